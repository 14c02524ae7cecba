// The parts of a Llama-architecture decode step that sit between the bitplane linears, for ONE new
// token: residual add + RMSNorm, SiLU(gate) * up, and rotary embedding + key/value cache append +
// attention over the cache.  The reference has no kernels for them: its model wrapper calls the Hugging
// Face modules (any_precision/modules/AnyPrecisionForCausalLM.py:88-97), which at batch 1 cost a dozen
// launch-bound library kernels per layer between two GEMVs.  fp16 in memory, fp32 arithmetic, one rounding
// per output.
#pragma once
#include <math.h>

#include <type_traits>

#include "ap_device.hpp"

namespace ap {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

constexpr int kAttnThreads = 1024;  // sixteen waves: the kernel is a chain of load latencies, more waves = more loads in flight
constexpr int kAttnMaxLen = 8192;  // cache rows one launch attends over: the limit of the entry point (the kernel itself keeps nothing per row)

// One workgroup per row of H elements (H % 8 == 0):
//     s = h + delta (rounded to fp16, as an fp16 add; delta only with DELTA), written to h_out;
//     x_out = s * rsqrt(mean(s^2) + eps) * weight.
// h_out may alias h.  A thread has HELD units of 8 elements in registers between the two passes, all of them (and their
// deltas and weights) requested before the first is used, without a branch on the way: a unit past the row's end loads the
// row's last one and counts for nothing.  What is past HELD units of longer rows is re-read.
// Bound by its chain at a decoder's one row (scalar arguments, one trip to memory for what the linear before has written from
// every XCD, the reduction, the store); with 256 threads and the units one after the other that were two to four trips.
// 48 tokens with 32 layers of 4096 (65 launches a token): 68.8 -> 66.2 ms, 0.85 us a launch.
constexpr int kNormMaxThreads = 1024;
template <int HELD, bool DELTA>
__global__ __launch_bounds__(kNormMaxThreads) void add_rmsnorm_kernel(const half_t *h, const half_t *delta,
                                                                      const half_t *__restrict__ weight, half_t *h_out,
                                                                      half_t *__restrict__ x_out, int H, float eps) {
    __shared__ float red[kNormMaxThreads / kWave];
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x, waves = (int)blockDim.x / kWave;
    const int step = (int)blockDim.x * 8;
    const half_t *hr = h + row * H;
    const half_t *dr = DELTA ? delta + row * H : nullptr;
    half_t *ho = h_out + row * H;
    const bool rewrite = DELTA || ho != hr;
    half8_t held[HELD], dheld[HELD], wheld[HELD];
#pragma unroll
    for (int c = 0; c < HELD; c++) {
        const int i = min(tid * 8 + c * step, H - 8);
        held[c] = *reinterpret_cast<const half8_t *>(hr + i);
        if (DELTA) dheld[c] = *reinterpret_cast<const half8_t *>(dr + i);
        wheld[c] = *reinterpret_cast<const half8_t *>(weight + i);
    }
    float ss = 0.f;
    auto add = [&](half8_t &a, const half8_t &b) {
#pragma unroll
        for (int e = 0; e < 8; e++) a[e] = (half_t)((float)a[e] + (float)b[e]);
    };
    auto squares = [&](const half8_t &a) {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) s += (float)a[e] * (float)a[e];
        return s;
    };
#pragma unroll
    for (int c = 0; c < HELD; c++) {
        if (DELTA) add(held[c], dheld[c]);
        ss += tid * 8 + c * step < H ? squares(held[c]) : 0.f;
    }
    if constexpr (HELD > 1)
        for (int i = tid * 8 + HELD * step; i < H; i += step) {
            half8_t a = *reinterpret_cast<const half8_t *>(hr + i);
            if (DELTA) add(a, *reinterpret_cast<const half8_t *>(dr + i));
            if (rewrite) *reinterpret_cast<half8_t *>(ho + i) = a;
            ss += squares(a);
        }
    ss = wave_sum(ss);
    if ((tid & (kWave - 1)) == kSumLane) red[tid / kWave] = ss;
    __syncthreads();
    // a lane takes the sum of one wave; rotations within the 16 lanes of a DPP row add them up in every lane
    static_assert(kNormMaxThreads / kWave == 16, "one DPP row holds the sums of all waves");
    const int w = tid & 15;
    float total = red[min(w, waves - 1)];
    total = w < waves ? total : 0.f;
    total = dpp_add<0x128>(total);  // row_ror:8
    total = dpp_add<0x124>(total);
    total = dpp_add<0x122>(total);
    total = dpp_add<0x121>(total);
    const float rs = rsqrtf(total / (float)H + eps);
    auto scaled = [&](const half8_t &a, const half8_t &g, int i) {
        half8_t y;
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = (half_t)((float)a[e] * rs * (float)g[e]);
        *reinterpret_cast<half8_t *>(x_out + row * H + i) = y;
    };
#pragma unroll
    for (int c = 0; c < HELD; c++) {
        const int i = tid * 8 + c * step;
        if (i < H) {
            // the last unit of an aliased row is read by other threads too: it is written behind the barrier
            if (rewrite) *reinterpret_cast<half8_t *>(ho + i) = held[c];
            scaled(held[c], wheld[c], i);
        }
    }
    if constexpr (HELD > 1) {
        const half_t *src = rewrite ? ho : hr;  // every thread re-reads exactly what it wrote
        for (int i = tid * 8 + HELD * step; i < H; i += step)
            scaled(*reinterpret_cast<const half8_t *>(src + i), *reinterpret_cast<const half8_t *>(weight + i), i);
    }
}

// out = gate / (1 + exp(-gate)) * up over n elements (n % 8 == 0).  out may be gate or up: a thread reads its 8 elements before
// it writes them, and no other thread touches them.
__global__ __launch_bounds__(256) void silu_mul_kernel(const half_t *gate, const half_t *up, half_t *out, long long n) {
    const long long stride = (long long)gridDim.x * blockDim.x * 8;
    for (long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * 8; i < n; i += stride) {
        const half8_t g = *reinterpret_cast<const half8_t *>(gate + i);
        const half8_t u = *reinterpret_cast<const half8_t *>(up + i);
        half8_t y;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x = (float)g[e];
            y[e] = (half_t)(x / (1.f + __expf(-x)) * (float)u[e]);
        }
        *reinterpret_cast<half8_t *>(out + i) = y;
    }
}

// Greedy token selection and the bookkeeping of a decode step in one workgroup:
//     t = argmax(logits[0 .. n))  (the first index of the maximum; a NaN counts as the maximum, as torch.argmax has it);
//     p = *pos + 1; if p < max_len: emitted[p] = t, *pos = p;  *tok = t.
// Replaces an argmax reduction, an increment, an indexed store and a copy -- four launch-bound library kernels.
constexpr int kAdvanceThreads = 1024;
__global__ __launch_bounds__(kAdvanceThreads) void decode_advance_kernel(const half_t *__restrict__ logits, int n,
                                                                        long long *pos, long long *tok, long long *emitted,
                                                                        int max_len) {
    __shared__ float best_v[kAdvanceThreads / kWave];
    __shared__ int best_i[kAdvanceThreads / kWave];
    const int tid = threadIdx.x;
    // a > b in the order "NaN above everything, then by value, then the lower index"
    auto better = [](float av, int ai, float bv, int bi) {
        const bool an = av != av, bn = bv != bv;
        if (an != bn) return an;
        if (!an && av != bv) return av > bv;
        return ai < bi;
    };
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    const int nv = n / 8;  // whole 16-byte groups; the rest one by one
    constexpr int AHEAD = 4;  // 16-byte groups requested together: the scan is one chain of load latencies otherwise
    for (int g0 = tid; g0 < nv; g0 += AHEAD * kAdvanceThreads) {
        half8_t v[AHEAD];
#pragma unroll
        for (int a = 0; a < AHEAD; a++) {
            const int g = g0 + a * kAdvanceThreads;
            v[a] = reinterpret_cast<const half8_t *>(logits)[g < nv ? g : g0];
        }
#pragma unroll
        for (int a = 0; a < AHEAD; a++) {
            const int g = g0 + a * kAdvanceThreads;
            if (g < nv) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float f = (float)v[a][e];
                    if (better(f, g * 8 + e, bv, bi)) {
                        bv = f;
                        bi = g * 8 + e;
                    }
                }
            }
        }
    }
    for (int i = nv * 8 + tid; i < n; i += kAdvanceThreads) {
        const float f = (float)logits[i];
        if (better(f, i, bv, bi)) {
            bv = f;
            bi = i;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float ov = __shfl_xor(bv, off, kWave);
        const int oi = __shfl_xor(bi, off, kWave);
        if (better(ov, oi, bv, bi)) {
            bv = ov;
            bi = oi;
        }
    }
    if ((tid & (kWave - 1)) == 0) {
        best_v[tid / kWave] = bv;
        best_i[tid / kWave] = bi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kAdvanceThreads / kWave; w++)
            if (better(best_v[w], best_i[w], bv, bi)) {
                bv = best_v[w];
                bi = best_i[w];
            }
        const long long p = *pos + 1;
        if (p >= 0 && p < max_len) {
            emitted[p] = bi;
            *pos = p;
        }
        *tok = bi;
    }
}

// Attention of one new token at cache row pos = *pos_p, one workgroup per query head; `group` query heads share a key head.
//   qkv     [n_heads + 2 n_kv_heads, HD]: the token's query, key and value heads before the rotary embedding
//   cosT, sinT [max_len, HD / 2] fp32: cos / sin of position * inverse frequency i
//   kcache, vcache [n_kv_heads, max_len, HD]: rows 0 .. pos-1 are read; row pos is written (rotated key, value)
//           by the first query head of each key/value group -- every workgroup uses its own copy of that row
//           from LDS, never the one in memory
//   out     [n_heads * HD]
// Rotary convention of the Hugging Face Llama model: x * cos + rotate_half(x) * sin with
// rotate_half(x) = (-x[HD/2:], x[:HD/2]).  Scores = (q . k) * scale, softmax and the weighted sum in fp32.
// A position outside 0 .. max_len-1 makes every workgroup return without touching memory.
//
// A chain of latencies at a decoder's lengths: arguments, position, rows, and what stands between the barriers.  So a wave takes its keys all the way
// -- scores, softmax with its own running maximum, weighted sum -- and the workgroup meets twice: behind the rotary embedding, with the
// first rows on their way, and to add the waves' parts, each scaled from its maximum to the largest.  LPK lanes share a key, 8 elements each; a
// step is the KPW keys of every wave, and up to four are requested together (no loads of keys that are not there: they cost more than a
// later start).  us with the phases one after the other and six barriers / so: 32 heads of 128 at position 40 4.95 / 3.68, at 80 5.20 / 3.85, at 383
// 7.2 / 5.6, at 2000 35 / 22; 8 heads of 256 at 383 13.4 / 7.8; 16 heads of 64 at 80 5.13 / 4.01.  Results further than half an ulp of
// fp16 from the exact ones, of 69632 (heads of 128, up to 60 keys): 63 / 46.
template <int HD>
__global__ __launch_bounds__(kAttnThreads) void decode_attention_kernel(
    const half_t *__restrict__ qkv, const float *__restrict__ cosT, const float *__restrict__ sinT, half_t *kcache,
    half_t *vcache, const long long *__restrict__ pos_p, half_t *__restrict__ out, int nh, int nkv, int group,
    int max_len, float scale) {
    constexpr int HALF = HD / 2;
    constexpr int NW = kAttnThreads / kWave;
    constexpr int LPK = HD / 8;             // lanes per key
    constexpr int KPW = kWave / LPK;        // keys per wave and step
    constexpr int STEP = NW * KPW;
    constexpr int MOST = 4;                 // steps requested together
    static_assert(HD % 32 == 0 && HD <= 256 && HD <= kAttnThreads, "");
    __shared__ __attribute__((aligned(16))) float q_s[HD], kn_s[HD], vn_s[HD];
    __shared__ float max_s[NW], sum_s[NW];
    __shared__ __attribute__((aligned(16))) float part_s[NW][HD];

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int head = blockIdx.x, kvh = head / group;
    const bool writer = head == kvh * group;
    const int dl = lane % LPK, sub = lane / LPK;

    // ---- waves 0, 1, 2: the query, the new key (and the new row of the cache) and the new value into LDS
    const half_t *const mine = qkv + (size_t)(wave == 0 ? head : (wave == 1 ? nh + kvh : nh + nkv + kvh)) * HD;
    constexpr int PER = (HALF + kWave - 1) / kWave;
    half_t lo[PER], hi[PER];
    if (wave < 3)
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int i = min(lane + r * kWave, HALF - 1);
            lo[r] = mine[i];
            hi[r] = mine[i + HALF];
        }
    const long long p64 = *pos_p;
    if (p64 < 0 || p64 >= max_len) return;  // uniform over the grid
    const int pos = (int)p64;
    const int steps = (pos + STEP - 1) / STEP;
    const half_t *const kbase = kcache + (size_t)kvh * max_len * HD + dl * 8, *const vbase = vcache + (size_t)kvh * max_len * HD + dl * 8;
    const int first = wave * KPW + sub;     // this lane's key of step 0

    auto fresh_rows = [&]() {
        if (wave >= 3) return;
        float *const dst = wave == 0 ? q_s : (wave == 1 ? kn_s : vn_s);
#pragma unroll
        for (int r = 0; r < PER; r++) {
            const int i = lane + r * kWave;
            if (i >= HALF) break;
            float a = (float)lo[r], b = (float)hi[r];
            if (wave < 2) {
                const float c = cosT[(size_t)pos * HALF + i], s = sinT[(size_t)pos * HALF + i];
                if (wave == 0) {
                    const float x1 = a, x2 = b, base2 = scale * 1.44269504088896341f;   // scores to base 2
                    a = (x1 * c - x2 * s) * base2;
                    b = (x2 * c + x1 * s) * base2;
                } else {
                    // rounded by the instruction that adds, as the rows of a prompt are
                    const half_t y1 = (half_t)((float)lo[r] * c - (float)hi[r] * s), y2 = (half_t)((float)hi[r] * c + (float)lo[r] * s);
                    a = (float)y1;
                    b = (float)y2;
                }
            }
            dst[i] = a;
            dst[i + HALF] = b;
            if (wave > 0 && writer) {
                half_t *const row = (wave == 1 ? kcache : vcache) + ((size_t)kvh * max_len + pos) * HD;
                row[i] = (half_t)a;
                row[i + HALF] = (half_t)b;
            }
        }
    };
    auto over_key = [](float s) {           // the sum over the lanes of a key
        s = dpp_add<0xB1>(s);
        s = dpp_add<0x4E>(s);
        if constexpr (LPK >= 8) s = dpp_add<0x141>(s);
        if constexpr (LPK >= 16) s = dpp_add<0x140>(s);
        if constexpr (LPK >= 32) s += __shfl_xor(s, 16, kWave);
        return s;
    };
    float m = -INFINITY, l = 0.f, acc[8];   // of this lane's keys: maximum, sum of exp(score - m), weighted sum of 8 elements
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.f;
    float q[8];
    // The rotary embedding, and what needs no row of the cache: the new key is the first wave's first.  The rows requested before stay on their way
    // in the waves that only wait here; waves 0 to 2 have theirs when they come to the barrier: loads complete in order, cosines and sines
    // come behind them, and wave 2 shares the wait.
    auto meet = [&]() {
        fresh_rows();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
        for (int e = 0; e < 8; e++) q[e] = q_s[dl * 8 + e];
        if (wave == 0) {
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) s += kn_s[dl * 8 + e] * q[e];
            s = over_key(s);
            if (sub == 0) {
                m = s;
                l = s == -INFINITY ? 0.f : s - s + 1.f;    // nothing at -inf, as any other key; NaN where the score is NaN or +inf
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] = l * vn_s[dl * 8 + e];
            }
        }
    };
    // scores of U keys and their values (score -inf: no key)
    auto take = [&](auto u_c, const float (&s)[MOST], const half8_t (&v)[MOST]) {
        constexpr int U = decltype(u_c)::value;
        float top = m;
#pragma unroll
        for (int u = 0; u < U; u++) top = fmaxf(top, s[u]);
        const float base = top == -INFINITY ? 0.f : top, old = __builtin_amdgcn_exp2f(m - base);
        l *= old;
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] *= old;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const float p = __builtin_amdgcn_exp2f(s[u] - base);
            l += p;
#pragma unroll
            for (int e = 0; e < 8; e++) acc[e] += p * (float)v[u][e];
        }
        m = top;
    };
    // U steps from step t on, the last of which may have lanes past the end; FIRST: the query is not there yet
    auto run = [&](auto u_c, auto first_c, int t) {
        constexpr int U = decltype(u_c)::value;
        half8_t k[MOST], v[MOST];
        float s[MOST];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = min(first + (t + u) * STEP, pos - 1);
            k[u] = *reinterpret_cast<const half8_t *>(kbase + (size_t)j * HD);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = min(first + (t + u) * STEP, pos - 1);
            v[u] = *reinterpret_cast<const half8_t *>(vbase + (size_t)j * HD);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(first_c)::value) meet();
#pragma unroll
        for (int u = 0; u < U; u++) {
            float a = 0.f, b = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                a += (float)k[u][e] * q[e];
                b += (float)k[u][e + 1] * q[e + 1];
            }
            s[u] = over_key(a + b);
            if (u == U - 1 && first + (t + u) * STEP >= pos) {
                s[u] = -INFINITY;
                v[u] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
            }
        }
        take(u_c, s, v);
    };
    int t = 0;
    if (steps == 0) meet();
    else if (steps == 1) run(std::integral_constant<int, 1>{}, std::true_type{}, 0);
    else if (steps == 2) run(std::integral_constant<int, 2>{}, std::true_type{}, 0);
    else if (steps == 3) run(std::integral_constant<int, 3>{}, std::true_type{}, 0);
    else {
        run(std::integral_constant<int, 4>{}, std::true_type{}, 0);
        for (t = 4; t + 4 <= steps; t += 4) run(std::integral_constant<int, 4>{}, std::false_type{}, t);
        const int left = steps - t;
        if (left == 1) run(std::integral_constant<int, 1>{}, std::false_type{}, t);
        else if (left == 2) run(std::integral_constant<int, 2>{}, std::false_type{}, t);
        else if (left == 3) run(std::integral_constant<int, 3>{}, std::false_type{}, t);
    }
    // ---- the wave's keys together, then the waves'
    float top = m;
#pragma unroll
    for (int off = kWave / 2; off >= LPK; off /= 2) top = fmaxf(top, __shfl_xor(top, off, kWave));
    const float f = __builtin_amdgcn_exp2f(m - (top == -INFINITY ? 0.f : top));
    l *= f;
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] *= f;
#pragma unroll
    for (int off = kWave / 2; off >= LPK; off /= 2) {
        l += __shfl_xor(l, off, kWave);
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] += __shfl_xor(acc[e], off, kWave);
    }
    if (sub == 0) {
#pragma unroll
        for (int e = 0; e < 8; e++) part_s[wave][dl * 8 + e] = acc[e];
    }
    if (lane == 0) {
        max_s[wave] = top;
        sum_s[wave] = l;
    }
    __syncthreads();
    if (tid >= HD) return;
    float all = max_s[0], sum = 0.f, g[NW], y = 0.f;
#pragma unroll
    for (int w = 1; w < NW; w++) all = fmaxf(all, max_s[w]);
#pragma unroll
    for (int w = 0; w < NW; w++) {
        g[w] = __builtin_amdgcn_exp2f(max_s[w] - all);
        sum += sum_s[w] * g[w];
    }
    const float whole = 1.f / sum;
#pragma unroll
    for (int w = 0; w < NW; w++) y += part_s[w][tid] * g[w];
    out[(size_t)head * HD + tid] = (half_t)(y * whole);
}

}  // namespace ap
