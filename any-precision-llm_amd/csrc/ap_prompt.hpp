// The parts of a Llama-architecture prompt that sit between the bitplane linears: rotary embedding + key/value cache
// write, and causal attention of the prompt's tokens over each other.  The reference calls the Hugging Face modules
// (any_precision/modules/AnyPrecisionForCausalLM.py:88-97); as torch ops they are fourteen launches a layer, among them
// two batched products over the whole static cache and four copies that only rearrange.
#pragma once
#include <math.h>

#include "ap_device.hpp"

namespace ap {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kPromptRopeThreads = 256;

// qkv [T, (nh + 2 nkv) HD]: token t's query, key and value heads before the rotary embedding; cache row of token t is t.
// Queries are rotated where they are, keys go to the cache rotated, values as they are.  A thread takes 8 dimensions of
// the lower half of a head and their partners in the upper half.  128 tokens of 3 x 32 heads of 128: 5 us, launch included
// (6 MB in and out; three torch ops and an indexed copy took 30).
template <int HD>
__global__ __launch_bounds__(kPromptRopeThreads) void prompt_rope_kernel(half_t *qkv, const float *__restrict__ cosT,
                                                                         const float *__restrict__ sinT, half_t *__restrict__ kcache,
                                                                         half_t *__restrict__ vcache, int T, int nh, int nkv, int max_len) {
    constexpr int HALF = HD / 2, UNITS = HALF / 8;
    const int heads = nh + 2 * nkv;
    const int per_token = heads * UNITS;
    const long long id = (long long)blockIdx.x * kPromptRopeThreads + threadIdx.x;
    const int t = (int)(id / per_token), u = (int)(id % per_token);
    if (t >= T) return;
    const int head = u / UNITS, i = (u % UNITS) * 8;
    half_t *src = qkv + ((size_t)t * heads + head) * HD + i;
    const half8_t a = *reinterpret_cast<const half8_t *>(src), b = *reinterpret_cast<const half8_t *>(src + HALF);
    if (head >= nh + nkv) {
        half_t *dst = vcache + ((size_t)(head - nh - nkv) * max_len + t) * HD + i;
        *reinterpret_cast<half8_t *>(dst) = a;
        *reinterpret_cast<half8_t *>(dst + HALF) = b;
        return;
    }
    const float *c = cosT + (size_t)t * HALF + i, *s = sinT + (size_t)t * HALF + i;
    half8_t lo, hi;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        lo[e] = (half_t)((float)a[e] * c[e] - (float)b[e] * s[e]);
        hi[e] = (half_t)((float)b[e] * c[e] + (float)a[e] * s[e]);
    }
    half_t *dst = head < nh ? src : kcache + ((size_t)(head - nh) * max_len + t) * HD + i;
    *reinterpret_cast<half8_t *>(dst) = lo;
    *reinterpret_cast<half8_t *>(dst + HALF) = hi;
}

// Rotary embedding of x [rows, heads, hd] (token-major, as a projection leaves it) into out of the same layout, with
// cos / sin [cos_rows, hd] in fp16 as the Hugging Face Llama model passes them; row r takes their row r % cos_rows.  fp32
// arithmetic, one rounding.  A thread takes 8 dimensions of the lower half of a head and their partners in the upper
// half.  Bound by memory: 1024 tokens of 32 heads of 128 (16 MB in and out) 6 us, launch included; as torch ops (two
// products, a sum, a negation and a concatenation, each over memory) 44 us.
__global__ __launch_bounds__(kPromptRopeThreads) void rope_heads_kernel(const half_t *__restrict__ x, const half_t *__restrict__ cosT,
                                                                        const half_t *__restrict__ sinT, half_t *__restrict__ out,
                                                                        int rows, int cos_rows, int heads, int hd) {
    const int half = hd / 2, units = hd / 16;
    const uint32_t per_row = (uint32_t)(heads * units), id = blockIdx.x * (uint32_t)kPromptRopeThreads + threadIdx.x;
    const uint32_t r = id / per_row, u = id % per_row;
    if (r >= (uint32_t)rows) return;
    const uint32_t head = u / (uint32_t)units, i = (u % (uint32_t)units) * 8;
    const size_t at = ((size_t)r * heads + head) * hd + i, tab = (size_t)(r % (uint32_t)cos_rows) * hd + i;
    const half8_t a = *reinterpret_cast<const half8_t *>(x + at), b = *reinterpret_cast<const half8_t *>(x + at + half);
    const half8_t c0 = *reinterpret_cast<const half8_t *>(cosT + tab), c1 = *reinterpret_cast<const half8_t *>(cosT + tab + half);
    const half8_t s0 = *reinterpret_cast<const half8_t *>(sinT + tab), s1 = *reinterpret_cast<const half8_t *>(sinT + tab + half);
    half8_t lo, hi;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        lo[e] = (half_t)((float)a[e] * (float)c0[e] - (float)b[e] * (float)s0[e]);
        hi[e] = (half_t)((float)b[e] * (float)c1[e] + (float)a[e] * (float)s1[e]);
    }
    *reinterpret_cast<half8_t *>(out + at) = lo;
    *reinterpret_cast<half8_t *>(out + at + half) = hi;
}

// Causal attention of queries first .. T-1 over keys 0 .. query; out [T - first, nh HD].
// A workgroup is one head and 64 queries, a wave 16 of them.  Scores are computed transposed, keys x queries: a lane then
// holds scores of ONE query (column l % 16) in every register, so maximum, rescaling and sum are per lane (four lanes
// share a query and meet by two exchanges), and the probabilities are already the B operand of the second product, output
// dimensions x queries, if its 32 keys are numbered as they lie: lane group g has keys 4g .. 4g+3 and 16+4g .. 16+4g+3.
// The matching A operand, values by dimension, comes from the tile of 32 values that the workgroup writes to LDS
// transposed; keys are read from the cache as they are (their rows are the A operand of the first product).
// fp16 operands, fp32 scores, softmax and sums.
// Bound by the chain of tiles of the last queries at short prompts: 128 tokens x 32 heads of 128, 64 workgroups, 10 us
// (11.4 with the keys loaded where they are used); torch's batched products, masks and copies took 60.
constexpr int kPromptAttnThreads = 256;
constexpr int kPromptQueries = 64;
template <int HD>
__global__ __launch_bounds__(kPromptAttnThreads) void prompt_attention_kernel(const half_t *__restrict__ qkv, int ldq,
                                                                              const half_t *__restrict__ kcache,
                                                                              const half_t *__restrict__ vcache,
                                                                              half_t *__restrict__ out, int first, int T, int nh,
                                                                              int group, int max_len, float scale_log2) {
    constexpr int NC = HD / 32, ND = HD / 16, KEYS = 32;
    constexpr int LD = KEYS + 8;                                   // halfs of a row of the transposed tile: 80 bytes
    constexpr int VPT = KEYS * HD / 8 / kPromptAttnThreads > 0 ? KEYS * HD / 8 / kPromptAttnThreads : 1;
    __shared__ __attribute__((aligned(16))) half_t vt[2][HD][LD];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave, col = lane & 15, g = lane >> 4;
    const int head = blockIdx.y, kvh = head / group;
    const int tile = (int)gridDim.x - 1 - (int)blockIdx.x;        // the longest rows of keys first
    const int q0 = first + tile * kPromptQueries + 16 * wave, query = q0 + col;
    const int last = min(first + tile * kPromptQueries + kPromptQueries, T) - 1;  // of the workgroup
    const half_t *kbase = kcache + (size_t)kvh * max_len * HD, *vbase = vcache + (size_t)kvh * max_len * HD;

    half8_t qf[NC];
    const half_t *qrow = qkv + (size_t)min(query, T - 1) * ldq + (size_t)head * HD;
#pragma unroll
    for (int c = 0; c < NC; c++) qf[c] = *reinterpret_cast<const half8_t *>(qrow + 32 * c + 8 * g);
    f32x4_t o[ND];
#pragma unroll
    for (int d = 0; d < ND; d++) o[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    // values of a tile: thread = key tid % 32 and units of 8 dimensions; rows past the prompt repeat its last one
    half8_t v[VPT];
    const int vkey = tid % KEYS, vunit = tid / KEYS;
    auto fetch = [&](int k0) {
        const half_t *row = vbase + (size_t)min(k0 + vkey, T - 1) * HD;
#pragma unroll
        for (int i = 0; i < VPT; i++) {
            const int u = vunit + i * (kPromptAttnThreads / KEYS);
            if (u < HD / 8) v[i] = *reinterpret_cast<const half8_t *>(row + 8 * u);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < VPT; i++) {
            const int u = vunit + i * (kPromptAttnThreads / KEYS);
            if (u < HD / 8)
#pragma unroll
                for (int e = 0; e < 8; e++) vt[buf][8 * u + e][vkey] = v[i][e];
        }
    };
    // keys of a tile, as the first product takes them; requested a tile ahead like the values: a tile is then one round of
    // products and not two trips to memory
    half8_t kf[2][NC];
    auto fetch_keys = [&](int k0) {
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
            const half_t *krow = kbase + (size_t)min(k0 + 16 * sub + col, T - 1) * HD + 8 * g;
#pragma unroll
            for (int c = 0; c < NC; c++) kf[sub][c] = *reinterpret_cast<const half8_t *>(krow + 32 * c);
        }
    };
    fetch(0);
    fetch_keys(0);
    stage(0);
    __syncthreads();
    for (int k0 = 0, buf = 0; k0 <= last; k0 += KEYS, buf ^= 1) {
        const bool more = k0 + KEYS <= last;
        if (more) fetch(k0 + KEYS);
        if (k0 <= q0 + 15) {  // some query of this wave sees the tile
            f32x4_t s[2];
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {
                s[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < NC; c++) s[sub] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[sub][c], qf[c], s[sub], 0, 0, 0);
            }
            if (more) fetch_keys(k0 + KEYS);
            float p[8], top = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int key = k0 + 16 * (i / 4) + 4 * g + i % 4;
                p[i] = key <= query ? s[i / 4][i % 4] * scale_log2 : -INFINITY;
                top = fmaxf(top, p[i]);
            }
            top = fmaxf(top, __shfl_xor(top, 16, kWave));
            top = fmaxf(top, __shfl_xor(top, 32, kWave));
            // -inf while every score so far is (keys that overflowed): measured against 0 then, so that such keys weigh nothing
            // and not NaN once a finite score follows
            const float mn = fmaxf(m, top), ref = mn == -INFINITY ? 0.f : mn;
            const float alpha = exp2f(m - ref);
            m = mn;
            half8_t pb;
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float e = exp2f(p[i] - ref);
                sum += e;
                pb[i] = (half_t)e;
            }
            l = l * alpha + sum;
#pragma unroll
            for (int d = 0; d < ND; d++) {
                const half4_t lo = *reinterpret_cast<const half4_t *>(&vt[buf][16 * d + col][4 * g]);
                const half4_t hi = *reinterpret_cast<const half4_t *>(&vt[buf][16 * d + col][16 + 4 * g]);
                const half8_t va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                o[d] *= alpha;
                o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb, o[d], 0, 0, 0);
            }
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (query < T) {
        const float r = 1.f / l;
        half_t *dst = out + ((size_t)(query - first) * nh + head) * HD + 4 * g;
#pragma unroll
        for (int d = 0; d < ND; d++) {
            half4_t y;
#pragma unroll
            for (int i = 0; i < 4; i++) y[i] = (half_t)(o[d][i] * r);
            *reinterpret_cast<half4_t *>(dst + 16 * d) = y;
        }
    }
}

}  // namespace ap
