// Staged K-split fused bitplane dequant -> MFMA GEMM for gfx950, 1 <= M <= 32 activation rows:
//     out[m,n] = sum_k x[m,k] * lut[n, index_b(n,k)]      (fp16 operands, fp32 accumulate)
//
// What bounds such a call is the time a wave spends waiting, not the rate of any unit: a linear of a decoder layer has 5..60 MB of planes, a few us
// at the rate of memory, on workgroups that live for a few steps each.  So a workgroup is small -- 16 weight rows, 4 waves that share the words
// of K, two or three workgroups a CU -- and every wave keeps its whole next step in flight: the planes in registers, the activations in a ring in
// LDS that is the wave's own, so that no barrier stands between the tables' and the last one.  The waits count (load_to_lds, GemmsOrder): a
// stage is waited for ahead of its first read, while the loads behind it stay out.  The loads of a wave's first step are the exception: the release
// ahead of the tables' barrier is for LDS, which direct loads write, and waits for all that is outstanding.
//  - Activations come by direct loads of rows of 256 bytes, a byte group of a step each; read from global memory by every wave's lanes in
//    pieces of 16 or 64 bytes, as the other K-split kernel does, they cost more than the weights from 9 rows on.  A row's 16-byte units are
//    permuted by its number, and the reads of an octet are free of conflicts.
//  - Tables lie [entry][slot], 16 weight rows x up to 4 copies: a lane's bank depends on its slot only.  Pairs of entries at 3 and 4 bits.
//  - Weights are the matrix instruction's first operand, so that a lane ends with 4 weight rows of one activation row: one store of 8 bytes.
//  - The waves' sums meet in LDS in the place of the first stage, and are added in the order of the waves.
// Measured, us before / here: 4096 x 11008 at 16 rows, 3 bits 17.6 / 11.0 (the floor of its planes 2.6), 5 bits 21.3 / 15.3, 8 bits 27.3 / 21.0;
// 4096 x 4096 at 16 rows, 4 bits 8.4 / 6.9; 4096 x 14336 at 4 rows, 4 bits 15.7 / 11.3; 14336 x 4096 at 8 rows, 4 bits 17.8 / 13.8.
// Slower: 8 waves (11008 x 4096 at 16 rows, 4 bits 13.4 -> 18.2), 2 waves, 16 waves on 2 words each, a ring of 2 stages (10-25 %), workgroups
// that walk over blocks of weight rows with their tables fetched ahead.
#pragma once
#include <type_traits>

#include "ap_bitplane.hpp"
#include "ap_device.hpp"
#include "ap_gemms_launch.hpp"

namespace ap {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// What a workgroup takes of the LDS: the tables, and of every wave a ring of stages.  Four stages, all of a step, wherever a single copy of
// the tables leaves room (with two, the loads of a step's second half start when its first half is done: 4096 x 11008 at 4 rows, 4 bits
// 10.7 -> 12.8 us), then as many copies of the tables as fit: 64 slots give every lane a bank of its own, and addresses by one v_perm_b32.
// The limit is two workgroups a CU, three up to 8 rows (14336 x 4096 at 4 rows, 4 bits: 12.7 us with three, 15.7 with two).
template <int BITS, int ROWS>
struct GemmsLds {
    static constexpr bool kPair = BITS <= 4;
    static constexpr int kEntries = kPair ? 1 << (2 * BITS) : 1 << BITS;
    static constexpr int kStage = ROWS * 256;              // a wave's activations of one byte group of a step
    static constexpr int kSums = ROWS > 16 ? 2048 : 1024;  // a wave's sums; they take the place of its first stage
    static_assert(kSums <= kStage, "");
    static constexpr int kLimit = (ROWS <= 8 ? 53 : 80) * 1024;
    static constexpr bool fits(int ring, int slots) { return kEntries * slots * 4 + kGemmsWaves * ring * kStage <= kLimit; }
    static constexpr int kRing = fits(4, 16) ? 4 : 2;
    static constexpr int kSlots = fits(kRing, 64) ? 64 : (fits(kRing, 32) ? 32 : 16);
    static_assert(fits(kRing, kSlots), "");
    static constexpr int kCopies = kSlots / 16;
};

// What a wave has requested behind a stage when the first read of that stage is due, in the order in which run_step requests: the stages of the
// ring (DMA loads each) lie ahead of the step; with NEXT its first loads are the BITS planes of the next one; a stage's buffer is refilled
// behind its last products -- in a ring of four after the first reads of the stage behind it, in a ring of two before them.  Loads
// complete in order: when no more than behind(j) are outstanding, stage j has landed.
template <int BITS, int RING, int DMA, bool NEXT>
struct GemmsOrder {
    static constexpr int behind(int j) {
        int requested = RING * DMA, landed[4] = {};  // landed[k]: requests up to the last of stage k
        for (int k = 0; k < RING; k++) landed[k] = (k + 1) * DMA;
        if (NEXT) requested += BITS;
        for (int k = 0; k < j; k++) {  // the end of stage k, up to the reads of stage k + 1
            if (RING == 4 && k + 1 == j) break;
            if (RING == 4 ? NEXT : (k < 2 || NEXT)) requested += DMA;
            if (RING == 2 && k < 2) landed[k + 2] = requested;
        }
        return requested - landed[j];
    }
    static_assert(RING == 2 || RING == 4, "");
    static_assert(behind(0) == (RING - 1) * DMA + (NEXT ? BITS : 0), "");
    static_assert(RING == 4 || (behind(1) == behind(0) && behind(2) == DMA && behind(3) == (NEXT ? DMA : 0)), "");
    static_assert(RING == 2 || !NEXT || (behind(1) == 2 * DMA + BITS && behind(2) == behind(1) && behind(3) == behind(1)), "");
    static_assert(RING == 2 || NEXT || (behind(1) == 2 * DMA && behind(2) == DMA && behind(3) == 0), "");
};

// Grid: a workgroup of (64, 4) threads per block of 16 weight rows of all members.  ROWS: activation rows staged (M <= ROWS).
template <int BITS, int ROWS>
__global__ __launch_bounds__(kGemmsWaves *kWave, ROWS <= 8 ? 3 : 2) void gemms_kbit_kernel(const half_t *__restrict__ x, const GemmsMembers mem,
                                                                                          int M, int K) {
    using Lds = GemmsLds<BITS, ROWS>;
    constexpr bool PAIR = Lds::kPair;
    constexpr int NC = 1 << BITS, SLOTS = Lds::kSlots, RING = Lds::kRing, COPIES = Lds::kCopies, WAVES = kGemmsWaves;
    constexpr int MB = ROWS > 16 ? 2 : 1;
    constexpr int DMA = ROWS / 4;  // direct loads of a stage
    __shared__ __attribute__((aligned(256))) uint32_t tables[Lds::kEntries * SLOTS];
    __shared__ u32x4 x0[WAVES][ROWS][16], x1[WAVES][ROWS][16];
    __shared__ u32x4 x2[RING == 4 ? WAVES : 1][RING == 4 ? ROWS : 1][16], x3[RING == 4 ? WAVES : 1][RING == 4 ? ROWS : 1][16];

    const int lane = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int row = lane & 15, quad = lane >> 4;

    uint64_t x_i = reinterpret_cast<uint64_t>(x), q_i = reinterpret_cast<uint64_t>(mem.qweight[0]), lut_i = reinterpret_cast<uint64_t>(mem.lut[0]),
             out_i = reinterpret_cast<uint64_t>(mem.out[0]), bias_i = reinterpret_cast<uint64_t>(mem.bias);
    int N = mem.N[0], count = mem.count, b1 = mem.block0[1], b2 = mem.block0[2], b3 = mem.block0[3];
    long long ldo = mem.ldo[0];
    asm volatile("" : "+s"(x_i), "+s"(q_i), "+s"(lut_i), "+s"(out_i), "+s"(bias_i), "+s"(N), "+s"(count), "+s"(b1), "+s"(b2), "+s"(b3), "+s"(ldo),
                      "+s"(M), "+s"(K));
    const int block = blockIdx.x;
    int first = 0;
    if (count > 1) {
        int g = block >= b1 ? 1 : 0;
        g = (count > 2 && block >= b2) ? 2 : g;
        g = (count > 3 && block >= b3) ? 3 : g;
        if (g > 0) {
            q_i = reinterpret_cast<uint64_t>(mem.qweight[g]);
            lut_i = reinterpret_cast<uint64_t>(mem.lut[g]);
            out_i = reinterpret_cast<uint64_t>(mem.out[g]);
            N = mem.N[g];
            ldo = mem.ldo[g];
            first = g == 1 ? b1 : (g == 2 ? b2 : b3);
        }
    }
    const global_ptr<const char> planes = (global_ptr<const char>)q_i, luts = (global_ptr<const char>)lut_i;
    const uint32_t x_bytes = (uint32_t)M * (uint32_t)K * 2u;
    const int W = K >> 5, T = (W + 15) >> 4;
    const int n0 = (block - first) * kGemmsRows;
    const size_t plane_bytes = (size_t)N * W * 4;
    const uint32_t prow = (uint32_t)min(n0 + row, N - 1) * (uint32_t)W * 4u;

    // ---- planes of a step: 16 words of the 16 rows, a lane the words 4 quad .. + 3 of its row
    u32x4 q[BITS];
    auto fetch = [&](int step) {
        const uint32_t off = prow + 4u * (uint32_t)min(16 * step + 4 * quad, W - 4);
#pragma unroll
        for (int p = 0; p < BITS; p++) q[p] = load_at_nt<u32x4>(planes + p * plane_bytes, off);
    };

    // ---- tables: [entry][slot] dwords, slot = 16 copy + row; an item is 8 entries of one row and copy
    constexpr int PARTS = Lds::kEntries / 8, ITEMS = 16 * COPIES * PARTS, THREADS = WAVES * kWave;
    constexpr int PER = (ITEMS + THREADS - 1) / THREADS;
    const int tid = wave * kWave + lane;
    u32x4 t4[PER];
    auto fetch_tables = [&]() {
#pragma unroll
        for (int it = 0; it < PER; it++) {
            const int item = min(tid + it * THREADS, ITEMS - 1), r = item & 15, part = item / (16 * COPIES);
            const uint32_t at = (uint32_t)min(n0 + r, N - 1) * (uint32_t)(2 * NC);
            if constexpr (PAIR) {
                const uint32_t g = (uint32_t)part;
                const uint32_t f = BITS == 3 ? ((g >> 1) & 2u) | (g & 1u) : ((g >> 2) & 4u) | ((g >> 1) & 2u) | (g & 1u);
                const uint32_t s = BITS == 3 ? (g >> 1) & 1u : ((g >> 2) & 2u) | ((g >> 1) & 1u);
                t4[it][0] = load_at<uint32_t>(luts, at + 4u * f);
                const u32x2 v = load_at<u32x2>(luts, at + 8u * s);
                t4[it][1] = v[0];
                t4[it][2] = v[1];
            } else {
                t4[it] = load_at<u32x4>(luts, at + 16u * (uint32_t)part);
            }
        }
    };
    auto put_tables = [&]() {
#pragma unroll
        for (int it = 0; it < PER; it++) {
            const int item = tid + it * THREADS;
            if (ITEMS % THREADS != 0 && item >= ITEMS) break;
            const int r = item & 15, copy = (item >> 4) % COPIES, part = item / (16 * COPIES);
            uint32_t *dst = tables + part * 8 * SLOTS + copy * 16 + r;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                uint32_t v;
                if constexpr (PAIR)  // low half: weight f0 of the first word, high half: weight s0 of the second
                    v = __builtin_amdgcn_perm(t4[it][1 + (k >> 2)], t4[it][0], ((k & 1) ? 0x07060000u : 0x05040000u) | ((k & 2) ? 0x0302u : 0x0100u));
                else
                    v = (k & 1) ? t4[it][k / 2] >> 16 : t4[it][k / 2] & 0xffffu;
                dst[k * SLOTS] = v;
            }
        }
    };

    // ---- activations of a stage (byte group j of a step): ROWS rows of 256 bytes, a direct load brings four of them, the 16-byte units of a
    // row permuted by its number
    uint32_t xrow[DMA], xunit[DMA];
#pragma unroll
    for (int i = 0; i < DMA; i++) {
        const int m = 4 * i + quad;
        xunit[i] = (uint32_t)(row ^ (m & 15));
        xrow[i] = (uint32_t)min(m, M - 1) * (uint32_t)K * 2u;
    }
    auto ring = [&](auto b_c) -> auto & {
        constexpr int b = decltype(b_c)::value;
        if constexpr (b == 0) return x0;
        else if constexpr (b == 1) return x1;
        else if constexpr (b == 2) return x2;
        else return x3;
    };
    auto stage = [&](int step, auto j_c) {
        constexpr int j = decltype(j_c)::value;
        auto &buf = ring(std::integral_constant<int, j % RING>{});
        const int w0 = 16 * step, chunk = w0 >> 5;
        const uint32_t stride = chunk == (W >> 5) ? (uint32_t)(W & 31) * 16u : 512u;
        const uint32_t at = ((uint32_t)chunk << 11) + ((uint32_t)(w0 & 31) << 4) + (uint32_t)j * stride;
        const uint32_t last = (uint32_t)(W - 1 - w0);  // units past the row's end fetch its last one
#pragma unroll
        for (int i = 0; i < DMA; i++)
            load_to_lds(x_i, x_bytes, (__attribute__((address_space(3))) void *)&buf[wave][4 * i][0], xrow[i] + 16u * min(xunit[i], last), at);
    };

    typedef __attribute__((address_space(3))) uint16_t lds_u16_t;
    typedef __attribute__((address_space(3))) uint32_t lds_u32_t;
    typedef __attribute__((address_space(3))) uint8_t lds_u8_t;
    const lds_u8_t *const tables_lds = (const lds_u8_t *)&tables[0];
    const uint32_t slot_byte = (uint32_t)(lane & (SLOTS - 1)) * 4u;

    float4_t acc[MB];
    constexpr int NRAW = PAIR ? 4 : 8;
    uint32_t idx[4][NRAW];
    auto convert = [&]() {
#pragma unroll
        for (int w = 0; w < 4; w++) {
            uint32_t pl[BITS];
#pragma unroll
            for (int p = 0; p < BITS; p++) pl[p] = q[p][w];
            if constexpr (PAIR) {  // as planes_to_adjacent_pairs, the entry in the low bits of its byte
                uint32_t r[4] = {pl[BITS - 1], pl[BITS - 2], pl[BITS - 3], BITS == 4 ? pl[0] : 0u};
                swap_blocks<4, 0x0F0F0F0Fu>(r[0], r[2]);
                swap_blocks<4, 0x0F0F0F0Fu, false, BITS == 3>(r[1], r[3]);
                swap_blocks<2, 0x33333333u>(r[0], r[1]);
                swap_blocks<2, 0x33333333u>(r[2], r[3]);
#pragma unroll
                for (int i = 0; i < 4; i++) idx[w][i] = r[3 - i];
            } else {
                planes_to_indices<BITS>(pl, idx[w]);
            }
        }
    };
    half8_t af[2][2][MB];
    uint32_t raw[2][2][NRAW];
    const int xm = row & (ROWS < 16 ? ROWS - 1 : 15);
    // operands of octets 2 h, 2 h + 1 (words of the lane's quad) of stage j into set s
    auto request = [&](auto j_c, auto h_c, auto s_c) {
        constexpr int j = decltype(j_c)::value, h = decltype(h_c)::value, s = decltype(s_c)::value, c = 3 - j;
        auto &buf = ring(std::integral_constant<int, j % RING>{});
#pragma unroll
        for (int o = 0; o < 2; o++) {
#pragma unroll
            for (int i = 0; i < NRAW; i++) {
                uint32_t a;
                const uint32_t word = idx[2 * h + o][i];
                if constexpr (SLOTS == 64) a = __builtin_amdgcn_perm(word, slot_byte, 0x0c0c0000u | ((4u + c) << 8));
                else a = (__builtin_amdgcn_ubfe(word, 8 * c, 8) * (4u * SLOTS)) | slot_byte;
                if constexpr (PAIR) raw[s][o][i] = *reinterpret_cast<const lds_u32_t *>(tables_lds + a);
                else raw[s][o][i] = *reinterpret_cast<const lds_u16_t *>(tables_lds + a);
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
                af[s][o][mb] = __builtin_bit_cast(half8_t, buf[wave][16 * mb + xm][(4 * quad + 2 * h + o) ^ xm]);
        }
    };
    auto multiply = [&](auto s_c, auto check_c, bool live) {
        constexpr int s = decltype(s_c)::value;
#pragma unroll
        for (int o = 0; o < 2; o++) {
            u32x4 bw;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (PAIR) bw[i] = raw[s][o][i];
                else bw[i] = raw[s][o][2 * i] | (raw[s][o][2 * i + 1] << 16);
                if constexpr (decltype(check_c)::value) bw[i] = live ? bw[i] : 0u;
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                u32x4 a = __builtin_bit_cast(u32x4, af[s][o][mb]);
                if constexpr (decltype(check_c)::value)
#pragma unroll
                    for (int i = 0; i < 4; i++) a[i] = live ? a[i] : 0u;
                acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, bw), __builtin_bit_cast(half8_t, a), acc[mb], 0, 0, 0);
            }
        }
    };
    auto wait = [&](auto n_c) {
        constexpr int n = decltype(n_c)::value;
        static_assert(n < 64, "");
        __builtin_amdgcn_s_waitcnt(0x0f70 | (n & 15) | ((n >> 4) << 14));
        asm volatile("s_nop 0");
        __builtin_amdgcn_sched_barrier(0);
    };
    // One step.  NEXT: the wave has another, step + WAVES.
    auto run_step = [&](auto next_c, auto check_c, int step) {
        constexpr bool NEXT = decltype(next_c)::value;
        using Order = GemmsOrder<BITS, RING, DMA, NEXT>;
        const bool live = 16 * step + 4 * quad < W;
        convert();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NEXT) fetch(step + WAVES);
        __builtin_amdgcn_sched_barrier(0);
        auto ready = [&](auto j_c) { wait(std::integral_constant<int, Order::behind(decltype(j_c)::value)>{}); };
        ready(std::integral_constant<int, 0>{});
        request(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
        // units of two octets, the operands of the next requested before the products of the current
        static_for<8>([&](auto u_c) {
            constexpr int u = decltype(u_c)::value, j = u / 2, v = u + 1, vj = v / 2;
            constexpr bool last = u % 2 == 1;  // of the stage
            auto ahead = [&]() {
                if constexpr (v < 8) {
                    if constexpr (last) ready(std::integral_constant<int, vj>{});
                    request(std::integral_constant<int, vj>{}, std::integral_constant<int, v % 2>{}, std::integral_constant<int, v & 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if constexpr (RING == 4 || !last) ahead();
            multiply(std::integral_constant<int, u & 1>{}, check_c, live);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (last) {  // every read of the stage has been used: its buffer is free
                if constexpr (RING == 4) {
                    if constexpr (NEXT) stage(step + WAVES, std::integral_constant<int, j>{});
                } else {
                    if constexpr (j < 2) stage(step, std::integral_constant<int, j + 2>{});
                    else if constexpr (NEXT) stage(step + WAVES, std::integral_constant<int, j - 2>{});
                    __builtin_amdgcn_sched_barrier(0);
                    ahead();
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        // the planes of the next: behind them came the stages of one step
        if constexpr (NEXT) wait(std::integral_constant<int, 4 * DMA>{});
    };
    const int step0 = min(wave, T - 1);  // rows of fewer steps than waves: the others do the last one again, and their sums are left out
    fetch_tables();
    __builtin_amdgcn_sched_barrier(0);
    fetch(step0);
    __builtin_amdgcn_sched_barrier(0);
    static_for<RING>([&](auto j_c) { stage(step0, j_c); });
    __builtin_amdgcn_sched_barrier(0);
    wait(std::integral_constant<int, BITS + RING * DMA>{});  // the tables, ahead of planes and stages
    put_tables();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    wait(std::integral_constant<int, RING * DMA>{});  // the planes: holds by the release already, which compiles to a wait for every load
#pragma unroll
    for (int mb = 0; mb < MB; mb++) acc[mb] = float4_t{0.f, 0.f, 0.f, 0.f};
    int step = step0;
    for (; step + WAVES < T; step += WAVES) run_step(std::true_type{}, std::false_type{}, step);
    if (16 * step + 16 <= W) run_step(std::false_type{}, std::false_type{}, step);
    else run_step(std::false_type{}, std::true_type{}, step);

    // ---- the waves' sums meet in LDS and are added in the order of the waves.  D: lane l holds activation row l % 16 and weight rows
    // 4 (l / 16) .. + 3
    auto sums = [&](int w) { return reinterpret_cast<float4_t *>(&x0[w][0][0]); };
#pragma unroll
    for (int mb = 0; mb < MB; mb++) sums(wave)[mb * kWave + lane] = acc[mb];
    __syncthreads();
    if (wave >= MB) return;
    const int waves = min(T, WAVES), m = 16 * wave + row;
    float4_t sum = sums(0)[wave * kWave + lane];
#pragma unroll
    for (int w = 1; w < WAVES; w++) {
        const float4_t v = sums(w)[wave * kWave + lane];
        if (w < waves)
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] += v[e];
    }
    if (m >= M) return;
    const int n = n0 + 4 * quad;
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    half4_t y = {(half_t)sum[0], (half_t)sum[1], (half_t)sum[2], (half_t)sum[3]};
    const global_ptr<const half_t> bias = (global_ptr<const half_t>)bias_i;
    if (bias_i != 0)  // as on the finished result
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = (half_t)((float)y[e] + (float)bias[min(n + e, N - 1)]);
    const global_ptr<half_t> o = (global_ptr<half_t>)out_i + ((size_t)m * ldo + n);
    if ((ldo & 3) == 0 && (out_i & 7u) == 0 && n + 3 < N) {
        *(global_ptr<half4_t>)o = y;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < N) o[e] = y[e];
    }
}

}  // namespace ap
