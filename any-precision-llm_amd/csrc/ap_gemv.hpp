// Bitplane GEMV / skinny GEMM for gfx950, 1 <= M <= 8:
//     out[m,n] = sum_k x[m,k] * lut[n, index_b(n,k)]      (fp32 accumulate, fp16 out)
//
// Replaces the reference's matmul_kbit_32<maxm,bits,use_ksplit>
// (any_precision/modules/kernels/matmul.cuh:16-167); the reference sums in
// fp16, this kernel in fp32.
//
// Per weight the path costs a table lookup, so besides HBM it loads the VALU and the LDS
// gather pipe; the design minimises instructions per weight and keeps every wave short:
//   * A workgroup is the S waves of R consecutive rows; wave s owns K-segment s (64*WPL
//     consecutive words = 2048*WPL elements).  The row's table sits at a compile-time LDS
//     address and a gather address is a single SDWA byte-extract-and-shift.
//   * The activations a lane needs are the same for every row: they are loaded into
//     registers once, as they sit in memory.
//   * Per row a lane streams WPL words per plane (one load per plane, a wave covers
//     256*WPL contiguous bytes), rebuilds its indices with a butterfly transpose in
//     registers, gathers from LDS and feeds v_dot2c_f32_f16.
//   * 3 and 4 bits use a pair table (reference idea: matmul.cuh:24,41-49,
//     dequant.cuh:13-30,56-67) of two ADJACENT elements (ap_lookup.hpp): 4^b entries of
//     two fp16, one 32-bit gather per two weights and no packing.  5..8 bits gather single
//     fp16 entries and pack two of them per dot2.
//   * Lane partials of all R x M sums are folded together (wave_sums, ap_device.hpp); when S > 1 the segment partials
//     of a row meet in LDS and are added in a fixed order: results are deterministic.
// The kernel is bound by instructions and by the launch, not by HBM: with every plane in L2 a gate/up launch of 2 x 11008
// x 4096 at 3 bits takes 9.6 us against 10.3 from HBM.  A wave of that launch issues 168 vector instructions, 92 of them
// transposes, lookups and products; with one sum after the other and longer table lane arithmetic they were 181.5.  The more
// sums a wave has, the more the folding saves (vector instructions a wave, registers and us in the kernel trace, before ->
// after: 4096 x 14336 at 3 rows, 4 bits 552 -> 462, 88 -> 80, 15.1 -> 13.3; 5120 x 5120 at 4 rows, 8 bits 921 -> 803,
// 116 -> 112, 14.8 -> 14.1; 4096 x 11008 at 2 rows, 6 bits 665 -> 606, 74 -> 69, 16.8 -> 16.1; 1024 x 4096 at 8 rows, 8 bits
// 752 -> 635, 166 -> 167, 6.7 -> 6.1; 4096 x 4096 at one row, 3 bits the same).
#pragma once
#include <type_traits>

#include "ap_bitplane.hpp"
#include "ap_device.hpp"
#include "ap_gemv_launch.hpp"
#include "ap_lookup.hpp"

namespace ap {


template <int WPL>
struct WordVec;
template <>
struct WordVec<1> { typedef uint32_t type; };
template <>
struct WordVec<2> { typedef u32x2 type; };

template <int WPL>
__device__ __forceinline__ uint32_t word_of(const typename WordVec<WPL>::type &v, int i) {
    if constexpr (WPL == 1) return v; else return v[i];
}

// Whether all lookups of a word are asked to come before its first product.  Left to the scheduler they are issued a pair at
// a time from three activation rows on, each pair's products waiting for it, and the first of them for all activations: one
// LDS round trip after the other.  Together they also pass the time until the activations are there.  us without -> with:
// 1024 x 4096 at 3 rows, 5 bits 4.66 -> 4.28; 2048 x 2048 at 6 rows, 6 bits 4.95 -> 4.42; over thirteen shapes of 64 to
// 14336 rows 2-13 % at 3 to 8 rows.  One or two rows are scheduled well as they are; the sixteen registers that the lookups
// take spill at three and four rows of 8 bits, cost one of three waves per SIMD at eight rows (5120 x 5120 at 8 bits 18.7 ->
// 20.2), and are needed otherwise in workgroups of more than four waves (1024 x 14336 at 6 rows, 3 bits 7.9 -> 9.5).
constexpr bool gemv_lookups_first(int bits, int m, int threads) {
    return threads <= 256 && m >= (bits == 8 ? 5 : 3) && m <= 7;
}

// One row x one lane: rebuild the indices of this lane's WPL words, gather from
// `table` (an LDS array at a compile-time address) and accumulate the M dot products.
template <int BITS, int M, int WPL, bool FIRST>
__device__ __forceinline__ void row_dot(const typename WordVec<WPL>::type (&q)[BITS],
                                        const uint8_t (&table)[LookupTable<BITS>::kBytes],
                                        const uint32_t (&X)[M][WPL][4][4], float (&acc)[M][2]) {
#pragma unroll
    for (int wi = 0; wi < WPL; wi++) {
        uint32_t qq[BITS];
#pragma unroll
        for (int p = 0; p < BITS; p++) qq[p] = word_of<WPL>(q[p], wi);
        uint32_t w[16];  // w[4 i + c]: elements 2 i and 2 i + 1 of byte c
        auto product = [&](auto i_c, auto c_c) {
            constexpr int i = decltype(i_c)::value, c = decltype(c_c)::value;
#pragma unroll
            for (int m = 0; m < M; m++) acc[m][c & 1] = dot2(w[4 * i + c], X[m][wi][3 - c][i], acc[m][c & 1]);
        };
        auto all = [&](auto &&lookup) {
            static_for<4>([&](auto i_c) {
                static_for<4>([&](auto c_c) {
                    w[4 * decltype(i_c)::value + decltype(c_c)::value] = lookup(i_c, c_c);
                    if constexpr (!FIRST) product(i_c, c_c);
                });
            });
            if constexpr (FIRST) {
                asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]),
                                  "+v"(w[8]), "+v"(w[9]), "+v"(w[10]), "+v"(w[11]), "+v"(w[12]), "+v"(w[13]), "+v"(w[14]),
                                  "+v"(w[15]));
                static_for<4>([&](auto i_c) { static_for<4>([&](auto c_c) { product(i_c, c_c); }); });
            }
        };
        if constexpr (LookupTable<BITS>::kPair) {
            uint32_t apair[4];
            // byte = entry number (4 bits) or the entry's byte offset (3 bits); a table entry is 4 bytes
            planes_to_adjacent_pairs<BITS>(qq, apair);
            all([&](auto i_c, auto c_c) -> uint32_t {
                constexpr int i = decltype(i_c)::value, c = decltype(c_c)::value;
                return *reinterpret_cast<const uint32_t *>(&table[byte_offset<c, BITS == 4 ? 2 : 0>(apair[i])]);
            });
        } else {
            uint32_t idx[8];
            planes_to_indices<BITS>(qq, idx);
            all([&](auto i_c, auto c_c) -> uint32_t {
                constexpr int i = decltype(i_c)::value, c = decltype(c_c)::value;
                const uint32_t lo = *reinterpret_cast<const uint16_t *>(&table[byte_offset<c, 1>(idx[2 * i])]);
                const uint32_t hi = *reinterpret_cast<const uint16_t *>(&table[byte_offset<c, 1>(idx[2 * i + 1])]);
                return lo | (hi << 16);
            });
        }
    }
}

// The GEMV kernel.  A workgroup is the S waves of R consecutive rows (R = 1, 2 or 4,
// compile time).  Every wave issues all the global loads it will ever need -- the tables,
// the planes of its R rows, its activations -- before it computes anything, so the
// memory pipe is full from the first cycle and there is no loop-carried prefetch.  Every
// table sits at a compile-time LDS address.
// Grid: ceil(N / R) workgroups per member, of (64, S) threads (S is also an argument: it arrives with the
// others instead of through a load of its own from the dispatch packet); S*64 <= THREADS.  THREADS (256, 512 or
// 1024) only bounds the workgroup size, so that small workgroups may use more registers
// per lane (M x WPL x 16 of them hold the activations).
//
// One launch serves up to kGemvMaxGroup linears that share x, K and the bit-width (the
// q/k/v or gate/up projections of a decoder layer): `mem` lists them and the workgroup
// range of each; a plain call is a set of one.
//
// PAIR (R = 2 only): the two rows of a workgroup are row n of member 0 and row n of member 1 (two linears of
// equal shape), and what is stored is silu(member 0) * member 1 -- the gate and up projections of a SwiGLU
// MLP with their activation function, one output per row pair, nothing written in between.
// Waves per SIMD the register allocator is asked to keep room for (1 = no request).  At 8 bits with two to
// four activation rows the allocator, left alone, settles two or three registers above a step of the
// occupancy table (83 where 80 fit six waves, 99 where 96 fit five) and a workgroup fewer fits the CU; the
// request is what the registers a lane holds by design allow -- 16 per activation row for x, one per plane
// and row, about 14 more -- out of 512 per SIMD lane in blocks of 8.  No instance spills with it; at fewer
// bits the pair-table lookups in flight need more than the estimate, and the allocator does well alone.
constexpr int gemv_waves_per_simd(int bits, int m, int wpl, int r) {
    if (bits != 8 || wpl > 1 || m < 2 || m > 4) return 1;
    const int need = 16 * m + r * bits + 14;
    const int waves = 512 / ((need + 7) / 8 * 8);
    return waves > 8 ? 8 : waves;
}

template <int BITS, int M, int WPL, int R, int THREADS, bool PAIR = false, typename Members = GemvMembers>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(gemv_waves_per_simd(BITS, M, WPL, R))))
void gemv_kbit_kernel(const half_t *__restrict__ x, const Members mem, int K, int S) {
    static_assert(!PAIR || R == 2, "a pair is two rows");
    constexpr bool BIAS = std::is_same<Members, GemvBiasMembers>::value;
    constexpr int NC = 1 << BITS;
    constexpr int MAXS = THREADS / kWave;
    typedef typename WordVec<WPL>::type wvec_t;
    __shared__ __attribute__((aligned(16))) uint8_t tables[R][LookupTable<BITS>::kBytes];
    __shared__ float partial[MAXS * R * M];

    // Which member this workgroup belongs to.  Written without branches, so that every kernel argument
    // arrives with the first clause of scalar loads (a branch per member costs a dependent scalar load
    // each) and the selects stay in scalar registers; no indexed access to the arguments.
    const int bid = blockIdx.x;
    // Member 0 (the only one of a plain call; with PAIR also member 1) and the scalars every workgroup
    // needs, named in ONE empty statement that wants them in scalar registers: the compiler then fetches
    // them with its first clause of scalar loads and waits once.  Left alone it loads each argument where
    // it is first used, a dependent round trip to the scalar cache every time.
    const uint32_t *q0 = mem.qweight[0], *q1 = mem.qweight[PAIR ? 1 : 0];
    const uint16_t *lut0 = mem.lut[0], *lut1 = mem.lut[PAIR ? 1 : 0];
    uint16_t *out0 = mem.out[0];
    const uint16_t *bias0 = nullptr;
    if constexpr (BIAS) bias0 = mem.bias;
    int n0 = mem.n[0], end0 = mem.wg_end[0], end1 = mem.wg_end[1], end2 = mem.wg_end[2], count = mem.count;
    if constexpr (PAIR)
        asm volatile("" : "+s"(q0), "+s"(q1), "+s"(lut0), "+s"(lut1), "+s"(out0), "+s"(n0), "+s"(K), "+s"(S), "+s"(x));
    else if constexpr (BIAS)
        asm volatile("" : "+s"(q0), "+s"(lut0), "+s"(out0), "+s"(n0), "+s"(K), "+s"(S), "+s"(x), "+s"(bias0));
    else
        asm volatile("" : "+s"(q0), "+s"(lut0), "+s"(out0), "+s"(n0), "+s"(end0), "+s"(end1), "+s"(end2), "+s"(count),
                          "+s"(K), "+s"(S), "+s"(x));
    const uint32_t *__restrict__ qweight = q0;
    const half_t *__restrict__ lut = reinterpret_cast<const half_t *>(lut0);
    half_t *__restrict__ out = reinterpret_cast<half_t *>(out0);
    int N = n0, wg0 = 0;
    if constexpr (!PAIR && !BIAS) {
        if (count > 1) {
            // a launch of several linears (a scalar branch; plain calls skip it): which member the workgroup
            // belongs to, then that member's fields by index -- one more clause of scalar loads, cheaper than
            // selecting each field among four
            int g = bid >= end0 ? 1 : 0;  // wg_end ascends
            g = (count > 2 && bid >= end1) ? 2 : g;
            g = (count > 3 && bid >= end2) ? 3 : g;
            if (g > 0) {
                qweight = mem.qweight[g];
                lut = reinterpret_cast<const half_t *>(mem.lut[g]);
                out = reinterpret_cast<half_t *>(mem.out[g]);
                N = mem.n[g];
                wg0 = g == 1 ? end0 : (g == 2 ? end1 : end2);
            }
        }
    }

    // blockDim.x is the wave size, so threadIdx.y is wave-uniform: say so, to keep row
    // addresses in scalar registers
    const int lane = threadIdx.x;
    const int s = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int W = K >> 5;
    const uint32_t w0 = (uint32_t)(s * kWave + lane) * WPL;
    const bool valid = w0 < (uint32_t)W;
    const uint32_t wl = valid ? w0 : 0u;  // lanes past the row end read word 0; their sums are dropped
    const int row0 = PAIR ? bid : (bid - wg0) * R;
    // row r of this workgroup: its number, the address of its first plane word and of its table (all
    // wave-uniform: a load is a scalar base plus the lane's 32-bit byte offset)
    const size_t plane_bytes = (size_t)N * W * sizeof(uint32_t);
    const uint32_t lane_bytes = wl * (uint32_t)sizeof(uint32_t);
    const char *plane_row[R];
    global_ptr<const half_t> table_row[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int n = PAIR ? row0 : min(row0 + r, N - 1);
        plane_row[r] = reinterpret_cast<const char *>((PAIR ? (r == 0 ? q0 : q1) : qweight) + (size_t)n * W);
        table_row[r] = scalar_ptr((PAIR ? reinterpret_cast<const half_t *>(r == 0 ? lut0 : lut1) : lut) + (size_t)n * NC);
    }

    // Issue order matters: the tables first (tiny; staging them to LDS then overlaps the
    // plane loads -- issued last, the table was the last thing to arrive and cost 15-20 %),
    // then the planes (HBM: the requests must go out at once), then the activations (L2
    // hits; issued before the planes they cost up to 1 us at 3-5 bits).  Rows past N (last
    // workgroup only) re-read row N-1 and are not stored.
    // wave r % S fetches and stages the table of row r; r < 4, so up to three conditional subtractions
    // instead of a division by a run-time S
    auto stages = [&](int r) {
        int owner = r;
#pragma unroll
        for (int i = 0; i < R - 1; i++) owner = owner >= S ? owner - S : owner;
        return s == owner;
    };
    const PairLane<BITS> pl = pair_lane<BITS>(lane);
    TableWords<BITS> t[R];
#pragma unroll
    for (int r = 0; r < R; r++)
        if (stages(r)) t[r] = lookup_table_fetch<BITS>(table_row[r], lane, pl);
    wvec_t q[R][BITS];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int p = 0; p < BITS; p++)  // streamed once: non-temporal, so x and the tables keep their cache lines
            q[r][p] = load_at_nt<wvec_t>(scalar_ptr(plane_row[r] + p * plane_bytes), lane_bytes);
    uint32_t X[M][WPL][4][4];
    load_activations_plain<M, WPL>(x, K, (int)wl, X);

#pragma unroll
    for (int r = 0; r < R; r++)
        if (stages(r)) {
            lookup_table_arrive<BITS>(t[r]);
            lookup_table_stage<BITS>(t[r], tables[r], lane);
        }
    if (S > 1) lds_only_barrier(); else __builtin_amdgcn_wave_barrier();

    // stores go through a pointer typed as global memory (the argument pointers left the statement above
    // without an address space, and a store through them would be a flat one)
    const global_ptr<half_t> out_g = (global_ptr<half_t>)reinterpret_cast<uint64_t>(out);
    constexpr int NS = R * M;
    // Seven and eight activation rows in a workgroup of more than eight waves (at most 128 registers a lane, which the
    // activations fill): every sum is finished and stored at once; held for the folding they more than double what goes to
    // scratch memory (us folded -> at once: 512 x 17408 at 7 rows, 5 bits 30.3 -> 13.9; 2048 x 20480 at 8 rows, 8 bits 180 -> 70).
    // The order within a sum is the same.
    constexpr bool FOLD = M <= 6 || THREADS <= 512;
    float lane_sum[NS];
    static_for<R>([&](auto r_c) {
        constexpr int r = decltype(r_c)::value;
        float acc[M][2];
#pragma unroll
        for (int m = 0; m < M; m++) acc[m][0] = acc[m][1] = 0.f;
        row_dot<BITS, M, WPL, gemv_lookups_first(BITS, M, THREADS)>(q[r], tables[r], X, acc);
#pragma unroll
        for (int m = 0; m < M; m++) {
            float v = acc[m][0] + acc[m][1];
            if constexpr (FOLD) {
                // a row's sums are finished before the next row's lookups start, outside of any "if (valid)" region: left to the
                // optimiser the lookups of all rows are interleaved and take up to 30 registers more (8 bits: scratch memory)
                asm volatile("" : "+v"(v));
                lane_sum[r * M + m] = valid ? v : 0.f;
            } else {
                const float one[1] = {valid ? v : 0.f};
                float sum[1];
                wave_sums<1>(one, sum);
                if (lane == 0) partial[s * NS + r * M + m] = sum[0];
            }
        }
    });
    // sum number r M + m
    float tot[(NS + 3) / 4];
    if constexpr (FOLD) wave_sums<NS>(lane_sum, tot);

    // What is stored: the sum as fp16, plus the bias of its row in fp16 arithmetic, as the operation on the finished result has it.  A
    // bias as an operation of its own costs a launch and half as much again of the host's time (1999 x 2720, 3 rows, 6 bits: 10.9 us a
    // call, 7.0 with it here).
    auto finished = [&](float v, int n) {
        const half_t y = (half_t)v;
        if constexpr (BIAS) return (half_t)((float)y + (float)((global_ptr<const half_t>)reinterpret_cast<uint64_t>(bias0))[n]);
        else return y;
    };
    auto swiglu = [](float gate, float up) { return gate / (1.f + __expf(-gate)) * up; };
    if (FOLD && S == 1 && !PAIR) {
#pragma unroll
        for (int h = 0; h < (NS + 3) / 4; h++) {
            int i;
            if (sum_lane<NS>(h, lane, i) && row0 + i / M < N) out_g[(size_t)(i % M) * N + row0 + i / M] = finished(tot[h], row0 + i / M);
        }
    } else {
#pragma unroll
        for (int h = 0; FOLD && h < (NS + 3) / 4; h++) {
            int i;
            if (sum_lane<NS>(h, lane, i)) partial[s * NS + i] = tot[h];
        }
        __syncthreads();
        const int tid = s * kWave + lane;
        if constexpr (PAIR) {
            if (tid < M) {
                float g = 0.f, u = 0.f;
                for (int ss = 0; ss < S; ss++) {
                    g += partial[(ss * R) * M + tid];
                    u += partial[(ss * R + R - 1) * M + tid];
                }
                out_g[(size_t)tid * N + row0] = (half_t)swiglu(g, u);
            }
        } else if (tid < R * M) {  // S >= 2 waves hold at least 128 threads >= R * M
            const int m = tid % M, r = tid / M;
            float v = 0.f;
            if (S == 2) {  // rows of up to 4096 elements: both partials in one LDS read instead of a loop of two
                v = partial[r * M + m] + partial[(R + r) * M + m];
            } else {
                for (int ss = 0; ss < S; ss++) v += partial[(ss * R + r) * M + m];
            }
            if (row0 + r < N) out_g[(size_t)m * N + row0 + r] = finished(v, row0 + r);
        }
    }
}

}  // namespace ap
