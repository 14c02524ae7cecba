// Block-tile fused bitplane dequant -> MFMA GEMM for gfx950, for tens to thousands of activation rows:
//     out[m,n] = sum_k x[m,k] * lut[n, index_b(n,k)]      (fp16 operands, fp32 accumulate)
//
// A workgroup owns 32 WN weight rows x 32 MB activation rows for the whole of K: WN waves side by side over the weight rows, WK
// such groups each on its share of K (their sums meet in LDS at the end, in the order of the groups).
//   * A wave owns 32 weight rows and all the activation rows of the tile: a weight is rebuilt once per tile, in the registers of the
//     lane that feeds it to v_mfma_f32_32x32x16_f16 (lane = weight row l % 32 and words of quad l / 32; one operand is one byte group
//     of a word), and serves MB matrix instructions.  The tiled kernel (ap_gemmt.hpp) has 16 weight rows a wave, so twice the LDS
//     reads of activations a matrix instruction.
//   * Tables sit in LDS by entry and slot, 256 bytes an entry: the address of a lookup is the index byte over the byte of the lane's
//     slot, one v_perm_b32, and lanes served together read different banks.  Up to 4 bits a table of pairs where it fits.
//   * Activations come by direct global -> LDS loads in stages of 64 elements of every row (runs of 128 bytes: a run of 64 costs the
//     load pipe as much, 19 TB/s from L2 instead of 33), two or four stages in flight, units XOR-swizzled.
//   * What a matrix instruction leaves free is planned, not left to the scheduler: 32 cycles each, of which about six vector
//     instructions of either wave of the SIMD fit in 24.  Every slot holds its share of the lookups of the next octet, of the index
//     arithmetic of the NEXT half-step, of the loads, an activation read, fenced.  Bursts of any of them stood before: the index
//     arithmetic at the start of a half-step, loads by all waves behind the barrier, planes at once (4096 x 4096, 128 rows, 128 x 128
//     tile, 5 bits: 45 us so, 43 with reads interleaved only, 38 with the loads spread and half the barriers, 36 fenced,
//     33 with waits that leave the stages ahead outstanding).
// What bounds it (same tile, 5 bits, taken on the form of 36 us): matrix cores alone 14 us, with the vector instructions 15.5, with the LDS reads 24, and 7
// for launch, tables, first loads and the sums at the end.
// Measured (us, planes from HBM; before = the better of tiled kernel and dequantise + library product), rows / 3 / 5 / 8 bits:
//   4096 x 11008, 128: 34 -> 26, 53 -> 37, 71 -> 49;   512: 81 -> 57, 99 -> 67, 102 -> 91
//   14336 x 4096, 192: 41 -> 29, 58 -> 38, 77 -> 49;   512: 88 -> 62, 88 -> 71, 92 -> 79 (0.98 / 0.85 / 0.77 PFLOP/s)
#pragma once
#include <type_traits>

#include "ap_bitplane.hpp"
#include "ap_device.hpp"
#include "ap_gemmb_launch.hpp"
#include "ap_reciprocal.hpp"

namespace ap {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

// What a direct load fetches for a 16-byte unit that lies past the end of its row.
__device__ const uint32_t kGemmbZeros[64] = {};

// Lookup tables in LDS, [entry][64 slots] dwords: slot = 32 (wave & 1) + weight row of the wave.  Plain tables hold one fp16 entry, waves 2
// and 3 in the high half of the dwords; pair tables (3 bits, and 4 bits with up to two waves side by side where 64 KB are free) the entries
// of two adjacent elements, one array for every two waves.  Then what a tile takes of the LDS: four stages where they fit.
template <int BITS, int MB, int WN, int WK>
struct GemmbLds {
    static constexpr int kStage = WK * MB * 4096;  // one stage of every group of waves
    static constexpr bool kPair = BITS == 3 || (BITS == 4 && WN <= 2 && 65536 + 2 * kStage <= 160 * 1024);
    static constexpr int kEntries = kPair ? 1 << (2 * BITS) : 1 << BITS;
    static constexpr int kArrays = kPair ? (WN + 1) / 2 : 1;
    static constexpr int kTable = kArrays * kEntries * 256;
    static constexpr int kBufs = kTable + 4 * kStage <= 160 * 1024 ? 4 : 2;
    static constexpr bool kFits = kTable + kBufs * kStage <= 160 * 1024;
};

// How a wave's loads are spread over the octets of a step (32 of them: two half-steps of four stages of four octets), so that
// the eight waves of a workgroup do not queue for the load pipe while the matrix cores wait.  The waves meet every kSync stages,
// before the last octet of a stage with (stage + 1) % kSync == 0: the buffers of these kSync stages are free then, and the next
// kSync stages must have landed.  The direct loads that refill the buffers begin in that octet, kPieces at a time; the two loads
// of plane p of the next step go into octets kPlanes + 2 p and kPlanes + 2 p + 1.
template <int BITS, int MB, int WN, int WK>
struct GemmbLoads {
    static constexpr int kBufs = GemmbLds<BITS, MB, WN, WK>::kBufs;
    static constexpr int kSync = kBufs / 2;
    static constexpr int kDirect = 4 * MB / WN;                  // direct loads of a wave per stage
    static constexpr int kOctets = 2 * kSync;                    // octets that they are spread over: half of what a meeting lies ahead
    static constexpr int kPieces = (kSync * kDirect + kOctets - 1) / kOctets;
    static constexpr int kLast = (kSync * kDirect - 1) / kPieces;  // octets from the first to the last of them
    static_assert(kPieces < 16, "");
    static constexpr int kPlanes = 14 - 2 * BITS;                // the last two words of the planes before are done with by octet 30
    // of the loads that refill the buffers of the stages up to a meeting, those of the i-th stage that `octets` octets have brought
    static constexpr int refilled(int i, int octets) {
        const int n = octets * kPieces - (i - (kBufs - kSync)) * kDirect;
        return i < kBufs - kSync ? kDirect : (n < 0 ? 0 : (n > kDirect ? kDirect : n));
    }
    // direct loads ahead of the first step: every stage as far as the octet before it has brought it
    static constexpr int first() {
        int n = 0;
        for (int i = 0; i < kBufs; i++) n += refilled(i, 1);
        return n;
    }
    // Loads that were requested after the last of the direct loads that this meeting (before octet 4 s + 3) waits for.  Loads
    // complete in order: waiting until no more than these are outstanding means that the direct loads have landed.  Plane loads
    // of the octet that holds the last direct load are not counted: the order within an octet is the compiler's.
    static constexpr int outstanding(int s, bool planes) {
        int n = 0;
        if (planes)
            for (int o = 4 * (s - kSync) + 3 + kLast + 1; o <= 4 * s + 2; o++) {
                const int at = (o + 64) % 32;
                n += (at >= kPlanes && at < kPlanes + 2 * BITS) || at - 32 >= kPlanes;
            }
        return n;
    }
};

template <int BITS, int MB, int WN, int WK>
__global__ __launch_bounds__(WN *WK *kWave) void gemmb_kbit_kernel(const half_t *__restrict__ x, const GemmbMembers mem, int M,
                                                                   int K, int grid_m, uint32_t tile_div, uint32_t tile_magic) {
    using Lds = GemmbLds<BITS, MB, WN, WK>;
    constexpr bool PAIR = Lds::kPair;
    constexpr int NC = 1 << BITS;
    constexpr int BN = kGemmbRows * WN, BM = 32 * MB;
    constexpr int NBUF = Lds::kBufs;  // stages in flight
    using Loads = GemmbLoads<BITS, MB, WN, WK>;
    constexpr int ND = Loads::kDirect;
    static_assert(4 * MB % WN == 0 && WN <= 4, "");
    __shared__ __attribute__((aligned(256))) uint32_t tables[Lds::kTable / 4];
    __shared__ u32x4 xt0[WK][BM][8], xt1[WK][BM][8];
    __shared__ u32x4 xt2[NBUF == 4 ? WK : 1][NBUF == 4 ? BM : 1][8], xt3[NBUF == 4 ? WK : 1][NBUF == 4 ? BM : 1][8];

    const int lane = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int wn = wave % WN, kh = wave / WN;
    const int row = lane & 31, h = lane >> 5;

    uint64_t x_i = reinterpret_cast<uint64_t>(x), q_i = reinterpret_cast<uint64_t>(mem.qweight[0]),
             lut_i = reinterpret_cast<uint64_t>(mem.lut[0]), out_i = reinterpret_cast<uint64_t>(mem.out[0]);
    int N0 = mem.N[0], count = mem.count, t1 = mem.tile0[1], t2 = mem.tile0[2], t3 = mem.tile0[3], t4 = mem.tile0[4];
    long long ldo0 = mem.ldo[0];
    asm volatile("" : "+s"(x_i), "+s"(q_i), "+s"(lut_i), "+s"(out_i), "+s"(N0), "+s"(count), "+s"(t1), "+s"(t2), "+s"(t3),
                      "+s"(t4), "+s"(ldo0), "+s"(M), "+s"(K), "+s"(grid_m), "+s"(tile_div), "+s"(tile_magic));
    const int W = K >> 5;
    // Workgroup -> tile and its linear, as in the tiled kernel (ap_gemmt.hpp): up to 8 tiles of activation rows the tiles of one block of
    // weight rows get workgroup numbers 8 apart, on one XCD at about the same time, so that the planes come from HBM once.
    const int tiles = count <= 1 ? t1 : (count == 2 ? t2 : (count == 3 ? t3 : t4));
    uint32_t wq, wr;
    divmod_by_reciprocal(blockIdx.x, tile_div, tile_magic, wq, wr);
    int tile_n, tile_m;
    if (grid_m <= 8) {
        tile_n = 8 * (int)wq + (int)(wr & 7u);
        tile_m = (int)(wr >> 3);
    } else {
        tile_n = (int)wr;
        tile_m = (int)wq;
    }
    if (tile_n >= tiles) return;
    int N = N0, first_tile = 0;
    long long ldo = ldo0;
    if (count > 1) {
        int g = tile_n >= t1 ? 1 : 0;
        g = (count > 2 && tile_n >= t2) ? 2 : g;
        g = (count > 3 && tile_n >= t3) ? 3 : g;
        if (g > 0) {
            q_i = reinterpret_cast<uint64_t>(mem.qweight[g]);
            lut_i = reinterpret_cast<uint64_t>(mem.lut[g]);
            out_i = reinterpret_cast<uint64_t>(mem.out[g]);
            N = mem.N[g];
            ldo = mem.ldo[g];
            first_tile = g == 1 ? t1 : (g == 2 ? t2 : t3);
        }
    }
    const global_ptr<const char> xg = (global_ptr<const char>)x_i;
    const global_ptr<const char> qg = (global_ptr<const char>)q_i;
    const half_t *__restrict__ lut = (const half_t *)(global_ptr<const half_t>)lut_i;
    half_t *__restrict__ out = (half_t *)(global_ptr<half_t>)out_i;
    const int nb = (tile_n - first_tile) * BN, n0 = nb + wn * kGemmbRows, m0 = tile_m * BM;
    const size_t plane_bytes = (size_t)N * W * 4;

    // ---- this group's share of K in whole half-steps of 8 words (256 elements): the first H_full % WK groups have one more.  What is
    // left of a row, fewer than 8 words, is group 0's, at the end.  A group without any walks nothing (and loads what half-step 0 has).
    const int H_full = W >> 3, most = (H_full + WK - 1) / WK;
    const int own = H_full / WK + (kh < H_full % WK ? 1 : 0);
    const int hs0 = own > 0 ? kh * (H_full / WK) + min(kh, H_full % WK) : 0, hs_end = hs0 + own;

    // ---- planes: step = 16 words; load 0 covers rows 0..15, load 1 rows 16..31 of the wave: 64 contiguous bytes of a row by
    // the lanes row % 16 + 16 {0, 2, 1, 3}.  One exchange of odd and even groups of 16 lanes between the two
    // (v_permlane16_swap) then leaves lane = (row % 32, quad 0 or 1) in the first and (row % 32, quad 2 or 3) in the second.
    uint32_t prow[2];
#pragma unroll
    for (int r = 0; r < 2; r++) prow[r] = (uint32_t)min(n0 + 16 * r + (lane & 15), N - 1) * (uint32_t)W * 4u;
    const int quad = ((lane >> 4) & 1) * 2 + (lane >> 5);
    uint32_t q[2][BITS][4];   // as they arrive
    uint32_t q1[BITS][4];     // of half-step 1
    typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
    auto fetch_plane = [&](auto check_c, int hs, int p, int r) {  // rows 16 r .. 16 r + 15, half-steps hs, hs + 1
        const int w = 8 * hs + 4 * quad;
        const int wc = min(w, W - 4);  // quads past the half-steps that are used stay inside the row
        const global_ptr<const char> plane = qg + p * plane_bytes;
        if constexpr (decltype(check_c)::value) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                q[r][p][i] = *(global_ptr<const uint32_t>)(plane + (prow[r] + 4u * (uint32_t)min(w + i, W - 1)));
        } else {
            const u32x4 v = *(global_ptr<const u32x4_a4>)(plane + (prow[r] + 4u * (uint32_t)wc));
#pragma unroll
            for (int i = 0; i < 4; i++) q[r][p][i] = v[i];
        }
    };
    auto fetch = [&](auto check_c, int hs) {
#pragma unroll
        for (int p = 0; p < BITS; p++) {
            fetch_plane(check_c, hs, p, 0);
            fetch_plane(check_c, hs, p, 1);
        }
    };

    // ---- activation stages
    const int full_chunks = W >> 5;
    const uint32_t tail_stride = (uint32_t)(W & 31) * 16u;
    const uint32_t x_bytes = (uint32_t)M * (uint32_t)K * 2u;
    uint32_t xoff[ND];
    int xunit[ND];
#pragma unroll
    for (int i = 0; i < ND; i++) {
        const int r = 8 * (wn + WN * i) + (lane >> 3);  // row of the tile
        xunit[i] = (lane & 7) ^ ((r >> 1) & 7);
        xoff[i] = (uint32_t)min(m0 + r, M - 1) * (uint32_t)K * 2u + 16u * (uint32_t)xunit[i];
    }
    auto stage_buffer = [&](auto buf_c) -> auto & {
        constexpr int buf = decltype(buf_c)::value;
        if constexpr (buf == 0) return xt0;
        else if constexpr (buf == 1) return xt1;
        else if constexpr (buf == 2) return xt2;
        else return xt3;
    };
    // direct loads [first, last) of this wave for stage j of half-step hs
    auto stage_dma = [&](auto check_c, int hs, int j, auto buf_c, int first, int last) {
        auto &xt = stage_buffer(buf_c);
        constexpr bool CHECK = decltype(check_c)::value;
        // past the end of the group's share: some half-step of it again, nobody reads it
        const int s = !CHECK && hs >= hs_end ? hs0 : hs;
        const int w0 = 8 * s, chunk = w0 >> 5;
        const uint32_t koff = ((uint32_t)chunk << 11) + ((uint32_t)(w0 & 31) << 4) + (uint32_t)j * (chunk == full_chunks ? tail_stride : 512u);
        const global_ptr<const char> base = xg + koff;
#pragma unroll
        for (int i = 0; i < ND; i++) {
            if (i < first || i >= last) continue;
            const auto to = (__attribute__((address_space(3))) void *)&xt[kh][8 * (wn + WN * i)][0];
            if constexpr (CHECK) {
                const char *const src = w0 + xunit[i] < W ? (const char *)(base + xoff[i]) : reinterpret_cast<const char *>(kGemmbZeros) + 16 * (lane & 7);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, to, 16, 0, 0);
            } else {
                // the compiler's own waits count behind this one (14336 x 4096 at 512 rows, 5 bits 77.6 -> 74.2 us; 22016 x 4096 at 128 rows 40.9 -> 40.7)
                load_to_lds(x_i, x_bytes, to, xoff[i], koff);
            }
        }
    };

    fetch(std::false_type{}, hs0);
    __builtin_amdgcn_sched_barrier(0);
    // this lane's share of its row's table: all of it for a pair table (built from registers), else 1 / PARTS of its entries
    constexpr int PARTS = PAIR ? 1 : (2 * WK * 8 <= NC ? 2 * WK : NC / 8);
    constexpr int TQ = NC / PARTS / 8;
    const int part = PAIR ? 0 : (2 * kh + h) % PARTS;
    u32x4 table_row[TQ];
    {
        const u32x4 *src = reinterpret_cast<const u32x4 *>(lut + (size_t)min(n0 + row, N - 1) * NC) + part * TQ;
#pragma unroll
        for (int i = 0; i < TQ; i++) table_row[i] = src[i];
    }
    static_for<NBUF>([&](auto t_c) {
        constexpr int t = decltype(t_c)::value;
        stage_dma(std::false_type{}, hs0, t, std::integral_constant<int, t>{}, 0, Loads::refilled(t, 1));
    });

    const uint32_t array_bits = BITS == 3 && WN == 4 ? (wn >> 1 ? 0x55555555u : 0u) : 0u;
    constexpr int NRAW = PAIR ? 4 : 8;  // table reads per octet of weights
    uint32_t idx[2][4][NRAW];           // per half-step: the indices of its four words of the lane
    // Word w of a half-step from its planes to its indices, in four pieces (one an octet) of four parts that go between the matrix
    // instructions.
    uint32_t work[8];
    auto convert = [&](auto half_c, auto w_c, auto piece_c, auto part_c) {
        constexpr int half = decltype(half_c)::value, w = decltype(w_c)::value, piece = decltype(piece_c)::value, part = decltype(part_c)::value;
        if constexpr (piece == 0) {
            if constexpr (half == 0)
#pragma unroll
                for (int p = part; p < BITS; p += 4) {
                    const auto a = __builtin_amdgcn_permlane16_swap(q[0][p][w], q[1][p][w], false, false);
                    q[0][p][w] = a[0];
                    q1[p][w] = a[1];
                }
            return;
        }
        if constexpr (piece == 1 && part == 0) {
            auto plane = [&](int p) { return half == 0 ? q[0][p][w] : q1[p][w]; };
            if constexpr (PAIR) {
                // as planes_to_adjacent_pairs, the entry in the low bits of its byte; at 3 bits the two above choose the array
                work[0] = plane(BITS - 1);
                work[1] = plane(BITS - 2);
                work[2] = plane(BITS - 3);
                work[3] = BITS == 4 ? plane(0) : array_bits;
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) work[i] = i < BITS ? plane(i < BITS ? BITS - 1 - i : 0) : 0u;
            }
        }
        if constexpr (PAIR) {
            if constexpr (piece == 1 && part == 0) swap_blocks<4, 0x0F0F0F0Fu>(work[0], work[2]);
            if constexpr (piece == 1 && part == 2) swap_blocks<4, 0x0F0F0F0Fu, false, BITS == 3 && WN != 4>(work[1], work[3]);
            if constexpr (piece == 2 && part == 0) swap_blocks<2, 0x33333333u>(work[0], work[1]);
            if constexpr (piece == 2 && part == 2) swap_blocks<2, 0x33333333u>(work[2], work[3]);
            if constexpr (piece == 3 && part == 3)
#pragma unroll
                for (int i = 0; i < 4; i++) idx[half][w][i] = work[3 - i];
        } else {
            if constexpr (piece == 1) swap_index_rows<BITS, 0, 4, 0x0F0F0F0Fu, part, 0>(work);
            if constexpr (piece == 2) swap_index_rows<BITS, 0, 2, 0x33333333u, (part & 1) + 2 * (part & 2), 1>(work);
            if constexpr (piece == 3) {
                swap_index_rows<BITS, 0, 1, 0x55555555u, 2 * part, 2>(work);
                idx[half][w][7 - 2 * part] = work[2 * part];
                idx[half][w][6 - 2 * part] = work[2 * part + 1];
            }
        }
    };
    auto convert_all = [&](auto half_c) {
        static_for<4>([&](auto w_c) {
            static_for<4>([&](auto piece_c) { static_for<4>([&](auto part_c) { convert(half_c, w_c, piece_c, part_c); }); });
        });
    };

    // The planes were requested first: their index arithmetic while the tables and the activations, every load behind them, are on
    // their way.  (Fenced on both sides, or the scheduler takes the arithmetic ahead of the wait; and an instruction between, or the
    // compiler joins the wait with its own at the first use.  That one was for every load while the direct loads were global_load_lds,
    // which are of the FLAT family; then, us so, and with all loads waited for: 1024 x 512 at 512 rows, 4 bits 6.68 / 6.92; 4096 x 768 at 128 rows, 3 bits 5.79 / 5.97; 4096 x 11008 at
    // 128 rows, 4 bits 29.9 / 30.2; of rows of 4096 elements 1 % at most.)
    __builtin_amdgcn_sched_barrier(0);
    {
        constexpr int keep = TQ + Loads::first();
        static_assert(keep < 64, "");
        __builtin_amdgcn_s_waitcnt(0x0f70 | (keep & 15) | ((keep >> 4) << 14));
    }
    asm volatile("s_nop 0");
    __builtin_amdgcn_sched_barrier(0);
    convert_all(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);  // (the loads below stay behind it: 4096 x 768 at 8 bits, 128 rows 9.9 us with them ahead, 9.7)
    static_for<(Loads::kPlanes < 0 ? -Loads::kPlanes : 0)>([&](auto n_c) {  // what a step before would have requested
        constexpr int n = decltype(n_c)::value;
        fetch_plane(std::false_type{}, hs0 + 2 < hs_end ? hs0 + 2 : hs0, n / 2, n % 2);
    });

    // ---- tables
    {
        const int slot = 32 * (wn & 1) + row;
        if constexpr (PAIR) {
            // entry e = (.. f1 s1 f0 s0) holds (lut[f], lut[s]); group kh and half h of the wave write PER consecutive ones:
            // the low bits of f and s come by constant index, the others select once
            constexpr int PER = (NC * NC) / (2 * WK), LB = __builtin_ctz(PER), FB = 1 << (LB / 2), SB = 1 << ((LB + 1) / 2);
            uint32_t v[NC];
#pragma unroll
            for (int k = 0; k < NC / 8; k++) {
                const u32x4 t = table_row[k];
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    v[8 * k + 2 * d] = t[d] & 0xffffu;
                    v[8 * k + 2 * d + 1] = t[d] >> 16;
                }
            }
            const int e0 = PER * (2 * kh + h);
            const int f0 = ((e0 >> 1) & 1) | ((e0 >> 2) & 2) | ((e0 >> 3) & 4) | ((e0 >> 4) & 8);
            const int s0 = (e0 & 1) | ((e0 >> 1) & 2) | ((e0 >> 2) & 4) | ((e0 >> 3) & 8);
            uint32_t F[FB], S[SB];
#pragma unroll
            for (int a = 0; a < FB; a++) {
                F[a] = v[a];
#pragma unroll
                for (int k = 1; k < NC / FB; k++) F[a] = f0 == FB * k ? v[FB * k + a] : F[a];
            }
#pragma unroll
            for (int a = 0; a < SB; a++) {
                S[a] = v[a];
#pragma unroll
                for (int k = 1; k < NC / SB; k++) S[a] = s0 == SB * k ? v[SB * k + a] : S[a];
                S[a] <<= 16;
            }
            uint32_t *dst = tables + (wn >> 1) * (NC * NC * 64) + e0 * 64 + slot;
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const int f = ((i >> 1) & 1) | ((i >> 2) & 2), s = (i & 1) | ((i >> 1) & 2) | ((i >> 2) & 4);
                dst[i * 64] = F[f] | S[s];
            }
        } else {
            // plain: halves of a dword by wn >> 1; lane half and group share the entries
            uint16_t *dst = reinterpret_cast<uint16_t *>(tables) + 2 * slot + (WN == 4 ? (wn >> 1) : 0);
            constexpr int PER = NC / PARTS;
            if (2 * kh + h < PARTS)
#pragma unroll
                for (int i = 0; i < TQ; i++)
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        const int e = part * PER + 8 * i + 2 * d;
                        dst[e * 128] = (uint16_t)(table_row[i][d] & 0xffffu);
                        dst[(e + 1) * 128] = (uint16_t)(table_row[i][d] >> 16);
                    }
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();

    typedef __attribute__((address_space(3))) uint16_t lds_u16_t;
    typedef __attribute__((address_space(3))) uint32_t lds_u32_t;
    typedef __attribute__((address_space(3))) uint8_t lds_u8_t;
    const lds_u8_t *const tables_lds = (const lds_u8_t *)&tables[0];
    // low byte of a lookup address: the lane's slot (and, plain tables, its half of the dword)
    const uint32_t slot_byte = (uint32_t)(32 * (wn & 1) + row) * 4u + (!PAIR && WN == 4 ? 2u * (uint32_t)(wn >> 1) : 0u);

    float16_t acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[mb][v] = 0.f;

    half8_t afrag[MB];                  // activation operands: each is read anew once its matrix instruction has been issued
    uint32_t raw[2][NRAW];              // table entries of their weights as they come from LDS
    const int sw = (lane >> 1) & 7;
    auto issue_a = [&](auto buf_c, auto wi_c, auto m_c) {
        constexpr int wi = decltype(wi_c)::value, m = decltype(m_c)::value;
        auto &xt = stage_buffer(buf_c);
        afrag[m] = __builtin_bit_cast(half8_t, xt[kh][m * 32 + row][(4 * h + wi) ^ sw]);
    };
    auto issue_b = [&](auto j_c, const uint32_t(&word)[NRAW], uint32_t(&r)[NRAW], auto first_c, auto last_c) {
        constexpr int c = 3 - decltype(j_c)::value, first = decltype(first_c)::value, last = decltype(last_c)::value < NRAW ? decltype(last_c)::value : NRAW;
#pragma unroll
        for (int i = first; i < last; i++) {
            // address = index byte * 256 + slot byte
            const uint32_t a = __builtin_amdgcn_perm(word[i], slot_byte, 0x0c0c0000u | ((4u + c) << 8));
            if constexpr (PAIR) r[i] = *reinterpret_cast<const lds_u32_t *>(tables_lds + a);
            else r[i] = *reinterpret_cast<const lds_u16_t *>(tables_lds + a);
        }
    };
    auto finish_b = [&](auto check_c, const uint32_t(&r)[NRAW], bool alive) {
        u32x4 bw;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t packed;
            if constexpr (PAIR) packed = r[i];
            else packed = r[2 * i] | (r[2 * i + 1] << 16);
            if constexpr (decltype(check_c)::value) bw[i] = alive ? packed : 0u;
            else bw[i] = packed;
        }
        return __builtin_bit_cast(half8_t, bw);
    };
    // One half-step: four stages (byte group j of its 8 words) of four octets (word wi of a lane's quad).
    // NEXT: a half-step follows, so that planes are requested and indices made for it.  (The counts of loads in flight depend on it: without a
    // use for them the compiler drops the plane loads.)
    auto run_half = [&](auto check_c, auto next_c, auto half_c, int hs) {
        constexpr bool CHECK = decltype(check_c)::value, NEXT = decltype(next_c)::value;
        constexpr int half = decltype(half_c)::value;
        bool live[4];
#pragma unroll
        for (int wi = 0; wi < 4; wi++) live[wi] = !CHECK || 8 * hs + 4 * h + wi < W;
        static_for<16>([&](auto t_c) {
            constexpr int t = decltype(t_c)::value, j = t / 4, wi = t % 4, cur = t & 1, nxt = cur ^ 1;
            constexpr int SYNC = Loads::kSync;
            if constexpr (wi == 3 && (j + 1) % SYNC == 0) {
                // Every read of these stages has been requested.  When they are done in every wave the buffers can be refilled;
                // and the next stages have landed (GemmbLoads::outstanding).
                constexpr int keep = Loads::outstanding(4 * half + j, NEXT);
                static_assert(keep < 64, "");
                __builtin_amdgcn_s_waitcnt(0x0070 | (keep & 15) | ((keep >> 4) << 14));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (NEXT && half == 1 && t == 0) {
                // The planes of the next step are used from here on; what was requested after them, in the octet before, stays
                // outstanding.
                __builtin_amdgcn_s_waitcnt(0x0f70 | (Loads::kPieces & 15));
                __builtin_amdgcn_sched_barrier(0);
            }
            const half8_t w = finish_b(check_c, raw[cur], live[wi]);
            // One matrix instruction a slot, and behind it what runs in its shadow: table reads for the next octet (in the first
            // half of the octet, so that they are back at its end), the activations of this block of rows for the next octet, a
            // part of the index arithmetic of the next half-step, and in some slots a load.
            static_for<MB>([&](auto m_c) {
                constexpr int m = decltype(m_c)::value;
                acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, afrag[m], acc[m], 0, 0, 0);
                constexpr int FRONT = (MB + 1) / 2, LOOK = (NRAW + FRONT - 1) / FRONT;
                if constexpr (m < FRONT)
                    issue_b(std::integral_constant<int, (wi == 3 ? j + 1 : j) % 4>{}, idx[t == 15 ? half ^ 1 : half][(wi + 1) % 4], raw[nxt],
                            std::integral_constant<int, m * LOOK>{}, std::integral_constant<int, (m + 1) * LOOK>{});
                issue_a(std::integral_constant<int, (wi == 3 ? j + 1 : j) % NBUF>{}, std::integral_constant<int, (wi + 1) % 4>{}, m_c);
                // the loads that refill the buffers of the stages up to the last meeting
                constexpr int since = (t + 1) % (4 * SYNC);                                  // octets since the meeting
                constexpr int s0 = ((t + 1) / (4 * SYNC) - 1) * SYNC;                        // first of its stages, from this half-step on
                if constexpr (since <= Loads::kLast)
                    static_for<Loads::kPieces>([&](auto p_c) {
                        constexpr int load = since * Loads::kPieces + decltype(p_c)::value, i = load / ND, st = s0 + i + NBUF;
                        if constexpr (i < SYNC && decltype(p_c)::value * MB / Loads::kPieces == m)
                            stage_dma(check_c, hs + st / 4, st % 4, std::integral_constant<int, st % NBUF>{}, load % ND, load % ND + 1);
                    });
                if constexpr (NEXT) {
                    static_for<4>([&](auto part_c) {
                        if constexpr (decltype(part_c)::value * MB / 4 == m)
                            convert(std::integral_constant<int, half ^ 1>{}, std::integral_constant<int, j>{}, std::integral_constant<int, wi>{}, part_c);
                    });
                    // the planes of the next step
                    constexpr int n = 16 * half + t - Loads::kPlanes, load = n >= 32 ? n - 32 : n;
                    if constexpr (m == MB - 1 && load >= 0 && load < 2 * BITS) {
                        const int nx = half == 0 ? hs + 2 : hs + 3;  // first half-step of the step whose planes are requested
                        fetch_plane(std::false_type{}, nx < hs_end ? nx : hs0, load / 2, load % 2);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };
    auto first_reads = [&]() {
        static_for<MB>([&](auto m_c) { issue_a(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, m_c); });
        issue_b(std::integral_constant<int, 0>{}, idx[0][0], raw[0], std::integral_constant<int, 0>{}, std::integral_constant<int, NRAW>{});
    };
    auto idle_half = [&]() {
#pragma unroll
        for (int i = 0; i < 4 / Loads::kSync; i++) __builtin_amdgcn_s_barrier();
    };
    first_reads();
    // (an odd half-step runs a copy of its own: left through the middle, the loop has an edge on which plane loads are pending, and the
    // compiler waits for every load at its head)
    int hs = hs0;
    for (; hs + 1 < hs_end; hs += 2) {
        run_half(std::false_type{}, std::true_type{}, std::integral_constant<int, 0>{}, hs);
        run_half(std::false_type{}, std::true_type{}, std::integral_constant<int, 1>{}, hs + 1);
    }
    if (hs < hs_end) run_half(std::false_type{}, std::false_type{}, std::integral_constant<int, 0>{}, hs);
    if (own < most) idle_half();
    if (W & 7) {
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        if (kh == 0) {
            fetch(std::true_type{}, H_full);
            static_for<NBUF>([&](auto t_c) {
                constexpr int t = decltype(t_c)::value;
                stage_dma(std::true_type{}, H_full, t, std::integral_constant<int, t>{}, 0, Loads::refilled(t, 1));
            });
            convert_all(std::integral_constant<int, 0>{});
        }
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        if (kh == 0) {
            first_reads();
            run_half(std::true_type{}, std::false_type{}, std::integral_constant<int, 0>{}, H_full);
        } else {
            idle_half();
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();

    // ---- epilogue.  D: lane l holds activation row l % 32 and weight rows 8 (v / 4) + 4 (l / 32) + v % 4
    // The finished values go through LDS once more, as fp16 rows of the tile ([activation row][16-byte unit ^ row]), so that a
    // row's results leave in 16-byte stores side by side.
    constexpr int UNITS = BN / 8;
    constexpr int PASSES = BM * BN * 2 > (int)sizeof(xt0) ? 2 : 1;  // parts of the tile by activation rows, as one stage buffer holds them
    constexpr int PM = BM / PASSES;
    static_assert(PM * BN * 2 <= (int)sizeof(xt0) && (PASSES == 1 || WK == 1), "");
    uint8_t *const tile = reinterpret_cast<uint8_t *>(NBUF == 4 ? &xt2[0][0][0] : &xt0[0][0][0]);
    auto finish4 = [&](int r, const float(&v)[4]) {  // accumulators r .. r + 3
        typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
        const int m = (32 * (r / 16)) % PM + row, unit = 4 * wn + (r % 16) / 4;
        *reinterpret_cast<half4_t *>(tile + (m * UNITS + (unit ^ (m & (UNITS - 1)))) * 16 + 8 * h) =
            half4_t{(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
    };
    constexpr int REGS = 16 * MB, PART = REGS / WK;  // accumulators of a wave; group g finishes PART of them
    // what is parked stays in the first two buffers: with four the finished tile goes to the third, with no barrier between
    static_assert(PART % 4 == 0 && WN * (WK - 1) <= 2 * WK, "");
    if constexpr (WK > 1) {
        // what a wave of group `from` leaves for the wave of group `to` over the same weight rows: PART accumulators
        auto parked = [&](int to, int from) {
            const int block = (wn * WK + to) * (WK - 1) + (from < to ? from : from - 1), buf = block / (WK * WK);
            float4_t *base = reinterpret_cast<float4_t *>(buf == 0 ? &xt0[0][0][0] : &xt1[0][0][0]);
            return base + block % (WK * WK) * (PART / 4 * kWave) + lane;
        };
        static_for<WK>([&](auto to_c) {
            constexpr int to = decltype(to_c)::value;
            if (kh == to) return;
            float4_t *p = parked(to, kh);
#pragma unroll
            for (int i = 0; i < PART; i += 4) {
                constexpr int r0 = to * PART;
                p[i / 4 * kWave] = float4_t{acc[(r0 + i) / 16][(r0 + i) % 16], acc[(r0 + i) / 16][(r0 + i) % 16 + 1],
                                            acc[(r0 + i) / 16][(r0 + i) % 16 + 2], acc[(r0 + i) / 16][(r0 + i) % 16 + 3]};
            }
        });
        __syncthreads();
        float sum[PART / 4][4];
        static_for<WK>([&](auto own_c) {
            constexpr int own = decltype(own_c)::value;
            if (kh != own) return;
#pragma unroll
            for (int i = 0; i < PART; i += 4) {
                constexpr int r0 = own * PART;
                const int r = r0 + i;
                float(&v)[4] = sum[i / 4];
#pragma unroll
                for (int g = 0; g < WK; g++) {  // in the order of the groups, whoever adds
                    float4_t part;
                    if (g == own) part = float4_t{acc[r / 16][r % 16], acc[r / 16][r % 16 + 1], acc[r / 16][r % 16 + 2], acc[r / 16][r % 16 + 3]};
                    else part = parked(own, g)[i / 4 * kWave];
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = g == 0 ? part[e] : v[e] + part[e];
                }
            }
        });
        if constexpr (NBUF == 2) __syncthreads();  // the tile takes the place of what was parked
        static_for<WK>([&](auto own_c) {
            constexpr int own = decltype(own_c)::value;
            if (kh != own) return;
#pragma unroll
            for (int i = 0; i < PART; i += 4) finish4(own * PART + i, sum[i / 4]);
        });
    }
    const global_ptr<const half_t> bias = (global_ptr<const half_t>)reinterpret_cast<uint64_t>(mem.bias);
    const bool wide = (ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#pragma unroll
    for (int pass = 0; pass < PASSES; pass++) {
        if constexpr (WK == 1) {
            if (pass > 0) __syncthreads();
#pragma unroll
            for (int r = pass * (REGS / PASSES); r < (pass + 1) * (REGS / PASSES); r += 4) {
                const float v[4] = {acc[r / 16][r % 16], acc[r / 16][r % 16 + 1], acc[r / 16][r % 16 + 2], acc[r / 16][r % 16 + 3]};
                finish4(r, v);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i * WN * WK * kWave < PM * UNITS; i++) {
            const int at = i * (WN * WK * kWave) + wave * kWave + lane, r = at / UNITS, u = at % UNITS;
            if (at >= PM * UNITS) break;
            const int m = m0 + pass * PM + r, n = nb + 8 * u;
            half8_t v = *reinterpret_cast<const half8_t *>(tile + (r * UNITS + (u ^ (r & (UNITS - 1)))) * 16);
            if (m >= M) continue;
            if (bias != nullptr)  // as on the finished result
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = (half_t)((float)v[e] + (float)bias[min(n + e, N - 1)]);
            half_t *o = out + (size_t)m * ldo + n;
            if (wide && n + 7 < N) {
                *reinterpret_cast<half8_t *>(o) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (n + e < N) o[e] = v[e];
            }
        }
    }
}

}  // namespace ap
