// moe_ffn_tiled.hip -- LDS-tiled schedule of the MoeExpertFFN grouped GEMMs (many rows per expert, prefill).
//
// Reference: op_kernel/moe_expert_ffn.cpp (ComputeSwiGLU :265-333, ComputeDownProj :339-394, scatter :250-257);
// oracle: tests/moe_cpu_sim.cpp:245-296 (W_gate, W_up [I, H]; W_down [H, I]).
//
// With ~1000 rows per expert (T = 8192, K = 2, E = 16) the GEMMs have an arithmetic intensity of ~1500 flop/B
// against HBM, far above the MFMA ridge. Both are "NT": activation rows and weight rows are contiguous along the
// reduction dim k.
//   macro tile   256 activation rows x 256 weight rows x 64 k per stage; 8 waves (2 x 4), each 128 x 64 as two
//                halves of 64 rows (4 x 4 v_mfma_f32_16x16x32_f16 tiles each, 128 fp32 accumulators per lane in
//                all). The weight fragment is the MFMA's first operand, so each lane ends with 4 consecutive output
//                columns of one row.
//   copies       each stage is copied from global memory straight into LDS (buffer_load ... lds: no staging
//                registers, no LDS store instructions; 32-bit offsets against buffer resources whose range ends
//                at the buffer, so a read past it returns zeros instead of faulting)
//   ticks        a stage is two pairs of ticks, one pair per activation half: a memory tick (LDS reads of the
//                half's fragments, copies) and a compute tick (32 MFMAs), a barrier after each. Waves 4-7 run one
//                tick behind waves 0-3, and wave w shares its SIMD with wave w + 4, so on every SIMD one wave's
//                MFMAs run beside the other's reads and copies.
//   ring         two LDS slots of four 16 KB half tiles (two of activation rows, two of weight rows). A half tile is
//                free one tick after its last read and is refilled at once, a whole stage ahead of its use, with
//                counted waits (all but the youngest 8 copies of a wave). With the 8 copies a wave issues per stage
//                sent together after the stage's one barrier (64 KB in a quarter of its MFMA time) the waves
//                stalled on issuing them. Kernel times on one box each, that kernel -> this one (an in-between
//                form with four tick pairs of 16 MFMAs a stage in the middle):
//                  T = 8192, H = 2048, E = 16, K = 2, I = 8192: gate/up 1024 -> 917 -> 888 us, down 506 -> 440 -> 438
//                  T = 16384, H = 2048, E = 64, K = 6, I = 1408: gate/up 1093 -> 965 -> 940 us, down 587 -> 515 -> 513
//                What bounds it now is power: on all-zero inputs the first gate/up takes 700 us (942 us in the old
//                kernel), on random ones the clock falls to ~1.6 GHz. Timing-only copies of the forms on the way,
//                on zeros: with four tick pairs a stage (734 us) 615 without any copies after the first stages, 640
//                without the epilogue, 733 without the LDS reads; with two pairs but 8-byte hidden stores (728 us)
//                613 with every copy an L2 hit. Measured and not kept: 32x32x16 MFMAs (9 % slower), MFMAs that share
//                the weight instead of the activation fragment (1 % slower), copies issued between the MFMAs of the
//                compute ticks (2-7 % slower, they leave later), the first k-stage rotated per XCD and other cache
//                policies of the copies (level), s_setprio around the compute tick (level), skipping the second
//                half's ticks in tiles of at most 128 rows (1-3 % slower: such a tile takes as long, and the
//                workgroups that share its weight tile drift apart).
//   persistent   one workgroup per CU walks its tiles back to back and the ring runs on across them: the
//                copies of a tile's first two stages go out during the previous tile's last two. The tile table
//                (per-expert tile prefix and row offsets) is built once per workgroup in LDS, so finding a tile
//                is a short search from the last tile's expert on; the next tile's 256 sorted-slot
//                entries are copied into LDS a tile ahead.
//   split        (down) the down projection has only ~2 tiles per CU at prefill, so a count-based schedule
//                leaves the last round mostly idle: the tiles left over after the full rounds are split over k
//                into pieces, one per workgroup, that write fp32 partial tiles; ffn_tiled_fixup_kernel adds them
//                in piece order. The split is a separate instantiation (SPLIT), so gate/up keeps its register
//                allocation at tile changes.
//   LDS layout   unpadded 128-byte rows of 8 granules of 16 B; granule g of row r is stored at g ^ ((r >> 1) & 7),
//                so the 16 rows one ds_read_b128 touches (same logical granule) spread over all banks
//   gate/up      weight half 0 of a tile is 128 W_gate rows, half 1 the matching W_up rows, so each wave holds gate
//                and up of the same (row, i) and applies SwiGLU in registers (hardware exp2 and reciprocal, ~1 ulp
//                each). Lanes exchange halves of their columns (v_permlane16_swap) and store 16 bytes each, 64 B a
//                row (8-byte stores, 32 B a row: 905 instead of 892 us at prefill).
//   down         weight rows are W_down rows (output columns); the epilogue writes expert_out[slot] directly
//   scheduling   tiles are (expert, n-tile, m-tile) with m fastest. Workgroups are dispatched round-robin over
//                the 8 XCDs; each XCD owns a contiguous range of tiles, so the m-tiles that share a weight tile
//                share that XCD's L2.
// Rows past an expert's count read zeros (past the buffer) and are masked on store. A reduction
// extent that is an odd multiple of 32 ends with a half stage (KT instantiation): only its first 32-k step is
// multiplied.

#include "moe_device.h"
#include "moe_launch.h"

namespace moe {

namespace {

constexpr int kBM = 256;           // activation rows per tile
constexpr int kBN = 256;           // weight rows per tile
constexpr int kBK = 64;            // k per stage
constexpr int kPitch = kBK;        // LDS row pitch in halfs (granules XOR-swizzled)
constexpr int kThreads = 512;      // 8 waves
constexpr int kStageHalfs = (kBM + kBN) * kPitch;
constexpr int kHalfTile = 128 * kPitch;  // halfs of one of a stage's four half tiles
constexpr int kNStage = 2;
constexpr int kLdsBytes = kNStage * kStageHalfs * 2;  // the ring; the tile table follows it
constexpr int kEpiStageBytes = kThreads / kWave * 2048;  // down epilogue: 16 rows x 128 B per wave
// LDS of a launch: the ring, the tile table (tab, offs: 2 (E + 1) ints), three row tables, then (down) the
// epilogue's staging rows at the next 16-byte boundary
__host__ __device__ constexpr int tiled_epi_stage_offset(int E) {
    return (kLdsBytes + 8 * (E + 1) + 3 * kBM * 4 + 15) / 16 * 16;
}
__host__ __device__ constexpr int tiled_lds_bytes(int E, bool down) {
    return down ? tiled_epi_stage_offset(E) + kEpiStageBytes : kLdsBytes + 8 * (E + 1) + 3 * kBM * 4;
}
constexpr int kLdsMax = 160 * 1024;
constexpr int kXcds = 8;
constexpr int kCopyPolicy = 1;  // cache-policy bits of the stage copies: sc0
// Partial tiles of the split leftover round: one fp32 kBM x kBN tile per workgroup of a persistent launch.
constexpr int kMaxParts = 256;
constexpr int kFixThreads = 256;
constexpr int kFixRows = 16;  // tile rows per fix-up workgroup
// The split pays off only while the leftover round is a large share of the down projection. The whole FFN, leftover
// round whole / split (us, one box):
//   H = 2048, E = 16, K = 2, I = 8192   T = 1000 383 / 389, T = 2048 535 / 540, T = 4096 878 / 845,
//                                       T = 8192 1470 / 1437, T = 12000 2010 / 1957,
//                                       T = 16384 (5 rounds by the bound) 2737 / 2705
//   H = 4096, E = 8, K = 2, I = 14336   T = 4096 2467 / 2382, T = 8192 (5 rounds) 4556 / 4461
//   H = 2048, E = 64, K = 6, I = 1408   T = 1531 275 / 279, T = 4096 478 / 479, T = 16384 (13-14 rounds) 1457 / 1464
//   H = 1056, E = 24, K = 3, I = 736    T = 3001 83.1 / 87.6
// so at few rounds of short tiles the fix-up launch costs 1-5 % more than it saves, and at 5 rounds of 128 or 224
// stages it would still save 1-2 %.
constexpr int kSplitMaxRounds = 4;

struct TiledArgs {
    const uint16_t* act;         // x [T, H] (gate/up, gathered) or hidden [T*K, I] (down)
    const int32_t* sorted_slot;
    const int32_t* offsets;
    const uint16_t* w;           // expert_weights
    uint16_t* out;               // hidden or expert_out
    int T, E, K, H, I;
    int kdim;                    // H or I
    // [kMaxParts, kBM, kBN] fp32 partial tiles of the split leftover round. It stands between the ints: next to kdim,
    // ntiles_n and gather would be one scalar load with it and prefill 0.2-0.3 % slower (other scalar registers).
    float* partial;
    int ntiles_n;                // n-tiles per expert: 128 i of gate and up, or 256 columns of H (down)
    int gather;                  // gate/up: activation row r -> x[sorted_slot[r] / K]
    int split;                   // split the leftover tiles of each XCD over k (persistent grid <= kMaxParts)
};

// Work of one XCD: its tiles [base, base + n) are dealt to its nloc workgroups in R full rounds; the L tiles
// left over are each split over k into S pieces of at least two stages, one piece per workgroup, so the last
// round keeps every workgroup busy instead of L of them. S = 1 runs the leftover tiles whole.
struct XcdSched {
    int base, n, R, L, S;
};
__device__ __forceinline__ XcdSched xcd_sched(int x, int total, int nloc, int nst, int split) {
    XcdSched s;
    const int per_xcd = (total + kXcds - 1) / kXcds;
    s.base = x * per_xcd;
    s.n = max(0, min(per_xcd, total - s.base));
    s.R = s.n / nloc;
    s.L = s.n - s.R * nloc;
    s.S = 1;
    if (split && s.L > 0) s.S = max(1, min(nloc / s.L, nst / 2));
    return s;
}

// Barrier between two ticks. The only LDS writes of the main loop are the direct-to-LDS copies, which the memory
// ticks' explicit vmcnt waits cover, and the memory ticks also wait for their LDS reads. A workgroup-scope release
// fence would wait for the copies still in flight too (vmcnt(0)).
__device__ __forceinline__ void ring_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    __builtin_amdgcn_sched_barrier(0);
}

// silu(g) * u with the hardware exp2 and reciprocal (each about 1 ulp): g * rcp(1 + 2^(-g log2 e)) * u.
__device__ __forceinline__ float swiglu_fast(float g, float u) {
#pragma clang fp contract(off)
    const float e = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
    return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
}

// The lane index read afresh. Values derived from lane_id() are loop-invariant, so the compiler computes them
// once and keeps them live across the main loop, where the accumulators and fragments leave no room for them:
// they are spilled, and each reload in the tile change or the epilogue waits (vmcnt) for every stage copy in
// flight. A volatile read cannot be hoisted, so what make_plan, the tile search and the epilogue derive from it is
// recomputed there. Of the six instantiations only the down projection with both SPLIT and KT still spills (one
// VGPR, to 8 bytes of scratch).
__device__ __forceinline__ int lane_fresh() {
    int v;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(v));
    return v;
}

// Two fp32 values as packed fp16, each rounded to nearest even.
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef f16 f16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, f16x2));
}

enum Epilogue { kSwiGLU = 0, kScatter = 1 };

// One work item: tile (e, mt, nt), k-stages [k0, k0 + nk), and the partial slot it writes (-1: the whole k
// range, written through the epilogue).
struct TileRef {
    int e, mt, nt, off, ne;
    int k0, nk, part;
};

// Copy plan of one tile. A stage is four half tiles of 128 rows x 128 B (activation rows 0-127 and 128-255, and the
// two weight halves); per half tile wave w issues 2 instructions j, each filling 8 whole LDS rows
// r = (2 w + j) * 8 + lane / 8; lane fetches global granule (lane % 8) ^ ((r >> 1) & 7). ao / bo are byte offsets of
// those granules at k = 0 in the activation and weight buffers ar / wr; the second weight half lies bhalf bytes
// after the first (and, for hidden rows, the second activation half ahalf bytes after the first).
struct CopyPlan {
    uint32_t ao[4], bo[2];
    __amdgpu_buffer_rsrc_t ar, wr;
};

// SPLIT: the leftover round may be split over k (p.split); a separate instantiation, so the kernel without it
// keeps its register allocation at tile changes. KT: the reduction extent is an odd multiple of 32, so the last
// k-stage holds 32 valid columns; its copies read on into the next row (or past the buffer, as zeros), and those
// columns are not multiplied.
template <int EPI, bool SPLIT, bool KT = false>
__global__ __launch_bounds__(kThreads) void ffn_tiled_kernel(TiledArgs p) {
    extern __shared__ __align__(16) uint16_t lds[];
    const int tid = static_cast<int>(threadIdx.x);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = lane_id();
    const int row16 = lane & 15, kg = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;  // 2 x 4 waves: rows wm*128.., weight rows wn*64..

    // Tile table in LDS after the ring: tab[e] = tiles of the experts before e (tab[E] = all tiles), offs[e] =
    // first sorted row of expert e. Tiles are (expert, n-tile, m-tile), m fastest.
    int* tab = reinterpret_cast<int*>(lds + kNStage * kStageHalfs);
    int* offs = tab + (p.E + 1);
    // Three row tables of 256 sorted-slot entries, one per tile in flight (tile k uses table k % 3): the copy rows
    // of gate/up gather x rows by them, the down epilogue scatters by them. Wave 0 copies tile k + 1's table
    // straight into LDS at the start of tile k; it lands before the next ring barrier.
    int* rowtab = reinterpret_cast<int*>(lds + kNStage * kStageHalfs) + 2 * (p.E + 1);
    if (wave == 0) {
        int carry = 0;
        for (int base = 0; base <= p.E; base += kWave) {
            const int e = base + lane;
            int o0 = 0, tiles = 0;
            if (e <= p.E) {
                o0 = p.offsets[e];
                offs[e] = o0;
            }
            if (e < p.E) tiles = (p.offsets[e + 1] - o0 + kBM - 1) / kBM * p.ntiles_n;
            int incl = tiles;  // inclusive scan over the wave
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int v = __shfl_up(incl, d, kWave);
                if (lane >= d) incl += v;
            }
            if (e < p.E) tab[e + 1] = carry + incl;
            carry += __shfl(incl, kWave - 1, kWave);
        }
        if (lane == 0) tab[0] = 0;
    }
    __syncthreads();
    const int total = tab[p.E];

    // Persistent: the grid is a multiple of 8 workgroups, at most one per CU. Workgroups are dispatched
    // round-robin over the 8 XCDs, so workgroup b runs on XCD x = b % 8 as that XCD's li = b / 8-th workgroup.
    // XCD x owns tiles [x * per_xcd, (x + 1) * per_xcd) (m-tiles of one weight tile are consecutive, so they
    // share that XCD's L2), and its workgroups take them round-robin: li, li + nloc, li + 2 nloc, ...; with
    // p.split the tiles left over after the full rounds are split over k (xcd_sched).
    const int nst = (p.kdim + kBK - 1) / kBK;  // >= 2
    const int nloc = static_cast<int>(gridDim.x) / kXcds;
    const int x = static_cast<int>(blockIdx.x) % kXcds, li = static_cast<int>(blockIdx.x) / kXcds;
    const int per_xcd = (total + kXcds - 1) / kXcds;
    XcdSched xs{};
    if (SPLIT) xs = xcd_sched(x, total, nloc, nst, p.split);
    auto tile_at = [&](int k, TileRef& T) __attribute__((always_inline)) -> bool {
        int t;
        T.k0 = 0;
        T.nk = nst;
        T.part = -1;
        if (!SPLIT) {
            const int loc = li + k * nloc;
            t = x * per_xcd + loc;
            if (loc >= per_xcd || t >= total) return false;
        } else {
            int loc;
            if (k < xs.R) {
                loc = li + k * nloc;
            } else if (k == xs.R && xs.S == 1) {
                if (li >= xs.L) return false;
                loc = xs.R * nloc + li;
            } else if (k == xs.R) {  // piece pc of leftover tile j
                const int j = li / xs.S, pc = li - j * xs.S;
                if (j >= xs.L) return false;
                loc = xs.R * nloc + j;
                T.k0 = pc * nst / xs.S;
                T.nk = (pc + 1) * nst / xs.S - T.k0;
                T.part = static_cast<int>(blockIdx.x);
            } else {
                return false;
            }
            t = xs.base + loc;
        }
        // the expert with tab[lo] <= t < tab[lo + 1], from the last tile's on: 64 experts a step (one LDS read, where a
        // search one by one or by halves waits for up to E or log2(E) of them in turn)
        int lo = T.e, past;
        do {
            past = __builtin_popcountll(__ballot(tab[min(lo + 1 + lane_fresh(), p.E)] <= t));
            lo += past;
        } while (past == kWave);
        T.e = lo;
        T.off = __builtin_amdgcn_readfirstlane(offs[lo]);
        T.ne = __builtin_amdgcn_readfirstlane(offs[lo + 1]) - T.off;
        const int mtiles = (T.ne + kBM - 1) / kBM;
        const int local = t - __builtin_amdgcn_readfirstlane(tab[lo]);
        T.nt = __builtin_amdgcn_readfirstlane(local / mtiles);  // the division runs on the VALU
        T.mt = local - T.nt * mtiles;
        return true;
    };
    TileRef cur;
    cur.e = 0;
    if (!tile_at(0, cur)) return;

    // activation rows a tile copies: gate/up gathers token rows (x), down reads its own sorted hidden rows
    const uint32_t act_rows = static_cast<uint32_t>(p.T);
    const uint32_t kbytes = static_cast<uint32_t>(p.kdim) * 2;
    const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(p.sorted_slot), 0,
                                                                          p.T * p.K * 4, 0x00020000);
    auto load_rows = [&](const TileRef& T, int buf) __attribute__((always_inline)) {
        if (wave == 0) {
#pragma unroll
            for (int jj = 0; jj < kBM / kWave; ++jj) {
                const int r = jj * kWave + lane;
                const int row = T.off + min(T.mt * kBM + r, T.ne - 1);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    srsrc, (__attribute__((address_space(3))) void*)(rowtab + buf * kBM + jj * kWave), 4, row * 4, 0, 0,
                    0);
            }
        }
    };
    auto make_plan = [&](const TileRef& T, int buf, CopyPlan& P) __attribute__((always_inline)) {
        const int ln = lane_fresh();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = (wave * 2 + j) * 8 + ln / 8;
            const uint32_t gq = static_cast<uint32_t>((ln % 8) ^ ((r >> 1) & 7));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // rows past the tile's last are past the buffer: zeros, and no memory traffic
                if (p.gather) {
                    const uint32_t row = static_cast<uint32_t>(rowtab[buf * kBM + h * 128 + r] / p.K);
                    P.ao[h * 2 + j] = T.mt * kBM + h * 128 + r < T.ne ? row * kbytes + gq * 16 : 0x80000000u;
                } else {  // rows relative to the tile's first row
                    P.ao[h * 2 + j] = static_cast<uint32_t>(h * 128 + r) * kbytes + gq * 16;
                }
            }
            if (EPI == kSwiGLU) {  // half 0: W_gate rows, half 1: the matching W_up rows
                const int ic = min(T.nt * 128 + r, p.I - 1);
                P.bo[j] = static_cast<uint32_t>(ic) * static_cast<uint32_t>(p.H) * 2 + gq * 16;
            } else {  // half h of wave column wn: output columns wn * 64 + h * 32 + [0, 32); past H: past the buffer
                const int n = T.nt * kBN + (r >> 5) * 64 + (r & 31);
                P.bo[j] = (2u * static_cast<uint32_t>(p.I) * p.H + static_cast<uint32_t>(n) * p.I) * 2 + gq * 16;
            }
        }
        if (p.gather) {
            P.ar = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.act), 0,
                                                     static_cast<int>(act_rows * kbytes), 0x00020000);
        } else {  // the tile's own rows only: any T*K*I stays within 32-bit offsets
            const int row0 = T.off + T.mt * kBM;
            const int rows = min(kBM, T.ne - T.mt * kBM);
            P.ar = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint16_t*>(p.act + static_cast<size_t>(row0) * p.kdim), 0,
                static_cast<int>(static_cast<uint32_t>(rows) * kbytes), 0x00020000);
        }
        const size_t ebase = static_cast<size_t>(T.e) * 3 * static_cast<size_t>(p.I) * p.H;
        P.wr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(p.w + ebase), 0,
            static_cast<int>(3u * static_cast<uint32_t>(p.I) * p.H * 2), 0x00020000);
    };

    // copies one half tile of stage kc of plan P into ring slot q % 2. The data is consumed from LDS, so the loads
    // bypass the L1 (sc0); they still allocate in L2, where the other m-tiles of the weight tile find them (a
    // non-temporal hint there made the kernel 35 % slower).
    const int bhalf = EPI == kSwiGLU ? p.I * p.H * 2 : 32 * p.I * 2;  // bytes from weight half 0 to half 1
    auto copyA = [&](int q, int h, int kc, const CopyPlan& P) __attribute__((always_inline)) {
        uint16_t* s = lds + (q % kNStage) * kStageHalfs + h * kHalfTile;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                P.ar, (__attribute__((address_space(3))) void*)(s + (wave * 2 + j) * 8 * kPitch), 16,
                static_cast<int>(P.ao[h * 2 + j]), kc * kBK * 2, 0, kCopyPolicy);
    };
    auto copyB = [&](int q, int h, int kc, const CopyPlan& P) __attribute__((always_inline)) {
        uint16_t* s = lds + (q % kNStage) * kStageHalfs + (2 + h) * kHalfTile;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                P.wr, (__attribute__((address_space(3))) void*)(s + (wave * 2 + j) * 8 * kPitch), 16,
                static_cast<int>(P.bo[j]), kc * kBK * 2 + h * bhalf, 0, kCopyPolicy);
    };
    // Accumulators acc[hA][hB]: 4 x 2 blocks of 16 x 16. Fragments: one activation half (4 blocks, both 32-k steps)
    // and both weight halves (2 blocks each).
    using Acc = f32x4[2][4][2];
    f16x8 fa[2][4], fb0[2][2], fb1[2][2];
    const int sw = (row16 >> 1) & 7;
    auto rdA = [&](int q, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const uint16_t* s = lds + (q % kNStage) * kStageHalfs + h * kHalfTile + (wm * 64 + row16) * kPitch +
                                (((kk * 4 + kg) ^ sw) * 8);
#pragma unroll
            for (int i = 0; i < 4; ++i) fa[kk][i] = *reinterpret_cast<const f16x8*>(s + i * 16 * kPitch);
        }
    };
    auto rdB = [&](int q, int h, f16x8 (&fb)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const uint16_t* s = lds + (q % kNStage) * kStageHalfs + (2 + h) * kHalfTile + (wn * 32 + row16) * kPitch +
                                (((kk * 4 + kg) ^ sw) * 8);
#pragma unroll
            for (int j = 0; j < 2; ++j) fb[kk][j] = *reinterpret_cast<const f16x8*>(s + j * 16 * kPitch);
        }
    };
    // Ends a memory tick: the fragments just read are in registers, and all but this wave's youngest 8 copies have
    // landed, the half tiles of the next memory tick among them; the barrier publishes them. `stores` (0, 8 or 16):
    // at least that many stores of the last tile's epilogue are younger than the copies waited for and need not
    // have ended.
    auto tick_m = [&](int stores = 0) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if (stores == 8) __builtin_amdgcn_s_waitcnt(vmcnt_imm(16) & 0xf0ffu);
        else if (stores == 16) __builtin_amdgcn_s_waitcnt(vmcnt_imm(24) & 0xf0ffu);
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm(8) & 0xf0ffu);
        ring_barrier();
    };
    // A compute tick: D[weight row][activation row], each lane ends with 4 consecutive output columns of one row.
    // half: the last stage of an odd multiple of 32, only its first 32-k step is multiplied.
    auto tick_c = [&](Acc& c, bool zero, bool half) __attribute__((always_inline)) {
        auto mma = [&](int kk) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    c[j >> 1][i][j & 1] =
                        mfma16x16x32(j < 2 ? fb0[kk][j & 1] : fb1[kk][j & 1], fa[kk][i],
                                     zero && kk == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : c[j >> 1][i][j & 1]);
        };
        mma(0);
        if (!KT || !half) mma(1);
        ring_barrier();
    };
    // The two tick pairs of 64-k stage q. half1 reads the first activation half and both weight halves, half2 the
    // second activation half. Each refills what the memory tick before it read last: half1 the second activation
    // half of stage q + 1 (stage kc of plan P), half2 the other three half tiles of stage q + 2 (again kc of P).
    int stores = 0;  // stores of this wave's last epilogue, younger than the copies that stage 0 waits for
    auto half1 = [&](Acc (&acc)[2], int q, bool first, int kc, const CopyPlan& P, bool half)
                     __attribute__((always_inline)) {
        rdA(q, 0);
        rdB(q, 0, fb0);
        rdB(q, 1, fb1);
        copyA(q + 1, 1, kc, P);
        tick_m(first ? stores : 0);
        tick_c(acc[0], first, half);
    };
    auto half2 = [&](Acc (&acc)[2], int q, bool first, int kc, const CopyPlan& P, bool half)
                     __attribute__((always_inline)) {
        rdA(q, 1);
        copyA(q, 0, kc, P);
        copyB(q, 0, kc, P);
        copyB(q, 1, kc, P);
        tick_m(first ? stores : 0);
        tick_c(acc[1], first, half);
    };

    // Epilogue: a lane of acc[a][b][i][j] holds D[weight row 4 * kg + r of block j of weight half b][activation row
    // row16 of block i of activation half a], i.e. 4 consecutive output columns of one row.
    auto epilogue = [&](const Acc (&acc)[2], const TileRef& cur, const int* rows) __attribute__((always_inline)) {
        const int lane_e = lane_fresh(), row16 = lane_e & 15, kg = lane_e >> 4;
        if (SPLIT && cur.part >= 0) {
            // a piece of a split tile: the raw fp32 sums of its k-range, [activation row][weight row] of the tile
            float* dst =
                p.partial + static_cast<size_t>(cur.part) * (kBM * kBN) + (wm * 64 + row16) * kBN + wn * 64 + kg * 4;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<f32x4*>(dst + ((i >> 2) * 128 + (i & 3) * 16) * kBN + j * 16) =
                        acc[i >> 2][j >> 1][i & 3][j & 1];
            }
        } else if (EPI == kSwiGLU) {
            // stored through a buffer that ends with the tile's rows; columns past I go past it too
            const int row0 = cur.mt * kBM;
            const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(
                p.out + static_cast<size_t>(cur.off + row0) * p.I, 0, min(kBM, cur.ne - row0) * p.I * 2, 0x00020000);
            const int col = cur.nt * 128 + wn * 32 + (kg & 1) * 16 + (kg >> 1) * 8;
            const uint32_t at = col < p.I ? static_cast<uint32_t>((wm * 64 + row16) * p.I + col) * 2 : 0x80000000u;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint32_t v[2][2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const f32x4 g = acc[i >> 2][0][i & 3][j], u = acc[i >> 2][1][i & 3][j];
                    // each value converted by itself: the last product and the rounding to fp16 are then one
                    // v_fma_mixlo_f16, rounded once
                    v[j][0] = f32_to_f16_bits(swiglu_fast(g[0], u[0])) |
                              (static_cast<uint32_t>(f32_to_f16_bits(swiglu_fast(g[1], u[1]))) << 16);
                    v[j][1] = f32_to_f16_bits(swiglu_fast(g[2], u[2])) |
                              (static_cast<uint32_t>(f32_to_f16_bits(swiglu_fast(g[3], u[3]))) << 16);
                }
                // odd rows of 16 lanes of block 0 against even ones of block 1: each lane then holds 8 columns in a row
                const auto lo = __builtin_amdgcn_permlane16_swap(v[0][0], v[1][0], false, false);
                const auto hi = __builtin_amdgcn_permlane16_swap(v[0][1], v[1][1], false, false);
                // The row's offset goes into the vector offset. With a scalar one the compiler leaves no wait state
                // between a 16-byte buffer store and the next write of its data registers (it counts that case as
                // safe), and where the next instruction was such a write, lanes 12-15 of each row stored the next
                // value.
                const uint32_t row = static_cast<uint32_t>(((i >> 2) * 128 + (i & 3) * 16) * p.I) * 2;
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo[0], hi[0], lo[1], hi[1]}, hr,
                                                       static_cast<int>(at + row), 0, 0);
            }
        } else {
            // Whole-line stores: the wave's 128 x 64 sub-tile leaves as 16 instructions of 8 rows x 128 B. Row
            // block i passes through the wave's own 2 KB of LDS (16 rows x 128 B; 16-byte granule g of row r at
            // g ^ (r & 7)): lane (row16, kg) writes its four packed 4-column groups, then lane L reads granule
            // L % 8 of row h * 8 + L / 8 (h = 0, 1). Stored straight from the MFMA layout (16 rows x 32 B per
            // instruction) the epilogue cost ~100 us per DeepSeek-V2-Lite down launch (T = 16384, E = 64, K = 6).
            uint8_t* stg = reinterpret_cast<uint8_t*>(lds) + tiled_epi_stage_offset(p.E) + wave * 2048;
            // Rows past the tile's last and columns past H repeat the last valid row or granule, its data too: no
            // divergent branch, and a full tile issues exactly 16 stores.
            const int ncol = p.H - cur.nt * kBN - wn * 64;  // valid columns of the wave
            if (ncol <= 0) return;
            const int rr = lane_e >> 3, gq = min(lane_e & 7, (ncol - 1) >> 3);
            const int col = cur.nt * kBN + wn * 64 + gq * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r0 = (i >> 2) * 128 + wm * 64 + (i & 3) * 16;  // the block's first row of the tile
                const int last = min(15, cur.ne - cur.mt * kBM - r0 - 1);
                if (last < 0) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 v = acc[i >> 2][j >> 1][i & 3][j & 1];
                    *reinterpret_cast<uint2*>(stg + row16 * 128 + (((2 * j + (kg >> 1)) ^ (row16 & 7)) << 4) +
                                              ((kg & 1) << 3)) =
                        make_uint2(pack_f16(v[0], v[1]), pack_f16(v[2], v[3]));
                }
                // the reads take what other lanes of this wave just wrote (LDS operations of one wave run in order)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                u32x4 v[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = min(h * 8 + rr, last);
                    v[h] = *reinterpret_cast<const u32x4*>(stg + r * 128 + ((gq ^ (r & 7)) << 4));
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // read before the next block's writes
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int r = r0 + min(h * 8 + rr, last);
                    *reinterpret_cast<u32x4*>(p.out + static_cast<size_t>(rows[r]) * p.H + col) = v[h];
                }
            }
        }
    };

    CopyPlan plan;
    load_rows(cur, 0);
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();
    make_plan(cur, 0, plan);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        const int kc = (SPLIT ? cur.k0 : 0) + st;
        copyA(st, 0, kc, plan);
        copyB(st, 0, kc, plan);
        copyB(st, 1, kc, plan);
        __builtin_amdgcn_sched_barrier(0);
        if (st == 0) copyA(st, 1, kc, plan);
        __builtin_amdgcn_sched_barrier(0);  // stage 0 first: the counted wait below covers its first three half tiles
    }
    tick_m();  // the first half tiles of stage 0
    int q0 = 0;  // ring index of the current item's first stage
    for (int k = 0;; ++k) {
        TileRef nxt = cur;
        const bool has_next = tile_at(k + 1, nxt);
        // table k + 1 % 3 was last read two tiles ago; the barriers of tile k - 1 separate those reads from this copy
        if (has_next) load_rows(nxt, (k + 1) % 3);
        // the last two stages copy the next item's first two (or, after the last item, repeat this one's last)
        const int k0 = SPLIT ? cur.k0 : 0, nk = SPLIT ? cur.nk : nst;  // nk >= 2
        const int nk0 = SPLIT ? nxt.k0 : 0;
        const int kc0 = has_next ? nk0 : k0 + nk - 1, kc1 = has_next ? nk0 + 1 : k0 + nk - 1;
        const bool tail = KT && k0 + nk == nst;  // this item ends with the 32-column k-stage
        if (nk < 4) {  // the next plan is needed before the counted waits cover its row table's copy: wait here
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
            __syncthreads();
        }
        if (wm) ring_barrier();  // waves 4-7 run one tick behind waves 0-3
        Acc acc[2];
        auto full = [&](int s, bool first) __attribute__((always_inline)) {
            half1(acc, q0 + s, first, k0 + s + 1, plan, false);
            half2(acc, q0 + s, first, k0 + s + 2, plan, false);
        };
        if (nk > 2) {
            full(0, true);
            for (int s = 1; s + 2 < nk; ++s) full(s, false);
            half1(acc, q0 + nk - 2, false, k0 + nk - 1, plan, false);
            if (has_next) make_plan(nxt, (k + 1) % 3, plan);
            half2(acc, q0 + nk - 2, false, kc0, plan, false);
        } else {
            half1(acc, q0, true, k0 + 1, plan, false);
            if (has_next) make_plan(nxt, (k + 1) % 3, plan);
            half2(acc, q0, true, kc0, plan, false);
        }
        half1(acc, q0 + nk - 1, false, kc0, plan, tail);
        half2(acc, q0 + nk - 1, false, kc1, plan, tail);
        if (!wm) ring_barrier();
        epilogue(acc, cur, rowtab + (k % 3) * kBM);
        // every lane of gate/up stores (past the buffer where there is no row), down skips blocks of rows or columns
        // that are not there
        stores = EPI == kSwiGLU ? 8 : (cur.ne - cur.mt * kBM >= kBM && (cur.nt + 1) * kBN <= p.H ? 16 : 0);
        if (!has_next) break;
        cur = nxt;
        q0 += nk;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the surplus copies have landed before the workgroup ends
}

// Down projection: adds the pieces of each split leftover tile in piece order (fixed, so the result does not
// depend on timing) and scatters the fp16 rows to expert_out. Workgroup (g, rb) takes rows [rb * kFixRows, +kFixRows)
// of leftover tile j = g / 8 of XCD x = g % 8; piece pc of that tile is in the partial slot of workgroup
// (j * S + pc) * 8 + x of the tiled launch, whose grid had nloc workgroups per XCD. The tile is found from offsets
// (each wave scans the experts 64 at a time).
__global__ __launch_bounds__(kFixThreads) void ffn_tiled_fixup_kernel(TiledArgs p, int nloc) {
    constexpr int nrb = kBM / kFixRows;
    const int rb = static_cast<int>(blockIdx.x) % nrb, g = static_cast<int>(blockIdx.x) / nrb;
    const int x = g % kXcds, j = g / kXcds;
    const int lane = lane_id();
    auto tiles_of = [&](int e) {
        return e < p.E ? (p.offsets[e + 1] - p.offsets[e] + kBM - 1) / kBM * p.ntiles_n : 0;
    };
    int total = 0;
    for (int base = 0; base < p.E; base += kWave) {
        int v = tiles_of(base + lane);
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) v += __shfl_xor(v, d, kWave);
        total += v;
    }
    const XcdSched xs = xcd_sched(x, total, nloc, (p.kdim + kBK - 1) / kBK, 1);
    if (xs.S < 2 || j >= xs.L) return;
    const int t = xs.base + xs.R * nloc + j;
    // expert e with prefix(e) <= t < prefix(e) + tiles(e), prefix(e) = tiles of the experts before e
    int e = -1, before = 0, carry = 0;
    for (int base = 0; base < p.E && e < 0; base += kWave) {
        const int te = tiles_of(base + lane);
        int incl = te;
#pragma unroll
        for (int d = 1; d < kWave; d <<= 1) {
            const int v = __shfl_up(incl, d, kWave);
            if (lane >= d) incl += v;
        }
        const uint64_t hit = __ballot(te > 0 && carry + incl - te <= t && t < carry + incl);
        if (hit) {
            const int l = __builtin_ctzll(hit);
            e = base + l;
            before = carry + __shfl(incl - te, l, kWave);
        }
        carry += __shfl(incl, kWave - 1, kWave);
    }
    const int mt_count = (p.offsets[e + 1] - p.offsets[e] + kBM - 1) / kBM;
    const int local = t - before, nt = local / mt_count, mt = local - nt * mt_count;
    const int off = p.offsets[e], rows = min(kBM, p.offsets[e + 1] - off - mt * kBM);
    const float* part0 = p.partial + static_cast<size_t>(j * xs.S * kXcds + x) * (kBM * kBN);
    const size_t pstride = static_cast<size_t>(kXcds) * (kBM * kBN);  // next piece: li + 1
    const int tid = static_cast<int>(threadIdx.x);
    // 64 threads per row, 4 consecutive output columns each; 4 rows per thread, loaded together
    constexpr int kRows = kFixRows / (kFixThreads / 64);
    const int c = (tid % 64) * 4, r0 = rb * kFixRows + tid / 64;
    const float* src = part0 + r0 * kBN + c;
    f32x4 v[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) v[u] = *reinterpret_cast<const f32x4*>(src + u * (kFixThreads / 64) * kBN);
#pragma unroll 2
    for (int pc = 1; pc < xs.S; ++pc)
#pragma unroll
        for (int u = 0; u < kRows; ++u)
            v[u] += *reinterpret_cast<const f32x4*>(src + pc * pstride + u * (kFixThreads / 64) * kBN);
    const int col = nt * kBN + c;
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
        const int r = r0 + u * (kFixThreads / 64);
        if (r >= rows || col >= p.H) continue;
        const uint32_t lo = f32_to_f16_bits(v[u][0]) | (static_cast<uint32_t>(f32_to_f16_bits(v[u][1])) << 16);
        const uint32_t hi = f32_to_f16_bits(v[u][2]) | (static_cast<uint32_t>(f32_to_f16_bits(v[u][3])) << 16);
        const int slot = p.sorted_slot[off + mt * kBM + r];
        *reinterpret_cast<uint2*>(p.out + static_cast<size_t>(slot) * p.H + col) = make_uint2(lo, hi);
    }
}

// Persistent grid: at most the workgroups the device holds at once, a multiple of the XCD count. SPLIT (the down
// projection): with p.split set, the leftover tiles are split over k and the fix-up kernel follows.
template <int EPI, bool SPLIT, bool KT>
hipError_t launch_tiled(TiledArgs p, int grid, const char* name, hipStream_t stream) {
    const void* fn = reinterpret_cast<const void*>(&ffn_tiled_kernel<EPI, SPLIT, KT>);
    const int lds = tiled_lds_bytes(p.E, EPI == kScatter);
    const int resident = resident_workgroups(fn, kThreads, lds);
    if (resident > 0 && resident < grid) grid = resident;
    grid = grid / kXcds * kXcds;
    if (grid < kXcds) grid = kXcds;
    // the leftover round is sized by the workgroups per XCD, so a split needs the grid to be all resident; each
    // workgroup owns one partial slot
    p.split = (SPLIT && p.split && resident > 0 && grid <= kMaxParts) ? 1 : 0;
    {
        TraceScope trace(name, stream);
        ffn_tiled_kernel<EPI, SPLIT, KT><<<grid, kThreads, lds, stream>>>(p);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || !p.split) return err;
    {
        TraceScope trace("moe_ffn_down_fixup", stream);
        ffn_tiled_fixup_kernel<<<grid * (kBM / kFixRows), kFixThreads, 0, stream>>>(p, grid / kXcds);
    }
    return hipGetLastError();
}

}  // namespace

// Both k extents need at least two stages (the ring runs two ahead) and the tile table must fit in the LDS left
// over by the ring.
bool tiled_shape_supported(int64_t H, int64_t E, int64_t I) {
    if (H % 32 != 0 || I % 32 != 0 || H <= kBK || I <= kBK) return false;
    return tiled_lds_bytes(static_cast<int>(E), true) <= kLdsMax;
}
// The buffer offsets are 32-bit: gathered x rows (T*H*2 bytes), one expert's weights (3*I*H*2) and the sorted
// slots (T*K*4) must stay below 2 GiB. The down projection addresses hidden per tile, so T*K*I has no such bound.
bool tiled_size_supported(int64_t T, int64_t H, int64_t K, int64_t I) {
    const int64_t lim = int64_t(1) << 31;
    return T * H * 2 < lim && 3 * I * H * 2 < lim && T * K * 4 < lim && static_cast<int64_t>(kBM) * I * 2 < lim;
}
bool tiled_supported(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I) {
    return tiled_shape_supported(H, E, I) && tiled_size_supported(T, H, K, I);
}
hipError_t prepare_ffn_tiled() {
    for (const void* fn : {reinterpret_cast<const void*>(&ffn_tiled_kernel<kSwiGLU, false, false>),
                           reinterpret_cast<const void*>(&ffn_tiled_kernel<kScatter, false, false>),
                           reinterpret_cast<const void*>(&ffn_tiled_kernel<kScatter, true, false>),
                           reinterpret_cast<const void*>(&ffn_tiled_kernel<kSwiGLU, false, true>),
                           reinterpret_cast<const void*>(&ffn_tiled_kernel<kScatter, false, true>),
                           reinterpret_cast<const void*>(&ffn_tiled_kernel<kScatter, true, true>)}) {
        const hipError_t err = ensure_lds_limit(fn, kLdsMax);
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}
int tiled_block_threads() { return kThreads; }
// The down projection splits leftover tiles into pieces of at least two k-stages (so only when I / kBK >= 4), and
// only when its tiles (bounded by tiled_down_grid) fill at most kSplitMaxRounds rounds of kMaxParts workgroups
// (one per CU on MI355X); a piece writes the partial slot of its workgroup, and the launch has at most
// min(kMaxParts, tiled_down_grid) workgroups.
bool tiled_down_splits(int T, int E, int K, int H, int I) {
    const int rounds = (tiled_down_grid(T, E, K, H) + kMaxParts - 1) / kMaxParts;
    return (I + kBK - 1) / kBK >= 4 && rounds <= kSplitMaxRounds;
}
size_t tiled_partial_bytes(int T, int H, int E, int K, int I) {
    if (!tiled_down_splits(T, E, K, H, I)) return 0;
    const int slots = min(kMaxParts, tiled_down_grid(T, E, K, H));
    return static_cast<size_t>(slots) * kBM * kBN * sizeof(float);
}
int tiled_rows_per_tile() { return kBM; }
// Upper bound on the tile count (sum over experts of ceil(rows_e / kBM) <= ceil(T*K / kBM) + E), rounded up to
// a multiple of the XCD count so that the XCD-contiguous remap in the kernel is a bijection on [0, grid).
int tiled_grid(int T, int E, int K, int ntiles_n) {
    const int m_bound = (T * K + kBM - 1) / kBM + E;
    const int g = m_bound * ntiles_n;
    return (g + kXcds - 1) / kXcds * kXcds;
}
int tiled_gateup_grid(int T, int E, int K, int I) { return tiled_grid(T, E, K, (I + 127) / 128); }
int tiled_down_grid(int T, int E, int K, int H) { return tiled_grid(T, E, K, (H + kBN - 1) / kBN); }

hipError_t launch_ffn_tiled(const uint16_t* x, const uint16_t* expert_weights, uint16_t* expert_out,
                            const FfnWorkspace& ws, int T, int H, int E, int K, int I, hipStream_t stream,
                            bool allow_split) {
    TiledArgs p{};
    p.sorted_slot = ws.sorted_slot;
    p.offsets = ws.offsets;
    p.w = expert_weights;
    p.T = T;
    p.E = E;
    p.K = K;
    p.H = H;
    p.I = I;
    p.act = x;
    p.out = ws.hidden;
    p.kdim = H;
    p.ntiles_n = (I + 127) / 128;
    p.gather = 1;
    p.partial = ws.partial;
    // an odd multiple of 32 along the reduction runs the KT instantiation, which multiplies only the first 32-k step of
    // the last stage
    const int ggrid = tiled_gateup_grid(T, E, K, I);
    const hipError_t err = H % kBK != 0
                               ? launch_tiled<kSwiGLU, false, true>(p, ggrid, "moe_ffn_gateup_swiglu", stream)
                               : launch_tiled<kSwiGLU, false, false>(p, ggrid, "moe_ffn_gateup_swiglu", stream);
    if (err != hipSuccess) return err;
    p.act = ws.hidden;
    p.out = expert_out;
    p.kdim = I;
    p.ntiles_n = (H + kBN - 1) / kBN;
    p.gather = 0;
    p.split = (allow_split && tiled_down_splits(T, E, K, H, I) && ws.partial != nullptr) ? 1 : 0;
    const int dgrid = tiled_down_grid(T, E, K, H);
    if (I % kBK != 0) {
        if (p.split) return launch_tiled<kScatter, true, true>(p, dgrid, "moe_ffn_down", stream);
        return launch_tiled<kScatter, false, true>(p, dgrid, "moe_ffn_down", stream);
    }
    if (p.split) return launch_tiled<kScatter, true, false>(p, dgrid, "moe_ffn_down", stream);
    return launch_tiled<kScatter, false, false>(p, dgrid, "moe_ffn_down", stream);
}

}  // namespace moe
