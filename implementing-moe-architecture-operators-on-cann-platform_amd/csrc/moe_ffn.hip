// moe_ffn.hip -- MoeExpertFFN: workspace layout and schedule dispatch of the grouped GEMMs.
//
// Reference: op_kernel/moe_expert_ffn.cpp:613-621 (kernel entry), op_host/moe_ops.cpp:340-349 (workspace).
// The expert FFN runs on one stream as
//   permute              expert-sorted slot order + per-expert offsets (workspace): moe_permute.hip for the
//                        tiled schedule; the streaming gate/up kernel finds its rows itself
//   gate/up + SwiGLU     hidden[r, :] = silu(x_t W_gate_e^T) * (x_t W_up_e^T) for sorted row r = (t, k), fp16
//   down + scatter       expert_out[t, k, :] = hidden[r, :] W_down_e^T, fp16
// The grouped GEMMs have two schedules, chosen on the host from the average number of rows per expert
// (the actual per-expert counts exist only on the device):
//   moe_ffn_stream.hip  weight streaming, for few rows per expert (HBM-bound: every weight byte read once)
//   moe_ffn_tiled.hip   256x256 LDS-tiled MFMA tiles, for many rows per expert (MFMA-bound)

#include "moe_device.h"
#include "moe_launch.h"
#include "moe_slot_rank.h"

namespace moe {

namespace {

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Average rows per expert from which the tiled schedule runs. The 32-row streaming kernels stream every expert's
// weights once per 32 rows, so they degrade once experts exceed 32 rows; the wide streaming kernels take up to 128
// rows per pass and run in their place from 32 rows at the latest (moe_ffn_stream.hip); the tiled kernels cost about
// the same from 32 to ~110 rows per expert (their 256-row tiles are then mostly padding). The host sees only the
// average: the wide kernels' time is that of the fullest experts, so it grows with uneven loads, the tiled kernels'
// hardly. The FFN alone, ids drawn uniformly (wide / tiled, us, one box):
//   H = 2048, E = 16, K = 2, I = 8192   32 rows 305 / 362, 48 rows 323 / 360, 56 rows 370 / 363, 64 rows 376 / 362,
//     (1.6 GB)                          72 rows 397 / 369, 96 rows 452 / 375, 112 rows 484 / 384, 128 rows 699 / 394
//   H = 4096, E = 8, K = 2, I = 14336   40 rows 559 / 599, 56 rows 597 / 612, 64 rows 664 / 622, 72 rows 707 / 624,
//     (2.8 GB)                          96 rows 794 / 641, 112 rows 839 / 657
//   H = 2048, E = 64, K = 6, I = 1408   32 rows 241 / 236, 40 rows 248 / 233, 56 rows 280 / 239, 72 rows 304 / 246
//     (1.1 GB)
//   H = 4096, E = 128, K = 8, I = 1536  32 rows 868 / 900, 40 rows 915 / 911, 56 rows 1059 / 942, 70 rows 1161 / 951
//   H = 7168, E = 256, K = 8, I = 2048  37 rows 4001 / 4202, 48 rows 4788 / 4300, 64 rows 5339 / 4397
//   H = 1024, E = 64, K = 4, I = 3072   32 rows 253 / 255, 40 rows 265 / 257, 64 rows 308 / 266  (1.2 GB)
//   H = 5120, E = 16, K = 2, I = 1536   40 rows 185 / 202, 56 rows 213 / 206, 72 rows 237 / 205  (0.75 GB)
//   H = 1024, E = 96, K = 4, I = 1024   40 rows 144 / 174, 64 rows 177 / 181, 72 rows 200 / 184  (0.6 GB)
//   H = 2048, E = 32, K = 4, I = 1408   48 rows 157 / 158, 64 rows 168 / 161, 72 rows 179 / 162  (0.55 GB)
//   H = 1536, E = 12, K = 2, I = 6144   66 rows 198 / 219, 80 rows 215 / 220, 96 rows 228 / 225, 104 rows 235 / 229
//     (0.7 GB)
//   H = 1024, E = 32, K = 4, I = 4096   48 rows 194 / 202, 56 rows 208 / 204, 65 rows 215 / 205, 80 rows 238 / 211,
//     (0.8 GB)                          96 rows 255 / 215
//   Zipf-skewed ids: H = 2048, E = 16, I = 8192 56 rows 940 / 425, 96 rows 1665 / 455; H = 2048, E = 64, I = 1408
//   32 rows 732 / 256, 64 rows 1373 / 307; H = 1024, E = 32, I = 4096 48 rows 542 / 220, 80 rows 873 / 252
// Three lines:
//   32 rows      shapes the wide kernels cannot run.
//   72 rows, and 97 from I = 4096   expert weights below 1 GB. Both were drawn on a slower tiled kernel: by the table
//                the present one wins from ~56-68 rows (H = 1536, E = 12 from ~90).
//   40 rows (E >= 64), 66 rows      expert weights of at least 1 GB, streamed from HBM whichever schedule runs for long
//                enough that the tiled one's permute and fix-up launches do not show. Calls without the split leftover
//                round's workspace (splits.tiled off) and sizes past the tiled kernels' offsets keep the lines above.
// Where the 1 GB line loses on even loads: 1 GB over few down output columns (E * H / 256 tiles) means a long I and few
// down tiles, each split over k. 64 tiles: H = 1024, E = 16, I = 14336 66 rows 352 / 426, 95 rows 411 / 445; H = 2048,
// E = 8, I = 14336 66 rows 365 / 420; H = 512, E = 32, I = 14336 66 rows 388 / 451; H = 256, E = 64, I = 14336 40 rows
// 424 / 477. 80 tiles: H = 2560, E = 8, I = 9216 66 rows 300 / 325, 85 rows 345 / 338. 96 tiles: H = 384, E = 64,
// I = 12288 40 rows 473 / 504, 52 rows 522 / 507; H = 768, E = 32, I = 8192 66 rows 342 / 329. It holds there all the
// same, for with a gate of Zipf-scaled columns the same sizes take (wide / tiled) 686 / 487 and 1006 / 492, 391 / 431
// (80 rows 572 / 448), 1477 / 499, 1256 / 495; H = 1280, E = 16, I = 9216 66 rows 598 / 371; 1412 / 490 at E = 64,
// H = 384.
constexpr int64_t kTiledMinRowsPerExpert = 32;
constexpr int64_t kWideMaxRowsPerExpert = 97;
constexpr int64_t kWideMaxRowsSmallI = 72;
constexpr int64_t kWideLargeI = 4096;
constexpr int64_t kLargeWeightBytes = int64_t{1} << 30;
constexpr int64_t kManyExperts = 64;
constexpr int64_t kLargeTiledMinRowsMany = 40;  // from kManyExperts experts
constexpr int64_t kLargeTiledMinRows = 66;

}  // namespace

int ffn_schedule(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, FfnSplits splits) {
    const bool stream_ok = stream_supported(static_cast<int>(H), static_cast<int>(I), splits.gateup);
    const int64_t wide_limit = I >= kWideLargeI ? kWideMaxRowsPerExpert : kWideMaxRowsSmallI;
    const int64_t limit = stream_wide_supported(static_cast<int>(H), static_cast<int>(I)) ? wide_limit
                                                                                          : kTiledMinRowsPerExpert;
    if (splits.tiled && 6 * E * I * H >= kLargeWeightBytes &&
        T * K >= (E >= kManyExperts ? kLargeTiledMinRowsMany : kLargeTiledMinRows) * E && tiled_supported(T, H, E, K, I))
        return 1;
    const bool many_rows = T * K >= limit * E;
    if (tiled_shape_supported(H, E, I) && (many_rows || !stream_ok))
        return tiled_size_supported(T, H, K, I) ? 1 : -1;
    if (stream_ok) return 0;
    return -1;
}

// Layout (each region 256-byte aligned): offsets [E+1] i32 | sorted_slot [T*K] i32 | hidden [T*K, I] fp16, then
// for the weight-streaming schedule: fp32 partial sums, [nsplit, T*K, H] when the down projection is split over K
// and [nsplit, T*K, 2*I] when the 32-row gate/up kernel splits H (the larger of the two; one serves both in turn) |
// slot_row [T*K] i32; for the tiled schedule: the permute's scratch (rank [T*K] i32, counts [chunks, E] i32),
// then with splits.tiled up to 256 fp32 partial tiles of 256 x 256 (64 MiB; one per workgroup of the down launch)
// for the leftover round it splits over k (none when I < 256 or when the down tiles fill more than 4 rounds).
size_t ffn_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, FfnSplits splits) {
    const size_t S = static_cast<size_t>(T) * static_cast<size_t>(K);
    size_t bytes = align_up(sizeof(int32_t) * static_cast<size_t>(E + 1), 256);
    bytes += align_up(sizeof(int32_t) * S, 256);
    bytes += align_up(sizeof(uint16_t) * S * static_cast<size_t>(I), 256);
    const int schedule = ffn_schedule(T, H, E, K, I, splits);
    if (schedule == 0) {
        bytes += align_up(stream_partial_bytes(static_cast<int>(T), static_cast<int>(H), static_cast<int>(E),
                                               static_cast<int>(K), static_cast<int>(I), stream_wide(T, H, E, K, I),
                                               splits.gateup), 256);
        bytes += align_up(sizeof(int32_t) * S, 256);
    } else if (schedule == 1) {
        bytes += align_up(permute_scratch_bytes(static_cast<int>(S), static_cast<int>(E)), 256);
        if (splits.tiled)
            bytes += align_up(tiled_partial_bytes(static_cast<int>(T), static_cast<int>(H), static_cast<int>(E),
                                                  static_cast<int>(K), static_cast<int>(I)), 256);
    }
    return bytes;
}

FfnWorkspace ffn_workspace_carve(void* base, int64_t T, int64_t H, int64_t E, int64_t K, int64_t I,
                                 FfnSplits splits) {
    const size_t S = static_cast<size_t>(T) * static_cast<size_t>(K);
    char* p = static_cast<char*>(base);
    FfnWorkspace ws;
    ws.offsets = reinterpret_cast<int32_t*>(p);
    p += align_up(sizeof(int32_t) * static_cast<size_t>(E + 1), 256);
    ws.sorted_slot = reinterpret_cast<int32_t*>(p);
    p += align_up(sizeof(int32_t) * S, 256);
    ws.hidden = reinterpret_cast<uint16_t*>(p);
    p += align_up(sizeof(uint16_t) * S * static_cast<size_t>(I), 256);
    ws.partial = nullptr;
    ws.slot_row = nullptr;
    ws.pscratch = nullptr;
    const int schedule = ffn_schedule(T, H, E, K, I, splits);
    if (schedule == 0) {
        ws.partial = reinterpret_cast<float*>(p);
        p += align_up(stream_partial_bytes(static_cast<int>(T), static_cast<int>(H), static_cast<int>(E),
                                           static_cast<int>(K), static_cast<int>(I), stream_wide(T, H, E, K, I),
                                           splits.gateup), 256);
        ws.slot_row = reinterpret_cast<int32_t*>(p);
    } else if (schedule == 1) {
        ws.pscratch = reinterpret_cast<int32_t*>(p);
        p += align_up(permute_scratch_bytes(static_cast<int>(S), static_cast<int>(E)), 256);
        if (splits.tiled && tiled_partial_bytes(static_cast<int>(T), static_cast<int>(H), static_cast<int>(E),
                                               static_cast<int>(K), static_cast<int>(I)) > 0)
            ws.partial = reinterpret_cast<float*>(p);
    }
    return ws;
}

namespace {

// Without the partial tiles of the split leftover round: the schedule lines below 1 GB of expert weights, and the
// workspace of calls streamed under them.
constexpr FfnSplits kNoPartialTiles = {/*tiled=*/false, /*gateup=*/true};

// A size that only the rule for 1 GB of expert weights takes to the tiled schedule. Its need then differs from the
// streaming one, either way (74.4 MB tiled and 7.3 MB streamed at T = 432, H = 2048, E = 64, K = 6, I = 1408; 61.3 MB
// and 75.7 MB at T = 264, H = 4096, E = 8, K = 2, I = 14336), while its neighbours below the line stream.
bool tiled_by_weight_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I) {
    return ffn_schedule(T, H, E, K, I) == 1 && ffn_schedule(T, H, E, K, I, kNoPartialTiles) == 0;
}

size_t need_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, FfnSplits splits, bool layer) {
    return layer ? layer_workspace_bytes(T, H, E, K, I, splits) : ffn_workspace_bytes(T, H, E, K, I, splits);
}

}  // namespace

// A workspace that holds what streaming needs, but not the tiled schedule's regions, is enough for such a size (it may
// have been sized for another T): the call streams. Every other size needs its whole workspace.
FfnSplits workspace_splits(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, size_t bytes, bool layer) {
    if (bytes < need_bytes(T, H, E, K, I, {}, layer) && tiled_by_weight_bytes(T, H, E, K, I) &&
        bytes >= need_bytes(T, H, E, K, I, kNoPartialTiles, layer))
        return kNoPartialTiles;
    return {};
}

// The larger of the two needs there, so that a workspace sized for such a T also holds the smaller T that stream.
size_t workspace_query(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, bool layer) {
    const size_t need = need_bytes(T, H, E, K, I, {}, layer);
    if (!tiled_by_weight_bytes(T, H, E, K, I)) return need;
    const size_t streamed = need_bytes(T, H, E, K, I, kNoPartialTiles, layer);
    return need > streamed ? need : streamed;
}

FfnGrid ffn_grid(int T, int H, int E, int K, int I) {
    FfnGrid g;
    g.schedule = ffn_schedule(T, H, E, K, I);
    if (g.schedule == 1) {
        g.block_threads = tiled_block_threads();
        g.gateup_blocks = tiled_gateup_grid(T, E, K, I);
        g.down_blocks = tiled_down_grid(T, E, K, H);
        g.rows_per_tile = tiled_rows_per_tile();
    } else {
        g.block_threads = stream_block_threads();
        g.gateup_blocks = stream_gateup_grid(T, H, E, K, I, stream_wide(T, H, E, K, I));
        g.down_blocks = stream_down_grid(T, H, E, K, I, stream_wide(T, H, E, K, I));
        g.rows_per_tile = stream_rows_per_pass();
    }
    return g;
}

hipError_t launch_ffn(const uint16_t* x, const int32_t* expert_ids, const uint16_t* expert_weights,
                      uint16_t* expert_out, FfnWorkspace ws, int T, int H, int E, int K, int I, hipStream_t stream,
                      FfnSplits splits) {
    switch (ffn_schedule(T, H, E, K, I, splits)) {
        case 1: {
            hipError_t err = prepare_permute(T * K, E);
            if (err == hipSuccess) err = prepare_ffn_tiled();
            if (err == hipSuccess) err = launch_permute(expert_ids, T * K, E, H, ws, expert_out, stream);
            if (err != hipSuccess) return err;
            return launch_ffn_tiled(x, expert_weights, expert_out, ws, T, H, E, K, I, stream, splits.tiled);
        }
        case 0: {
            const hipError_t err = prepare_ffn_stream(H, I);
            if (err != hipSuccess) return err;
            return launch_ffn_stream(x, expert_ids, expert_weights, expert_out, ws, T, H, E, K, I, stream, nullptr,
                                     nullptr, splits.gateup);
        }
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ffn_combine(const uint16_t* x, const int32_t* expert_ids, const uint16_t* weights,
                              const uint16_t* expert_weights, uint16_t* expert_out, uint16_t* y, FfnWorkspace ws,
                              int T, int H, int E, int K, int I, hipStream_t stream, FfnSplits splits) {
    if (ffn_schedule(T, H, E, K, I, splits) == 0) {
        const hipError_t err = prepare_ffn_stream(H, I);
        if (err != hipSuccess) return err;
        return launch_ffn_stream(x, expert_ids, expert_weights, expert_out, ws, T, H, E, K, I, stream, weights, y,
                                 splits.gateup);
    }
    const hipError_t err = launch_ffn(x, expert_ids, expert_weights, expert_out, ws, T, H, E, K, I, stream, splits);
    if (err != hipSuccess) return err;
    return launch_combine(expert_out, weights, y, T, H, K, stream);
}

size_t layer_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t K, int64_t I, FfnSplits splits) {
    size_t bytes = ffn_workspace_bytes(T, H, E, K, I, splits);
    // counts for the routing blocks of any routing kernel: at most one block per 16 tokens
    if (ffn_schedule(T, H, E, K, I, splits) == 1)
        bytes += align_up(sizeof(int32_t) * static_cast<size_t>((T + 15) / 16) * counts_stride(static_cast<int>(E)), 256);
    else  // the split routing's quarter sums (small batches, E > 64)
        bytes += align_up(routing_split_workspace_bytes(static_cast<int>(T), static_cast<int>(E)), 256);
    return bytes;
}

hipError_t launch_layer(const uint16_t* x, const uint16_t* w_gate, const uint16_t* expert_weights, int32_t* ids,
                        uint16_t* weights, uint16_t* expert_out, uint16_t* y, void* workspace, int T, int H, int E,
                        int K, int I, hipStream_t stream, FfnSplits splits) {
    const FfnWorkspace ws = ffn_workspace_carve(workspace, T, H, E, K, I, splits);
    // what follows the FFN's regions: the routing blocks' counts (tiled) or the split routing's sums (streaming)
    char* const tail = static_cast<char*>(workspace) + ffn_workspace_bytes(T, H, E, K, I, splits);
    switch (ffn_schedule(T, H, E, K, I, splits)) {
        case 1: {
            hipError_t err = prepare_ffn_tiled();
            if (err != hipSuccess) return err;
            int32_t* rank = ws.pscratch;  // [T*K] in the permute's scratch
            int32_t* counts = reinterpret_cast<int32_t*>(tail);
            err = launch_routing_topk(x, w_gate, ids, weights, T, H, E, K, stream, counts, rank);
            if (err != hipSuccess) return err;
            const bool lw = routing_lds_weights(w_gate, H, E);  // the same choice the routing launch makes
            const int nblocks = routing_blocks(T, H, E, lw);
            err = launch_permute_scatter(ids, T * K, E, H, counts, rank, nblocks, routing_tokens_per_block(T, H, E, lw) * K,
                                         permute_scatter_chunks_per_block(nblocks), ws, expert_out, stream);
            if (err != hipSuccess) return err;
            err = launch_ffn_tiled(x, expert_weights, expert_out, ws, T, H, E, K, I, stream, splits.tiled);
            if (err != hipSuccess) return err;
            return launch_combine(expert_out, weights, y, T, H, K, stream);
        }
        case 0: {
            hipError_t err = prepare_ffn_stream(H, I);  // the FFN kernels' attributes before the first launch
            if (err != hipSuccess) return err;
            if (routing_split_applies(T, H, E, routing_lds_weights(w_gate, H, E))) {
                err = launch_routing_split(x, w_gate, ids, weights, T, H, E, K, reinterpret_cast<float*>(tail), stream);
            } else {
                err = launch_routing_topk(x, w_gate, ids, weights, T, H, E, K, stream);
            }
            if (err != hipSuccess) return err;
            return launch_ffn_combine(x, ids, weights, expert_weights, expert_out, y, ws, T, H, E, K, I, stream,
                                      splits);
        }
        default: return hipErrorInvalidValue;
    }
}

}  // namespace moe
