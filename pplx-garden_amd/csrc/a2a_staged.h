// Staging buffers and kernels of the split calls (one logical rank per call).
//
// They keep the reference's structure: a send stages the rows of its tokens
// (a2a_dispatch_send.cu:341-367), a recv lays out what it received and copies
// it into the caller's buffers (a2a_worker.rs:526-703 on the CPU there, then
// a2a_dispatch_recv.cu:122-156), combine-send copies expert rows back to the
// staging row of the copy they answer (a2a_combine_send.cu:119-138,182-207)
// and combine-recv gathers them (a2a_combine_recv.cu:94-148).
//
// Differences that follow from every rank living in one HBM: a token is staged
// ONCE (quantised), not once per route, and the receiver finds it through a
// position -> token table; the private / overflow split of the receive buffer
// (max_private_tokens) moves no row here, but the recv still writes the two
// offset tables that encode it (source_dispatch_offset, combine_send_offset),
// bit for bit what the reference's host worker computes.
#pragma once

#include <string>

#include "a2a_internal.h"

namespace a2a {

struct Staging {
    bool allocated = false;
    void *arena = nullptr;
    uint8_t *send_buf = nullptr;         // [N][max_num_tokens][disp_stride]: payload, scales, 16 spare bytes (+ padding to whole lines)
    uint32_t *pos_token = nullptr;       // [N][max_tk]: token behind each row of a sender's expert-sorted order
                                         // (the other way round, copy -> position, is in the workspace's route_slot)
    uint8_t *comb_buf = nullptr;         // [N][max_tk][comb_stride]: combine rows at the sender's positions
    uint32_t *padded_index = nullptr;    // [N][max_recv]
    uint32_t *source_rank = nullptr;     // [N][max_recv]
    uint32_t *source_position = nullptr; // [N][max_recv]
    uint32_t *source_dispatch_offset = nullptr;  // [N][max_recv]  a2a_worker.rs:636-656
    uint32_t *combine_send_offset = nullptr;     // [N][max_recv]  a2a_worker.rs:659-667
    uint4 *moves = nullptr;              // [N][max_recv]: what the copies need of a received row, side by side: its row in the
                                         // receiver's buffer, the staged row it comes from (sender * max_tokens + token), its
                                         // source and its position there
    uint32_t *num_recv = nullptr;        // [N][2]: received rows, rows from other nodes
    size_t disp_stride = 0;
    size_t comb_stride = 0;
    uint32_t payload_bytes = 0;          // offset of the scales inside a staged dispatch row
    uint32_t max_recv = 0;               // rows per receiver in the tables above
    uint32_t max_tokens = 0;
    uint32_t recv_mask = 0;              // receivers whose tables are valid in this step
    uint32_t combine_sent_mask = 0;
};

struct StageSendArgs {
    PushSrc src;
    uint32_t rank;
    uint32_t row_bytes;
    uint32_t hidden_dim;
    uint32_t hidden_dim_scale;
    uint32_t topk_magic;      // ceil(2^32 / K) (0 for K = 1), for entry -> token without a division
    uint32_t resolver_wave;   // resolving send: wavefront that resolves the routes (set by the launcher)
};

// What stage_send_quick_kernel needs (kShortArguments); buffers and tables are those of the sender's dp group.
struct SendQuickArgs {
    const uint8_t *x;
    const float *x_scale;
    const int32_t *indices;
    const int32_t *bound_m;
    uint64_t x_stride;        // bytes
    uint8_t *staged;
    uint32_t *pos_token;
    uint32_t *num_routed;
    uint32_t *token_offset;
    uint32_t *route_slot;
    uint32_t xs_stride_elem;  // elements
    uint32_t xs_stride_token;
    uint32_t num_tokens;
    uint32_t num_scales;
    uint32_t sizes;           // from bit 0: sixteen-byte pieces of a row (10), experts (11), routes per token (7)
    uint32_t distances;       // from num_routed on: to expert_offsets in kTableUnit (10), to the context's flags in words (22)

    __device__ __forceinline__ uint32_t pieces() const { return sizes & 0x3FF; }
    __device__ __forceinline__ uint32_t num_experts() const { return sizes >> 10 & 0x7FF; }
    __device__ __forceinline__ uint32_t topk() const { return sizes >> 21; }
    __device__ __forceinline__ uint32_t *expert_offsets() const { return num_routed + kTableUnit * (distances & 0x3FF); }
    __device__ __forceinline__ uint32_t *flags() const { return num_routed + (distances >> 10); }
};
static_assert(sizeof(SendQuickArgs) <= kShortArguments, "");
static_assert(holds(10, 1024 - kWave) && holds(11, A2A_MAX_EXPERTS) && holds(11, A2A_MAX_EXPERTS_PER_TOKEN), "sizes");
constexpr uint32_t kSenderTable = (A2A_MAX_WORLD_SIZE * A2A_MAX_EXPERTS + kTableUnit - 1) / kTableUnit;   // of the largest, in kTableUnit
static_assert(holds(10, kSenderTable) && holds(22, 3ull * kSenderTable * kTableUnit), "distances");

// A grid of wavefronts over the pieces (128 sixteen-byte chunks) of a receiver's rows.
struct PieceGrid {
    uint32_t pieces;          // of a row
    uint32_t magic;           // n / pieces = mulhi(n, magic) for the wavefronts of a grid (0 for one piece a row)
    uint32_t step_rows;       // wavefronts of the grid = step_rows * pieces + step_pieces
    uint32_t step_pieces;
};

// The staged row's stride: the reference's format (payload, scales, spare bytes; rows are whole 16-byte chunks) rounded up
// to whole cache lines.
__host__ __device__ inline size_t staged_row_stride(size_t row_bytes, size_t num_scales) {
    return (row_bytes + (num_scales * 4 + 15) / 16 * 16 + 16 + 255) / 256 * 256;
}

struct StageRecvArgs {   // of a recv as the host has it, and of the kernels that lay receivers out
    PushDst dst;
    int32_t *out_num_tokens;  // rows per local expert for the caller, may be null
    uint32_t rank;
    uint32_t row_bytes;
    uint32_t hidden_dim_scale;
    uint32_t max_rows;        // upper bound of received rows known to the host
    bool streamed;            // the copies are written past the Infinity Cache (received_past_cache)
    // the first recv of a step only: it lays out every receiver
    uint32_t valid_mask;      // sources that sent tokens in this step (the others count as empty)
    uint32_t max_private;     // rows per source in the private part of a receive region (a2a_worker.rs:646-656)
    uint32_t copy_blocks;     // few rows: workgroups that serve the caller's rank; the others lay out the other receivers (launcher)
    uint32_t slices;          // workgroups per receiver that is laid out for later recvs (launcher)
};

// What the kernel needs that copies a receiver's rows (kShortArguments).
struct RecvRowsArgs {
    uint8_t *out_x;
    float *out_scale;
    int32_t *out_num_tokens;  // may be null
    const uint8_t *staged;
    const uint4 *moves;       // the receiver's
    const uint32_t *num_recv; // the receiver's
    uint32_t *counts;         // rows of its experts
    uint64_t out_stride;      // bytes
    uint32_t os_stride_elem;  // elements
    uint32_t os_stride_token;
    uint32_t out_rows;
    uint32_t row_bytes;
    uint32_t num_scales;
    uint32_t max_recv;
    uint32_t pieces, magic, step_rows, step_pieces;   // PieceGrid
    uint32_t scale_blocks;    // workgroups in front of the grid that move scales by column
    // experts of the receiver, from their counts on to their first rows (in kTableUnit), and back to the context's flags (words)
    uint32_t num_local : 11, to_first_rows : 5, to_flags : 16;

    __device__ __forceinline__ uint32_t *flags() const { return counts - to_flags; }
};
static_assert(sizeof(RecvRowsArgs) <= kShortArguments, "");
// (the last receiver's first expert may lie up to a receiver's share behind the last one)
static_assert(holds(11, A2A_MAX_EXPERTS) && holds(5, (A2A_MAX_EXPERTS + kTableUnit - 1) / kTableUnit) &&
              holds(16, kTableUnit + A2A_MAX_EXPERTS + A2A_MAX_WORLD_SIZE), "num_local, to_first_rows, to_flags");

struct CombineSendArgs {
    const uint8_t *y;
    uint64_t y_stride;
    uint32_t y_rows;
    uint32_t row_bytes;
    // the launcher's
    uint8_t *staged;
    uint64_t staged_stride;
    const uint4 *moves;       // the receiver's
    const uint32_t *num_recv; // the receiver's
    uint32_t *err;
    uint32_t max_recv;
    uint32_t max_tk;
    PieceGrid grid;
};
static_assert(sizeof(CombineSendArgs) <= kShortArguments, "");

struct CombineRecvArgs {
    CombDst dst;
    uint32_t rank;
    uint32_t hidden_dim;
    uint32_t accumulate;
};

int staging_allocate(Staging &st, const a2a_config &cfg, std::string *error);
void staging_free(Staging &st);
// Device pointer of a receive-side table of `rank`, or null when none exists.
const uint32_t *staging_table(const Staging &st, const a2a_config &cfg, uint32_t rank, uint32_t which,
                              size_t *limit);

hipError_t launch_stage_send(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                             bool quantize, hipStream_t stream, KernelTiming timing = KernelTiming());
// One-launch send (routing counted inside) for small steps: whether a step qualifies, and the launch
// (dense index rows and a wavefront to spare: the kernel in which a spare wavefront resolves the
// positions while the others stage the row; otherwise the one in which every wavefront does both).
bool stage_send_small_fits(const StageSendArgs &args, const Workspace &ws);
hipError_t launch_stage_send_small(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                   bool quantize, hipStream_t stream, KernelTiming timing = KernelTiming());
// One-launch send for steps of up to 8192 entries that are too large for the small-step kernel
// (a workgroup counts once for several tokens): whether a step qualifies, and the launch (with a
// wavefront to spare, again the kernel in which it resolves the positions beside the teams).
bool stage_send_single_fits(const StageSendArgs &args, const Workspace &ws, bool quantize);
hipError_t launch_stage_send_single(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                    bool quantize, hipStream_t stream, KernelTiming timing = KernelTiming());
// One-launch send for larger steps (up to 65535 entries): the routing runs in workgroups beside those that stage the rows.
bool stage_send_beside_fits(const StageSendArgs &args, const Workspace &ws);
hipError_t launch_stage_send_beside(const StageSendArgs &args, const Workspace &ws, const Staging &st, bool quantize,
                                    hipStream_t stream, KernelTiming timing = KernelTiming());
// The send of a large step after launch_route_accumulate(..., for_send = true).
hipError_t launch_stage_send_resolve(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                     bool quantize, hipStream_t stream, KernelTiming timing = KernelTiming());
// `first_of_step`: no recv has run since the step's sends; all receivers are laid out first (`layout_timing`: where that
// is a launch of its own).
hipError_t launch_stage_recv(const StageRecvArgs &args, const Workspace &ws, const Staging &st, bool first_of_step,
                             hipStream_t stream, KernelTiming timing = KernelTiming(),
                             KernelTiming layout_timing = KernelTiming());
// `max_rows`: upper bound of the receiver's rows known to the host.
hipError_t launch_combine_send(const CombineSendArgs &args, uint32_t rank, uint32_t max_rows, const Workspace &ws,
                               const Staging &st, hipStream_t stream, KernelTiming timing = KernelTiming());
hipError_t launch_combine_recv(const CombineRecvArgs &args, const Workspace &ws, const Staging &st,
                               uint32_t in_dtype, uint32_t out_dtype, hipStream_t stream,
                               KernelTiming timing = KernelTiming());

}  // namespace a2a
