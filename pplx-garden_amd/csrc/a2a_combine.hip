// Combine: for every token, gather the K expert-output rows of its routes,
// weight them, accumulate in float and write one output row in token order.
//
// What it replaces: the reference's combine-send kernel (copy of every
// expert_y row back to the sender's staging buffer, a2a_combine_send.cu:
// 119-138,182-207) fused with its combine-recv kernel (weighted gather,
// a2a_combine_recv.cu:94-148).  Here the rows are read in place from the
// receivers' expert_y buffers, which live in the same HBM: one read per row,
// no staging write.
//
// Design for CDNA4: one wavefront per (token, slab of 64 sixteen-byte chunks);
// a lane owns 16 bytes of every source row, so K independent 16-byte loads are
// in flight per lane before the first multiply-add.  Row pointers and weights
// are resolved once by the first K lanes and read back as wave-uniform scalars:
// each row is a buffer descriptor (uniform base, one offset register for all
// rows) whose bound stands in for every condition.  Accumulation is an explicit
// float fused multiply-add chain, k ascending, then one round-to-nearest-even to
// the output type (combine_utils.cuh:108-114,14-23).
//
// What bounds it is HBM: reads alone of the 4096-token shape take 69 us, the
// output adds what 59 MB of writes cost between them.  4096 tokens of 14 KB
// rows, K = 8: 91.3 -> 89.7 us (5.9 TB/s) against loads under a condition each (means
// of several runs, which differ by 1.5 us); for float rows the compiler made
// copies of all rows' registers at each such condition and waited for every
// load by itself: 228.9 -> 101.4 us (4096 tokens of 16 KB rows).  Loads are non-temporal (ordinary
// ones 127 us; how the output is written: kStreamedOutput), and so is the load of what a combine
// accumulates onto (6000 tokens of 8 KB rows, K = 6: 76.5 -> 67.4 us).
#include "a2a_device.h"
#include "a2a_internal.h"
#include "a2a_rules.h"

namespace a2a {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Bf16 {};
struct F16 {};
struct F32 {};

template <typename T> struct Elem;
template <> struct Elem<Bf16> { static constexpr int kSize = 2; };
template <> struct Elem<F16> { static constexpr int kSize = 2; };
template <> struct Elem<F32> { static constexpr int kSize = 4; };

// Elements per 16-byte source chunk (vector.cuh:14-27: 8 for the 16-bit
// types, 4 for float).
template <typename T> constexpr int vec_elems() { return 16 / Elem<T>::kSize; }

template <typename T, int V>
__device__ __forceinline__ void load_elems(const uint8_t *p, float (&f)[V]) {
    if constexpr (Elem<T>::kSize == 4) {
        static_assert(V == 4 || V == 8, "");
#pragma unroll
        for (int h = 0; h < V / 4; ++h) {
            const u32x4 *q = reinterpret_cast<const u32x4 *>(p) + h;
            const u32x4 v = __builtin_nontemporal_load(q);
#pragma unroll
            for (int j = 0; j < 4; ++j) f[4 * h + j] = __uint_as_float(v[j]);
        }
    } else if constexpr (V == 8) {
        const u32x4 *q = reinterpret_cast<const u32x4 *>(p);
        const u32x4 v = __builtin_nontemporal_load(q);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (__is_same(T, Bf16)) {
                f[2 * j] = __uint_as_float(v[j] << 16);
                f[2 * j + 1] = __uint_as_float(v[j] & 0xFFFF0000u);
            } else {
                f[2 * j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[j] & 0xFFFF));
                f[2 * j + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[j] >> 16));
            }
        }
    } else {  // V == 4, 16-bit type: 8 bytes
        const u32x2 *q = reinterpret_cast<const u32x2 *>(p);
        const u32x2 v = __builtin_nontemporal_load(q);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (__is_same(T, Bf16)) {
                f[2 * j] = __uint_as_float(v[j] << 16);
                f[2 * j + 1] = __uint_as_float(v[j] & 0xFFFF0000u);
            } else {
                f[2 * j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[j] & 0xFFFF));
                f[2 * j + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[j] >> 16));
            }
        }
    }
}

template <typename U>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (__is_same(U, Bf16)) {
        const uint16_t lo = __builtin_bit_cast(uint16_t, (__bf16)a);
        const uint16_t hi = __builtin_bit_cast(uint16_t, (__bf16)b);
        return (uint32_t)lo | ((uint32_t)hi << 16);
    } else {
        const uint16_t lo = __builtin_bit_cast(uint16_t, (_Float16)a);
        const uint16_t hi = __builtin_bit_cast(uint16_t, (_Float16)b);
        return (uint32_t)lo | ((uint32_t)hi << 16);
    }
}

typedef int32_t i32x2 __attribute__((ext_vector_type(2)));

// The V elements of chunk `chunk` of the output row at `row`; lanes past the row's end (`bytes`) store nothing.
template <typename U, int V, int POLICY>
__device__ __forceinline__ void store_elems(uint64_t row, uint32_t bytes, uint32_t chunk, const float (&f)[V]) {
    const uint32_t offset = chunk * V * Elem<U>::kSize;
    if constexpr (Elem<U>::kSize == 4) {
#pragma unroll
        for (int h = 0; h < V / 4; ++h) {
            u32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __float_as_uint(f[4 * h + j]);
            store_row_chunk<POLICY>(v, row, bytes, offset + 16 * h);
        }
    } else if constexpr (V == 8) {
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = pack2<U>(f[2 * j], f[2 * j + 1]);
        store_row_chunk<POLICY>(v, row, bytes, offset);
    } else {
        i32x2 v;
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] = (int32_t)pack2<U>(f[2 * j], f[2 * j + 1]);
        __builtin_amdgcn_raw_buffer_store_b64(v, row_descriptor(row, bytes), (int)offset, 0, POLICY);
    }
}

// Convert one 16-byte source chunk (raw) and fuse it into the accumulators.
template <typename T, int V>
__device__ __forceinline__ void fma_chunk(const u32x4 raw, float w, float (&acc)[V]) {
    if constexpr (Elem<T>::kSize == 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(w, __uint_as_float(raw[j]), acc[j]);
    } else if constexpr (__is_same(T, Bf16)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[2 * j] = __builtin_fmaf(w, __uint_as_float(raw[j] << 16), acc[2 * j]);
            acc[2 * j + 1] = __builtin_fmaf(w, __uint_as_float(raw[j] & 0xFFFF0000u), acc[2 * j + 1]);
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[2 * j] = __builtin_fmaf(
                w, (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j] & 0xFFFF)), acc[2 * j]);
            acc[2 * j + 1] = __builtin_fmaf(
                w, (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j] >> 16)), acc[2 * j + 1]);
        }
    }
}

constexpr uint32_t kOneRankMaxTokens = 2048;   // largest step that takes the ONE_RANK variant of the gather

// How the gather writes: non-temporally, but past the Infinity Cache where the step's copies went past it
// (copies_past_cache in a2a_rules.h has the figures) or the tokens themselves are kStreamedOutput bytes or more (behind
// copies that went past it, non-temporal / past: 80 MB 126.0 / 122.1 us, 88 MB 138 / 133, 235 MB 371 / 360).  The ONE_RANK
// variant's outputs stay non-temporal (15 MB 23.4 us, past 24.0), and so do those of rows that were staged (they are
// written between the launches of the other ranks' calls).
constexpr uint64_t kStreamedOutput = 84000000;

// With eight loads a lane, 16 wavefronts a compute unit are enough to keep HBM busy, and more of them only have more
// rows open at a time.  us per combine, all wavefronts / bounded, K = 8: 470 MB of output past the cache 740 / 670-700,
// 4096 tokens of 14 KB rows 89.3 / 86.2, 8 x 512 tokens 89.9 / 87.9, 6000 tokens 131.1 / 127.2, 2668 tokens of 10 KB rows
// 43.1 / 42.2, 8 x 128 tokens 23.8 / 23.7.  What counts is the loads in flight, 128 a lane and compute unit: with K = 6
// (rows of 8 KB) 16 wavefronts make 2048 tokens slower (24.0 / 24.3), 21 do not (24.5 / 24.1; 6000 tokens 66.7 / 64.8, 12 000
// 132.9 / 127.8), K = 5 59.2 / 58.3; up to four loads a lane need all wavefronts (K = 2: 70.5 / 80.7 with 18).  Behind
// copies and in front of tokens that go past the cache 96 are enough: whole steps with 16 / 14 / 12 / 11 wavefronts, K = 8,
// 6000 tokens 216.6 / 214.1 / 212.7 / 214.2, 8 x 4096 tokens 1161 / 1145 / 1139 / 1152, 8 x 2048 tokens of 5 KB fp8 rows 416.1 /
// 410.2 / 406.7 / 409.3, float rows of 8 KB, 8 x 3000 tokens 663.7 / 657.5 / 655.4 / 656.7; K = 6 with 21 / 18 / 16, 8 x 4096
// tokens 894.5 / 888.6 / 878.0 (in the cache 14 are 0.9 us better at 4096 tokens and 0.3 worse at 2668, 12 worse).  The launch
// asks for LDS that nothing uses to bound them; with all of a compute unit's LDS given out, a kernel of another stream that
// wants some waits for wavefronts to end, as it does without the bound, where they take all the wave slots.  Eight combines
// beside bf16 matrix products on another stream, us for both, all wavefronts / bounded: 4096 tokens and eight products of
// 4096 x 2048 x 7168 1370 / 1350, of 4096 x 7168 x 7168 2974 / 2917, 32 of 512 x 7168 x 2048 1393 / 1380; 8 x 512 tokens 1374 / 1365,
// 2963 / 2933, 1403 / 1402.  The ONE_RANK variant is left alone (1024 tokens 23.6 / 23.4-23.7), and so are
// steps whose wavefronts fit the GPU all at once (kAllAtOnce): bounded to 16 they take a second, half empty round (rows of
// 14 KB: 8 x 40 tokens 9.08 / 8.68 us unbounded, 8 x 64 13.14 / 12.53; level where 16 hold them all and at 8064 wavefronts).
constexpr uint64_t kAllAtOnce = 32 * 256;

inline size_t lds_to_bound_waves(uint32_t topk, bool past_cache) {
    if (topk <= 4) return 0;
    constexpr size_t kLds = 160 * 1024, kBlock = 1280;   // of a compute unit, and what it is given out in
    const size_t waves = (past_cache ? 96 : 128) / (topk < 8 ? topk : 8);
    return kLds / waves / kBlock * kBlock;
}

// PIECES slabs of a token's output row, from piece `slab` * PIECES on: the rows that lanes 0..K-1 hold (address 0: not there),
// weighted and added up.
template <typename T, typename U, int GROUP, int PIECES, int LOAD, int OUT>
__device__ __forceinline__ void gather_slabs(uint64_t row_ptr, float weight, uint32_t K, uint32_t num_chunks, uint32_t slab,
                                             uint32_t lane, uint8_t *out_row, bool accumulate) {
    constexpr int V = vec_elems<T>();
    const uint32_t first = slab * PIECES * kWave + lane;
    float acc[PIECES][V];
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const uint32_t chunk = first + p * kWave;
#pragma unroll
        for (int j = 0; j < V; ++j) acc[p][j] = 0.0f;
        if (accumulate && chunk < num_chunks) load_elems<U, V>(out_row + (size_t)chunk * V * Elem<U>::kSize, acc[p]);
    }

    // GROUP routes at a time, all their loads asked for before the first is used.  A row is read through
    // a buffer descriptor of its own: uniform base, one offset register for all rows, and the descriptor's
    // bound takes the place of every condition (lanes past the row's end and rows that are not there read
    // zeros without touching memory).
    const uint64_t there = __ballot(row_ptr != 0);
    const uint32_t row_bytes = num_chunks * 16;
    for (uint32_t k0 = 0; k0 < K; k0 += GROUP) {
        u32x4 raw[GROUP][PIECES];
        float w[GROUP];
#pragma unroll
        for (int k = 0; k < GROUP; ++k) {
            const uint64_t row = read_lane64(row_ptr, k0 + k);
            w[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), (int)(k0 + k)));
#pragma unroll
            for (int p = 0; p < PIECES; ++p) raw[k][p] = load_row_chunk<LOAD>(row, row_bytes, (first + p * kWave) * 16);
        }
        const uint32_t have = (uint32_t)(there >> k0) & ((1u << GROUP) - 1);
        if (have == (1u << GROUP) - 1) {
#pragma unroll
            for (int k = 0; k < GROUP; ++k) {
#pragma unroll
                for (int p = 0; p < PIECES; ++p) fma_chunk<T, V>(raw[k][p], w[k], acc[p]);
            }
        } else {
            // (a row that is not there adds nothing, also with a weight that is not finite)
#pragma unroll
            for (int k = 0; k < GROUP; ++k) {
                if (!(have >> k & 1)) continue;
#pragma unroll
                for (int p = 0; p < PIECES; ++p) fma_chunk<T, V>(raw[k][p], w[k], acc[p]);
            }
        }
    }
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
        store_elems<U, V, OUT>((uint64_t)out_row, num_chunks * V * Elem<U>::kSize, first + p * kWave, acc[p]);
}

// T: type of the expert_y rows, U: type of out_tokens.  One WAVEFRONT handles
// one slab (PIECES of them) of 64 sixteen-byte chunks of one token; wavefronts share nothing, so
// a compute unit keeps many of them in flight and the latency of resolving a
// token's routes is hidden by the loads of its neighbours.  GROUP routes are
// loaded before the first is used: the smallest of 1, 2, 4, 8 that holds K, or
// groups of 8 (a load that fills a group up costs its issue only, but at K = 1
// three of them were 10 %: 96.7 -> 106.4 us for 16000 tokens).  PIECES: slabs a wavefront moves (two_pieces_a_lane in
// a2a_rules.h).  ONE_RANK: one rank
// alone has tokens and the step is small; its descriptor is read from a fixed
// place in the argument block, which takes two dependent scalar loads out of
// the head of every wavefront (0.1-0.4 us of a step of 128 to 1024 tokens; a
// 4096-token step hides them and is 0.3 us faster without the variant).
template <typename T, typename U, int GROUP, int PIECES, bool ONE_RANK, int OUT>
__global__ __launch_bounds__(kWave) void combine_gather_kernel(const CombArgs args, const Workspace ws) {
    constexpr int LOAD = OUT == kNonTemporal ? kNonTemporal : kDeviceNonTemporal;
    if constexpr (ONE_RANK) {
        // everything the head of a wavefront needs from the argument block, asked for in one go
        A2A_PIN(args.token_start[kMaxWorld]);
        A2A_PIN(args.single_rank);
        A2A_PIN(args.hidden_dim);
        A2A_PIN(args.accumulate);
        A2A_PIN(args.single.out);
        A2A_PIN(args.single.indices);
        A2A_PIN(args.single.weights);
        A2A_PIN(args.single.bound_m);
        A2A_PIN(args.single.out_stride);
        A2A_PIN(args.single.indices_stride);
        A2A_PIN(args.single.weights_stride);
        A2A_PIN(args.single.num_tokens);
        A2A_PIN(ws.world);
        A2A_PIN(ws.dp_size);
        A2A_PIN(ws.num_experts);
        A2A_PIN(ws.experts_per_rank);
        A2A_PIN(ws.le_magic);
        A2A_PIN(ws.max_tk);
        A2A_PIN(ws.route_slot);
        A2A_PIN(ws.err);
    }
    if constexpr (!ONE_RANK) {
        // (here too; measured on the 4096-token step: 0.7 us a step.  The same in the pack of that step cost
        // 1.2 us and is left out there.)
        A2A_PIN(args.token_start[0]);
        A2A_PIN(args.token_start[1]);
        A2A_PIN(args.layer_rows);
        A2A_PIN(args.hidden_dim);
        A2A_PIN(args.accumulate);
        A2A_PIN(ws.world);
        A2A_PIN(ws.dp_size);
        A2A_PIN(ws.num_experts);
        A2A_PIN(ws.experts_per_rank);
        A2A_PIN(ws.le_magic);
        A2A_PIN(ws.max_tk);
        A2A_PIN(ws.route_slot);
        A2A_PIN(ws.err);
    }
    const uint32_t lane = threadIdx.x;
    const uint32_t E = ws.num_experts;
    const uint32_t K = ws.topk;
    const uint32_t num_chunks = args.hidden_dim / vec_elems<T>();
    // the grid: slabs of a token side by side, then its tokens (no division stands in front of the loads)
    const uint32_t token_global = ONE_RANK ? blockIdx.y : blockIdx.z * args.layer_rows + blockIdx.y;
    const uint32_t slab = blockIdx.x;
    uint32_t g = 0, token = token_global;
    if constexpr (ONE_RANK) {
        if (token_global >= args.token_start[kMaxWorld]) return;   // the total, at a fixed place
        g = args.single_rank - 1;
    } else {
        if (token_global >= args.token_start[ws.world]) return;
        // the last rank that starts at or before this token, eight starts at a time asked for together
        // (the array is non-decreasing and ends in copies of the total)
        uint32_t start = 0;
        for (uint32_t r0 = 1; r0 < ws.world; r0 += 8) {
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                if (r0 + i < (uint32_t)kMaxWorld) {
                    const uint32_t first = args.token_start[r0 + i];
                    if (token_global >= first) {
                        g = r0 + i;
                        start = first;
                    }
                }
            }
        }
        token = token_global - start;
    }
    const CombDst &dst = ONE_RANK ? args.single : args.dst[g];
    const uint32_t group = g / ws.dp_size;   // the routing tables belong to the rank's dp group
    if (token >= effective_tokens(dst.bound_m, dst.num_tokens)) return;

    // Lane r holds the descriptor of receiver r; lanes 0..K-1 resolve a route
    // each and pick their receiver's descriptor with a lane shuffle.
    uint64_t y_base = 0, y_stride = 0;
    uint32_t y_rows = 0;
    if (lane < ws.world) {
        y_base = (uint64_t)args.src[lane].y;
        y_stride = args.src[lane].y_stride;
        y_rows = args.src[lane].y_rows;
    }
    uint32_t expert = 0, slot = 0;
    float weight = 0.0f;
    if (lane < K) {
        expert = (uint32_t)dst.indices[(size_t)token * dst.indices_stride + lane];
        weight = dst.weights[(size_t)token * dst.weights_stride + lane];
        slot = ws.route_slot[(size_t)group * ws.max_tk + token * K + lane];
    }
    const bool expert_ok = expert < E;
    const uint32_t r = expert_ok ? owner_of_expert(ws, expert) : 0;
    const uint64_t r_base = __shfl(y_base, (int)r);
    const uint64_t r_stride = __shfl(y_stride, (int)r);
    const uint32_t r_rows = __shfl(y_rows, (int)r);
    uint64_t row_ptr = 0;
    if (lane < K) {
        bool ok = false;
        if (expert_ok && r_base != 0 && slot < r_rows) {
            row_ptr = r_base + (uint64_t)slot * r_stride;
            ok = true;
        }
        if (!ok && slab == 0) atomicOr(ws.err, A2A_DEV_BAD_SLOT);
    }

    gather_slabs<T, U, GROUP, PIECES, LOAD, OUT>(row_ptr, weight, K, num_chunks, slab, lane, dst.out + (size_t)token * dst.out_stride,
                                        args.accumulate != 0);
}

// The combine's recv of the split calls: the rows are the staged ones of ONE sender, at the positions its send recorded
// per copy (a2a_combine_recv.cu:67-73 = exclusive offset of the expert + token offset), so that there is no receiver to
// look up and no second, dependent load in front of the rows.  What it needs is passed as the few words that they are
// (kShortArguments); otherwise as combine_gather_kernel.
template <typename T, typename U, int GROUP, int PIECES>
__global__ __launch_bounds__(kWave) void combine_staged_kernel(const CombineStagedArgs args) {
    A2A_PIN(args.out);
    A2A_PIN(args.indices);
    A2A_PIN(args.weights);
    A2A_PIN(args.bound_m);
    A2A_PIN(args.route_slot);
    A2A_PIN(args.staged);
    A2A_PIN(args.out_stride);
    A2A_PIN(args.staged_stride);
    A2A_PIN(args.indices_stride);
    A2A_PIN(args.weights_stride);
    A2A_PIN(args.num_tokens);
    A2A_PIN(args.layer_rows);
    A2A_PIN(args.max_tk);
    A2A_PIN(args.hidden_dim);
    A2A_PIN(args.num_experts);
    A2A_PIN(args.topk);
    A2A_PIN(args.accumulate);
    const uint32_t lane = threadIdx.x;
    const uint32_t K = args.topk;
    const uint32_t slab = blockIdx.x;
    const uint32_t token = blockIdx.z * args.layer_rows + blockIdx.y;
    if (token >= effective_tokens(args.bound_m, args.num_tokens)) return;
    float weight = 0.0f;
    uint64_t row_ptr = 0;
    if (lane < K) {
        const uint32_t expert = (uint32_t)args.indices[(size_t)token * args.indices_stride + lane];
        weight = args.weights[(size_t)token * args.weights_stride + lane];
        const uint32_t slot = args.route_slot[token * K + lane];
        if (expert < args.num_experts && slot < args.max_tk) {
            row_ptr = (uint64_t)(args.staged + (size_t)slot * args.staged_stride);
        } else if (slab == 0) {
            atomicOr(args.err, A2A_DEV_BAD_SLOT);
        }
    }
    gather_slabs<T, U, GROUP, PIECES, kNonTemporal, kNonTemporal>(row_ptr, weight, K, args.hidden_dim / vec_elems<T>(), slab, lane,
                                                         args.out + (size_t)token * args.out_stride, args.accumulate != 0);
}

// The combine of a small step with one sender, whose launch is what it costs: the words of kShortArguments instead of every
// rank's descriptors.  A receiver's rows are found by their distance from the first receiver's, which lane r holds for receiver r.
// Steps of 128 tokens, host's pace, medians of 14 processes a side in turn (which lie up to 10 % apart): hidden 7168 10.7 -> 9.8 us,
// 2048 10.7 -> 9.9; other steps of one sender (bounds, strided rows,
// more receivers, buffers of different lengths) keep the kernel above.
template <typename T, typename U, int GROUP, int PIECES>
__global__ __launch_bounds__(kWave) void combine_sole_kernel(const CombineSoleArgs args) {
    A2A_PIN(args.y);
    A2A_PIN(args.out);
    A2A_PIN(args.indices);
    A2A_PIN(args.weights);
    A2A_PIN(args.route_slot);
    A2A_PIN(args.y_stride);
    A2A_PIN(args.y_rows);
    A2A_PIN(args.out_stride);
    A2A_PIN(args.hidden_dim);
    A2A_PIN(args.le_magic);
    A2A_PIN(args.sizes);
    const uint32_t lane = threadIdx.x;
    const uint32_t K = args.topk();
    const uint32_t slab = blockIdx.x, token = blockIdx.y;
    const int32_t distance = args.y_offset[lane < kSoleReceivers ? lane : 0];
    uint32_t expert = 0, slot = 0;
    float weight = 0.0f;
    if (lane < K) {
        expert = (uint32_t)args.indices[token * K + lane];
        weight = args.weights[token * K + lane];
        slot = args.route_slot[token * K + lane];
    }
    const bool expert_ok = expert < args.num_experts();
    const uint32_t r = !expert_ok ? 0 : args.experts_per_rank() > 1 ? __umulhi(expert, args.le_magic) : expert;
    const int64_t r_distance = (int64_t)__shfl(distance, (int)r) * 16;
    uint64_t row_ptr = 0;
    if (lane < K) {
        if (expert_ok && slot < args.y_rows) {
            row_ptr = (uint64_t)(args.y + r_distance + (size_t)slot * args.y_stride * 16);
        } else if (slab == 0) {
            atomicOr(args.err, A2A_DEV_BAD_SLOT);
        }
    }
    gather_slabs<T, U, GROUP, PIECES, kNonTemporal, kNonTemporal>(
        row_ptr, weight, K, args.hidden_dim / vec_elems<T>(), slab, lane, args.out + (size_t)token * args.out_stride * 8,
        args.accumulate());
}

// Whether a step of one sender with rank `sender`'s tokens can be described by CombineSoleArgs, and the words.
static bool sole_args(const CombArgs &given, const Workspace &ws, uint32_t sender, CombineSoleArgs &a) {
    const CombDst &dst = given.dst[sender];
    const CombSrc &first = given.src[0];
    if (ws.world > kSoleReceivers || dst.bound_m != nullptr || dst.indices_stride != ws.topk || dst.weights_stride != ws.topk)
        return false;
    if (first.y_stride / 16 > 0xFFFFFFFFull || dst.out_stride / 8 > 0xFFFFFFFFull) return false;
    for (uint32_t r = 0; r < kSoleReceivers; ++r) {
        const CombSrc &src = given.src[r < ws.world ? r : 0];
        if (src.y == nullptr || src.y_stride != first.y_stride || src.y_rows != first.y_rows) return false;
        const int64_t distance = (src.y - first.y) / 16;   // (rows are 16-byte aligned)
        if (distance != (int32_t)distance) return false;
        a.y_offset[r] = (int32_t)distance;
    }
    a.y = first.y;
    a.out = dst.out;
    a.indices = dst.indices;
    a.weights = dst.weights;
    a.route_slot = ws.route_slot + (size_t)(sender / ws.dp_size) * ws.max_tk;
    a.err = ws.err;
    a.y_stride = (uint32_t)(first.y_stride / 16);
    a.y_rows = first.y_rows;
    a.out_stride = (uint32_t)(dst.out_stride / 8);
    a.hidden_dim = given.hidden_dim;
    a.le_magic = ws.le_magic;
    a.sizes = ws.num_experts | ws.topk << 11 | ws.experts_per_rank << 18 | (given.accumulate != 0 ? 1u : 0u) << 29;
    return true;
}

template <typename T, typename U>
static hipError_t launch_typed(const CombArgs &given, const Workspace &ws, uint32_t total_tokens,
                               bool streamed, hipStream_t stream, KernelTiming timing) {
    constexpr int V = vec_elems<T>();
    CombArgs args = given;
    uint32_t ranks_with_tokens = 0;
    args.single_rank = 0;
    for (uint32_t r = 0; r < ws.world; ++r) {
        if (given.dst[r].num_tokens == 0) continue;
        ++ranks_with_tokens;
        args.single_rank = r + 1;
    }
    if (ranks_with_tokens != 1 || total_tokens > kOneRankMaxTokens || streamed) args.single_rank = 0;
    if (args.single_rank != 0) args.single = given.dst[args.single_rank - 1];
    const uint32_t chunks = args.hidden_dim / V;
    const bool two = two_pieces_a_lane(ws.topk, (uint64_t)((chunks + kWave - 1) / kWave) * total_tokens);
    const uint32_t width = two ? 2 * kWave : kWave;
    const uint32_t slabs = (chunks + width - 1) / width;
    const TokenLayers layers = token_layers(total_tokens);
    args.layer_rows = layers.rows;
    const dim3 grid(slabs, layers.rows, layers.layers);
    const bool past_cache =
        args.single_rank == 0 && (streamed || (uint64_t)total_tokens * args.hidden_dim * Elem<U>::kSize >= kStreamedOutput);
    const size_t lds = (uint64_t)slabs * total_tokens <= kAllAtOnce ? 0 : lds_to_bound_waves(ws.topk, past_cache);
    CombineSoleArgs sole;
    if (args.single_rank != 0 && sole_args(given, ws, args.single_rank - 1, sole)) {
#define A2A_LAUNCH_SOLE(GROUP, PIECES)                                                                         \
    hipExtLaunchKernelGGL((combine_sole_kernel<T, U, GROUP, PIECES>), grid, dim3(kWave), 0, stream,            \
                          timing.start, timing.stop, 0, sole)
        if (ws.topk > 4) A2A_LAUNCH_SOLE(8, 1);
        else if (ws.topk > 2) A2A_LAUNCH_SOLE(4, 1);
        else if (ws.topk > 1 && two) A2A_LAUNCH_SOLE(2, 2);
        else if (ws.topk > 1) A2A_LAUNCH_SOLE(2, 1);
        else if (two) A2A_LAUNCH_SOLE(1, 2);
        else A2A_LAUNCH_SOLE(1, 1);
#undef A2A_LAUNCH_SOLE
        return hipGetLastError();
    }
#define A2A_LAUNCH_GATHER(GROUP, PIECES, ONE, OUT, LDS)                                                        \
    hipExtLaunchKernelGGL((combine_gather_kernel<T, U, GROUP, PIECES, ONE, OUT>), grid, dim3(kWave), LDS,      \
                          stream, timing.start, timing.stop, 0, args, ws)
#define A2A_LAUNCH_GATHER_RANKS(GROUP, PIECES)                                                                 \
    do {                                                                                                       \
        if (args.single_rank != 0) A2A_LAUNCH_GATHER(GROUP, PIECES, true, kNonTemporal, 0);                    \
        else if (past_cache) A2A_LAUNCH_GATHER(GROUP, PIECES, false, kSystemNonTemporal, lds);                 \
        else A2A_LAUNCH_GATHER(GROUP, PIECES, false, kNonTemporal, lds);                                       \
    } while (0)
    if (ws.topk > 4) A2A_LAUNCH_GATHER_RANKS(8, 1);
    else if (ws.topk > 2) A2A_LAUNCH_GATHER_RANKS(4, 1);
    else if (ws.topk > 1 && two) A2A_LAUNCH_GATHER_RANKS(2, 2);
    else if (ws.topk > 1) A2A_LAUNCH_GATHER_RANKS(2, 1);
    else if (two) A2A_LAUNCH_GATHER_RANKS(1, 2);
    else A2A_LAUNCH_GATHER_RANKS(1, 1);
#undef A2A_LAUNCH_GATHER_RANKS
#undef A2A_LAUNCH_GATHER
    return hipGetLastError();
}

hipError_t launch_combine_gather(const CombArgs &args, const Workspace &ws, uint32_t in_dtype,
                                 uint32_t out_dtype, uint32_t total_tokens, bool streamed, hipStream_t stream,
                                 KernelTiming timing) {
    if (total_tokens == 0) return hipSuccess;
#define A2A_COMBINE_CASE(IN_TAG, IN_T, OUT_TAG, OUT_T) \
    if (in_dtype == IN_TAG && out_dtype == OUT_TAG)    \
        return launch_typed<IN_T, OUT_T>(args, ws, total_tokens, streamed, stream, timing);
    A2A_COMBINE_CASE(A2A_BF16, Bf16, A2A_BF16, Bf16)
    A2A_COMBINE_CASE(A2A_BF16, Bf16, A2A_F32, F32)
    A2A_COMBINE_CASE(A2A_BF16, Bf16, A2A_F16, F16)
    A2A_COMBINE_CASE(A2A_F16, F16, A2A_F16, F16)
    A2A_COMBINE_CASE(A2A_F16, F16, A2A_F32, F32)
    A2A_COMBINE_CASE(A2A_F16, F16, A2A_BF16, Bf16)
    A2A_COMBINE_CASE(A2A_F32, F32, A2A_F32, F32)
    A2A_COMBINE_CASE(A2A_F32, F32, A2A_BF16, Bf16)
    A2A_COMBINE_CASE(A2A_F32, F32, A2A_F16, F16)
#undef A2A_COMBINE_CASE
    return hipErrorInvalidValue;
}

template <typename T, typename U>
static hipError_t launch_staged_typed(const CombineStagedArgs &given, hipStream_t stream, KernelTiming timing) {
    CombineStagedArgs args = given;
    const uint32_t chunks = args.hidden_dim / vec_elems<T>();
    const bool two = two_pieces_a_lane(args.topk, (uint64_t)((chunks + kWave - 1) / kWave) * args.num_tokens);
    const uint32_t width = two ? 2 * kWave : kWave;
    const uint32_t slabs = (chunks + width - 1) / width;
    const TokenLayers layers = token_layers(args.num_tokens);
    args.layer_rows = layers.rows;
    const dim3 grid(slabs, layers.rows, layers.layers);
    const bool bounded = args.num_tokens > kOneRankMaxTokens && (uint64_t)slabs * args.num_tokens > kAllAtOnce;
    const size_t lds = bounded ? lds_to_bound_waves(args.topk, false) : 0;
#define A2A_LAUNCH_STAGED(GROUP, PIECES)                                                                      \
    hipExtLaunchKernelGGL((combine_staged_kernel<T, U, GROUP, PIECES>), grid, dim3(kWave), lds, stream,       \
                          timing.start, timing.stop, 0, args)
    if (args.topk > 4) A2A_LAUNCH_STAGED(8, 1);
    else if (args.topk > 2) A2A_LAUNCH_STAGED(4, 1);
    else if (args.topk > 1 && two) A2A_LAUNCH_STAGED(2, 2);
    else if (args.topk > 1) A2A_LAUNCH_STAGED(2, 1);
    else if (two) A2A_LAUNCH_STAGED(1, 2);
    else A2A_LAUNCH_STAGED(1, 1);
#undef A2A_LAUNCH_STAGED
    return hipGetLastError();
}

hipError_t launch_combine_staged(const CombineStagedArgs &args, uint32_t in_dtype, uint32_t out_dtype, hipStream_t stream,
                                 KernelTiming timing) {
    if (args.num_tokens == 0) return hipSuccess;
    // (staged rows have elements as wide as those of the output)
#define A2A_STAGED_CASE(IN_TAG, IN_T, OUT_TAG, OUT_T) \
    if (in_dtype == IN_TAG && out_dtype == OUT_TAG) return launch_staged_typed<IN_T, OUT_T>(args, stream, timing);
    A2A_STAGED_CASE(A2A_BF16, Bf16, A2A_BF16, Bf16)
    A2A_STAGED_CASE(A2A_BF16, Bf16, A2A_F16, F16)
    A2A_STAGED_CASE(A2A_F16, F16, A2A_F16, F16)
    A2A_STAGED_CASE(A2A_F16, F16, A2A_BF16, Bf16)
    A2A_STAGED_CASE(A2A_F32, F32, A2A_F32, F32)
#undef A2A_STAGED_CASE
    return hipErrorInvalidValue;
}

}  // namespace a2a
