// Kernels of the split calls; see a2a_staged.h for what they mirror.
#include "a2a_rules.h"
#include "a2a_staged.h"

#include <algorithm>
#include <cstring>

#include "a2a_device.h"
#include "a2a_scan.h"

namespace a2a {

namespace {

size_t align_up_sz(size_t n, size_t a) { return (n + a - 1) / a * a; }

// ---------------------------------------------------------------------------
// dispatch send: stage one (quantised) row per token, record which token sits
// behind every row of the sender's expert-sorted order.
// ---------------------------------------------------------------------------

// Stages the row of `token` (payload, then scales).  Whole workgroup.
// PRE: the thread's first piece of the row was asked for earlier and is passed in.
template <bool QUANT, bool PRE = false>
__device__ __forceinline__ void stage_row(const StageSendArgs &args, const Staging &st, uint32_t g, uint32_t token,
                                          uint32_t staging_threads, u32x4 pre_a = u32x4{0, 0, 0, 0},
                                          u32x4 pre_b = u32x4{0, 0, 0, 0}, uint32_t first_thread = 0) {
    // the row is the work of threads first_thread .. first_thread + staging_threads - 1 of the workgroup
    const uint32_t tid = threadIdx.x - first_thread;
    if (tid >= staging_threads) return;   // (threads below first_thread wrap around to large numbers)
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const PushSrc &src = args.src;
    const uint8_t *x_row = src.x + (size_t)token * src.x_stride;
    uint8_t *row = st.send_buf + ((size_t)g * st.max_tokens + token) * st.disp_stride;
    float *row_scale = reinterpret_cast<float *>(row + st.payload_bytes);

    if constexpr (QUANT) {
        const uint32_t num_chunks = args.hidden_dim / 16;
        for (uint32_t base = wave * kWave; base < num_chunks; base += staging_threads) {
            const uint32_t c = base + lane;
            const bool active = c < num_chunks;
            u32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
            if (PRE && base == wave * kWave) {
                a = pre_a;
                b = pre_b;
            } else if (active) {
                const u32x4 *p = reinterpret_cast<const u32x4 *>(x_row + (size_t)c * 32);
                a = __builtin_nontemporal_load(p);
                b = __builtin_nontemporal_load(p + 1);
            }
            float scale;
            const u32x4 q = quantize16(a, b, &scale);
            if (active) {
                reinterpret_cast<u32x4 *>(row)[c] = q;
                if ((lane & 7) == 0) row_scale[c / 8] = scale;
            }
        }
    } else {
        const uint32_t num_chunks = args.row_bytes / 16;
        for (uint32_t c = tid; c < num_chunks; c += staging_threads) {
            reinterpret_cast<u32x4 *>(row)[c] =
                PRE && c == tid ? pre_a : __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row) + c);
        }
        if (src.x_scale != nullptr) {
            const float *xs = src.x_scale + (size_t)token * src.xs_stride_token;
            for (uint32_t j = tid; j < args.hidden_dim_scale; j += staging_threads) {
                row_scale[j] = xs[(size_t)j * src.xs_stride_elem];
            }
        }
    }
}

template <bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_kernel(const StageSendArgs args, const Workspace ws,
                                                          const Staging st) {
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t E = ws.num_experts;
    const uint32_t K = ws.topk;
    const uint32_t g = args.rank / ws.dp_size;   // ranks of a dp group hold the same tokens
    const uint32_t token = blockIdx.x;
    const PushSrc &src = args.src;
    if (token >= effective_tokens(src.bound_m, src.num_tokens)) return;

    if (wave == 0 && lane < K) {
        const uint32_t entry = token * K + lane;
        const uint32_t expert = (uint32_t)src.indices[(size_t)token * src.indices_stride + lane];
        uint32_t toff = 0, at = kInvalidSlot;
        if (expert < E) {
            toff = ws.block_prefix[((size_t)g * ws.nb_max + entry / kRouteBlock) * E + expert] +
                   ws.local_rank[(size_t)g * ws.max_tk + entry];
            // position of the copy (a2a_dispatch_send.cu:54)
            const uint32_t excl = expert > 0 ? ws.expert_offsets[g * E + expert - 1] : 0;
            at = excl + toff;
            st.pos_token[(size_t)g * ws.max_tk + at] = token;
        }
        ws.token_offset[(size_t)g * ws.max_tk + entry] = toff;
        ws.route_slot[(size_t)g * ws.max_tk + entry] = at;   // (the combine-recv of the step reads the position here)
    }
    stage_row<QUANT>(args, st, g, token, blockDim.x);
}

// The send of a small step in ONE launch (the reference's dispatch-send kernel
// is one launch too, a2a_dispatch_send.cu:158-523): every token workgroup
// counts the entries of the sender per expert and those before its
// own token (LDS atomics; counts do not depend on arrival order), scans the
// counts over the experts, and has the position of each of its K copies in the
// sender's expert-sorted order.  The workgroup of token 0 publishes the counts
// and their scan.  Cost grows with tokens x entries, so the host uses it for
// small steps only.  Dynamic LDS: 3 * E words.
template <bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_small_kernel(const StageSendArgs args, const Workspace ws,
                                                                const Staging st) {
    extern __shared__ uint32_t s_send[];
    __shared__ uint32_t scratch[kRouteWaves];
    __shared__ uint32_t s_carry;
    // everything the head of a workgroup takes from the argument block, asked for in one go
    A2A_PIN(args.src.x);
    A2A_PIN(args.src.indices);
    A2A_PIN(args.src.bound_m);
    A2A_PIN(args.src.x_stride);
    A2A_PIN(args.src.indices_stride);
    A2A_PIN(args.src.num_tokens);
    A2A_PIN(args.rank);
    A2A_PIN(args.hidden_dim);
    A2A_PIN(args.row_bytes);
    A2A_PIN(args.topk_magic);
    A2A_PIN(ws.num_experts);
    A2A_PIN(ws.topk);
    A2A_PIN(ws.dp_size);
    A2A_PIN(ws.max_tk);
    A2A_PIN(ws.num_routed);
    A2A_PIN(ws.expert_offsets);
    A2A_PIN(ws.token_offset);
    A2A_PIN(ws.err);
    A2A_PIN(st.send_buf);
    A2A_PIN(st.pos_token);
    A2A_PIN(st.disp_stride);
    A2A_PIN(st.payload_bytes);
    A2A_PIN(st.max_tokens);
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;   // read once: used after LDS atomics it is fetched again every time
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t E = ws.num_experts;
    const uint32_t K = ws.topk;
    const uint32_t g = args.rank / ws.dp_size;
    const uint32_t token = blockIdx.x;
    const PushSrc &src = args.src;
    const uint32_t eff = effective_tokens(src.bound_m, src.num_tokens);
    const uint32_t entries = eff * K;
    const uint32_t my_first = token * K;
    uint32_t *cnt = s_send;          // [E] entries of the sender per expert
    uint32_t *prior = cnt + E;       // [E] those of the tokens before mine
    uint32_t *excl = prior + E;      // [E] exclusive scan of cnt

    // The first batch of entries is asked for before the tables are cleared and counted in
    // straight-line code, each entry waited for by itself.
    auto load_batch = [&](uint32_t f0, uint32_t (&expert)[8]) {
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t f = f0 + j * nthreads + tid;
            expert[j] = 0xFFFFFFFFu;
            if (f < entries) {
                const uint32_t t = K > 1 ? __umulhi(f, args.topk_magic) : f;
                expert[j] = (uint32_t)src.indices[(size_t)t * src.indices_stride + (f - t * K)];
            }
        }
    };
    auto count_batch = [&](uint32_t f0, const uint32_t (&expert)[8]) {
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t x = expert[j];
            if (x >= E) continue;
            atomicAdd(&cnt[x], 1u);
            if (f0 + j * nthreads + tid < my_first) atomicAdd(&prior[x], 1u);
        }
    };
    uint32_t first_batch[8];
    load_batch(0, first_batch);
    uint32_t my_expert = 0xFFFFFFFFu;
    if (lane < K) my_expert = (uint32_t)src.indices[(size_t)token * src.indices_stride + lane];
    // The row is asked for here, after the entries, and travels while they are counted.  Without a
    // condition (a thread without a piece asks for one it ignores), and every barrier up to its use
    // waits for LDS only: otherwise something on the way would wait for it by accident.
    u32x4 pre_a, pre_b = {0, 0, 0, 0};
    {
        const uint8_t *x_row = src.x + (size_t)token * src.x_stride;
        if constexpr (QUANT) {
            const uint32_t pieces = args.hidden_dim / 16;
            const u32x4 *piece = reinterpret_cast<const u32x4 *>(x_row + (size_t)(tid < pieces ? tid : 0) * 32);
            pre_a = __builtin_nontemporal_load(piece);
            pre_b = __builtin_nontemporal_load(piece + 1);
        } else {
            const uint32_t pieces = args.row_bytes / 16;
            pre_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row) + (tid < pieces ? tid : 0));
        }
    }

    for (uint32_t i = tid; i < 2 * E; i += nthreads) s_send[i] = 0;
    lds_barrier();
    count_batch(0, first_batch);
    for (uint32_t f0 = 8 * nthreads; f0 < entries; f0 += 8 * nthreads) {
        uint32_t expert[8];
        load_batch(f0, expert);
        count_batch(f0, expert);
    }
    lds_barrier();

    // Scan over the experts (a2a_dispatch_send.cu:236-242); token 0 publishes.
    uint32_t carry = 0;
    for (uint32_t e0 = 0; e0 < E; e0 += nthreads) {
        const uint32_t e = e0 + tid;
        const uint32_t c = e < E ? cnt[e] : 0;
        const uint32_t incl = carry + block_inclusive_scan<true>(c, scratch);
        if (e < E) {
            excl[e] = incl - c;
            if (token == 0) {
                ws.num_routed[g * E + e] = c;
                ws.expert_offsets[g * E + e] = incl;
            }
        }
        if (e0 + nthreads < E) {   // uniform: another round follows
            if (tid == nthreads - 1) s_carry = incl;
            lds_barrier();
            carry = s_carry;
        }
    }
    lds_barrier();
    if (token >= eff) return;   // past bound_m: nothing to stage (uniform)

    if (wave == 0) {
        uint32_t repeats = 0;   // copies of this token to the same expert at an earlier k
        for (uint32_t k = 0; k + 1 < K; ++k) {
            const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)my_expert, (int)k);
            if (k < lane && other == my_expert) ++repeats;
        }
        if (lane < K) {
            const uint32_t entry = token * K + lane;
            uint32_t toff = 0, at = kInvalidSlot;
            if (my_expert < E) {
                toff = prior[my_expert] + repeats;
                // position of the copy (a2a_dispatch_send.cu:54)
                at = excl[my_expert] + toff;
                st.pos_token[(size_t)g * ws.max_tk + at] = token;
            } else {
                atomicOr(ws.err, A2A_DEV_BAD_EXPERT_ID);
            }
            ws.token_offset[(size_t)g * ws.max_tk + entry] = toff;
            ws.route_slot[(size_t)g * ws.max_tk + entry] = at;
        }
    }
    stage_row<QUANT, true>(args, st, g, token, nthreads, pre_a, pre_b);
}

// The scan over a sender's per-expert counts (a2a_dispatch_send.cu:236-242) by ONE wavefront, for the
// sends in which a spare wavefront resolves positions.  `s_cnt[e]`: low half of a word the entries of
// expert e.  W passes of 64 experts at a time: their reads, scans and lane exchanges do not depend on
// each other, only the running total `run` does.  A lane whose route's expert `my_id` lies in a pass
// takes the expert's word and the entries of the experts before it from the lane that holds them; with
// `publish` the counts and their inclusive scan go to memory.  Whole wavefront.
template <uint32_t W>
__device__ __forceinline__ void scan_counts_passes(const uint32_t *s_cnt, uint32_t E, uint32_t e0, uint32_t lane,
                                                   uint32_t my_id, bool publish, uint32_t *num_routed,
                                                   uint32_t *expert_offsets, uint32_t &run, uint32_t &my_word,
                                                   uint32_t &my_excl) {
    uint32_t word[W], incl[W];
#pragma unroll
    for (uint32_t u = 0; u < W; ++u) {
        const uint32_t x = e0 + u * kWave + lane;
        word[u] = s_cnt[x < E ? x : 0];
        if (x >= E) word[u] = 0;
    }
#pragma unroll
    for (uint32_t u = 0; u < W; ++u) incl[u] = wave_inclusive_scan(word[u] & 0xFFFFu, lane);
#pragma unroll
    for (uint32_t u = 0; u < W; ++u) {
        const uint32_t x = e0 + u * kWave + lane;
        const uint32_t c = word[u] & 0xFFFFu;
        const uint32_t rel = my_id - (e0 + u * kWave);   // (an id below the pass wraps around to a large number)
        const uint32_t their_word = (uint32_t)__shfl((int)word[u], (int)(rel & (kWave - 1)));   // every lane takes part
        const uint32_t their_excl = (uint32_t)__shfl((int)(incl[u] - c), (int)(rel & (kWave - 1)));
        if (rel < (uint32_t)kWave) {
            my_word = their_word;
            my_excl = run + their_excl;
        }
        if (publish && x < E) {
            num_routed[x] = c;
            expert_offsets[x] = run + incl[u];
        }
        run += (uint32_t)__builtin_amdgcn_readlane((int)incl[u], kWave - 1);
    }
}

// The whole scan: four passes at a time while more than two are left, then two (256 experts: 3.6 ->
// 3.4 us per send of 128 tokens against one pass at a time; a step with 128 experts takes two at a
// time, with four it was 0.1 us slower).
__device__ __forceinline__ void scan_counts_for_routes(const uint32_t *s_cnt, uint32_t E, uint32_t lane, uint32_t my_id,
                                                       bool publish, uint32_t *num_routed, uint32_t *expert_offsets,
                                                       uint32_t &my_word, uint32_t &my_excl) {
    uint32_t run = 0, e0 = 0;
    my_word = my_excl = 0;
    for (; e0 + 2 * kWave < E; e0 += 4 * kWave) {
        scan_counts_passes<4>(s_cnt, E, e0, lane, my_id, publish, num_routed, expert_offsets, run, my_word, my_excl);
    }
    if (e0 < E) scan_counts_passes<2>(s_cnt, E, e0, lane, my_id, publish, num_routed, expert_offsets, run, my_word, my_excl);
}

// The quick form of the one-launch send of a small step: dense index rows and a row that is one piece
// per thread (16 elements to quantise, or 16 bytes to move as they are) with a wavefront to spare (the
// host launches one more than the row has pieces for).  Where a row is staged does not depend on the
// routing (one row per token, at the token's own place), so the wavefronts that move the row count
// their entries, say so (a word in LDS, not a barrier) and then quantise and store without waiting for
// anybody; the spare wavefront (the RESOLVER) does not count: it holds the token's ids, waits until
// every counting wavefront has said that its entries are in the table, scans the table by itself (64
// experts an instruction, no workgroup scan with its barriers), and writes the token's positions; the
// resolver of token 0 publishes the counts and their scan on the way.  In stage_send_small_kernel every
// wavefront walks count, workgroup scan, routes and row one after the other: 128 tokens of 7168,
// 4.1 -> 3.6 us per send at the GPU's own pace; hidden 2048: 3.9 -> 3.2.
// NB: entries a counting thread asks for at the head (the host picks the smallest of 1, 2, 3, 4, 8 that
// covers the step; entries beyond are counted by a loop).  Dynamic LDS: E words (low half of a word:
// the entries of the expert, high half: those of the tokens before this one; a step of this kernel
// has fewer than 2^16 entries).
constexpr uint32_t kSendQuickSpinLimit = 1u << 22;   // (a resolver that gives up flags A2A_DEV_INTERNAL; never seen)

template <uint32_t NB, bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_quick_kernel(const SendQuickArgs args) {
    extern __shared__ uint32_t s_cnt[];
    __shared__ uint32_t s_counted;   // counting wavefronts whose entries are in the table
    // everything the head of a workgroup takes from the argument block, asked for in one go
    A2A_PIN(args.x);
    A2A_PIN(args.x_scale);
    A2A_PIN(args.indices);
    A2A_PIN(args.bound_m);
    A2A_PIN(args.x_stride);
    A2A_PIN(args.staged);
    A2A_PIN(args.pos_token);
    A2A_PIN(args.num_routed);
    A2A_PIN(args.token_offset);
    A2A_PIN(args.route_slot);
    A2A_PIN(args.num_tokens);
    A2A_PIN(args.num_scales);
    A2A_PIN(args.sizes);
    A2A_PIN(args.distances);
    const uint32_t tid = threadIdx.x;
    const uint32_t num_chunks = args.pieces();   // pieces of a row, one per thread
    const uint32_t counters = (num_chunks + kWave - 1) / kWave * kWave;   // threads that count entries and move the row
    const uint32_t nthreads = counters + kWave;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t waves = nthreads / kWave;
    const bool resolver = wave == waves - 1;
    const uint32_t E = args.num_experts();
    const uint32_t K = args.topk();
    const uint32_t token = blockIdx.x;
    const uint32_t tokens = args.num_tokens;  // the grid: one workgroup per token
    const uint32_t entries = tokens * K;      // > 0
    const uint32_t my_first = token * K;
    const bool has_piece = tid < num_chunks;

    // What each kind of wavefront takes from memory, asked for before anything else is done: the
    // entries, then the thread's piece of the row (and the first of the caller's scales it copies);
    // the resolver its token's ids (lane k: route k).
    uint32_t early[NB] = {};
    u32x4 pre_a = {0, 0, 0, 0}, pre_b = {0, 0, 0, 0};
    float first_scale = 0.0f;
    uint32_t my_id = 0xFFFFFFFFu;
    if (!resolver) {
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
            const uint32_t f = j * counters + tid;
            early[j] = (uint32_t)args.indices[f < entries ? f : entries - 1];
        }
        const uint8_t *x_row = args.x + (size_t)token * args.x_stride;
        if (has_piece) {
            if constexpr (QUANT) {
                const u32x4 *piece = reinterpret_cast<const u32x4 *>(x_row + (size_t)tid * 32);
                pre_a = __builtin_nontemporal_load(piece);
                pre_b = __builtin_nontemporal_load(piece + 1);
            } else {
                pre_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row) + tid);
            }
        }
        if constexpr (!QUANT) {
            if (args.x_scale != nullptr && tid < args.num_scales) {
                first_scale = args.x_scale[(size_t)token * args.xs_stride_token + (size_t)tid * args.xs_stride_elem];
            }
        }
    } else {
        // (the resolver shares its SIMD with wavefronts that quantise while the positions are resolved)
        __builtin_amdgcn_s_setprio(3);
        my_id = (uint32_t)args.indices[my_first + (lane < K ? lane : 0)];
    }
    const uint32_t eff = effective_tokens(args.bound_m, tokens);
    const uint32_t flat_entries = eff * K;
    const bool live = token < eff;   // uniform

    for (uint32_t i = tid; i < E; i += nthreads) s_cnt[i] = 0;
    if (tid == 0) s_counted = 0;
    lds_barrier();

    if (!resolver) {
        // The first batch in straight-line code: each of its values is waited for by itself, and the
        // row asked for after them stays in flight meanwhile.
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
            const uint32_t f = j * counters + tid;
            const uint32_t x = f < flat_entries ? early[j] : 0xFFFFFFFFu;
            if (x < E) atomicAdd(&s_cnt[x], f < my_first ? 0x10001u : 1u);
        }
        for (uint32_t f0 = NB * counters; f0 < flat_entries; f0 += NB * counters) {
            uint32_t x[NB];
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                const uint32_t f = f0 + j * counters + tid;
                x[j] = f < flat_entries ? (uint32_t)args.indices[f] : 0xFFFFFFFFu;
            }
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                const uint32_t f = f0 + j * counters + tid;
                if (x[j] < E) atomicAdd(&s_cnt[x[j]], f < my_first ? 0x10001u : 1u);
            }
        }
        // this wavefront's entries are in the table before its arrival is counted
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) atomicAdd(&s_counted, 1u);
        if (!live) return;   // past bound_m: nothing to stage (uniform)

        uint8_t *row = args.staged + (size_t)token * staged_row_stride(num_chunks * 16, args.num_scales);
        float *row_scale = reinterpret_cast<float *>(row + num_chunks * 16);
        if constexpr (QUANT) {
            float scale;
            const u32x4 q = quantize16(pre_a, pre_b, &scale);
            if (has_piece) {
                reinterpret_cast<u32x4 *>(row)[tid] = q;
                if ((lane & 7) == 0) row_scale[tid / 8] = scale;
            }
        } else {
            if (has_piece) reinterpret_cast<u32x4 *>(row)[tid] = pre_a;
            if (args.x_scale != nullptr) {
                if (tid < args.num_scales) row_scale[tid] = first_scale;
                const float *xs = args.x_scale + (size_t)token * args.xs_stride_token;
                for (uint32_t j = tid + counters; j < args.num_scales; j += counters) {
                    row_scale[j] = xs[(size_t)j * args.xs_stride_elem];
                }
            }
        }
        return;
    }

    // ---- the resolver ----
    // copies of this token to the same expert at an earlier k: what no count decides
    uint32_t repeats = 0;
    for (uint32_t k = 0; k + 1 < K; ++k) {
        const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)my_id, (int)k);
        if (k < lane && other == my_id) ++repeats;
    }
    // until the counting wavefronts have all said that their entries are in the table (at the lowest
    // priority: the wavefronts that share this SIMD are among those waited for)
    __builtin_amdgcn_s_setprio(0);
    for (uint32_t spins = 0; __hip_atomic_load(&s_counted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != waves - 1;) {
        if (++spins == kSendQuickSpinLimit) {
            if (lane == 0) atomicOr(args.flags(), A2A_DEV_INTERNAL);
            break;
        }
    }
    __builtin_amdgcn_s_setprio(3);
    asm volatile("" ::: "memory");

    // Scan over the experts; a route takes its expert's word and the entries of the experts before it.
    // Token 0 publishes.
    uint32_t my_word, my_excl;
    scan_counts_for_routes(s_cnt, E, lane, my_id, token == 0, args.num_routed, args.expert_offsets(), my_word, my_excl);
    if (!live) return;   // past bound_m: no positions to write (uniform)
    if (lane < K) {
        uint32_t toff = 0, at = kInvalidSlot;
        if (my_id < E) {
            toff = (my_word >> 16) + repeats;
            // position of the copy (a2a_dispatch_send.cu:54)
            at = my_excl + toff;
            args.pos_token[at] = token;
        } else {
            atomicOr(args.flags(), A2A_DEV_BAD_EXPERT_ID);
        }
        args.token_offset[my_first + lane] = toff;
        args.route_slot[my_first + lane] = at;
    }
}

// The send of a step too large for stage_send_small_kernel and of at most kSendSingleMaxEntries
// entries (448 to 1024 tokens at top-8), in ONE launch: what makes the small kernel expensive as steps
// grow is that every token's workgroup counts every entry of the sender; here a workgroup counts once
// for `per_group` tokens (the host picks it so that the workgroups are about as many as the compute
// units) and stages them with teams of wavefronts, one token per team and round.  One LDS word per
// expert holds its entries (low half) and those of the tokens before the workgroup's first (high half).
// The rows of the first two rounds are asked for at the head and travel while the entries are counted
// (every barrier up to their use waits for LDS only).  Dynamic LDS: 2 * E words.
constexpr uint32_t kSendSingleMaxEntries = 8192;
constexpr uint32_t kSendTokensPerGroup = 4;

template <bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_single_kernel(const StageSendArgs args, const Workspace ws,
                                                                 const Staging st, const uint32_t team_threads,
                                                                 const uint32_t per_group) {
    extern __shared__ uint32_t s_single[];
    __shared__ uint32_t s_route_expert[kSendTokensPerGroup * A2A_MAX_EXPERTS_PER_TOKEN];
    __shared__ uint32_t scratch[kRouteWaves];
    __shared__ uint32_t s_carry;
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    const uint32_t E = ws.num_experts, K = ws.topk;
    const uint32_t g = args.rank / ws.dp_size;
    const PushSrc &src = args.src;                     // index rows are dense (the host checks)
    const uint32_t tokens = effective_tokens(src.bound_m, src.num_tokens);
    const uint32_t flat_entries = tokens * K;
    const uint32_t first_token = blockIdx.x * per_group;
    const uint32_t my_first = first_token * K;         // flat index of my first entry
    if (blockIdx.x != 0 && first_token >= tokens) return;   // nothing to stage; the first workgroup publishes

    constexpr uint32_t kBatch = 10;   // 8192 entries over 896 threads in one batch
    uint32_t early[kBatch];
#pragma unroll
    for (uint32_t j = 0; j < kBatch; ++j) {
        const uint32_t f = j * nthreads + tid;
        early[j] = f < flat_entries ? (uint32_t)src.indices[f] : 0xFFFFFFFFu;
    }
    const uint32_t my_routes = per_group * K;          // one thread each
    uint32_t my_expert = 0xFFFFFFFFu;
    if (tid < my_routes && my_first + tid < flat_entries) my_expert = (uint32_t)src.indices[my_first + tid];
    const uint32_t teams = nthreads / team_threads;
    const uint32_t team = tid / team_threads;
    const uint32_t team_tid = tid - team * team_threads;
    u32x4 pre_a, pre_b = {0, 0, 0, 0};
    u32x4 next_a = {0, 0, 0, 0}, next_b = {0, 0, 0, 0};
    {
        const uint32_t last_token = src.num_tokens - 1;
        const uint32_t any_token = first_token + team < src.num_tokens ? first_token + team : last_token;
        const uint32_t second = first_token + teams + team;
        const uint8_t *x_row = src.x + (size_t)any_token * src.x_stride;
        const uint8_t *x_next = src.x + (size_t)(second < src.num_tokens ? second : last_token) * src.x_stride;
        const bool two_rounds = per_group > teams;     // uniform: a branch, not a select
        if constexpr (QUANT) {
            const uint32_t pieces = args.hidden_dim / 16;
            const size_t at = (size_t)(team_tid < pieces ? team_tid : 0) * 32;
            if (two_rounds) {
                next_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_next + at));
                next_b = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_next + at) + 1);
            }
            pre_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row + at));
            pre_b = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row + at) + 1);
        } else {
            const uint32_t pieces = args.row_bytes / 16;
            const uint32_t at = team_tid < pieces ? team_tid : 0;
            if (two_rounds) next_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_next) + at);
            pre_a = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row) + at);
        }
    }

    uint32_t *cnt = s_single;      // [E] low half: entries per expert, high half: those before my first token
    uint32_t *excl = cnt + E;      // [E] exclusive scan of the entries per expert
    for (uint32_t i = tid; i < E; i += nthreads) cnt[i] = 0;
    lds_barrier();
    auto count_batch = [&](const uint32_t (&expert)[kBatch], uint32_t f0) {
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t x = expert[j];
            if (x >= E) continue;
            atomicAdd(&cnt[x], f0 + j * nthreads + tid < my_first ? 0x10001u : 1u);
        }
    };
    count_batch(early, 0);
    for (uint32_t f0 = kBatch * nthreads; f0 < flat_entries; f0 += kBatch * nthreads) {
        uint32_t expert[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t f = f0 + j * nthreads + tid;
            expert[j] = f < flat_entries ? (uint32_t)src.indices[f] : 0xFFFFFFFFu;
        }
        count_batch(expert, f0);
    }
    if (tid < my_routes) s_route_expert[tid] = my_expert;
    lds_barrier();

    // Scan over the experts (a2a_dispatch_send.cu:236-242); the first workgroup publishes.
    uint32_t carry = 0;
    for (uint32_t e0 = 0; e0 < E; e0 += nthreads) {
        const uint32_t e = e0 + tid;
        const uint32_t c = e < E ? cnt[e] & 0xFFFFu : 0;
        const uint32_t incl = carry + block_inclusive_scan<true>(c, scratch);
        if (e < E) {
            excl[e] = incl - c;
            if (blockIdx.x == 0) {
                ws.num_routed[g * E + e] = c;
                ws.expert_offsets[g * E + e] = incl;
            }
        }
        if (e0 + nthreads < E) {   // uniform: another round follows
            if (tid == nthreads - 1) s_carry = incl;
            lds_barrier();
            carry = s_carry;
        }
    }
    lds_barrier();

    // One thread per route of my tokens: its rank inside its expert and the row of the sender's
    // expert-sorted order it stands for (a2a_dispatch_send.cu:54).
    if (tid < my_routes && my_first + tid < flat_entries) {
        uint32_t toff = 0, at = kInvalidSlot;
        if (my_expert < E) {
            uint32_t earlier = 0;
            for (uint32_t q = 0; q < tid; ++q) earlier += s_route_expert[q] == my_expert ? 1u : 0u;
            toff = (cnt[my_expert] >> 16) + earlier;
            at = excl[my_expert] + toff;
            st.pos_token[(size_t)g * ws.max_tk + at] = first_token + tid / K;
        } else {
            atomicOr(ws.err, A2A_DEV_BAD_EXPERT_ID);
        }
        ws.token_offset[(size_t)g * ws.max_tk + my_first + tid] = toff;
        ws.route_slot[(size_t)g * ws.max_tk + my_first + tid] = at;
    }

    // The teams stage one token each per round.
    for (uint32_t first = 0; first < per_group; first += teams) {
        const uint32_t token = first_token + first + team;
        if (first + team >= per_group || token >= tokens) continue;   // (no barrier below: teams work alone)
        if (first == 0) {
            stage_row<QUANT, true>(args, st, g, token, team_threads, pre_a, pre_b, team * team_threads);
        } else if (first == teams) {
            stage_row<QUANT, true>(args, st, g, token, team_threads, next_a, next_b, team * team_threads);
        } else {
            stage_row<QUANT>(args, st, g, token, team_threads, u32x4{0, 0, 0, 0}, u32x4{0, 0, 0, 0}, team * team_threads);
        }
    }
}

// stage_send_single_kernel with the division of labour of stage_send_quick_kernel, for steps whose
// rows are one piece per thread of a team and leave room for a spare wavefront: the teams count the
// step's entries, say so, and quantise and stage their tokens' rows (at most two rounds, both rounds'
// pieces asked for at the head) without waiting for anybody; the spare wavefront holds the routes of
// the workgroup's tokens (a lane each, at most 64), counts for each the earlier routes of the workgroup
// to the same expert, waits for the counting wavefronts, scans the counts by itself and writes the
// positions.  1024 tokens of 7168: 8.5 -> 7.0 us per send at the GPU's own pace.
// NB: entries a counting thread asks for at the head.  Dynamic LDS: E words.
template <uint32_t NB, uint32_t ROUNDS, bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_teams_kernel(const StageSendArgs args, const Workspace ws,
                                                                const Staging st, const uint32_t team_threads,
                                                                const uint32_t per_group) {
    extern __shared__ uint32_t s_cnt[];
    __shared__ uint32_t s_counted;   // counting wavefronts whose entries are in the table
    // everything the head of a workgroup takes from the argument block, asked for in one go
    A2A_PIN(args.src.x);
    A2A_PIN(args.src.x_scale);
    A2A_PIN(args.src.indices);
    A2A_PIN(args.src.bound_m);
    A2A_PIN(args.src.x_stride);
    A2A_PIN(args.src.num_tokens);
    A2A_PIN(args.rank);
    A2A_PIN(args.hidden_dim);
    A2A_PIN(args.row_bytes);
    A2A_PIN(args.topk_magic);
    A2A_PIN(ws.num_experts);
    A2A_PIN(ws.topk);
    A2A_PIN(ws.dp_size);
    A2A_PIN(ws.max_tk);
    A2A_PIN(ws.num_routed);
    A2A_PIN(ws.expert_offsets);
    A2A_PIN(ws.token_offset);
    A2A_PIN(ws.err);
    A2A_PIN(st.send_buf);
    A2A_PIN(st.pos_token);
    A2A_PIN(st.disp_stride);
    A2A_PIN(st.payload_bytes);
    A2A_PIN(st.max_tokens);
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t waves = nthreads / kWave;
    const bool resolver = wave == waves - 1;
    const uint32_t counters = nthreads - kWave;   // threads that count entries and move rows
    const uint32_t E = ws.num_experts;
    const uint32_t K = ws.topk;
    const uint32_t g = args.rank / ws.dp_size;
    const PushSrc &src = args.src;              // index rows are dense (the host checks)
    const uint32_t tokens = src.num_tokens;     // the grid: a workgroup per `per_group` tokens
    const uint32_t entries = tokens * K;        // > 0
    const uint32_t first_token = blockIdx.x * per_group;
    const uint32_t my_first = first_token * K;  // flat index of the workgroup's first entry
    const uint32_t routes = per_group * K;      // <= 64 (the host checks)
    const uint32_t num_chunks = QUANT ? args.hidden_dim / 16 : args.row_bytes / 16;   // pieces of a row, one per thread of a team
    const uint32_t teams = counters / team_threads;
    const uint32_t team = tid / team_threads;
    const uint32_t member = tid - team * team_threads;
    const bool has_piece = member < num_chunks;

    uint32_t early[NB] = {};
    u32x4 pre_a[ROUNDS], pre_b[ROUNDS];
    float first_scale[ROUNDS];
    uint32_t my_id = 0xFFFFFFFFu;
    if (!resolver) {
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
            const uint32_t f = j * counters + tid;
            early[j] = (uint32_t)src.indices[f < entries ? f : entries - 1];
        }
#pragma unroll
        for (uint32_t round = 0; round < ROUNDS; ++round) {
            const uint32_t token = first_token + round * teams + team;
            const uint8_t *x_row = src.x + (size_t)(token < tokens ? token : tokens - 1) * src.x_stride;
            pre_a[round] = pre_b[round] = u32x4{0, 0, 0, 0};
            first_scale[round] = 0.0f;
            if (has_piece) {
                if constexpr (QUANT) {
                    const u32x4 *piece = reinterpret_cast<const u32x4 *>(x_row + (size_t)member * 32);
                    pre_a[round] = __builtin_nontemporal_load(piece);
                    pre_b[round] = __builtin_nontemporal_load(piece + 1);
                } else {
                    pre_a[round] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x_row) + member);
                }
            }
            if constexpr (!QUANT) {
                if (src.x_scale != nullptr && member < args.hidden_dim_scale) {
                    first_scale[round] = src.x_scale[(size_t)(token < tokens ? token : tokens - 1) * src.xs_stride_token +
                                                     (size_t)member * src.xs_stride_elem];
                }
            }
        }
    } else {
        // (the resolver shares its SIMD with wavefronts that quantise while the positions are resolved)
        __builtin_amdgcn_s_setprio(3);
        const uint32_t f = my_first + lane;
        my_id = (uint32_t)src.indices[f < entries ? f : entries - 1];
    }
    const uint32_t eff = effective_tokens(src.bound_m, tokens);
    const uint32_t flat_entries = eff * K;
    if (blockIdx.x != 0 && first_token >= eff) return;   // nothing to stage (uniform); the first workgroup publishes

    for (uint32_t i = tid; i < E; i += nthreads) s_cnt[i] = 0;
    if (tid == 0) s_counted = 0;
    lds_barrier();

    if (!resolver) {
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
            const uint32_t f = j * counters + tid;
            const uint32_t x = f < flat_entries ? early[j] : 0xFFFFFFFFu;
            if (x < E) atomicAdd(&s_cnt[x], f < my_first ? 0x10001u : 1u);
        }
        for (uint32_t f0 = NB * counters; f0 < flat_entries; f0 += NB * counters) {
            uint32_t x[NB];
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                const uint32_t f = f0 + j * counters + tid;
                x[j] = f < flat_entries ? (uint32_t)src.indices[f] : 0xFFFFFFFFu;
            }
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                const uint32_t f = f0 + j * counters + tid;
                if (x[j] < E) atomicAdd(&s_cnt[x[j]], f < my_first ? 0x10001u : 1u);
            }
        }
        // this wavefront's entries are in the table before its arrival is counted
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) atomicAdd(&s_counted, 1u);

#pragma unroll
        for (uint32_t round = 0; round < ROUNDS; ++round) {
            const uint32_t token = first_token + round * teams + team;
            if (round * teams + team >= per_group || token >= eff) continue;   // (no barrier below: teams work alone)
            uint8_t *row = st.send_buf + ((size_t)g * st.max_tokens + token) * st.disp_stride;
            float *row_scale = reinterpret_cast<float *>(row + st.payload_bytes);
            if constexpr (QUANT) {
                float scale;
                const u32x4 q = quantize16(pre_a[round], pre_b[round], &scale);
                if (has_piece) {
                    reinterpret_cast<u32x4 *>(row)[member] = q;
                    if ((lane & 7) == 0) row_scale[member / 8] = scale;
                }
            } else {
                if (has_piece) reinterpret_cast<u32x4 *>(row)[member] = pre_a[round];
                if (src.x_scale != nullptr) {
                    if (member < args.hidden_dim_scale) row_scale[member] = first_scale[round];
                    const float *xs = src.x_scale + (size_t)token * src.xs_stride_token;
                    for (uint32_t j = member + team_threads; j < args.hidden_dim_scale; j += team_threads) {
                        row_scale[j] = xs[(size_t)j * src.xs_stride_elem];
                    }
                }
            }
        }
        return;
    }

    // ---- the resolver: lane l holds route l of the workgroup's tokens ----
    const bool route_live = lane < routes && my_first + lane < flat_entries;
    if (!route_live) my_id = 0xFFFFFFFFu;
    // routes of the workgroup before this one (earlier tokens, earlier k) to the same expert: what no count decides
    uint32_t earlier = 0;
    for (uint32_t l = 0; l + 1 < routes; ++l) {
        const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)my_id, (int)l);
        if (l < lane && other == my_id) ++earlier;
    }
    // until the counting wavefronts have all said that their entries are in the table (at the lowest
    // priority: the wavefronts that share this SIMD are among those waited for)
    __builtin_amdgcn_s_setprio(0);
    for (uint32_t spins = 0; __hip_atomic_load(&s_counted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != waves - 1;) {
        if (++spins == kSendQuickSpinLimit) {
            if (lane == 0) atomicOr(ws.err, A2A_DEV_INTERNAL);
            break;
        }
    }
    __builtin_amdgcn_s_setprio(3);
    asm volatile("" ::: "memory");

    // Scan over the experts; a route takes its expert's word and the entries of the experts before it.
    // The first workgroup publishes.
    uint32_t my_word, my_excl;
    scan_counts_for_routes(s_cnt, E, lane, my_id, blockIdx.x == 0, ws.num_routed + g * E, ws.expert_offsets + g * E,
                           my_word, my_excl);

    if (route_live) {
        uint32_t toff = 0, at = kInvalidSlot;
        if (my_id < E) {
            toff = (my_word >> 16) + earlier;
            // position of the copy (a2a_dispatch_send.cu:54)
            const uint32_t token = first_token + (K > 1 ? __umulhi(lane, args.topk_magic) : lane);
            at = my_excl + toff;
            st.pos_token[(size_t)g * ws.max_tk + at] = token;
        } else {
            atomicOr(ws.err, A2A_DEV_BAD_EXPERT_ID);
        }
        ws.token_offset[(size_t)g * ws.max_tk + my_first + lane] = toff;
        ws.route_slot[(size_t)g * ws.max_tk + my_first + lane] = at;
    }
}

// The send of a larger step (up to kSendBesideMaxEntries entries) in ONE launch: where a row is staged does not depend on
// the routing, so the routing runs beside the rows, in workgroups of its own at the head of the grid.  Such a workgroup
// has a chunk of as many entries as it has threads.  It counts ALL entries of the sender per expert, with those in front
// of its chunk in the high half of the word, ranks its own entries among equal ones with ballots (and a scan over the
// wavefronts), scans the counts over the experts, and then has the position of each of its entries without having
// waited for anybody.  The counting is redundant, but it runs on compute units that the rows, which are bound by memory,
// do not fill.  All other workgroups stage rows, a team of wavefronts per token, and nothing else.
//
// us per send at the GPU's own pace, two launches (routing, then rows that resolve their own positions) / this one:
//   fp8 rows of 7168 bytes, K = 8, 1100 tokens   11.5 /  7.3     2048   15.9 / 10.2     4096   20.8 / 14.7     8000   32.7 / 24.5
//   quantised rows, 2048 tokens                  18.4 / 11.8     4096   26.0 / 19.7
//   bf16 rows of 14 KB, 2048 tokens              22.4 / 14.4     of 8 KB, K = 4, 4000 tokens   24.8 / 14.5
//   rows of 2048 bytes, 512 experts, 2000 tokens 10.6 /  7.4     of 1024 bytes, 3000 tokens     9.0 /  7.7
// (Whole steps of 8 x 2048 tokens through the split calls: 1431 -> 1385.)
//
// Dynamic LDS: 2 * E words and, per wavefront, E half words.
constexpr uint32_t kSendBesideMaxEntries = 65535;   // (the halves of a word)
constexpr uint32_t kSendBesideAhead = 8;            // entries a thread has on their way while it counts as many

template <bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_beside_kernel(const StageSendArgs args, const Workspace ws,
                                                                 const Staging st, const uint32_t team_threads,
                                                                 const uint32_t chunks) {
    extern __shared__ uint32_t s_beside[];
    __shared__ uint32_t scratch[kRouteWaves];
    __shared__ uint32_t s_carry;
    A2A_PIN(args.src.x);
    A2A_PIN(args.src.x_scale);
    A2A_PIN(args.src.indices);
    A2A_PIN(args.src.bound_m);
    A2A_PIN(args.src.x_stride);
    A2A_PIN(args.src.num_tokens);
    A2A_PIN(args.rank);
    A2A_PIN(args.hidden_dim);
    A2A_PIN(args.row_bytes);
    A2A_PIN(args.topk_magic);
    A2A_PIN(ws.num_experts);
    A2A_PIN(ws.topk);
    A2A_PIN(ws.dp_size);
    A2A_PIN(ws.max_tk);
    A2A_PIN(ws.token_offset);
    A2A_PIN(ws.err);
    A2A_PIN(st.send_buf);
    A2A_PIN(st.pos_token);
    A2A_PIN(st.disp_stride);
    A2A_PIN(st.payload_bytes);
    A2A_PIN(st.max_tokens);
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    const uint32_t K = ws.topk;
    const uint32_t g = args.rank / ws.dp_size;
    const PushSrc &src = args.src;
    if (blockIdx.x >= chunks) {
        // ---- rows
        const uint32_t teams = nthreads / team_threads, team = tid / team_threads;
        const uint32_t token = (blockIdx.x - chunks) * teams + team;
        if (token >= effective_tokens(src.bound_m, src.num_tokens)) return;   // (no barrier below)
        stage_row<QUANT>(args, st, g, token, team_threads, u32x4{0, 0, 0, 0}, u32x4{0, 0, 0, 0}, team * team_threads);
        return;
    }

    // ---- positions
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t waves = nthreads / kWave;
    const uint32_t E = ws.num_experts;
    uint32_t *const cnt = s_beside;                                     // [E]
    uint32_t *const excl = cnt + E;                                     // [E] entries of the experts before e
    uint16_t *const hist = reinterpret_cast<uint16_t *>(excl + E);      // [waves][E] entries of my chunk
    const uint32_t entries = src.num_tokens * K;                        // > 0
    auto id_of = [&](uint32_t f) { return (uint32_t)src.indices[f < entries ? f : entries - 1]; };   // (dense rows)
    const uint32_t chunk_first = blockIdx.x * nthreads;
    const uint32_t entry = chunk_first + tid;
    const uint32_t my_id = id_of(entry);
    constexpr uint32_t NB = kSendBesideAhead;
    uint32_t now[NB];
#pragma unroll
    for (uint32_t j = 0; j < NB; ++j) now[j] = id_of(j * nthreads + tid);
    const uint32_t live_entries = effective_tokens(src.bound_m, src.num_tokens) * K;
    if (blockIdx.x != 0 && chunk_first >= live_entries) return;   // uniform (the first workgroup publishes)
    for (uint32_t i = tid; i < E; i += nthreads) cnt[i] = 0;
    for (uint32_t i = tid; i < waves * E; i += nthreads) hist[i] = 0;
    lds_barrier();

    // my chunk: lanes of this wavefront that hold the same expert id, matched bit by bit
    const bool in = entry < live_entries;
    const bool valid = in && my_id < E;
    uint64_t peers = __ballot(valid);
    const uint32_t nbits = 32 - __clz((int)(E - 1) | 1);
    for (uint32_t b = 0; b < nbits; ++b) {
        const bool bit = (my_id >> b) & 1;
        const uint64_t set = __ballot(valid && bit);
        peers &= bit ? set : ~set;
    }
    const uint32_t rank_in_wave = __popcll(peers & ((1ull << lane) - 1));
    if (valid && rank_in_wave == 0) hist[wave * E + my_id] = (uint16_t)__popcll(peers);

    // all entries, the next ones on their way while these are counted
    for (uint32_t f0 = 0;;) {
        const uint32_t next = f0 + NB * nthreads;
        uint32_t then[NB];
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) then[j] = id_of(next + j * nthreads + tid);
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
            const uint32_t f = f0 + j * nthreads + tid;
            if (f < live_entries && now[j] < E) atomicAdd(&cnt[now[j]], f < chunk_first ? 0x10001u : 1u);
        }
        if (next >= live_entries) break;
        f0 = next;
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) now[j] = then[j];
    }
    lds_barrier();

    // per expert: my wavefronts' entries in order, and the scan over the experts (a2a_dispatch_send.cu:236-242)
    uint32_t carry = 0;
    for (uint32_t e0 = 0; e0 < E; e0 += nthreads) {
        const uint32_t e = e0 + tid;
        uint32_t run = 0;
        if (e < E) {
            for (uint32_t w = 0; w < waves; ++w) {
                const uint32_t c = hist[w * E + e];
                hist[w * E + e] = (uint16_t)run;
                run += c;
            }
        }
        const uint32_t c = e < E ? cnt[e] & 0xFFFFu : 0;
        const uint32_t incl = carry + block_inclusive_scan<true>(c, scratch);
        if (e < E) {
            excl[e] = incl - c;
            if (blockIdx.x == 0) {
                ws.num_routed[g * E + e] = c;
                ws.expert_offsets[g * E + e] = incl;
            }
        }
        if (e0 + nthreads < E) {   // uniform: another round follows
            if (tid == nthreads - 1) s_carry = incl;
            lds_barrier();
            carry = s_carry;
        }
    }
    lds_barrier();
    if (!in) return;
    uint32_t toff = 0, at = kInvalidSlot;
    if (valid) {
        toff = (cnt[my_id] >> 16) + hist[wave * E + my_id] + rank_in_wave;
        // position of the copy (a2a_dispatch_send.cu:54)
        at = excl[my_id] + toff;
        st.pos_token[(size_t)g * ws.max_tk + at] = K > 1 ? __umulhi(entry, args.topk_magic) : entry;
    } else {
        atomicOr(ws.err, A2A_DEV_BAD_EXPERT_ID);
    }
    ws.token_offset[(size_t)g * ws.max_tk + entry] = toff;
    ws.route_slot[(size_t)g * ws.max_tk + entry] = at;
}

// The send of a large step, after a routing launch that left the chunk counts,
// the in-chunk rank of every entry and the sender's totals per expert and per
// owning rank.  No launch in between scans anything: wavefront 0 of a token
// workgroup finds the position of each of its K copies in the sender's
// expert-sorted order itself, eight lanes per route, from three short sums
// (copies of the same expert in earlier chunks; copies for the ranks before
// the expert's owner; copies for the owner's experts before it), while the
// other wavefronts stage the row.  Workgroup 0 is not a token: it publishes the
// sender's counts and their scan (a2a_dispatch_send.cu:199-204,236-242) and
// hands the totals over to the next send.
template <bool QUANT>
__global__ __launch_bounds__(1024) void stage_send_resolve_kernel(const StageSendArgs args, const Workspace ws,
                                                                  const Staging st) {
    __shared__ uint32_t scratch[kRouteWaves];
    __shared__ uint32_t s_carry;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t E = ws.num_experts, K = ws.topk, Le = ws.experts_per_rank;
    const uint32_t g = args.rank / ws.dp_size;
    const uint32_t use = ws.send_turn[1] & 1u;
    const uint32_t *per_expert = ws.send_totals + (size_t)use * (E + ws.world);   // [E]
    const uint32_t *per_rank = per_expert + E;                                     // [N]

    if (blockIdx.x == 0) {
        uint32_t carry = 0;
        for (uint32_t e0 = 0; e0 < E; e0 += blockDim.x) {
            const uint32_t e = e0 + tid;
            const uint32_t c = e < E ? per_expert[e] : 0;
            const uint32_t incl = carry + block_inclusive_scan(c, scratch);
            if (e < E) {
                ws.num_routed[g * E + e] = c;
                ws.expert_offsets[g * E + e] = incl;
            }
            if (e0 + blockDim.x < E) {   // uniform: another round follows
                if (tid == blockDim.x - 1) s_carry = incl;
                __syncthreads();
                carry = s_carry;
            }
        }
        if (tid == 0) ws.send_turn[0] = use ^ 1u;
        return;
    }

    const uint32_t token = blockIdx.x - 1;
    const PushSrc &src = args.src;
    if (token >= effective_tokens(src.bound_m, src.num_tokens)) return;

    // With a wavefront to spare the last one resolves and stages nothing, so that no wavefront
    // has both chains of memory trips to walk; otherwise wavefront 0 does both.
    const uint32_t staging_threads = args.resolver_wave != 0 ? args.resolver_wave * kWave : blockDim.x;
    if (wave == args.resolver_wave) {
        const uint32_t *counts = ws.chunk_counts + (size_t)g * E * ws.nb_max;   // [E][nb_max]
        const uint32_t part = lane & 7, route = lane >> 3;
        for (uint32_t k0 = 0; k0 < K; k0 += 8) {
            const uint32_t k = k0 + route;
            const bool in = k < K;
            const uint32_t kk = in ? k : 0;   // a lane without a route reads route 0 and is dropped below
            const uint32_t id = (uint32_t)src.indices[(size_t)token * src.indices_stride + kk];
            const uint32_t local = ws.local_rank[(size_t)g * ws.max_tk + token * K + kk];
            const bool live = in && id < E;
            const uint32_t e = live ? id : 0;
            const uint32_t upto = live ? (token * K + k) / kRouteBlock : 0;   // chunk of this entry
            const uint32_t r = owner_of_expert(ws, e);
            const uint32_t le = live ? e - r * Le : 0;
            const uint32_t ranks_before = live ? r : 0;
            // four terms of each sum per lane without a branch (clamped index, masked value)
            uint32_t v_chunk[4], v_rank[4], v_expert[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t n = part + 8 * i;
                v_chunk[i] = counts[(size_t)e * ws.nb_max + (n < upto ? n : 0)];
                v_rank[i] = per_rank[n < ranks_before ? n : 0];
                v_expert[i] = per_expert[r * Le + (n < le ? n : 0)];
            }
            uint32_t earlier = 0, excl = 0;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t n = part + 8 * i;
                earlier += n < upto ? v_chunk[i] : 0;
                excl += n < ranks_before ? v_rank[i] : 0;
                excl += n < le ? v_expert[i] : 0;
            }
            // longer sums (more than 32 chunks, more than 32 experts in a rank)
            for (uint32_t c = 32 + part; c < upto; c += 8) earlier += counts[(size_t)e * ws.nb_max + c];
            for (uint32_t q = 32 + part; q < le; q += 8) excl += per_expert[r * Le + q];
            earlier = group8_sum(earlier);
            excl = group8_sum(excl);
            if (part == 0 && in) {
                uint32_t toff = 0, at = kInvalidSlot;
                if (live) {
                    toff = earlier + local;
                    // position of the copy (a2a_dispatch_send.cu:54)
                    at = excl + toff;
                    st.pos_token[(size_t)g * ws.max_tk + at] = token;
                }
                ws.token_offset[(size_t)g * ws.max_tk + token * K + k] = toff;
                ws.route_slot[(size_t)g * ws.max_tk + token * K + k] = at;
            }
        }
    }
    stage_row<QUANT>(args, st, g, token, staging_threads);
}

constexpr uint32_t kPieceThreads = 256;   // threads of a workgroup of the kernels that copy rows in pieces
constexpr uint32_t kPieceLoads = 2;       // sixteen-byte chunks of a piece that a lane moves, both in flight
constexpr uint32_t kPieceChunks = kPieceLoads * kWave;

// A team of `team` threads (one or more whole wavefronts) copies a staged row of `num_chunks` 16-byte pieces:
// eight loads per thread in flight.  Ordinary loads, because the recvs of the other ranks its token was routed to read
// the row again (non-temporal ones here, in the step's first recv: whole steps of one sender of 512 tokens 86.9 -> 89.7
// us, of 1024 tokens on 16 ranks 164.3 -> 170.5).
__device__ __forceinline__ void copy_row_by_team(const u32x4 *src, u32x4 *dst, uint32_t num_chunks, uint32_t member,
                                                 uint32_t team) {
    for (uint32_t c0 = 0; c0 < num_chunks; c0 += 8 * team) {
        u32x4 v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t c = c0 + u * team + member;
            if (c < num_chunks) v[u] = src[c];
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t c = c0 + u * team + member;
            if (c < num_chunks) dst[c] = v[u];
        }
    }
}

// Payload and scales of one received row, by a team.  The scales are asked for before the payload
// moves: behind the payload's stores their trip would begin only when those have been acknowledged
// (memory operations of a wavefront complete in order).
__device__ __forceinline__ void copy_received_row(const uint8_t *src, uint32_t payload_bytes, uint32_t num_chunks,
                                                  uint32_t num_scales, const PushDst &dst, uint32_t dst_row,
                                                  uint32_t member, uint32_t team) {
    const float *ss = reinterpret_cast<const float *>(src + payload_bytes);
    float first_scale = 0.0f;
    const bool scales = dst.out_scale != nullptr;
    if (scales && member < num_scales) first_scale = ss[member];
    copy_row_by_team(reinterpret_cast<const u32x4 *>(src),
                     reinterpret_cast<u32x4 *>(dst.out_x + (size_t)dst_row * dst.out_stride), num_chunks, member, team);
    if (scales) {
        float *os = dst.out_scale + (size_t)dst_row * dst.os_stride_token;
        if (member < num_scales) os[(size_t)member * dst.os_stride_elem] = first_scale;
        for (uint32_t q = member + team; q < num_scales; q += team) os[(size_t)q * dst.os_stride_elem] = ss[q];
    }
}

// ---------------------------------------------------------------------------
// dispatch recv.  The receivers of a step are laid out ONCE per step, by the step's
// first recv (the reference's host worker runs process_routing_info once per rank
// and step, a2a_worker.rs:526-703).  A layout is made in LDS from the published
// per-source counts of a receiver's experts (a2a_worker.rs:577-606,621-694: rows per
// expert, padded first row of every expert, first row of every (source, expert) run
// inside it, and the order in which the runs ARRIVE: sources in the worker's order,
// experts inside a source); then one thread per received row writes the row's
// metadata (padded_index, source_rank, source position and the two offset tables:
// a2a_worker.rs:636-671) and the staged row it comes from (the token behind its
// position in the sender's order).
//
// stage_layout_kernel does that for every receiver, in front of the first recv's
// copy.  Where the rows are few, stage_recv_first_few_kernel does layout and copy in
// one launch: its first workgroups lay out the OTHER receivers, those behind them
// lay the calling rank out, each for the row it copies.
//
// stage_recv_kernel is the copy: where a row comes from and where it goes is read
// from the tables (a2a_dispatch_recv.cu:139-155); its first workgroup hands the
// receiver's counts to the caller.
//
// Dynamic LDS of a layout: 5 * G * Le + 1 + 3 * G + Le words.
// ---------------------------------------------------------------------------
struct ReceiverTables {   // in LDS, see lay_out_receiver
    uint32_t *tot;       // [g][le]  copies source g sends to local expert le
    uint32_t *excl;      // [g][le]  position of the run in the sender's expert-sorted order
    uint32_t *run_row;   // [i][le]  first row of the run in the receiver's buffer (i = order index)
    uint32_t *seg;       // [i][le]  first ARRIVAL index of the run; seg[items] = rows received
    uint32_t *grp_dst;   // [g]      position of source g's first row for this receiver in g's send order
    uint32_t *grp_src;   // [g]      rows this receiver gets from the sources numbered below g
    uint32_t *grp_cnt;   // [g]      rows this receiver gets from source g
    const uint8_t *order;  // [i]    the i-th source this receiver lays out
    uint32_t rows;       // rows received
    // (w = i * Le + le is the run of the i-th source visited and local expert le)
    uint32_t *pos;       // [w]      position of the run in the sender's expert-sorted order (excl, by run)
    uint32_t own_g, own_pos, own_seg, own_end, own_row;   // run w = threadIdx.x of this thread (if there is one), in registers
};

// What the receiver's tables say of arrival `row` of run `s` (seg[s] <= row < seg[s + 1]).
struct RowMeta {
    uint32_t g;        // source (dp group)
    uint32_t pos;      // position in the source's expert-sorted order
    uint32_t dst_row;  // row in the receiver's buffer
};

// Writes the five per-row tables of the reference's host worker for arrival `row` of receiver `r`
// (a2a_worker.rs:633-671).  One thread.
__device__ __forceinline__ void write_row_tables(const ReceiverTables &t, const Workspace &ws, const Staging &st,
                                                 uint32_t r, uint32_t row, const RowMeta &m, uint32_t max_private) {
    const uint32_t G = ws.num_groups;
    const size_t at = (size_t)r * st.max_recv + row;
    st.padded_index[at] = m.dst_row;
    // the member of the group that sends to this rank (a2a_worker.rs:633)
    const uint32_t peer = m.g * ws.dp_size + r % ws.dp_size;
    st.source_rank[at] = peer;
    st.source_position[at] = m.pos;
    // How the reference addresses the row on its way in and on its way back (a2a_worker.rs:636-667).
    // Nothing here reads these two: they are what a rank on a GPU of its own would consume.
    const uint32_t index_on_rank = m.pos - t.grp_dst[m.g];     // rows of this source before this one
    const bool same_node = peer / ws.node_size == r / ws.node_size;
    uint32_t sdo = m.pos, cso = m.pos;                         // own rows: the sender's position
    if (peer != r) {
        if (index_on_rank < max_private) {
            sdo = max_private * m.g + index_on_rank;                               // private region
        } else if (same_node) {
            sdo = m.pos | 0x80000000u;                                             // read from the peer's send buffer
        } else {
            sdo = t.grp_src[m.g] + index_on_rank + max_private * (G - 1);          // overflow region
        }
    }
    if ((peer != r || ws.dp_size > 1) && !same_node) cso = t.grp_src[m.g] + index_on_rank;
    st.source_dispatch_offset[at] = sdo;
    st.combine_send_offset[at] = cso;
}

// Lays out receiver `r` in LDS.  Whole workgroup.  `publish`: this workgroup also writes the
// receiver's tables to memory and (if given) its counts to the caller.  Returns false, before the
// expensive part, when the workgroup's first row `first_row` lies beyond the rows received and it
// does not publish: the host sizes grids for an upper bound, a receiver typically gets 1/N of it.
// In the tables run_row, seg and pos a run is w = i * Le + le, i the source's place in the order of
// the layout.
//
// The work is spread over all threads, one run (source in the order of the layout, local expert)
// each, and what counts is the number of dependent LDS trips and barriers between the arrival of the
// counts and the first row's load (each about 0.1 us): everything that can be asked for together is,
// reads before writes.  One wavefront doing the layout alone, in loops over the sources with one trip
// per step, was 1.5 us of the 2.2 us a small step's recv waited for its layout.
// After the last barrier inside, a thread's OWN runs (w = tid, tid + blockDim.x, ...) are complete in
// LDS and the first of them is in t.own_*; `all_visible` adds the barrier after which every thread
// may read every run.
__device__ __forceinline__ bool lay_out_receiver(uint32_t valid_mask, const Workspace &ws, const Staging &st, uint32_t r,
                                                 bool publish, uint32_t first_row, int32_t *out_num_tokens,
                                                 uint32_t out_rows, uint32_t *s_recv, uint8_t *s_order,
                                                 ReceiverTables &t, bool all_visible) {
    const uint32_t G = ws.num_groups, E = ws.num_experts, Le = ws.experts_per_rank;
    const uint32_t first = r * Le;
    const uint32_t n_local = first >= E ? 0 : (E - first < Le ? E - first : Le);
    const uint32_t items = G * Le;
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    uint32_t *tot = t.tot = s_recv;
    uint32_t *excl = t.excl = tot + items;
    uint32_t *pos_of = t.pos = excl + items;
    uint32_t *run_row = t.run_row = pos_of + items;
    uint32_t *seg = t.seg = run_row + items;
    uint32_t *grp_dst = t.grp_dst = seg + items + 1;
    uint32_t *grp_src = t.grp_src = grp_dst + G;
    uint32_t *grp_cnt = t.grp_cnt = grp_src + G;
    uint32_t *poff = grp_cnt + G;   // [le] rows of a local expert, then its padded first row
    t.order = s_order;

    // The order in which this receiver lays out its sources (one byte per source, from the table the
    // context computed once) is asked for with the counts: every thread takes the first two words (the
    // first eight sources) for its loops over the sources, the first eight threads copy the table's row
    // to LDS for whoever needs the i-th source with an i of its own.  All loads of a thread are asked
    // for before the first is used, none under a condition of its own (a word that does not count is
    // read from a valid place and dropped): waited for one by one they are a trip to memory each.
    const uint32_t *order_row = ws.order + r * (kMaxWorld / 4);
    const uint32_t order_lo = order_row[0], order_hi = order_row[1];
    const uint32_t order_mine = order_row[tid & (kMaxWorld / 4 - 1)];
    uint32_t *order_words = reinterpret_cast<uint32_t *>(s_order);
    for (uint32_t w = tid; w < items; w += nthreads) {
        const uint32_t g = Le > 1 ? __umulhi(w, ws.le_magic) : w;
        const uint32_t le = w - g * Le;
        const uint32_t e = first + le;
        const bool live = le < n_local && (valid_mask >> g & 1);
        const uint32_t at = live ? g * E + e : 0;
        const uint32_t count = ws.num_routed[at];
        const uint32_t upto = ws.expert_offsets[at > 0 ? at - 1 : 0];
        tot[w] = live ? count : 0;
        excl[w] = live && e > 0 ? upto : 0;
    }
    if (tid < (uint32_t)kMaxWorld / 4) order_words[tid] = order_mine;
    __syncthreads();
    const uint32_t o0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)order_lo);
    const uint32_t o1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)order_hi);

    // Rows of local expert `le` from the sources visited before the i-th, and from all of them.
    auto sums_over_sources = [&](uint32_t i, uint32_t le, uint32_t &below, uint32_t &total) {
        below = total = 0;
        for (uint32_t b = 0; b < G; b += 8) {
            // eight sources at a time: their numbers are the same for every thread (scalar), their
            // counts are asked for together
            const uint32_t w0 = b == 0 ? o0 : (uint32_t)__builtin_amdgcn_readfirstlane((int)order_words[b / 4]);
            const uint32_t w1 = b == 0 ? o1 : (uint32_t)__builtin_amdgcn_readfirstlane((int)order_words[b / 4 + 1]);
            uint32_t c[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                const uint32_t g = ((u < 4 ? w0 : w1) >> (8 * (u & 3))) & 0xFFu;   // (0 past the last source)
                c[u] = tot[g * Le + le];
            }
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                if (b + u < G) total += c[u];
                if (b + u < i) below += c[u];
            }
        }
    };

    // ---- first trip: everything that needs only the counts.  Run w = tid of this thread first.
    // (A wavefront none of whose threads has a run skips what only runs need: what every wavefront
    // of a workgroup executes costs the SIMDs they share as much time as what one executes alone.)
    const bool has_runs = tid - lane < items;   // the same for a whole wavefront
    const uint32_t w_own = tid < items ? tid : 0;
    const uint32_t i_own = Le > 1 ? __umulhi(w_own, ws.le_magic) : w_own;
    const uint32_t le_own = w_own - i_own * Le;
    const bool source_lane = lane < G && n_local != 0;
    const uint32_t last = source_lane ? lane * Le + n_local - 1 : 0;
    const uint32_t excl_last = excl[last], tot_last = tot[last], excl_first = excl[source_lane ? lane * Le : 0];
    uint32_t visited = 0, g_own = 0, below_own = 0, total_own = 0;
    if (has_runs) {
        visited = s_order[lane < G ? lane : 0];   // lane i: the i-th source in the order of the layout
        g_own = s_order[i_own];
        sums_over_sources(i_own, le_own, below_own, total_own);
    }

    // Rows this receiver gets from source g (lane g; there are at most kMaxWorld <= 64 sources): the
    // sender's scan over its experts gives them without a sum.  Every wavefront adds them up by itself.
    const uint32_t from_source = source_lane ? excl_last + tot_last - excl_first : 0;
    const uint32_t from_lower = wave_inclusive_scan(from_source, lane);   // inclusive over the sources
    const uint32_t rows = t.rows = (uint32_t)__builtin_amdgcn_readlane((int)from_lower, kWave - 1);
    if (!publish && first_row >= rows) return false;   // uniform

    // ---- second trip: the rows of the i-th source visited (lane i), the position and rows of the own run
    uint32_t theirs = 0, pos0_own = 0, pos_own = 0, tot_own = 0;
    if (has_runs) {
        theirs = (uint32_t)__shfl((int)from_source, (int)visited);   // every lane of the wavefront takes part
        pos0_own = excl[g_own * Le];
        pos_own = excl[g_own * Le + le_own];
        tot_own = tot[g_own * Le + le_own];
    }

    // Padded first row of every local expert: a scan over the experts, by the first wavefront, whose
    // thread `le` has the expert's rows already (thread le is run (0, le)).  With more than 64 local
    // experts the counts go through LDS and a barrier.
    const uint32_t pad = ws.expert_padding;
    const bool wide = Le > (uint32_t)kWave;   // uniform
    if (wide) {
        if (tid < Le) poff[tid] = total_own;
        for (uint32_t le = tid + nthreads; le < Le; le += nthreads) {
            uint32_t below, total;
            sums_over_sources(0, le, below, total);
            poff[le] = total;
        }
        __syncthreads();
    }
    if (wave == 0) {
        uint32_t carry = 0;
        for (uint32_t l0 = 0; l0 < Le; l0 += kWave) {
            const uint32_t le = l0 + lane;
            const bool mine = le < n_local;
            const uint32_t tpe = !mine ? 0 : (wide ? poff[le] : total_own);
            const uint32_t padded = pad > 1 ? (tpe + pad - 1) / pad * pad : tpe;
            const uint32_t scan = wave_inclusive_scan(padded, lane);
            const uint32_t mine_off = carry + scan - padded;
            if (le < Le) poff[le] = mine_off;
            if (mine && publish) {
                const uint32_t e = first + le;
                ws.tokens_per_expert[e] = tpe;
                ws.padded_offset[e] = mine_off;
                if (out_num_tokens != nullptr) out_num_tokens[le] = (int32_t)tpe;
                if (mine_off + tpe > out_rows) atomicOr(ws.err, A2A_DEV_RECV_OVERFLOW);
            }
            carry += (uint32_t)__builtin_amdgcn_readlane((int)scan, kWave - 1);
        }
    }

    // Arrival order: sources as the worker visits them, local experts inside a source.  Lane i of every
    // wavefront has the rows of the i-th source visited and those that arrive before them.
    uint32_t arrive = 0, before = 0, seg_own = 0;
    if (has_runs) {
        arrive = lane < G ? theirs : 0;
        before = wave_inclusive_scan(arrive, lane) - arrive;
        // ---- third trip: the own run's source in that order
        const uint32_t base_own = (uint32_t)__shfl((int)before, (int)i_own);    // every lane of the wavefront takes part
        const uint32_t count_own = (uint32_t)__shfl((int)arrive, (int)i_own);
        seg_own = base_own + (le_own < n_local ? pos_own - pos0_own : count_own);
    }
    t.own_g = g_own;
    t.own_pos = pos_own;
    t.own_seg = seg_own;
    t.own_end = seg_own + tot_own;   // (the run after this one begins where this one's rows end)

    // ---- writes
    if (tid < items) {
        seg[tid] = seg_own;
        pos_of[tid] = pos_own;
    }
    if (wave == 0 && lane < G) {
        // Per source: where its rows for this receiver begin in its own send order (dst_group_offset,
        // a2a_worker.rs:571-575) and how many rows the lower-numbered sources send here
        // (src_group_offset, a2a_worker.rs:582-590: numeric order, not the order of arrival).
        grp_dst[lane] = excl_first;
        grp_cnt[lane] = from_source;
        grp_src[lane] = from_lower - from_source;
    }
    if (tid == 0) {
        seg[items] = rows;
        if (publish) {
            if (rows > st.max_recv) atomicOr(ws.err, A2A_DEV_RECV_OVERFLOW);
            st.num_recv[2 * r] = rows;
        }
    }
    // the runs beyond the first of a thread (more runs than threads): the same, one at a time
    for (uint32_t w0 = nthreads; w0 < items; w0 += nthreads) {
        const uint32_t w = w0 + tid;
        const bool real = w < items;
        const uint32_t wc = real ? w : 0;
        const uint32_t i = Le > 1 ? __umulhi(wc, ws.le_magic) : wc;
        const uint32_t le = wc - i * Le;
        uint32_t below, total;
        sums_over_sources(i, le, below, total);
        const uint32_t g = s_order[i];
        const uint32_t p0 = excl[g * Le];
        const uint32_t p = excl[g * Le + le];
        const uint32_t base = (uint32_t)__shfl((int)before, (int)i);    // every lane takes part
        const uint32_t count = (uint32_t)__shfl((int)arrive, (int)i);
        if (real) {
            run_row[w] = below;
            seg[w] = base + (le < n_local ? p - p0 : count);
            pos_of[w] = p;
        }
    }
    __syncthreads();

    // First row of every run: behind the rows of the expert from the sources visited earlier.
    t.own_row = below_own + poff[le_own];
    if (tid < items) {
        run_row[tid] = t.own_row;
        if (publish && le_own < n_local) ws.slot_base[g_own * E + first + le_own] = t.own_row;
    }
    for (uint32_t w = tid + nthreads; w < items; w += nthreads) {
        const uint32_t i = Le > 1 ? __umulhi(w, ws.le_magic) : w;
        const uint32_t le = w - i * Le;
        const uint32_t row = run_row[w] + poff[le];
        run_row[w] = row;
        if (publish && le < n_local) ws.slot_base[(uint32_t)s_order[i] * E + first + le] = row;
    }
    if (publish && tid == 0) {
        // rows that come from other nodes (num_efa_tokens, a2a_worker.rs:681-687)
        const uint32_t remote_segs = (ws.world / ws.node_size - 1) * (ws.node_size / ws.dp_size) * Le;
        st.num_recv[2 * r + 1] = remote_segs < items ? seg[remote_segs] : rows;
    }
    if (all_visible) __syncthreads();
    return true;
}

// What the tables say of arrival `row` of run `s` (seg[s] <= row < seg[s + 1]): one LDS trip.
__device__ __forceinline__ RowMeta row_of_run(const ReceiverTables &t, const Workspace &ws, uint32_t s, uint32_t row) {
    const uint32_t Le = ws.experts_per_rank;
    const uint32_t i = Le > 1 ? __umulhi(s, ws.le_magic) : s;
    RowMeta m;
    m.g = t.order[i];
    const uint32_t j = row - t.seg[s];
    m.pos = t.pos[s] + j;
    m.dst_row = t.run_row[s] + j;
    return m;
}

// Slice `slice` of the work that lays out receiver `r`: the layout in LDS, then one thread per received
// row writes the row's tables and the staged row it comes from.
__device__ __forceinline__ void lay_out_rows(const StageRecvArgs &args, const Workspace &ws, const Staging &st, uint32_t r,
                                             uint32_t slice, uint32_t *s_recv, uint8_t *s_order) {
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    ReceiverTables t;
    if (!lay_out_receiver(args.valid_mask, ws, st, r, slice == 0, slice * nthreads, nullptr, 0xFFFFFFFFu,
                                 s_recv, s_order, t, true))
        return;
    const uint32_t total = t.rows < st.max_recv ? t.rows : st.max_recv;   // beyond: flagged and dropped
    for (uint32_t row = slice * nthreads + tid; row < total; row += args.slices * nthreads) {
        // the run this arrival belongs to: the last one with seg[s] <= row (runs without rows share
        // their first arrival with the run after them, so the last such run is the one with rows)
        uint32_t lo = 0, hi = ws.num_groups * ws.experts_per_rank;   // seg[lo] <= row < seg[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (t.seg[mid] <= row) lo = mid; else hi = mid;
        }
        const RowMeta m = row_of_run(t, ws, lo, row);
        // the token behind the position: asked for first, used last
        const uint32_t token = m.pos < ws.max_tk ? st.pos_token[(size_t)m.g * ws.max_tk + m.pos] : 0;
        write_row_tables(t, ws, st, r, row, m, args.max_private);
        st.moves[(size_t)r * st.max_recv + row] = uint4{m.dst_row, m.g * st.max_tokens + token, m.g, m.pos};
    }
}

// The step's first recv when the step has few rows (the host gave every row a workgroup as wide as the
// row): layout and copy in one launch; the whole workgroup serves one row at a time, and the thread whose
// run holds the row says so to the others.
// Dynamic LDS: 5 * G * Le + 1 + 3 * G + Le words.
__global__ __launch_bounds__(1024) void stage_recv_first_few_kernel(const StageRecvArgs args, const Workspace ws,
                                                                    const Staging st) {
    extern __shared__ uint32_t s_recv[];
    __shared__ __align__(16) uint8_t s_order[kMaxWorld];
    __shared__ uint32_t s_meta[3];
    const uint32_t tid = threadIdx.x;
    const uint32_t nthreads = blockDim.x;
    const uint32_t items = ws.num_groups * ws.experts_per_rank;
    ReceiverTables t;

    // The workgroups of the other receivers come first in the grid: their chain (layout, run and token
    // of every row, the row's tables) is as long as the calling rank's (layout, row, copy), and started
    // behind its workgroups they were what the kernel's end waited for (0.15 us).
    const uint32_t other_blocks = gridDim.x - args.copy_blocks;
    if (blockIdx.x < other_blocks) {
        // ---- one of the other receivers: layout, then one thread per received row ----
        uint32_t r = blockIdx.x / args.slices;
        const uint32_t slice = blockIdx.x - r * args.slices;
        if (r >= args.rank) ++r;   // the caller's rank is served by the workgroups behind these
        lay_out_rows(args, ws, st, r, slice, s_recv, s_order);
        return;
    }

    // ---- the caller's rank: layout, then the workgroup's row ----
    const uint32_t r = args.rank;
    const PushDst &dst = args.dst;
    const uint32_t num_chunks = args.row_bytes / 16;
    const uint32_t block = blockIdx.x - other_blocks;
    if (!lay_out_receiver(args.valid_mask, ws, st, r, block == 0, block, args.out_num_tokens,
                                 args.dst.out_rows, s_recv, s_order, t, false))
        return;
    for (uint32_t row = block; row < t.rows; row += args.copy_blocks) {
        if (row != block) __syncthreads();   // the row before this one has been taken from s_meta
        if (tid < items && t.own_seg <= row && row < t.own_end) {   // in the thread's first run: all in registers
            s_meta[0] = t.own_g;
            s_meta[1] = t.own_pos + (row - t.own_seg);
            s_meta[2] = t.own_row + (row - t.own_seg);
        }
        for (uint32_t w = tid + nthreads; w < items; w += nthreads) {
            // (a thread's own runs are complete, and every run's first arrival is there)
            if (t.seg[w] <= row && row < t.seg[w + 1]) {
                const RowMeta mine = row_of_run(t, ws, w, row);
                s_meta[0] = mine.g;
                s_meta[1] = mine.pos;
                s_meta[2] = mine.dst_row;
            }
        }
        __syncthreads();
        RowMeta m;
        m.g = s_meta[0];
        m.pos = s_meta[1];
        m.dst_row = s_meta[2];
        if (row >= st.max_recv) continue;   // flagged by the layout: more rows than the receive region was sized for
        const uint32_t token = st.pos_token[(size_t)m.g * ws.max_tk + m.pos];
        if (tid == 0) {
            write_row_tables(t, ws, st, r, row, m, args.max_private);
            st.moves[(size_t)r * st.max_recv + row] = uint4{m.dst_row, m.g * st.max_tokens + token, m.g, m.pos};
        }
        if (dst.out_x != nullptr) {
            if (m.dst_row >= dst.out_rows) {
                if (tid == 0) atomicOr(ws.err, A2A_DEV_RECV_OVERFLOW);
            } else {
                const uint8_t *src = st.send_buf + ((size_t)m.g * st.max_tokens + token) * st.disp_stride;
                copy_received_row(src, st.payload_bytes, num_chunks, args.hidden_dim_scale, dst, m.dst_row, tid, nthreads);
            }
        }
    }
}

// The receiver's counts for the caller (a2a_dispatch_recv.cu:220-224).  One workgroup of a recv that did
// not lay the receiver out itself.
__device__ __forceinline__ void hand_over_counts(const RecvRowsArgs &args) {
    for (uint32_t le = threadIdx.x; le < args.num_local; le += kPieceThreads) {
        const uint32_t tpe = args.counts[le];
        if (args.out_num_tokens != nullptr) args.out_num_tokens[le] = (int32_t)tpe;
        if (args.counts[kTableUnit * args.to_first_rows + le] + tpe > args.out_rows)
            atomicOr(args.flags(), A2A_DEV_RECV_OVERFLOW);
    }
}

// Lays out every receiver of a step whose rows are copied by the kernels below (the first recv of the
// step launches it in front of its copy): the same layout as above, then one thread per received row.
// Dynamic LDS as stage_recv_first_few_kernel.
__global__ __launch_bounds__(1024) void stage_layout_kernel(const StageRecvArgs args, const Workspace ws,
                                                            const Staging st) {
    extern __shared__ uint32_t s_recv[];
    __shared__ __align__(16) uint8_t s_order[kMaxWorld];
    const uint32_t r = blockIdx.x / args.slices;
    lay_out_rows(args, ws, st, r, blockIdx.x - r * args.slices, s_recv, s_order);
}

// Rows cut into pieces of kPieceChunks sixteen-byte chunks, a wavefront each: wavefront w of the grid takes the
// pieces w, w + wavefronts, ... of all rows counted through.
struct PieceWalk {
    uint32_t row, piece;

    __device__ __forceinline__ void start(const PieceGrid &grid, uint32_t unit) {
        row = grid.pieces > 1 ? __umulhi(unit, grid.magic) : unit;
        piece = unit - row * grid.pieces;
    }
    __device__ __forceinline__ void advance(const PieceGrid &grid) {
        row += grid.step_rows;
        piece += grid.step_pieces;
        if (piece >= grid.pieces) {
            piece -= grid.pieces;
            ++row;
        }
    }
};

// A recv that did not lay the receivers out.  It only moves rows, and what bounds it is the write side of
// HBM while the reads can come from the Infinity Cache: every staged row is read by the recvs of all the
// ranks its token was routed to.  Hence
//  - the rows are walked in the order of arrival by a grid of wavefronts, two 16-byte chunks a lane, so that
//    reads and writes each advance as ONE front through memory.  A wavefront per row with eight chunks a
//    lane in flight kept 4096 rows half open at a time: rows of 7392 bytes, 16384 a launch (8 ranks x 2048
//    tokens), 52.1 us = 4.65 TB/s of reads and writes then, 42.1 us in this order;
//  - staged rows are loaded with ordinary loads, which keep them in that cache, and where the copies of a step
//    are more than it can keep for their reader (STREAM: received_past_cache in a2a_rules.h) they are stored
//    non-temporally, which keeps THEM out of it: 37.0 us = 6.5 TB/s (rows of 14 KB, 235 MB staged: 84.3 -> 69.3 us;
//    470 MB staged, more than the cache holds: 172 -> 143 us with non-temporal loads as the other side).
// A row's scales travel with its first pieces; they are 3 us of the 42 (rows of scales are not whole cache
// lines: their ends are written by two wavefronts at different times).  Scales that the caller wants by COLUMN would be a
// cache line a word that way, written by as many wavefronts as it has words: COLUMNS moves them in workgroups of their own in
// front of the grid, a wavefront for kScaleColumns columns of 64 rows in the order of arrival, whose rows lie side by side run
// by run (an expert's rows of one source).  Step of 8 x 2048 tokens of 7168 bytes 1422 -> 1382 us, of 8 x 400 353 -> 347, one
// sender of 4096 367 -> 356.  Their chain (entries, staged words, stores) is longer than a piece's, so with few words to
// move (kColumnWords, of a typical receiver) the pieces carry them: 1600 rows of 56 (90 thousand) 222 us against 225,
// 4800 of 16 (77) 212 against 217, 8192 of 8 (66) 202 against 211; on the other side 2400 of 56 (134) 291 against 288, 2048 of
// 56 (115) 210 against 208.6, 9600 of 16 (154) 332.5 against 329.7.
constexpr uint32_t kScaleColumns = 8;
constexpr uint64_t kColumnWords = 112 * 1024;

// The scales of the received rows, by column.  `unit`, `units`: of the wavefronts that do this.
__device__ __forceinline__ void receive_scale_columns(const RecvRowsArgs &args, uint32_t total, uint32_t unit, uint32_t units) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t num_scales = args.num_scales;
    const size_t staged_stride = staged_row_stride(args.row_bytes, num_scales);
    const uint32_t slices = (num_scales + kScaleColumns - 1) / kScaleColumns;
    for (; unit / slices * kWave < total; unit += units) {
        const uint32_t row = unit / slices * kWave + lane;
        const uint32_t first = unit % slices * kScaleColumns;
        const uint4 move = args.moves[row < total ? row : total - 1];
        if (row >= total || move.x >= args.out_rows) continue;   // (rows that do not fit are flagged where they are copied)
        const u32x4 *from = reinterpret_cast<const u32x4 *>(args.staged + (size_t)move.y * staged_stride + args.row_bytes) +
                            first / 4;
        float *to = args.out_scale + (size_t)move.x * args.os_stride_token + (size_t)first * args.os_stride_elem;
        // (a staged row has 16 spare bytes behind its scales)
        u32x4 v[kScaleColumns / 4];
#pragma unroll
        for (uint32_t i = 0; i < kScaleColumns / 4; ++i) v[i] = first + 4 * i < num_scales ? from[i] : u32x4{0, 0, 0, 0};
#pragma unroll
        for (uint32_t j = 0; j < kScaleColumns; ++j) {
            if (first + j < num_scales) to[(size_t)j * args.os_stride_elem] = __uint_as_float(v[j / 4][j % 4]);
        }
    }
}

template <bool STREAM, bool COLUMNS>
__global__ __launch_bounds__(kPieceThreads) void stage_recv_kernel(const RecvRowsArgs args) {
    // everything a wavefront takes from the argument block, asked for in one go
    A2A_PIN(args.out_x);
    A2A_PIN(args.out_scale);
    A2A_PIN(args.out_stride);
    A2A_PIN(args.os_stride_elem);
    A2A_PIN(args.os_stride_token);
    A2A_PIN(args.out_rows);
    A2A_PIN(args.row_bytes);
    A2A_PIN(args.num_scales);
    A2A_PIN(args.pieces);
    A2A_PIN(args.magic);
    A2A_PIN(args.step_rows);
    A2A_PIN(args.step_pieces);
    if constexpr (COLUMNS) A2A_PIN(args.scale_blocks);
    A2A_PIN(args.staged);
    A2A_PIN(args.moves);
    A2A_PIN(args.num_recv);
    A2A_PIN(args.max_recv);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t num_chunks = args.row_bytes / 16;
    const uint4 *const moves = args.moves;
    const PieceGrid grid = {args.pieces, args.magic, args.step_rows, args.step_pieces};
    // The first piece's table entry is asked for together with the number of rows received
    // (a row index the tables do not hold reads entry 0 and is dropped by the loop's bound).
    const size_t staged_stride = staged_row_stride(args.row_bytes, args.num_scales);
    PieceWalk at;
    const uint32_t scale_blocks = COLUMNS ? args.scale_blocks : 0;
    const uint32_t block = blockIdx.x - scale_blocks;   // (wraps around for the workgroups in front: they move scales)
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    at.start(grid, COLUMNS && blockIdx.x < scale_blocks ? 0 : block * (kPieceThreads / kWave) + wave);
    const uint32_t probe = at.row < args.max_recv ? at.row : 0;
    uint4 move = moves[probe];
    uint32_t total = *args.num_recv;
    if (total > args.max_recv) total = args.max_recv;   // flagged by the layout: more rows than the region was sized for

    if (COLUMNS && blockIdx.x < scale_blocks) {
        receive_scale_columns(args, total, blockIdx.x * (kPieceThreads / kWave) + wave,
                              scale_blocks * (kPieceThreads / kWave));
        return;
    }
    if (block == 0) hand_over_counts(args);
    if (args.out_x == nullptr) return;

    while (at.row < total) {
        const uint32_t dst_row = move.x;
        const uint8_t *src = args.staged + (size_t)move.y * staged_stride;
        const uint32_t chunk = at.piece * kPieceChunks + lane, c = at.piece * kWave + lane;   // c: of the scales
        const bool fits = dst_row < args.out_rows;
        const bool scaled = !COLUMNS && fits && args.out_scale != nullptr && c < args.num_scales;
        u32x4 v[kPieceLoads];
        float scale = 0.0f;
#pragma unroll
        for (uint32_t u = 0; u < kPieceLoads; ++u) {
            v[u] = u32x4{0, 0, 0, 0};
            if (fits && chunk + u * kWave < num_chunks) v[u] = reinterpret_cast<const u32x4 *>(src)[chunk + u * kWave];
        }
        if (scaled) scale = reinterpret_cast<const float *>(src + args.row_bytes)[c];
        // the next piece's entry travels while this one is copied
        PieceWalk next = at;
        next.advance(grid);
        const uint32_t next_probe = next.row < total ? next.row : at.row;
        const uint4 next_move = moves[next_probe];
        u32x4 *const to = reinterpret_cast<u32x4 *>(args.out_x + (size_t)dst_row * args.out_stride) + chunk;
#pragma unroll
        for (uint32_t u = 0; u < kPieceLoads; ++u) {
            if (!fits || chunk + u * kWave >= num_chunks) continue;
            if constexpr (STREAM) __builtin_nontemporal_store(v[u], to + u * kWave); else store_copy(v[u], to + u * kWave);
        }
        if (scaled) args.out_scale[(size_t)dst_row * args.os_stride_token + (size_t)c * args.os_stride_elem] = scale;
        if (!COLUMNS && fits && args.out_scale != nullptr) {
            // rows with more scales than pieces have lanes
            for (uint32_t q = c + grid.pieces * kWave; q < args.num_scales; q += grid.pieces * kWave) {
                args.out_scale[(size_t)dst_row * args.os_stride_token + (size_t)q * args.os_stride_elem] =
                    reinterpret_cast<const float *>(src + args.row_bytes)[q];
            }
        }
        if (!fits && at.piece == 0 && lane == 0) atomicOr(args.flags(), A2A_DEV_RECV_OVERFLOW);
        at = next;
        move = next_move;
    }
}

// ---------------------------------------------------------------------------
// combine send: copy expert_y[padded_index[i]] to the staging row of the copy
// it answers, i.e. row `source_position[i]` of sender `source_rank[i]`
// (a2a_combine_send.cu:124-136,196-205).  Walked in pieces as stage_recv_kernel is, and for the same
// reason: in the order of arrival the rows written are consecutive per source and the rows read per
// (source, expert), so both sides are fronts through memory.  16384 rows of 14 KB: 105.5 us = 4.45 TB/s
// with a wavefront per row, 76.5 us = 6.1 TB/s in this order with one chunk a lane (a plain copy of as many rows in the
// same order, examples/ceilings.hip: 67.6 us; both sides come from and go to HBM, so loads and stores keep nothing).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kPieceThreads) void combine_send_kernel(const CombineSendArgs args) {
    // everything a wavefront takes from the argument block, asked for in one go
    A2A_PIN(args.y);
    A2A_PIN(args.y_stride);
    A2A_PIN(args.y_rows);
    A2A_PIN(args.row_bytes);
    A2A_PIN(args.grid.pieces);
    A2A_PIN(args.grid.magic);
    A2A_PIN(args.grid.step_rows);
    A2A_PIN(args.grid.step_pieces);
    A2A_PIN(args.max_tk);
    A2A_PIN(args.staged);
    A2A_PIN(args.moves);
    A2A_PIN(args.num_recv);
    A2A_PIN(args.staged_stride);
    A2A_PIN(args.max_recv);
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t num_chunks = args.row_bytes / 16;
    const uint4 *const moves = args.moves;
    PieceWalk at;
    at.start(args.grid, __builtin_amdgcn_readfirstlane(blockIdx.x * (kPieceThreads / kWave) + threadIdx.x / kWave));
    const uint32_t probe = at.row < args.max_recv ? at.row : 0;
    uint4 move = moves[probe];
    uint32_t total = *args.num_recv;
    if (total > args.max_recv) total = args.max_recv;
    while (at.row < total) {
        const uint32_t c = at.piece * kPieceChunks + lane;
        const uint32_t row = move.x, g = move.z, pos = move.w;   // (every member of a dp group reads the same staging rows)
        const bool fits = row < args.y_rows && pos < args.max_tk;
        const u32x4 *const from = reinterpret_cast<const u32x4 *>(args.y + (size_t)row * args.y_stride) + c;
        u32x4 v[kPieceLoads];
#pragma unroll
        for (uint32_t u = 0; u < kPieceLoads; ++u) {
            v[u] = u32x4{0, 0, 0, 0};
            if (fits && c + u * kWave < num_chunks) v[u] = __builtin_nontemporal_load(from + u * kWave);
        }
        // the next piece's entry travels while this one is copied
        PieceWalk next = at;
        next.advance(args.grid);
        const uint32_t next_probe = next.row < total ? next.row : at.row;
        const uint4 next_move = moves[next_probe];
        u32x4 *const to = reinterpret_cast<u32x4 *>(args.staged + ((size_t)g * args.max_tk + pos) * args.staged_stride) + c;
#pragma unroll
        for (uint32_t u = 0; u < kPieceLoads; ++u) {
            if (fits && c + u * kWave < num_chunks) store_copy(v[u], to + u * kWave);
        }
        if (!fits && at.piece == 0 && lane == 0) atomicOr(args.err, A2A_DEV_BAD_SLOT);
        at = next;
        move = next_move;
    }
}

uint32_t block_for_chunks(uint32_t chunks) {
    uint32_t threads = (chunks + kWave - 1) / kWave * kWave;
    if (threads < (uint32_t)kWave) threads = kWave;
    if (threads > 1024) threads = 1024;
    return threads;
}

// The rows of a receiver are copied in pieces by a grid of wavefronts that walks all pieces of all rows in
// order.  The host knows an upper bound of the rows (every copy of every sender); a receiver typically gets
// 1/N of it.
//   - combine-send, and recvs of receivers that typically get kInOrderRows rows (`in_order`): a wavefront per piece of the
//     typical receiver (more loop), so that the hardware, which starts workgroups in order, keeps the front of reads and
//     writes tight, but not fewer than the wavefronts that fit the GPU at once.
//   - other recvs: 2048 workgroups, those that fit (4096 and 8192: 43.7 and 43.9 us against 42.1 at 16384 rows of 7 KB, one
//     chunk a lane).
// Two chunks a lane instead of one, one table entry instead of three words, whole split steps, us: 8 x 128 tokens of 14 KB
// bf16 rows 187.8 -> 184.1 (of 8 KB 147 -> 143, of 2 KB 105.5 -> 100.4), 8 x 512 of 7 KB 418.6 -> 407.4, one sender of 4096
// 367.1 -> 352.0, 8 x 2048 1391 -> 1362, 4 x 3000 983 -> 962.  In order or not (recv): 8 x 512 409.4 / 407.4, one sender of 4096
// (4096 rows a receiver) 353.7 / 352.0, 8 x 2048 (16384) 1362 / 1372, 4 x 3000 (24000) 962 / 969.  Four chunks a lane in
// the combine-send: 8 x 2048 1402 against 1380, the others level.
constexpr uint32_t kPieceWorkgroups = 2048;
constexpr uint32_t kInOrderRows = 8192;

uint32_t piece_grid(uint32_t max_rows, uint32_t world, uint32_t chunks, bool in_order, PieceGrid &grid) {
    constexpr uint32_t waves = kPieceThreads / kWave;
    grid.pieces = (chunks + kPieceChunks - 1) / kPieceChunks;
    const uint64_t most = ((uint64_t)max_rows * grid.pieces + waves - 1) / waves;
    uint64_t blocks = kPieceWorkgroups;
    if (in_order && most / world > blocks) blocks = most / world;
    if (blocks > 1u << 16) blocks = 1u << 16;   // (keeps wavefront numbers far below 2^32 / pieces)
    if (blocks > most) blocks = most;
    if (blocks < 1) blocks = 1;
    grid.magic = grid.pieces > 1 ? 0xFFFFFFFFu / grid.pieces + 1 : 0;
    grid.step_rows = (uint32_t)blocks * waves / grid.pieces;
    grid.step_pieces = (uint32_t)blocks * waves % grid.pieces;
    return (uint32_t)blocks;
}

// The launch that lays the receivers out and copies the caller's rows (first_recv_in_one_launch in a2a_rules.h).
constexpr uint32_t kFewRowWorkgroups = 512;

}  // namespace

int staging_allocate(Staging &st, const a2a_config &cfg, std::string *error) {
    if (st.allocated) return A2A_OK;
    const size_t N = cfg.world_size;
    const size_t K = cfg.num_experts_per_token;
    const size_t max_tk = (size_t)cfg.max_num_tokens * K;
    // The staged rows keep the reference's format (payload, scales, spare bytes: a2a_dispatch_send.cu:586-588)
    // at a stride rounded up to whole cache lines: the buffer is the library's own, and rows that begin in
    // the middle of a line cost every recv that reads them (4096 tokens: 120.7 -> 115.4 us for the recvs of
    // eight ranks).
    st.disp_stride = staged_row_stride((size_t)cfg.hidden_dim * cfg.in_elemsize, cfg.hidden_dim_scale);
    st.comb_stride = a2a_combine_token_stride(&cfg);
    st.payload_bytes = (uint32_t)align_up_sz((size_t)cfg.hidden_dim * cfg.in_elemsize, 16);
    st.max_tokens = cfg.max_num_tokens;
    // Rows of the per-receiver tables: what the caller sized a rank's receive region for
    // (max_recv_tokens), and never more than every copy of every sender.  A receiver that gets
    // more rows than that is flagged (A2A_DEV_RECV_OVERFLOW) and the rows beyond are dropped.
    size_t max_recv = N * max_tk;
    if (cfg.max_recv_tokens != 0 && cfg.max_recv_tokens < max_recv) max_recv = cfg.max_recv_tokens;
    if (max_recv > 0x7FFFFFFFull) {
        if (error) *error = "world_size * max_num_tokens * num_experts_per_token too large";
        return A2A_ERR_UNSUPPORTED;
    }
    st.max_recv = (uint32_t)max_recv;
    if (N * cfg.max_num_tokens > 0xFFFFFFFFull) {   // a staged row is named by sender * max_num_tokens + token
        if (error) *error = "world_size * max_num_tokens too large";
        return A2A_ERR_UNSUPPORTED;
    }

    size_t off = 0;
    auto carve = [&off](size_t bytes) {
        const size_t at = off;
        off = align_up_sz(off + bytes, 256);
        return at;
    };
    const size_t o_send = carve(N * cfg.max_num_tokens * st.disp_stride);
    const size_t o_pos = carve(N * max_tk * sizeof(uint32_t));
    const size_t o_comb = carve(N * max_tk * st.comb_stride);
    const size_t o_pidx = carve(N * max_recv * sizeof(uint32_t));
    const size_t o_srank = carve(N * max_recv * sizeof(uint32_t));
    const size_t o_spos = carve(N * max_recv * sizeof(uint32_t));
    const size_t o_sdo = carve(N * max_recv * sizeof(uint32_t));
    const size_t o_cso = carve(N * max_recv * sizeof(uint32_t));
    const size_t o_moves = carve(N * max_recv * sizeof(uint4));
    const size_t o_nrecv = carve(N * 2 * sizeof(uint32_t));
    hipError_t e = hipMalloc(&st.arena, off);
    if (e != hipSuccess) {
        if (error) {
            *error = "hipMalloc(staging, " + std::to_string(off) + " bytes): " + hipGetErrorString(e);
        }
        st.arena = nullptr;
        return A2A_ERR_OUT_OF_MEMORY;
    }
    uint8_t *base = static_cast<uint8_t *>(st.arena);
    st.send_buf = base + o_send;
    st.pos_token = reinterpret_cast<uint32_t *>(base + o_pos);
    st.comb_buf = base + o_comb;
    st.padded_index = reinterpret_cast<uint32_t *>(base + o_pidx);
    st.source_rank = reinterpret_cast<uint32_t *>(base + o_srank);
    st.source_position = reinterpret_cast<uint32_t *>(base + o_spos);
    st.source_dispatch_offset = reinterpret_cast<uint32_t *>(base + o_sdo);
    st.combine_send_offset = reinterpret_cast<uint32_t *>(base + o_cso);
    st.moves = reinterpret_cast<uint4 *>(base + o_moves);
    st.num_recv = reinterpret_cast<uint32_t *>(base + o_nrecv);
    // Tables are read before they are written only through misuse; start from zero.
    e = hipMemset(base + o_pos, 0, o_comb - o_pos);
    if (e == hipSuccess) e = hipMemset(base + o_pidx, 0, off - o_pidx);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        if (error) *error = std::string("hipMemset(staging): ") + hipGetErrorString(e);
        (void)hipFree(st.arena);
        st.arena = nullptr;
        return (int)e;
    }
    st.allocated = true;
    return A2A_OK;
}

void staging_free(Staging &st) {
    if (st.arena != nullptr) (void)hipFree(st.arena);
    st = Staging();
}

const uint32_t *staging_table(const Staging &st, const a2a_config &cfg, uint32_t rank, uint32_t which,
                              size_t *limit) {
    (void)cfg;
    if (!st.allocated || !(st.recv_mask >> rank & 1)) return nullptr;
    switch (which) {
        case A2A_TABLE_PADDED_INDEX:
            *limit = st.max_recv;
            return st.padded_index + (size_t)rank * st.max_recv;
        case A2A_TABLE_SOURCE_RANK:
            *limit = st.max_recv;
            return st.source_rank + (size_t)rank * st.max_recv;
        case A2A_TABLE_SOURCE_POSITION:
            *limit = st.max_recv;
            return st.source_position + (size_t)rank * st.max_recv;
        case A2A_TABLE_NUM_RECV_TOKENS:
            *limit = 2;
            return st.num_recv + (size_t)rank * 2;
        case A2A_TABLE_SOURCE_DISPATCH_OFFSET:
            *limit = st.max_recv;
            return st.source_dispatch_offset + (size_t)rank * st.max_recv;
        case A2A_TABLE_COMBINE_SEND_OFFSET:
            *limit = st.max_recv;
            return st.combine_send_offset + (size_t)rank * st.max_recv;
        default:
            return nullptr;
    }
}

hipError_t launch_stage_send(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                             bool quantize, hipStream_t stream, KernelTiming timing) {
    if (args.src.num_tokens == 0) return hipSuccess;
    const uint32_t threads = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    if (quantize) {
        hipExtLaunchKernelGGL(stage_send_kernel<true>, dim3(args.src.num_tokens), dim3(threads), 0, stream,
                              timing.start, timing.stop, 0, args, ws, st);
    } else {
        hipExtLaunchKernelGGL(stage_send_kernel<false>, dim3(args.src.num_tokens), dim3(threads), 0, stream,
                              timing.start, timing.stop, 0, args, ws, st);
    }
    return hipGetLastError();
}

bool stage_send_small_fits(const StageSendArgs &args, const Workspace &ws) {
    const uint64_t T = args.src.num_tokens;
    const uint64_t entries = T * ws.topk;
    return T != 0 && entries <= kSmallMaxEntries && entries * T <= kSmallMaxVisits;
}

hipError_t launch_stage_send_small(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                   bool quantize, hipStream_t stream, KernelTiming timing) {
    // The quick form: dense index rows, a piece of the row per thread and a wavefront beside them.
    const uint32_t pieces = quantize ? args.hidden_dim / 16 : args.row_bytes / 16;
    if (args.src.indices_stride == ws.topk && pieces + kWave <= 1024) {
        const uint32_t counters = (pieces + kWave - 1) / kWave * kWave;
        const uint32_t per_thread = (args.src.num_tokens * ws.topk + counters - 1) / counters;
        const size_t quick_lds = (size_t)ws.num_experts * sizeof(uint32_t);
        const size_t g = args.rank / ws.dp_size;
        SendQuickArgs q;
        q.x = args.src.x;
        q.x_scale = args.src.x_scale;
        q.indices = args.src.indices;
        q.bound_m = args.src.bound_m;
        q.x_stride = args.src.x_stride;
        q.staged = st.send_buf + g * st.max_tokens * st.disp_stride;
        q.pos_token = st.pos_token + g * ws.max_tk;
        q.num_routed = ws.num_routed + g * ws.num_experts;
        q.token_offset = ws.token_offset + g * ws.max_tk;
        q.route_slot = ws.route_slot + g * ws.max_tk;
        q.xs_stride_elem = args.src.xs_stride_elem;
        q.xs_stride_token = args.src.xs_stride_token;
        q.num_tokens = args.src.num_tokens;
        q.num_scales = args.hidden_dim_scale;
        q.sizes = pieces | ws.num_experts << 10 | ws.topk << 21;
        const ptrdiff_t to_offsets = ws.expert_offsets - ws.num_routed, to_flags = ws.err - q.num_routed;
        if (to_offsets % kTableUnit != 0 || !fits_field(to_offsets / kTableUnit, 10) || !fits_field(to_flags, 22))
            return hipErrorInvalidValue;
        q.distances = (uint32_t)to_offsets / kTableUnit | (uint32_t)to_flags << 10;
#define A2A_LAUNCH_SEND_QUICK(NB)                                                                                    \
    do {                                                                                                             \
        if (quantize)                                                                                                \
            hipExtLaunchKernelGGL((stage_send_quick_kernel<NB, true>), dim3(args.src.num_tokens),                    \
                                  dim3(counters + kWave), quick_lds, stream, timing.start, timing.stop, 0, q);       \
        else                                                                                                         \
            hipExtLaunchKernelGGL((stage_send_quick_kernel<NB, false>), dim3(args.src.num_tokens),                   \
                                  dim3(counters + kWave), quick_lds, stream, timing.start, timing.stop, 0, q);       \
    } while (0)
        if (per_thread <= 1) A2A_LAUNCH_SEND_QUICK(1);
        else if (per_thread <= 2) A2A_LAUNCH_SEND_QUICK(2);
        else if (per_thread <= 3) A2A_LAUNCH_SEND_QUICK(3);
        else if (per_thread <= 4) A2A_LAUNCH_SEND_QUICK(4);
        else A2A_LAUNCH_SEND_QUICK(8);
#undef A2A_LAUNCH_SEND_QUICK
        return hipGetLastError();
    }
    const uint32_t threads = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    const size_t lds = 3 * (size_t)ws.num_experts * sizeof(uint32_t);
    if (quantize) {
        hipExtLaunchKernelGGL(stage_send_small_kernel<true>, dim3(args.src.num_tokens), dim3(threads), lds, stream,
                              timing.start, timing.stop, 0, args, ws, st);
    } else {
        hipExtLaunchKernelGGL(stage_send_small_kernel<false>, dim3(args.src.num_tokens), dim3(threads), lds, stream,
                              timing.start, timing.stop, 0, args, ws, st);
    }
    return hipGetLastError();
}

uint32_t send_single_tokens_per_group(uint32_t tokens) {
    constexpr uint32_t kComputeUnits = 256;
    const uint32_t per_group = (tokens + kComputeUnits - 1) / kComputeUnits;
    return per_group < 1 ? 1 : per_group > kSendTokensPerGroup ? kSendTokensPerGroup : per_group;
}

bool stage_send_single_fits(const StageSendArgs &args, const Workspace &ws, bool quantize) {
    const uint64_t T = args.src.num_tokens;
    const uint32_t team = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    const uint32_t per_group = send_single_tokens_per_group((uint32_t)T);
    uint32_t teams = 1024 / team;
    if (teams > per_group) teams = per_group;
    // dense index rows (the entries are read as one flat array), one thread per route of a workgroup's tokens
    return T != 0 && T * ws.topk <= kSendSingleMaxEntries && args.src.indices_stride == ws.topk &&
           per_group * ws.topk <= teams * team;
}

hipError_t launch_stage_send_single(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                    bool quantize, hipStream_t stream, KernelTiming timing) {
    const uint32_t team = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    const uint32_t per_group = send_single_tokens_per_group(args.src.num_tokens);
    uint32_t teams = 1024 / team;
    if (teams > per_group) teams = per_group;
    const uint32_t blocks = (args.src.num_tokens + per_group - 1) / per_group;
    {
        // With a spare wavefront beside the teams, rows of one piece per thread of a team, a lane of
        // the spare wavefront per route of a workgroup's tokens and at most two rounds: the kernel in
        // which the teams do not wait for the routes.
        const uint32_t pieces = quantize ? args.hidden_dim / 16 : args.row_bytes / 16;
        uint32_t spare_teams = (1024 - kWave) / team;
        if (spare_teams > per_group) spare_teams = per_group;
        const uint32_t rounds = spare_teams != 0 ? (per_group + spare_teams - 1) / spare_teams : 3;
        if (pieces <= team && per_group * ws.topk <= (uint32_t)kWave && rounds <= 2) {
            const uint32_t counters = spare_teams * team;
            const uint32_t per_thread = (args.src.num_tokens * ws.topk + counters - 1) / counters;
            const size_t teams_lds = (size_t)ws.num_experts * sizeof(uint32_t);
#define A2A_LAUNCH_SEND_TEAMS(NB, ROUNDS)                                                                            \
    do {                                                                                                             \
        if (quantize)                                                                                                \
            hipExtLaunchKernelGGL((stage_send_teams_kernel<NB, ROUNDS, true>), dim3(blocks),                         \
                                  dim3(counters + kWave), teams_lds, stream, timing.start, timing.stop, 0, args,     \
                                  ws, st, team, per_group);                                                          \
        else                                                                                                         \
            hipExtLaunchKernelGGL((stage_send_teams_kernel<NB, ROUNDS, false>), dim3(blocks),                        \
                                  dim3(counters + kWave), teams_lds, stream, timing.start, timing.stop, 0, args,     \
                                  ws, st, team, per_group);                                                          \
    } while (0)
#define A2A_LAUNCH_SEND_TEAMS_NB(ROUNDS)                                                                             \
    do {                                                                                                             \
        if (per_thread <= 4) A2A_LAUNCH_SEND_TEAMS(4, ROUNDS);                                                       \
        else if (per_thread <= 8) A2A_LAUNCH_SEND_TEAMS(8, ROUNDS);                                                  \
        else if (per_thread <= 10) A2A_LAUNCH_SEND_TEAMS(10, ROUNDS);                                                \
        else A2A_LAUNCH_SEND_TEAMS(16, ROUNDS);                                                                      \
    } while (0)
            if (rounds <= 1) A2A_LAUNCH_SEND_TEAMS_NB(1);
            else A2A_LAUNCH_SEND_TEAMS_NB(2);
#undef A2A_LAUNCH_SEND_TEAMS_NB
#undef A2A_LAUNCH_SEND_TEAMS
            return hipGetLastError();
        }
    }
    const size_t lds = 2 * (size_t)ws.num_experts * sizeof(uint32_t);
    if (quantize) {
        hipExtLaunchKernelGGL(stage_send_single_kernel<true>, dim3(blocks), dim3(teams * team), lds, stream,
                              timing.start, timing.stop, 0, args, ws, st, team, per_group);
    } else {
        hipExtLaunchKernelGGL(stage_send_single_kernel<false>, dim3(blocks), dim3(teams * team), lds, stream,
                              timing.start, timing.stop, 0, args, ws, st, team, per_group);
    }
    return hipGetLastError();
}

bool stage_send_beside_fits(const StageSendArgs &args, const Workspace &ws) {
    return args.src.num_tokens != 0 && args.src.indices_stride == ws.topk &&
           (uint64_t)args.src.num_tokens * ws.topk <= kSendBesideMaxEntries;
}

hipError_t launch_stage_send_beside(const StageSendArgs &args, const Workspace &ws, const Staging &st, bool quantize,
                                    hipStream_t stream, KernelTiming timing) {
    const uint32_t team = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    const uint32_t teams = team < 512 ? 512 / team : 1;
    const uint32_t threads = teams * team;
    const uint32_t chunks = (args.src.num_tokens * ws.topk + threads - 1) / threads;
    const uint32_t blocks = chunks + (args.src.num_tokens + teams - 1) / teams;
    const size_t lds = (size_t)ws.num_experts * (2 * sizeof(uint32_t) + threads / kWave * sizeof(uint16_t));
    if (quantize) {
        hipExtLaunchKernelGGL(stage_send_beside_kernel<true>, dim3(blocks), dim3(threads), lds, stream, timing.start,
                              timing.stop, 0, args, ws, st, team, chunks);
    } else {
        hipExtLaunchKernelGGL(stage_send_beside_kernel<false>, dim3(blocks), dim3(threads), lds, stream, timing.start,
                              timing.stop, 0, args, ws, st, team, chunks);
    }
    return hipGetLastError();
}

hipError_t launch_stage_send_resolve(const StageSendArgs &args, const Workspace &ws, const Staging &st,
                                     bool quantize, hipStream_t stream, KernelTiming timing) {
    uint32_t threads = block_for_chunks(quantize ? args.hidden_dim / 16 : args.row_bytes / 16);
    const uint32_t blocks = args.src.num_tokens + 1;
    StageSendArgs a = args;
    a.resolver_wave = 0;
    if (threads + kWave <= 1024) {   // a wavefront of its own for the routes (measured: 27.3 against 28.5 us)
        a.resolver_wave = threads / kWave;
        threads += kWave;
    }
    if (quantize) {
        hipExtLaunchKernelGGL(stage_send_resolve_kernel<true>, dim3(blocks), dim3(threads), 0, stream, timing.start,
                              timing.stop, 0, a, ws, st);
    } else {
        hipExtLaunchKernelGGL(stage_send_resolve_kernel<false>, dim3(blocks), dim3(threads), 0, stream, timing.start,
                              timing.stop, 0, a, ws, st);
    }
    return hipGetLastError();
}

hipError_t launch_stage_recv(const StageRecvArgs &args, const Workspace &ws, const Staging &st, bool first_of_step,
                             hipStream_t stream, KernelTiming timing, KernelTiming layout_timing) {
    const uint32_t chunks = args.row_bytes / 16;
    const size_t items = (size_t)ws.num_groups * ws.experts_per_rank;
    const size_t lds = (5 * items + 1 + 3 * (size_t)ws.num_groups + ws.experts_per_rank) * sizeof(uint32_t);
    const uint32_t typical = (args.max_rows + ws.world - 1) / ws.world;
    StageRecvArgs a = args;
    const uint32_t threads = block_for_chunks(chunks);
    if (first_of_step && first_recv_in_one_launch(typical, args.row_bytes, (uint32_t)items, threads)) {
        uint32_t blocks = args.max_rows < kFewRowWorkgroups ? args.max_rows : kFewRowWorkgroups;
        if (blocks == 0) blocks = 1;    // the counts are handed over even when nothing was sent
        // Beside the caller's workgroups: a few per other receiver, enough threads for the rows a receiver
        // typically gets (1/N of the host's upper bound); each repeats that receiver's layout in LDS.
        a.copy_blocks = blocks;
        a.slices = (typical + threads - 1) / threads;
        if (a.slices < 1) a.slices = 1;
        if (a.slices > 16) a.slices = 16;
        hipExtLaunchKernelGGL(stage_recv_first_few_kernel, dim3(blocks + (ws.world - 1) * a.slices), dim3(threads),
                              lds, stream, timing.start, timing.stop, 0, a, ws, st);
        return hipGetLastError();
    }
    if (first_of_step) {
        constexpr uint32_t layout_threads = 512;
        a.slices = (typical + layout_threads - 1) / layout_threads;
        if (a.slices < 1) a.slices = 1;
        if (a.slices > 32) a.slices = 32;
        hipExtLaunchKernelGGL(stage_layout_kernel, dim3(ws.world * a.slices), dim3(layout_threads), lds, stream,
                              layout_timing.start, layout_timing.stop, 0, a, ws, st);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    PieceGrid grid;
    const uint32_t blocks = piece_grid(args.max_rows, ws.world, chunks, typical >= kInOrderRows, grid);
    const uint32_t first = args.rank * ws.experts_per_rank;
    RecvRowsArgs m;
    m.out_x = args.dst.out_x;
    m.out_scale = args.dst.out_scale;
    m.out_num_tokens = args.out_num_tokens;
    m.staged = st.send_buf;
    m.moves = st.moves + (size_t)args.rank * st.max_recv;
    m.num_recv = st.num_recv + 2 * args.rank;
    m.counts = ws.tokens_per_expert + first;
    m.out_stride = args.dst.out_stride;
    m.os_stride_elem = args.dst.os_stride_elem;
    m.os_stride_token = args.dst.os_stride_token;
    m.out_rows = args.dst.out_rows;
    m.row_bytes = args.row_bytes;
    m.num_scales = args.hidden_dim_scale;
    m.max_recv = st.max_recv;
    m.pieces = grid.pieces;
    m.magic = grid.magic;
    m.step_rows = grid.step_rows;
    m.step_pieces = grid.step_pieces;
    m.num_local = first >= ws.num_experts ? 0 : std::min(ws.num_experts - first, ws.experts_per_rank);
    const ptrdiff_t to_first_rows = ws.padded_offset - ws.tokens_per_expert, to_flags = m.counts - ws.err;
    if (to_first_rows % kTableUnit != 0 || !fits_field(to_first_rows / kTableUnit, 5) || !fits_field(to_flags, 16))
        return hipErrorInvalidValue;
    m.to_first_rows = (uint32_t)to_first_rows / kTableUnit;
    m.to_flags = (uint32_t)to_flags;
    // Scales by column: a wavefront for every kScaleColumns columns of 64 rows that the receiver typically gets.
    const bool columns = args.dst.out_x != nullptr && scales_by_column(args.dst) &&
                         (uint64_t)typical * args.hidden_dim_scale >= kColumnWords;
    m.scale_blocks = 0;
    if (columns) {
        const uint64_t units = ((uint64_t)typical + kWave - 1) / kWave *
                               ((args.hidden_dim_scale + kScaleColumns - 1) / kScaleColumns);
        const uint64_t blocks_of_units = (units + kPieceThreads / kWave - 1) / (kPieceThreads / kWave);
        m.scale_blocks = blocks_of_units < 1 ? 1 : blocks_of_units < kPieceWorkgroups ? (uint32_t)blocks_of_units : kPieceWorkgroups;
    }
#define A2A_LAUNCH_RECV(STREAM, COLUMNS)                                                                            \
    hipExtLaunchKernelGGL((stage_recv_kernel<STREAM, COLUMNS>), dim3(blocks + m.scale_blocks), dim3(kPieceThreads), 0, \
                          stream, timing.start, timing.stop, 0, m)
    if (args.streamed) {
        if (columns) A2A_LAUNCH_RECV(true, true); else A2A_LAUNCH_RECV(true, false);
    } else {
        if (columns) A2A_LAUNCH_RECV(false, true); else A2A_LAUNCH_RECV(false, false);
    }
#undef A2A_LAUNCH_RECV
    return hipGetLastError();
}

hipError_t launch_combine_send(const CombineSendArgs &args, uint32_t rank, uint32_t max_rows, const Workspace &ws,
                               const Staging &st, hipStream_t stream, KernelTiming timing) {
    if (max_rows == 0) return hipSuccess;
    const uint32_t chunks = args.row_bytes / 16;
    CombineSendArgs a = args;
    a.staged = st.comb_buf;
    a.staged_stride = st.comb_stride;
    a.moves = st.moves + (size_t)rank * st.max_recv;
    a.num_recv = st.num_recv + 2 * rank;
    a.err = ws.err;
    a.max_recv = st.max_recv;
    a.max_tk = ws.max_tk;
    const uint32_t blocks = piece_grid(max_rows, ws.world, chunks, true, a.grid);
    hipExtLaunchKernelGGL(combine_send_kernel, dim3(blocks), dim3(kPieceThreads), 0, stream, timing.start, timing.stop,
                          0, a);
    return hipGetLastError();
}

hipError_t launch_combine_recv(const CombineRecvArgs &args, const Workspace &ws, const Staging &st,
                               uint32_t in_dtype, uint32_t out_dtype, hipStream_t stream, KernelTiming timing) {
    const size_t g = args.rank / ws.dp_size;
    CombineStagedArgs a;
    a.out = args.dst.out;
    a.indices = args.dst.indices;
    a.weights = args.dst.weights;
    a.bound_m = args.dst.bound_m;
    a.route_slot = ws.route_slot + g * ws.max_tk;
    a.staged = st.comb_buf + g * ws.max_tk * st.comb_stride;
    a.err = ws.err;
    a.out_stride = args.dst.out_stride;
    a.staged_stride = st.comb_stride;
    a.indices_stride = args.dst.indices_stride;
    a.weights_stride = args.dst.weights_stride;
    a.num_tokens = args.dst.num_tokens;
    a.layer_rows = 0;
    a.max_tk = ws.max_tk;
    a.hidden_dim = args.hidden_dim;
    a.num_experts = ws.num_experts;
    a.topk = ws.topk;
    a.accumulate = args.accumulate;
    return launch_combine_staged(a, in_dtype, out_dtype, stream, timing);
}

}  // namespace a2a
