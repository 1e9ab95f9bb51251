// Rules of the launchers that depend on sizes alone: plain host code, checked without a GPU.
#pragma once

#include <cstdint>

namespace a2a {

// The combine's grid: `layers` of `rows` tokens, as even as they come, so that no more than layers - 1 rows are
// empty; one layer is as large as the grid's second dimension takes.  Empty workgroups cost what they cost: with full
// layers 33 000 tokens were a grid of 65 536, 352.1 us against 236.8 (K = 2, hidden 7168; 32 768 tokens 236.5) and
// 258.9 against 207.1 (K = 8, hidden 2048), 66 000 tokens 585.6 against 469.3.
constexpr uint32_t kTokensPerLayer = 32768;

struct TokenLayers {
    uint32_t layers, rows;
};

inline TokenLayers token_layers(uint32_t tokens) {
    TokenLayers t;
    t.layers = (uint32_t)(((uint64_t)tokens + kTokensPerLayer - 1) / kTokensPerLayer);
    if (t.layers < 1) t.layers = 1;
    t.rows = (uint32_t)(((uint64_t)tokens + t.layers - 1) / t.layers);
    return t;
}

// Whether a wavefront of the gather moves two slabs of a token's row instead of one.  With one or two copies a token a slab is
// one or two loads a lane behind a chain of arguments, ids and places: all the wavefronts that fit have too few of them in flight,
// and the dispatcher starts no more than some 4300 a us.  us per combine, bf16 rows unless said otherwise, one slab / two / four:
//                          K = 1                    K = 2                    K = 4
//    8 x 3000 of 2 KB    24.9 /  19.8 /  20.4     28.8 /  28.0 /  29.6     42.8 /  43.3 /  43.5
//             of 5.9 KB  67.1 /  48.6 /  55.0     74.6 /  70.7 /  76.2    115.5 / 118.7 / 125.3
//             of 8 KB    88.4 /  66.7 /  68.5     99.9 /  97.8 /  99.8    163.3 / 166.9 / 168.1
//             of 14 KB  137.2 / 114.7 / 121.4    174.1 / 169.6 / 174.2
//    8 x 800  of 8 KB    26.3 /  21.0 /  21.4     30.4 /  29.5 /  29.3     45.4 /  45.9 /  46.1
//        float of 28 KB  72.9 /  63.1 /  63.7     93.3 /  91.1 /  93.0    149.0 / 152.7 / 157.7
//    8 x 200  of 5.9 KB   7.9 /   6.7 /   6.8      8.4 /   8.0 /   8.4     11.1 /  10.9 /  11.6
//    8 x 40   of 8 KB     4.4 /   3.8 /   3.9      4.6 /   4.1 /   4.2      5.1 /   4.8 /   5.0
//             of 4 KB     3.45 /  3.47 /  3.63     3.5 /   3.7 /   3.9      (1280 wavefronts)
//    8 x 4    of 14 KB    3.2 /   3.35 /  3.45     3.3 /   3.3 /   3.6      (448)
// Eight copies lose 1 to 6 % with two.  Steps of few wavefronts end with the chain, which is shorter with one slab.
constexpr uint64_t kFewSlabs = 1536;

inline bool two_pieces_a_lane(uint32_t topk, uint64_t slabs) { return topk <= 2 && slabs > kFewSlabs; }

// Cache policy of a large step's copies and of its combined tokens.  From kStreamCopies bytes of copies on the pack
// sends them past the 256 MB Infinity Cache (device scope and non-temporal) and the combine sends its tokens past it
// too: such a step cannot stay there until it is read, and lines that are not left dirty need not be written back
// while the next kernels read.  Below the line copies stay where the experts, which read them next, find them.
// Whole steps, us, copies kept / past the cache, with nothing between dispatch and combine (no user's step; their
// difference is the writing back that the combine no longer waits for), with a sweep that reads the received rows, and
// with one that reads them and writes expert_y (buffers not those of the step before):
//   quantised rows of 7168 bytes, K = 8
//      117 MB   79.3 /  82.7    136.3 / 139.8     507.2 /  525.3
//      235 MB  162.1 / 153.8    245.2 / 248.5     954.7 /  958.5
//      355 MB  240.0 / 228.2    365.1 / 359.6    1392.1 / 1385.7
//     1879 MB 1251.2 / 1185.0  2377.8 / 2330.1   11770.7 / 11731.8
//   fp8 rows of 5120 bytes, K = 8
//      109 MB   81.5 /  78.2    130.3 / 133.1     455.7 /  476.4
//      307 MB  215.1 / 203.1    329.8 / 324.2    1197.5 / 1188.5
//      983 MB  648.3 / 595.5    951.3 / 916.9    3409.3 / 3379.9
//   bf16 rows of 8 KB, K = 6 (the ones that gain least)
//      201 MB   96.2 /  91.2    158.6 / 166.5     193.3 /  186.0
//      295 MB  139.1 / 132.3    231.0 / 235.2     276.5 /  270.2
//      344 MB  158.6 / 150.2    267.4 / 267.3     315.8 /  307.3
//      786 MB  352.8 / 338.0    585.2 / 593.0     707.9 /  693.7
//     1573 MB  690.0 / 649.9   1136.0 / 1113.1   1439.6 / 1424.5
// One goes with the other (copies kept, tokens into the cache instead: up to 11 us more), so the pack decides and the
// combine follows what the pack did.  Rows that are not quantised and have at most two copies are kept at every size
// (rows of 2 KB, K = 1: 44.0 us against 46.6 past the cache; 8 KB, K = 2: 91.0 against 94.5).
constexpr uint64_t kStreamCopies = 320000000;

inline bool copies_past_cache(uint64_t copies, bool quantize, uint32_t topk) {
    return copies >= kStreamCopies && (quantize || topk > 2);
}

// Whether copies that stay in the Infinity Cache, are not quantised and bring no scales are stored at device scope.  Ordinary
// stores leave them dirty in eight L2s, which write them back in an order of their own; written through, they reach memory as
// the rows are worked off, but every store is held until it is there.  What decides is how much of its last 4 KB a row fills
// (an L2's 16 channels of 256 bytes repeat after 4 KB: the fuller the rows, the more evenly the stores of a workgroup lie on
// them) and how many copies a load feeds.  us per step whose buffers are not those of the step before, ordinary / written
// through, with nothing between dispatch and combine | with a sweep that reads the received rows | with one that reads them
// and writes expert_y:
//                        K = 6, 280 MB                                K = 8, 280 MB
//    4608 bytes  131.9 / 136.5 | 236.1 / 240.1 | 263.6 / 266.0  122.4 / 124.4 | 228.5 / 231.2 | 260.1 / 262.2
//    6144        125.5 / 127.4 | 231.2 / 234.2 | 259.4 / 262.2  124.7 / 119.3 | 226.0 / 228.3 | 254.6 / 256.9
//    7168        127.9 / 124.8 | 230.9 / 232.5 | 258.8 / 260.6  125.9 / 120.9 | 226.2 / 226.9 | 257.6 / 258.7
//    8192        130.6 / 125.8 | 228.7 / 229.0 | 258.2 / 255.8  126.5 / 122.3 | 229.0 / 227.0 | 259.8 / 257.1
//    9216        125.1 / 126.1 | 235.8 / 236.5 | 263.6 / 264.9  124.7 / 119.7 | 230.9 / 231.8 | 265.3 / 265.1
//   10240        125.1 / 124.8 | 234.2 / 235.5 | 263.7 / 265.1  125.6 / 120.3 | 230.9 / 231.2 | 264.0 / 264.3
//   12288        129.9 / 123.9 | 231.1 / 231.0 | 261.4 / 260.7  125.7 / 121.3 | 231.5 / 230.4 | 263.9 / 262.5
//   12800        126.6 / 126.6 | 240.8 / 241.4 | 273.9 / 274.4  122.8 / 119.5 | 235.0 / 235.4 | 271.8 / 270.4
//   28672        129.7 / 125.7 | 249.3 / 245.5 | 281.9 / 279.7  123.9 / 122.1 | 249.9 / 248.9 | 285.8 / 284.7
// Of 23 lengths between 4096 and 28672 bytes, K = 6 to 8, nothing between, every one with topk * (share of whole 4 KB filled)
// of at least 5 is level or gains, up to 5 %, and every one below is level or loses, up to 3.4 %; K = 7 turns at 5888 bytes
// (0.719).  Behind a sweep the rows that are less than three quarters full lose 1 to 1.7 % also with K = 8 (5120: 224.1 /
// 228.0), those above lie between -1 and +2 %.  Steps over the same buffers again and again, as no user's are, gain less or
// lose: 280 MB of 8 KB 110.8 / 110.6, of 4 KB 112.8 / 116.0.
// It loses with few copies a token (K = 4 behind a reader 245.6 / 247.4; not where a thread moves several pieces,
// pieces_per_lane, which are written through at every size: fp8 rows of 5 KB, K = 4 73.9 / 73.5, bf16 of 14 KB, K = 1 275 / 267,
// behind a reader 391 / 384), with rows of 2 KB (131.7 / 134.1), with rows that
// bring scales (fp8 rows of 5120 bytes 75.3 / 77.5, of 4096 behind a reader 300 / 308), and below kWrittenThrough bytes of copies
// (4 KB rows, 79 MB: dispatch 24.0 / 24.9; 108 MB level).
constexpr uint64_t kWrittenThrough = 120000000;

inline bool copies_written_through(uint64_t copies, uint32_t row_bytes, uint32_t topk) {
    constexpr uint64_t kPeriod = 4096;
    const uint64_t whole = (row_bytes + kPeriod - 1) / kPeriod * kPeriod;
    return copies >= kWrittenThrough && topk >= 6 && row_bytes >= kPeriod && 4ull * row_bytes >= 3 * whole &&
           (uint64_t)topk * row_bytes >= 5 * whole;
}

// Sixteen-byte pieces of a copy that a thread of the resolving pack moves, and with it the wavefronts of a token's workgroup.
// All of a workgroup's wavefronts are held through the chain of look-ups that ends in the rows' places, and a token with few
// copies brings few bytes for it: with a piece a thread and one or two copies the pack ran at 3.0 to 3.8 TB/s where a push of
// the same rows without any look-ups does 5.4.  Fewer wavefronts a token are more tokens in flight.  With many copies it is
// the rows held open at a time that cost.  us per step, ordinary rows with one piece (what there was before) / 1, 2 and 4
// pieces, all at device scope:
//                     K = 1                     K = 2                     K = 4                     K = 6
//    bf16  2 KB   80.7 /  81  68  68       94.4 /  98  85  85       94.1 /  96  92  92       88.3 /  89  87  87
//    bf16  4 KB  142.5 / 147 120 116      116.9 / 121 106 108       91.3 /  92  92  93       84.5 /  84  87  87
//    bf16  5.9 KB 233.0 / 236 165 157     139.6 / 139 107 108       99.6 / 101  91  92       86.9 /  88  87  87
//    bf16 14 KB  301.7 / 299 216 196      197.1 / 192 152 155      138.4 / 138 131 133      147.6 / 147 156 158
//    f32  28 KB  458.9 / 469 440 381      320.7 / 320 297 300      289.3 / 289 299 304      292.5 / 293 300 304
//    fp8   5 KB  273.3 / 283 219 205      188.4 / 197 158 156      140.2 / 146 132 132      126.6 / 132 127 126
//    fp8   7 KB  297.4 / 296 235 222      186.6 / 188 156 157      140.6 / 142 131 132      129.5 / 129 126 126
//    quantised 4 KB 217 / 217 195 195     175.8 / 176 169 170      135.7 / 136 137 139      126.1 / 126 128 129
//    quantised 5 KB 302 / 297 236 232     202.8 / 200 172 173      144.8 / 145 140 141      130.5 / 130 131 132
//    quantised 7 KB 312 / 307 257 253     191.1 / 189 170 173      141.6 / 140 138 141      128.4 / 129 131 132
// and with a sweep between dispatch and combine that reads the received rows, before / as it is: K = 1, bf16 rows of 14 KB
// 535 / 385, quantised of 7 KB 372 / 316; K = 2, bf16 of 5.9 KB 169 / 144, fp8 of 7 KB 243 / 215; K = 4, fp8 of 5 KB
// 125.5 / 120.7, bf16 of 14 KB 253 / 236.  (K = 2 with rows of 28 KB: two pieces 461, four 438.)
// K = 3, 8 x 2000 tokens, before / as it is: bf16 of 2 KB 60.9 / 56.5, 5.9 KB 168 / 143, 14 KB 374 / 323; f32 of 16 KB 403 / 377; fp8 of
// 5 KB 204 / 182; quantised of 4 KB 158.2 / 156.6, 7 KB 279 / 257.  Copies that go past the Infinity Cache: quantised of 7 KB,
// 16 x 4096, K = 1 810 / 594, 8 x 3000, K = 3 413 / 380; fp8 of 5 KB, 8 x 4096, K = 3 406 / 342; bf16 of 5.9 KB, 8 x 4096, K = 4 396 / 358.
// Four copies a token: two pieces where a piece a thread makes workgroups that do not fill a compute unit's 32 places for
// wavefronts (3, 5, 6, 7, 14 of them, not 1, 4, 8 or 16), and for the shortest unquantised rows; not where scales go out by
// column, which workgroups of fewer than 256 threads leave to the rows (fp8 rows of 2944 bytes 116.6 / 121.5, of 5120 level;
// with K = 1 and 2 the pieces gain more than that: 158 / 136 and 150 / 138).
// A workgroup has a thread per local expert in any case.  Where these are as many as pieces, several pieces a thread make no
// wavefront fewer and the stores at device scope cost 1 to 4 %.  us per dispatch of 2 x 12 000 tokens, several pieces / one: 128
// local experts, bf16 of 2 KB, K = 1, 2, 4 47.1 / 46.1, 57.0 / 55.4, 74.8 / 72.8; 256, bf16 of 1.3 KB 79.8 / 77.6, 92.7 / 89.6,
// 111.1 / 107.0, fp8 of 4 KB, K = 1, 2 98.0 / 94.5, 119.7 / 118.5; 512, fp8 of 5 KB 217.6 / 210.5, 262.1 / 257.2, 309.6 / 315.5,
// float of 8 KB, K = 1, 2 218.0 / 217.1, 264.7 / 266.9.  The last of the fp8 and of the float rows lie
// beyond kLongCopies: with 16 KB of copies a token and more the stores at device scope are level or gain.  (Quantised rows, at
// device scope either way: level.)
// Rows of at most 64 pieces have one wavefront in any case too and gain by the stores: us per step, several pieces / one, K = 1,
// 2, 3, bf16 of 1 KB 48.7 / 49.7, 43.3 / 44.2, 49.6 / 50.5, of 512 bytes 46.4 / 47.7, 39.1 / 39.9, 40.6 / 41.7; fp8 of 1 KB
// 59.9 / 60.0, 57.8 / 57.9, 67.8 / 68.6.
constexpr uint32_t kLongCopies = 1024;   // pieces of a token's copies

inline uint32_t pieces_per_lane(uint32_t topk, uint32_t chunks, bool quantize, bool by_column, uint32_t experts_per_rank) {
    const bool held = chunks > 64 && chunks <= (experts_per_rank + 63) / 64 * 64;
    if (held && topk * chunks < kLongCopies) return 1;
    if (topk == 1) return 4;
    if (topk <= 3) return chunks > 1024 ? 4 : 2;
    if (topk > 4 || by_column) return 1;
    const uint32_t waves = (chunks + 63) / 64;
    const bool fills = waves > 16 || (waves & (waves - 1)) == 0;
    return !fills || (!quantize && waves == 2) ? 2 : 1;
}

// Whether a step of eight copies a token that the one launch of several sources can hold with a workgroup per compute unit, of
// `one` > 4 tokens each, has two per compute unit instead, of `two` tokens.  With up to 32 routes a workgroup's resolver has two
// lanes a route, with up to 64 one, and what a route waits for last is the sum over the earlier experts of its receiver, four of
// them a lane and the others one after another.  So two workgroups gain the more the more experts a receiver has, and while
// `two` <= 4.  Against that stand the tables that more workgroups count, and quantised rows, which want their tokens spread
// evenly: six on a compute unit with two workgroups of three where one has five.  us per step, one / two:
//   quantised 4 KB, E experts   8 x 130  E = 64 27.6 / 28.2, 256 28.7 / 26.6;  4 x 290  E = 64 29.9 / 29.5;
//                               16 x 65  E = 64 27.8 / 28.5, 256 28.4 / 28.4;  8 x 159  E = 64 31.0 / 31.5, 256 32.0 / 29.8
//             3 KB              8 x 130  E = 64 22.6 / 23.2, 256 23.7 / 22.0;  one source of 1400, E = 64 27.1 / 26.4
//             5 KB              8 x 145  E = 64 34.6 / 35.1, 256 35.6 / 33.0;  8 x 180, E = 128 41.0 / 39.4
//             2 KB, 6 KB, 7 KB  8 x 160  E = 64 20.5 / 20.3, 42.5 / 41.8, 48.6 / 46.8;  four tokens a workgroup, 7 KB 58.1 / 59.0
//   bf16 2 KB, 4 KB, 7 KB, 8 KB 8 x 160  E = 64 15.7 / 14.2, 22.0 / 20.5, 33.8 / 31.6, 37.8 / 35.1
//   fp8  2 KB, 5 KB, 7 KB       8 x 160  E = 64 19.8 / 18.4, 36.1 / 34.1, 47.0 / 46.3
// (The few that lose all the same: uneven loads with few experts a receiver, one / two for 460, 0, 153, 1, ... tokens, E = 64, 3 KB
// 25.4 / 25.1, 4 KB 30.7 / 30.4.)
// Four tokens of four units each are two rounds of eight wavefronts, too few to count for many sources: bf16 of 4 KB, 8 x 220
// 28.9 / 28.1, 16 x 110 28.3 / 28.8.  2048 tokens are more than two workgroups of four on each compute unit, and with five routes
// have a lane each: short rows lose (8 x 256: bf16 of 2 KB 19.6 / 20.5, of 3 KB 25.4 / 25.8, 4 KB level, 5 KB 38.2 / 37.4, 7 KB
// 50.0 / 49.7; fp8 of 2 KB 26.7 / 27.4; but 16 x 128, E = 384, bf16 of 2 KB 22.6 / 21.2, fp8 29.2 / 28.4), and with scales longer
// ones whose receivers have few experts (fp8 of 4 KB, 8 x 256, E = 64 44.8 / 45.1, 256 46.2 / 45.6, 2 x 1024, E = 64 47.8 / 46.8;
// 5 KB 53.4 / 54.2, 54.8 / 53.8, 53.9 / 52.8; 6 KB 60.7 / 61.4, 62.4 / 61.6, 62.6 / 61.9).
inline bool two_workgroups_a_unit(bool quantize, bool scaled, uint32_t one, uint32_t two, uint32_t units, uint32_t experts_per_rank,
                                  uint32_t senders) {
    if (quantize) return two <= 3 && (one > 5 || experts_per_rank > 8 || units < 3 || units > 5);
    if (two <= 4) return two * units != 16 || senders <= 8;
    if (units < 4) return senders > 8 && experts_per_rank > 16;
    return !scaled || units > 5 || experts_per_rank > 16;
}

// copies_past_cache for the recvs of the split calls, from kStreamReceived bytes of copies in all of a step's recvs on.  What this
// keeps in the cache are the STAGED rows, which the recvs of all the ranks a token was routed to read, and the copies of the
// first recvs are gone anyway by the time the last one has run.  Whole steps, us, copies kept / past the cache, with a
// sweep that reads the received rows, and with one that reads them and writes expert_y:
//   fp8 rows of 7168 bytes, K = 8: 184 MB (2 ranks)  320.4 / 332.0   813.3 / 823.1
//                                  206 MB (1 sender) 416.1 / 411.1  1058.3 / 1052.8
//                                  229 MB (8 ranks)  503.2 / 494.7  1210.9 / 1196.3
//                                  940 MB           1804.7 / 1740.6 4332.2 / 4261.9
//                           K = 4: 161 MB            386.4 / 394.1   858.0 / 863.0
//                                  206 MB            480.5 / 476.4  1072.1 / 1060.0
//                           K = 2:  80 MB            267.7 / 265.4   477.3 / 500.2
//                                  161 MB            432.1 / 431.5   887.5 / 880.6
//                                  229 MB            571.9 / 554.9  1201.4 / 1179.0
//   bf16 rows of 14 KB,     K = 4: 184 MB            328.8 / 328.1   353.4 / 348.5
//                           K = 8: 229 MB            391.1 / 380.1   417.6 / 409.5
constexpr uint64_t kStreamReceived = 200000000;

inline bool received_past_cache(uint64_t copies) { return copies >= kStreamReceived; }

// The first recv of a step is ONE launch that lays the receivers out and copies the caller's rows, a workgroup per row,
// where a receiver typically gets at most kFewRows rows, or up to kOneLaunchRows of no more than 8 KB each and
// kOneLaunchBytes together if every thread of a workgroup has at most one of the `items` runs to lay out; otherwise the
// layout is a launch in front of the copy.  us, layout apart / one launch, rank 0's four calls with one sender and the whole step:
//   8 ranks, rows of 7168 bytes:   256 rows  21.8 / 19.5    69.5 /  67.2      512 rows  31.4 / 29.0    89.2 /  86.9
//                                 1024 rows  49.2 / 47.9   121.5 / 119.9     2048 rows  86.3 / 86.3   220.4 / 220.6
//     8 senders:                   512 rows       -        133.1 / 131.5     1024 rows       -        166.3 / 165.3
//   16 ranks, 384 experts:         512 rows  47.0 / 44.6   166.9 / 164.3
//   32 ranks, 512 experts:         475 rows  72.4 / 74.5   333.4 / 335.6     (512 runs, 448 threads)
//   rows of 2048 bytes:           1024 rows  24.5 / 23.0    74.8 /  73.0     1400 rows  31.0 / 31.7    84.4 /  85.0
//   rows of 14 KB:                 256 rows  22.3 / 23.2    71.5 /  72.5      512 rows  33.1 / 33.4    93.9 /  94.1
//                                 1024 rows  53.5 / 57.0   138.8 / 142.0
constexpr uint32_t kFewRows = 256, kOneLaunchRows = 1024;
constexpr uint64_t kOneLaunchBytes = 7500000;

inline bool first_recv_in_one_launch(uint32_t typical_rows, uint32_t row_bytes, uint32_t items, uint32_t threads) {
    if (typical_rows <= kFewRows) return true;
    return typical_rows <= kOneLaunchRows && row_bytes <= 8192 &&
           (uint64_t)typical_rows * row_bytes <= kOneLaunchBytes && items <= threads;
}

}  // namespace a2a
