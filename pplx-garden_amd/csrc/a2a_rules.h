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

}  // namespace a2a
