"""The launchers' rules on sizes (csrc/a2a_rules.h), compiled as plain C++ and called on the CPU."""

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

from test_gpu_pieces import GATHERS, HELD, MOVED, QUANTISED
from test_gpu_shapes import STREAMED, STREAMED_QUANTISED, copies_of
from test_gpu_split import PIECES
from test_gpu_written_through import STEPS

CSRC = Path(__file__).resolve().parent.parent / "pplx-garden_amd" / "csrc"

SOURCE = """
#include "a2a_rules.h"
extern "C" {
uint32_t layers(uint32_t tokens) { return a2a::token_layers(tokens).layers; }
uint32_t layer_rows(uint32_t tokens) { return a2a::token_layers(tokens).rows; }
int past_cache(uint64_t copies, int quantize, uint32_t k) { return a2a::copies_past_cache(copies, quantize != 0, k); }
int received_past_cache(uint64_t copies) { return a2a::received_past_cache(copies); }
int written_through(uint64_t copies, uint32_t row_bytes, uint32_t k) {
    return a2a::copies_written_through(copies, row_bytes, k);
}
uint32_t pieces(uint32_t k, uint32_t chunks, int quantize, int by_column) {
    return a2a::pieces_per_lane(k, chunks, quantize != 0, by_column != 0, 1);
}
uint32_t pieces_beside(uint32_t k, uint32_t chunks, uint32_t experts) {
    return a2a::pieces_per_lane(k, chunks, false, false, experts);
}
int two_workgroups(int quantize, int scaled, uint32_t one, uint32_t two, uint32_t units, uint32_t experts, uint32_t senders) {
    return a2a::two_workgroups_a_unit(quantize != 0, scaled != 0, one, two, units, experts, senders);
}
int two_pieces(uint32_t k, uint64_t slabs) { return a2a::two_pieces_a_lane(k, slabs); }
int one_launch(uint32_t rows, uint32_t row_bytes, uint32_t items, uint32_t threads) {
    return a2a::first_recv_in_one_launch(rows, row_bytes, items, threads);
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("needs a C++ compiler")
    folder = tmp_path_factory.mktemp("rules")
    (folder / "rules.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", str(CSRC),
                    str(folder / "rules.cpp"), "-o", str(folder / "rules.so")], check=True)
    lib = ctypes.CDLL(str(folder / "rules.so"))
    lib.past_cache.argtypes = [ctypes.c_uint64, ctypes.c_int, ctypes.c_uint32]
    lib.received_past_cache.argtypes = [ctypes.c_uint64]
    lib.written_through.argtypes = [ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32]
    return lib


@pytest.mark.parametrize("tokens", [1, 7, 32767, 32768, 32769, 33000, 65536, 65537, 100001, 1048577, 2147483647])
def test_the_gathers_grid_has_every_token_and_next_to_no_empty_rows(rules, tokens):
    layers, rows = rules.layers(tokens), rules.layer_rows(tokens)
    assert layers * rows >= tokens and rows <= 32768 and layers <= 65536
    assert layers * rows - tokens < layers
    assert layers == -(-tokens // 32768)


def test_copies_that_the_infinity_cache_can_hold_stay_there_for_their_reader(rules):
    """The experts read the copies next: only what the 256 MB cache cannot hold until then goes past it."""
    for tokens in (1900, 2048, 3072, 4096):      # 109 to 235 MB of quantised rows of 7168 bytes
        assert not rules.past_cache(tokens * 8 * 7168, 1, 8)
    assert not rules.past_cache(256 << 20, 1, 8) and not rules.past_cache(256 << 20, 0, 6)
    assert rules.past_cache(8 * 4096 * 8 * 7168, 1, 8)       # eight ranks of 4096 tokens
    assert rules.past_cache(1 << 30, 0, 3) and rules.past_cache(1 << 30, 1, 1) and not rules.past_cache(1 << 30, 0, 2)


@pytest.mark.parametrize("row,hidden,scales,k,tokens,streamed", STREAMED)
def test_the_gpu_tests_of_streamed_steps_lie_on_the_side_they_are_meant_for(rules, row, hidden, scales, k, tokens, streamed):
    assert bool(rules.past_cache(copies_of(row, hidden, k, tokens), 0, k)) == streamed


def test_the_gpu_tests_of_streamed_quantised_rows_are_streamed_and_move_the_pieces_they_are_meant_for(rules):
    for hidden, k, tokens, pieces in STREAMED_QUANTISED:
        assert rules.past_cache(sum(tokens) * k * hidden, 1, k), (hidden, k)
        assert rules.pieces(k, hidden // 16, 1, 0) == pieces, (hidden, k)


def test_rows_that_leave_much_of_their_last_4_kb_empty_are_not_written_through(rules):
    size = 200000000
    assert all(rules.written_through(size, row, k) for row in (4096, 7168, 8192, 12288, 14336, 16384, 28672) for k in (6, 7, 8))
    assert not any(rules.written_through(size, row, 6) for row in (2048, 4080, 4112, 4608, 5120, 5888, 6144, 6656, 8704, 9216))
    assert rules.written_through(size, 6144, 7) and rules.written_through(size, 9216, 8) and rules.written_through(size, 12800, 7)
    assert not any(rules.written_through(size, row, k) for row in (4352, 5888, 6128, 8704) for k in (7, 8, 64))
    assert not any(rules.written_through(size, 8192, k) for k in (1, 4, 5)) and not rules.written_through(119999999, 8192, 8)
    assert rules.written_through(size, 0xFFFFF000, 64)


@pytest.mark.parametrize("tokens,experts,topk,hidden,dtype,through", STEPS)
def test_the_gpu_tests_of_written_through_steps_lie_on_the_side_they_are_meant_for(rules, tokens, experts, topk, hidden, dtype,
                                                                                   through):
    row = hidden * dtype.itemsize
    assert sum(tokens) * topk > 16384 and not rules.past_cache(sum(tokens) * topk * row, 0, topk)
    assert bool(rules.written_through(sum(tokens) * topk * row, row, topk)) == through


def test_pieces_of_a_thread(rules):
    # the fewer copies a token has, the more of its row a thread moves; never with five copies and more
    assert [rules.pieces(k, 320, 0, 0) for k in (1, 2, 3, 4, 5, 8, 64)] == [4, 2, 2, 2, 1, 1, 1]
    # four copies: where a piece a thread makes workgroups of 3, 5, 6, 7 or 14 wavefronts (and 2, unquantised)
    waves = [w for w in range(1, 40) if rules.pieces(4, 64 * w, 1, 0) == 2]
    assert waves == [3, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15]
    assert rules.pieces(4, 128, 0, 0) == 2 and rules.pieces(4, 128, 1, 0) == 1 and rules.pieces(4, 320, 0, 1) == 1
    for k, hidden, dtype, scales, layout, pieces in MOVED:
        assert rules.pieces(k, hidden * dtype.itemsize // 16, 0, layout == "col") == pieces, (k, hidden)
    for k, hidden, pieces in QUANTISED:
        assert rules.pieces(k, hidden // 16, 1, 0) == pieces, (k, hidden)


def test_pieces_of_a_thread_where_the_local_experts_hold_the_workgroup(rules):
    # as many threads for experts as pieces: no wavefront fewer with several pieces, so one, with the stores it had
    assert [rules.pieces_beside(1, chunks, 128) for chunks in (64, 65, 128, 129)] == [4, 1, 1, 4]
    assert [rules.pieces_beside(2, 128, experts) for experts in (8, 64, 65, 96, 128, 1024)] == [2, 2, 1, 1, 1, 1]
    # unless a token's copies are long
    assert [rules.pieces_beside(2, chunks, 512) for chunks in (511, 512)] == [1, 2]
    assert [rules.pieces_beside(4, chunks, 512) for chunks in (192, 255, 320)] == [1, 1, 2]
    for topk, ranks, experts, hidden, dtype, scales, layout, pieces in HELD:
        chunks = hidden * dtype.itemsize // 16
        assert rules.pieces_beside(topk, chunks, -(-experts // ranks)) == pieces, (topk, hidden)


def test_two_workgroups_a_compute_unit_where_they_gain(rules):
    # quantised rows, five tokens a workgroup or three: receivers of many experts, or rows of few or many units
    assert [rules.two_workgroups(1, 1, 5, 3, 4, le, 8) for le in (4, 8, 9, 32)] == [0, 0, 1, 1]
    assert [rules.two_workgroups(1, 1, 5, 3, units, 8, 8) for units in range(1, 9)] == [1, 1, 0, 0, 0, 1, 1, 1]
    # six on a compute unit either way; never four
    assert rules.two_workgroups(1, 1, 6, 3, 4, 8, 8) and not rules.two_workgroups(1, 1, 6, 4, 2, 32, 8)
    # rows as they are: always with up to four tokens, but for two rounds of eight wavefronts and many sources
    assert all(rules.two_workgroups(0, 0, one, two, units, 8, 16) for one, two in ((5, 3), (6, 3), (7, 4)) for units in (1, 2, 3, 5, 7))
    assert [rules.two_workgroups(0, 0, 7, 4, 4, 8, senders) for senders in (1, 8, 9, 16)] == [1, 1, 0, 0]
    # with five, which have a lane a route, only rows of 4 KB and more, of 6 KB where they have scales and few experts
    assert [rules.two_workgroups(0, 0, 8, 5, units, 8, 8) for units in range(1, 8)] == [0, 0, 0, 1, 1, 1, 1]
    assert [rules.two_workgroups(0, 1, 8, 5, units, 8, 8) for units in range(1, 8)] == [0, 0, 0, 0, 0, 1, 1]
    assert [rules.two_workgroups(0, 1, 8, 5, units, 17, 8) for units in range(1, 8)] == [0, 0, 0, 1, 1, 1, 1]
    assert [rules.two_workgroups(0, 1, 8, 5, 2, 24, senders) for senders in (8, 9, 16)] == [0, 1, 1]


def test_pieces_of_the_gather(rules):
    for ranks, tokens, topk, hidden, dtype, two in GATHERS:
        slabs = -(-hidden * dtype.itemsize // 1024) * ranks * tokens
        assert bool(rules.two_pieces(topk, slabs)) == two, (tokens, topk)


def test_received_rows_that_the_cache_can_keep_stay_there(rules):
    for tokens, k in ((5600, 2), (5600, 4)):     # 8 x 700 tokens of 7168 bytes: 80 and 161 MB of copies, 42 MB staged
        assert not rules.received_past_cache(tokens * k * 7168)
    assert rules.received_past_cache(8 * 2048 * 8 * 7168)
    sides = {cfg.name: rules.received_past_cache(cfg.world_size * cfg.max_num_tokens * cfg.num_experts_per_token *
                                                 cfg.hidden_dim * cfg.in_dtype.itemsize) for cfg in PIECES}
    assert sides.pop("past-the-cache") and not any(sides.values())


def test_first_recvs_in_one_launch(rules):
    # rows a receiver typically gets, bytes of one, (source, expert) runs, threads of a workgroup
    assert rules.one_launch(512, 7168, 16 * 24, 448)            # 1024 tokens on 16 ranks with 384 experts
    assert rules.one_launch(1024, 7168, 8 * 32, 448) and rules.one_launch(256, 16384, 1024, 64)
    assert not rules.one_launch(475, 7168, 32 * 16, 448)        # more runs than threads
    assert not rules.one_launch(512, 14336, 8 * 16, 896) and not rules.one_launch(1025, 1024, 8, 64)
    sides = {}
    for cfg in PIECES:
        row = cfg.hidden_dim * cfg.in_dtype.itemsize
        runs = cfg.world_size * -(-cfg.num_experts // cfg.world_size)
        sides[cfg.name] = rules.one_launch(cfg.max_num_tokens * cfg.num_experts_per_token, row, runs,
                                           min(max(-(-row // 1024) * 64, 64), 1024))
    assert [n for n in sides if sides[n]] == ["more-scales-than-lanes", "256-rows", "257-rows-one-run-a-thread",
                                                  "1024-rows", "915-rows-of-8-KB"]
