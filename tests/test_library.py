"""The C-ABI library (CPU side): it loads, exports every entry point
include/wptv.h declares, and answers its host-only queries (no kernel runs
here)."""

import ctypes
import re
from pathlib import Path
from types import SimpleNamespace

import pytest
import torch

from wpt_amd import _lib, layers
from wpt_amd.decoder import LARGE, MQADecoder

HEADER = Path(__file__).resolve().parents[1] / "include" / "wptv.h"


def declared():
    text = HEADER.read_text()
    return sorted(set(re.findall(r"^(?:int|const char\*)\s+(wptv_\w+)\(", text, flags=re.M)))


def test_the_header_declares_the_entry_points_the_loader_binds():
    assert declared() == sorted(_lib.SIGNATURES)


def test_the_library_loads_and_exports_every_declared_entry_point():
    library = _lib.lib()
    for name in declared():
        assert hasattr(library, name), name
    assert library.wptv_abi_version() == _lib.ABI_VERSION


def test_the_workspace_query_plans_the_verify_attention_workload():
    library = _lib.lib()
    splits, size = ctypes.c_int(8), ctypes.c_size_t(0)
    status = library.wptv_attention_workspace(32, 5, 16, 128, 4096, 0, _lib.WPTV_BF16, 0, ctypes.byref(splits),
                                              ctypes.byref(size))
    assert status == 0 and splits.value == 8
    # eight parts of 80 query rows x 128 bf16 values plus an FP32
    # log-sum-exp each
    assert size.value >= 32 * 8 * 80 * (128 * 2 + 4)
    status = library.wptv_attention_workspace(32, 5, 16, 128, 4096, 0, _lib.WPTV_BF16, _lib.KEY_SPLIT,
                                              ctypes.byref(splits), ctypes.byref(size))
    assert status == 0 and size.value >= 32 * 8 * 80 * (128 * 2 + 4)


def test_bad_arguments_are_reported_with_a_message():
    library = _lib.lib()
    splits, size = ctypes.c_int(0), ctypes.c_size_t(0)
    status = library.wptv_attention_workspace(0, 5, 16, 128, 4096, 0, _lib.WPTV_BF16, 0, ctypes.byref(splits),
                                              ctypes.byref(size))
    assert status == -1
    assert b"positive" in library.wptv_last_error()
    with pytest.raises(ValueError, match="positive"):
        _lib.check(status, "attention_workspace")
    status = library.wptv_attention_workspace(1, 1, 1, 128, 8, 0, 7, 0, ctypes.byref(splits), ctypes.byref(size))
    with pytest.raises(NotImplementedError):
        _lib.check(status, "attention_workspace")


def chosen_parts(B, T, H, c, N, window=0, dtype=_lib.WPTV_BF16, flags=_lib.RANGE_FROM_POSITIONS):
    splits, size = ctypes.c_int(0), ctypes.c_size_t(0)
    assert _lib.lib().wptv_attention_workspace(B, T, H, c, N, window, dtype, flags, ctypes.byref(splits),
                                               ctypes.byref(size)) == 0
    return splits.value


@pytest.mark.parametrize("B, T, N", [(256, 5, 4100), (257, 5, 4100), (300, 5, 4100), (384, 5, 8000), (4, 600, 3600),
                                     (300, 1, 5000)])
def test_a_call_that_fills_the_compute_units_has_one_bf16_rounding(B, T, N):
    # parts are held in bf16: where a workgroup a (batch row, query group) fills the 256 compute units, a
    # second part would only add its rounding (the sums of one part are FP32 throughout)
    assert chosen_parts(B, T, 16, 128, N) == 1


def test_sparse_calls_that_fill_the_compute_units_have_one_bf16_rounding():
    splits, size = ctypes.c_int(0), ctypes.c_size_t(0)
    assert _lib.lib().wptv_sparse_attention_workspace(60, 5, 16, 128, 3900, 128, 20000, _lib.WPTV_BF16,
                                                      ctypes.byref(splits), ctypes.byref(size)) == 0
    assert splits.value == 1


@pytest.mark.parametrize("B, T, H, N, parts", [
    (200, 2, 16, 4100, 2), (171, 2, 16, 2048, 2), (100, 2, 16, 3000, 5), (150, 4, 8, 1500, 3),  # two workgroups a unit
    (200, 2, 16, 1029, 1), (23, 2, 16, 4100, 11), (255, 2, 16, 2048, 1),  # a part over costs more than it gives
    (100, 3, 16, 4100, 5), (47, 5, 16, 4100, 5), (171, 3, 16, 1500, 1),   # three blocks and more: a round each
    (39, 1, 16, 4500, 7)])                                               # one block: the parts cover the units
def test_the_parts_at_head_width_64(B, T, H, N, parts):
    assert chosen_parts(B, T, H, 64, N) == parts


@pytest.mark.parametrize("B, T, c, N, parts, alone", [
    (1, 1, 128, 320, 3, 1), (64, 1, 128, 320, 3, 1), (128, 1, 128, 320, 1, 1), (1, 1, 128, 160, 1, 1),  # one block
    (80, 1, 128, 256, 2, 1), (32, 2, 128, 288, 3, 1), (72, 3, 128, 320, 3, 1), (72, 3, 128, 256, 1, 1),
    (1, 5, 128, 300, 3, 1), (16, 5, 128, 320, 3, 1), (32, 5, 128, 320, 1, 1),
    (1, 16, 128, 288, 3, 1), (8, 31, 128, 320, 1, 1), (1, 5, 64, 320, 1, 1),
    (1, 5, 128, 700, 6, 6), (32, 5, 128, 4100, 8, 8)])
def test_short_ranges_are_cut_for_graphs_and_left_whole_for_calls_one_by_one(B, T, c, N, parts, alone):
    assert chosen_parts(B, T, 16, c, N) == parts
    assert chosen_parts(B, T, 16, c, N, flags=_lib.RANGE_FROM_POSITIONS | _lib.CALL_BY_CALL) == alone


def test_a_reading_whose_stream_passes_4_gb_keeps_the_product_it_had():
    # wptv_gemm_wide_swiglu refuses operands of 4 GB and more, hipBLASLt does not
    assert layers.swiglu_tiles(976562, 11264, 2048)
    assert not layers.swiglu_tiles(976563, 11264, 2048)
    assert _lib.lib().wptv_gemm_wide_swiglu(16, 2048, 16, 2048, 976563, 11264, 2048, 16, 5632, None) == -3
    assert b"4 GB" in _lib.lib().wptv_last_error()


@pytest.mark.parametrize("M, N, K, faster", [
    (513, 11264, 2048, True), (1281, 11264, 2048, True), (4096, 11264, 2048, True), (1281, 22016, 4096, True),
    (513, 5632, 1024, True), (2000, 768, 256, True), (1000, 2048, 512, True),
    (1000, 4096, 2048, False), (513, 22016, 4096, False), (513, 2048, 512, False), (1000, 768, 256, False)])
def test_a_gate_up_product_of_few_tiles_stays_off_them(M, N, K, faster):
    # measured on the MI355X at these sizes (layers.swiglu_tiles)
    assert layers.swiglu_tiles(M, N, K) == faster


@pytest.mark.parametrize("rows", [1, 160, 161, 235, 288, 289, 320, 321])
@pytest.mark.parametrize("any_rows", [False, True])
def test_the_decoder_s_answer_about_fm_rows_is_the_products(rows, any_rows):
    # a program that asks fm_rows and then calls the products without any_rows must not be refused
    shapes = {"qkv": (2304, 2048), "out": (2048, 2048), "gate_up_tiles": (11264, 2048), "down": (2048, 5632)}
    model = SimpleNamespace(dtype=torch.bfloat16, config=LARGE, _fm_rows={},
                            fm={f"layers.0.{name}": SimpleNamespace(shape=shape) for name, shape in shapes.items()})
    taken = all(layers.fm_plan(rows, *shape, swiglu=name == "gate_up_tiles", any_rows=any_rows) is not None
                for name, shape in shapes.items())
    assert taken == (rows <= 160 or 289 <= rows <= 320 or any_rows and rows <= 320)
    assert MQADecoder.fm_rows(model, rows, *([True] if any_rows else [])) == taken
