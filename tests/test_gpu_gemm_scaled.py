"""The block-scaled FP6 x FP4 token GEMM: the bits of the int8 kernels (themselves checked against the oracle) on
every output, at the edges of its tiles (64 tokens, 128, 256 or 384 rows, 8-row pitch), with group counts of every remainder
of its three-step rounds, an odd chunk count, all three epilogues, a bias and a padded output stride; and a sample of
token rows against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

import ternary_oracle as T
from _util import assert_bits_equal, device_matrix, make_layer, to_np

pytestmark = pytest.mark.gpu

NAMES = {"store": "gemm_tile_store", "residual": "gemm_tile_residual", "silu_pair": "gemm_tile_silu_pair"}


# The last figure is the row tiles per wave (32 rows each) the rule takes on 256 CUs.
@pytest.mark.parametrize("m,k,rows,tiles", [
    (777, 4096, 12288, 3), (705, 4224, 12290, 3), (704, 4352, 12286, 1), (640, 2112, 30002, 2), (2047, 2048, 14338, 3),
    (777, 11008, 4096, 1), (833, 11072, 4098, 1), (2048, 8192, 8192, 2), (2001, 8320, 8194, 3), (513, 4096, 14338, 1),
    (514, 9138, 14390, 1), (391, 20434, 9326, 1), (897, 4096, 16386, 2), (300, 4100, 22018, 2)])
@pytest.mark.parametrize("epilogue", sorted(NAMES))
def test_gemm_scaled_matches_the_int8_kernels(cuda, oracle, m, k, rows, tiles, epilogue):
    import torch
    from ivonar_amd import ops, runtime

    lib = runtime.library()
    assert lib.ivonar_gemm_row_tiles(m, rows, k) == tiles
    assert lib.ivonar_gemm_work(m, rows, k) > 0
    rng = np.random.default_rng(m + k + rows)
    codes, packed, scale_bits, bias = make_layer(rng, rows, k, bias=m % 2 == 1)
    matrix = device_matrix(packed, scale_bits, k, bias=bias, device=cuda)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 5] *= 40.0
    q8, xsum, sx = ops.quantize_rows(torch.from_numpy(x).to(cuda))
    q8[1, 7] = -128  # the quantizer stops at -127, a caller's buffer need not
    width = rows // 2 if epilogue == "silu_pair" else rows
    base = torch.randn(m, width + 3, generator=torch.Generator(device=cuda).manual_seed(m), device=cuda)
    expected, out = base.clone(), base.clone()
    args = (matrix.rows, k, matrix.row_bytes, matrix.groups)
    status = getattr(lib, NAMES[epilogue])(
        runtime.current_stream(cuda), q8.data_ptr(), xsum.data_ptr(), sx.data_ptr(), matrix.packed.data_ptr(),
        matrix.scales.data_ptr(), None if bias is None else matrix.bias.data_ptr(), expected.data_ptr(), *args,
        matrix.lanes, width + 3, m)
    assert status == 0
    ops.gemm(matrix, q8, xsum, sx, out=out, epilogue=epilogue, out_stride=width + 3)
    assert torch.equal(out, expected)
    if epilogue == "store":
        assert runtime.gemm_plan(m, rows, k) == 1
        rows_checked = [0, 63, 64, m - 1]
        eq8, exsum, esx = oracle.quantize_rows(T.MODE_PLAIN, x[rows_checked], k)
        reference = oracle.gemm_split(T.EPI_STORE, eq8, exsum, esx, packed, scale_bits, bias,
                                      np.zeros((len(rows_checked), rows), np.float32), k, rows, len(rows_checked), 1)
        assert_bits_equal(to_np(out[rows_checked, :width].contiguous()), reference, "sampled tokens")


# Measured (us, graph replays on one MI355X): the int8 kernel, then 1, 2 and 3 row tiles, the lay-out included.
MEASURED = [
    (777, 2048, 6144, 26.7, 26.3, 27.4, 27.7), (1024, 2048, 6144, 27.7, 28.5, 29.3, 30.4),
    (2048, 2048, 6144, 46.4, 46.9, 45.4, 43.6), (777, 4096, 4096, 30.4, 30.2, 33.9, 39.7),
    (900, 4096, 4096, 31.8, 31.8, 35.0, 41.0), (1300, 4096, 4096, 50.3, 40.8, 43.2, 43.5),
    (2048, 4096, 4096, 54.5, 56.8, 50.2, 60.4), (300, 4096, 12288, 31.2, 31.4, 34.4, 40.1),
    (391, 4096, 12288, 46.7, 39.5, 41.5, 42.4), (777, 4096, 12288, 78.3, 61.1, 65.7, 59.1),
    (514, 4096, 14336, 75.9, 53.2, 47.2, 56.2), (2048, 4096, 14336, 167.6, 150.5, 137.4, 140.8),
    (777, 4096, 22016, 123.4, 101.1, 101.0, 93.1), (640, 5120, 5120, 36.5, 34.1, 39.0, 46.5),
    (391, 8192, 8192, 55.8, 47.3, 53.3, 65.5), (2048, 8192, 8192, 178.8, 171.0, 154.8, 167.1),
    (128, 8192, 28672, 57.6, 57.8, 64.4, 76.5), (2048, 8192, 28672, 558.6, 548.4, 517.8, 507.0),
    (777, 11008, 4096, 71.9, 55.4, 64.1, 79.9), (1536, 11008, 4096, 114.0, 95.7, 92.2, 119.0),
    (777, 14336, 4096, 92.1, 70.4, 81.5, 102.6), (391, 28672, 8192, 184.4, 140.2, 162.1, 204.8),
]


@pytest.mark.parametrize("m,k,rows,times", [(*row[:3], row[3:]) for row in MEASURED])
def test_the_rule_takes_what_was_measured_fastest(cuda, m, k, rows, times):
    """Within 8% of the fastest (the rule asks for 3% before it leaves the int8 kernel, and its fit has an error of
    4%), and never more than 2% behind the int8 kernel."""
    from ivonar_amd import runtime

    taken = times[runtime.library().ivonar_gemm_row_tiles(m, rows, k)]
    assert taken <= 1.08 * min(times) and taken <= 1.02 * times[0]


def test_small_workspace_runs_the_int8_kernel(cuda):
    import torch
    from ivonar_amd import ops, runtime

    lib = runtime.library()
    m, k, rows = 777, 4096, 12288
    rng = np.random.default_rng(2)
    _, packed, scale_bits, _ = make_layer(rng, rows, k)
    matrix = device_matrix(packed, scale_bits, k, device=cuda)
    q8, xsum, sx = ops.quantize_rows(torch.randn(m, k, device=cuda))
    expected = ops.gemm(matrix, q8, xsum, sx)
    for work, size in ((None, 0), (torch.empty(64, dtype=torch.uint8, device=cuda), 64)):
        out = torch.zeros(m, rows, device=cuda)
        assert lib.ivonar_gemm(runtime.current_stream(cuda), 0, q8.data_ptr(), xsum.data_ptr(), sx.data_ptr(),
                               matrix.packed.data_ptr(), matrix.scales.data_ptr(), None, out.data_ptr(), rows, k,
                               matrix.row_bytes, matrix.groups, rows, m,
                               None if work is None else work.data_ptr(), size) == 0
        assert torch.equal(out, expected)
    assert lib.ivonar_gemm(0, 3, *([None] * 7), rows, k, matrix.row_bytes, matrix.groups, rows, m, None, 0) != 0


def test_no_memory_for_the_workspace_runs_the_int8_kernel(cuda, monkeypatch):
    """The allocation of the block-scaled kernel's workspace fails (forced here): the call runs without it."""
    import torch
    from ivonar_amd import ops

    m, k, rows = 777, 4096, 12288
    rng = np.random.default_rng(4)
    _, packed, scale_bits, _ = make_layer(rng, rows, k)
    matrix = device_matrix(packed, scale_bits, k, device=cuda)
    x = torch.randn(m, k, device=cuda)
    expected = ops.ternary_linear(x, matrix)
    buffers = ops.quantize_rows(x)
    refused, real = [], torch.empty

    def empty(*args, **kwargs):
        if kwargs.get("dtype") == torch.uint8 and args[0] > m * k * 2:
            refused.append(args[0])
            raise torch.OutOfMemoryError("forced")
        return real(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", empty)
    assert torch.equal(ops.ternary_linear(x, matrix), expected)
    assert torch.equal(ops.gemm(matrix, *buffers), expected)
    assert len(refused) == 2


def test_graph_replays_with_the_workspace(cuda):
    import torch
    from ivonar_amd import ops

    m, k, rows = 777, 4096, 12288
    rng = np.random.default_rng(3)
    _, packed, scale_bits, _ = make_layer(rng, rows, k)
    matrix = device_matrix(packed, scale_bits, k, device=cuda)
    x = torch.randn(m, k, device=cuda)
    ops.ternary_linear(x, matrix)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.ternary_linear(x, matrix)
    for seed in range(3):
        x.copy_(torch.randn(m, k, generator=torch.Generator(device=cuda).manual_seed(seed), device=cuda))
        expected = ops.ternary_linear(x, matrix)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, expected)
