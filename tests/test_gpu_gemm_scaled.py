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


# Row tiles per wave: three, and one and two where they fill the CUs better (11008 inputs to 4096 rows; 8192 to 8194).
@pytest.mark.parametrize("m,k,rows", [(777, 4096, 12288), (705, 4224, 12290), (704, 4352, 12286), (640, 2112, 30002),
                                      (2047, 2048, 14338), (777, 11008, 4096), (833, 11072, 4098), (2048, 8192, 8192),
                                      (2001, 8320, 8194)])
@pytest.mark.parametrize("epilogue", sorted(NAMES))
def test_gemm_scaled_matches_the_int8_kernels(cuda, oracle, m, k, rows, epilogue):
    import torch
    from ivonar_amd import ops, runtime

    lib = runtime.library()
    need = lib.ivonar_gemm_work(m, rows, k)
    if need == 0:
        pytest.skip("the rule does not pick the block-scaled kernel for this shape on this device")
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
