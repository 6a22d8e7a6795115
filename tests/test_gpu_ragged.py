"""Token GEMM on matrices whose sizes fit no tile, against the CPU oracle's restatement of the kernel's order."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import ternary_oracle as T
from _util import assert_bits_equal, device_matrix, make_layer, to_np, token_gemm_expected, token_gemm_order

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 17, 33, 77])
@pytest.mark.parametrize("k,rows", [(1100, 33), (300, 17), (384, 5), (2100, 97)])
def test_gemm_odd_scale_count(cuda, oracle, m, k, rows):
    """An odd number of group scales in all (odd rows, odd groups): the last row's last scale is half a dword."""
    from ivonar_amd import ops

    rng = np.random.default_rng(m * 100 + k + rows)
    codes, packed, scale_bits, b = make_layer(rng, rows, k, bias=True)
    assert scale_bits.size % 2 == 1
    x = rng.standard_normal((m, k)).astype(np.float32)
    matrix = device_matrix(packed, scale_bits, k, bias=b, device=cuda)
    y = to_np(ops.gemm(matrix, *ops.quantize_rows(torch.from_numpy(x).to(cuda))))
    q8, xsum, sx = oracle.quantize_rows(T.MODE_PLAIN, x, k)
    expected = token_gemm_expected(oracle, T.EPI_STORE, q8, xsum, sx, packed, scale_bits, b,
                                   np.zeros((m, rows), np.float32), k, rows, m)
    assert_bits_equal(y, expected, f"gemm m={m} {k}->{rows} (order {token_gemm_order(m, rows, k)})")


@pytest.mark.parametrize("m", [1, 2, 12, 17, 33, 77, 200])
@pytest.mark.parametrize("k,rows", [(1100, 33), (300, 17), (384, 5), (1024, 64), (4352, 97), (2048, 3334)])
def test_scales_off_a_dword_boundary(cuda, oracle, m, k, rows):
    """A caller's scales may start in the middle of a dword: the halfwords around them (NaN here) are not used, and
    the last scale is, whatever the parity of the count."""
    from ivonar_amd import ops, runtime

    rng = np.random.default_rng(m * 10 + k + rows)
    codes, packed, scale_bits, b = make_layer(rng, rows, k, bias=True)
    matrix = device_matrix(packed, scale_bits, k, bias=b, device=cuda)
    around = np.full(scale_bits.size + 4, 0x7E00, dtype=np.uint16)
    around[1:1 + scale_bits.size] = scale_bits.reshape(-1)
    scales = torch.from_numpy(around.view(np.int16)).to(cuda)
    assert (scales.data_ptr() + 2) % 4 == 2
    x = rng.standard_normal((m, k)).astype(np.float32)
    q8d, xsumd, sxd = ops.quantize_rows(torch.from_numpy(x).to(cuda))
    y = torch.empty(m, rows, device=cuda)
    status = runtime.library().gemm_tile_store(
        runtime.current_stream(cuda), q8d.data_ptr(), xsumd.data_ptr(), sxd.data_ptr(), matrix.packed.data_ptr(),
        scales.data_ptr() + 2, matrix.bias.data_ptr(), y.data_ptr(), rows, k, matrix.row_bytes, matrix.groups,
        matrix.lanes, rows, m)
    assert status == 0
    q8, xsum, sx = oracle.quantize_rows(T.MODE_PLAIN, x, k)
    expected = token_gemm_expected(oracle, T.EPI_STORE, q8, xsum, sx, packed, scale_bits, b,
                                   np.zeros((m, rows), np.float32), k, rows, m)
    assert_bits_equal(to_np(y), expected, f"gemm m={m} {k}->{rows}")
