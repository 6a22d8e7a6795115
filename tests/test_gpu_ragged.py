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
