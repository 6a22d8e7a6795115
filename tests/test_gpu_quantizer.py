"""The quantizer's register-resident rows at the edges of their layouts, bit for bit against the oracle:
each row length one past or at a kernel's capacity, odd lengths, rows that start off a 16-byte boundary, and
lengths past the last layout (the slice kernel)."""

from __future__ import annotations

import numpy as np
import pytest

import ternary_oracle as T
from _util import assert_bits_equal, to_np

pytestmark = pytest.mark.gpu


def _check(actual, expected):
    for what, a, e in zip(("q8", "xsum", "scale"), actual, expected):
        assert_bits_equal(to_np(a), e, what)


def _rows(rng, m, n):
    x = (rng.standard_normal((m, n)) * rng.choice([1e-4, 1.0, 30.0], size=(m, 1))).astype(np.float32)
    x[0] = np.rint(x[0] * 4) / 2  # ties at half-integer quotients where the scale allows them
    x[0, n // 2] = 63.5
    return x


@pytest.mark.parametrize("m,n", [(3, 1028), (2, 4100), (513, 2052), (512, 4100), (513, 8192), (2, 8196), (2, 16388),
                                 (1, 32768), (1, 32772), (2, 1023), (3, 2049), (2, 4097), (1, 8191), (1, 8193)])
def test_plain_rows(cuda, oracle, m, n):
    import torch
    from ivonar_amd import ops

    x = _rows(np.random.default_rng(m + n), m, n)
    _check(ops.quantize_rows(torch.from_numpy(x).to(cuda)), oracle.quantize_rows(T.MODE_PLAIN, x, n))


@pytest.mark.parametrize("n,stride,offset", [(1024, 1027, 1), (4096, 4098, 2), (8192, 8193, 3), (6000, 6004, 4)])
def test_plain_rows_off_alignment(cuda, oracle, n, stride, offset):
    import torch
    from ivonar_amd import ops

    x = _rows(np.random.default_rng(n), 3, n)
    flat = torch.full((3 * stride + 8,), 7.0, device=cuda)
    rows = flat[offset:offset + 3 * stride].view(3, stride)[:, :n]
    rows.copy_(torch.from_numpy(x))
    _check(ops.quantize_rows(rows, n=n), oracle.quantize_rows(T.MODE_PLAIN, x, n))


@pytest.mark.parametrize("n", [1, 1025, 2048, 2049, 4097, 8191, 8193])
def test_norm_rows(cuda, oracle, n):
    import torch
    from ivonar_amd import ops

    rng = np.random.default_rng(n)
    x = _rows(rng, 3, n)
    weight = (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)
    actual = ops.quantize_rows(torch.from_numpy(x).to(cuda), mode=ops.MODE_NORM, aux=torch.from_numpy(weight).to(cuda))
    _check(actual, oracle.quantize_rows(T.MODE_NORM, x, n, aux=weight, eps=1e-6))


# head_dim * heads inputs: one, two, four and eight words per thread, pairs beyond the LDS table (5000), and
# rows beyond the last layout.
@pytest.mark.parametrize("head_dim,heads,splits", [(64, 64, 1), (64, 65, 8), (48, 171, 3), (128, 128, 2),
                                                   (64, 512, 8), (5, 1000, 5), (64, 513, 1)])
def test_attn_rows(cuda, oracle, head_dim, heads, splits):
    import torch
    from ivonar_amd import ops, runtime

    rng = np.random.default_rng(head_dim + heads)
    parts = rng.standard_normal((2, heads, splits, head_dim + 2)).astype(np.float32)
    parts[..., 0] *= 8.0
    parts[..., 1] = np.abs(parts[..., 1]) + 0.5
    if splits > 1:
        parts[0, 3, 1, 0] = -np.inf  # an empty split
    n, stride = heads * head_dim, heads * splits * (head_dim + 2)
    flat = parts.reshape(2, stride)
    assert runtime.library().ivonar_define(b"HEAD_DIM", head_dim) == 0
    try:
        actual = ops.quantize_rows(torch.from_numpy(flat).to(cuda), mode=ops.MODE_ATTN, splits=splits, n=n)
        _check(actual, oracle.quantize_rows(T.MODE_ATTN, flat, n, splits=splits, head_dim=head_dim, m=2,
                                            in_stride=stride))
    finally:
        runtime.library().ivonar_define(b"HEAD_DIM", 64)


# Rows on both sides of the rules that hand few long rows to several blocks: PLAIN rows of float4 in slices of 4096
# inputs (fewer than the register layout has room for, a last one in part), rows off a 16-byte boundary and NORM
# rows in the slice kernel or in one block each.
@pytest.mark.parametrize("m,n,offset", [(36, 28672, 0), (37, 28672, 0), (51, 20000, 0), (52, 20000, 0), (85, 9000, 0),
                                        (86, 9000, 0), (65, 12292, 0), (128, 8192, 0), (129, 8192, 0), (170, 2050, 0),
                                        (171, 2050, 0), (128, 4096, 1), (129, 4096, 1), (102, 4097, 0), (103, 4097, 0),
                                        (64, 8191, 0), (65, 8191, 0)])
def test_plain_rows_shared_by_blocks(cuda, oracle, m, n, offset):
    import torch
    from ivonar_amd import ops

    x = _rows(np.random.default_rng(m + n), m, n)
    rows = torch.empty(m * n + offset, device=cuda)[offset:].view(m, n)
    rows.copy_(torch.from_numpy(x))
    _check(ops.quantize_rows(rows), oracle.quantize_rows(T.MODE_PLAIN, x, n))


@pytest.mark.parametrize("m,n", [(64, 4096), (65, 4096), (64, 3076), (3, 3072), (51, 4097), (52, 4097), (32, 8191),
                                 (33, 8191), (86, 2051)])
def test_norm_rows_shared_by_blocks(cuda, oracle, m, n):
    import torch
    from ivonar_amd import ops

    rng = np.random.default_rng(m + n)
    x = _rows(rng, m, n)
    weight = (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)
    actual = ops.quantize_rows(torch.from_numpy(x).to(cuda), mode=ops.MODE_NORM, aux=torch.from_numpy(weight).to(cuda))
    _check(actual, oracle.quantize_rows(T.MODE_NORM, x, n, aux=weight, eps=1e-6))


@pytest.mark.parametrize("mode", ["plain", "norm"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 191, 255, 256, 257])
def test_rows_of_one_input_per_thread(cuda, oracle, mode, n):
    """Up to 256 inputs a thread holds one; 256 is the last such row."""
    import torch
    from ivonar_amd import ops

    rng = np.random.default_rng(n)
    x = _rows(rng, 5, n)
    rows = torch.full((5 * (n + 1) + 1,), 7.0, device=cuda)[1:].view(5, n + 1)[:, :n]
    rows.copy_(torch.from_numpy(x))
    weight = (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32) if mode == "norm" else None
    code = ops.MODE_NORM if mode == "norm" else ops.MODE_PLAIN
    actual = ops.quantize_rows(rows, mode=code, n=n, aux=None if weight is None else torch.from_numpy(weight).to(cuda))
    _check(actual, oracle.quantize_rows(T.MODE_NORM if mode == "norm" else T.MODE_PLAIN, x, n, aux=weight, eps=1e-6))
