"""ternary_linear on half rows: the bits of the same call on the rows converted to fp32 first, for every layout the
quantizer reads half rows in (aligned, off alignment, odd widths, past the last layout) and for strided inputs."""

from __future__ import annotations

import numpy as np
import pytest

from _util import device_matrix, make_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("m,k", [(1, 1024), (1, 4100), (1, 8192), (1, 1101), (2, 8192), (12, 28672), (77, 1100),
                                 (300, 4096), (5, 8190), (3, 8194), (3, 40000), (513, 2052), (257, 8192)])
def test_half_rows(cuda, dtype, m, k):
    import torch
    from ivonar_amd import ops

    rng = np.random.default_rng(m + k)
    _, packed, scale_bits, bias = make_layer(rng, 130, k, bias=m % 2 == 1)
    matrix = device_matrix(packed, scale_bits, k, bias=bias, device=cuda)
    flat = torch.randn(m * k + 8, generator=torch.Generator(device=cuda).manual_seed(k), device=cuda)
    flat[m * k // 2] = 60000.0
    flat = flat.to(getattr(torch, dtype))
    for offset in (0, 1, 2):  # 16-, 2- and 4-byte aligned rows
        x = flat[offset:offset + m * k].view(m, k)
        assert torch.equal(ops.ternary_linear(x, matrix), ops.ternary_linear(x.float(), matrix)), f"offset {offset}"
    wide = torch.randn(m, k + 6, device=cuda).to(flat.dtype)
    strided = wide[:, 3:3 + k]
    assert torch.equal(ops.ternary_linear(strided, matrix), ops.ternary_linear(strided.float().contiguous(), matrix))
    batched = flat[:m * k].view(1, m, k)
    assert ops.ternary_linear(batched, matrix).shape == (1, m, 130)


@pytest.mark.parametrize("m,k", [(64, 1101), (65, 1101), (65, 8190), (65, 1100), (2, 8194), (70, 8194)])
def test_strided_rows(cuda, m, k):
    """One copy at most before the call (the half types are converted by it or by the quantizer): the bits of the
    rows converted first, for each type."""
    import torch
    from ivonar_amd import ops
    from torch.utils._python_dispatch import TorchDispatchMode

    class Copies(TorchDispatchMode):
        made = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.made += func.overloadpacket in (torch.ops.aten.clone, torch.ops.aten._to_copy, torch.ops.aten.copy_)
            return func(*args, **(kwargs or {}))

    rng = np.random.default_rng(m + k)
    _, packed, scale_bits, _ = make_layer(rng, 130, k)
    matrix = device_matrix(packed, scale_bits, k, device=cuda)
    wide = torch.randn(m, k + 6, device=cuda)
    for dtype in (torch.float16, torch.bfloat16, torch.float64, torch.float32):
        x = wide.to(dtype)[:, 3:3 + k]
        expected = ops.ternary_linear(x.float().contiguous(), matrix)
        with Copies() as copies:
            y = ops.ternary_linear(x, matrix)
        assert torch.equal(y, expected), dtype
        assert copies.made == 1, dtype


def test_linear_matches_the_separate_calls(cuda):
    import torch
    from ivonar_amd import ops

    rng = np.random.default_rng(5)
    _, packed, scale_bits, bias = make_layer(rng, 333, 1100, bias=True)
    matrix = device_matrix(packed, scale_bits, 1100, bias=bias, device=cuda)
    for m in (1, 2, 33, 500):
        x = torch.randn(m, 1100, device=cuda)
        q8, xsum, scale = ops.quantize_rows(x)
        expected = ops.gemm(matrix, q8, xsum, scale) if m > 1 else ops.gemv(matrix, x[0]).reshape(1, -1)
        assert torch.equal(ops.ternary_linear(x, matrix), expected)
        assert torch.equal(ops.ternary_linear(x.double(), matrix), expected)


def test_linear_refuses_what_it_cannot_run(cuda):
    import torch
    from ivonar_amd import ops, runtime

    rng = np.random.default_rng(6)
    _, packed, scale_bits, _ = make_layer(rng, 64, 256)
    matrix = device_matrix(packed, scale_bits, 256, device=cuda)
    with pytest.raises(runtime.KernelError):
        ops.ternary_linear(torch.zeros(0, 256, device=cuda), matrix)
    with pytest.raises(runtime.KernelError):
        ops.ternary_linear(torch.zeros(2, 255, device=cuda), matrix)
    with pytest.raises(runtime.KernelError):
        ops.ternary_linear(torch.zeros(2, 256), matrix)
    x, out = torch.zeros(2, 256, device=cuda), torch.zeros(2, 64, device=cuda)
    tail = (matrix.packed.data_ptr(), matrix.scales.data_ptr(), None, out.data_ptr(), 64, 256, matrix.row_bytes, 2)
    for dtype, work, size in ((3, x.data_ptr(), 2048), (0, None, 2048), (0, x.data_ptr(), 16)):  # type, no or little work
        assert runtime.library().ivonar_linear(0, x.data_ptr(), dtype, 2, work, size, *tail) != 0
