"""GPU: the many-row int8 GEMM (more than 128 rows, and gate||up above 64 rows)
against the product of the same quantized weights in float64.

Bound: fp32 accumulation of K terms (K * 2^-24 of the sum of their magnitudes), then one rounding to
fp16 (2^-11 relative, 2^-25 at the smallest); the SwiGLU epilogue rounds gate, up, silu and product.
"""

from __future__ import annotations

import sys

import pytest
import torch

import runtime_amd.phase2  # noqa: F401

il = sys.modules["runtime_amd.phase2.int8_linear"]
pytestmark = pytest.mark.gpu
DEV = "cuda"
U, SUB = 2.0**-11, 2.0**-25


def _weights(n, k, g):
    q = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int32).to(torch.int8)
    scale = (torch.rand(n, generator=g, device=DEV) * 2e-3 + 1e-3).half()
    return q, scale, q.double() * scale.double()[:, None]


def _product(x, w, bias=None):
    """x W^T (+ bias) in float64 and the bound of an fp32 sum of it rounded to fp16."""
    y = x.double() @ w.T.contiguous()
    if bias is not None:
        y = y + bias.double()
    mag = x.double().abs() @ w.abs().T.contiguous() + (bias.double().abs() if bias is not None else 0)
    return y, U * y.abs() + SUB + (x.shape[1] + 2) * 2.0**-24 * mag


# Every instance of the launch (row tiles of 32, 64, 96 and 128 rows, 128 and 256 channels) with remainders
# of both, n-tiles past the last one, one k-tile, k-tile counts around the unrolled loops' 2, 3 and 12, and
# shapes that split K; test_int8_rows_plan.py checks that these shapes still reach them.
LINEAR = [
    (129, 1152, 896, True), (777, 1152, 896, True), (160, 4096, 4096, False), (256, 896, 4864, True),
    (1531, 4096, 1024, False), (2049, 4112, 192, True), (1000, 16, 64, False), (130, 272, 64, True),
    (385, 6144, 4096, False), (4096, 2048, 128, False), (191, 4096, 14336, False),
    (256, 4096, 14336, False), (1531, 4096, 14336, False), (700, 28672, 832, True), (2048, 28672, 1600, False),
    (130, 6144, 704, False), (140, 2048, 768, True), (150, 1024, 1600, False),
    (4167, 832, 832, True), (300, 4096, 4096, False), (198, 28560, 960, False), (4218, 784, 1792, False),
    (2814, 17568, 1920, False), (2814, 17568, 1984, True), (164, 22208, 1792, False),
    (3377, 528, 1856, True),
]
GATEUP = [
    (65, 4864, 896, False), (128, 4864, 896, True), (129, 4864, 896, False), (777, 1032, 192, True),
    (2048, 14336, 256, False), (300, 14336, 4096, False), (150, 8, 64, False), (96, 14336, 4096, False),
    (128, 14336, 4096, True), (66, 5632, 2048, False), (2000, 14336, 1088, False), (64, 4864, 896, False),
    (98, 12560, 128, False), (260, 14336, 4096, True), (4167, 416, 832, True), (198, 14280, 960, False),
    (71, 10912, 1920, False), (4218, 392, 1792, False), (2814, 8784, 1920, True), (2814, 8784, 1984, False), (164, 11104, 1792, True),
]


@pytest.mark.parametrize("m,n,k,bias", LINEAR)
def test_linear(m, n, k, bias):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    q, scale, w = _weights(n, k, g)
    b = torch.randn(n, generator=g, device=DEV).half() if bias else None
    x = torch.randn(m, k, generator=g, device=DEV).half()
    packed = il.pack_weight(q)
    y = il.int8_linear(x, packed, scale, b, n)
    want, bound = _product(x, w, b)
    assert ((y.double() - want).abs() <= bound).all()
    # An output at an odd element (no 8-byte stores), and strided x rows, give the same bytes.
    odd = torch.empty(m * n + 1, dtype=torch.float16, device=DEV)[1:]
    il.int8_linear(x, packed, scale, b, n, out=odd)
    assert torch.equal(odd.view(m, n), y)
    wide = torch.empty(m, k + 72, dtype=torch.float16, device=DEV)
    wide[:, :k] = x
    assert torch.equal(il.int8_linear(wide[:, :k], packed, scale, b, n), y)


def test_without_workspace_runs_in_one_range():
    from runtime_amd.phase2 import _hip

    m, n, k = 160, 4096, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    q, scale, w = _weights(n, k, g)
    x = torch.randn(m, k, generator=g, device=DEV).half()
    packed = il.pack_weight(q)
    y = torch.empty(m, n, dtype=torch.float16, device=DEV)
    _hip.check(_hip.load().mx_w8a16_linear(x.data_ptr(), m, k, k, packed.data_ptr(), scale.data_ptr(), None, y.data_ptr(),
                                           n, n, None, 0, _hip.stream_handle(x.device)), "mx_w8a16_linear")
    want, bound = _product(x, w)
    assert ((y.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("m,inter,k,bias", GATEUP)
def test_gateup(m, inter, k, bias):
    g = torch.Generator(device=DEV).manual_seed(m + inter + k)
    parts = [_weights(inter, k, g) for _ in range(2)]
    biases = [torch.randn(inter, generator=g, device=DEV).half() for _ in range(2)] if bias else [None, None]
    x = torch.randn(m, k, generator=g, device=DEV).half()
    packed = il.pack_weight(il.gateup_interleave(parts[0][0], parts[1][0]))
    scale = il.gateup_interleave(parts[0][1], parts[1][1])
    y = il.int8_gateup_swiglu(x, packed, scale, il.gateup_interleave(*biases) if bias else None, inter)
    (gate, eg), (up, eu) = (_product(x, p[2], b) for p, b in zip(parts, biases))
    s = gate * torch.sigmoid(gate)
    es = 1.1 * eg + (U + 1e-6) * s.abs() + SUB
    want = s * up
    bound = es * up.abs() + eu * (s.abs() + es) + U * want.abs() + SUB
    assert ((y.double() - want).abs() <= bound * (1 + U)).all()
