"""GPU: the prompt branch of the block_paged attention hook (mx_prefill_attn) against softmax attention in float64.

Bound: the kernel's scores and softmax are fp32 (1e-4 relative covers sums of D products and exp2
over the drawn scores), the weights are rounded once to the element type (relative u, or half the
smallest subnormal), and the output is the product of those rounded weights with V, rounded again.
"""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from runtime_amd.phase2 import block_paged_attention as bpa

pytestmark = pytest.mark.gpu
DEV = "cuda"
UNIT = {torch.float16: (2.0**-11, 2.0**-25), torch.bfloat16: (2.0**-8, 0.0)}


def _reference(q, k, v, scaling, groups):
    q, k, v = (t.double().cpu() for t in (q, k, v))
    k, v = (t.repeat_interleave(groups, dim=1) for t in (k, v))
    p, s = q.shape[2], k.shape[2]
    scores = torch.matmul(q, k.transpose(2, 3).contiguous()) * scaling
    w = torch.softmax(scores.masked_fill(bpa._causal_block(p, s, q.device), float("-inf")), dim=-1)
    return w, torch.matmul(w, v), torch.matmul(w, v.abs()), v.abs().sum(dim=2, keepdim=True)


def _check(q, k, v, scaling, groups):
    assert bpa._prefill_kernel_takes(q, k, v, scaling, groups)
    out, weights = bpa.block_paged_attention_forward(
        SimpleNamespace(num_key_value_groups=groups, training=False), q, k, v, None, scaling)
    w, o, wv, vsum = _reference(q, k, v, scaling, groups)
    u, sub = UNIT[q.dtype]
    b, hq, p, d = q.shape
    assert out.shape == (b, p, hq, d) and out.is_contiguous() and weights.shape == w.shape
    rel = u + 1e-4
    assert ((weights.double().cpu() - w).abs() <= rel * w + sub + 1e-9).all()
    assert (weights.cpu()[w == 0] == 0).all()
    bound = (rel + u) * wv + u * o.abs() + sub * vsum + 1e-7
    assert ((out.transpose(1, 2).double().cpu() - o).abs() <= bound).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hkv,groups,p,past", [
    (1, 1, 2, 0), (2, 7, 15, 0), (2, 4, 16, 1), (1, 4, 17, 47), (2, 7, 33, 31), (1, 3, 63, 0), (2, 1, 64, 64),
    (1, 4, 65, 0), (2, 7, 129, 176), (8, 4, 1030, 0), (8, 8, 520, 24),
])
def test_against_float64(d, dtype, hkv, groups, p, past):
    g = torch.Generator().manual_seed(1000 * p + past + d)
    s = p + past

    def rows(t, h):  # [1, h, t, d] strided as a decoder layer's reshaped projection
        return torch.randn(1, t, h, d, generator=g).to(dtype).to(DEV).transpose(1, 2)

    _check(rows(p, hkv * groups), rows(s, hkv), rows(s, hkv), d**-0.5, groups)


@pytest.mark.parametrize("form", ["contiguous", "sliced", "batch", "expanded"])
def test_strides(form):
    g = torch.Generator().manual_seed(3)
    b = 3 if form in ("batch", "expanded") else 1
    q = torch.randn(b, 6, 40, 64, generator=g).half().to(DEV)
    k, v = (torch.randn(1 if form == "expanded" else b, 2, 72, 64, generator=g).half().to(DEV) for _ in range(2))
    if form == "sliced":  # a gathered row: whole blocks, cut to the length
        k, v = k[:, :, :59], v[:, :, :59]
    if form == "expanded":
        k, v = k.expand(b, -1, -1, -1), v.expand(b, -1, -1, -1)
    _check(q, k, v, 0.125, 3)


def test_a_non_finite_row_is_nan_everywhere_and_leaves_the_others_alone():
    g = torch.Generator().manual_seed(4)
    q = torch.randn(1, 2, 100, 64, generator=g).half().to(DEV)
    k, v = (torch.randn(1, 2, 100, 64, generator=g).half().to(DEV) for _ in range(2))
    clean = bpa.block_paged_attention_forward(SimpleNamespace(num_key_value_groups=1, training=False), q, k, v, None, 0.125)
    q[0, 1, 5, 3] = float("nan")
    q[0, 1, 70, 3] = float("inf")
    out, weights = bpa.block_paged_attention_forward(SimpleNamespace(num_key_value_groups=1, training=False), q, k, v,
                                                     None, 0.125)
    bad = torch.zeros(2, 100, dtype=torch.bool, device=DEV)
    bad[1, 5] = bad[1, 70] = True
    assert weights[0][bad].isnan().all() and torch.equal(weights[0][~bad], clean[1][0][~bad])
    rows = bad.t()
    assert out[0][rows].isnan().all() and torch.equal(out[0][~rows], clean[0][0][~rows])


def test_what_the_kernel_leaves_to_the_eager_chain():
    q = torch.randn(1, 4, 8, 64, device=DEV, dtype=torch.float16)
    k = torch.randn(1, 2, 8, 64, device=DEV, dtype=torch.float16)
    takes = bpa._prefill_kernel_takes
    assert takes(q, k, k, 0.125, 2)
    assert not takes(q.float(), k.float(), k.float(), 0.125, 2)
    assert not takes(q[..., :32], k[..., :32], k[..., :32], 0.125, 2)
    assert not takes(q, k[:, :, :7], k[:, :, :7], 0.125, 2)   # fewer keys than queries
    assert not takes(q, k, k, -0.125, 2) and not takes(q, k, k, torch.tensor(0.125), 2)
    assert not takes(q[:, :, 1:2], k, k, 0.125, 2)            # one query: every key is visible, no launch saved
    odd = torch.randn(1, 2, 8, 66, device=DEV, dtype=torch.float16)[..., 1:65]
    assert not takes(q, odd, odd, 0.125, 2)
    assert not takes(q.clone().requires_grad_(), k, k, 0.125, 2)
    with torch.no_grad():
        assert takes(q.clone().requires_grad_(), k, k, 0.125, 2)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not takes(q, k, k, 0.125, 2)
    with torch.autograd.forward_ad.dual_level():
        assert not takes(q, k, k, 0.125, 2)
    seen = []
    torch.vmap(lambda x: seen.append(takes(x, k, k, 0.125, 2)) or x)(torch.stack([q, q]))
    assert seen == [False]
    module = SimpleNamespace(num_key_value_groups=2, training=True)
    qg = q.clone().requires_grad_()
    out, _ = bpa.block_paged_attention_forward(module, qg, k, k, None, 0.125)
    out.float().sum().backward()
    assert qg.grad is not None


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,s", [(64, 100), (128, 320), (64, 129)])
def test_a_row_whose_visible_scores_are_all_minus_infinity_is_nan_everywhere(dtype, d, s):
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn(1, 2, s, d, generator=g).to(DEV, dtype) for _ in range(3))
    module = SimpleNamespace(num_key_value_groups=1, training=False)
    k[0, :, 0, 3] = -1.0
    q[0, 1, 0, 3] = float("inf")  # row 0 sees token 0 alone: its score is -inf
    base = bpa.block_paged_attention_forward(module, q[:, :1], k[:, :1], v[:, :1], None, 0.125)
    out, weights = bpa.block_paged_attention_forward(module, q, k, v, None, 0.125)
    assert weights[0, 1, 0].isnan().all() and out[0, 0, 1].isnan().all()
    assert torch.equal(weights[0, :1], base[1][0]) and torch.equal(out[0, :, :1], base[0][0])
    assert weights[0, 1, 1:].isfinite().all() and out[0, 1:, 1].isfinite().all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("scaling", [1e-50, 1e-42, 1e-37, 2.9e38, True])
def test_any_positive_scale_gives_the_eager_chain_s_weights(dtype, scaling):
    """Scales that fp32 does not hold, or not times log2(e), are left to the eager chain."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 2, 80, 64, generator=g).to(DEV, dtype) for _ in range(3))
    q, k = q / 64, k / 64
    if scaling > 1:  # the scores stay finite: 0
        q = torch.zeros_like(q)
    out, weights = bpa.block_paged_attention_forward(
        SimpleNamespace(num_key_value_groups=1, training=False), q, k, v, None, scaling)
    scores = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3).contiguous()) * scaling
    w = torch.softmax(scores.masked_fill(bpa._causal_block(80, 80, scores.device), float("-inf")), dim=-1)
    u, sub = UNIT[dtype]
    # The eager chain rounds a score twice to the element type: at most 2 u |score| on each exponent.
    rel = u + 1e-4 + 2 * (2 * u) * scores.abs().max().item()
    assert ((weights.double().cpu() - w).abs() <= rel * w + sub + 1e-9).all()
    assert out.isfinite().all()
