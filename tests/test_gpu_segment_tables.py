"""Segment tables around the entries one launch takes (128, gaps included): the
scatter against per-parameter copies and the segmented update against scatter
then update, bit for bit."""

from __future__ import annotations

import pytest
import torch

import churten_amd.kernels  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("gaps", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 300])
def test_tables(n, gaps, dtype):
    R = 3
    g = torch.Generator(device="cuda").manual_seed(n)
    widths = torch.randint(1, 700, (n,), generator=torch.Generator().manual_seed(n)).tolist()
    cols, at = [], 0
    for i, w in enumerate(widths):
        at += (1 + i % 3) if gaps else 0
        cols.append(at)
        at += w
    T = at + (5 if gaps else 0)

    def rt(std):
        return torch.randn(R, T, device="cuda", generator=g).mul_(std).to(dtype)

    def vec(x):
        return torch.full((R,), x, device="cuda", dtype=dtype)

    grads = [torch.randn(R, w, device="cuda", generator=g).to(dtype) for w in widths]
    dst = rt(1.0)
    want = dst.clone()
    for c, t in zip(cols, grads):
        want[:, c:c + t.shape[1]] = t
    torch.ops.churten.scatter_grads_(dst, grads, cols)
    assert torch.equal(dst, want)

    mask = torch.tensor([True, False, True], device="cuda")
    start = [rt(0.1), rt(0.01), rt(0.01).abs_(), rt(0.01).abs_()]
    hyp = [vec(1e-2), vec(0.9), vec(0.98), vec(1e-3), vec(1e-2)]
    kw = dict(amsgrad=False, maximize=False, decoupled_weight_decay=True)
    a, sa = [t.clone() for t in start], vec(3.0)
    torch.ops.churten.adam_step_segments_(a[0], grads, cols, a[1], a[2], a[3], None, sa, *hyp,
                                          mask, **kw)
    b, sb = [t.clone() for t in start], vec(3.0)
    torch.ops.churten.scatter_grads_(b[1], grads, cols)
    torch.ops.torchstrap.adam_step_(*b, None, sb, *hyp, mask, **kw)
    assert torch.equal(sa, sb)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
