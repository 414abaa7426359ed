"""Launches on both sides of the sizes where the dense and segmented drivers
change their shape or their accesses (plain or non-temporal, by the bytes of the
operands): the same element math, so the same bits as one replica at a time,
whose calls stay below every such size."""

from __future__ import annotations

import pytest
import torch

import churten_amd.kernels  # noqa: F401

pytestmark = pytest.mark.gpu

MB = 1 << 20
# Operand bytes around 16, 27/28, 48 and 100 MiB, and a consolidated gradient
# around 88 MiB (float32 Adam: 20 bytes per element with it).
SIZES = [15 * MB, 17 * MB, 26 * MB, 29 * MB, 47 * MB, 49 * MB, 99 * MB, 101 * MB]


def operands(R, T, dtype, state, slots, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rt(dt):
        return torch.randn(R, T, device="cuda", generator=g).mul_(0.1).to(dt)

    return [rt(dtype), rt(dtype)] + [rt(state).abs_() for _ in range(slots)]


def step(opt, bufs, steps, hyp, mask, segs=None):
    ops, seg = torch.ops.torchstrap, torch.ops.churten
    if opt == "adam":
        kw = dict(amsgrad=False, maximize=False, decoupled_weight_decay=True)
        if segs is None:
            return ops.adam_step_(*bufs[:4], None, steps, *hyp, mask, **kw)
        return seg.adam_step_segments_(bufs[0], *segs, bufs[1], *bufs[2:4], None, steps, *hyp,
                                       mask, **kw)
    if opt == "sgd":
        kw = dict(nesterov=True, maximize=False)
        if segs is None:
            return ops.sgd_step_(*bufs[:3], steps, *hyp[:4], mask, **kw)
        return seg.sgd_step_segments_(bufs[0], *segs, bufs[1], bufs[2], steps, *hyp[:4], mask,
                                      **kw)
    if segs is None:
        return ops.adagrad_step_(*bufs[:3], steps, *hyp[:4], mask, maximize=False)
    return seg.adagrad_step_segments_(bufs[0], *segs, bufs[1], bufs[2], steps, *hyp[:4], mask,
                                      maximize=False)


def check(opt, dtype, state, nbytes, segmented):
    R, slots = 3, 2 if opt == "adam" else 1
    es, ss = torch.finfo(dtype).bits // 8, torch.finfo(state).bits // 8
    per = 2 * es + slots * ss + (es if segmented else 0)
    T = nbytes // per // R + 1  # just past the size, ragged rows
    bufs = operands(R, T, dtype, state, slots, seed=nbytes % 1000)
    hyp = [torch.full((R,), x, device="cuda", dtype=dtype)
           for x in (1e-2, 0.875, 0.96875, 1e-3, 1e-2)]
    if opt == "adagrad":
        hyp = [hyp[0], hyp[4], hyp[4], hyp[3]]
    if opt == "sgd":
        hyp = [hyp[0], hyp[1], hyp[4], hyp[4]]
    steps = torch.tensor([0.0, 3.0, 7.0], device="cuda", dtype=dtype)
    mask = torch.tensor([True, True, False], device="cuda")
    grads = None
    if segmented:
        cut = T // 3 + 1
        grads = [bufs[1][:, :cut].clone(), bufs[1][:, cut:T - 3].clone()]
        cols = [0, cut]
    want = [b.clone() for b in bufs]
    if segmented:
        bufs[1].fill_(0.25)
        want[1].fill_(0.25)
        want[1][:, :T - 3] = torch.cat(grads, dim=1)
    s2 = steps.clone()
    step(opt, bufs, steps, hyp, mask, (grads, cols) if segmented else None)
    for r in range(R):
        # A quarter row at a time: far below every size, in the dense driver.
        for lo in range(0, T, T // 4 + 1):
            hi = min(T, lo + T // 4 + 1)
            one = s2[r:r + 1].clone()
            step(opt, [b[r:r + 1, lo:hi] for b in want], one, [h[r:r + 1] for h in hyp],
                 mask[r:r + 1])
        s2[r] = one[0]
    assert torch.equal(steps, s2)
    for i, (a, b) in enumerate(zip(bufs, want)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("nbytes", SIZES)
@pytest.mark.parametrize("opt,dtype,state", [
    ("adam", torch.float32, torch.float32), ("adam", torch.float32, torch.bfloat16),
    ("adam", torch.bfloat16, torch.bfloat16), ("adam", torch.float64, torch.float64),
    ("sgd", torch.float32, torch.float32), ("sgd", torch.float16, torch.float16),
    ("sgd", torch.float64, torch.float64), ("adagrad", torch.float32, torch.float32)])
def test_dense_sizes(opt, dtype, state, nbytes):
    check(opt, dtype, state, nbytes, segmented=False)


@pytest.mark.parametrize("nbytes", [100 * MB, 255 * MB, 257 * MB])
def test_sgd_sizes_on_the_small_tile(nbytes):
    check("sgd", torch.float32, torch.float32, nbytes, segmented=False)
    check("sgd", torch.float32, torch.bfloat16, nbytes, segmented=False)


@pytest.mark.parametrize("nbytes", [639 * MB, 641 * MB])
def test_dense_sizes_in_one_and_two_launches(nbytes):
    check("adagrad", torch.float32, torch.bfloat16, nbytes, segmented=False)


@pytest.mark.parametrize("nbytes", [26 * MB, 28 * MB, 99 * MB, 101 * MB, 430 * MB, 450 * MB])
@pytest.mark.parametrize("opt,dtype,state", [
    ("adam", torch.float32, torch.float32), ("adam", torch.float32, torch.bfloat16),
    ("adam", torch.bfloat16, torch.bfloat16), ("sgd", torch.float32, torch.float32),
    ("adagrad", torch.float32, torch.float32)])
def test_segmented_sizes(opt, dtype, state, nbytes):
    check(opt, dtype, state, nbytes, segmented=True)
