"""A call whose workspace has room for its entries (128 bytes per replica) runs
as one launch: the update's own head workgroups bump the steps and publish the
per-replica constants (optim_drivers.h, "One launch per call"). Whatever a
workgroup finds in its entry -- this launch's constants, an earlier launch's, or
what the memory held before -- the results are those of the two-launch form,
bit for bit. Same inputs through both, three calls on one workspace."""

from __future__ import annotations

import ctypes
from pathlib import Path

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
_P, _I64, _U32, _SZ = ctypes.c_void_p, ctypes.c_int64, ctypes.c_uint32, ctypes.c_size_t
AMSGRAD, ADAMW, NESTEROV, BUMP, STATE_BF16, ADAGRAD_F32 = 0x1, 0x2, 0x8, 0x10, 0x20, 0x40
CODES = {torch.float32: 0, torch.float64: 1, torch.float16: 2, torch.bfloat16: 3}
F32, F64, F16, BF16 = torch.float32, torch.float64, torch.float16, torch.bfloat16


class RtBuf(ctypes.Structure):
    _fields_ = [("data", _P), ("stride_r", _I64), ("stride_t", _I64)]


class Segment(ctypes.Structure):
    _fields_ = [("data", _P), ("stride_r", _I64), ("col", _I64), ("numel", _I64)]


LIB = ctypes.CDLL(str(Path(__file__).resolve().parents[1] / "churten_amd" / "lib"
                      / "libchurten_optim.so"))
LIB.ts_single_launch_bytes.restype = _SZ
LIB.ts_single_launch_bytes.argtypes = [_I64]

# (optimizer, parameter dtype, state dtype, flags, state buffers)
KINDS = [("adam", F32, F32, 0, 2), ("adam", F32, F32, ADAMW | AMSGRAD, 3),
         ("adam", F32, BF16, ADAMW, 2), ("adam", F64, F64, 0, 2), ("adam", F16, F16, 0, 2),
         ("adam", BF16, BF16, 0, 2), ("sgd", F32, F32, NESTEROV, 1), ("sgd", F32, F32, 0, 0),
         ("sgd", BF16, BF16, 0, 1), ("sgd", F64, F64, 0, 1), ("adagrad", F32, F32, 0, 1),
         ("adagrad", F16, F16, 0, 1), ("adagrad", F32, BF16, ADAGRAD_F32, 1)]
CONSTANTS = {"adam": 2, "sgd": 1, "adagrad": 1}


def make(kind, R, T, seed, strided=False):
    op, dt, st, _, n = kind
    g = torch.Generator(device=DEV).manual_seed(seed)

    def rt(std, dtype):
        t = torch.randn(R, T, device=DEV, generator=g).mul_(std)
        return t.to(dtype)

    bufs = [rt(0.1, dt), rt(0.01, dt)] + [rt(0.01, st).abs_() for _ in range(n)]
    steps = torch.randint(0, 3, (R,), device=DEV, generator=g).to(dt)
    mask = torch.rand(R, device=DEV, generator=g) < 0.8
    mask[0] = True
    if R > 2:
        mask[1], steps[1] = False, 0.0  # frozen before its first step
        for b in bufs[2:]:
            b[1] = float("nan")
    u = torch.rand(R, device=DEV, generator=g)
    hyp = {"adam": [u * 1e-2, 0.8 + u * 0.1, 0.9 + u * 0.09, u * 0 + 1e-3, u * 1e-2],
           "sgd": [u * 1e-2, 0.5 + u * 0.4, u * 0.1, u * 1e-2],
           "adagrad": [u * 1e-2, u * 1e-2, u * 1e-2, u * 0 + 1e-3]}[op]
    return bufs, steps, mask, [h.to(dt) for h in hyp]


def call(kind, bufs, steps, mask, hyp, ws, ws_bytes, bump=True, segs=None):
    """One call; ``segs``: (col, tensor) gradients, bufs[1] receiving them."""
    op, dt, st, flags, _ = kind
    R, T = bufs[0].shape
    if bump:
        flags |= BUMP
    if st != dt:
        flags |= STATE_BF16
    rt = [RtBuf(b.data_ptr(), b.stride(0), b.stride(1)) if b is not None else RtBuf(None, 0, 1)
          for b in bufs]
    table = (RtBuf * 5)(*(rt + [RtBuf(None, 0, 1)] * (5 - len(rt))))
    out = torch.full((), 7.0, device=DEV, dtype=dt)
    args = [table]
    name = f"ts_{op}_step_ws"
    if segs is not None:
        name = f"ts_{op}_step_segments_ws"
        args += [(Segment * len(segs))(*[Segment(t.data_ptr(), t.stride(0), c, t.shape[1])
                                         for c, t in segs]), ctypes.c_int(len(segs))]
    args += [ctypes.c_int(CODES[dt]), _P(steps.data_ptr()), *[_P(h.data_ptr()) for h in hyp],
             _P(mask.data_ptr()), _I64(R), _I64(T), _U32(flags), _P(out.data_ptr()),
             _P(ws.data_ptr()), _SZ(ws_bytes),
             _P(torch.cuda.current_stream().cuda_stream)]
    assert getattr(LIB, name)(*args) == 0
    return out


def clone(bufs):
    return [None if b is None else b.clone() for b in bufs]


def bits(t):
    size = {2: torch.int16, 4: torch.int32, 8: torch.int64}[t.element_size()]
    return t.view(size)


def check_same(kind, bufs, steps, mask, hyp, fill, calls=3, bump=True, segs=None):
    R = mask.numel()
    assert LIB.ts_single_launch_bytes(R) == 128 * R
    one, two = clone(bufs), clone(bufs)
    s1, s2 = steps.clone(), steps.clone()
    w1 = torch.full((128 * R,), fill, device=DEV, dtype=torch.uint8)
    w2 = torch.full((16 * R,), fill, device=DEV, dtype=torch.uint8)
    for k in range(calls):
        before = w1.view(R, 128).clone()
        z = call(kind, one, s1, mask, hyp, w1, 128 * R, bump, segs)
        call(kind, two, s2, mask, hyp, w2, 16 * R, bump, segs)
        torch.cuda.synchronize()
        assert float(z) == 0.0
        assert torch.equal(bits(s1), bits(s2)), k
        for i, (a, b) in enumerate(zip(one, two)):
            if a is not None:
                assert torch.equal(bits(a), bits(b)), (k, i)
        # The launch published: every active replica's entry is new, and
        # nothing else of the workspace has changed.
        words = 16 * CONSTANTS[kind[0]]
        changed = w1.view(R, 128) != before
        assert bool(changed[:, :words].any(dim=1)[mask].all())
        assert not bool(changed[~mask].any()) and not bool(changed[:, words:].any())


# One element, less than a pack, a row and a bit over one tile, a ragged row
# over several, rows past the workgroups that look at memory first (4096), and
# the most replicas a single launch takes.
SHAPES = [(1, 1), (3, 3), (3, 4), (5, 1027), (4, 70001), (2, 4_500_001), (1024, 36)]


@pytest.mark.parametrize("kind", KINDS, ids=lambda k: f"{k[0]}-{k[1]}-{k[2]}-{k[3]}-{k[4]}")
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_single_launch_matches_two(kind, shape):
    args = make(kind, *shape, seed=shape[1] + 31 * len(kind))
    check_same(kind, *args, fill=(0xFF if shape[0] > 2 else 0), calls=3)


@pytest.mark.parametrize("kind", [KINDS[0], KINDS[6], KINDS[10]], ids=lambda k: k[0])
def test_steps_not_bumped(kind):
    check_same(kind, *make(kind, 6, 3001, seed=3), fill=0, bump=False)


@pytest.mark.parametrize("kind", [KINDS[0], KINDS[2], KINDS[5], KINDS[6], KINDS[8], KINDS[11]],
                         ids=lambda k: f"{k[0]}-{k[1]}-{k[2]}")
@pytest.mark.parametrize("kept", [True, False])
@pytest.mark.parametrize("n_segs", [1, 70])
def test_segments(kind, kept, n_segs):
    """70 segments with gaps take more than one launch: only the first has the
    heads."""
    R, width = 5, 700
    T = n_segs * width + 13
    bufs, steps, mask, hyp = make(kind, R, T, seed=n_segs)
    g = torch.Generator(device=DEV).manual_seed(9)
    segs = [(i * width + 3, torch.randn(R, width - 5, device=DEV, generator=g).to(kind[1]))
            for i in range(n_segs)]
    if not kept:
        bufs[1] = None
    check_same(kind, bufs, steps, mask, hyp, fill=0x5A, segs=segs)


SGD = [KINDS[6], KINDS[7], KINDS[8], KINDS[9], ("sgd", F32, BF16, 0, 1)]


@pytest.mark.parametrize("kind", SGD, ids=lambda k: f"{k[1]}-{k[2]}-{k[4]}")
@pytest.mark.parametrize("n_segs", [0, 1, 70])
@pytest.mark.parametrize("n", [3, 70001])
def test_sgd_counters_below_zero(kind, n, n_segs):
    """A counter may start anywhere. From -1 the new step is 0, which is also
    the old step of a first one: the momentum buffer is read and kept there, and
    a first step is where the *new* step is 1 (so also from a counter that a bump
    rounds to 1). The 70 segments take two launches, the second after the bump."""
    R, T = 9, max(n, 70 * 7 if n_segs else n)
    bufs, steps, mask, hyp = make(kind, R, T, seed=5)
    eps = 2.0 ** -26 if kind[1] == F32 else 2.0 ** -10 if kind[1] == BF16 else 2.0 ** -55
    steps.copy_(torch.tensor([-1, -2, -1, 0, -0.0, -1 + 4 * eps, eps, 1, -3], dtype=F64))
    mask[:] = True
    mask[2] = False
    for b in bufs[2:]:
        b[1] = 0.5
    segs = None
    if n_segs:
        g = torch.Generator(device=DEV).manual_seed(8)
        w = T // n_segs
        segs = [(i * w + 1, torch.randn(R, w - 2, device=DEV, generator=g).to(kind[1]))
                for i in range(n_segs)]
    check_same(kind, bufs, steps, mask, hyp, fill=0, calls=4, segs=segs)


def test_launches_share_one_counter():
    """The tags of a launch come from one counter whatever entry point it went
    through, so an entry that another optimizer's launch left is never taken for
    this one's. They are read back from the workspaces: word i of an entry holds
    tag i % 2 in its high half, and the low tag is the counter times an odd
    number."""
    odd, counts = 0x9E3779B1, []
    for i, kind in enumerate([KINDS[0], KINDS[6], KINDS[10]] * 2):
        for segmented in (False, True):
            bufs, steps, mask, hyp = make(kind, 2, 64, seed=i)
            segs = [(0, bufs[1].clone())] if segmented else None
            ws = torch.zeros(128 * 2, device=DEV, dtype=torch.uint8)
            call(kind, bufs, steps, mask, hyp, ws, 128 * 2, segs=segs)
            words = ws.view(torch.int64).cpu().tolist()
            low = (words[0] >> 32) & 0xFFFFFFFF
            counts.append(low * pow(odd, -1, 2 ** 32) % 2 ** 32)
    assert [(c - counts[0]) % 2 ** 32 for c in counts] == list(range(len(counts)))


def test_replica_limit():
    assert LIB.ts_single_launch_bytes(1024) == 128 * 1024
    assert LIB.ts_single_launch_bytes(1025) == 0 and LIB.ts_single_launch_bytes(0) == 0
    kind = KINDS[0]
    bufs, steps, mask, hyp = make(kind, 1025, 36, seed=1)
    other, s2 = clone(bufs), steps.clone()
    ws = torch.zeros(128 * 1025, device=DEV, dtype=torch.uint8)
    call(kind, bufs, steps, mask, hyp, ws, 128 * 1025)
    call(kind, other, s2, mask, hyp, ws, 16 * 1025)
    assert torch.equal(steps, s2)
    for a, b in zip(bufs, other):
        assert torch.equal(bits(a), bits(b))


def test_operands_without_unit_inner_stride():
    """A (T, R) buffer seen as (R, T) takes the other drivers, in two launches."""
    kind = KINDS[0]
    bufs, steps, mask, hyp = make(kind, 6, 515, seed=2)
    minor = [b.t().contiguous().t() for b in bufs]
    s2 = steps.clone()
    ws = torch.zeros(128 * 6, device=DEV, dtype=torch.uint8)
    call(kind, minor, steps, mask, hyp, ws, 128 * 6)
    call(kind, bufs, s2, mask, hyp, ws, 16 * 6)
    assert torch.equal(steps, s2)
    for a, b in zip(minor, bufs):
        assert torch.equal(bits(a.contiguous()), bits(b))
