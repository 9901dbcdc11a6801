"""The input producers' many-token kernel (more than 32 tokens, or rmsfold with an output over its input, of rows that are not
narrow) against the few-token one on the same rows: 8 columns a thread instead of one changes no pair of the transform and no order of the norm,
so every output has the same bits; odd strides and alignments take its scalar loads and stores."""
import numpy as np
import pytest
import torch

from kt_cases import say, dev, rng

pytestmark = pytest.mark.gpu
FEW = 32


def _in(t, pad, shift):
    """the rows of t in a wider buffer: row stride + pad elements, base shifted by `shift` elements"""
    M, C = t.shape
    buf = torch.full((M * (C + pad) + shift + 8,), float("nan") if t.dtype == torch.float32 else 7, dtype=t.dtype, device="cuda")
    v = buf[shift:shift + M * (C + pad)].view(M, C + pad)[:, :C]
    v.copy_(t)
    return v


def _act(lin, M, C, hp, pad):
    Mq = 2 * M if hp else M
    q = torch.zeros((Mq, C + pad), dtype=torch.int8, device="cuda")[:, :C]
    return lin.Act(q, torch.empty((Mq, C // 128), device="cuda"),
                   torch.empty((Mq, C // 128), dtype=torch.int32, device="cuda"), M, C, False, hp)


def _same(a, b):
    return torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# HB 512 (a wave), 1024 (two), 4096 (eight); widths of one wave, of a partial last 4096-column chunk, of many chunks
@pytest.mark.parametrize("C,HB", [(512, 512), (1536, 512), (1024, 1024), (5120, 1024), (6144, 1024), (4096, 4096), (8192, 4096)])
@pytest.mark.parametrize("hp", [False, True])
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 4), (1, 3)])
def test_many_equals_few(C, HB, hp, pad, shift):
    from kindi_amd import linear as lin
    M, nparts = 37, 2
    say("fold many", C, HB, hp, pad, shift)
    r = rng(C + HB + pad)
    x = _in(dev(r.standard_normal((M, C)).astype(np.float32)), pad, shift)
    b = _in(dev(r.standard_normal((M, C)).astype(np.float32)), pad, shift)
    x[3] = 0.0
    x[4, :128] *= 1e-30
    parts = dev(r.standard_normal((M, nparts * C)).astype(np.float32))
    w = _in(dev((1 + 0.2 * r.standard_normal((1, C))).astype(np.float32)), 0, shift)[0]
    sg = _in(dev(np.where(r.random((1, C)) < 0.5, -1, 1).astype(np.float32)), 0, shift)[0]
    perm = (C // 512, 128, 4) if C % 1024 else (24, C // 48, 2) if C % 48 == 0 else (C // 64, 32, 2)

    def run(rows, order):
        o = [_in(torch.zeros((rows.stop - rows.start, C), device="cuda"), pad, shift) for _ in range(5)]
        acts = [_act(lin, rows.stop - rows.start, C, hp, pad) for _ in range(3)]
        lin.rmsfold(x[rows], w, sg, HB, r=parts[rows], nparts=nparts, xw=o[0], xn=o[1], xo=o[2], out=acts[0], hp=hp)
        lin.fold(x[rows], sg, HB, xo=o[3], out=acts[1], hp=hp)
        lin.smfold(x[rows], b[rows], sg, HB, perm=order, xo=o[4], out=acts[2], hp=hp)
        return o + [t for a in acts for t in (a.XQ, a.XS, a.XA)]

    for order in ((1, 1, 1), perm):
        many = run(slice(0, M), order)
        few = [run(slice(i, min(i + FEW, M)), order) for i in range(0, M, FEW)]
        for k, t in enumerate(many):
            assert _same(t, torch.cat([f[k] for f in few])), (k, order)


@pytest.mark.parametrize("C,HB,few", [(512, 512, "rmsfold smfold"), (1024, 1024, "rmsfold smfold"), (1024, 512, "rmsfold"), (1536, 512, ""),
                                      (2048, 1024, "")])
def test_narrow_rows_route(C, HB, few):
    """more than 32 tokens of narrow rows stay with the few-token kernel (no dynamic LDS): the other one's waves would idle"""
    from kindi_amd import linear as lin
    M = 40
    x, sg = torch.randn((M, C), device="cuda"), torch.ones(C, device="cuda")
    xw, act = torch.empty_like(x), _act(lin, M, C, False, 0)
    calls = {"rmsfold": lambda: lin.rmsfold(x, sg, sg, HB, r=x, nparts=1, xw=xw, out=act),
             "fold": lambda: lin.fold(x, sg, HB, out=act), "smfold": lambda: lin.smfold(x, x, sg, HB, out=act)}
    for name, fn in calls.items():
        plan = lin.Plan(fn, 2)
        assert plan.n == 1 and (plan.recs[0].shmem == 0) == (name in few.split()), (name, plan.recs[0].shmem)


def test_outputs_over_inputs():
    """rmsfold's outputs over x (any token count), narrow rows among them"""
    from kindi_amd import linear as lin
    M, C = 40, 6144
    r = rng(9)
    for n, hb in ((512, 512), (1024, 512), (1024, 1024)):                # narrow rows: the few-token kernel, a block a row
        x, b = (dev(r.standard_normal((M, n)).astype(np.float32)) for _ in range(2))
        sg = dev(np.where(r.random(n) < 0.5, -1, 1).astype(np.float32))
        for m in (1, M):
            out = torch.empty((m, n), device="cuda")
            a0 = lin.rmsfold(x[:m], sg, sg, hb, r=b[:m], nparts=1, xw=out)
            y = x[:m].clone()
            a1 = lin.rmsfold(y, sg, sg, hb, r=b[:m], nparts=1, xw=y)
            assert _same(y, out) and _same(a0.XQ, a1.XQ) and _same(a0.XS, a1.XS)
    x, b = (dev(r.standard_normal((M, C)).astype(np.float32)) for _ in range(2))
    w, sg = torch.ones(C, device="cuda"), dev(np.where(r.random(C) < 0.5, -1, 1).astype(np.float32))
    for m in (1, M):
        out = [torch.empty((m, C), device="cuda") for _ in range(3)]
        a0 = lin.rmsfold(x[:m], w, sg, 1024, r=b[:m], nparts=1, xw=out[0], xn=out[1], xo=out[2])
        y = x[:m].clone()
        a1 = lin.rmsfold(y, w, sg, 1024, r=b[:m], nparts=1, xo=y)
        assert _same(y, out[2]) and _same(a0.XQ, a1.XQ) and _same(a0.XS, a1.XS)


# one token to more than the few-token kernel's 32, rows of one chunk and of several, up to the widest that LDS holds
@pytest.mark.parametrize("M,C,HB,perm", [(1, 6144, 1024, (128, 24, 2)), (32, 6144, 1024, (128, 24, 2)), (40, 6144, 1024, (128, 24, 2)),
                                         (1, 12288, 4096, (128, 16, 6)), (40, 12288, 4096, (128, 16, 6)), (3, 1024, 1024, (128, 2, 4)),
                                         (3, 1024, 512, (128, 2, 4)), (2, 36352, 512, (256, 2, 71)), (2, 35840, 1024, (256, 20, 7)), (2, 32768, 4096, (128, 128, 2))])
@pytest.mark.parametrize("over", ["a", "b"])
def test_smfold_in_place_grouped_heads(M, C, HB, perm, over):
    """smfold's xo over one of its inputs in the grouped-head order, where a chunk reads other chunks' columns: the outputs
    of the call with an xo of its own"""
    from kindi_amd import linear as lin
    say("smfold in place", M, C, HB, perm, over)
    r = rng(C + M)
    a, b = (dev(r.standard_normal((M, C)).astype(np.float32)) for _ in range(2))
    sg = dev(np.where(r.random(C) < 0.5, -1, 1).astype(np.float32))
    want = torch.empty_like(a)
    a0 = lin.smfold(a, b, sg, HB, perm=perm, xo=want)
    y = (a if over == "a" else b).clone()
    a1 = lin.smfold(y if over == "a" else a, y if over == "b" else b, sg, HB, perm=perm, xo=y)
    assert _same(y, want) and all(_same(u, v) for u, v in zip((a0.XQ, a0.XS, a0.XA), (a1.XQ, a1.XS, a1.XA)))


def test_smfold_in_place_refused_past_lds():
    from kindi_amd import gpudrv, linear as lin
    C, sg = 36864, torch.ones(36864, device="cuda")
    a, b = torch.randn((1, C), device="cuda"), torch.randn((1, C), device="cuda")
    with pytest.raises(gpudrv.KernelError):
        lin.smfold(a, b, sg, 512, perm=(128, 144, 2), xo=a)
    lin.smfold(a, b, sg, 512, perm=(128, 144, 2), xo=torch.empty_like(a))       # not in place, and the plain order: taken
    lin.smfold(a, b, sg, 512, perm=(18432, 1, 2), xo=a)


# rows of one buffer that lie between one another and do not meet: [a | b | xo] of one stride, and an xo of twice a's stride;
# widths that LDS holds and wider
@pytest.mark.parametrize("C", [6144, 36864])
@pytest.mark.parametrize("M", [1, 3, 40])
def test_smfold_between_rows(C, M):
    from kindi_amd import linear as lin
    say("smfold between rows", M, C)
    r = rng(C + M)
    sg = dev(np.where(r.random(C) < 0.5, -1, 1).astype(np.float32))
    a, b = (dev(r.standard_normal((M, C)).astype(np.float32)) for _ in range(2))
    want = torch.empty_like(a)
    perm = (128, C // 256, 2)
    a0 = lin.smfold(a, b, sg, 512, perm=perm, xo=want)
    one = torch.zeros((M, 3 * C), device="cuda")
    two = torch.zeros((2 * M, 2 * C), device="cuda")
    for av, xo in ((one[:, :C], one[:, 2 * C:]), (two[:M, :C], two.view(M, 4 * C)[:, C:2 * C])):
        av.copy_(a)
        a1 = lin.smfold(av, b, sg, 512, perm=perm, xo=xo)
        assert _same(xo, want) and _same(av, a) and all(_same(u, v) for u, v in zip((a0.XQ, a0.XS, a0.XA), (a1.XQ, a1.XS, a1.XA)))
