"""The many-token q8_0 product (k_q8_gemm), grouped and dense, and the dense dispatch around it: kt_q8_gemv's bits at every
list length and width, int32 unit values exact against the oracle."""
import re
import os
import subprocess

import numpy as np
import pytest
import torch

import oracle as orc
from kt_cases import say, q8_case, dev, host, rng

gpu = pytest.mark.gpu


def _single(W, Q, D):
    """the product a token at a time (the one-token kernel, pinned to the oracle's tree elsewhere)"""
    return torch.cat([W.gemv(Q[i:i + 1].contiguous(), D[i:i + 1].contiguous()) for i in range(Q.shape[0])])


# widths: units 1, 3, 8 (one step), 9, 17 and 58 (a short last step), 84 (slices of one and two steps), 128, 136 (more
# than 8 slices) and 512 (16 slices); list lengths around the tile of 32 and the pass of 64, an empty list among them
LENS = [0, 1, 31, 32, 33, 64, 65, 130]


@gpu
@pytest.mark.parametrize("C", [32, 96, 256, 288, 544, 1856, 2688, 4096, 4352, 16384])
@pytest.mark.parametrize("R", [8, 100, 129])
def test_grouped_lists(R, C):
    assert sum(LENS) >= 10 * len(LENS)
    _grouped(R, C, LENS)


# 4 to 6 entries an expert: k_q8_mma (its lists around the pass of 16; one and several slices a wave, odd counts)
FEW = [0, 1, 3, 15, 16, 2, 17, 1]


@gpu
@pytest.mark.parametrize("C", [32, 96, 288, 544, 1536, 1856, 2688, 4096])
@pytest.mark.parametrize("R", [8, 100])
def test_grouped_few(R, C):
    assert 4 * len(FEW) <= sum(FEW) < 7 * len(FEW)
    _grouped(R, C, FEW)


# lists of more than one pass a block: 64 P entries a round of the P blocks that share a row tile (P = 3 below 64 entries an
# expert on average, 7 from there on), so second and third passes of one and two tiles, and blocks with no pass at all
LONG3 = [0, 1, 420, 33, 2, 3, 0, 5]
LONG3B = [193, 0, 257, 1, 0, 2, 1, 0]
LONG7 = [0, 1, 449, 520, 64, 96, 3, 30]


@gpu
@pytest.mark.parametrize("lens", [LONG3, LONG3B, LONG7], ids=["three", "three_b", "seven"])
@pytest.mark.parametrize("C", [256, 512, 1856, 2688, 4352])       # one slice, one of two steps, 4, 6 (the last short), 9 slices
def test_grouped_passes(C, lens):
    mean = sum(lens) // len(lens)
    assert 12 <= mean and (mean >= 64) == (lens is LONG7) and max(lens) > 64 * (7 if mean >= 64 else 3)
    _grouped(100, C, lens)


# k_q8_mma's activations straight into the operand and through LDS: 5 and 8 entries an expert over 1 to 8 slices, lists around a
# pass of 16 and of two passes
FIVE = [0, 1, 16, 17, 2, 3, 1, 0]
EIGHT = [0, 1, 16, 17, 30, 2, 1, 0]


@gpu
@pytest.mark.parametrize("lens", [FIVE, EIGHT], ids=["five", "eight"])
@pytest.mark.parametrize("C", [512, 768, 1856, 2688, 3584, 4096])
def test_grouped_either_way(C, lens):
    assert sum(lens) // len(lens) == (5 if lens is FIVE else 8)
    _grouped(100, C, lens)


# few entries an expert on a small grid: the blocks with the lists' first passes before all others (a second pass of the first
# ones at 200 entries), numbers of row tiles that are no multiple of 8, an idle expert last
FIRST = [200, 0, 70, 33, 1] + [0] * 8 + [2, 1, 64, 0, 0, 0, 0, 7, 0, 0, 0, 5, 0]


@gpu
@pytest.mark.parametrize("R,C", [(100, 512), (129, 1856), (300, 2688), (129, 4352)])
def test_grouped_first_passes_first(R, C):
    assert 11 * len(FIRST) <= sum(FIRST) < 16 * len(FIRST) and max(FIRST) > 192
    _grouped(R, C, FIRST)


def _active(cnt):
    """the active experts in ascending order (E entries, the tail unused) and how many there are"""
    on = np.flatnonzero(cnt)
    act = np.zeros(len(cnt), np.int32)
    act[:len(on)] = on
    return act, np.array([len(on)], np.int32)


@pytest.mark.parametrize("lens", [LENS, FEW, LONG3, LONG3B, LONG7, FIVE, EIGHT, FIRST])
def test_lists_are_whole(lens):
    """the lists that the tests here hand to the kernel, which trusts them: every active expert once, none past the table"""
    act, nact = _active(np.array(lens, np.int32))
    assert nact[0] <= len(act) == len(lens) and sorted(act[:nact[0]]) == [e for e, c in enumerate(lens) if c]


def _grouped(R, C, lens):
    from kindi_amd import moe
    say("grouped", R, C, lens)
    E, n = len(lens), sum(lens)
    cases = [q8_case(R, C, 1000 * R + C + e) for e in range(E)]
    W = moe.Q8Experts([c[0] for c in cases], R, C)
    M = 70                                                                # input rows, reached through xrow
    Q, D = moe.q8_quantize(dev(rng(C).normal(0, 1, (M, C)).astype(np.float32)))
    cnt = np.array(lens, np.int32)
    off = np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int32)
    xrow = rng(7).integers(0, M, n).astype(np.int32)
    act, nact = _active(cnt)
    lists = (dev(cnt), dev(off), dev(xrow), dev(np.zeros(n, np.int32)), dev(act), dev(nact))
    Y = torch.full((n, R), float("nan"), device="cuda")
    dbg = torch.empty((n, R, C // 32), dtype=torch.int32, device="cuda")
    W.grouped(lists, M, Q, D, Y, dbg=dbg)
    y, g, q = host(Y), host(dbg), host(Q)
    Y2 = torch.full((n, R), float("nan"), device="cuda")
    W.grouped(lists, M, Q, D, Y2)
    assert np.array_equal(host(Y2), y)
    Qe, De = Q[dev(xrow).long()].contiguous(), D[dev(xrow).long()].contiguous()
    Y3 = torch.full((n, R), float("nan"), device="cuda")
    W.grouped(lists, M, Qe, De, Y3, xrow=False)
    assert np.array_equal(host(Y3), y), "entries' own rows"
    for e in range(E):
        if cnt[e] == 0:
            continue
        sl = slice(int(off[e]), int(off[e] + cnt[e]))
        assert np.array_equal(g[sl], orc.q8_acc(cases[e][0], R, C, q[xrow[sl]])), "int32 unit values"
        one = moe.Q8Matrix(cases[e][0], R, C)
        assert np.array_equal(y[sl], host(_single(one, Qe[sl], De[sl]))), (e, int(cnt[e]))


@gpu
@pytest.mark.parametrize("R,C,M", [(8, 32, 3), (100, 96, 9), (2688, 1856, 5), (4096, 2688, 50), (4100, 2688, 330),
                                   (8192, 4096, 4), (8190, 1024, 161), (4100, 2688, 400), (8190, 1024, 200), (130, 4352, 64), (136, 16384, 65), (136, 8192, 65), (40, 8192, 70),
                                   (8190, 512, 48), (8190, 512, 49), (8190, 1024, 96), (8190, 1024, 97), (136, 4352, 88), (4100, 4352, 16), (4100, 4352, 17), (4090, 4352, 25), (4090, 4352, 43), (4090, 4352, 44),
                                   (5919, 2528, 34), (4130, 1632, 49), (7365, 1696, 242)])
def test_dense_routes(R, C, M):
    from kindi_amd import moe
    say("q8 dense", R, C, M)
    rows, codes, sc = q8_case(R, C, R + C)
    W = moe.Q8Matrix(rows, R, C)
    Q, D = moe.q8_quantize(dev(rng(M).normal(0, 1, (M, C)).astype(np.float32)))
    y = host(W.gemv(Q, D))
    pick = sorted({0, M // 2, M - 1, min(M - 1, 16), min(M - 1, 33), min(M - 1, 64)})
    assert np.array_equal(y[pick], host(_single(W, Q[pick].contiguous(), D[pick].contiguous())))
    if R * C * M < 1 << 26:
        dbg = torch.empty((M, R, C // 32), dtype=torch.int32, device="cuda")
        assert np.array_equal(host(W.gemv(Q, D, dbg=dbg)), y)
        assert np.array_equal(host(dbg), orc.q8_acc(rows, R, C, host(Q)))


def test_refill_load_count(tmp_path):
    """k_q8_gemm waits for its DMAs with the 24 loads of a weight refill still in flight: the compiled kernels hold exactly
    the initial and one refill's loads (16 of codes, 8 of scales each), so that count is the one issued"""
    from kindi_amd import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("hipcc is not installed")
    out = str(tmp_path / "q.s")
    r = subprocess.run([build.HIPCC] + build.FLAGS + ["-S", "--cuda-device-only", os.path.join(build.CSRC, "kt_q8gemm.hip"),
                                                     "-o", out], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    kernels = re.findall(r"^(_Z9k_q8_gemm\w*):(.*?)^\s*\.section", open(out).read(), re.S | re.M)
    assert len(kernels) == 4
    for name, body in kernels:
        if "Lb0EEv" not in name:                                          # the debug kernels wait for everything
            continue
        ops = [l.split(";")[0].split() for l in body.split("\n")]
        x4 = [o for o in ops if o and o[0] == "buffer_load_dwordx4" and "lds" not in o]
        u16 = [o for o in ops if o and o[0].startswith("buffer_load_") and ("ushort" in o[0] or "d16" in o[0])]
        assert (len(x4), len(u16)) == (32, 16), (name, len(x4), len(u16))
        assert any(o[:2] == ["s_waitcnt", "vmcnt(24)"] for o in ops if o)
