"""The prefill product's kernels at the edges of their dispatch (kt_tern_gemm): a tile a block with its groups dealt over
4 or (one tile a CU, 4096 columns or more) 8 waves (up to 2 tiles of 32 x 32 a CU), one tile a wave (up to 12), two tiles a wave. Every one applies the reference
expression group after group, so the int32 group values and the fp32 outputs are the oracle's, bit for bit."""
import numpy as np
import pytest
import torch

import oracle as orc
from kt_cases import say, tern_case, dev, host, rng

pytestmark = pytest.mark.gpu


def _tiles(R, M):
    return -(-R // 32) * -(-M // 32)


def _route(R, M):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if _tiles(R, M) <= 2 * cus:
        return "split"
    return "one" if -(-R // 128) * -(-M // 32) <= 3 * cus else "two"


# group counts around the 4 groups of a round, the 3 stages and the 8 units of a kt2 step; ragged rows and tokens
@pytest.mark.parametrize("R,C,M,route", [
    (8, 128, 1, "split"), (40, 256, 17, "split"), (100, 384, 33, "split"), (31, 512, 64, "split"), (65, 640, 31, "split"),
    (257, 1152, 45, "split"), (96, 1664, 96, "split"), (5120, 1408, 61, "split"),
    (40, 4096, 33, "split"), (31, 4224, 64, "split"), (257, 5248, 17, "split"), (1024, 6016, 70, "split"),
    (8200, 128, 70, "one"), (8200, 256, 95, "one"), (8193, 384, 65, "one"), (8260, 512, 100, "one"), (8300, 1152, 97, "one"),
    (8200, 128, 400, "two"), (8197, 256, 385, "two"), (8200, 384, 449, "two"), (8300, 1280, 390, "two")])
@pytest.mark.parametrize("per_row", [False, True])
def test_gemm_routes(R, C, M, route, per_row):
    from kindi_amd import linear
    say("gemm route", R, C, M, route, per_row)
    assert _route(R, M) == route
    dig, bc, dpm = tern_case(R, C, R + C + M)
    L = linear.Linear({"w": linear.TernaryMatrix(bc, dpm, R, C)})
    X = rng(M + 5).normal(0, 1, (M, C)).astype(np.float32)
    act = linear.quantize(dev(X), per_row=per_row)
    Q, XS, XA = orc.quant_q8(X, per_row=per_row)
    acc = orc.tern_acc(bc, R, C, Q)
    want = (orc.tern_out_rs if per_row else orc.tern_out)(acc, XS, dpm, R, C)
    dbg = torch.empty((M, R, C // 128), dtype=torch.int32, device="cuda")
    Y = torch.empty((M, R), dtype=torch.float32, device="cuda")
    Y16 = torch.empty((M, R), dtype=torch.float16, device="cuda")
    L.gemm("w", act, Y=Y, Y16=Y16, dbg=dbg)
    assert np.array_equal(host(dbg), acc), "int32 group values"
    assert np.array_equal(host(Y), want), "debug instantiation"
    assert np.array_equal(host(Y16), want.astype(np.float16))
    assert np.array_equal(host(L.gemm("w", act)), want)
    wide = torch.full((M, R + 3), -7.0, device="cuda")                    # rows of a wider buffer: the pad untouched
    L.gemm("w", act, Y=wide[:, :R])
    assert np.array_equal(host(wide[:, :R]), want) and bool((wide[:, R:] == -7.0).all())


# the 16-token decode product with its activations straight into the operand and through LDS: both sides of 5 rows (3 above 2
# tiles a CU of 3 slices or more) and of slices x rows 16 at a tile a CU; whole slices, slices over 4 waves, more slices than 4
# groups, over 2 waves; a second pass of one token; the two-row form
@pytest.mark.parametrize("R,C,Ms", [(40, 384, (3, 5, 6, 15, 16, 17)), (100, 2048, (4, 16, 17)), (8200, 2048, (5, 6)), (1000, 4096, (8, 9)), (520, 6144, (5, 6)),
                                    (16648, 5120, (3, 4)), (136, 9216, (5, 6, 9, 17)), (100, 12288, (3, 5, 6, 8, 9, 16))])
@pytest.mark.parametrize("hp", [False, True])
def test_decode_rows_either_way(R, C, Ms, hp):
    from kindi_amd import linear
    dig, bc, dpm = tern_case(R, C, R + C)
    L = linear.Linear({"w": linear.TernaryMatrix(bc, dpm, R, C)})
    X = dev(rng(C).normal(0, 1, (max(Ms), C)).astype(np.float32))
    one = torch.empty((max(Ms), R), device="cuda")
    for i in range(max(Ms)):                                              # a token at a time: the same bits in any company
        L.gemv_q(["w"], linear.quantize(X[i:i + 1], hp=hp), [one[i:i + 1]])
    for M in Ms:
        say("decode rows", R, C, M, hp)
        act = linear.quantize(X[:M], hp=hp)
        Y = torch.empty((M, R), device="cuda")
        L.gemv_q(["w"], act, [Y])
        assert torch.equal(Y, one[:M]), M
        rows = act.XQ.shape[0]
        if rows * R * C <= 1 << 25:
            dbg = torch.empty((rows, R, C // 128), dtype=torch.int32, device="cuda")
            Y2 = torch.empty((M, R), device="cuda")
            L.gemv_q(["w"], act, [Y2], dbg=dbg)
            assert torch.equal(Y2, one[:M]) and np.array_equal(host(dbg), orc.tern_acc(bc, R, C, host(act.XQ))), M


@pytest.mark.parametrize("R,M,route", [(256, 64, "split"), (8200, 70, "one"), (8200, 400, "two")])
def test_gemm_scale_extremes(R, M, route):
    """token scales whose product with a row scale is subnormal, overflows, or is not a number: the element scale is
    XS d rounded once on every route (the two-tile route makes it on the matrix cores)"""
    from kindi_amd import linear
    say("gemm scales", R, M, route)
    assert _route(R, M) == route
    C = 384
    dig, bc, dpm = tern_case(R, C, 77)
    L = linear.Linear({"w": linear.TernaryMatrix(bc, dpm, R, C)})
    act = linear.quantize(dev(rng(3).normal(0, 1, (M, C)).astype(np.float32)))
    sc = np.array([1e-38, 3e-40, 1.4e-45, 0.0, 2e38, np.inf, np.nan, 1.0, -0.5, 1.1754944e-38], np.float32)
    act.XS.copy_(dev(np.tile(sc, (M * (C // 128) + 9) // 10)[:M * (C // 128)].reshape(M, C // 128)))
    with np.errstate(all="ignore"):
        want = orc.tern_out(orc.tern_acc(bc, R, C, host(act.XQ)), host(act.XS), dpm, R, C)
    got = host(L.gemm("w", act))
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), (int((~same).sum()), got[~same][:4], want[~same][:4])
