"""The activation quantizer (kt_quant_q8) where its dispatch changes: per row, the groups a wave keeps in registers (4, 8,
16, 32, or read twice); per group and two-row, the chunks a row is cut into by the number of rows."""
import numpy as np
import pytest
import torch

from kt_cases import say, dev, host, orc, rng

pytestmark = pytest.mark.gpu


def _same(X, mode, pad):
    from kindi_amd import linear
    M, C = X.shape
    wide = torch.full((M, C + pad), float("nan"), device="cuda")
    wide[:, :C] = dev(X)
    act = linear.quantize(wide[:, :C], per_row=mode == 1, hp=mode == 2)
    for got, want, what in zip((act.XQ, act.XS, act.XA), orc.quant_q8(X, mode), ("rows", "scales", "sums")):
        assert np.array_equal(host(got), want), what


# both sides of 32, 64, 128 and 256 groups, fewer groups than the 8 waves, and a last wave without a group
@pytest.mark.parametrize("NG", [1, 7, 8, 9, 32, 33, 57, 64, 65, 128, 129, 256, 257])
def test_per_row_widths(NG):
    say("quant row", NG)
    X = rng(NG).normal(0, 1, (5, NG * 128)).astype(np.float32)
    X[1] = 0.0
    X[2, :128] *= 1e4                                       # the row's maximum in its first group, and in its last
    X[3, -1] = -3e4
    X[4] *= 1e-30
    _same(X, 1, 2)


# a group a wave, chunks that do not divide the row (NG 9, 45), and one block a row from 4096 rows
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("NG,M", [(1, 1), (3, 3), (9, 1), (45, 100), (45, 1000), (9, 1500), (9, 4095), (9, 4096), (5, 5000)])
def test_group_chunks(NG, M, mode):
    say("quant groups", NG, M, mode)
    X = rng(NG + M).normal(0, 1, (M, NG * 128)).astype(np.float32)
    X[0, :128] = 0.0
    X[-1] *= 1e-30
    _same(X, mode, 6)


# rows of fewer groups than a block has waves otherwise (blocks of 1, 2 and 4 waves per row, of NG per group), and the two-row form
# around the line at which its sums go over the LDS crossbar (16 groups, 4096 rows)
@pytest.mark.parametrize("NG,M,mode", [(1, 3, 1), (2, 5, 1), (3, 5, 1), (4, 6, 1), (5, 5, 1), (2, 4100, 1), (1, 4100, 0), (2, 9, 0), (3, 4096, 2),
                                       (15, 4096, 2), (16, 4095, 2), (16, 4096, 2), (17, 4099, 2)])
def test_narrow_rows_and_two_row_line(NG, M, mode):
    say("quant narrow", NG, M, mode)
    X = rng(NG * M).normal(0, 1, (M, NG * 128)).astype(np.float32)
    X[0, -128:] = 0.0
    X[1, :128] *= 1e4
    X[2] *= 1e-30
    _same(X, mode, 2)
