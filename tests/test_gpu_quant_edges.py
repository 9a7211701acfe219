"""The 2-D quantize's edge loads (rows that are not 16-byte aligned, chunks
that run past a row's end, rows shorter than a chunk, tiles partly or wholly
of padding) and the one-launch form of the just-in-time quantize for small
inputs, against the oracle: codes, transposed codes, their zero padding,
absmax and scale bit for bit, column sums within binary32 summation error."""
import numpy as np
import pytest
import torch

import deepfuse_amd as df
from deepfuse_amd import Fmt
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
# one value, rows shorter than a 16-byte chunk, one value past / short of a
# chunk and of a tile, 128 KB of input on, below and above (the one-launch form's limit in 2 and 4 byte types),
# tiles on and past the small kernel's limit
SHAPES = [(1, 1), (3, 3), (5, 7), (129, 5), (2, 9), (127, 129), (128, 127), (130, 136), (257, 131), (8, 1600),
          (16, 1024), (16, 1025), (31, 264), (64, 128), (8, 1023), (300, 77),
          (64, 1024), (64, 1025), (32, 1024), (33, 1024), (2048, 2048), (2049, 2056),
          (40000, 1)]


def tensor(rows, cols, dt, dev, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * 3
    if rows * cols > 16:  # specials, one in the last row and column
        flat = x.view(-1)
        at = torch.randperm(rows * cols - 1, generator=g)[:5]
        flat[at] = torch.tensor([float("nan"), float("inf"), float("-inf"), 0.0, -0.0])
        flat[-1] = 11.5  # the absmax, in the last chunk
    return x.to(dt).to(dev)


def host(x):
    return x.float().cpu().numpy()  # exact for the 2-byte types


@pytest.mark.parametrize("rows,cols", SHAPES)
@pytest.mark.parametrize("dt", [F32, BF16, F16])
@pytest.mark.parametrize("fmt", [Fmt.E4M3, Fmt.E5M2])
def test_edges(dev, rows, cols, dt, fmt):
    x = tensor(rows, cols, dt, dev, rows * 1009 + cols)
    h = host(x)
    am, sc, q, qt, cs = df.quantize_2d_jit(x, fmt, want_qt=True, colsum=True)
    s = orc.scale(orc.absmax(h), int(fmt))
    assert am.item() == orc.absmax(h) and sc.item() == np.float32(s)
    codes = orc.quantize(h, s, int(fmt))

    def check(q, qt):
        qh, th = q.cpu().numpy(), qt.cpu().numpy()
        assert np.array_equal(qh[:, :cols], codes) and not qh[:, cols:].any()
        assert np.array_equal(th[:, :rows], codes.T) and not th[:, rows:].any()

    check(q, qt)
    finite = np.isfinite(h).all(axis=0)
    ref = h.astype(np.float64).sum(axis=0)
    # binary32 sums of `rows` values: at most rows * 2^-24 of the sum of magnitudes
    bound = rows * 2.0 ** -24 * np.abs(h.astype(np.float64)).sum(axis=0) + 1e-30
    assert (np.abs(cs.cpu().numpy()[finite] - ref[finite]) <= bound[finite]).all()
    # the same without column sums, the plain pass at that scale, and the
    # rows of a wider matrix (a stride that is not a multiple of 16 bytes)
    _, sc2, q2, qt2 = df.quantize_2d_jit(x, fmt, want_qt=True)
    assert sc2.item() == sc.item()
    check(q2, qt2)
    check(*df.quantize_2d(x, sc, fmt, want_qt=True))
    wide = torch.full((rows, cols + 3), float("nan"), dtype=dt, device=dev)
    wide[:, :cols].copy_(x)
    check(*df.quantize_2d(wide[:, :cols], sc, fmt, want_qt=True))


# tile rows (of 128) on and past the counts from which the column sums of a
# matrix of one or two strips of 128 columns are added up by a launch of their own
@pytest.mark.parametrize("rows,cols,dt", [(49152, 3, BF16), (49153, 3, F16), (49153, 128, F32), (262145, 9, BF16),
                                          (131072, 130, BF16), (131073, 130, BF16), (131073, 129, F32)])
def test_tall_column_sums(dev, rows, cols, dt):
    """Either way the sums are those of df_quantize_2d_colsum, bit for bit,
    and absmax, scale and codes those of the calls without sums."""
    x = tensor(rows, cols, dt, dev, rows + cols)
    x = torch.where(torch.isfinite(x), x, torch.zeros_like(x))
    am, sc, q, qt, cs = df.quantize_2d_jit(x, Fmt.E5M2, want_qt=True, colsum=True)
    am1, sc1 = df.absmax_scale(x, Fmt.E5M2)
    q1, qt1, cs1 = df.quantize_2d(x, sc1, Fmt.E5M2, want_qt=True, colsum=True)
    assert am.item() == am1.item() == x.float().abs().max().item() and sc.item() == sc1.item()
    assert torch.equal(q, q1) and torch.equal(qt, qt1)
    assert torch.equal(cs.view(torch.int32), cs1.view(torch.int32))
    ref = x.double().sum(0)
    bound = rows * 2.0 ** -24 * x.double().abs().sum(0)
    assert bool(((cs.double() - ref).abs() <= bound).all())


# rows of whole 16-byte chunks below, at and past what a wave's registers hold,
# row counts that leave waves with fewer rows than their share, rows too wide
# for the registers in whole and part rounds of sixteen values a lane
@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 512), (130, 1600), (67, 2048), (9, 1024), (8193, 64), (16387, 72),
                                       (6, 2056), (3, 6400), (4, 3001)])
@pytest.mark.parametrize("dt", [F32, BF16, F16])
@pytest.mark.parametrize("affine", [True, False])
def test_layernorm_codes(dev, rows, cols, dt, affine):
    """The fused LayerNorm's codes and scale are those of the quantize of its
    own y, and y is within rounding of binary64 (a NaN row and a constant row
    among them)."""
    g = torch.Generator().manual_seed(rows + 31 * cols)
    x = torch.randn(rows, cols, generator=g) * 2 + 0.25
    if rows > 4:
        x[1, cols // 2] = float("nan")
        x[2] = 0.5
    x = x.to(dt).to(dev)
    gamma = (1 + 0.1 * torch.randn(cols, generator=g)).to(dt).to(dev) if affine else None
    beta = (0.1 * torch.randn(cols, generator=g)).to(dt).to(dev) if affine else None
    y0 = df.layernorm(x, gamma, beta)
    y, q, qt, sc = df.layernorm(x, gamma, beta, fmt=Fmt.E4M3, want_y=True, want_qt=True)
    bits = torch.int32 if dt == F32 else torch.int16
    assert torch.equal(y.view(bits), y0.view(bits))
    _, sy, q2, qt2 = df.quantize_2d_jit(y.contiguous(), Fmt.E4M3, want_qt=True)
    assert sc.item() == sy.item() and torch.equal(q, q2) and torch.equal(qt, qt2)
    xd = x.double()
    ref = (xd - xd.mean(1, keepdim=True)) / (xd.var(1, unbiased=False, keepdim=True) + 1e-5).sqrt()
    if affine:
        ref = ref * gamma.double() + beta.double()
    ok = torch.isfinite(ref)
    # half a unit in the last place of a p-bit significand is at most 2^-p of the value (p = 24, 8, 11); behind it
    # binary32 sums of `cols` values of magnitude below 8
    ulp = {F32: 2.0 ** -24, BF16: 2.0 ** -8, F16: 2.0 ** -11}[dt]
    err = (y.double() - ref).abs()[ok]
    bound = ulp * ref.abs()[ok] + cols * 2.0 ** -24 * 8 + 2.0 ** -25
    assert bool((err <= bound).all()) and bool(torch.isnan(y[~ok]).all())


@pytest.mark.parametrize("rows,cols", [(130, 1600), (33, 771), (9, 2056), (20, 3001)])
@pytest.mark.parametrize("dt", [F32, BF16, F16])
def test_layernorm_codes_overflow(dev, rows, cols, dt):
    """Values that overflow the element type when y is rounded to it: infinite
    in y, left out of the absmax, saturated as codes.  Columns with a gamma
    that takes most values past the range, and columns whose beta is the
    largest finite value and whose gamma is about its unit in the last place:
    y is rounded to that value on one side of it, to infinity on the other."""
    g = torch.Generator().manual_seed(rows + 7 * cols)
    x = (torch.randn(rows, cols, generator=g) * 2 + 0.25).to(dt).to(dev)
    gamma, beta = torch.ones(cols), torch.zeros(cols)
    top = torch.finfo(dt).max
    gamma[::97] = top / 1.5
    gamma[5::97], beta[5::97] = {F32: 2.0e31, BF16: 1.4e36, F16: 32.0}[dt], top
    gamma, beta = gamma.to(dt).to(dev), beta.to(dt).to(dev)
    y0 = df.layernorm(x, gamma, beta)
    h = host(y0)
    assert np.isinf(h[:, ::97]).any() and np.isinf(h[:, 5::97]).any() and (h[:, 5::97] == top).any()
    s = orc.scale(orc.absmax(h), int(Fmt.E4M3))
    y, q, qt, sc = df.layernorm(x, gamma, beta, fmt=Fmt.E4M3, want_y=True, want_qt=True)
    bits = torch.int32 if dt == F32 else torch.int16
    assert torch.equal(y.view(bits), y0.view(bits)) and sc.item() == np.float32(s)
    codes = orc.quantize(h, s, int(Fmt.E4M3))
    assert np.array_equal(q.cpu().numpy()[:, :cols], codes)
    assert np.array_equal(qt.cpu().numpy()[:, :rows], codes.T)


# one and three partials past the count (8192) up to which every tile block of
# the fused LayerNorm folds them all: rows of odd width have a partial per 4
# rows, rows of whole 16-byte chunks one per 32
@pytest.mark.parametrize("rows,cols,per", [(32772, 33, 4), (32777, 5, 4), (262176, 64, 32)])
@pytest.mark.parametrize("at", ["first", "middle", "last"])
def test_layernorm_many_rows(dev, rows, cols, per, at):
    """A long list of absmax partials is folded before the tile pass, whose
    every block would otherwise read all of it: the folded values lie behind
    the list in the workspace, and codes, scale and absmax are those of the
    quantize of y wherever the largest |y| stands."""
    g = torch.Generator().manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g).clamp_(-2, 2)
    r = {"first": 0, "middle": rows // 2, "last": rows - 1}[at]
    x[r] = 0.0
    x[r, cols // 2] = 100.0  # a one-hot row has the largest normalized value of all
    x = x.to(BF16).to(dev)
    y = df.layernorm(x)
    am, sy, q2, qt2 = df.quantize_2d_jit(y, Fmt.E4M3, want_qt=True)
    q, qt = torch.empty_like(q2), torch.empty_like(qt2)
    sc, ab = torch.empty(1, device=dev), torch.empty(1, device=dev)
    nbytes = df.lib().df_layernorm_workspace_bytes(rows, cols, q.shape[1], qt.shape[1])
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev)
    df.call("df_layernorm_quantize", int(df.DType.BFLOAT16), x.data_ptr(), rows, cols, cols, None, None, 1e-5, None, 0,
            int(Fmt.E4M3), sc.data_ptr(), ab.data_ptr(), q.data_ptr(), q.shape[1], qt.data_ptr(), qt.shape[1],
            ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
    assert sc.item() == sy.item() and ab.item() == am.item() == y[r].float().abs().max().item()
    assert torch.equal(q, q2) and torch.equal(qt, qt2)
    parts = ws[(rows * 8 + 15) // 16 * 16:].view(torch.float32)
    n = (rows + per - 1) // per
    few = parts[n:n + 4]
    assert n > 8192 and bool(torch.isfinite(parts[:n + 4]).all())
    assert parts[:n].max().item() == few.max().item() == am.item()
