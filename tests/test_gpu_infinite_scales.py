"""Blocks whose fp16 scale is infinite (the format holds them and the quantisers write them
where a weight overflows) through every form of the expert FFN: decode, the 4x4x4 items of up
to 8 tokens and the tiles of 16 on both sides of it, with one expert so that an item holds the
batch. The reference adds d * dot per group of four weights (q40.h:162-207): a row whose
groups all have one sign ends at that infinity, any other at NaN."""
import numpy as np
import pytest

import zzref as Z
import zunzuncito_amd as zz
from test_gpu_parity import gpu_layer

pytestmark = pytest.mark.gpu

BB = {Z.FMT_Q40: 18, Z.FMT_Q80: 34}
SIZES = (1, 4, 5, 8, 9, 17, 40, 64, 70)
INF = np.array([np.inf], np.float16).view(np.uint8)


@pytest.fixture(scope="module")
def dev():
    return zz.init()


def _blocks(L, t):
    """Tensor t (gate, up, down) of expert 0 as a writable [rows, blocks, bytes] view."""
    sizes = L.tensor_sizes()
    off, (O, I), bb = sum(sizes[:t]), ((L.MI, L.D), (L.MI, L.D), (L.D, L.MI))[t], BB[L.fmts[t]]
    return L.experts[off:off + O * (I // 32) * bb].reshape(O, I // 32, bb)


def _layer(fmt):
    """up = gate, so that the hidden g^2 sigmoid(g) is positive; 34 blocks of input, whose
    last chunk is short (and holds positive values, below), and 10 of hidden."""
    L = Z.make_layer("lfm", seed=61, E=1, K=1, D=1088, MI=320, fmts=(fmt, fmt, fmt))
    _blocks(L, 1)[:] = _blocks(L, 0)
    return L


def _make_infinite(fmt, blk, neg):
    """An infinite scale and one code throughout, of either sign."""
    blk[:2] = INF
    if fmt == Z.FMT_Q40:
        blk[2:] = 0x55 if neg else 0xbb                      # codes 5 - 8 and 11 - 8
    else:
        blk[2:] = np.int8(-9 if neg else 9).view(np.uint8)


def _run(L):
    m = gpu_layer(L)
    try:
        for S in SIZES:
            print("case", L.fmts, "S", S, flush=True)
            x = Z.make_input(L, S, 70 + S)
            x[:, -64:] = np.abs(x[:, -64:])
            out, _, _ = m.forward(x)
            with np.errstate(all="ignore"):
                want = Z.oracle_moe(L, x).out
            yield S, out.reshape(S, L.D), want.reshape(S, L.D)
    finally:
        m.close()


@pytest.mark.parametrize("fmt", [Z.FMT_Q40, Z.FMT_Q80])
def test_down_rows(dev, fmt):
    """Infinite blocks in some down rows: the oracle's infinities with their signs, finite
    rows within the fp32 tier (1e-3 relative L2)."""
    L = _layer(fmt)
    b = _blocks(L, 2)
    rows = np.arange(3, L.D, 37)
    for k, r in enumerate(rows):
        _make_infinite(fmt, b[r, (0, 4, 9)[k % 3]], neg=k % 2 == 0)
    for S, out, want in _run(L):
        fin = np.ones(L.D, bool)
        fin[rows] = False
        inf = np.isinf(want)
        assert inf[:, rows].mean() > 0.8, "the oracle's rows are meant to be infinite"
        assert not np.isfinite(out[:, rows]).any()
        assert np.array_equal(out[inf], want[inf])
        assert Z.rel_l2(out[:, fin], want[:, fin]) < 1e-3


@pytest.mark.parametrize("fmt", [Z.FMT_Q40, Z.FMT_Q80])
@pytest.mark.parametrize("t", [0, 1])
def test_gate_and_up_rows(dev, fmt, t):
    """An infinite block in a gate or up row: an infinite hidden, whose q8_0 block has an
    infinite scale, so that no output of the layer is finite."""
    L = _layer(fmt)
    _make_infinite(fmt, _blocks(L, t)[37, (33, 32)[t]], neg=False)
    for S, out, want in _run(L):
        assert not np.isfinite(want).any()
        assert not np.isfinite(out).any(), (S, int(np.isfinite(out).sum()))
