"""The matrix-core FFN where its tiles and chunks end: rows of 34 and 10 blocks (the last
chunk of a row holds 2), every number of token tiles, and ternary codes of all four bit
patterns (a weight of +2 where a record holds code 3, which the reference's c - 1 gives)."""
import numpy as np
import pytest

import zzref as Z
import zunzuncito_amd as zz
from test_gpu_int_dots import check_dots
from test_gpu_parity import check_layer, gpu_layer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return zz.init()


@pytest.mark.parametrize("kind,fmts", [("gemma", (1, 1, 1)), ("lfm", (2, 2, 2)), ("lfm", (1, 2, 1)),
                                       ("maple", (3, 3, 3))])
def test_short_chunks_and_tiles(dev, kind, fmts):
    """Exact int32 dots, and layer outputs within the float tier (check_layer's 1e-3)."""
    print("case", kind, fmts, flush=True)
    L = Z.make_layer(kind, seed=29, E=4, K=2, D=1088, MI=320, **({} if kind == "maple" else {"fmts": fmts}))
    if kind == "maple":                          # every code byte, 3s among the codes
        rng = np.random.default_rng(4)
        g, u, d = L.tensor_sizes()
        for e in range(L.E):
            for off, O, I in ((0, L.MI, L.D), (g, L.MI, L.D), (g + u, L.D, L.MI)):
                o = e * L.esz + off + 4 * O
                L.experts[o:o + O * I // 4] = rng.integers(0, 256, O * I // 4, dtype=np.uint8)
    m = gpu_layer(L)
    try:
        for S in (6, 20, 50, 80, 130):           # ~3, 10, 25, 40 and 65 tokens an expert
            print("  S", S, flush=True)
            x = Z.make_input(L, S, 31)
            check_layer(m, L, x, Z.oracle_moe(L, x))
            if S <= 80:
                check_dots(L, m, x, f"{kind} {fmts} S={S}")
    finally:
        m.close()


def test_tq2_large_sums(dev):
    """Ternary dots of up to 3e38: the sums are of the dots themselves, so what is finite in
    the reference (whose clamp then makes it an ordinary hidden value) stays finite."""
    L = Z.make_layer("maple", seed=29, E=4, K=2, D=1088, MI=320)
    m = gpu_layer(L)
    try:
        for S in (3, 6, 20, 50, 130):
            print("case large sums", S, flush=True)
            x = Z.make_input(L, S, 31) * np.float32(5e35)
            check_layer(m, L, x, Z.oracle_moe(L, x))
    finally:
        m.close()
