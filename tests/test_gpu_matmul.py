"""gpu_matmul where its splits end: rows of one block and one past a workgroup's 2048
weights, row counts off the workgroup's four, every number of tokens a workgroup takes and
the calls split over several, tensors that start at an odd byte of their mapping, and
infinite block scales."""
import os
import subprocess
import sys

import numpy as np
import pytest

import zzref as Z
import zunzuncito_amd as zz

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return zz.init()


def _weights(rng, fmt, O, I):
    if fmt == Z.FMT_TQ2:
        return Z.make_expert_tq2(rng, O, I)
    if fmt == Z.FMT_Q4A:
        return Z.q4a_rows(rng, O, I)
    return Z.quant_rows(fmt, (rng.standard_normal((O, I)) * 0.02).astype(np.float32))


@pytest.mark.parametrize("fmt", [Z.FMT_Q40, Z.FMT_Q80, Z.FMT_TQ2, Z.FMT_Q4A])
def test_edges(dev, fmt):
    """Within 1e-5 of the largest output: 32-bit sums of up to 4160 products whose
    rounding errors are each below 2^-24 of a partial sum."""
    rng = np.random.default_rng(71)
    small = 64 if fmt in (Z.FMT_TQ2, Z.FMT_Q4A) else 32
    for O, I, S in [(1, small, 1), (5, small, 9), (3, 2048 + small, 2), (7, 4160, 3), (66, 1088, 4), (9, 320, 5),
                    (130, 2112, 6), (4, 2048, 7), (33, 704, 8), (6, 192, 17)]:
        print("case", fmt, O, I, S, flush=True)
        W = _weights(rng, fmt, O, I)
        odd = np.zeros(W.size + 1, np.uint8)
        odd[1:] = W
        Wm = zz.gpu_map(odd)[1:]
        x = rng.standard_normal((S, I)).astype(np.float32)
        y = zz.gpu_matmul(fmt, Wm, x, O, I)
        ref = np.zeros((S, O), np.float32)
        Z.oracle().orc_matmul_f32(fmt, Z.ptr(ref), Z.ptr(W), Z.ptr(x), O, I, S)
        assert np.abs(y - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("fmt,bb", [(Z.FMT_Q40, 18), (Z.FMT_Q80, 34), (Z.FMT_Q4A, 36)])
def test_infinite_scales(dev, fmt, bb):
    """An infinite d times a block's whole partial sum: the reference's infinities."""
    rng = np.random.default_rng(73)
    O, I, S = 10, 512, 3
    W = np.array(_weights(rng, fmt, O, I))
    blocks = W.reshape(O, -1, bb)
    for r in range(O):
        blocks[r, r % blocks.shape[1], :2] = np.array([np.inf], np.float16).view(np.uint8)
    x = rng.standard_normal((S, I)).astype(np.float32)
    y = zz.gpu_matmul(fmt, zz.gpu_map(W), x, O, I)
    ref = np.zeros((S, O), np.float32)
    Z.oracle().orc_matmul_f32(fmt, Z.ptr(ref), Z.ptr(W), Z.ptr(x), O, I, S)
    assert not np.isfinite(ref).any() and np.array_equal(y, ref, equal_nan=True)


@pytest.mark.parametrize("fmt", [Z.FMT_Q40, Z.FMT_TQ2])
@pytest.mark.parametrize("O,I,S", [(64, 4096, 64), (40, 4096, 65), (8191, 64, 33), (4099, 2112, 70)])
def test_staged_and_copied_calls(dev, fmt, O, I, S):
    """Up to 2^18 values of x and of y go through the pinned staging (the first shape just
    does), larger ones by copies (x, y, both); in each the weights are rewritten on the host
    and the next call forms the product again. Within 1e-5 of the largest output, as above."""
    print("case", fmt, O, I, S, flush=True)
    rng = np.random.default_rng(77)
    Wm = zz.gpu_map(np.array(_weights(rng, fmt, O, I)))
    for k in range(3):
        x = rng.standard_normal((S, I)).astype(np.float32)
        n0 = zz.lib().zz_gpu_map_refreshes()
        if k == 1:
            Wm[:] = _weights(rng, fmt, O, I)
        y = zz.gpu_matmul(fmt, Wm, x, O, I)
        assert zz.lib().zz_gpu_map_refreshes() - n0 == (k == 1)
        ref = np.zeros((S, O), np.float32)
        Z.oracle().orc_matmul_f32(fmt, Z.ptr(ref), Z.ptr(Wm), Z.ptr(x), O, I, S)
        assert np.abs(y - ref).max() <= 1e-5 * np.abs(ref).max()


_CHILD = """
import numpy as np
import zunzuncito_amd as zz

def maps():
    return {l.split()[0] for l in open("/proc/self/maps") if "/dev/dri/" in l}

def product():
    W = zz.gpu_map(np.full(64 * 2 * 18, 0x44, np.uint8))
    return zz.gpu_matmul(zz.GPU_FMT_Q40, W, np.ones((3, 64), np.float32), 64, 64)

size = lambda m: int(m.split("-")[1], 16) - int(m.split("-")[0], 16)
zz.init()
before = maps()
y = product()
staging = {m for m in maps() - before if size(m) == 2 << 20}
zz.lib().gpu_shutdown()
print("staging", len(staging), "left", len(staging & maps()), flush=True)
for _ in range(2):
    zz.init()
    assert np.array_equal(product(), y)
    zz.lib().gpu_shutdown()
print("done")
"""


def test_shutdown_gives_the_staging_back():
    """The 2 MiB pinned staging leaves the process with gpu_shutdown, and calls after another
    gpu_init have theirs again. In a process of its own: a shutdown takes every layer."""
    r = subprocess.run([sys.executable, "-c", _CHILD], cwd=Z.ROOT, capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=Z.ROOT))
    assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr
    assert "staging 1 left 0" in r.stdout, r.stdout
