"""Several-vector GEMV (gs_gemv with 2..8 quantized vectors) at the edges of its plans: rows around one
tile of 16 and one tile per CU, K of one super-block, of odd counts, over one chunk and of several
chunks; rows off 16- and 4-byte boundaries; padded strides; accumulation. Each vector quantizes by itself
and its products are exact integer dots, so against the oracle only the f32 scaling and the order of the
sums differ: relative errors of 2^-24 at random signs over K / 32 terms (rel L2 about 1e-7 here), bounded
at 1e-5 as for the one-vector kernels."""
import sys

import numpy as np
import pytest

import glmssd as G
from glmssd import GgmlType as T
from glmssd import synth
import oracle as O

pytestmark = pytest.mark.gpu
REL = 1e-5
HALVES = {T.Q8_0: ([0], 3e-4), T.Q4_K: ([0, 2], 3e-4), T.Q5_K: ([0, 2], 2e-4), T.Q6_K: ([208], 2e-5)}
TYPES = list(HALVES)


def run(ty, K, rows, B, accumulate=False, x_pad=0, y_pad=0, row_pad=0, w_off=0):
    rng = np.random.default_rng([ty, K, rows, B])
    rb = G.row_bytes(ty, K)
    raw = synth.random_blocks(rng, ty, rows * K, HALVES[ty][1], HALVES[ty][0])
    X = rng.standard_normal((B, K + x_pad)).astype(np.float32)
    want = O.gemv(ty, raw, rb, K, rows, X, B, K + x_pad, nthreads=8)
    ys = rows + y_pad
    y0 = (rng.standard_normal((B, ys)) * np.std(want)).astype(np.float32)
    padded = np.zeros((rows, rb + row_pad), np.uint8)
    padded[:, :rb] = raw.reshape(rows, rb)
    dw = G.DeviceBuffer(padded.nbytes + w_off)
    dw.upload(padded.reshape(-1), None, w_off)
    dx, dy = G.DeviceBuffer.from_array(X), G.DeviceBuffer.from_array(y0)
    print(f"gemv {G.TYPE_NAMES[ty]} K={K} rows={rows} B={B} pad={row_pad}", flush=True)
    sys.stdout.flush()
    G.ops.gemv(ty, dw.ptr(w_off), rb + row_pad, K, rows, dx, K + x_pad, dy, ys, B, accumulate)
    got = dy.download(np.float32, B * ys).reshape(B, ys)
    G.ops.wait_status()
    assert np.array_equal(got[:, rows:], y0[:, rows:])   # nothing past the rows
    g = got[:, :rows].astype(np.float64) - (y0[:, :rows] if accumulate else 0.0)
    # per vector: a wrong vector does not hide among the others
    return max(float(np.linalg.norm(g[b] - want[b]) / np.linalg.norm(want[b])) for b in range(B))


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("K,rows,vectors", [
    (256, 1, (5, 8)), (2048, 17, (5, 7)), (1280, 100, (5, 6)), (4096, 4096, (3, 4, 5, 8)), (4096, 4113, (4, 7)),
    (512, 16400, (5, 8)), (2304, 14600, (3, 6)), (4352, 33, (3, 5, 8)), (6144, 2750, (2, 3, 8)), (12288, 47, (3, 4, 8)),
    (12288, 2740, (2, 6, 8)), (16640, 515, (3, 8))])
def test_edges(ty, K, rows, vectors):
    for B in vectors:
        assert run(ty, K, rows, B) <= REL


@pytest.mark.parametrize("ty", TYPES)
def test_strides_accumulate_offsets(ty):
    assert run(ty, 1024, 333, 6, True, x_pad=4, y_pad=3) <= REL
    assert run(ty, 6144, 333, 3, True, x_pad=8, y_pad=1, row_pad=16) <= REL
    assert run(ty, 8192, 300, 8, True, row_pad=4, w_off=4) <= REL
    assert run(ty, 2048, 300, 5, row_pad=2, w_off=2) <= REL      # off dwords: Q6_K here, the others streamed
    assert run(ty, 6144, 100, 4, x_pad=1) <= REL                 # vectors off 16 bytes: streamed
    assert run(ty, 512, 5000, 8, row_pad=6, w_off=2) <= REL
