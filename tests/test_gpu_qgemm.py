"""The quantized GEMM of row-tile workgroups (qgemm.hip) at the sizes where its tiling can go wrong:
one and several row blocks with a ragged last one, token blocks of 1 .. 6 sixteens and of 128 with
ragged ends, one to several raw chunks of a row, K slices, f32 and f16-slab activations, strides,
batches, accumulate, rows off dword boundaries. Reference: the f64 product of the oracle's
dequantized weights and the activations, both rounded to f16 (the GEMM's operands); the bound is
f32 accumulation's: K products of relative error 2^-24 summed in blocks, at most 1e-5 as for every
GEMM path here."""
import sys

import numpy as np
import pytest

import glmssd as G
from glmssd import GgmlType as T
from glmssd import synth
import oracle as O

pytestmark = pytest.mark.gpu
REL = 1e-5
HALVES = {T.Q8_0: ([0], 3e-4), T.Q4_K: ([0, 2], 3e-4), T.Q5_K: ([0, 2], 2e-4), T.Q6_K: ([208], 2e-5), T.IQ2_XXS: ([0], 5e-4),
          T.IQ3_XXS: ([0], 2e-4)}
TYPES = list(HALVES)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def run(ty, K, rows, N, work_bytes=None, accumulate=False, x_pad=0, y_pad=0, row_pad=0, w_off=0, nb=1, seed=0):
    """rel-L2 of gs_gemm_ex against the f64 product; work_bytes None: gs_gemm."""
    rng = np.random.default_rng([seed, ty, K, rows, N])
    rb = G.row_bytes(ty, K)
    raw = synth.random_blocks(rng, ty, nb * rows * K, HALVES[ty][1], HALVES[ty][0])
    X = rng.standard_normal((nb, N, K + x_pad)).astype(np.float32)
    w16 = O.dequantize(ty, raw, nb * rows * K).reshape(nb, rows, K).astype(np.float16).astype(np.float64)
    x16 = X[:, :, :K].astype(np.float16).astype(np.float64)
    want = np.stack([x16[z] @ w16[z].T for z in range(nb)])
    ys = rows + y_pad
    y0 = (rng.standard_normal((nb, N, ys)) * np.std(want)).astype(np.float32)
    padded = np.zeros((nb * rows, rb + row_pad), np.uint8)
    padded[:, :rb] = raw.reshape(nb * rows, rb)
    dw = G.DeviceBuffer(padded.nbytes + w_off)
    dw.upload(padded.reshape(-1), None, w_off)
    dx, dy = G.DeviceBuffer.from_array(X), G.DeviceBuffer.from_array(y0)
    rs = rb + row_pad
    say(f"qgemm {G.TYPE_NAMES[ty]} K={K} rows={rows} N={N} work={work_bytes} batches={nb}")
    if work_bytes is None:
        G.ops.gemm(ty, dw.ptr(w_off), rs, K, rows, dx, K + x_pad, dy, ys, N, accumulate, nb, rows * rs, N * (K + x_pad), N * ys)
    else:
        wk = G.DeviceBuffer(work_bytes)
        G.ops.gemm_ex(ty, dw.ptr(w_off), rs, K, rows, dx, K + x_pad, dy, ys, N, accumulate, nb, rows * rs, N * (K + x_pad), N * ys,
                      wk, work_bytes)
    got = dy.download(np.float32, nb * N * ys).reshape(nb, N, ys)
    G.ops.wait_status()
    assert np.array_equal(got[:, :, rows:], y0[:, :, rows:])   # nothing past the rows
    g = got[:, :, :rows].astype(np.float64) - (y0[:, :, :rows] if accumulate else 0.0)
    return float(np.linalg.norm(g - want) / np.linalg.norm(want))


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("K,rows,N", [
    (256, 1, 9), (512, 17, 16), (2304, 47, 17),        # one block, one super-block, nine of them
    (1280, 2000, 33), (768, 4097, 50), (512, 12301, 77), (256, 12288, 96), (512, 9000, 100), (512, 3000, 192)])
def test_no_workspace(ty, K, rows, N):
    assert run(ty, K, rows, N) <= REL


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("K,rows,N", [(256, 12289, 65), (1536, 4100, 96), (4096, 300, 90), (2048, 2500, 129), (1024, 12300, 257),
                                      (512, 130, 512), (6144, 1030, 200)])
def test_workspace(ty, K, rows, N):
    assert run(ty, K, rows, N, 256 << 20) <= REL


@pytest.mark.parametrize("ty", [T.Q4_K, T.Q6_K, T.Q8_0])
def test_accumulate_strides_batches(ty):
    assert run(ty, 512, 333, 45, None, True, x_pad=4, y_pad=3, nb=2) <= REL
    assert run(ty, 1024, 2600, 70, 64 << 20, True, x_pad=8, y_pad=5, nb=2) <= REL
    assert run(ty, 1024, 5000, 200, 128 << 20, True, y_pad=1) <= REL


@pytest.mark.parametrize("ty", TYPES)
def test_rows_off_dwords(ty):
    # rows 2 bytes past a dword: formats of whole-dword blocks take the other tiles
    assert run(ty, 512, 300, 40, row_pad=2, w_off=2) <= REL
    assert run(ty, 512, 5000, 200, 128 << 20, row_pad=2) <= REL


def test_results_repeat():
    ty, K, rows, N = T.Q4_K, 4096, 2048, 200
    rng = np.random.default_rng(5)
    raw = synth.random_blocks(rng, ty, rows * K, 3e-4, [0, 2])
    dw, dx = G.DeviceBuffer.from_array(raw), G.DeviceBuffer.from_array(rng.standard_normal((N, K)).astype(np.float32))
    wk = G.DeviceBuffer(64 << 20)
    outs = []
    for _ in range(3):
        dy = G.DeviceBuffer(N * rows * 4)
        G.ops.gemm_ex(ty, dw, G.row_bytes(ty, K), K, rows, dx, K, dy, rows, N, work=wk, work_bytes=wk.nbytes)
        outs.append(dy.download(np.uint32, N * rows))
    assert all(np.array_equal(o, outs[0]) for o in outs[1:])
