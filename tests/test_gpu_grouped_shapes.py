"""The grouped MoE GEMM of prompts under each tile shape its kernel picks from the routing: pair counts on
both sides of its 16- and 32-pair chunks, from one round of the smallest tiles to more tiles of the
largest than CUs take at once, every token to one expert. Against the CPU oracle with the bounds of
test_gpu_grouped.py: 1e-4 of the exact-weight result (f16 activations, f32 sums in any order)."""
import numpy as np
import pytest

import glmssd as G
from glmssd import GgmlType as T
from glmssd import moe as M
import oracle as O

pytestmark = pytest.mark.gpu
REL = 1e-4
CUS = 256


def shape(counts, rows, kind, iq3):
    """The kernel's rule: rounds of the persistent grid times a tile's cost (grouped.hip grouped_auto)."""
    n16, n32 = sum(-(-m // 16) for m in counts), sum(-(-m // 32) for m in counts)
    rb = 256 if kind == 1 else 512
    c = (100, 57, 52) if kind == 1 else (100, 48, 43) if iq3 else (100, 55, 51)
    rounds = (-(-n32 * -(-rows // rb) // CUS), -(-n32 * -(-rows // (rb // 2)) // CUS), -(-n16 * -(-rows // (rb // 2)) // CUS))
    return min(range(3), key=lambda i: rounds[i] * c[i])


def counts_of(case):
    n, lo, hi, extra = case
    return list(np.random.default_rng(case).integers(lo, hi + 1, n)) + list(extra)


CASES = [(40, 1, 16, ()), (60, 17, 32, (0, 1)), (100, 17, 32, (0, 16, 33)), (136, 17, 32, (0, 31, 32, 33, 97)), (30, 31, 34, (15, 16, 17))]


@pytest.mark.parametrize("ty_gu,ty_down", [(T.IQ2_XXS, T.IQ3_XXS), (T.IQ3_XXS, T.IQ2_XXS)])
@pytest.mark.parametrize("case", CASES)
def test_shapes(case, ty_gu, ty_down):
    n_embd, n_ff = 512, 768
    counts = counts_of(case)
    n_exp, n_tok = len(counts), int(sum(counts))
    print(f"grouped {G.TYPE_NAMES[ty_gu]}/{G.TYPE_NAMES[ty_down]} {n_exp} experts {n_tok} pairs", flush=True)
    rng = np.random.default_rng([n_exp, ty_gu])
    owner = rng.permutation(np.repeat(np.arange(n_exp), counts))
    routes = [[(int(e), float(w))] for e, w in zip(owner, rng.random(n_tok) + 0.1)]
    orng = O.Rng(77 + n_exp)
    gate = [orng.random_blocks(ty_gu, n_ff * n_embd) for _ in range(n_exp)]
    up = [orng.random_blocks(ty_gu, n_ff * n_embd) for _ in range(n_exp)]
    down = [orng.random_blocks(ty_down, n_embd * n_ff) for _ in range(n_exp)]
    x = rng.standard_normal((n_tok, n_embd)).astype(np.float32)
    layer = M.ResidentMoeLayer(gate, up, down, n_embd, n_ff, ty_gu, ty_down)
    offs, idx, w, pe = layer.upload_routes(routes)
    want = O.moe_ffn(ty_gu, ty_down, gate, up, down, layer.rs_gu, layer.rs_down, n_embd, n_ff, x, idx, pe, w, lim=5.0,
                     nthreads=8, act="f16sx")
    s = G.Stream()
    dx, dy = G.DeviceBuffer.from_array(x), G.DeviceBuffer.from_array(np.zeros((n_tok, n_embd), np.float32))
    layer.forward(dx, dy, n_tok, 5.0, s)
    got = dy.download(np.float32, n_tok * n_embd, s).reshape(n_tok, n_embd).astype(np.float64)
    G.ops.wait_status(s)
    # per token: one expert's wrong tile does not hide among the others
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 20 * REL and np.linalg.norm(got - want) <= REL * np.linalg.norm(want)


def test_cases_reach_every_shape():
    for kind, rows in ((1, 768), (2, 512)):
        for iq3 in (False, True):
            # IQ3_XXS down never takes the largest tiles
            assert {shape(counts_of(c), rows, kind, iq3) for c in CASES} == ({1, 2} if kind == 2 and iq3 else {0, 1, 2})
