"""Routing of whole batches (glmssd.moe.route) bit for bit against the same formula one token and one
expert at a time: expert counts around the array kernels' widths, ties, infinite logits, k up to all."""
import numpy as np
import pytest

from glmssd.moe import route


def one_by_one(logits, bias, k, norm, scale):
    out = []
    for row in logits:
        scores = [np.float32(1.0) / (np.float32(1.0) + np.exp(-row[e:e + 1])[0]) for e in range(row.size)]
        order = sorted(range(row.size), key=lambda e: -(scores[e] + bias[e]))[:k]
        wsum = np.float32(0.0 if norm else 1.0)
        for e in order if norm else []:
            wsum = wsum + scores[e]
        out.append([(e, float(scores[e] / (wsum + np.float32(1e-20)) * np.float32(scale))) for e in order])
    return out


@pytest.mark.parametrize("t,ne,k", [(1, 1, 1), (1, 7, 7), (3, 16, 2), (5, 33, 8), (4, 288, 8), (17, 31, 9), (2, 5, 9)])
@pytest.mark.parametrize("norm,scale", [(True, 2.5), (False, 1.0)])
def test_batches_match_one_by_one(t, ne, k, norm, scale):
    rng = np.random.default_rng([t, ne, k])
    logits = np.round(rng.standard_normal((t, ne)) * 3, 1).astype(np.float32)   # rounded: ties
    bias = np.round(rng.standard_normal(ne) * 0.2, 1).astype(np.float32)
    logits[0, 0] = np.inf
    logits[-1, ne // 2] = -np.inf
    assert route(logits, bias, k, norm, scale) == one_by_one(logits, bias, k, norm, scale)
