"""The one-row top-k's selection floor (the smallest of the threads' t-th
largest keys) and its keys-per-thread variants, bit-exact against the oracle's
stable top-k: row widths at the variants' edges, K at the edges of t, and rows
where the floor says little (visible keys in few threads, ties, one value,
infinities)."""
import numpy as np
import pytest
import torch

from oracle.indexer import stable_topk as oracle_topk

pytestmark = pytest.mark.gpu


def _rows(S, kind, rng):
    x = rng.randn(3, S).astype(np.float32)
    if kind == "ties":
        x = np.round(x * 4) / 4
    elif kind == "masked":       # few visible keys, all at the front; none; every other one
        x[0, min(S, 37):] = -np.inf
        x[1] = -np.inf
        x[2, ::2] = -np.inf
    elif kind == "spread":       # large outliers and an infinity: all keys but a few in one bin
        x[0, S // 2] = 1e30
        x[1, S - 1] = np.inf
        x[2] = x[2] * 1e-20 + 1.0
    elif kind == "same":
        x[:] = np.float32(0.25)
        x[1, S // 3] = -0.0
        x[2] *= -1
    return x


@pytest.mark.parametrize("kind", ["normal", "ties", "masked", "spread", "same"])
@pytest.mark.parametrize("S", [1, 5, 1023, 1025, 8192, 8193, 16384, 16387, 24576, 24577, 32768])
def test_bit_exact(S, kind):
    from dsa_triton_ascend_amd.lightning_indexer import stable_topk
    x = _rows(S, kind, np.random.RandomState(S))
    for K in (1, 1024, 1025, 2048, 2049, 4096):
        print(f"[topk floor] S={S} {kind} K={K}", flush=True)
        idx, val = stable_topk(torch.from_numpy(x).cuda(), K)
        ei, ev = oracle_topk(x, K)
        assert np.array_equal(idx.cpu().numpy(), ei)
        assert np.array_equal(val.cpu().numpy(), ev)
