"""The fast forward's two routes: one pass over a query block's key tiles, or the
even and odd tiles by two groups of waves that meet in LDS (grids of at most one
workgroup per CU whose rows can see more than ten 64-key tiles).  Both against
the float64 oracle, on each side of the rule, with the parity tests' bounds.
"""
import numpy as np
import pytest
import torch

from femtochat_amd import MFMAFast
from oracle import attention_ref as R
from tests.helpers import TOL, TOL_LSE, gpu_forward, lse_err, rel_err, to_np
from tests.test_gpu_parity import _check_case

pytestmark = pytest.mark.gpu

CASES = [
    # B, T, H, Hkv, D, window: 640 keys (ten tiles) take one pass, 641 two parts
    (1, 640, 2, 1, 64, (-1, 0)),
    (1, 641, 2, 1, 64, (-1, 0)),
    (2, 700, 4, 2, 128, (-1, 0)),
    (1, 777, 2, 2, 16, (-1, 0)),
    (1, 650, 3, 1, 32, (-1, 5)),
    (1, 900, 2, 1, 48, (512, 1)),
    (1, 900, 2, 1, 80, (512, 0)),
    (1, 900, 2, 2, 96, (600, 300)),
    (1, 770, 2, 2, 112, (700, -5)),
    (2, 800, 2, 1, 128, (1000, 1000)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_windows_and_head_dims(gpu, case):
    B, T, H, Hkv, D, window = case
    _check_case(gpu, "fast", B, T, H, Hkv, D, window, seed=T + D)


@pytest.mark.parametrize("D", [64, 128])
def test_documents(gpu, D):
    """Rows that see keys of one part alone (documents of 1 to 200 tokens)."""
    rng = np.random.default_rng(D)
    pos = np.zeros((2, 800), np.int32)
    for b in range(2):
        t = 0
        while t < 800:
            n = int(rng.integers(1, 200))
            pos[b, t:t + n] = np.arange(min(n, 800 - t))
            t += n
    _check_case(gpu, "fast", 2, 800, 2, 1, D, (-1, 0), seed=D, positions=pos)


@pytest.mark.parametrize("tile", [0, 1, 10, 11])
@pytest.mark.parametrize("growth", [40.0, 140.0])
def test_references_of_the_parts_differ(gpu, tile, growth):
    """One 64-key tile's base-2 scores lie `growth` above the others': from the
    first tile of a part the parts' references differ by it (at 140 the other
    part's factor underflows, as its exact share of 2^-140 does); in a later tile
    a part's probabilities grow by it (at 140 its rows are recomputed)."""
    B, T, H, Hkv, D = 1, 760, 2, 1, 64
    rng = np.random.Generator(np.random.PCG64(tile))
    c2 = np.log2(np.e) / np.sqrt(D)
    Q = (2.0 + 0.05 * rng.standard_normal((B, T, H, D))).astype(np.float32)
    K = (0.05 * rng.standard_normal((B, T, Hkv, D))).astype(np.float32)
    K[:, 64 * tile:64 * tile + 64] += np.float32(growth / (c2 * 2.0 * D))
    V = rng.standard_normal((B, T, Hkv, D)).astype(np.float32)
    Q, K, V = (torch.from_numpy(x).bfloat16().float().numpy() for x in (Q, K, V))
    O, l, m = gpu_forward(MFMAFast(), *(torch.from_numpy(x).to(gpu, torch.bfloat16) for x in (Q, K, V)), (-1, 0))
    torch.cuda.synchronize()
    O_ref, l_ref, m_ref = R.forward(Q, K, V, (-1, 0))
    assert np.all(np.isfinite(to_np(O))) and rel_err(to_np(O), O_ref) <= TOL["fast"]
    # |L| reaches 100: float32 statistics, the bound is relative to it
    L = to_np(m).astype(np.float64) + np.log(to_np(l).astype(np.float64))
    L_ref = m_ref + np.log(l_ref)
    assert np.max(np.abs(L - L_ref) / np.maximum(1.0, np.abs(L_ref))) <= TOL_LSE


@pytest.mark.parametrize("key", [3, 70])
def test_nan_and_infinity_stay_in_their_rows(gpu, key):
    """A NaN query: its row alone; an infinite V element in either part: the rows
    whose 32-key block holds it, in its column."""
    B, T, H, Hkv, D = 1, 700, 2, 1, 64
    rng = np.random.Generator(np.random.PCG64(key))
    Q, K, V = (torch.from_numpy(rng.standard_normal((B, T, h, D)).astype(np.float32)).bfloat16().float().numpy()
               for h in (H, Hkv, Hkv))
    O_ref, l_ref, m_ref = R.forward(Q, K, V, (-1, 0))
    Qn, Vn = Q.copy(), V.copy()
    Qn[0, 680, 1, 5] = np.nan
    Vn[0, key, 0, 7] = np.inf
    O, l, m = gpu_forward(MFMAFast(), *(torch.from_numpy(x).to(gpu, torch.bfloat16) for x in (Qn, K, Vn)), (-1, 0))
    torch.cuda.synchronize()
    O, l, m = (to_np(x).copy() for x in (O, l, m))
    assert np.all(np.isnan(O[0, 680, 1])) and (np.isnan(l[0, 1, 680]) or np.isnan(m[0, 1, 680]))
    O[0, 680, 1], l[0, 1, 680], m[0, 1, 680] = O_ref[0, 680, 1], l_ref[0, 1, 680], m_ref[0, 1, 680]
    seen = O[0, key:, :, 7]
    assert np.all(np.isinf(seen[np.arange(T - key) != 680 - key]))
    O[0, :, :, 7] = O_ref[0, :, :, 7]
    assert rel_err(O, O_ref) <= TOL["fast"] and lse_err(l, m, l_ref, m_ref) <= TOL_LSE
