"""Exact mode at the ends of the float32 range: the products of three bf16
parts stand for float32 products while inputs stay below 2^111 and scores below
2^96; rows that meet others are computed again with fp32 products.

Scaling by a power of two is exact, so a scaled problem must give the scaled
results of the plain one (itself compared with the float64 oracle); both
paths differ from the exact value by at most a few 1e-6 (2-norm: float32
sums of up to 300 terms, n 2^-24 = 2e-5 at the very worst), and the bound is
twice that.
"""
import numpy as np
import pytest
import torch

from femtochat_amd import MFMAExact
from femtochat_amd import kernels as Kn
from oracle import attention_ref as R
from tests.helpers import TOL, gpu_forward, rel_err, to_np

pytestmark = pytest.mark.gpu
BOUND = 4e-5


def _inputs(D, T=300, B=2, H=4, Hkv=2, seed=0):
    rng = np.random.Generator(np.random.PCG64(seed + D))
    Q, K, V, dO = (rng.standard_normal((B, T, h, D), dtype=np.float32) for h in (H, Hkv, Hkv, H))
    return [np.clip(x, -1.9, 1.9) for x in (Q, K, V)] + [0.1 * dO]


def _run(gpu, Q, K, V, dO, window=(-1, 0)):
    t = [torch.from_numpy(np.ascontiguousarray(x)).to(gpu) for x in (Q, K, V, dO)]
    st = Kn.attention_state(MFMAExact(), *t[:3], window)
    g = [torch.empty_like(x) for x in t[:3]]
    Kn.delta_attention_(MFMAExact(), *g, t[3], *t[:3], st.O, st.l, st.m, window, accumulate=False)
    torch.cuda.synchronize()
    return [to_np(x).astype(np.float64) for x in (st.O, *g)]


def _close(x, y):
    return np.linalg.norm(x - y) <= BOUND * np.linalg.norm(y)


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("q,k,v,do", [(-100, 100, 0, 0), (110, -110, 0, 0), (0, 0, 116, -126), (0, 0, 0, -110),
                                      (0, 0, -112, 0), (0, 0, -60, 60)])
def test_scaled_inputs(gpu, D, q, k, v, do):
    Q, K, V, dO = _inputs(D)
    plain = _run(gpu, Q, K, V, dO)
    l_ref = R.forward(Q, K, V, (-1, 0))
    assert rel_err(plain[0], l_ref[0]) <= TOL["exact"]
    f = [np.float32(2.0) ** np.float32(e) for e in (q, k, v, do)]
    scaled = _run(gpu, Q * f[0], K * f[1], V * f[2], dO * f[3])
    fs = [float(x) for x in f]
    for x, y, s in zip(scaled, plain, (fs[2], fs[2] * fs[3] / fs[0], fs[2] * fs[3] / fs[1], fs[3])):
        assert np.all(np.isfinite(x)) and _close(x / s, y)


@pytest.mark.parametrize("D", [16, 64, 112, 128])
@pytest.mark.parametrize("v,do", [(-24, -92), (-56, -56), (-60, -60)])
def test_small_score_gradients(gpu, D, v, do):
    """V and dO whose product, and with it dS, falls to 2^-112 .. 2^-120 while
    neither is small for a float32: dS keeps its 24 bits.  What float32 itself
    loses are sums' terms below 2^-149 (2^-26 of a dS of 2^-123, few of them:
    6e-8 in all at v + do = -120 in fp32 products); the bound is 1e-6."""
    Q, K, V, dO = _inputs(D)
    plain = _run(gpu, Q, K, V, dO)
    fv, fd = 2.0 ** v, 2.0 ** do
    scaled = _run(gpu, Q, K, V * np.float32(fv), dO * np.float32(fd))
    for name, x, y, s in zip(("O", "dQ", "dK", "dV"), scaled, plain, (fv, fv * fd, fv * fd, fd)):
        e = np.linalg.norm(x / s - y) / np.linalg.norm(y)
        assert e <= 1e-6, f"{name} {e}"


@pytest.mark.parametrize("D", [64, 96])
@pytest.mark.parametrize("which", ["Q", "K", "V", "dO"])
def test_tiny_column(gpu, D, which):
    """One column of 2^-118 times its neighbours: the output column that it alone
    makes (of dK, dQ, O, dV) has the relative precision of the others, a few
    1e-7 (float32 sums of 300 terms); the bound is 2e-6."""
    t = dict(zip(("Q", "K", "V", "dO"), _inputs(D, B=1)))
    t[which][..., 3] *= np.float32(2.0) ** np.float32(-118)
    Q, K, V, dO = t.values()
    out = dict(zip(("O", "dQ", "dK", "dV"), _run(gpu, Q, K, V, dO)))
    O, l, m = R.forward(Q, K, V, (-1, 0))
    ref = dict(zip(("O", "dQ", "dK", "dV"), (O, *R.backward(dO, Q, K, V, O, l, m, (-1, 0)))))
    name = dict(Q="dK", K="dQ", V="O", dO="dV")[which]
    x, y = out[name][..., 3], ref[name][..., 3]
    e = np.linalg.norm(x - y) / np.linalg.norm(y)
    assert e <= 2e-6, f"{name} {e}"


@pytest.mark.parametrize("B,T,H,Hkv,D,window", [(2, 333, 4, 2, 128, (-1, 0)), (1, 300, 6, 2, 64, (200, 3)),
                                                (2, 270, 4, 1, 80, (-1, 0)), (1, 257, 2, 2, 16, (-1, 0))])
def test_float32_precision(gpu, B, T, H, Hkv, D, window):
    """O and the gradients within 2e-6 (2-norm) of float64, as float32 products
    give them; without the products of the third parts the error is above 3e-6
    (tests/test_exact_split.py)."""
    Q, K, V, dO = _inputs(D, T=T, B=B, H=H, Hkv=Hkv)
    O, l, m = R.forward(Q, K, V, window)
    ref = (O, *R.backward(dO, Q, K, V, O, l, m, window))
    for name, x, y in zip(("O", "dQ", "dK", "dV"), _run(gpu, Q, K, V, dO, window), ref):
        e = np.linalg.norm(x - y) / np.linalg.norm(y)
        assert e <= 2e-6, f"{name} {e}"


@pytest.mark.parametrize("D", [32, 128])
def test_infinite_value_and_nan_query(gpu, D):
    """An infinite V element reaches the queries that see its key (and, as 0
    times infinity, those whose 32-key tile holds it), in its column alone; a
    NaN in a query stays in that query's row."""
    Q, K, V, dO = _inputs(D, B=1, H=2, Hkv=1)
    plain = _run(gpu, Q, K, V, dO)[0]
    V2 = V.copy()
    V2[0, 150, 0, 3] = np.inf
    O = _run(gpu, Q, K, V2, dO)[0]
    assert np.all(O[0, 150:, :, 3] == np.inf) and np.all(np.isfinite(O[0, :128]))
    others = [d for d in range(D) if d != 3]
    assert _close(O[..., others], plain[..., others]) and _close(O[0, :128], plain[0, :128])
    Q2 = Q.copy()
    Q2[0, 77, 1, 5] = np.nan
    O = _run(gpu, Q2, K, V, dO)[0]
    assert np.all(np.isnan(O[0, 77, 1]))
    O[0, 77, 1] = plain[0, 77, 1]
    assert _close(O, plain)


@pytest.mark.parametrize("D", [16, 128])
def test_large_values_behind_growing_scores(gpu, D):
    """Probabilities of up to 2^40 against the first tile's maximum times values
    of 2^100: the sum leaves the float32 range unless the reference moves."""
    Q, K, V, dO = _inputs(D, B=1, H=2, Hkv=1)
    Q, K = np.abs(Q) + 0.5, np.abs(K) + 0.5
    K *= np.where(np.arange(K.shape[1]) < 256, 0.1, 1.0).astype(np.float32)[None, :, None, None]
    S = np.einsum("thd,kd->htk", Q[0], K[0, :, 0]) * np.log2(np.e) / np.sqrt(D)
    Q *= np.float32(45.0 / S.max())  # base-2 scores up to 45, at most 6 in the first 256 keys
    V *= np.float32(2.0) ** np.float32(100)
    O = _run(gpu, Q, K, V, dO)[0]
    assert np.all(np.isfinite(O)) and rel_err(O, R.forward(Q, K, V, (-1, 0))[0]) <= TOL["exact"]


@pytest.mark.parametrize("D", [16, 128])
def test_growing_scores(gpu, D):
    """Scores that grow along the keys by far more than 2^64 between tiles."""
    Q, K, V, dO = _inputs(D, seed=9)
    Q = np.abs(Q) + 0.5
    K = (np.abs(K) + 0.5) * (np.arange(K.shape[1], dtype=np.float32)[None, :, None, None] / 4)
    O, dQ, dK, dV = _run(gpu, Q, K, V, dO)
    O_ref, l_ref, m_ref = R.forward(Q, K, V, (-1, 0))
    g_ref = R.backward(dO, Q, K, V, O_ref, l_ref, m_ref, (-1, 0))
    # scores of up to 600 carry a rounding of 600 log2(e) 2^-24 in the exponent
    for x, r in zip((O, dV), (O_ref, g_ref[2])):
        assert rel_err(x, r) <= 3 * TOL["exact"]


@pytest.mark.parametrize("D", [64, 128])
def test_growing_scores_leave_the_other_rows(gpu, D):
    """A query whose scores grow by far more than 2^64 behind the first tile
    changes its own row alone: the other rows of its wave keep their bits (they
    would not, were the wave's products done again another way)."""
    g = torch.Generator(device=gpu).manual_seed(D)
    Q, K, V = (torch.randn(1, 500, 2, D, device=gpu, generator=g) for _ in range(3))
    plain = gpu_forward(MFMAExact(), Q, K, V, (-1, 0))
    Q2 = Q.clone()
    Q2[0, 400, 1] = 40.0 * K[0, 200, 1]
    O, l, m = gpu_forward(MFMAExact(), Q2, K, V, (-1, 0))
    torch.cuda.synchronize()
    O_ref, l_ref, m_ref = R.forward(*(to_np(x) for x in (Q2, K, V)), (-1, 0))
    assert m_ref[0, 1, 400] > 200 and rel_err(to_np(O), O_ref) <= TOL["exact"]
    for x, y, at in zip((O, l, m), plain, ((0, 400, 1), (0, 1, 400), (0, 1, 400))):
        x[at] = y[at]
        assert torch.equal(x, y)


@pytest.mark.parametrize("D", [16, 48, 80, 112])
def test_head_dims_between_blocks_ignore_old_lds(gpu, D):
    """Tiles of these head dims leave LDS columns unwritten (or read past 16 of
    them): what an earlier launch left there must not send rows to the
    recomputation.  The same bits after a launch that fills LDS with NaN as after
    one that fills it with ones."""
    g = torch.Generator(device=gpu).manual_seed(D)
    Q, K, V = (torch.randn(2, 200, 4, D, device=gpu, generator=g) for _ in range(3))
    results = []
    for fill in (float("nan"), 1.0):
        X = torch.full((8, 1024, 16, 128), fill, device=gpu)  # enough workgroups for every CU
        gpu_forward(MFMAExact(), X, X, X, (-1, 0))
        results.append(gpu_forward(MFMAExact(), Q, K, V, (-1, 0)))
    for x, y in zip(*results):
        assert torch.equal(x, y)
