"""GPU checks of the column route of the forward sums (csrc/col.hip) at the edges of its workgroup shapes: the element
counts N + M where the threads or elements per thread change, the switch from two channels per workgroup to one, odd
channel counts, one-sided sizes and the last size before the ranges take over.

Against the fp64 oracle on a subsample of the queries, at the bar of every forward sum: 1e-5 of sum |term|. The fp32
error of these sums is a few roundings of partial sums no larger than sum |term| (measured: below 1e-6), so 1e-5 has room.
"""

import numpy as np
import pytest
import torch

from oracle import brute, inputs

pytestmark = pytest.mark.gpu

REL = 1e-5
# N + M just at and past every capacity of col_plan (threads x elements per thread), CH = 2 up to 20352 elements
EDGES = [768, 769, 1024, 1025, 1536, 1537, 2048, 2049, 4096, 4097, 6144, 6145, 8192, 8193, 10240, 10241, 12288, 12289,
         16384, 16385, 20352, 20353, 20480, 20481, 24576, 24577, 28672, 28673, 32768, 32769]


def _data(P, D, N, M, C, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "ties":
        q = (rng.integers(-6, 7, size=(P, D, M)) / 4).astype(np.float32)
        k = (rng.integers(-6, 7, size=(P, D, N)) / 4).astype(np.float32)
    else:
        q = rng.standard_normal((P, D, M), dtype=np.float32)
        k = rng.standard_normal((P, D, N), dtype=np.float32)
        if kind == "far":                          # offset by 300, with keys and queries far out on both sides
            q += 300
            k += 300
            q[..., 0] = -4000
            k[..., -1] = 9000
    return q, k, rng.standard_normal((P, N, C), dtype=np.float32)


def _check(dev, P, D, N, M, C, kind, seed):
    from weighted_abs_sum import weighted_abs_sum_full
    from weighted_laplace_sum import weighted_laplace_sum
    print(f"columns P={P} D={D} N={N} M={M} C={C} {kind}", flush=True)
    q, k, v = _data(P, D, N, M, C, kind, seed)
    tq, tk, tv = (torch.from_numpy(a).to(dev) for a in (q, k, v))
    idx = inputs.query_subsample(P, M, per_p=24, seed=seed)
    for name, op, oracle in (("abs", lambda *a: weighted_abs_sum_full(*a, backend="cuda"), brute.abs_sum),
                             ("laplace", weighted_laplace_sum, brute.laplace_sum)):
        w, u = (t.cpu().numpy() for t in op(tq, tk, tv))
        assert np.isfinite(w).all() and np.isfinite(u).all(), name
        ow, ou, nw = oracle(q, k, v, qidx=idx)
        w = np.stack([w[p][idx[p]] for p in range(P)])
        u = np.stack([u[p][idx[p]] for p in range(P)])
        assert float(brute.rel_err(w, ow, nw).max()) <= REL, f"{name} out_w"
        assert float(brute.rel_err(u, ou, ou).max()) <= REL, f"{name} out_u"


@pytest.fixture
def no_dense(pin_route):
    pin_route("columns")


@pytest.mark.parametrize("kind", ["normal", "ties"])
@pytest.mark.parametrize("n", EDGES)
def test_column_capacity_edges(dev, no_dense, n, kind):
    N = n // 2 + 3
    _check(dev, 1, 3, N, n - N, 3, kind, seed=n)


@pytest.mark.parametrize("shape", [(1, 1, 17, 1, 1), (2, 1, 18, 40, 2), (1, 2, 32000, 700, 5), (1, 2, 700, 32000, 2),
                                   (2, 5, 600, 610, 1), (1, 2, 9000, 8000, 1), (3, 33, 900, 1100, 7),
                                   (40, 2, 1200, 900, 128), (2, 64, 5003, 3001, 33)])
@pytest.mark.parametrize("kind", ["normal", "far"])
def test_column_shapes(dev, no_dense, shape, kind):
    _check(dev, *shape, kind, seed=sum(shape))


def test_one_channel_and_many_features(dev, no_dense):
    # 60000 features: with 10240 elements a segment, as one channel once took, a p's stream passes 32-bit offsets
    _check(dev, 1, 60000, 20, 600, 1, "normal", seed=2)


def test_laplace_infinite_keys_and_queries(dev, no_dense):
    # an infinite key adds 0 to every finite query, an infinite query sums to 0 over finite keys; neighbours stay exact
    from weighted_laplace_sum import weighted_laplace_sum
    P, D, N, M, C = 1, 2, 2000, 1500, 3
    q, k, v = _data(P, D, N, M, C, "normal", 5)
    k[0, 0, [3, 40]] = np.inf
    k[0, 1, 7] = -np.inf
    q[0, 0, 11] = np.inf
    w, u = (t.cpu().numpy() for t in weighted_laplace_sum(*(torch.from_numpy(a).to(dev) for a in (q, k, v))))
    with np.errstate(invalid="ignore"):            # inf - inf, set below
        a = [np.exp(-np.abs(q[0, d, :, None].astype(np.float64) - k[0, d][None])) for d in range(D)]
    a[0][11, [3, 40]] = 1.0                        # equal infinities are 0 apart
    A = a[0] + a[1]
    assert float(brute.rel_err(w[0], A @ v[0], A @ np.abs(v[0]).astype(np.float64)).max()) <= REL
    assert float(brute.rel_err(u[0], A.sum(1), A.sum(1)).max()) <= REL


@pytest.mark.parametrize("kind", ["normal", "ties", "runs"])
@pytest.mark.parametrize("shape", [(1, 3, 18, 19, 1), (2, 2, 400, 369, 3), (1, 3, 700, 800, 65), (1, 2, 2100, 1990, 5),
                                   (1, 2, 5000, 5239, 2), (1, 2, 9000, 7385, 9), (1, 2, 9900, 10453, 3),
                                   (1, 2, 16384, 16384, 18), (1, 2, 31000, 900, 2), (2, 1, 900, 30000, 1)])
def test_column_backward(dev, no_dense, shape, kind):
    # grad_q, grad_k, grad_v with and without g_u, and the sgn sum, at the workgroup shapes' edges; "ties": runs of
    # equal queries and keys that cross threads and waves, "runs": one value for long stretches. Ties count -1 (sgn:
    # +1).
    from weighted_abs_sum import _ext, weighted_sgn_sum
    P, D, N, M, C = shape
    print(f"column backward {shape} {kind}", flush=True)
    q, k, v = _data(P, D, N, M, C, "normal" if kind == "normal" else "ties", seed=sum(shape))
    if kind == "runs":
        q[..., : M // 2] = 0.25
        k[..., : N // 2] = 0.25
    rng = np.random.default_rng(1)
    g = rng.standard_normal((P, M, C), dtype=np.float32)
    gu = rng.standard_normal((P, M), dtype=np.float32)
    iq, ik = inputs.query_subsample(P, M, per_p=12, seed=2), inputs.query_subsample(P, N, per_p=12, seed=3)
    t = [torch.from_numpy(a).to(dev) for a in (q, k, v, g, gu)]
    pick = lambda a, i, ax: np.stack([np.take(a[p], i[p], axis=ax) for p in range(P)])  # noqa: E731
    for u in (gu, None):
        got = (_ext.weighted_abs_sum_full_backward(*t) if u is not None else _ext.weighted_abs_sum_backward(*t[:4]))
        got = [x.cpu().numpy() for x in got]
        (wq, wk, wv), (nq, nk, nv) = brute.abs_backward_sub(q, k, v, g, u, iq, ik)
        for name, a, w, nn in (("grad_q", pick(got[0], iq, 1), wq, nq), ("grad_k", pick(got[1], ik, 1), wk, nk),
                               ("grad_v", pick(got[2], ik, 0), wv, nv)):
            assert float(brute.rel_err(a, w, nn).max()) <= REL, name
    sgn = weighted_sgn_sum(*t[:4], backend="cuda").cpu().numpy()
    (wq, _, _), (nq, _, _) = brute.abs_backward_sub(q, k, v, g, None, iq, ik)
    assert float(brute.rel_err(pick(sgn, iq, 1), -wq, nq).max()) <= REL


# ---- layers; queries and keys that are not finite, or huge: their own row only

BAD = {"inf": np.inf, "-inf": -np.inf, "nan": np.nan, "-nan": -np.nan, "huge": 3e38}


def _layer64(kernel, q, k, v, keep, M):
    """float64 num (rows, C) and den (rows) of one p's layer at queries q (D, rows) over its kept keys k (D, N) with
    rows v, and the sums of |term| that the abs or Laplace sums and the epilogue form them from: each is within REL of those."""
    from qlka import layers
    n_pad = int((~keep).sum())
    q, k, v = q.astype(np.float64), k[:, keep].astype(np.float64), v[keep].astype(np.float64)
    x = q[:, :, None] - k[:, None]
    if kernel == "add_laplace":
        A = S = np.exp(-np.abs(x)).sum(0)
    elif kernel == "add_bump":
        A = np.maximum(0, 1 - np.abs(x)).sum(0)
        S = ((np.abs(x + 1) + np.abs(x - 1)) / 2 + np.abs(x)).sum(0)
    else:
        near, far = np.abs(x).sum(0), np.abs(q).sum(0)[:, None] + np.abs(k).sum(0)[None] + layers.EPS
        A, S = far - near, far + near
    den, sden = A.sum(1), S.sum(1)
    if kernel == "add_riesz":                      # it counts M keys (attention.py:78), less the masked ones
        den = den + (np.abs(q).sum(0) + layers.EPS) * (M - n_pad - k.shape[1])
    return A @ v, np.maximum(den, layers.CLAMP), S @ np.abs(v), sden


def _assert_layer(kernel, got, q, k, v, keep, M):
    num, den, snum, sden = _layer64(kernel, q, k, v, keep, M)
    assert np.isfinite(got).all(), kernel
    err = np.abs(got * den[:, None] - num)
    np.testing.assert_array_less(err, REL * (snum + np.abs(got) * sden[:, None]) + 1e-30, err_msg=kernel)


@pytest.mark.parametrize("kernel", ["add_laplace", "add_riesz", "add_bump"])
@pytest.mark.parametrize("N,M,C", [(1030, 1020, 6), (3111, 3111, 64), (12000, 9000, 31)])
def test_masked_layer_columns(dev, no_dense, kernel, N, M, C):
    # masked rows weigh 0 whatever they hold (NaN in v, large k), against the float64 layer over the kept keys
    from qlka import layers
    P, D = 2, 4
    q, k, v = _data(P, D, N, M, C, "normal", N)
    keep = np.random.default_rng(N).random((P, N)) < 0.7
    k[np.broadcast_to(~keep[:, None], k.shape)] = 50.0
    v[~keep] = np.nan
    got = layers.layer_forward(kernel, *(torch.from_numpy(a).to(dev) for a in (q, k, v)),
                               keep=torch.from_numpy(keep).to(dev)).cpu().numpy()
    rows = np.arange(0, M, max(1, M // 50))
    for p in range(P):
        _assert_layer(kernel, got[p][rows], q[p][:, rows], k[p], v[p], keep[p], M)


@pytest.mark.parametrize("bad", sorted(BAD))
@pytest.mark.parametrize("shape", [(2, 3, 700, 650, 5), (1, 2, 12000, 11000, 3), (1, 2, 16000, 16000, 2)])
def test_a_bad_query_spoils_only_its_row(dev, no_dense, shape, bad):
    # as by the walks: abs and layer rows of an infinite or NaN query are NaN, Laplace's are 0 for an infinite one;
    # every other row is what the oracle says. A huge finite query (differences past the largest float) spoils no other
    # row.
    from qlka import layers
    from weighted_abs_sum import weighted_abs_sum, weighted_abs_sum_full
    from weighted_laplace_sum import weighted_laplace_sum
    P, D, N, M, C = shape
    print(f"bad query {shape} {bad}", flush=True)
    q, k, v = _data(P, D, N, M, C, "normal", 3)
    at = 7
    q[0, 1, at] = BAD[bad]
    if bad == "huge":
        q[0, 0, at] = -3e38
    tq, tk, tv = (torch.from_numpy(a).to(dev) for a in (q, k, v))
    assert bool(torch.signbit(tq[0, 1, at])) == bad.startswith("-")
    idx = inputs.query_subsample(P, M, per_p=16, seed=5)
    idx = [i[i != at] for i in idx]
    rows = lambda a, p: a[p][idx[p]]  # noqa: E731
    for name, op, oracle in (("abs", lambda: weighted_abs_sum_full(tq, tk, tv, backend="cuda"), brute.abs_sum),
                             ("plain", lambda: (weighted_abs_sum(tq, tk, tv, backend="cuda"), None), brute.abs_sum),
                             ("laplace", lambda: weighted_laplace_sum(tq, tk, tv), brute.laplace_sum)):
        w, u = (t if t is None else t.cpu().numpy() for t in op())
        for p in range(P):
            ow, ou, nw = oracle(q[p:p + 1], k[p:p + 1], v[p:p + 1], qidx=idx[p:p + 1])
            assert float(brute.rel_err(rows(w, p)[None], ow, nw).max()) <= REL, name
            if u is not None:
                assert float(brute.rel_err(rows(u, p)[None], ou, ou).max()) <= REL, name
        if bad != "huge" and (name != "laplace" or "nan" in bad):
            assert np.isnan(w[0, at]).all() and (u is None or np.isnan(u[0, at])), name
        elif bad != "huge":                        # the features of a finite value alone
            ow, ou, nw = oracle(np.delete(q, 1, 1), np.delete(k, 1, 1), v, qidx=[np.array([at])] * P)
            assert float(brute.rel_err(w[:1, at:at + 1], ow[:1], nw[:1]).max()) <= REL
    keep = np.random.default_rng(N).random((P, N)) < 0.7
    for kernel in layers.KINDS:
        for mask in (np.ones_like(keep), keep):
            arg = None if mask.all() else torch.from_numpy(mask).to(dev)
            got = layers.layer_forward(kernel, tq, tk, tv, keep=arg).cpu().numpy()
            for p in range(P):
                _assert_layer(kernel, rows(got, p), q[p][:, idx[p]], k[p], v[p], mask[p], M)
            if bad != "huge" and (kernel != "add_laplace" or "nan" in bad):
                assert np.isnan(got[0, at]).all(), kernel


@pytest.mark.parametrize("bad", ["inf", "nan", "-nan"])
@pytest.mark.parametrize("shape", [(2, 3, 700, 650, 5), (1, 2, 12000, 11000, 3)])
def test_a_bad_key_spoils_only_its_row_of_grad_v(dev, no_dense, shape, bad):
    from weighted_abs_sum import _ext
    P, D, N, M, C = shape
    q, k, v = _data(P, D, N, M, C, "normal", 4)
    g = np.random.default_rng(6).standard_normal((P, M, C), dtype=np.float32)
    k[0, 1, 9] = BAD[bad]
    gv = _ext.weighted_abs_sum_backward(*(torch.from_numpy(a).to(dev) for a in (q, k, v, g)))[2].cpu().numpy()
    assert np.isnan(gv[0, 9]).all()
    idx = [i[i != 9] for i in inputs.query_subsample(P, N, per_p=16, seed=7)]
    for p in range(P):                             # grad_v: the abs sum with q and k exchanged
        w, _, nw = brute.abs_sum(k[p:p + 1], q[p:p + 1], g[p:p + 1], qidx=idx[p:p + 1])
        assert float(brute.rel_err(gv[p][idx[p]][None], w, nw).max()) <= REL


def test_a_thread_on_both_sides_of_the_median(dev, no_dense):
    # a far query, then the keys, all in the first thread's elements: the others' sums stay as precise as their
    # distances to the keys are (1.5e-3 of sum |term| where such a thread's values were relative to the far query)
    from weighted_abs_sum import weighted_abs_sum_full
    P, D, N, M, C = 2, 2, 17, 700, 3
    rng = np.random.default_rng(8)
    q = (300.2 + 0.5 * rng.random((P, D, M))).astype(np.float32)
    q[..., 0] = -4000
    k = np.tile((300 + 0.01 * np.arange(N)).astype(np.float32), (P, D, 1))
    v = rng.standard_normal((P, N, C), dtype=np.float32)
    w, u = (t.cpu().numpy() for t in weighted_abs_sum_full(*(torch.from_numpy(a).to(dev) for a in (q, k, v)),
                                                           backend="cuda"))
    ow, ou, nw = brute.abs_sum(q, k, v)
    assert float(brute.rel_err(w, ow, nw).max()) <= REL
    assert float(brute.rel_err(u, ou, ou).max()) <= REL


@pytest.mark.parametrize("kernel", ["add_laplace", "add_riesz", "add_bump"])
@pytest.mark.parametrize("far", ["low", "both", "nan"])
@pytest.mark.parametrize("N,M,kept", [(3000, 2000, 0.4), (3000, 2000, 0.01), (12000, 11000, 0.4),
                                      (12000, 11000, 0.001)])
def test_mostly_masked_keys_far_out(dev, no_dense, kernel, far, N, M, kept):
    # masked keys weigh nothing wherever they lie: most of a segment's keys masked and far below the kept ones, on both
    # sides of them, or NaN of either sign, with kept keys and queries of scale 1
    from qlka import layers
    P, D, C = 2, 3, 4
    print(f"mostly masked {kernel} N={N} kept={kept} {far}", flush=True)
    q, k, v = _data(P, D, N, M, C, "normal", N)
    rng = np.random.default_rng(N + 1)
    keep = rng.random((P, N)) < kept
    keep[1] = rng.random(N) < 0.7
    out = -1e4 * (1 + rng.random((P, D, N)))
    if far == "both":
        out *= np.where(rng.random((P, 1, N)) < 0.5, -1e3, 1.0)
    out = out.astype(np.float32)
    if far == "nan":
        out = np.where(rng.random((P, 1, N)) < 0.5, np.float32(np.nan), -np.float32(np.nan))
    k = np.where(keep[:, None], k, out).astype(np.float32)
    got = layers.layer_forward(kernel, *(torch.from_numpy(a).to(dev) for a in (q, k, v)),
                               keep=torch.from_numpy(keep).to(dev)).cpu().numpy()
    idx = inputs.query_subsample(P, M, per_p=24, seed=9)
    for p in range(P):
        _assert_layer(kernel, got[p][idx[p]], q[p][:, idx[p]], k[p], v[p], keep[p], M)


@pytest.mark.parametrize("kind", ["grid 1e-4", "grid 0.1", "grid 3", "uniform 2e-5", "normal 1e-5", "dyadic",
                                  "normal 1"])
@pytest.mark.parametrize("n", [1100, 3000, 8192, 16384])
def test_laplace_keys_whose_roundings_repeat(dev, no_dense, n, kind):
    # Decays between neighbours that are all alike (grids) or all below a rounding of 1 (narrow keys), where the errors
    # of a chain of products add up. Relative 2-norm: at most 31 products in a thread and 15 across waves, half of them
    # on average, each off by up to 2^-25 to the same side: 7e-7; by factors rounded one by one and multiplied up
    # through the scans 1.2e-6 to 6.1e-6 (measured, the grids and narrow keys here), by the walks up to 1.4e-6.
    from weighted_laplace_sum import weighted_laplace_sum
    P, D, C = 1, 4, 5
    print(f"repeating roundings {kind} n={n}", flush=True)
    rng = np.random.default_rng(n)

    def points():
        name, width = (kind.split() + ["1"])[:2]
        if name == "grid":
            x = np.linspace(-1, 1, n) * float(width)
            x = np.stack([rng.permutation(x) for _ in range(D)])
        elif name == "dyadic":
            x = np.stack([rng.permutation(n) for _ in range(D)]) / 1024.0
        else:
            x = float(width) * (rng.uniform(-1, 1, (D, n)) if name == "uniform" else rng.standard_normal((D, n)))
        return x[None].astype(np.float32)

    q, k, v = points(), points(), rng.standard_normal((P, n, C), dtype=np.float32)
    w, u = (t.cpu().numpy() for t in weighted_laplace_sum(*(torch.from_numpy(a).to(dev) for a in (q, k, v))))
    idx = inputs.query_subsample(P, n, per_p=64, seed=n)
    ow, ou, _ = brute.laplace_sum(q, k, v, qidx=idx)
    assert np.linalg.norm(w[0][idx[0]] - ow[0]) <= 1e-6 * np.linalg.norm(ow[0])
    assert np.linalg.norm(u[0][idx[0]] - ou[0]) <= 1e-6 * np.linalg.norm(ou[0])


@pytest.mark.parametrize("shape", [(1, 3, 63, 64, 2), (1, 3, 65, 127, 3), (2, 2, 4160, 4033, 5),
                                   (1, 2, 12352, 10000, 3)])
def test_columns_of_equal_and_padded_values(dev, no_dense, shape):
    # whole and broken blocks of 64 rows (their words are shuffled within whole ones), all values of a feature equal,
    # and a tail of keys that a mask made 0
    P, D, N, M, C = shape
    from weighted_abs_sum import weighted_abs_sum_full
    from weighted_laplace_sum import weighted_laplace_sum
    print(f"equal and padded {shape}", flush=True)
    q, k, v = _data(P, D, N, M, C, "normal", sum(shape))
    q[:, 0], k[:, 0] = 0.5, 0.5
    k[:, 1, N // 2:] = 0
    v[:, N // 2:] = 0
    g = np.random.default_rng(3).standard_normal((P, M, C), dtype=np.float32)
    t = [torch.from_numpy(a).to(dev) for a in (q, k, v, g)]
    idx, ik = inputs.query_subsample(P, M, per_p=24, seed=2), inputs.query_subsample(P, N, per_p=24, seed=3)
    take = lambda a, i, ax=0: np.stack([np.take(a[p], i[p], axis=ax) for p in range(P)])  # noqa: E731
    for op, oracle in ((lambda *a: weighted_abs_sum_full(*a, backend="cuda"), brute.abs_sum),
                       (weighted_laplace_sum, brute.laplace_sum)):
        w, u = (x.cpu().numpy() for x in op(*t[:3]))
        ow, ou, nw = oracle(q, k, v, qidx=idx)
        assert float(brute.rel_err(take(w, idx), ow, nw).max()) <= REL
        assert float(brute.rel_err(take(u, idx), ou, ou).max()) <= REL
    from weighted_abs_sum import _ext
    got = [x.cpu().numpy() for x in _ext.weighted_abs_sum_backward(*t)]
    (wq, wk, wv), (nq, nk, nv) = brute.abs_backward_sub(q, k, v, g, None, idx, ik)
    for a, w, n in ((take(got[0], idx, 1), wq, nq), (take(got[1], ik, 1), wk, nk), (take(got[2], ik), wv, nv)):
        assert float(brute.rel_err(a, w, n).max()) <= REL


# calls whose two routes were measured 1.3 x and more apart: the slower one is not taken
@pytest.mark.parametrize("op,shape,columns", [
    ("abs", (256, 1, 4000, 4000, 64), False), ("laplace", (256, 1, 4000, 4000, 64), False),      # one feature per p
    ("abs", (40, 4, 14000, 14000, 64), False), ("bwd", (256, 1, 4000, 4000, 64), False),
    ("add_bump", (12, 64, 20000, 600, 64), False),                  # the keys in three streams
    ("sgn", (2, 64, 5200, 5200, 64), False), ("sgn", (512, 4, 1100, 1100, 64), False),
    ("abs", (12, 64, 8192, 8192, 64), True), ("laplace", (12, 64, 8192, 8192, 64), True),
    ("bwd", (12, 64, 8192, 8192, 64), True), ("add_bump", (12, 64, 8192, 8192, 64), True),
    ("laplace", (2, 64, 1225, 703, 4), True), ("abs", (12, 64, 600, 20000, 64), True),
])
def test_the_measured_faster_route_is_taken(dev, op, shape, columns):
    from qlka import _lib, layers
    from weighted_abs_sum import _ext, weighted_abs_sum_full, weighted_sgn_sum
    from weighted_laplace_sum import weighted_laplace_sum
    P, D, N, M, C = shape
    print(f"route {op} {shape}", flush=True)
    g = torch.Generator(dev).manual_seed(1)
    q, k, v, gw = (torch.randn(s, generator=g, device=dev) for s in ((P, D, M), (P, D, N), (P, N, C), (P, M, C)))
    call = {"abs": lambda: weighted_abs_sum_full(q, k, v, backend="cuda"),
            "laplace": lambda: weighted_laplace_sum(q, k, v),
            "bwd": lambda: _ext.weighted_abs_sum_backward(q, k, v, gw),
            "sgn": lambda: weighted_sgn_sum(q, k, v, gw, backend="cuda"),
            "add_bump": lambda: layers.layer_forward("add_bump", q, k, v)}[op]
    lib = _lib.load()
    lib.qlka_timing_enable(1)
    try:
        before = [_lib.stage_time(s)[1] for s in ("col_sort", "col_merge")]
        call()
        torch.cuda.synchronize()
        ran = [_lib.stage_time(s)[1] for s in ("col_sort", "col_merge")] != before
    finally:
        lib.qlka_timing_enable(0)
    assert ran == columns
