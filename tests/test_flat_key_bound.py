"""The flat ranking score whose accumulator starts from ||q||^2 (k above 32)
against the exact squared distance, on the CPU: within flat_key_tau up to the
start value's own error, over float32 emulations of the bf16x3 products (sums
rounded once per step, after every product, and toward zero)."""

import numpy as np
import pytest

from test_proof_bounds import F32, bf16_split, bound_norm, flat_tau, seq_sum


def _score(a, b, start, order):
    ah, al = bf16_split(a)
    bh, bl = bf16_split(b)
    acc = np.broadcast_to(start, np.broadcast_shapes(a.shape[:-1], b.shape[:-1])).astype(F32)
    for t0 in range(0, a.shape[-1], 32):
        for x, y in ((ah, bl), (al, bh), (ah, bh)):
            p = x[..., t0:t0 + 32].astype(np.float64) * y[..., t0:t0 + 32].astype(np.float64)
            if order == "seq":
                for j in range(p.shape[-1]):
                    acc = (acc + p[..., j].astype(F32)).astype(F32)
                continue
            s = acc.astype(np.float64) + p.sum(-1)
            acc = s.astype(F32)
            if order == "trunc":
                acc = np.where(np.abs(acc.astype(np.float64)) > np.abs(s), np.nextafter(acc, F32(0)), acc).astype(F32)
    return acc


@pytest.mark.parametrize("kind", ["gaussian", "large_norm", "near_duplicate"])
@pytest.mark.parametrize("d", [33, 128, 256])
def test_started_score_within_its_bound(oracle, kind, d):
    rng = np.random.default_rng(d + len(kind))
    n, nq = 64, 12
    scale = 300.0 if kind == "large_norm" else 1.0
    X, Q = scale * rng.standard_normal((n, d)), scale * rng.standard_normal((nq, d))
    if kind == "near_duplicate":
        Q = X[rng.integers(0, n, nq)] + 1e-5 * rng.standard_normal((nq, d))
    X, Q = np.asarray(X, F32), np.asarray(Q, F32)
    xnorm, q2 = seq_sum((X * X).astype(F32), axis=1), seq_sum((Q * Q).astype(F32), axis=1)
    tau = flat_tau(d, 0, max(bound_norm(q) for q in Q), max(bound_norm(x) for x in X), -1)
    ref = np.array([[oracle.l2sq(q, x) for x in X] for q in Q], np.float64)
    start_err = q2.astype(np.float64) - (Q.astype(np.float64) ** 2).sum(1)
    for order in ("exact", "seq", "trunc"):
        acc = _score((F32(-2.0) * Q)[:, None, :].astype(F32), X[None], q2[:, None], order)
        v = (xnorm[None, :] + acc).astype(F32).astype(np.float64) - start_err[:, None]
        assert np.abs(v - ref).max() <= tau, (order, np.abs(v - ref).max(), tau)
