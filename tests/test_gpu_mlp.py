"""The MLP's MFMA kernels against the numpy oracle (oracle/mlp_oracle.py)."""
import numpy as np
import pytest

import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(16, 16, 32), (70, 50, 45), (129, 65, 200), (1, 300, 7),
                                   (100, 32, 2048), (300, 20, 700), (64, 96, 1536), (257, 33, 1000)])
def test_gemm_matches_bf16_oracle(gpu, ta, tb, shape):
    m, n, k = shape
    print(f"gemm m={m} n={n} k={k} ta={ta} tb={tb}", flush=True)
    rng = np.random.default_rng(m * 7 + n + k)
    a = rng.standard_normal((k, m) if ta else (m, k)).astype(np.float32)
    b = rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32)
    got = gpu.gemm(a, b, ta, tb)
    want = mo.matmul_bf16(a.T if ta else a, b.T if tb else b)
    # identical bf16 operands on both sides: only the FP32 summation order differs
    scale = mo.matmul_bf16(np.abs(a.T if ta else a), np.abs(b.T if tb else b)) + 1e-30
    assert np.all(np.abs(got - want) <= 1e-5 * scale), np.max(np.abs(got - want) / scale)


def test_gemm_lane_layout_identity(gpu):
    # A = identity picks rows of B exactly (bf16-representable B): catches any
    # transposed or shifted operand/result placement
    rng = np.random.default_rng(1)
    b = mo.bf16_round(rng.standard_normal((32, 48)).astype(np.float32))
    got = gpu.gemm(np.eye(32, dtype=np.float32), b)
    assert np.array_equal(got, b)
    perm = rng.permutation(32)
    got = gpu.gemm(np.eye(32, dtype=np.float32)[perm], b)
    assert np.array_equal(got, b[perm])


def _samples(rng, T, C, n):
    s = np.zeros(n, mo_sample_dtype())
    s["cur"] = rng.integers(0, T, n)
    s["octant"] = rng.integers(0, 8, n)
    s["depth"] = rng.uniform(0, 1, n)
    s["hist"] = rng.integers(0, T, (n, 4))
    s["hist"][rng.uniform(size=(n, 4)) < 0.2] = mo.NONE
    s["target"] = rng.integers(0, C, n)
    return s


def mo_sample_dtype():
    import rtx

    return rtx.MLP_SAMPLE_DTYPE


@pytest.mark.parametrize("T,C,n", [(40, 96, 300), (60, 2500, 700), (20, 17, 33)])
def test_loss_and_gradients_match_oracle(gpu, T, C, n):
    """Loss and every gradient block against the oracle.  The output layer is
    fused (logits only in registers): 2,500 classes span three row-statistics
    chunks and sixteen class splits of the dQ pass; 17 classes and 33 rows
    leave most of every tile empty."""
    rng = np.random.default_rng(5 + C)
    mlp = gpu.mlp(T, C, seed=9)
    try:
        vec = mlp.params()
        P = mo.unpack(vec.copy(), T, C)
        P["o"][:] = rng.standard_normal(C).astype(np.float32) * 0.1
        for k in ("b1", "b2", "b3"):
            P[k][:] = rng.standard_normal(P[k].shape).astype(np.float32) * 0.1
        vec = mo.pack(P, T, C)
        mlp.set_params(vec)
        s = _samples(rng, T, C, n)
        loss = mlp.loss_grad(s)
        g = mo.unpack(mlp.grads(), T, C)
        lo, G = mo.loss_and_grad(mo.unpack(vec, T, C), s, bf16=True)
        assert abs(loss - lo) <= 1e-4 * max(1.0, abs(lo)), (loss, lo)
        for k in G:
            d = np.linalg.norm(g[k] - G[k]) / (np.linalg.norm(G[k]) + 1e-12)
            assert d < 1e-2, (k, d)
        # the padded rows of W1 stay untouched by the gradient
        assert np.all(g["W1"][mo.IN:] == 0)
    finally:
        mlp.close()


def test_predict_matches_oracle_top4(gpu):
    T, C, n = 30, 200, 500
    rng = np.random.default_rng(6)
    mlp = gpu.mlp(T, C, seed=3)
    try:
        s = _samples(rng, T, C, n)
        top, prob = mlp.predict(s)
        P = mo.unpack(mlp.params(), T, C)
        otop, oprob = mo.top4(P, s, bf16=True)
        *_, L = mo.forward(P, s, bf16=True)
        Ls = -np.sort(-L, axis=1)
        clear = np.all(np.abs(np.diff(Ls[:, :5], axis=1)) > 1e-3, axis=1)  # no near-ties in the top 5
        assert clear.mean() > 0.5
        assert np.array_equal(top[clear], otop[clear])
        assert np.allclose(prob[clear], oprob[clear], rtol=1e-3, atol=1e-5)
        assert np.all(np.diff(prob, axis=1) <= 1e-7)
    finally:
        mlp.close()


def test_training_learns_a_treelet_rule(gpu):
    # next class = a fixed function of (cur, octant): the network must fit it
    T, C, n = 64, 128, 8192
    rng = np.random.default_rng(7)
    rule = rng.integers(0, C, (T, 8))
    s = _samples(rng, T, C, n)
    s["target"] = rule[s["cur"], s["octant"]]
    mlp = gpu.mlp(T, C, seed=1)
    try:
        buf = mlp.upload(s)
        l0 = mlp.loss_grad(buf, n)
        last = mlp.train(buf, n, epochs=30, batch=512, lr=3e-3)
        top, _ = mlp.predict(buf, n)
        acc = np.mean(top[:, 0] == s["target"])
        print(f"loss {l0:.3f} -> {last:.3f}, top-1 accuracy {acc:.3f}")
        assert last < 0.25 * l0 and acc > 0.9
    finally:
        mlp.close()


@pytest.mark.parametrize("T,C,n", [(30, 3, 5), (30, 17, 16), (50, 257, 65), (40, 1000, 4097), (20, 300, 2100)])
def test_predict_at_tile_edges(gpu, T, C, n):
    """Fewer than four classes, class counts around the MFMA tile and the LDS
    stage, row counts around the row tiles and the 4,096-row batches.  Both
    sides round operands to BF16; a sum of another order may flip one rounding
    of an activation (2^-8 relative), which moves a logit of this size by at
    most about 1e-3, so classes closer than 5e-3 may swap and probabilities
    agree to 5e-3."""
    rng = np.random.default_rng(C + n)
    mlp = gpu.mlp(T, C, seed=C)
    try:
        s = _samples(rng, T, C, n)
        top, prob = mlp.predict(s)
        P = mo.unpack(mlp.params(), T, C)
        *_, L = mo.forward(P, s, bf16=True)
        k = min(4, C)
        order = np.argsort(-L, axis=1, kind="stable")
        Ls = np.take_along_axis(L, order, axis=1)[:, :k + 1]
        clear = np.all(-np.diff(Ls, axis=1) > 5e-3, axis=1)
        assert clear.mean() > 0.5
        assert np.array_equal(top[clear, :k], order[clear, :k].astype(np.uint32))
        p = np.exp(L - L.max(axis=1, keepdims=True))
        p = np.take_along_axis(p / p.sum(axis=1, keepdims=True), order, axis=1)[:, :k]
        assert np.allclose(prob[clear, :k], p[clear], rtol=5e-3)
        assert np.all(top[:, k:] == 0xFFFFFFFF) and np.all(prob[:, k:] == 0)
    finally:
        mlp.close()


@pytest.mark.parametrize("T,C,n,batch", [(40, 33, 70, 33), (500, 300, 260, 129), (7, 1000, 40, 40)])
def test_training_matches_oracle_steps(gpu, T, C, n, batch):
    """Whole Adam epochs (row and class counts off the 16- and 32-wide tiles, a short
    last batch, embedding rows no sample names) against the oracle's gradients and a
    plain Adam.  A step moves a weight by at most lr, and BF16 flips change a gradient
    by about 1%, so after k steps weights agree to 0.1 * k * lr in the mean; a
    gradient near zero may change sign, which bounds a single weight by 2 * k * lr.
    Rows without samples stay as they were, bit for bit."""
    rng = np.random.default_rng(T + C)
    lr, epochs = 1e-3, 2
    mlp = gpu.mlp(T, C, seed=T)
    try:
        s = _samples(rng, T // 2, C, n)  # the upper half of the rows is never named
        vec = mlp.params()
        start = vec.copy()
        mlp.train(s, epochs=epochs, batch=batch, lr=lr)
        got, grads = mlp.params(), mlp.grads()
        m, v, k = np.zeros(len(vec)), np.zeros(len(vec)), 0
        p = vec.astype(np.float64)
        for _ in range(epochs):
            for b in range(0, n, batch):
                k += 1
                _, G = mo.loss_and_grad(mo.unpack(p.astype(np.float32), T, C), s[b:b + batch], bf16=True)
                g = mo.pack(G, T, C).astype(np.float64)
                m = 0.9 * m + 0.1 * g
                v = 0.999 * v + 0.001 * g * g
                p -= lr * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
        d = np.abs(got - p)
        moved = np.abs(p - start) > 0
        assert d.max() <= 2 * k * lr and d[moved].mean() <= 0.1 * k * lr
        rows = mo.unpack(got, T, C)["E"], mo.unpack(start, T, C)["E"]
        assert np.array_equal(rows[0][T // 2:T], rows[1][T // 2:T])
        # the last batch's gradients stay readable
        assert np.linalg.norm(grads - g) <= 0.1 * np.linalg.norm(g)
    finally:
        mlp.close()


@pytest.mark.parametrize("order", ["up", "down", "equal", "steps", "wide"])
@pytest.mark.parametrize("T,C,n", [(9, 4, 3), (9, 127, 70), (9, 129, 64), (9, 700, 17), (9, 3001, 300)])
def test_predict_of_ordered_classes(gpu, T, C, n, order):
    """Logits that are the class biases alone (zero weights): every class better than all
    before it, none after the first four, all equal, equal in runs, and a spread whose
    exponentials over- and underflow.  Equal logits go to the lower class.  The logits
    are exact, and a sum of at most 3,001 exponentials in FP32, each within 2^-22, in
    chains of at most 400, is within 400 * 2^-24 + 2^-22 < 3e-5 of its value."""
    c = np.arange(C, dtype=np.float32)
    o = dict(up=c * 0.01, down=-c * 0.01, equal=0 * c + 0.25, steps=np.floor(c / 37) % 5, wide=((c * 89) % C) / C * 180 - 90)[order]
    mlp = gpu.mlp(T, C, seed=1)
    try:
        p = np.zeros_like(mlp.params())
        p[-C:] = o.astype(np.float32)
        mlp.set_params(p)
        top, prob = mlp.predict(_samples(np.random.default_rng(C), T, C, n))
        o = p[-C:].astype(np.float64)
        best = np.argsort(-o, kind="stable")[:4]
        assert np.array_equal(top, np.tile(best.astype(np.uint32), (n, 1)))
        e = np.exp(o - o.max())
        assert np.allclose(prob, np.tile((e / e.sum())[best], (n, 1)), rtol=3e-5, atol=1e-30)
    finally:
        mlp.close()


def _bias_network(gpu, T, o):
    """A network whose logits are exactly the class biases o."""
    mlp = gpu.mlp(T, len(o), seed=1)
    p = np.zeros_like(mlp.params())
    p[-len(o):] = o
    mlp.set_params(p)
    return mlp


def test_probability_of_a_confident_class(gpu):
    """One class far above those before it, which met a lower maximum: its exponential
    dominates the sum.  To the top probability's relative error the hardware's 2^x and
    the two expf that refer sums to another maximum add at most 2^-23 each, and seven
    roundings (of the corrected exponential, the reference changes, three merges and the
    division) 2^-24 each."""
    C, T, tol = 160, 4, 13 * 2.0 ** -24
    rng = np.random.default_rng(3)
    s = _samples(np.random.default_rng(5), T, C, 33)
    for d in np.linspace(0.5, 31.5, 125):
        o = np.sort(rng.uniform(-0.4, 0.0, C).astype(np.float32))[::-1].copy()
        at = int(rng.integers(64, C))
        o[at] = np.float32(d) + np.float32(rng.uniform(0, 0.25))
        mlp = _bias_network(gpu, T, o)
        try:
            top, prob = mlp.predict(s)
        finally:
            mlp.close()
        e = np.exp(o.astype(np.float64) - float(o.max()))
        want = 1.0 / e.sum()
        assert np.all(top[:, 0] == at)
        assert np.all(np.abs(prob[:, 0] - want) <= tol * want), (d, np.max(np.abs(prob[:, 0] / want - 1)))


@pytest.mark.parametrize("C,nan", [(200, slice(0, 40)), (20, slice(4, 8)), (700, slice(0, 4)), (700, slice(690, 700))])
def test_a_nan_logit_reaches_probabilities_and_loss(gpu, C, nan):
    """A NaN among the logits makes the sum of exponentials NaN, wherever it stands: also in
    the classes that a lane meets first, and beside the padding of a tile."""
    T, n = 4, 40
    o = np.random.default_rng(C).uniform(-1, 1, C).astype(np.float32)
    o[nan] = np.nan
    s = _samples(np.random.default_rng(6), T, C, n)
    s["target"] = 10 if C != 200 else 100
    mlp = _bias_network(gpu, T, o)
    try:
        top, prob = mlp.predict(s)
        assert not np.isin(top, np.arange(C)[nan]).any()
        assert np.isnan(prob).all()
        assert np.isnan(mlp.loss_grad(s))
    finally:
        mlp.close()
