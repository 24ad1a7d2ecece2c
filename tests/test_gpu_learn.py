"""Learned initial guess: BF16-MFMA MLP kernels against the NumPy oracle, and
the POD + MLP guess against the zero guess on a family of elasticity cells.

Parity bar for the network: forward outputs, loss and every gradient match
the oracle evaluated with the same BF16 rounding of the matrix-product
operands (float64 elsewhere) to 1e-3 relative in norm -- the remaining
difference is the FP32 accumulation and tanhf of the device. The oracle's
own backward pass is pinned by finite differences in test_oracle.py.
"""

import numpy as np
import pytest

import mlp_oracle as M

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30)


@pytest.fixture(scope="module")
def net(B):
    nin, nh, nout = 4, 64, 40
    m = B.Mlp(nin, nh, nout, seed=3)
    rng = np.random.default_rng(7)
    _, npar = M.layout(nin, nh, nout)
    p = rng.normal(0, 0.3, npar).astype(np.float32)
    m.set_params(p)
    return m, p.astype(np.float64), (nin, nh, nout)


@pytest.mark.parametrize("batch", [1, 37, 256])
def test_mlp_forward_matches_oracle(B, ctx, net, batch):
    m, p, dims = net
    x = np.random.default_rng(batch).normal(size=(batch, dims[0])).astype(np.float32)
    y = m.forward(ctx, x)
    yo, _ = M.forward(p, x.astype(np.float64), *dims, bf16=True)
    assert relerr(y, yo) < 1e-3


def test_mlp_gradients_match_oracle(B, ctx, net):
    m, p, dims = net
    rng = np.random.default_rng(11)
    x = rng.normal(size=(83, dims[0])).astype(np.float32)
    t = rng.normal(size=(83, dims[2])).astype(np.float32)
    loss = m.backward(ctx, x, t)
    lo, go = M.loss_grad(p, x.astype(np.float64), t.astype(np.float64), *dims, bf16=True)
    g = m.grads().astype(np.float64)
    assert abs(loss - lo) <= 1e-4 * lo
    offs, _ = M.layout(*dims)
    for name, (o, shp) in zip(["W1", "b1", "W2", "b2", "W3", "b3"], offs):
        k = int(np.prod(shp))
        assert relerr(g[o:o + k], go[o:o + k]) < 1e-3, name


def test_mlp_adam_matches_oracle_and_learns(B, ctx):
    nin, nh, nout = 4, 32, 8
    m = B.Mlp(nin, nh, nout, seed=5)
    p0 = m.params().astype(np.float64)
    rng = np.random.default_rng(2)
    x = rng.uniform(-1, 1, size=(128, nin)).astype(np.float32)
    t = np.stack([np.sin(x[:, 0] + k * x[:, 1]) * np.cos(x[:, 2] - x[:, 3] * k / 3) for k in range(nout)],
                 axis=1).astype(np.float32)
    m.backward(ctx, x, t)
    g = m.grads().astype(np.float64)
    m.adam_step(ctx, 1e-2)
    pn, _, _ = M.adam(p0, g, np.zeros_like(p0), np.zeros_like(p0), 1, 1e-2)
    assert relerr(m.params(), pn) < 1e-6
    first = m.backward(ctx, x, t)
    for _ in range(400):
        m.backward(ctx, x, t)
        m.adam_step(ctx, 3e-3)
    last = m.backward(ctx, x, t)
    print(f"mlp loss {first:.4f} -> {last:.5f}", flush=True)
    assert last < 0.1 * first


def test_learned_guess_beats_zero_guess(B, ctx):
    """A small family of 4^3 elasticity cells: the POD + MLP guess trained on
    solved cells lowers the PCG iteration count of unseen cells."""
    mgrid, ntrain, ntest = 4, 48, 8
    rng = np.random.default_rng(20261205)

    def draw(k):
        return np.stack([rng.uniform(0.1, 0.45, k), rng.uniform(0, 3, k), rng.uniform(0.2, 0.45, k),
                         rng.uniform(-0.15, 0.15, k)], axis=1)

    def cells(prm):
        out = []
        order = None
        for r, lc, nu, sh in prm:
            mat, rhs = B.gen_elastic_cell(mgrid, r, 10 ** lc, nu, sh, 20261205)
            order = mat.rcm_order() if order is None else order  # one template: one ordering
            mo = mat.reorder(order)
            out.append((mo, B.Factor.ic2(mo, B.default_params(tau1=0.1, tau2=0.01)), mo.reorder_vector(order, rhs)))
        return out

    def solve(cs, x0=None, fallback=False):
        bt = B.Batch([(mo, f) for mo, f, _ in cs], prec_mask=0b010)
        b = bt.gather([c[2] for c in cs])
        db = B.DeviceArray.from_host(b)
        dx = B.DeviceArray.from_host(x0) if x0 is not None else B.DeviceArray(b.shape)
        if x0 is None:
            dx.zero()
        st, its, rr = bt.solve(ctx, db, dx, B.default_opts(kind=B.BLOCKPCG, eps=1e-10, precision=B.F32), 6,
                               fallback)
        assert st.converged == st.pairs
        return dx, its

    ptrain, ptest = draw(ntrain), draw(ntest)
    train = cells(ptrain)
    n = train[0][0].n
    g = B.Guess(n, 6, 4, nmodes=16, nhidden=64, capacity=ntrain, seed=9)
    for k0 in range(0, ntrain, 16):
        dx, _ = solve(train[k0:k0 + 16])
        g.add(ctx, ptrain[k0:k0 + 16], dx)
    rep = g.fit(ctx, steps=1500, lr=3e-3)
    print(f"guess fit: modes {rep.modes} energy {rep.pod_energy:.6f} loss {rep.loss_first:.3e} -> "
          f"{rep.loss_final:.3e}", flush=True)
    assert rep.pod_energy > 0.9 and rep.loss_final < 0.2 * rep.loss_first
    test = cells(ptest)
    dx0, its0 = solve(test)
    x0 = B.DeviceArray((n * ntest, 6))
    g.predict(ctx, ptest, x0)
    guess = x0.host()
    exact = dx0.host()
    err = np.linalg.norm(guess - exact) / np.linalg.norm(exact)
    _, its1 = solve(test, x0=guess, fallback=True)
    print(f"guess rel err {err:.3e}; iterations zero {its0.mean():.1f} learned {its1.mean():.1f}", flush=True)
    assert err < 0.3
    assert its1.mean() < its0.mean()


# Fused kernels: sizes around the 16-column and 32-step tiles, batches around
# the 16- and 32-row ones; the last two networks take the separate products.
@pytest.mark.parametrize("dims,batch", [((1, 1, 1), 1), ((4, 16, 16), 16), ((5, 17, 33), 31), ((33, 200, 47), 33),
                                        ((4, 256, 384), 1024), ((2, 31, 500), 100), ((8, 300, 40), 77),
                                        ((200, 64, 700), 65)])
def test_mlp_sizes_match_oracle(B, ctx, dims, batch):
    print(f"mlp {dims} batch {batch}", flush=True)
    m = B.Mlp(*dims, seed=9)
    rng = np.random.default_rng(sum(dims) + batch)
    offs, npar = M.layout(*dims)
    p = (rng.normal(size=npar) / np.sqrt(max(dims[1], dims[0]))).astype(np.float32)
    m.set_params(p)
    x = rng.normal(size=(batch, dims[0])).astype(np.float32)
    t = rng.normal(size=(batch, dims[2])).astype(np.float32)
    yo, _ = M.forward(p.astype(np.float64), x.astype(np.float64), *dims, bf16=True)
    # operands that round to the other BF16 neighbour after FP32 sums: 2^-9 each, over the few that are that close
    assert relerr(m.forward(ctx, x), yo) < 1e-3
    for _ in range(2):  # the second pass over the same buffers
        loss = m.backward(ctx, x, t)
        lo, go = M.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *dims, bf16=True)
        g = m.grads().astype(np.float64)
        assert abs(loss - lo) <= 1e-4 * lo
        for name, (o, shp) in zip(["W1", "b1", "W2", "b2", "W3", "b3"], offs):
            k = int(np.prod(shp))
            assert relerr(g[o:o + k], go[o:o + k]) < 2e-3, name
    p0, zero = m.params().astype(np.float64), np.zeros(npar)
    m.adam_step(ctx, 1e-2)
    pn, _, _ = M.adam(p0, g, zero, zero, 1, 1e-2)
    assert relerr(m.params(), pn) < 1e-6
    y1, _ = M.forward(m.params().astype(np.float64), x.astype(np.float64), *dims, bf16=True)
    assert relerr(m.forward(ctx, x), y1) < 1e-3  # the packed weights follow the update


# One buffer for input and output: the output starts where the input does, or
# inside it; rows of the output wider, narrower and as wide as the input's.
@pytest.mark.parametrize("dims,shift", [((4, 16, 8), 0), ((8, 16, 4), 0), ((6, 16, 6), 0), ((6, 16, 6), 3),
                                        ((4, 16, 8), 1000), ((200, 64, 700), 0)])
def test_mlp_forward_overlapping_buffers(B, ctx, dims, shift):
    nin, _, nout = dims
    batch = 20000 if nin < 10 else 500
    print(f"mlp {dims} one buffer, output {shift} floats behind the input", flush=True)
    m = B.Mlp(*dims, seed=4)
    x = np.random.default_rng(3).normal(size=(batch, nin)).astype(np.float32)
    want = m.forward(ctx, x)
    buf = np.zeros(shift + batch * max(nin, nout), np.float32)
    buf[:x.size] = x.ravel()
    d = B.DeviceArray.from_host(buf)
    B._check(B.lib().bcm_mlp_forward(ctx.h, m.h, batch, B.ptr(d), B.ptr(d) + 4 * shift))
    ctx.sync()
    assert np.array_equal(d.host()[shift:shift + batch * nout].reshape(batch, nout), want)


# An infinite weight saturates one unit. Rows past the batch, which fill up the
# last tile of rows, add nothing to any gradient then either.
@pytest.mark.parametrize("layer", [0, 2])
@pytest.mark.parametrize("batch", [17, 33, 64])
def test_mlp_infinite_weight(B, ctx, layer, batch):
    dims = (5, 20, 33)
    rng = np.random.default_rng(layer + batch)
    offs, npar = M.layout(*dims)
    p = rng.normal(0, 0.3, npar).astype(np.float32)
    p[offs[layer][0]] = np.inf
    x = rng.normal(size=(batch, dims[0])).astype(np.float32)
    t = rng.normal(size=(batch, dims[2])).astype(np.float32)
    print(f"mlp infinite weight layer {layer // 2 + 1} batch {batch}", flush=True)
    m = B.Mlp(*dims, seed=2)
    m.set_params(p)
    loss = m.backward(ctx, x, t)
    with np.errstate(invalid="ignore"):
        lo, go = M.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *dims, bf16=True)
    g = m.grads().astype(np.float64)
    assert abs(loss - lo) <= 1e-4 * lo
    assert np.array_equal(np.isfinite(g), np.isfinite(go))
    assert relerr(g[np.isfinite(go)], go[np.isfinite(go)]) < 2e-3  # as the gradients of finite weights


def test_mlp_more_rows_than_a_launch(B, ctx):
    """70 million rows: at 16 rows for 1024 threads more than one launch takes."""
    rows, dims = 70000000, (1, 250, 1)
    print(f"mlp {dims} rows {rows}", flush=True)
    m = B.Mlp(*dims, seed=6)
    part = np.random.default_rng(1).normal(size=(1000003, 1)).astype(np.float32)
    x = np.tile(part, (rows // len(part) + 1, 1))[:rows]
    want = m.forward(ctx, part)
    y = m.forward(ctx, x)
    for k in range(0, rows, len(part)):  # a row's result does not depend on where it stands
        assert np.array_equal(y[k:k + len(part)], want[:min(len(part), rows - k)]), k


def test_mlp_gradients_of_long_batches(B, ctx):
    """262144 rows: sums of a batch in FP32 from end to end would be off by some
    5e-7. Biases: 16 rows in FP32, then FP64, a few 2^-24. Weights: 32 steps of 32
    rows, then 64 such sums, each a random walk of 2^-25; what layers 1 and 2 add
    to it are gradients that round to the other BF16 neighbour."""
    dims, batch = (4, 16, 16), 262144
    rng = np.random.default_rng(3)
    offs, npar = M.layout(*dims)
    p = (rng.normal(size=npar) / 4.0).astype(np.float32)
    x = rng.normal(size=(batch, dims[0])).astype(np.float32)
    t = (rng.normal(size=(batch, dims[2])) + 0.3).astype(np.float32)
    print(f"mlp {dims} batch {batch}", flush=True)
    m = B.Mlp(*dims)
    m.set_params(p)
    m.backward(ctx, x, t)
    g = m.grads().astype(np.float64)
    _, go = M.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), *dims, bf16=True)
    for name, (o, shp), tol in zip(["W1", "b1", "W2", "b2", "W3", "b3"], offs, [1e-6, 2e-7, 5e-7, 2e-7, 4e-7, 2e-7]):
        k = int(np.prod(shp))
        e = relerr(g[o:o + k], go[o:o + k])
        print(f"{name} {e:.1e}", flush=True)
        assert e < tol, name
