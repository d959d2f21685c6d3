"""The counting sort's cell table: one launch for up to 4096 chunks of 2048 cells, three beyond
(about 8.4M cells).  The same particles in a small and in a large domain -- their cells differ, their
neighbours do not -- must take the same steps bitwise, statics and a ragged count included."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

H = np.float32(0.04)


def _run(side, x, v, dyn, steps):
    from implicitvelocityprojection_amd import _native as N
    from implicitvelocityprojection_amd.context import Context, IPParams
    n = len(x)
    t = lambda a, dt=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt)
    m = np.full(n, 0.0064, np.float32)
    minv = np.where(dyn == 1, np.float32(1) / m, np.float32(0)).astype(np.float32)
    # the lower corner clamps at the support radius in both; the upper one is out of reach
    ctx = Context(H, [0.0, 0.0, 0.0], [side, side, side], n, cache_size=80)
    ctx.set_particles(t(x), t(v), t(m), t(minv), t(np.full(n, 1000.0, np.float32)), t(dyn, torch.int32),
                      t(dyn, torch.int32))
    assert ctx.neighbors_build() == N.IVP_OK
    for _ in range(steps):
        res, _ = ctx.step(1e-3, (0.0, -9.81, 0.0), 0, 0.01, IPParams(tol_opt=1e-3, max_iteration_opt=100))
        assert res.status == 0
    out = [ctx.read(f, torch.zeros(s, device="cuda")).cpu().numpy().view(np.uint32)
           for f, s in ((N.FIELD_X, (n, 3)), (N.FIELD_V, (n, 3)), (N.FIELD_DENSITY, n), (N.FIELD_K, n))]
    ctx.close()
    return out


@pytest.mark.parametrize("side", [7.9, 8.6])     # about 4020 and 5100 chunks of cells
def test_large_cell_tables(side):
    rng = np.random.default_rng(3)
    g = np.stack(np.meshgrid(*[np.arange(k, dtype=np.float64) for k in (17, 15, 13)], indexing="ij"), -1).reshape(-1, 3)
    x = (0.1 + 0.0195 * g + 0.001 * rng.random(g.shape)).astype(np.float32)
    dyn = (g[:, 1] >= 2).astype(np.int32)
    v = np.where(dyn[:, None] == 1, 0.05 * rng.standard_normal(x.shape), 0.0).astype(np.float32)
    chunks = (int(np.ceil(side / (0.04 * 1.0009765625))) + 4) ** 3 / 2048
    assert (chunks <= 4096) == (side == 7.9)
    for a, b in zip(_run(1.0, x, v, dyn, 2), _run(side, x, v, dyn, 2)):
        assert np.array_equal(a, b)
