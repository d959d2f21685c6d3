"""The exact build pass that also finds the tile windows (rows of at most 64 slots): against the build
whose windows come from a pass of their own (one lane per row; rows of more than 64 slots) and against
the build without windows, at the edges of a tile's rows, of a row's slots and of the window cap."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

H = np.float32(0.04)


def _build(n, C, rows, lanes, windows):
    from implicitvelocityprojection_amd import _native as N
    from implicitvelocityprojection_amd.context import Context
    rng = np.random.default_rng(n)
    # about 15 neighbours per particle; a fifth of the particles are walls
    x = (0.3 + 0.026 * n ** (1 / 3) * rng.random((n, 3))).astype(np.float32)
    dyn = (np.arange(n) % 5 != 4).astype(np.int32)
    m = np.full(n, 0.0064, np.float32)
    minv = np.where(dyn == 1, np.float32(1) / m, np.float32(0)).astype(np.float32)
    t = lambda a, dt=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt)
    ctx = Context(H, [0.0, 0.0, 0.0], [2.0, 2.0, 2.0], n, cache_size=C)
    ctx.gradient_cache = rows
    ctx.build_lanes = lanes
    N.check(ctx.lib.ivp_set_option(ctx.h, N.OPT_TILE_WINDOWS, windows), "ivp_set_option")
    ctx.set_particles(t(x), t(np.zeros((n, 3), np.float32)), t(m), t(minv), t(np.full(n, 1000.0, np.float32)),
                      t(dyn, torch.int32), t(dyn, torch.int32))
    assert ctx.neighbors_build() == N.IVP_OK
    rho = ctx.read(N.FIELD_DENSITY, torch.zeros(n, device="cuda")).cpu().numpy()
    k = ctx.read(N.FIELD_K, torch.zeros(n, device="cuda")).cpu().numpy()
    stats = ctx.window_stats()
    ctx.write(N.FIELD_V, t(x))
    ctx.viscosity_weiler18(0.05, 1e-3)
    v = ctx.read(N.FIELD_V, torch.zeros((n, 3), device="cuda")).cpu().numpy()
    ctx.close()
    return stats, (rho.view(np.uint32), k.view(np.uint32), v.view(np.uint32))


@pytest.mark.parametrize("n", [1, 2, 79, 80, 81, 1283, 4000])
@pytest.mark.parametrize("C,rows,cap", [(57, 0, 1), (64, 0, 1), (64, 2, 1), (65, 0, 1), (64, 0, 260)])
def test_window_search_in_the_exact_pass(n, C, rows, cap):
    stats, got = _build(n, C, rows, 16, cap)
    ref_stats, ref = _build(n, C, rows, 1, cap)
    _, off = _build(n, C, rows, 16, 0)
    assert stats == ref_stats
    if cap == 1:
        assert stats[1] == stats[0], stats
    for a, b, c in zip(got, ref, off):
        assert np.array_equal(a, b) and np.array_equal(a, c)


def test_scene_windows_bitwise():
    """Independent scenes with four lanes per row: tiles that span two scenes, with and without windows."""
    from implicitvelocityprojection_amd import _native as N
    from implicitvelocityprojection_amd.scene_batch import SceneBatch
    from implicitvelocityprojection_amd.scenes import synthetic_batch
    out = []
    for windows in (1, 300, 0):
        b = SceneBatch(synthetic_batch(5, seed=3, count_range=(300, 2500)), chunk=2, lanes=4)
        N.check(b.ctx.lib.ivp_set_option(b.ctx.h, N.OPT_TILE_WINDOWS, windows), "ivp_set_option")
        assert b.ctx.neighbors_build() == N.IVP_OK
        tiles, windowed, _ = b.ctx.window_stats()
        assert (windowed == 0) == (windows == 0) and windowed <= tiles
        for _ in range(3):
            b.step()
        f = {N.FIELD_X: (b.n, 3), N.FIELD_V: (b.n, 3), N.FIELD_DENSITY: (b.n,), N.FIELD_DIVERGENCE: (b.n,)}
        out.append([b.ctx.read(k, torch.zeros(s, device="cuda")).cpu().numpy().view(np.uint32) for k, s in f.items()])
        b.close()
    for got in out[:2]:
        for x, y in zip(got, out[2]):
            assert np.array_equal(x, y)
