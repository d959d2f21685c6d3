"""The scan by cells (IVP_OPT_BUILD_LANES 64) and the four-lane exact pass where their rules change
over: particles outside the grid (clamped into its border cells, coordinates far from a segment's
centre), positions that are not finite, rows of cells with gaps along x, counts around a wave's
16 rows and a tile's 64, and row capacities that are not a multiple of 8.  Rows, density and k must
be bitwise those of the one-lane build."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

H = np.float32(0.04)


def _cloud(n, seed, spread):
    rng = np.random.default_rng(seed)
    x = (0.4 + spread * rng.random((n, 3))).astype(np.float32)
    dyn = (rng.random(n) < 0.8).astype(np.int32)
    dyn[:max(1, n // 2)] = 1
    return x, dyn


def _case(name):
    if name.startswith("count"):
        n = int(name[5:])
        x, _ = _cloud(n, n, 0.02 * max(1.0, n ** (1 / 3)))
        return x, np.ones(n, np.int32), 60
    x, dyn = _cloud(3000, 7, 0.3)
    if name == "outside":       # a group far below the domain and one far above, beside the cloud
        x[:400] = x[:400] - np.float32(3.0)
        x[400:700] += np.float32(5.0)
        x[700:900, 0] -= np.float32(40.0)
        return x, dyn, 61
    if name == "not_finite":
        x[5] = np.nan
        x[17, 1] = np.inf
        x[40, 2] = -np.inf
        x[2999] = np.nan
        return x, dyn, 60
    assert name == "gaps"       # clumps along x, one (y, z) row of cells
    q = np.repeat(np.arange(60, dtype=np.float32), 50)
    x[:, 0] = 0.1 + q * np.float32(0.031) + x[:, 0] * np.float32(0.05)
    x[:, 1:] = 0.4 + (x[:, 1:] - 0.4) * np.float32(0.1)
    return x, dyn, 200


@pytest.mark.parametrize("name", ["count1", "count15", "count16", "count17", "count63", "count65", "count129", "outside",
                                  "not_finite", "gaps"])
@pytest.mark.parametrize("rows", [0, 2], ids=["ids_only", "gradW_f16"])
def test_scan_by_cells_matches_one_lane(name, rows):
    from implicitvelocityprojection_amd import _native as N
    from implicitvelocityprojection_amd.context import Context
    x, dyn, C = _case(name)
    n = len(x)
    t = lambda a, dt=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt)
    m = np.full(n, 0.0064, np.float32)
    minv = np.where(dyn == 1, np.float32(1) / m, np.float32(0)).astype(np.float32)
    ctx = Context(H, [0.0, 0.0, 0.0], [2.4, 1.2, 1.2], n, cache_size=C)
    ctx.gradient_cache = rows
    ctx.set_particles(t(x), t(np.zeros((n, 3), np.float32)), t(m), t(minv), t(np.full(n, 1000.0, np.float32)),
                      t(dyn, torch.int32), t(dyn, torch.int32))
    got = {}
    for lanes in (1, 16, 64, 0):
        print(f"{name}: lanes {lanes}", flush=True)
        ctx.build_lanes = lanes
        assert ctx.neighbors_build() == N.IVP_OK
        rho = ctx.read(N.FIELD_DENSITY, torch.zeros(n, device="cuda")).cpu().numpy()
        k = ctx.read(N.FIELD_K, torch.zeros(n, device="cuda")).cpu().numpy()
        got[lanes] = (rho.view(np.uint32), k.view(np.uint32), ctx.pair_count())
        # the rows themselves, through a pass that walks them
        ctx.write(N.FIELD_V, t(np.nan_to_num(x, posinf=0.0, neginf=0.0)))
        ctx.viscosity_explicit(0.01, 1e-3)
        v = ctx.read(N.FIELD_V, torch.zeros((n, 3), device="cuda")).cpu().numpy()
        got[lanes] += (v.view(np.uint32),)
    for lanes in (16, 64, 0):
        for a, b in zip(got[1], got[lanes]):
            assert np.array_equal(a, b), (name, lanes)
    ctx.close()
