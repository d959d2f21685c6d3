"""The scan by cells on rows whose coordinates are far from their cells: a lattice of spacing h/2 (pairs
within float32 rounding of h, decided by the correctly rounded root) wholly or partly outside the grid,
so that its border cells hold hundreds of candidates, dynamic and static, in counts that fill a batch, a
quarter and a chunk or leave them ragged.  Rows, density and k must be bitwise those of the one-lane build."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

H = np.float32(0.04)


@pytest.mark.parametrize("n", [17, 64, 255, 256, 257, 700])
@pytest.mark.parametrize("shift", [0.3, -1.0, 9.0], ids=["across", "below", "above"])
def test_far_rows_match_one_lane(n, shift):
    from implicitvelocityprojection_amd import _native as N
    from implicitvelocityprojection_amd.context import Context
    g = np.arange(10, dtype=np.float32) * (H / np.float32(2))
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)[:n].astype(np.float32)
    # "across": the block straddles the lower border cells; the others lie outside the grid as a whole
    x[:, 0] += np.float32(shift if shift != 0.3 else -0.15)
    x[:, 1:] += np.float32(0.3)
    dyn = (np.arange(n) % 4 != 3).astype(np.int32)
    m = np.full(n, 0.0064, np.float32)
    minv = np.where(dyn == 1, np.float32(1) / m, np.float32(0)).astype(np.float32)
    t = lambda a, dt=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt)
    ctx = Context(H, [0.0, 0.0, 0.0], [1.2, 1.2, 1.2], n, cache_size=60)
    ctx.set_particles(t(x), t(np.zeros((n, 3), np.float32)), t(m), t(minv), t(np.full(n, 1000.0, np.float32)),
                      t(dyn, torch.int32), t(dyn, torch.int32))
    got = {}
    for lanes in (1, 64):
        print(f"n {n} shift {shift} lanes {lanes}", flush=True)
        ctx.build_lanes = lanes
        assert ctx.neighbors_build() == N.IVP_OK
        count = torch.zeros(n, dtype=torch.int32, device="cuda")
        ids = torch.zeros(n * 60, dtype=torch.int32, device="cuda")
        gradW = torch.zeros(n * 180, dtype=torch.float32, device="cuda")
        ctx.neighbors_export(count, ids, gradW)
        c = count.cpu().numpy()
        used = (np.arange(60)[None, :] < c[:, None]).reshape(-1)
        rho = ctx.read(N.FIELD_DENSITY, torch.zeros(n, device="cuda")).cpu().numpy()
        k = ctx.read(N.FIELD_K, torch.zeros(n, device="cuda")).cpu().numpy()
        got[lanes] = (c, ids.cpu().numpy()[used], rho.view(np.uint32), k.view(np.uint32))
    ctx.close()
    assert got[1][0].max() >= 3
    for a, b in zip(got[1], got[64]):
        assert np.array_equal(a, b)
