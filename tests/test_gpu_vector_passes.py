"""The CG's vector passes change their blocks with the row count (256 threads of one row; 1024 threads of one
to four rows; 256 threads again): the implicit viscosity solve on both sides of each line against the
same solve in float64.  Bar: 1e-5 relative (max norm), the repository's for a solve's velocities -- both stop at
r.r < 1e-5 and the float32 iterate differs by rounding alone."""

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(53, 50, 49), (64, 64, 32), (64, 64, 64), (65, 64, 64), (82, 80, 80), (93, 92, 92),
                                      (103, 102, 101)])
def test_viscosity_solve_at_the_block_lines(nx, ny, nz):
    from perf import cases
    case = dict(kind="w18", nx=nx, ny=ny, nz=nz, dam=True, coeff=0.1)
    s = cases.prepare(case, 5)
    v = cases.run(s)["v"].double()
    ref = cases.exact(case, 5)["v"]
    s["ctx"].close()
    err = float((v - ref).abs().max() / ref.abs().max())
    print(f"{nx * ny * nz} rows: {err:.2e}", flush=True)
    assert err <= 1e-5
