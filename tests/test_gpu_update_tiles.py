"""The curved-space stage update on its tiles (64 x1 cells by 4 x3 rows, or 32 by 8)
against the CPU oracle: widths that leave part of a tile idle, row counts that are
no multiple of a tile's, every floor frame and both inverters.  One step from an
evolved state, with the bars of the torus step parity: 1e-12 relative L1, or 10
times what the oracle's own FMA-contracted build differs by (the inversion turns
last-bit differences of floor-density zones into velocity differences of that
size).  The timestep of the step's CFL estimate too, so that no tile's partial is
missing or stale.
"""
import numpy as np
import pytest

from kharma_amd import problems as pr
from tests.helpers import install_library_geometry, interior_of, rel_l1

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    import kharma_amd
    kharma_amd.lib()


KASTAUN = dict(inverter="kastaun", err_tol=1e-12, iter_max=25)
CASES = {
    "w70_rows9": lambda: pr.torus_config(70, 18, 9),
    "w40_rows13_normal": lambda: dict(pr.torus_config(40, 21, 13), floor_frame="normal"),
    "w96_rows10_fluid": lambda: dict(pr.torus_config(96, 16, 10), floor_frame="fluid"),
    "w65_rows8_kastaun": lambda: dict(pr.torus_config(65, 16, 8), **KASTAUN),
    "w33_rows11_kastaun_normal": lambda: dict(pr.torus_config(33, 17, 11), floor_frame="normal", **KASTAUN),
    "2d_kastaun_fluid": lambda: dict(pr.torus_config(67, 35, 1), floor_frame="fluid", **KASTAUN),
}


def _oracle(oracle_lib, cfg, variant=""):
    ob = oracle_lib.OracleBlock(cfg, variant=variant)
    install_library_geometry(ob, cfg)
    return ob


@pytest.mark.parametrize("case", list(CASES))
def test_update_tiles_match_the_oracle(oracle_lib, case):
    import kharma_amd as kh
    cfg = CASES[case]()
    ob = _oracle(oracle_lib, cfg)
    ob.init_state(pr.torus_prims(cfg))
    ob.step(2)
    P, U = ob.state()
    dt = ob.dt
    print(f"[update tiles] {case}", flush=True)
    drv = kh.Driver(cfg)
    drv.init_prims(torch.from_numpy(np.ascontiguousarray(P)).cuda())
    drv.set_clock(ob.time, dt, 2)
    drv.step(1)
    out = {}
    for variant in ("", "fma"):
        ref = _oracle(oracle_lib, cfg, variant=variant)
        ref.set_state(P, U)
        ref.dt = dt
        ref.step(1)
        out[variant] = ref.state() + (ref.dt,)
    Pg, Ug = (x.detach().cpu().numpy() for x in drv.state())
    for A, Ao, Af in ((Pg, out[""][0], out["fma"][0]), (Ug, out[""][1], out["fma"][1])):
        sens = rel_l1(interior_of(Af, cfg), interior_of(Ao, cfg))
        r = rel_l1(interior_of(A, cfg), interior_of(Ao, cfg))
        assert np.all(r < np.maximum(1e-12, 10 * sens)), (r, sens)
        ra = rel_l1(A, Ao)
        assert np.all(ra < np.maximum(1e-12, 10 * rel_l1(Af, Ao))), ra
    new_dt = drv.scalars()["dt"]
    assert abs(new_dt - out[""][2]) <= 1e-12 * out[""][2], (new_dt, out[""][2])
