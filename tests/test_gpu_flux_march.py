"""The FP64 flux kernels of large 3-D blocks (lanes walking along the face normal,
along x3 for X1 faces) against the CPU oracle, at sizes just above the ones they
start from and ragged in every direction: column counts that leave part of a
wavefront, a chunk of faces that ends short, the smallest ghost depth.  Bars: those
of the other flux comparisons with the oracle, 1e-13 of the direction's largest
flux in flat space and 1e-12 on the torus.
"""
import numpy as np
import pytest

from kharma_amd import problems as pr
from tests.helpers import face_slices, install_library_geometry

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a HIP device")
    import kharma_amd
    kharma_amd.lib()


def _mode(n, **kw):
    cfg = pr.mhdmode_config(n=n[0], mode="fast", one_period=False, **kw)
    cfg["nx"] = n
    return cfg, pr.mhdmode_prims(cfg)


def _torus(n, **kw):
    cfg = dict(pr.torus_config(*n), **kw)
    return cfg, None


CASES = {
    "mode_weno5": lambda: _mode((81, 83, 79)),
    "mode_hlle_ppm_ng3": lambda: _mode((127, 65, 66), riemann="hlle", recon="ppm"),
    "torus_x2_x3": lambda: _torus((97, 74, 73)),
    "torus_x1": lambda: _torus((145, 89, 86)),
    "torus_x1_ng3": lambda: _torus((121, 101, 90)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_marching_fluxes_match_the_oracle(oracle_lib, case):
    import kharma_amd as kh
    cfg, P = CASES[case]()
    ob = oracle_lib.OracleBlock(cfg)
    if P is None:
        install_library_geometry(ob, cfg)
        P = pr.torus_prims(cfg)
    else:   # waves in every variable, so that no state or flux is uniform
        rng = np.random.default_rng(3)
        P = P * (1 + 1e-2 * pr.periodic_fill(rng.uniform(-1, 1, P.shape), cfg))
    ob.init_state(P)
    P, _ = ob.state()
    ocfg = cfg
    if case.endswith("ng3"):   # the oracle's faces reach one further and keep four ghosts
        cfg = dict(cfg, ng=3)
        P = P[:, 1:-1, 1:-1, 1:-1]
    blk = kh.Block(cfg)
    F, cmax, cmin = blk.new_fluxes()
    Pg = torch.from_numpy(np.ascontiguousarray(P)).cuda()
    bar = 1e-12 if cfg.get("coords") == "ks" else 1e-13
    for d in (1, 2, 3):
        blk.get_flux(d, Pg, F, cmax, cmin)
        ob.get_flux(d)
    torch.cuda.synchronize()
    Fo_all, speeds = ob.array(0), ((cmax.cpu().numpy(), ob.array(1)), (cmin.cpu().numpy(), ob.array(2)))
    for d in (1, 2, 3):
        sl, so = face_slices(cfg, d), face_slices(ocfg, d)
        Fo = Fo_all[d - 1][(slice(None),) + so]
        Fg = F[d - 1].cpu().numpy()
        err = np.abs(Fg[(slice(None),) + sl] - Fo).max()
        assert err <= bar * np.abs(Fo).max(), (case, d, err)
        for g, o in speeds:
            assert np.abs(g[d - 1][sl] - o[d - 1][so]).max() <= bar * np.abs(o[d - 1][so]).max(), (case, d)
        # nothing is written outside the faces the step consumes
        mask = np.ones(Fg.shape[1:], dtype=bool)
        mask[sl] = False
        assert not Fg[:, mask].any(), (case, d)
