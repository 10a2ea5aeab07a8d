"""The FP64 flux kernels whose lanes walk along the face normal, in every form that a
large 3-D block reaches them: each reconstruction, both Riemann fluxes, the smallest
ghost depth, contiguous containers and one pointer per variable (kh_get_flux_v, the
variables in allocations of their own).  Flat blocks from 917504 zones, the torus from
655360 (X1 faces from 1048576), ragged in every direction, against the CPU oracle
with the bars of the other flux comparisons: 1e-13 of the direction's largest flux
in flat space and 1e-12 on the torus.
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


# problem, zones, options, ghost depth, one pointer per variable
CASES = {
    "flat_weno5": ("mode", (101, 97, 99), dict(), 4, False),
    "flat_ppm_hlle_ng3": ("mode", (163, 75, 77), dict(recon="ppm", riemann="hlle"), 3, False),
    "flat_mc_vars": ("mode", (99, 98, 97), dict(recon="linear_mc"), 4, True),
    "flat_donor": ("mode", (131, 70, 102), dict(recon="donor_cell_c"), 4, False),
    "torus_mc_x2_x3": ("torus", (101, 86, 79), dict(recon="linear_mc"), 4, False),
    "torus_mc_vars": ("torus", (149, 89, 86), dict(recon="linear_mc"), 4, True),
    "torus_donor_hlle": ("torus", (139, 91, 84), dict(recon="donor_cell_c", riemann="hlle"), 4, False),
    "torus_ppm_ng3": ("torus", (121, 101, 90), dict(recon="ppm"), 3, True),
}


@pytest.mark.parametrize("case", list(CASES))
def test_marching_forms_match_the_oracle(oracle_lib, case):
    import kharma_amd as kh
    problem, n, kw, ng, per_var = CASES[case]
    if problem == "mode":
        ocfg = dict(pr.mhdmode_config(n=n[0], mode="fast", one_period=False), nx=n, **kw)
        P = pr.mhdmode_prims(ocfg)
        rng = np.random.default_rng(17)   # waves in every variable, so that no state or flux is uniform
        P = P * (1 + 1e-2 * pr.periodic_fill(rng.uniform(-1, 1, P.shape), ocfg))
    else:
        ocfg = dict(pr.torus_config(*n), **kw)
        P = pr.torus_prims(ocfg)
    ob = oracle_lib.OracleBlock(ocfg)
    if problem == "torus":
        install_library_geometry(ob, ocfg)
    ob.init_state(P)
    P, _ = ob.state()
    cut = ocfg.get("ng", 4) - ng          # the oracle's faces reach one further: it keeps four ghosts
    cfg = dict(ocfg, ng=ng)
    if cut:
        P = P[:, cut:-cut, cut:-cut, cut:-cut]
    print(f"[march forms] {case}", flush=True)
    blk = kh.Block(cfg)
    F, cmax, cmin = blk.new_fluxes()
    Pg = torch.from_numpy(np.ascontiguousarray(P)).cuda()
    Pv, Fv = [p.clone() for p in Pg], [[f.clone() for f in Fd] for Fd in F]
    for d in (1, 2, 3):
        if per_var:
            blk.get_flux_v(d, Pv, Fv[d - 1], cmax[d - 1], cmin[d - 1])
        else:
            blk.get_flux(d, Pg, F, cmax, cmin)
        ob.get_flux(d)
    torch.cuda.synchronize()
    Fo, omax, omin = ob.array(0), ob.array(1), ob.array(2)
    bar = 1e-12 if problem == "torus" else 1e-13
    for d in (1, 2, 3):
        sl, so = face_slices(cfg, d), face_slices(ocfg, d)
        Fg = (torch.stack(Fv[d - 1]) if per_var else F[d - 1]).cpu().numpy()
        ref = Fo[d - 1][(slice(None),) + so]
        assert np.abs(Fg[(slice(None),) + sl] - ref).max() <= bar * np.abs(ref).max(), (case, d)
        for g, o in ((cmax, omax), (cmin, omin)):
            o = o[d - 1][so]
            assert np.abs(g[d - 1].cpu().numpy()[sl] - o).max() <= bar * np.abs(o).max(), (case, d)
        mask = np.ones(Fg.shape[1:], dtype=bool)   # nothing is written outside the faces a step consumes
        mask[sl] = False
        assert not Fg[:, mask].any(), (case, d)
