"""Results do not depend on how a mesh is laid out or launched, also where the flux
kernels change with the size: as one block, as blocks in one launch and as blocks
launched one by one, and with the kernels timed (a launch a direction), equal bit
for bit, timesteps included.

FP64 3-D meshes on either side of the size from which the lanes walk along the face
normal: the two forms round differently, so the one that a mesh takes has to follow
from the whole mesh.  The sizes put one block and its split (whose blocks add ghost
zones of their own), or one launch over all blocks and one per block, on two sides
of a rule that counts a launch's faces ("deep" has more X3 faces than X2 faces), and
on both sides of one that counts the mesh's zones.
"""
import numpy as np
import pytest

from kharma_amd import problems as pr

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
    cfg["dt_start"] = 0.2 / max(n)
    rng = np.random.default_rng(11)
    P = pr.mhdmode_prims(cfg)
    return cfg, P * (1 + 1e-2 * pr.periodic_fill(rng.uniform(-1, 1, P.shape), cfg))


def _torus(n, **kw):
    cfg = dict(pr.torus_config(*n), **kw)
    return cfg, pr.torus_prims(cfg)


CASES = {
    "flat_78": (lambda: _mode((78, 78, 78)), (2, 2, 2)),
    "flat_deep": (lambda: _mode((80, 40, 153)), (1, 2, 1)),
    "flat_90_mc": (lambda: _mode((90, 78, 84), recon="linear_mc"), (1, 2, 2)),
    "torus_x2_x3": (lambda: _torus((96, 80, 64)), (2, 2, 4)),
    "flat_march": (lambda: _mode((100, 98, 96)), (2, 2, 2)),
    "flat_march_ppm_hlle": (lambda: _mode((100, 98, 96), recon="ppm", riemann="hlle"), (1, 1, 4)),
    "torus_x1": (lambda: _torus((136, 88, 80)), (2, 2, 4)),
    "torus_march": (lambda: _torus((152, 92, 80)), (2, 2, 4)),
    "torus_march_mc": (lambda: _torus((152, 92, 80), recon="linear_mc"), (2, 2, 1)),
}
STEPS = 2


def _state(d):
    P, U = d.state()
    torch.cuda.synchronize()
    return P.cpu(), U.cpu(), d.dt_history(STEPS), d.scalars()["dt"]


def _run(kind, cfg, P, nb):
    import kharma_amd as kh
    d = kh.Driver(cfg) if kind in ("block", "timed") else kh.Mesh(cfg, nb)
    if kind == "timed":
        d.set_kernel_timing(True)
    if kind == "per block":
        d.set_packed(False)
    d.init_prims(torch.from_numpy(np.ascontiguousarray(P)).cuda())
    d.step(STEPS)
    return _state(d)


def _same_by_every_route(case, cfg, P, nb):
    ref = _run("block", cfg, P, nb)
    for kind in ("timed", "packed", "per block"):
        print(f"[mesh routes] {case} {kind}", flush=True)
        out = _run(kind, cfg, P, nb)
        assert out[2] == ref[2] and out[3] == ref[3], (case, kind)
        worst = [float((a - b).abs().max()) for a, b in zip(out[:2], ref[:2])]
        assert worst == [0., 0.], (case, kind, worst)
    return ref[2:]


@pytest.mark.parametrize("case", list(CASES))
def test_layout_and_launch_do_not_change_the_result(case):
    mk, nb = CASES[case]
    _same_by_every_route(case, *mk(), nb)


# Small meshes: one block runs all directions' fluxes in one launch, blocks a launch a
# direction; a torus 64 zones wide updates on 64-wide tiles, its blocks on 32-wide ones.
# The first timestep is large enough for every signal speed to count: the CFL estimate,
# not the growth limit of twice the last step, sets the timestep after the run.
KASTAUN = dict(inverter="kastaun", err_tol=1e-12, iter_max=25)
SMALL = {
    "2d_hlle": (lambda: _mode((32, 24, 1), riemann="hlle"), (2, 1, 1)),
    "2d_split_ppm": (lambda: _mode((64, 40, 1), precision="split", recon="ppm"), (2, 2, 1)),
    "3d_donor": (lambda: _mode((21, 18, 16), recon="donor_cell_c"), (1, 2, 2)),
    "3d_split_mc": (lambda: _mode((33, 18, 16), precision="split", recon="linear_mc"), (1, 1, 2)),
    "torus2d": (lambda: _torus((36, 24, 1)), (2, 2, 1)),
    "torus2d_split_kastaun_fluid": (lambda: _torus((36, 24, 1), precision="split", floor_frame="fluid", **KASTAUN),
                                    (1, 2, 1)),
    "torus3d_ppm_normal": (lambda: _torus((64, 24, 16), recon="ppm", floor_frame="normal"), (2, 1, 2)),
    "torus3d_split_kastaun_fluid": (lambda: _torus((64, 24, 16), precision="split", floor_frame="fluid", **KASTAUN),
                                    (2, 1, 1)),
    "torus3d_mc_hlle_vl2": (lambda: _torus((64, 24, 16), recon="linear_mc", riemann="hlle", integrator="vl2"),
                            (2, 2, 1)),
}


@pytest.mark.parametrize("case", list(SMALL))
def test_small_meshes_too(case):
    mk, nb = SMALL[case]
    cfg, P = mk()
    cfg["dt_start"] = 0.04 if cfg.get("coords") == "ks" else 0.3 / max(cfg["nx"])
    dts, dt = _same_by_every_route(case, cfg, P, nb)
    assert dt < 1.99 * dts[-1], (dts, dt)
