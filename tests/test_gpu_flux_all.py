"""The flux kernel that takes all directions of a block in one launch, against one
launch per direction (which a driver runs while its kernels are timed): two
and three dimensions, sizes that leave tiles partly idle, both precisions.  A step's
states agree to rounding: 1e-13 of a variable's largest value with FP64 fluxes, and
with FP32 fluxes 1e-6, a few of their roundings.  On the torus the velocities, which
the inversion makes sensitive to rounding in floor-density zones, are left out.
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
    rng = np.random.default_rng(5)
    P = pr.mhdmode_prims(cfg)
    return cfg, P * (1 + 1e-2 * pr.periodic_fill(rng.uniform(-1, 1, P.shape), cfg))


def _torus(n, **kw):
    cfg = dict(pr.torus_config(*n), **kw)
    return cfg, pr.torus_prims(cfg)


CASES = {
    "2d": lambda: _mode((17, 13, 1)),
    "2d_split_hlle": lambda: _mode((67, 35, 1), precision="split", riemann="hlle"),
    "3d_ppm_ng3": lambda: _mode((21, 14, 9), recon="ppm", ng=3),
    "3d_split": lambda: _mode((33, 18, 11), precision="split"),
    "2d_torus": lambda: _torus((37, 22, 1)),
    "3d_torus_split_mc": lambda: _torus((41, 19, 10), precision="split", recon="linear_mc"),
}


@pytest.mark.parametrize("case", list(CASES))
def test_one_launch_matches_one_per_direction(case):
    import kharma_amd as kh
    cfg, P = CASES[case]()
    print(f"[flux all] {case}", flush=True)
    out = []
    for timed in (False, True):
        drv = kh.Driver(cfg)
        drv.set_kernel_timing(timed)
        drv.init_prims(torch.from_numpy(np.ascontiguousarray(P)).cuda())
        drv.step(1)
        torch.cuda.synchronize()
        out.append([x.cpu().numpy() for x in drv.state()])
    bar = 1e-6 if cfg.get("precision") == "split" else 1e-13
    use = [0, 1, 5, 6, 7] if cfg.get("coords") == "ks" else range(8)
    for a, b in zip(*out):
        for v in use:
            assert np.abs(a[v] - b[v]).max() <= bar * np.abs(b[v]).max(), (case, v)
