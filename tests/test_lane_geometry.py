"""The metric that the marching flux kernels keep per lane holds some components only:
the covariant ones but g_{t x2} and g_{x2 phi}, and of the contravariant ones the time
row and the face normal's diagonal.  Asking it for another has to fail at compile
time, and the two that it leaves out have to be exactly zero in the tables of every
coordinate system.
"""
import itertools
import os
import subprocess

import numpy as np
import pytest

from kharma_amd import build as kb
from kharma_amd import problems as pr

USE = """#include "kh_lane_geom.hpp"
__global__ void use(double* o) {
    __shared__ double s[kh::MG_N][256];
    kh::LaneGeom<%d> g{s, 0};
    o[0] = %s;
}
"""


def _compiles(tmp_path, direction, expr):
    src = tmp_path / "use.hip"
    src.write_text(USE % (direction, expr))
    r = subprocess.run([kb.HIPCC] + [f for f in kb.COMMON if f != "-fPIC"] +
                       ["--cuda-device-only", "-fsyntax-only", "-Wno-comment", str(src)], capture_output=True, text=True)
    assert r.returncode == 0 or "no slot for this component" in r.stderr, r.stderr
    return r.returncode == 0


def test_held_components_compile(tmp_path):
    cov = ["g.gcov<%d, %d>()" % ab for ab in itertools.product(range(4), repeat=2) if sorted(ab) not in ([0, 2], [2, 3])]
    con = ["kh::gcon_at<%d, %d>(g)" % ab for ab in ((0, 0), (0, 1), (2, 0), (0, 3), (2, 2))]
    assert _compiles(tmp_path, 2, " + ".join(cov + con))


@pytest.mark.parametrize("direction, expr", [(1, "g.gcov<0, 2>()"), (3, "g.gcov<3, 2>()"), (1, "kh::gcon_at<2, 2>(g)"),
                                             (3, "kh::gcon_at<1, 3>(g)")])
def test_missing_components_do_not_compile(tmp_path, direction, expr):
    assert not _compiles(tmp_path, direction, expr)


@pytest.mark.parametrize("transform", ["null", "mks", "fmks"])
@pytest.mark.parametrize("a", [0.0, 0.5, 0.9375])
def test_left_out_components_vanish(transform, a):
    import kharma_amd as kh
    cfg = dict(pr.torus_config(24, 16, 8, a=a), transform=transform)
    if transform == "null":
        cfg["bounds"] = ((1.2, 40.0), (0.0, np.pi), (0.0, 2 * np.pi))
    for loc in range(3):
        for comp in (2, 8):
            assert not np.any(kh.geometry_host(cfg, loc, comp)), (loc, comp)
