"""The choice of the automatic skin where steps run on the candidates (csrc/skin_choice.h, host code): followed over many
builds on model systems -- gaps as in a packing or a gas, one speed -- from thin and wide skins. It has to settle on lists
that last, or at the widest skin (where the cell sweep takes over), whatever skin it comes from."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUCKETS = 16
SRC = """
#include "skin_choice.h"
extern "C" void choose(double skin, double radius, double nCand, const uint32_t* gaps, double move, double least,
                       double* out) {
    const deme_int::SkinChoice c = deme_int::choose_skin({skin, radius, nCand, gaps, move, least});
    out[0] = c.skin;
    out[1] = c.ratio;
    out[2] = c.life;
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    d = tmp_path_factory.mktemp("skin")
    (d / "s.cpp").write_text(SRC)
    inc = os.path.join(ROOT, "dem-engine-sbel_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", "-I", inc, str(d / "s.cpp"), "-o",
                    str(d / "s.so")], check=True)
    lib = C.CDLL(str(d / "s.so"))
    lib.choose.argtypes = [C.c_double, C.c_double, C.c_double, C.c_void_p, C.c_double, C.c_double, C.c_void_p]

    def call(skin, radius, n_cand, gaps, move, least=0.0):
        out = np.zeros(3)
        lib.choose(skin, radius, n_cand, gaps.ctypes.data, move, least, out.ctypes.data)
        return out

    return call


def _partners(g, n, fill, touching):
    """Candidates with gaps below g (radius 1): those that touch, then the shells of a packing of that solid fraction."""
    return n * (touching + 0.5 * fill * ((2 + g) ** 3 - 8))


def _settle(choose, n, fill, touching, skin, move, builds=40):
    """(skin, steps its lists last) after so many builds, and whether it is steady."""
    seen = []
    for _ in range(builds):
        edges = _partners(np.arange(BUCKETS + 1) * skin / BUCKETS, n, fill, touching)
        edges[0] = 0.0
        gaps = np.round(np.diff(edges) / edges[-1] * 65536).astype(np.uint32)
        skin, ratio, life = choose(skin, 1.0, edges[-1], gaps, move)
        assert 0.0 < skin <= 0.8 and ratio > 0.0 and life == pytest.approx(0.5 * skin / move)
        seen.append(skin)
    return skin, 0.5 * skin / move, max(seen[-8:]) / min(seen[-8:]) < 1.6


@pytest.mark.parametrize("start", [0.01, 0.05, 0.2, 0.8])
@pytest.mark.parametrize("move", [1e-7, 1e-4, 0.005, 0.02, 0.04, 0.09, 0.2, 0.5])
@pytest.mark.parametrize("n,fill,touching", [(600, 0.6, 3.0), (20_000, 0.6, 3.0), (1_000_000, 0.55, 3.0), (2000, 0.05, 0.0),
                                             (1_000_000, 0.02, 0.0)])
def test_the_skin_settles_on_lists_that_last(choose, n, fill, touching, start, move):
    skin, life, steady = _settle(choose, n, fill, touching, start, move)
    assert steady
    assert life >= 4.0 or skin == 0.8
    # and not far from the best of all skins for this system
    def cost(s):
        k = _partners(s, n, fill, touching)
        return 14e-6 + 70e-12 * k + (300e-6 + 210e-12 * k) / (0.5 * s / move)

    good = [s for s in np.geomspace(0.01, 0.8, 200) if 0.5 * s / move >= 4.0]
    if good:
        assert cost(skin) <= 1.25 * min(map(cost, good))


def test_a_skin_is_kept_when_nothing_is_known(choose):
    none = np.zeros(BUCKETS, np.uint32)
    some = np.full(BUCKETS, 10, np.uint32)
    assert choose(0.2, 1.0, 1e5, none, 0.01)[0] == 0.2
    for move in (np.nan, np.inf):
        assert choose(0.2, 1.0, 1e5, some, move)[0] == 0.2


def test_no_skin_thinner_than_is_kept_is_chosen(choose):
    """A world so large for its spheres that the build positions' unit rules out skins that gaps and speed ask for."""
    skin, least = 0.2, 0.03
    for _ in range(20):
        edges = _partners(np.arange(BUCKETS + 1) * skin / BUCKETS, 1e6, 0.6, 3.0)
        edges[0] = 0.0
        gaps = np.round(np.diff(edges) / edges[-1] * 65536).astype(np.uint32)
        skin = choose(skin, 1.0, edges[-1], gaps, 1e-9, least)[0]
        assert skin >= least
    assert skin < 0.06
