"""The feature header compiled for the host by g++ and called directly (no GPU)."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")

SRC = r"""
#include "padenti/pd_features.hpp"

// a user's hook built on a shipped one
struct NegatedDepth : pd::DepthU16Feature {
  static float eval_prep(const pd::ImageView<uint16_t, 1> &im, int x, int y, Prep dp, const float *p)
  {
    return -pd::DepthU16Feature::eval_prep(im, x, y, dp, p);
  }
};

extern "C" {
int has_fast_depth(void) { return pd::has_fast<pd::DepthU16Feature>::value; }
int has_fast_rgbd(void) { return pd::has_fast<pd::RGBDFeature>::value; }
int has_fast_f32(void) { return pd::has_fast<pd::DepthF32Feature>::value; }
int has_fast_derived(void) { return pd::has_fast<NegatedDepth>::value; }
float depth_u16(const uint16_t *im, int w, int h, int x, int y, const float *p)
{
  return pd::DepthU16Feature::eval(pd::ImageView<uint16_t, 1>{im, w, h}, x, y, p);
}
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("features")
    src, lib = d / "features.cpp", d / "libfeatures.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-fPIC", "-shared", "-I",
                    os.path.join(ROOT, "include"), str(src), "-o", str(lib)], check=True)
    so = C.CDLL(str(lib))
    so.depth_u16.restype = C.c_float
    return so


def test_fast_form_is_not_inherited(host):
    """A hook derived from a shipped one with an eval_prep of its own has no
    fast form: training and prediction call its eval_prep."""
    assert host.has_fast_depth() == 1 and host.has_fast_rgbd() == 1
    assert host.has_fast_f32() == 0
    assert host.has_fast_derived() == 0


@pytest.mark.parametrize("p", [(np.inf, 0, 0, 0), (0, -np.inf, 0, 0), (3e38, 0, -np.inf, np.inf), (1e5, -1e5, 0, 7)])
def test_zero_depth_gives_zero_for_every_offset(host, p):
    im = np.full((5, 5), 1000, np.uint16)
    im[2, 2] = 0
    a = np.array(p, np.float32)
    assert host.depth_u16(im.ctypes.data_as(C.c_void_p), 5, 5, 2, 2, a.ctypes.data_as(C.c_void_p)) == 0.0
