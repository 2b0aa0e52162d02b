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

// a user's hook on the header's integer-depth probe
struct UserDepth {
  using ImgType = uint16_t;
  using FeatType = float;
  using Prep = pd::IntDivPrep;
  static constexpr int nChannels = 1;
  static constexpr int FeatDim = 4;
  static Prep prepare(const pd::ImageView<uint16_t, 1> &im, int x, int y)
  {
    return pd::int_div_prep((float)im.at(x, y, 0));
  }
  static float eval_prep(const pd::ImageView<uint16_t, 1> &im, int x, int y, Prep dp, const float *p)
  {
    if (!(dp.d > 0.0f)) return 0.0f;
    const int a = pd::probe_int(im, x, y, dp, p[0], p[1], 0, 10000);
    const int b = pd::probe_int(im, x, y, dp, p[2], p[3], 0, 10000);
    return (float)(a - b);
  }
};

extern "C" {
int has_fast_depth(void) { return pd::has_fast<pd::DepthU16Feature>::value; }
int has_fast_rgbd(void) { return pd::has_fast<pd::RGBDFeature>::value; }
int has_fast_f32(void) { return pd::has_fast<pd::DepthF32Feature>::value; }
int has_fast_derived(void) { return pd::has_fast<NegatedDepth>::value; }
// mismatches of the coordinate rules with x + roundf(p / d) at the quotients that
// are exactly halves, (n + 1/2) d <= 2^22 of every n for d in [d0, d1), and at the
// floats next to them, both signs
static uint64_t bad_at(uint32_t x, float p, uint32_t d, bool any)
{
  const pd::RecipPrep y = pd::recip_prep(d);
  const uint32_t want = x + (uint32_t)(int)roundf(p / (float)d);
  uint64_t bad = 0;
  if (fabsf(p) <= pd::RECIP_MAX) bad += pd::recip_coord(x, (double)p, y) != want;
  // (the general form takes every quotient from 2^20 on as outside)
  if (any && fabsf(p / (float)d) < 1048576.0f) bad += pd::recip_coord_any(x, p, y) != want;
  return bad;
}
uint64_t bad_halves(uint32_t d0, uint32_t d1)
{
  uint64_t bad = 0;
  for (uint32_t d = d0; d < d1; d++)
    for (uint64_t h = d; h <= 2ull << 22; h += 2ull * d) {   // h / 2 = (n + 1/2) d, a float
      const float p = (float)h * 0.5f, c[3] = {p, nextafterf(p, 0.0f), nextafterf(p, INFINITY)};
      const uint32_t x = (uint32_t)(h * 2654435761u) >> 16;
      for (float q : c) bad += bad_at(x, q, d, true) + bad_at(x, -q, d, true);
    }
  return bad;
}
uint64_t bad_of(uint64_t n, const uint32_t *x, const float *p, const uint32_t *d)
{
  uint64_t bad = 0;
  for (uint64_t i = 0; i < n; i++) bad += bad_at(x[i], p[i], d[i], true);
  return bad;
}
float depth_u16(const uint16_t *im, int w, int h, int x, int y, const float *p)
{
  return pd::DepthU16Feature::eval(pd::ImageView<uint16_t, 1>{im, w, h}, x, y, p);
}
float depth_u16_fast(const uint16_t *im, int w, int h, int x, int y, const float *p)
{
  using F = pd::DepthU16Feature;
  const pd::ImageView<uint16_t, 1> v{im, w, h};
  return F::eval_fast(v, x, y, F::prepare(v, x, y), F::fast_params(p));
}
float user_depth(const uint16_t *im, int w, int h, int x, int y, const float *p)
{
  const pd::ImageView<uint16_t, 1> v{im, w, h};
  return UserDepth::eval_prep(v, x, y, UserDepth::prepare(v, x, y), p);
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
    for f in (so.depth_u16, so.depth_u16_fast, so.user_depth):
        f.restype = C.c_float
    so.bad_halves.restype = so.bad_of.restype = C.c_uint64
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


def test_integer_depth_probe_for_user_hooks(host):
    """A hook written with int_div_prep / probe_int compiles and gives the
    shipped depth hook's response, in its general and its fast form."""
    rng = np.random.default_rng(8)
    im = rng.choice(np.array([0, 1, 2, 3, 64, 1000, 4096, 65535], np.uint16), (17, 23))
    pi = im.ctypes.data_as(C.c_void_p)
    for _ in range(3000):
        x, y = int(rng.integers(23)), int(rng.integers(17))
        d = max(int(im[y, x]), 1)
        # offsets of a few pixels, every other one on a half
        p = np.array([(int(k) / 2) * d for k in rng.integers(-30, 31, 4)], np.float32)
        p = np.clip(p, -4194304, 4194304) * (1 if rng.random() < 0.5 else np.float32(rng.uniform(0.9, 1.0)))
        pp = p.ctypes.data_as(C.c_void_p)
        want = host.user_depth(pi, 23, 17, x, y, pp)
        assert host.depth_u16(pi, 23, 17, x, y, pp) == want, (x, y, p)
        assert host.depth_u16_fast(pi, 23, 17, x, y, pp) == want, (x, y, p)


@pytest.mark.parametrize("d0,d1", [(1, 2), (2, 3), (3, 16), (16, 256), (256, 4096), (4096, 65536)])
def test_coordinate_of_every_half(host, d0, d1):
    """recip_coord and recip_coord_any against x + roundf(p / d) at every
    half-integer quotient of the fast form's range and the floats beside it."""
    assert host.bad_halves(d0, d1) == 0


def test_coordinate_of_random_offsets(host):
    rng = np.random.default_rng(6)
    n = 4_000_000
    d = rng.integers(1, 65536, n).astype(np.uint32)
    d[: n // 4] = rng.integers(1, 64, n // 4)
    x = rng.integers(0, 65536, n).astype(np.uint32)
    x[::3] = 0                                        # sums below zero
    p = rng.uniform(-4194304, 4194304, n)
    p[1::4] = np.exp(rng.uniform(-30, 26, n)[1::4]) * rng.choice([-1, 1], n)[1::4]   # every magnitude
    p[2::4] = rng.integers(-4194304, 4194305, n)[2::4]                                # whole numbers
    p[:8] = [4194304, -4194304, 4194303.5, -4194303.5, 0.0, -0.0, 1e-40, -1e-40]
    p = p.astype(np.float32)
    assert host.bad_of(C.c_uint64(n), x.ctypes.data_as(C.c_void_p), p.ctypes.data_as(C.c_void_p),
                       d.ctypes.data_as(C.c_void_p)) == 0
