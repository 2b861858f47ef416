"""Host checks of the numerics headers shared with the gfx950 kernels.

vramancer_amd/csrc/vrm_fdlibm_atan2f.h must reproduce the C library's float
atan2 (what PyTorch's CPU kernel calls on the reference's strided views) and
vramancer_amd/csrc/vrm_e4m3.h must reproduce torch's float8_e4m3fn cast.
Both headers are compiled here with g++ (no FP contraction, as on the GPU).
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
CSRC = os.path.join(ROOT, "vramancer_amd", "csrc")

SRC = r"""
#include "vrm_fdlibm_atan2f.h"
#include "vrm_e4m3.h"
#include "vrm_tq_bin.h"
#include <math.h>
#include <stdint.h>
extern "C" long atan2_mismatches(long n, uint64_t seed, int mode) {
  uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
  auto next = [&]() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; };
  long bad = 0;
  for (long i = 0; i < n; ++i) {
    float y, x;
    if (mode == 0) {  // random bit patterns
      y = vrm_fdlibm::bitsf((uint32_t)next()); x = vrm_fdlibm::bitsf((uint32_t)next());
    } else {          // moderate magnitudes with random signs and exponents in [-20, 20]
      uint32_t r = (uint32_t)next(), q = (uint32_t)next();
      y = ldexpf(1.0f + (r & 0xffffff) / 16777216.0f, (int)(r >> 26) % 21 - 10) * ((r >> 25) & 1 ? -1.f : 1.f);
      x = ldexpf(1.0f + (q & 0xffffff) / 16777216.0f, (int)(q >> 26) % 21 - 10) * ((q >> 25) & 1 ? -1.f : 1.f);
    }
    float a = vrm_fdlibm::atan2f(y, x), b = ::atan2f(y, x);
    if (vrm_fdlibm::fbits(a) != vrm_fdlibm::fbits(b) && !(isnan(a) && isnan(b))) ++bad;
  }
  return bad;
}
// bins off the sector edges that differ from the defining atan2; values drawn
// over 80 binary orders, at ratios within 2^-19 of 1 and within 1e-5 rad of an edge
template <int BITS, bool L0> static long bins(long n, uint64_t seed, long* edges) {
  uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
  auto next = [&]() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; };
  auto uni = [&]() { return (double)(next() >> 11) / 9007199254740992.0; };
  const float lo0 = (float)-3.141592653589793, r0 = (float)6.283185307179586, r1 = (float)1.5707963267948966;
  long bad = 0;
  for (long i = 0; i < n; ++i) {
    float x = (float)(4 * uni() - 2), y = (float)(4 * uni() - 2);
    if (i % 4 == 1) y = x * (1.0f + ldexpf((float)((int)(next() % 65) - 32), -24));
    if (i % 4 == 2) {
      const double step = (L0 ? 2 * M_PI : M_PI / 2) / (1 << BITS);
      const double th = (L0 ? -M_PI : 0.0) + step * (double)(next() % ((1 << BITS) + 1)) + (uni() - 0.5) * 2e-5;
      const double r = 0.01 + uni();
      x = (float)(r * cos(th)); y = (float)(r * sin(th));
    }
    if (i % 4 == 3) { x = ldexpf(x, -(int)(next() % 40)); y = ldexpf(y, -(int)(next() % 40)); }
    if (!L0) { x = fabsf(x); y = fabsf(y); }
    // the reciprocal off by up to one ulp either way
    const float rcp = vrm_fdlibm::bitsf(vrm_fdlibm::fbits(1.0f / fmaxf(fabsf(x), fabsf(y))) + (uint32_t)(next() % 3) - 1u);
    bool edge;
    const int got = vrm_tq_bin::fast_bin<BITS, L0>(x, y, rcp, edge);
    if (edge) { ++*edges; continue; }
    const float th = vrm_fdlibm::atan2f(y, x);
    const float d = th - lo0;
    const float nrm = L0 ? d / r0 : th / r1;
    const float t = nrm * (float)(1 << BITS);
    int ref = (int)t;
    ref = ref < 0 ? 0 : ref > (1 << BITS) - 1 ? (1 << BITS) - 1 : ref;
    if (got != ref) ++bad;
  }
  return bad;
}
extern "C" long fast_bin_mismatches(int bits, int level0, long n, uint64_t seed, long* edges) {
  switch (2 * bits + level0) {
    case 4: return bins<2, false>(n, seed, edges);
    case 5: return bins<2, true>(n, seed, edges);
    case 6: return bins<3, false>(n, seed, edges);
    case 7: return bins<3, true>(n, seed, edges);
    case 8: return bins<4, false>(n, seed, edges);
    default: return bins<4, true>(n, seed, edges);
  }
}
// Multiples of pi / 4, by operands of one magnitude and by signed zeros: bins
// that differ from the defining atan2, or that are left to it.
template <int BITS, bool L0> static long symmetric() {
  const float lo0 = (float)-3.141592653589793, r0 = (float)6.283185307179586, r1 = (float)1.5707963267948966;
  const float mags[] = {1e-37f, 3e-20f,  // normal: the reciprocal of a denormal overflows, which is an edge
                         1e-6f, 0.3f, 1.f, 2.7182817f, 5e4f, 1e15f};
  long bad = 0;
  for (float m : mags) {
    if (!L0 && m < 1e-6f) continue;  // radii carry a floor of 1e-6
    for (int c = 0; c < 32; ++c) {
      float x = c & 4 ? 0.f : m, y = c & 8 ? 0.f : m;
      if (c & 16) x *= 0.5f, y *= 0.5f;
      x = c & 1 ? -x : x;
      y = c & 2 ? -y : y;
      if (!L0) { x = m; y = m; }
      bool edge;
      const int got = vrm_tq_bin::fast_bin<BITS, L0>(x, y, 1.0f / fmaxf(fabsf(x), fabsf(y)), edge);
      const float th = vrm_fdlibm::atan2f(y, x);
      const float d = th - lo0;
      const float nrm = L0 ? d / r0 : th / r1;
      const float t = nrm * (float)(1 << BITS);
      int ref = (int)t;
      ref = ref < 0 ? 0 : ref > (1 << BITS) - 1 ? (1 << BITS) - 1 : ref;
      if (edge || got != ref) ++bad;
    }
  }
  return bad;
}
// The ends of the range above level 0: small angles to x and to y.
template <int BITS> static long ends(long n) {
  uint64_t s = 88172645463325252ull;
  auto next = [&]() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; };
  long bad = 0;
  for (long i = 0; i < n; ++i) {
    float x = ldexpf(1.0f + (float)(next() & 0x7fffff) / 8388608.0f, (int)(next() % 20));
    float y = x * ldexpf(1.0f + (float)(next() & 0x7fffff) / 8388608.0f, -20 - (int)(next() % 16));
    if (i & 1) { const float z = x; x = y; y = z; }
    bool edge;
    const int got = vrm_tq_bin::fast_bin<BITS, false>(x, y, 1.0f / fmaxf(x, y), edge);
    const float nrm = vrm_fdlibm::atan2f(y, x) / (float)1.5707963267948966;
    const float t = nrm * (float)(1 << BITS);
    int ref = (int)t;
    ref = ref > (1 << BITS) - 1 ? (1 << BITS) - 1 : ref;
    if (edge || got != ref) ++bad;
  }
  return bad;
}
extern "C" long end_mismatches(long n) { return ends<2>(n) + ends<3>(n) + ends<4>(n); }
// Above level 0, pi / 4 within 64 ulp: the same.
template <int BITS> static long middle(long n) {
  uint64_t s = 88172645463325252ull;
  auto next = [&]() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; };
  long bad = 0;
  for (long i = 0; i < n; ++i) {
    const float x = ldexpf(1.0f + (float)(next() & 0x7fffff) / 8388608.0f, (int)(next() % 60) - 19);
    const float y = vrm_fdlibm::bitsf(vrm_fdlibm::fbits(x) + (uint32_t)(next() % 129) - 64u);
    bool edge;
    const int got = vrm_tq_bin::fast_bin<BITS, false>(x, y, 1.0f / fmaxf(x, y), edge);
    const float nrm = vrm_fdlibm::atan2f(y, x) / (float)1.5707963267948966;
    const float t = nrm * (float)(1 << BITS);
    if (edge || got != (int)t) ++bad;
  }
  return bad;
}
extern "C" long middle_mismatches(long n) { return middle<2>(n) + middle<3>(n) + middle<4>(n); }
extern "C" long symmetric_mismatches() {
  return symmetric<2, false>() + symmetric<2, true>() + symmetric<3, false>() + symmetric<3, true>() +
         symmetric<4, false>() + symmetric<4, true>();
}
extern "C" uint32_t div_sqrt128_bits(float x) { return vrm_fdlibm::fbits(vrm_tq_bin::div_sqrt128(x)); }
extern "C" long div_sqrt128_mismatches(int exponent) {
  const volatile float root = (float)sqrt(128.0);
  long bad = 0;
  for (uint32_t m = 0; m < (1u << 23); ++m) {
    const float x = vrm_fdlibm::bitsf(((uint32_t)(exponent + 127) << 23) | m);
    if (x / root != vrm_tq_bin::div_sqrt128(x)) ++bad;
  }
  return bad;
}
extern "C" float atan2_one(float y, float x) { return vrm_fdlibm::atan2f(y, x); }
extern "C" void e4m3_encode(const float* x, uint8_t* y, long n) { for (long i = 0; i < n; ++i) y[i] = vrm_e4m3::encode(x[i]); }
extern "C" void e4m3_decode(const uint8_t* x, float* y, long n) { for (long i = 0; i < n; ++i) y[i] = vrm_e4m3::decode(x[i]); }
"""


@pytest.fixture(scope="module")
def hostlib(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostnum")
    src = d / "hostnum.cpp"
    src.write_text(SRC)
    so = d / "hostnum.so"
    subprocess.check_call(["g++", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                           f"-I{CSRC}", str(src), "-o", str(so), "-lm"])
    lib = ctypes.CDLL(str(so))
    lib.atan2_mismatches.restype = ctypes.c_long
    lib.atan2_mismatches.argtypes = [ctypes.c_long, ctypes.c_uint64, ctypes.c_int]
    lib.atan2_one.restype = ctypes.c_float
    lib.atan2_one.argtypes = [ctypes.c_float, ctypes.c_float]
    return lib


@pytest.mark.parametrize("mode", [0, 1])
def test_fdlibm_atan2f_matches_libm(hostlib, mode):
    assert hostlib.atan2_mismatches(4_000_000, 12345 + mode, mode) == 0


def test_fdlibm_atan2f_matches_torch_strided_atan2(hostlib):
    # torch's CPU atan2 on the reference's strided pair views is the libm routine
    g = torch.Generator().manual_seed(0)
    x = torch.randn(4096, 2, generator=g)
    t = torch.atan2(x[:, 1], x[:, 0])
    mine = torch.tensor([hostlib.atan2_one(float(b), float(a)) for a, b in x.tolist()])
    assert torch.equal(t, mine)


def test_fdlibm_atan2f_special_values(hostlib):
    sp = [0.0, -0.0, 1.0, -1.0, float("inf"), -float("inf"), 1e-40, -1e-40, 3.4e38, 1.17e-38]
    libm = ctypes.CDLL("libm.so.6")
    libm.atan2f.restype = ctypes.c_float
    libm.atan2f.argtypes = [ctypes.c_float, ctypes.c_float]
    for y in sp:
        for x in sp:
            a, b = hostlib.atan2_one(y, x), libm.atan2f(y, x)
            assert np.float32(a).view(np.uint32) == np.float32(b).view(np.uint32), (y, x)


@pytest.mark.parametrize("level0", [0, 1])
@pytest.mark.parametrize("bits", [2, 3, 4])
def test_fast_bin_is_the_defined_bin_off_the_edges(hostlib, bits, level0):
    edges = ctypes.c_long(0)
    hostlib.fast_bin_mismatches.restype = ctypes.c_long
    hostlib.fast_bin_mismatches.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_uint64, ctypes.c_void_p]
    n = 2_000_000
    assert hostlib.fast_bin_mismatches(bits, level0, n, 7 + bits, ctypes.byref(edges)) == 0
    # the ordinary quarter of the draws is hardly ever at an edge
    assert edges.value < 0.76 * n


def test_fast_bin_knows_the_multiples_of_a_quarter_pi(hostlib):
    hostlib.symmetric_mismatches.restype = ctypes.c_long
    assert hostlib.symmetric_mismatches() == 0


def test_fast_bin_decides_the_middle_of_the_range(hostlib):
    hostlib.middle_mismatches.restype = ctypes.c_long
    hostlib.middle_mismatches.argtypes = [ctypes.c_long]
    assert hostlib.middle_mismatches(3_000_000) == 0


def test_fast_bin_has_no_edge_at_the_ends_of_the_range(hostlib):
    hostlib.end_mismatches.restype = ctypes.c_long
    hostlib.end_mismatches.argtypes = [ctypes.c_long]
    assert hostlib.end_mismatches(2_000_000) == 0


def test_div_sqrt128_keeps_the_sign_of_zero(hostlib):
    hostlib.div_sqrt128_bits.restype = ctypes.c_uint32
    hostlib.div_sqrt128_bits.argtypes = [ctypes.c_float]
    assert hostlib.div_sqrt128_bits(0.0) == 0 and hostlib.div_sqrt128_bits(-0.0) == 0x80000000


@pytest.mark.parametrize("exponent", [-100, -3, 0, 1, 100])
def test_div_sqrt128_is_correctly_rounded(hostlib, exponent):
    # every significand of a binary order; the operation is the same in each
    hostlib.div_sqrt128_mismatches.restype = ctypes.c_long
    assert hostlib.div_sqrt128_mismatches(exponent) == 0


def test_e4m3_encode_matches_torch_cast(hostlib):
    rng = np.random.default_rng(0)
    bits = rng.integers(0, 2**32, size=1 << 22, dtype=np.uint64).astype(np.uint32)
    # add every float in [0, 512) on a fine grid, both signs
    grid = np.arange(0, 512, 1 / 4096, dtype=np.float32)
    f = np.concatenate([bits.view(np.float32), grid, -grid])
    f = f[~np.isnan(f)]
    mine = np.empty(f.size, np.uint8)
    hostlib.e4m3_encode(f.ctypes.data_as(ctypes.c_void_p), mine.ctypes.data_as(ctypes.c_void_p),
                        ctypes.c_long(f.size))
    ref = torch.from_numpy(f).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    assert np.array_equal(mine, ref)


def test_e4m3_decode_all_codes(hostlib):
    codes = np.arange(256, dtype=np.uint8)
    out = np.empty(256, np.float32)
    hostlib.e4m3_decode(codes.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p),
                        ctypes.c_long(256))
    ref = torch.from_numpy(codes).view(torch.float8_e4m3fn).float().numpy()
    nan = np.isnan(ref)
    assert np.array_equal(out[~nan], ref[~nan]) and np.isnan(out[nan]).all()
