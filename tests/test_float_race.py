"""The float32 race of csrc/choose.h on the CPU: its own source text, compiled for the host, with the hardware
logarithm and reciprocal replaced by ones that round and are then off by a unit in the last place.  The claim that makes
the picks exact: keys that surely_less orders are ordered as the 64-bit keys are, whatever the weights."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "dist-gpu-sampling_amd", "csrc", "choose.h")

PRELUDE = r"""
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __forceinline__ inline
static int log_off = 0, rcp_off = 0;   // units in the last place
static uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static float moved(double v, int off) {
  float f = float(v);
  for (; off > 0; --off) f = nextafterf(f, INFINITY);
  for (; off < 0; ++off) f = nextafterf(f, -INFINITY);
  return f;
}
static float __builtin_amdgcn_logf(float x) { return moved(log2(double(x)), log_off); }
static float __builtin_amdgcn_rcpf(float x) { return x == 0 || std::isinf(x) ? 1 / x : moved(1.0 / double(x), rcp_off); }
"""

DRIVER = r"""
static uint32_t key_of(uint32_t x, float w, uint32_t p) {
  const float e = approx_neg_log_u32(x);
  return plain_weight(w) ? __float_as_uint(e * __builtin_amdgcn_rcpf(w)) : uncommon_key(e, w, p);
}
static long double true_key(uint32_t x, float w) {  // 2e6: above every usable one
  return w > 0 ? (std::isinf(w) ? 0.0L : -logl((x + 0.5L) / 4294967296.0L) / w) : INFINITY;
}
extern "C" {
void set_off(int l, int r) { log_off = l; rcp_off = r; }
double worst_log_error(const uint32_t* x, int64_t n) {
  double worst = 0;
  for (int64_t i = 0; i < n; ++i) {
    const long double t = -logl((x[i] + 0.5L) / 4294967296.0L);
    worst = fmax(worst, double(fabsl(approx_neg_log_u32(x[i]) - t) / t));
  }
  return worst;
}
// pairs (x, w, position): how many are ordered surely and wrongly, and how many surely at all
void pairs(const uint32_t* xa, const float* wa, const uint32_t* pa, const uint32_t* xb, const float* wb, const uint32_t* pb,
           int64_t n, int64_t* wrong, int64_t* sure) {
  *wrong = *sure = 0;
  for (int64_t i = 0; i < n; ++i) {
    const uint32_t a = key_of(xa[i], wa[i], pa[i]), b = key_of(xb[i], wb[i], pb[i]);
    const long double ta = true_key(xa[i], wa[i]), tb = true_key(xb[i], wb[i]);
    const bool less = ta < tb || (ta == tb && pa[i] < pb[i]);
    const bool ab = surely_less(a, b), ba = surely_less(b, a);
    *sure += ab || ba;
    *wrong += (ab && !less) || (ba && less) || a == 0 || b == 0 || a >= kOutOfRace || b >= kOutOfRace;
  }
}
}
"""


def _function(text, name):
    head = r"^__device__ __forceinline__ \w+ %s\(" % name
    return re.search(head + r"[^\n]*}\n|" + head + r".*?\n}\n", text, re.S | re.M).group(0)


@pytest.fixture(scope="module")
def race(tmp_path_factory):
    text = open(SOURCE).read()
    parts = re.findall(r"^constexpr (?:uint32_t k\w+Key|uint32_t kOutOfRace|float kSureRatio) = .*$", text, re.M)
    parts += [_function(text, f) for f in ("approx_neg_log_u32", "plain_weight", "uncommon_key", "surely_less")]
    d = tmp_path_factory.mktemp("race")
    (d / "race.cpp").write_text(PRELUDE + "\n".join(parts) + DRIVER)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(d / "race.so"), str(d / "race.cpp")])
    lib = ctypes.CDLL(str(d / "race.so"))
    lib.worst_log_error.restype = ctypes.c_double
    return lib


def _words(rng, n):
    return rng.integers(0, 1 << 32, size=n, dtype=np.uint64).astype(np.uint32)


def _pairs(race, a, b):
    a, b = [np.ascontiguousarray(v) for v in a], [np.ascontiguousarray(v) for v in b]
    wrong, sure = ctypes.c_int64(), ctypes.c_int64()
    race.pairs(*[ctypes.c_void_p(v.ctypes.data) for v in a + b], ctypes.c_int64(a[0].size), ctypes.byref(wrong), ctypes.byref(sure))
    return wrong.value, sure.value


OFFS = [(l, r) for l in (-1, 0, 1) for r in (-1, 0, 1)]


@pytest.mark.parametrize("log_off,rcp_off", OFFS)
def test_logarithm_stays_within_the_stated_error(race, log_off, rcp_off):
    race.set_off(log_off, rcp_off)
    near = np.arange(1 << 16, dtype=np.uint64)
    half = np.uint64(1 << 31)
    x = np.concatenate([near, half - near, half + near, np.uint64((1 << 32) - 1) - near]).astype(np.uint32)
    x = np.concatenate([x, _words(np.random.default_rng(1), 1 << 20)])
    # (the card's own: 2.9e-7.)  Two keys: 2 x (this, 1.5 units of the reciprocal = 1.8e-7, a rounded product 6e-8) has to
    # stay below kSureRatio - 1 = 1.9e-6
    assert race.worst_log_error(ctypes.c_void_p(x.ctypes.data), ctypes.c_int64(x.size)) < 4e-7


def _weights(rng, kind, n):
    if kind == "plain":
        return (rng.random(n) + 0.01).astype(np.float32)
    if kind == "all":  # every exponent, denormal ones too
        return np.exp2(rng.uniform(-149, 128, size=n)).astype(np.float32).clip(max=np.float32(3.4028234e38))
    if kind == "ends":
        return rng.choice(np.array([1e-45, 1.1e-38, 7.5e-37, 7.53e-37, 1.2379e27, 1.238e27, 3.4e38, np.inf], dtype=np.float32), size=n)
    return rng.choice(np.array([0, -1, np.nan, np.inf, 1, 1e-40], dtype=np.float32), size=n)


@pytest.mark.parametrize("log_off,rcp_off", OFFS)
@pytest.mark.parametrize("ka,kb", [("plain", "plain"), ("all", "all"), ("ends", "all"), ("ends", "ends"), ("none", "none"), ("none", "all")])
def test_sure_order_is_the_order_of_the_64_bit_keys(race, ka, kb, log_off, rcp_off):
    race.set_off(log_off, rcp_off)
    rng = np.random.default_rng(7)
    n = 1 << 15
    pos = [rng.choice([0, 5, 1 << 20, 0xfffffd, 0xfffffe, 0xffffff, 1 << 28], size=n).astype(np.uint32) + rng.integers(0, 4, size=n).astype(np.uint32)
           for _ in range(2)]
    xa, xb, wa, wb = _words(rng, n), _words(rng, n), _weights(rng, ka, n), _weights(rng, kb, n)
    pos[1] += pos[0] == pos[1]
    wrong, _ = _pairs(race, (xa, wa, pos[0]), (xb, wb, pos[1]))
    assert wrong == 0
    # and where the second weight brings the two keys to within some 1e-6 of one another
    with np.errstate(all="ignore"):
        ea, eb = [-np.log((x.astype(np.float64) + 0.5) / 2.0**32) for x in (xa, xb)]
        close = (wa.astype(np.float64) * eb / ea * (1 + rng.uniform(-4e-6, 4e-6, size=n))).astype(np.float32)
    wrong, _ = _pairs(race, (xa, wa, pos[0]), (xb, close, pos[1]))
    assert wrong == 0


@pytest.mark.parametrize("weight", [np.inf, 1e-40, 1e-45, 3e38, 1e30, 0.0, np.nan])
def test_one_uncommon_weight_leaves_no_row_open(race, weight):
    """Its key is ordered against those of ordinary weights without the 64-bit ones."""
    race.set_off(1, -1)
    rng = np.random.default_rng(3)
    n = 20000
    p = np.arange(1, n + 1, dtype=np.uint32)
    odd = np.full(n, weight, dtype=np.float32)
    wrong, sure = _pairs(race, (_words(rng, n), odd, np.zeros(n, np.uint32)), (_words(rng, n), _weights(rng, "plain", n), p))
    assert wrong == 0 and sure == n


def test_infinite_weights_are_ordered_by_their_positions(race):
    rng = np.random.default_rng(3)
    n = 20000
    inf = np.full(n, np.inf, dtype=np.float32)
    p = np.arange(n, dtype=np.uint32)
    assert _pairs(race, (_words(rng, n), inf, p), (_words(rng, n), inf, p + np.uint32(1))) == (0, n)
