"""How a crowded bucket of the hashed pass is gone over (in_parts of csrc/buckets.h), compiled for the host: every id's hash is
taken by exactly one attempt, and the attempts, each a sweep of the bucket by one block, stay few whatever the ids are."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "dist-gpu-sampling_amd", "csrc", "buckets.h")
SLOTS = 16384

DRIVER = r"""
// hashes: those of the bucket's different ids.  taken[i]: by how many attempts that their table took
extern "C" int run(const uint32_t* hashes, int64_t n, int units, int log_buckets, uint32_t* taken, int64_t* sweeps) {
  *sweeps = 0;
  return in_parts(units, kHashSlots, log_buckets, [&](HashPart p) {
    ++*sweeps;
    int64_t held = 0;
    const auto mine = [&](uint32_t h) { return int((h >> 23) % uint32_t(p.parts)) == p.part && (h >> log_buckets) - p.lo < p.span; };
    for (int64_t i = 0; i < n; ++i) held += mine(hashes[i]);
    if (held > kHashSlots) return false;
    for (int64_t i = 0; i < n; ++i) taken[i] += mine(hashes[i]);
    return true;
  });
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    text = open(SOURCE).read()
    parts = [re.search(r"^constexpr int kHashSlots = \d+;", text, re.M).group(0),
             re.search(r"^struct HashPart \{.*?^};\n", text, re.S | re.M).group(0),
             *re.findall(r"^constexpr int kPartBit = .*$", text, re.M),
             re.search(r"^template <typename Attempt>\n__device__ __forceinline__ bool in_parts\(.*?\n}\n", text, re.S | re.M).group(0)]
    d = tmp_path_factory.mktemp("parts")
    (d / "parts.cpp").write_text("#include <cstdint>\n#define __device__\n#define __forceinline__ inline\n" + "\n".join(parts) + DRIVER)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "parts.so"), str(d / "parts.cpp")])
    lib = ctypes.CDLL(str(d / "parts.so"))

    def call(hashes, units, log_buckets):
        hashes = np.ascontiguousarray(hashes, dtype=np.uint32)
        taken, sweeps = np.zeros(hashes.size, dtype=np.uint32), ctypes.c_int64()
        ok = lib.run(hashes.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(hashes.size), ctypes.c_int(units), ctypes.c_int(log_buckets),
                     taken.ctypes.data_as(ctypes.c_void_p), ctypes.byref(sweeps))
        return ok, taken, sweeps.value

    return call


@pytest.mark.parametrize("log_buckets,units,values", [
    (8, 20_000, 512),      # spread evenly: the parts suffice
    (8, 100_000, 2),       # two whole values of the bits that choose a part, 32 768 hashes each
    (8, 300_000, 9),
    (9, 300_000, 19),      # a value is one table's worth
    (10, 300_000, 37),     # ... half of one
    (8, 5_000_000, 3),     # more parts than there are values: ids that come up often beside ones that crowd
])
def test_every_hash_is_taken_once_in_few_sweeps(run, log_buckets, units, values):
    rng = np.random.default_rng(units + log_buckets)
    per_value = 1 << (23 - log_buckets)
    top = rng.permutation(512)[:values].astype(np.uint32)
    low = np.arange(per_value, dtype=np.uint32)
    hashes = ((top[:, None] << np.uint32(23 - log_buckets) | low) << np.uint32(log_buckets)).ravel()
    hashes = rng.permutation(hashes)[:units]
    ok, taken, sweeps = run(hashes, units, log_buckets)
    assert ok and (taken == 1).all()
    assert sweeps <= 512 + 2 * 512 and sweeps <= -(-units // (SLOTS // 2)) + 2 * 512
    if values == 512:
        assert sweeps == -(-units // (SLOTS // 2))
