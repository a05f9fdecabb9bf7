"""The links that a hop's edge list is read by (rank_from of csrc/edges.h), compiled for the host: they lead to the
rank at the smallest position, and words that no launch leaves end the search inside the array."""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "dist-gpu-sampling_amd", "csrc", "edges.h")
LINK = 0x80000000


@pytest.fixture(scope="module")
def rank_from(tmp_path_factory):
    text = open(SOURCE).read()
    body = re.search(r"^__device__ __forceinline__ uint32_t rank_from\(.*?\n}\n", text, re.S | re.M).group(0)
    d = tmp_path_factory.mktemp("links")
    (d / "links.cpp").write_text("#include <cstdint>\n#define __device__\n#define __forceinline__ inline\n"
                                 + re.search(r"^constexpr uint32_t kLinkBit = .*$", text, re.M).group(0) + "\n" + body
                                 + 'extern "C" uint32_t run(const uint32_t* a, uint32_t at) { return rank_from(a, at, a[at]); }\n')
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(d / "links.so"), str(d / "links.cpp")])
    lib = ctypes.CDLL(str(d / "links.so"))
    lib.run.restype = ctypes.c_uint32
    return lambda a, at: lib.run(np.ascontiguousarray(a, dtype=np.uint32).ctypes.data_as(ctypes.c_void_p), ctypes.c_uint32(at))


def test_links_lead_to_the_rank(rank_from):
    a = [7, 0 | LINK, 5, 1 | LINK, 3 | LINK, 2 | LINK]
    assert [rank_from(a, p) for p in range(6)] == [7, 7, 5, 7, 7, 5]


@pytest.mark.parametrize("word", [2 | LINK, 3 | LINK, 100_000_000 | LINK, 0xffffffff])
def test_links_that_lead_nowhere_end(rank_from, word):
    """To the position itself, to a later one, beyond the array: one step, nothing read."""
    assert rank_from([7, 0, word, 2 | LINK], 2) == 0
    assert rank_from([7, 0, word, 2 | LINK], 3) == 0
