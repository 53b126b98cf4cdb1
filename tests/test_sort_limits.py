"""CPU test of the sort's index arithmetic at the most elements it takes: the
segments of a pass cover every element once, and no index that a pass's loops
form wraps in 32 bits."""
from __future__ import annotations

import os
import subprocess

import pytest

from mvgpubtree_amd import build

PROGRAM = r"""
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include "mvbt_sort.hpp"
#include "mvbt_bulk.hpp"
using namespace mvbt;
int main() {
  const uint64_t sizes[] = {64, 511, 512, 513, kSortMax / 2 + 1, kSortMax - 513, kSortMax - 1};
  for (uint64_t n : sizes)
    for (uint32_t G : {kSortSegments, 1024u}) {
      uint32_t next = 0;
      for (uint32_t g = 0; g < G; ++g) {
        uint32_t a, b;
        segment_of((uint32_t)n, g, G, a, b);
        if (a != next || b < a) return printf("n %llu: segment %u starts at %u, not %u\n", (unsigned long long)n, g, a, next), 1;
        // the furthest index a loop over the segment computes
        if ((uint64_t)b + 2ull * kSortEach * kSortBlock > 0xFFFFFFFFull) return printf("index wraps at n %llu\n", (unsigned long long)n), 1;
        next = b;
      }
      if (next != n) return printf("n %llu: %u elements covered\n", (unsigned long long)n, next), 1;
    }
  return 0;
}
"""


def test_segments_at_the_largest_sizes(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "segments.hip", tmp_path / "segments"
    src.write_text(PROGRAM)
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, f"-I{build.CSRC}", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_first_inserts_beyond_the_sort_are_staged():
    """mvbt_insert sorts a first insert only below the sort's limit."""
    with open(os.path.join(build.CSRC, "mvbt_capi.hip")) as f:
        body = f.read().split("mvbt_status first_insert(", 1)[1]
    assert "n >= kSortMax) return MVBT_OK;" in body[: body.index("hipLaunchKernelGGL")]
