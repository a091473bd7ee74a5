"""The grid of decode launches that run one wave per part (attention_subs),
on the CPU, from the launcher's own functions (ltkv_kernels.h): whole
work-groups cover every item once, every wave past the last item is refused
before it reads or writes anything, and the states of all parts lie inside
the buffer they are given. Fixed partitions (ltkv_set_attention_partition) of
odd multiples of 64 tokens and odd head counts leave such waves over; the
default policies' counts are multiples of a work-group."""

from __future__ import annotations

import os
import subprocess

import pytest

from langtrain_studio_amd import build

SOURCE = r"""
#include <cstdio>
#include <set>
#include "ltkv_kernels.h"
using namespace ltkv;

int main() {
  const int cu = 256;
  struct { int heads, kv, hd; } shapes[] = {{32, 8, 128}, {28, 4, 128}, {8, 1, 128}, {32, 4, 64}, {9, 3, 64},
                                            {14, 2, 64}, {40, 5, 128}, {24, 6, 128}, {6, 6, 64}};
  const int fixed[] = {0, kPartCap, 64, 128, 192, 320, 512, 576, 640, 768, 1024, 1088, 4096};
  const int lens[] = {64, 1000, 2048, 2064, 3088, 3200, 4096, 8192, 8208, 16384};
  long launches = 0, over = 0;
  for (auto &s : shapes)
    for (int elem = 1; elem <= 2; ++elem)
      for (int part : fixed)
        for (int max_len : lens)
          for (int64_t n = 1; n <= 300; ++n) {
            const int group = s.heads / s.kv;
            const bool pairs = group <= 4 && s.kv % 2 == 0;
            const int split = elem == 1 && pairs ? 2 : 1, groups = s.kv / (pairs ? 2 : 1);
            const int max_parts = max_partitions(max_len, part) * split;
            const int subs = attention_subs(elem, s.hd, group, s.kv, false, n, max_parts,
                                            max_partition_size(max_len, part, split), cu);
            if (subs == 0) continue;
            const int64_t per_query = (int64_t)max_parts * subs, items = n * per_query, waves = items * groups;
            const int nw = decode_group_waves(true, waves, cu);
            const int64_t grid_waves = (int64_t)decode_grid(waves, nw) * nw;
            if (grid_waves < waves || grid_waves - waves >= nw) return printf("grid of %ld waves\n", (long)waves), 1;
            ++launches;
            over += grid_waves > waves;
            for (int64_t w = waves - 1; w < grid_waves; ++w) {  // the last item's wave and those past it
              int64_t q;
              int index;
              const bool has = decode_wave_item((uint32_t)(w / groups), (uint32_t)per_query, n, q, index);
              if (has != (w < waves) || (has && (q != n - 1 || index != per_query - 1)))
                return printf("%d/%d/%d elem %d partition %d, %ld queries of %d: wave %ld of %ld\n", s.heads, s.kv, s.hd,
                              elem, part, (long)n, max_len, (long)w, (long)waves), 1;
            }
            if (n == 1)  // a query's parts have slots of their own, whatever its length
              for (int len = 1; len <= max_len; ++len) {
                const int pt = split_partition(len, part, split), st = sub_tokens(len, s.hd);
                if (div_up_tokens(len, pt) > max_parts || div_up_tokens(pt, st) > subs)
                  return printf("slots: partition %d, length %d of %d\n", part, len, max_len), 1;
              }
            if (n * s.heads * per_query * (s.hd + 2) * 4 > (int64_t)kPartsBytes) return printf("bytes\n"), 1;
          }
  printf("%ld %ld\n", launches, over);
}
"""


def test_parts_grid(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "grid.cpp", tmp_path / "grid"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, "-x", "c++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{build.CSRC}", str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    launches, over = map(int, out.stdout.split())
    assert launches > 1000 and over > 100  # launches with waves past the last item are among them
