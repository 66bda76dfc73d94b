"""
The shares of the one-pass 8 x 8 three-body kernel, on the host: for every
molecule of 0 to 256 atoms the search for a share's first tile ends, and the
shares together hold every chunk (tile, 8 third atoms) of the molecule once.
The functions are the kernel's own (``d4_internal.h``); the walk over the list
that follows the search is restated here.
"""

import os
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include <map>
#include <tuple>
#include <algorithm>
#include "csrc/d4_internal.h"
using namespace d4;
int main() {
  for (int n = 0; n <= kAtm1MaxN; ++n) {
    const int nb = (n + kAtm8 - 1) / kAtm8, nw = (nb + 1) / 2, V = atm8_chunks(nb);
    const int S = atm8_splits(n);
    if (n == 0 && (S != 0 || V != 0)) return std::printf("n = 0: %d parts of %d\n", S, V), 1;
    if (n > 0 && S < 1) return std::printf("n = %d: no part\n", n), 1;
    std::map<std::tuple<int, int, int>, int> seen;  // tile blocks and third-atom block
    int next = 0;
    for (int s = 0; s < S; ++s) {
      int pos = (int)((int64_t)V * s / S);
      const int end = (int)((int64_t)V * (s + 1) / S);
      if (pos != next || end <= pos) return std::printf("n = %d: empty part %d\n", n, s), 1;
      next = end;
      Atm8Start a = atm8_seek(nb, pos);
      while (pos < end) {
        const bool wt = a.t < nw;
        const int bx = wt ? -1 : a.bx, by = wt ? a.t : a.by, z1 = wt ? 0 : a.by + 1;
        if (!wt && !(a.bx < a.by && a.by <= nb - 2))
          return std::printf("n = %d part %d: no tile (%d, %d)\n", n, s, a.bx, a.by), 1;
        if (!wt && ++a.bx == a.by) {
          a.bx = 0;
          ++a.by;
        }
        const int len = (wt ? nb : nb - by - 1) + kAtm8TileCost;
        const int upto = std::min(len, a.off + end - pos);
        for (int c = std::max(0, a.off - kAtm8TileCost); c < upto - kAtm8TileCost; ++c)
          ++seen[{bx, by, z1 + c}];
        pos += upto - a.off;
        a.off = 0;
        ++a.t;
      }
    }
    if (next != V) return std::printf("n = %d: parts end at %d of %d\n", n, next, V), 1;
    size_t chunks = 0;
    for (int t = 0; t < nw; ++t)
      for (int z = 0; z < nb; ++z) chunks += seen.count({-1, t, z});
    for (int by = 1; by <= nb - 2; ++by)
      for (int bx = 0; bx < by; ++bx)
        for (int z = by + 1; z < nb; ++z) chunks += seen.count({bx, by, z});
    const size_t want = (size_t)nw * nb + (nb > 2 ? (size_t)(nb - 2) * (nb - 1) * nb / 6 : 0);
    if (chunks != want || seen.size() != want)
      return std::printf("n = %d: %zu and %zu chunks of %zu\n", n, chunks, seen.size(), want), 1;
    for (auto& e : seen)
      if (e.second != 1) return std::printf("n = %d: a chunk %d times\n", n, e.second), 1;
  }
  return 0;
}
"""


def test_every_chunk_in_one_share(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src = tmp_path / "shares.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "shares"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    # -ftrapv: a signed overflow ends the program
    subprocess.run([cxx, "-std=c++17", "-O1", "-ftrapv", "-w", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROOT / 'tad_dftd4_amd'}", f"-I{rocm}/include", str(src), "-o", str(exe)],
                   check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
