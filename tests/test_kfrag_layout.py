"""The packed K~ layouts (tree_kfrag and tree_kchunk of htree_tree_index.h, which
the build's stores and the operand reads share) on the CPU: within each block of 16 nodes
a permutation of the row-major elements, 4 consecutive d stay together (the
build's 8-byte stores), and lane (u16, kg) of operand load m reads 16 bytes at
1 KB * m + 16 * lane (load_kfrag)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include <cstdio>
#include <vector>
#include "htree_tree_index.h"
using namespace htree;
int main() {
  int bad = 0;
  for (int D : {32, 64, 128, 256}) for (int pairs : {0, 1}) {
    auto kfrag = [&](int64_t r) { return pairs ? tree_kfrag(D, r) : tree_kchunk(D, r); };
    std::vector<int> seen(48 * D, 0);
    for (int64_t n = 0; n < 48; ++n)
      for (int d = 0; d < D; ++d) {
        const int64_t o = kfrag(tree_krow(48, D, 0, n) + d);
        if (o < n / 16 * 16 * D || o >= (n / 16 + 1) * 16 * D) ++bad; else ++seen[o];
        // D = 32 in pair order: a lane holds both halves of RoPE pairs 4 kg .. 4 kg + 3
        const int m = d / 32, kg = pairs && D == 32 ? d % 16 / 4 : d % 32 / 8, lane = kg * 16 + (int)(n % 16);
        const int e = pairs && D == 32 ? d / 16 * 4 + d % 4 : d % 8;
        if (o != n / 16 * 16 * D + m * 512 + lane * 8 + e) ++bad;
        if (d % 4 && o != kfrag(tree_krow(48, D, 0, n) + d - 1) + 1) ++bad;
      }
    for (int s : seen) bad += s != 1;
  }
  std::printf("%d\n", bad);
  return bad != 0;
}
'''


def test_kfrag_layout(tmp_path):
    src = tmp_path / "kfrag.cpp"
    src.write_text(SRC)
    exe = tmp_path / "kfrag"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "htree_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "0", r.stdout
