"""Memory of result arrays (ArrayAllocator in nlm_host.hpp), compiled with g++: those of 256 KB to
3 MB have their pages mapped when they are allocated, whatever their place in the heap."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

SOURCE = r"""
#include <cstdio>
#include <cstring>
#include "nlm_host.hpp"
static size_t missing(char* p, size_t n) {  // whole pages within [p, p + n) that are not there
  size_t out = 0;
  for (size_t a = ((size_t)p + 4095) / 4096 * 4096; a + 4096 <= (size_t)p + n; a += 4096) {
    unsigned char v = 0;
    if (mincore((void*)a, 4096, &v) || !(v & 1)) out++;
  }
  return out;
}
int main() {
#ifndef MADV_POPULATE_WRITE
  return 77;
#else
  void* q = aligned_alloc(4096, 8192);
  if (madvise(q, 8192, MADV_POPULATE_WRITE)) return 77;  // an older kernel
  nlm::ArrayAllocator<nlm::cd> a;
  std::vector<nlm::cd*> kept;
  for (size_t n : {16384u, 16385u, 30000u, 65536u, 100001u, 196607u}) {
    nlm::cd* p = a.allocate(n);
    if (missing((char*)p, n * sizeof(nlm::cd))) return std::printf("%zu elements\n", n), 1;
    std::memset((void*)p, 1, n * sizeof(nlm::cd));
    kept.push_back(p);
  }
  for (nlm::cd* p : kept) a.deallocate(p, 0);
  for (size_t n : {0u, 1u, 100u, 16383u, 196608u, 400000u}) a.deallocate(a.allocate(n), n);
  nlm::Grid g;
  g.setZero(300, 200);
  for (int i = 0; i < 300; i++)
    for (int k = 0; k < 200; k++)
      if (g.row(i)[k] != nlm::cd(0, 0)) return 2;
  return 0;
#endif
}
"""


def test_pages_of_results_are_mapped(tmp_path):
    src, exe = tmp_path / "arrays.cpp", str(tmp_path / "arrays")
    src.write_text(SOURCE)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(HERE, "..", "multimodenonlinearoptics_amd", "csrc"),
                        "-I" + os.path.join(HERE, "..", "include"), str(src), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    if r.returncode == 77:
        pytest.skip("the system cannot map pages ahead")
    assert r.returncode == 0, r.stdout
