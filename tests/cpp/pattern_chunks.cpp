// pattern_chunks.cpp — the staging chunks of the pattern build (ikarus_amd/csrc/pattern.cpp) on the CPU, with test
// doubles in host memory for its calls into the HIP runtime.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../ikarus_amd/csrc/ik_internal.hh"

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "host test double"; }
}

namespace {

int bad = 0;

// an n0 x n1 x n2 block of EAS elements in grid order, or nodes and elements in random order: the sizes of its chunks,
// and the share of rows that are complete before the last one
void check(const char* name, int n0, int n1, int n2, bool shuffled, const std::vector<int64_t>& sizes,
           double minShare) {
  ik_handle h;
  const int v0 = n0 + 1, v1 = n1 + 1;
  h.nn   = (int64_t)v0 * v1 * (n2 + 1);
  h.ne   = (int64_t)n0 * n1 * n2;
  h.ndof = h.nn * 3;
  h.neas = 21;
  std::vector<int32_t> node(h.nn), elem(h.ne);
  for (size_t i = 0; i < node.size(); ++i) node[i] = (int32_t)i;
  for (size_t i = 0; i < elem.size(); ++i) elem[i] = (int32_t)i;
  if (shuffled) {
    std::mt19937 rng(3);
    std::shuffle(node.begin(), node.end(), rng);
    std::shuffle(elem.begin(), elem.end(), rng);
  }
  h.hX.resize(h.nn * 3);
  h.hfixed.assign(h.nn * 3, 0);
  h.hconn.resize(h.ne * 8);
  for (int64_t v = 0; v < h.nn; ++v) {
    const int64_t x[3] = {v % v0, v / v0 % v1, v / v0 / v1};
    for (int d = 0; d < 3; ++d) h.hX[node[v] * 3 + d] = (double)x[d];
  }
  for (int64_t e = 0; e < h.ne; ++e) {
    const int64_t i = elem[e] % n0, j = elem[e] / n0 % n1, k = elem[e] / n0 / n1;
    for (int a = 0; a < 8; ++a)
      h.hconn[e * 8 + a] = node[(i + (a & 1)) + v0 * ((j + ((a >> 1) & 1)) + v1 * (k + ((a >> 2) & 1)))];
  }
  ik::buildPattern(&h);
  std::vector<int64_t> got;
  for (size_t c = 1; c < h.chunkElem.size(); ++c) got.push_back(h.chunkElem[c] - h.chunkElem[c - 1]);
  const double share = (double)h.chunkRow[h.chunkRow.size() - 2] / (double)h.nn;
  const bool ok      = got == sizes && h.chunkRow.back() == h.nn && share >= minShare;
  std::printf("%s: %zu chunks, %.3f of the rows before the last%s\n", name, got.size(), share, ok ? "" : " FAILED");
  bad += !ok;
}

}  // namespace

int main() {
  unsetenv("IKARUS_AMD_CHUNK_ELEMENTS");
  check("141,987 grid", 57, 53, 47, false, {141987}, 0.0);
  check("201,898 grid", 59, 58, 59, false, {100949, 100949}, 0.45);
  check("201,898 random", 59, 58, 59, true, {201898}, 0.0);
  check("340,000 grid", 68, 50, 100, false, {113334, 113334, 113332}, 0.6);
  setenv("IKARUS_AMD_CHUNK_ELEMENTS", "1000", 1);
  check("2,400 grid, 1,000 each", 20, 12, 10, false, {1000, 1000, 400}, 0.0);
  check("2,400 random, 1,000 each", 20, 12, 10, true, {1000, 1000, 400}, 0.0);
  std::printf(bad ? "FAILED\n" : "OK\n");
  return bad ? 1 : 0;
}
