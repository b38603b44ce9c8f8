// pattern_chunks.cpp — what the pattern build (ikarus_amd/csrc/pattern.cpp) decides by the numbering of a mesh: staging
// chunks and the stores of K, on the CPU, with test doubles in host memory for its calls into the HIP runtime.
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

// the share of a tile's complete blocks that follow each other in K, in grid order and with nodes in random order (the
// numbering of the elements does not matter), and how K is then stored
void checkStores(const char* name, bool shuffledNodes, double lo, double hi) {
  ik_handle h;
  const int n = 20, v = n + 1;
  h.nn        = (int64_t)v * v * v;
  h.ne        = (int64_t)n * n * n;
  h.ndof      = h.nn * 3;
  std::vector<int32_t> node(h.nn), elem(h.ne);
  for (size_t i = 0; i < node.size(); ++i) node[i] = (int32_t)i;
  for (size_t i = 0; i < elem.size(); ++i) elem[i] = (int32_t)i;
  std::mt19937 rng(3);
  if (shuffledNodes) std::shuffle(node.begin(), node.end(), rng);
  std::shuffle(elem.begin(), elem.end(), rng);
  h.hX.resize(h.nn * 3);
  h.hfixed.assign(h.nn * 3, 0);
  h.hconn.resize(h.ne * 8);
  for (int64_t i = 0; i < h.nn; ++i) {
    const int64_t x[3] = {i % v, i / v % v, i / v / v};
    for (int d = 0; d < 3; ++d) h.hX[node[i] * 3 + d] = (double)x[d];
  }
  for (int64_t e = 0; e < h.ne; ++e) {
    const int64_t i = elem[e] % n, j = elem[e] / n % n, k = elem[e] / n / n;
    for (int a = 0; a < 8; ++a)
      h.hconn[e * 8 + a] = node[(i + (a & 1)) + v * ((j + ((a >> 1) & 1)) + v * (k + ((a >> 2) & 1)))];
  }
  ik::buildPattern(&h);
  bool ok = h.adjacent >= lo && h.adjacent <= hi;
  for (int kind : {IK_NEOHOOKE, IK_SVK}) {
    const size_t MB = 1000000;
    ok &= !ik::nonTemporalK(kind, 200 * MB, h.adjacent) && ik::nonTemporalK(kind, 500 * MB, h.adjacent);
    // beyond 600 MB a Neo-Hooke K goes through the caches where its blocks follow each other
    ok &= ik::nonTemporalK(kind, 800 * MB, h.adjacent) == (kind == IK_SVK || shuffledNodes);
  }
  std::printf("%s: adjacent %.3f%s\n", name, h.adjacent, ok ? "" : " FAILED");
  bad += !ok;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc > 1 && !std::strcmp(argv[1], "stores")) {
    checkStores("grid", false, 0.5, 0.8);
    checkStores("random", true, 0.0, 0.05);
    std::printf(bad ? "FAILED\n" : "OK\n");
    return bad ? 1 : 0;
  }
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
