// pattern.cpp — 3x3-block sparsity pattern, its sliced-ELL storage slots and element block-slot maps.
//
// Ikarus builds the scalar pattern from the union of element DOF cliques with Eigen setFromTriplets
// and keeps per element (3*8)^2 positions into the CSC value array (simpleassemblers.inl:207-222,
// 254-265; eigensparseaddon.hh:19-29). For FlatInterleaved DOFs (dof = 3*node + k, fehelper.hh:146-152)
// that scalar pattern is exactly the node-adjacency pattern expanded by 3x3 blocks, so the device keeps
// the block form: block row = node, sorted block columns (CSR order), each block stored at a sliced-ELL
// slot, and the maps from element blocks to staging slots in the gather order of their K blocks (per
// element for EAS, per tile group for the plain element). The scalar CSC is re-derived from it on demand.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <thread>

#include "host_parallel.hh"
#include "ik_internal.hh"

namespace ik {

// elements per staging chunk; IKARUS_AMD_CHUNK_ELEMENTS overrides it. Plain element: splitting the 64^3 mesh into
// chunks whose gathers overlap the next chunk's element work measured slower than one launch of each (the two kernels
// contend for the same memory path), so the default takes meshes up to 1 M elements in one chunk. EAS: the element
// kernel is bound by its arithmetic and leaves the memory to the gathers, so the mesh is cut into equal chunks of about
// kChunkElementsEas (a short last chunk leaves SIMDs idle), unless the numbering completes few rows before the last
// chunk, which leaves nothing to overlap. Assembly and update, us, in one chunk / chunks of 131,072 and a rest / by
// this rule, Neo-Hooke:
//  grid order    141,987 elements 1,382 / 1,444 / 1,378, 198,476: 1,877 / 1,875 / 1,863, 238,328: 2,216 / 2,190 /
//                2,196, 287,496: 2,645 / 2,606 / 2,604, 373,248: 3,387 / 3,307 / 3,308, 442,368: 3,986 / 3,879 /
//                3,877, 806,400: 7,089 / 6,924 / 6,898
//  random order  198,476: 1,990 / 2,033 / 1,991, 238,328: 2,350 / 2,399 / 2,349, 442,368: 4,324 / 4,401 / 4,329
//  442,368 in grid order in chunks of 262,144 / 196,608 / 131,072 / 98,304 / 65,536: 4,040 / 3,891 / 3,862 / 3,879 /
//                3,932
constexpr int64_t kChunkElements = 1 << 20, kChunkElementsEas = 1 << 17;

static int64_t chunkOverride() {
  if (const char* v = std::getenv("IKARUS_AMD_CHUNK_ELEMENTS")) {
    const long long c = std::atoll(v);
    if (c >= 64) return (int64_t)c;
  }
  return 0;
}

// the low 21 bits of v spread to every third bit (bit i -> bit 3i)
static uint64_t spread3(uint32_t v) {
  uint64_t x = v & 0x1FFFFFu;
  x          = (x | x << 32) & 0x1F00000000FFFFull;
  x          = (x | x << 16) & 0x1F0000FF0000FFull;
  x          = (x | x << 8) & 0x100F00F00F00F00Full;
  x          = (x | x << 4) & 0x10C30C30C30C30C3ull;
  x          = (x | x << 2) & 0x1249249249249249ull;
  return x;
}

// The mesh lattice: node bounds and, per axis, the median element extent, an element's extent along axis d
// being the largest |component d| of its three mean edge vectors (the average of the four edges along each
// reference axis), which node jitter leaves unbiased. On a structured grid the lattice is the grid itself.
static void meshLattice(ik_handle* h) {
  const int64_t ne = h->ne, nn = h->nn;
  const double* X     = h->hX.data();
  const int32_t* conn = h->hconn.data();
  const int64_t T     = chunkCount(nn);
  std::vector<double> plo((size_t)T * 3, 0.0), phi((size_t)T * 3, 0.0);
  parallelChunks(nn, [&](int64_t n0, int64_t n1, int64_t c) {
    for (int d = 0; d < 3; ++d) {
      double lo = X[n0 * 3 + d], hi = lo;
      for (int64_t n = n0 + 1; n < n1; ++n) {
        lo = std::min(lo, X[n * 3 + d]);
        hi = std::max(hi, X[n * 3 + d]);
      }
      plo[c * 3 + d] = lo;
      phi[c * 3 + d] = hi;
    }
  });
  HostVec<double> ext(ne);
  for (int d = 0; d < 3; ++d) {
    h->latLo[d] = plo[d];
    h->latHi[d] = phi[d];
    for (int64_t c = 1; c < T; ++c) {
      h->latLo[d] = std::min(h->latLo[d], plo[c * 3 + d]);
      h->latHi[d] = std::max(h->latHi[d], phi[c * 3 + d]);
    }
    parallelChunks(ne, [&](int64_t e0, int64_t e1, int64_t) {
      for (int64_t e = e0; e < e1; ++e) {
        double best = 0.0;
        for (int m = 0; m < 3; ++m) {
          double v = 0.0;  // 4 x component d of the mean edge vector along reference axis m
          for (int a = 0; a < 8; ++a)
            if (!((a >> m) & 1)) v += X[conn[e * 8 + (a | (1 << m))] * 3 + d] - X[conn[e * 8 + a] * 3 + d];
          best = std::max(best, std::fabs(0.25 * v));
        }
        ext[e] = best;
      }
    });
    std::nth_element(ext.begin(), ext.begin() + ne / 2, ext.end());
    h->latStep[d] = ext[ne / 2] > 0.0 ? ext[ne / 2] : 1.0;
  }
}

// Elements in Morton (Z) order of their centroids on the mesh lattice, ties by element index. On a
// structured grid 16 consecutive elements then form a 4x2x2 box (45 nodes) whose 576 upper element blocks
// fall on 341 distinct K blocks; on other meshes the order still keeps each tile compact.
static HostVec<int32_t> mortonOrder(const ik_handle* h) {
  const int64_t ne = h->ne;
  const double* X     = h->hX.data();
  const int32_t* conn = h->hconn.data();
  const double* lo = h->latLo;
  const double* step = h->latStep;
  HostVec<std::pair<uint64_t, int32_t>> key(ne);
  parallelChunks(ne, [&](int64_t e0, int64_t e1, int64_t) {
    for (int64_t e = e0; e < e1; ++e) {
      uint64_t k = 0;
      for (int d = 0; d < 3; ++d) {
        double c = 0.0;
        for (int a = 0; a < 8; ++a) c += X[conn[e * 8 + a] * 3 + d];
        const double q = std::floor((0.125 * c - lo[d]) / step[d]);
        const uint32_t qi = q <= 0.0 ? 0u : (q >= 2097151.0 ? 2097151u : (uint32_t)q);
        k |= spread3(qi) << d;
      }
      key[e] = {k, (int32_t)e};
    }
  });
  // sorted runs per thread, then merged pairwise (keys are distinct: the element index breaks ties)
  {
    const int64_t T = chunkCount(ne);
    std::vector<int64_t> b(T + 1);
    for (int64_t c = 0; c <= T; ++c) b[c] = ne * c / T;
    parallelChunks(ne, [&](int64_t e0, int64_t e1, int64_t) { std::sort(key.begin() + e0, key.begin() + e1); });
    for (int64_t w = 1; w < T; w *= 2) {
      std::vector<std::thread> th;
      for (int64_t c = 0; c + w < T; c += 2 * w)
        th.emplace_back([&, c] {
          std::inplace_merge(key.begin() + b[c], key.begin() + b[c + w], key.begin() + b[std::min(T, c + 2 * w)]);
        });
      for (auto& x : th) x.join();
    }
  }
  HostVec<int32_t> order(ne);
  parallelChunks(ne, [&](int64_t i0, int64_t i1, int64_t) {
    for (int64_t i = i0; i < i1; ++i) order[i] = key[i].second;
  });
  return order;
}

void buildPattern(ik_handle* h) {
  const int64_t nn = h->nn, ne = h->ne;
  const int32_t* conn = h->hconn.data();
  meshLattice(h);
  // node -> incidences e*8 + a (CSR, ordered by element): nlist; the incident elements are nlist / 8
  std::vector<int64_t> cnt(nn + 1, 0);
  for (int64_t e = 0; e < ne; ++e)
    for (int a = 0; a < 8; ++a) cnt[conn[e * 8 + a] + 1]++;
  for (int64_t i = 0; i < nn; ++i) cnt[i + 1] += cnt[i];
  require(cnt[nn] < (int64_t)INT32_MAX, IK_EINVAL, "mesh too large for int32 incidence lists");
  HostVec<int32_t> nlist(cnt[nn]);
  {
    std::vector<int64_t> pos(cnt.begin(), cnt.end() - 1);
    for (int64_t e = 0; e < ne; ++e)
      for (int a = 0; a < 8; ++a) nlist[pos[conn[e * 8 + a]]++] = (int32_t)(e * 8 + a);
  }
  auto inc = [&](int64_t k) { return (int64_t)(nlist[k] >> 3); };
  // rows: union of the nodes of incident elements (per chunk of rows, then placed by the row counts)
  h->hrowptr.assign(nn + 1, 0);
  {
    std::vector<std::vector<int32_t>> part(chunkCount(nn));
    HostVec<int64_t> rc(nn);
    parallelChunks(nn, [&](int64_t i0, int64_t i1, int64_t c) {
      std::vector<int32_t>& cols = part[c];
      cols.reserve((size_t)(i1 - i0) * 27);
      std::vector<int32_t> buf;
      for (int64_t i = i0; i < i1; ++i) {
        buf.clear();
        for (int64_t k = cnt[i]; k < cnt[i + 1]; ++k) {
          const int64_t e = inc(k);
          for (int b = 0; b < 8; ++b) buf.push_back(conn[e * 8 + b]);
        }
        std::sort(buf.begin(), buf.end());
        buf.erase(std::unique(buf.begin(), buf.end()), buf.end());
        cols.insert(cols.end(), buf.begin(), buf.end());
        rc[i] = (int64_t)buf.size();
      }
    });
    int64_t tot = 0;
    for (int64_t i = 0; i < nn; ++i) {
      tot += rc[i];
      require(tot < (int64_t)INT32_MAX, IK_EINVAL, "pattern too large for int32 block indices");
      h->hrowptr[i + 1] = (int32_t)tot;
    }
    h->hcolidx.clear();
    h->hcolidx.resize(tot);
    parallelChunks(nn, [&](int64_t i0, int64_t, int64_t c) {
      std::copy(part[c].begin(), part[c].end(), h->hcolidx.begin() + h->hrowptr[i0]);
    });
  }
  h->nnzb = (int64_t)h->hcolidx.size();
  h->hdiag.assign(nn, -1);
  parallelChunks(nn, [&](int64_t i0, int64_t i1, int64_t) {
    for (int64_t i = i0; i < i1; ++i) {
      const auto b = h->hcolidx.begin() + h->hrowptr[i], en = h->hcolidx.begin() + h->hrowptr[i + 1];
      h->hdiag[i] = (int32_t)(std::lower_bound(b, en, (int32_t)i) - h->hcolidx.begin());
    }
  });
  // Sliced-ELL slots of K: slice s (rows [64 s, 64 s + 64)) is as wide as its longest row; block j of row i
  // sits at slot sstart[s] + 64 j + (i mod 64). The last slice is padded to 64 rows too (rows past nn own only
  // padding slots, which the kernels never read).
  const int64_t nslices = (nn + kSellRows - 1) / kSellRows;
  std::vector<int32_t> sstart(nslices + 1, 0);
  {
    int64_t tot = 0;
    for (int64_t s = 0; s < nslices; ++s) {
      int32_t w = 0;
      for (int64_t i = s * kSellRows; i < std::min(nn, (s + 1) * kSellRows); ++i)
        w = std::max(w, h->hrowptr[i + 1] - h->hrowptr[i]);
      tot += (int64_t)w * kSellRows;
      require(tot < (int64_t)INT32_MAX, IK_EINVAL, "pattern too large for int32 block slots");
      sstart[s + 1] = (int32_t)tot;
    }
  }
  h->nsell = sstart[nslices];
  h->hpos.clear();
  h->hpos.resize(h->nnzb);  // every block gets its slot below
  HostVec<int32_t> scol(h->nsell);
  parallelChunks(nslices, [&](int64_t s0, int64_t s1, int64_t) {
    for (int64_t s = s0; s < s1; ++s) {
      const int32_t w = (sstart[s + 1] - sstart[s]) / kSellRows;
      for (int r = 0; r < kSellRows; ++r) {
        const int64_t i = s * kSellRows + r;
        const int32_t len = i < nn ? h->hrowptr[i + 1] - h->hrowptr[i] : 0;
        for (int32_t j = 0; j < w; ++j) {
          const int32_t slot = sstart[s] + j * kSellRows + r;
          if (j < len) {
            h->hpos[h->hrowptr[i] + j] = slot;
            scol[slot]                 = h->hcolidx[h->hrowptr[i] + j];
          } else {
            scol[slot] = (int32_t)std::min(i, nn - 1);
          }
        }
      }
    }
  }, 32);
  {
    // every block in its row's slice, at a slot of its own holding its column (slices are disjoint slot ranges,
    // so each thread marks only its own slices' slots)
    HostVec<uint8_t> seen = filled<uint8_t>(h->nsell, 0);
    parallelChunks(nslices, [&](int64_t s0, int64_t s1, int64_t) {
      for (int64_t i = s0 * kSellRows; i < std::min(nn, s1 * kSellRows); ++i)
        for (int32_t b = h->hrowptr[i]; b < h->hrowptr[i + 1]; ++b) {
          const int32_t sl = h->hpos[b];
          require(sl >= sstart[i / kSellRows] && sl < sstart[i / kSellRows + 1] && !seen[sl] &&
                      scol[sl] == h->hcolidx[b],
                  IK_EINVAL, "internal error: bad sliced-ELL slot");
          seen[sl] = 1;
        }
    }, 32);
  }
  h->sellStart.upload(sstart.data(), sstart.size(), h->stream);
  h->scol.upload(scol.data(), scol.size(), h->stream);
  // Element e computes its 36 upper blocks (a <= b) sb(a,b) = 8a - a(a-1)/2 + (b-a). Block (node_a, node_b)
  // is an upper block of K when node_a <= node_b and receives the element block as it is; otherwise the
  // upper block (node_b, node_a) receives its transpose. Staging slots are grouped by upper block and
  // ordered by staging unit (tile or element) inside each group, so the gather reads contiguous segments
  // and sums them in a fixed order.
  require((int64_t)ne * 36 < (int64_t)INT32_MAX / 2, IK_EINVAL, "mesh too large for int32 staging slots");
  HostVec<int32_t> slots((size_t)ne * 36);  // block index p of each element block
  parallelChunks(ne, [&](int64_t e0, int64_t e1, int64_t) {
    for (int64_t e = e0; e < e1; ++e)
      for (int a = 0; a < 8; ++a)
        for (int c = a; c < 8; ++c) {
          const int32_t na = conn[e * 8 + a], nc = conn[e * 8 + c];
          const int32_t r = na < nc ? na : nc, col = na < nc ? nc : na;
          const auto b = h->hcolidx.begin() + h->hrowptr[r], en = h->hcolidx.begin() + h->hrowptr[r + 1];
          slots[e * 36 + 8 * a - (a * (a - 1)) / 2 + (c - a)] =
              (int32_t)(std::lower_bound(b, en, col) - h->hcolidx.begin());
        }
  });
  // upper blocks and their transposes
  std::vector<int64_t> uptr(nn + 1, 0);  // first upper block of each row
  for (int64_t i = 0; i < nn; ++i) uptr[i + 1] = uptr[i] + (h->hrowptr[i + 1] - h->hdiag[i]);
  HostVec<int32_t> up(uptr[nn]), upT(uptr[nn]);
  parallelChunks(nn, [&](int64_t i0, int64_t i1, int64_t) {
    for (int64_t i = i0; i < i1; ++i)
      for (int32_t p = h->hdiag[i]; p < h->hrowptr[i + 1]; ++p) {
        const int32_t c = h->hcolidx[p];
        const auto b = h->hcolidx.begin() + h->hrowptr[c], en = h->hcolidx.begin() + h->hrowptr[c + 1];
        const int64_t q = uptr[i] + (p - h->hdiag[i]);
        up[q]           = p;
        upT[q]          = (int32_t)(std::lower_bound(b, en, (int32_t)i) - h->hcolidx.begin());
      }
  });
  const int64_t nup = uptr[nn];
  HostVec<int32_t> qOf = filled<int32_t>(h->nnzb, -1);
  parallelChunks(nup, [&](int64_t q0, int64_t q1, int64_t) {
    for (int64_t q = q0; q < q1; ++q) qOf[up[q]] = (int32_t)q;
  });
  // FULL Dirichlet treatment per upper block: bit 3k+l zeroes entry (k,l), bit 9+k sets a unit diagonal
  HostVec<uint16_t> mask(nup);
  parallelChunks(nn, [&](int64_t i0, int64_t i1, int64_t) {
    for (int64_t i = i0; i < i1; ++i)
      for (int32_t p = h->hdiag[i]; p < h->hrowptr[i + 1]; ++p) {
        const int64_t c = h->hcolidx[p];
        uint16_t m      = 0;
        for (int k = 0; k < 3; ++k)
          for (int l = 0; l < 3; ++l)
            if (h->hfixed[3 * i + k] | h->hfixed[3 * c + l]) {
              m |= (uint16_t)(1u << (3 * k + l));
              if (3 * i + k == 3 * c + l) m |= (uint16_t)(1u << (9 + k));
            }
        mask[uptr[i] + (p - h->hdiag[i])] = m;
      }
  });
  // upper blocks the gather assembles (the rest are written directly)
  HostVec<uint8_t> gathered = filled<uint8_t>(nup, 1);
  HostVec<int64_t> unitOf(ne);  // staging unit of each element: its tile (tiled) or itself
  h->tiled = h->neas == 0;
  int64_t ntiles = 0;
  HostVec<int32_t> tileElem;
  if (h->tiled) {
    // plain element: tiles of kTileElems, consecutive runs of the Morton order (compact boxes), then sorted by
    // their lowest node, so tiles running at the same time write neighbouring parts of the segments.
    const HostVec<int32_t> order = mortonOrder(h);
    ntiles = (ne + kTileElems - 1) / kTileElems;
    std::vector<std::pair<int32_t, int32_t>> tkey(ntiles);  // (lowest node, Morton tile)
    parallelChunks(ntiles, [&](int64_t m0, int64_t m1, int64_t) {
      for (int64_t m = m0; m < m1; ++m) {
        int32_t lo = INT32_MAX;
        for (int64_t i = m * kTileElems; i < std::min(ne, (m + 1) * kTileElems); ++i)
          for (int a = 0; a < 8; ++a) lo = std::min(lo, conn[(int64_t)order[i] * 8 + a]);
        tkey[m] = {lo, (int32_t)m};
      }
    });
    std::sort(tkey.begin(), tkey.end());
    tileElem = filled<int32_t>(ntiles * kTileElems, -1);
    parallelChunks(ntiles, [&](int64_t t0, int64_t t1, int64_t) {
      for (int64_t t = t0; t < t1; ++t) {
        const int64_t m = tkey[t].second;
        for (int64_t i = m * kTileElems; i < std::min(ne, (m + 1) * kTileElems); ++i) {
          tileElem[t * kTileElems + (i - m * kTileElems)] = order[i];
          unitOf[order[i]] = t;
        }
      }
    });
  } else {
    for (int64_t e = 0; e < ne; ++e) unitOf[e] = e;
  }
  const int64_t nunits = h->tiled ? ntiles : ne;
  // Staging chunks (ranges of staging units: tiles, or elements for EAS): a block row is complete once the
  // last unit touching it is staged. With the prefix maximum of that unit index over rows (monotone by
  // construction), rows [0, r) are complete after all units below pm[r-1], so each chunk's gather covers a
  // contiguous row range behind the chunk. Any numbering is correct.
  {
    std::vector<int64_t> last(nn, -1);
    for (int64_t i = 0; i < nn; ++i) {
      for (int64_t k = cnt[i]; k < cnt[i + 1]; ++k) last[i] = std::max(last[i], unitOf[inc(k)]);
      if (i > 0) last[i] = std::max(last[i], last[i - 1]);
    }
    auto cut = [&](int64_t chunk) {
      h->chunkElem.assign(1, 0);
      h->chunkRow.assign(1, 0);
      int64_t r = 0;
      for (int64_t u0 = 0; u0 < nunits; u0 += chunk) {
        const int64_t u1 = std::min(nunits, u0 + chunk);
        if (u1 == nunits)
          r = nn;
        else
          while (r < nn && last[r] < u1) ++r;
        h->chunkElem.push_back(u1);
        h->chunkRow.push_back(r);
      }
    };
    const int64_t given = chunkOverride();
    if (h->tiled) {
      cut(((given ? given : kChunkElements) + kTileElems - 1) / kTileElems);
    } else if (given) {
      cut(given);
    } else {
      const int64_t nc = std::max<int64_t>(1, (ne + kChunkElementsEas / 2) / kChunkElementsEas);
      cut((ne + nc - 1) / nc);
      // in grid order the share of rows complete before the last chunk is close to (nc - 1) / nc, in random order to 0
      if (nc > 1 && h->chunkRow[nc - 1] * 2 * nc < nn * (nc - 1)) cut(ne);
    }
  }
  const int64_t nchunks = (int64_t)h->chunkElem.size() - 1;
  // Gather order of the upper blocks: chunk by chunk (the rows each chunk completes), inside a chunk by storage
  // slot. For a fixed j the rows of a slice have adjacent slots, so the gather's consecutive lanes, and a tile's
  // consecutive groups, write neighbouring slots. Staging segments follow this order; qrank[q] = position of q.
  std::vector<int32_t> qord;
  HostVec<int32_t> qrank = filled<int32_t>(nup, -1);
  std::vector<int64_t> qchunk(nchunks + 1, 0);  // qord[qchunk[c] .. qchunk[c+1]) = upper blocks of chunk c
  {
    HostVec<int32_t> qAtSlot = filled<int32_t>(h->nsell, -1);
    parallelChunks(nup, [&](int64_t q0, int64_t q1, int64_t) {
      for (int64_t q = q0; q < q1; ++q) qAtSlot[h->hpos[up[q]]] = (int32_t)q;
    });
    qord.reserve(nup);
    for (int64_t c = 0; c < nchunks; ++c) {
      const int64_t r0 = h->chunkRow[c], r1 = h->chunkRow[c + 1];
      if (r1 > r0) {
        // the chunk's slices in ranges per thread, each collecting its upper blocks in slot order, then joined
        const int64_t sl0 = r0 / kSellRows, nsl = (r1 - 1) / kSellRows + 1 - sl0;
        std::vector<std::vector<int32_t>> part(chunkCount(nsl, 32));
        parallelChunks(nsl, [&](int64_t a0, int64_t a1, int64_t ch) {
          for (int64_t sl = sl0 + a0; sl < sl0 + a1; ++sl)
            for (int32_t slot = sstart[sl]; slot < sstart[sl + 1]; ++slot) {
              const int32_t q   = qAtSlot[slot];
              const int64_t row = sl * kSellRows + (slot - sstart[sl]) % kSellRows;
              if (q >= 0 && row >= r0 && row < r1) part[ch].push_back(q);
            }
        }, 32);
        for (const auto& v : part) qord.insert(qord.end(), v.begin(), v.end());
      }
      qchunk[c + 1] = (int64_t)qord.size();
    }
    parallelChunks((int64_t)qord.size(), [&](int64_t k0, int64_t k1, int64_t) {
      for (int64_t k = k0; k < k1; ++k) qrank[qord[k]] = (int32_t)k;
    });
    require((int64_t)qord.size() == nup, IK_EINVAL, "internal error: gather order misses upper blocks");
  }
  // staging segment of upper block q: [segBeg[q], segBeg[q] + segCnt[q]), segments laid out in gather order
  HostVec<int32_t> segBeg(nup), segCnt(nup);  // both written for every upper block below
  auto layoutSegments = [&]() {
    HostVec<int64_t> beg;
    parallelPrefix((int64_t)qord.size(), [&](int64_t k) { return (int64_t)segCnt[qord[k]]; }, beg);
    const int64_t tot = beg.back();
    require(tot < (int64_t)INT32_MAX, IK_EINVAL, "mesh too large for int32 staging slots");
    parallelChunks((int64_t)qord.size(), [&](int64_t k0, int64_t k1, int64_t) {
      for (int64_t k = k0; k < k1; ++k) segBeg[qord[k]] = (int32_t)beg[k];
    });
    return tot;
  };
  if (!h->tiled) {
    // EAS: one slot per element block, elements in increasing order inside each segment
    std::vector<int32_t> kcnt(h->nnzb, 0);  // element blocks per K block
    for (const int32_t p : slots) kcnt[p]++;
    for (int64_t q = 0; q < nup; ++q) segCnt[q] = kcnt[up[q]];
    h->nstage = layoutSegments();
    std::vector<int32_t> dest((size_t)ne * 36);
    std::vector<int32_t> pos(segBeg.begin(), segBeg.end());
    for (int64_t e = 0; e < ne; ++e)
      for (int a = 0; a < 8; ++a)
        for (int c = a; c < 8; ++c) {
          const int sb    = 8 * a - (a * (a - 1)) / 2 + (c - a);
          const int32_t q = qOf[slots[e * 36 + sb]];
          const bool tr   = conn[e * 8 + a] > conn[e * 8 + c];
          dest[e * 36 + sb] = (pos[q]++ << 1) | (tr ? 1 : 0);
        }
    for (int64_t q = 0; q < nup; ++q)
      require(pos[q] == segBeg[q] + segCnt[q], IK_EINVAL, "internal error: staging segments do not tile the slots");
    h->bdest.upload(dest.data(), dest.size(), h->stream);
  } else {
    // per tile: the entries j = 36 s + sb that fall on one upper block form a group. The tile adds its entries in LDS
    // in one step: a group of one or two entries has one accumulator (a sum of two does not depend on the order of the
    // adds), a larger group one accumulator per entry, summed in entry order when the group is stored. Groups come with
    // those of one accumulator first (group g: accumulator g), those staged before those written directly, then the
    // others, each kind in the gather order of its upper blocks, i.e. by staging slot and by K slot. epos[t*576 + j]
    // = accumulator | transposed << 15, kNoEntry for padding; gmul = first accumulator | count << 16 of the larger
    // groups, those of tile t at [tmptr[t], tmptr[t+1]); tmaxr[t] = the largest count. Each chunk of tiles lists its
    // groups' upper blocks in its own buffer; tgptr places them. tmeta[4 t ..] = first group, first larger group,
    // single-accumulator groups that are staged | single-accumulator groups << 10 | larger groups << 20, number of
    // accumulators | largest count << 16.
    HostVec<uint16_t> epos((size_t)ntiles * kTileEntries);
    std::vector<uint8_t> tmaxr(ntiles);
    std::vector<int32_t> tgptr(ntiles + 1, 0), tmptr(ntiles + 1, 0);
    HostVec<int32_t> gq;
    HostVec<uint32_t> gmul;
    std::vector<int64_t> tng(ntiles), tnm(ntiles);
    int maxGroups = 0, maxAcc = 0;  // largest numbers of groups and accumulators of a tile
    // a tile's upper blocks -> group: open-addressing table of 2048 slots (a tile touches at most 576 upper blocks),
    // a slot valid when its stamp is the current tile
    constexpr int kHash = 2048;
    std::vector<std::vector<int32_t>> gpart(chunkCount(ntiles, 256));
    std::vector<std::vector<uint32_t>> mpart(chunkCount(ntiles, 256));
    parallelChunks(ntiles, [&](int64_t t0, int64_t t1, int64_t ch) {
      std::vector<int32_t> hkey(kHash), hval(kHash), touched;
      std::vector<int32_t> entQ(kTileEntries), cntQ(kTileEntries), accOf(kTileEntries);
      std::vector<int64_t> hstamp(kHash, -1);
      std::vector<uint16_t> entTr(kTileEntries);
      std::vector<int32_t>& out = gpart[ch];
      auto slotOf = [&](int32_t q, int64_t t) {  // the table slot of q in tile t (free or holding q)
        uint32_t k = ((uint32_t)q * 2654435761u) & (kHash - 1);
        while (hstamp[k] == t && hkey[k] != q) k = (k + 1) & (kHash - 1);
        return k;
      };
      for (int64_t t = t0; t < t1; ++t) {
        touched.clear();
        int nvalid = 0;
        for (int s = 0; s < kTileElems; ++s) {
          const int32_t e = tileElem[t * kTileElems + s];
          if (e < 0) continue;
          ++nvalid;
          for (int a = 0; a < 8; ++a)
            for (int c = a; c < 8; ++c) {
              const int sb    = 8 * a - (a * (a - 1)) / 2 + (c - a);
              const int j     = 36 * s + sb;
              const int32_t q = qOf[slots[(int64_t)e * 36 + sb]];
              entQ[j]         = q;
              entTr[j]        = conn[(int64_t)e * 8 + a] > conn[(int64_t)e * 8 + c] ? 0x8000u : 0u;
              const uint32_t k = slotOf(q, t);
              if (hstamp[k] != t) {
                hstamp[k] = t;
                hkey[k]   = q;
                hval[k]   = 0;
                touched.push_back(q);
              }
              ++hval[k];  // entries of the group
            }
        }
        // gather order: sort the ranks, then map back to upper blocks
        for (auto& q : touched) q = qrank[q];
        std::sort(touched.begin(), touched.end());
        for (auto& q : touched) q = qord[q];
        const int ng = (int)touched.size();
        const int n1 = (int)(std::stable_partition(touched.begin(), touched.end(),
                                                   [&](int32_t q) { return hval[slotOf(q, t)] <= 2; }) -
                             touched.begin());
        int nacc = n1, maxc = 1;
        for (int g = 0; g < ng; ++g) {
          int32_t& v = hval[slotOf(touched[g], t)];
          cntQ[g]    = v;
          v          = g;
          accOf[g]   = g < n1 ? g : nacc;
          if (g >= n1) {
            mpart[ch].push_back((uint32_t)nacc | (uint32_t)cntQ[g] << 16);
            nacc += cntQ[g];
            maxc = std::max(maxc, (int)cntQ[g]);
          }
        }
        uint16_t* ep = epos.data() + t * kTileEntries;
        for (int j = 0; j < kTileEntries; ++j) {
          if (j >= 36 * nvalid) {
            ep[j] = kNoEntry;
            continue;
          }
          const int g = hval[slotOf(entQ[j], t)];
          ep[j]       = (uint16_t)(accOf[g] | entTr[j]);
          if (g >= n1) ++accOf[g];
        }
        tmaxr[t] = (uint8_t)maxc;
        tnm[t]   = ng - n1;
        out.insert(out.end(), touched.begin(), touched.end());
        tng[t] = ng;
      }
    }, 256);
    {
      int64_t tot = 0;
      for (int64_t t = 0; t < ntiles; ++t) {
        tot += tng[t];
        maxGroups = std::max(maxGroups, (int)tng[t]);
        tmptr[t + 1] = tmptr[t] + (int32_t)tnm[t];
        require(tot < (int64_t)INT32_MAX, IK_EINVAL, "mesh too large for int32 staging slots");
        tgptr[t + 1] = (int32_t)tot;
      }
      gq.resize(tot);
      gmul.resize(tmptr[ntiles]);
      for (int64_t t = 0; t < ntiles; ++t) maxAcc = std::max(maxAcc, (int)(tng[t] - tnm[t]));
      parallelChunks(ntiles, [&](int64_t t0, int64_t, int64_t ch) {  // the same chunks as the loop above
        std::copy(gpart[ch].begin(), gpart[ch].end(), gq.begin() + tgptr[t0]);
        std::copy(mpart[ch].begin(), mpart[ch].end(), gmul.begin() + tmptr[t0]);
      }, 256);
    }
    // An upper block that only one tile touches is complete after that tile's group sum, which the tile
    // writes straight into K (with the FULL mask and the mirror block). The others are staged, in gather
    // order: segments in the order qord, each ordered by tile. gdst[g] = slot, or -(K block + 1) with
    // gpt[g] = the mirror block and gmsk[g] = the mask of a direct group.
    HostVec<int32_t> ntile = filled<int32_t>(nup, 0);
    parallelChunks((int64_t)gq.size(), [&](int64_t g0, int64_t g1, int64_t) {
      for (int64_t g = g0; g < g1; ++g) __atomic_fetch_add(&ntile[gq[g]], 1, __ATOMIC_RELAXED);
    });
    parallelChunks(nup, [&](int64_t q0, int64_t q1, int64_t) {
      for (int64_t q = q0; q < q1; ++q) {
        gathered[q] = ntile[q] > 1;
        segCnt[q]   = gathered[q] ? ntile[q] : 0;
      }
    });
    // the staged ones of a tile's single-accumulator groups move in front of the directly written ones
    std::vector<int32_t> tns(ntiles);
    parallelChunks(ntiles, [&](int64_t t0, int64_t t1, int64_t) {
      std::vector<int32_t> perm(kTileEntries), old(kTileEntries);
      for (int64_t t = t0; t < t1; ++t) {
        int32_t* g   = gq.data() + tgptr[t];
        const int n1 = (int)(tng[t] - tnm[t]);
        int at       = 0;
        std::copy(g, g + n1, old.begin());
        for (int pass = 0; pass < 2; ++pass) {
          for (int j = 0; j < n1; ++j)
            if ((gathered[old[j]] != 0) == (pass == 0)) {
              perm[j] = at;
              g[at++] = old[j];
            }
          if (pass == 0) tns[t] = at;
        }
        uint16_t* ep = epos.data() + t * kTileEntries;
        for (int j = 0; j < kTileEntries; ++j)
          if (ep[j] != kNoEntry && (ep[j] & 0x7FFF) < n1) ep[j] = (uint16_t)(perm[ep[j] & 0x7FFF] | (ep[j] & 0x8000));
      }
    });
    h->nstage = layoutSegments();
    // A staged group's slot is its upper block's segment start plus its rank among that block's groups by
    // increasing group index (= tile order). Groups are dropped into their segment through a per-block cursor
    // (any order), each segment (at most 8 groups: one per tile touching the block) is then sorted, and the
    // k-th group of segment q gets slot segBeg[q] + k. A direct group stores -(K slot + 1), its mirror's K
    // slot and its FULL mask.
    const int64_t ngq = (int64_t)gq.size();
    HostVec<int32_t> gdst(ngq), gpt(ngq), cursor = filled<int32_t>(nup, 0), segG(h->nstage);
    HostVec<uint16_t> gmsk(ngq);
    parallelChunks(ngq, [&](int64_t g0, int64_t g1, int64_t) {
      for (int64_t g = g0; g < g1; ++g) {
        const int32_t q = gq[g];
        if (gathered[q]) {
          segG[segBeg[q] + __atomic_fetch_add(&cursor[q], 1, __ATOMIC_RELAXED)] = (int32_t)g;
          gpt[g]  = 0;
          gmsk[g] = 0;
        } else {
          gdst[g] = -(h->hpos[up[q]] + 1);
          gpt[g]  = h->hpos[upT[q]];
          gmsk[g] = mask[q];
        }
      }
    });
    parallelChunks(nup, [&](int64_t q0, int64_t q1, int64_t) {
      for (int64_t q = q0; q < q1; ++q) {
        if (!gathered[q]) continue;
        require(cursor[q] == segCnt[q], IK_EINVAL, "internal error: staging segment not filled");
        int32_t* b = segG.data() + segBeg[q];
        std::sort(b, b + segCnt[q]);
        for (int32_t k = 0; k < segCnt[q]; ++k) gdst[b[k]] = segBeg[q] + k;
      }
    });
    // the kernel's indexing relies on these: in every tile the accumulators of the single-accumulator groups come first
    // and get one or two entries each, those of the other groups follow without gaps and get one each, all below
    // maxAcc; the slots are a permutation of [0, nstage) with each group inside its own upper block's segment (the
    // segments are disjoint consecutive ranges, each filled exactly by its cursor), and every upper block is either
    // staged by two or more tiles or written by exactly one
    for (int64_t t = 0; t < ntiles; ++t)
      if (tmptr[t + 1] > tmptr[t]) {
        const uint32_t m = gmul[tmptr[t + 1] - 1];
        maxAcc           = std::max(maxAcc, (int)((m & 0xFFFFu) + (m >> 16)));
      }
    {
      parallelChunks(nup, [&](int64_t q0, int64_t q1, int64_t) {
        for (int64_t q = q0; q < q1; ++q)
          require(ntile[q] >= 1 && segCnt[q] == (gathered[q] ? ntile[q] : 0) &&
                      cursor[q] == (gathered[q] ? segCnt[q] : 0),
                  IK_EINVAL, "internal error: upper block without a tile or a segment not filled");
      });
      parallelChunks((int64_t)gq.size(), [&](int64_t g0, int64_t g1, int64_t) {
        for (int64_t g = g0; g < g1; ++g) {
          const int32_t sl = gdst[g], q = gq[g];
          if (sl < 0)
            require(!gathered[q] && -sl - 1 == h->hpos[up[q]] && gpt[g] == h->hpos[upT[q]], IK_EINVAL,
                    "internal error: bad direct group");
          else
            require(sl >= segBeg[q] && sl < segBeg[q] + segCnt[q], IK_EINVAL,
                    "internal error: staging slot outside its segment");
        }
      });
      parallelChunks(ntiles, [&](int64_t t0, int64_t t1, int64_t) {
        std::vector<int32_t> fill(kTileEntries);  // entries per accumulator
        for (int64_t t = t0; t < t1; ++t) {
          const int ng = tgptr[t + 1] - tgptr[t], nm = tmptr[t + 1] - tmptr[t], n1 = ng - nm;
          int nvalid = 0;
          while (nvalid < kTileElems && tileElem[t * kTileElems + nvalid] >= 0) ++nvalid;
          for (int s = nvalid; s < kTileElems; ++s)
            require(tileElem[t * kTileElems + s] < 0, IK_EINVAL, "internal error: bad tile padding");
          require(nvalid >= 1 && ng >= 1 && n1 >= 0 && ng <= 36 * nvalid && ng <= maxGroups, IK_EINVAL,
                  "internal error: bad tile");
          int nacc = n1;
          for (int m = 0; m < nm; ++m) {
            const uint32_t v = gmul[tmptr[t] + m];
            require((int)(v & 0xFFFFu) == nacc && (v >> 16) >= 3 && (v >> 16) <= tmaxr[t], IK_EINVAL,
                    "internal error: bad tile accumulators");
            nacc += (int)(v >> 16);
          }
          require(nacc <= maxAcc && nacc <= kTileEntries && tns[t] <= n1, IK_EINVAL,
                  "internal error: bad tile accumulators");
          for (int g = 0; g < n1; ++g)
            require((gdst[tgptr[t] + g] >= 0) == (g < tns[t]), IK_EINVAL, "internal error: bad tile group order");
          std::fill(fill.begin(), fill.begin() + nacc, 0);
          const uint16_t* ep = epos.data() + t * kTileEntries;
          for (int j = 0; j < kTileEntries; ++j) {
            if (j >= 36 * nvalid) {
              require(ep[j] == kNoEntry, IK_EINVAL, "internal error: bad padding entry");
              continue;
            }
            const int g = ep[j] & 0x7FFF;
            require(g < nacc && ++fill[g] <= (g < n1 ? 2 : 1), IK_EINVAL, "internal error: bad tile entry");
          }
          for (int g = 0; g < nacc; ++g) require(fill[g] >= 1, IK_EINVAL, "internal error: empty tile accumulator");
        }
      });
    }
    h->ntiles = ntiles;
    h->tileElem.upload(tileElem.data(), tileElem.size(), h->stream);
    h->gdst.upload(gdst.data(), gdst.size(), h->stream);
    h->gpt.upload(gpt.data(), gpt.size(), h->stream);
    h->gmsk.upload(gmsk.data(), gmsk.size(), h->stream);
    h->epos.upload(epos.data(), epos.size(), h->stream);
    HostVec<int32_t> tmeta(ntiles * 4), tileNode(ntiles * kTileElems * 8);
    std::atomic<int64_t> direct{0}, adjacent{0};
    parallelChunks(ntiles, [&](int64_t t0, int64_t t1, int64_t) {
      int64_t nd = 0, na = 0;
      for (int64_t t = t0; t < t1; ++t) {
        for (int32_t g = tgptr[t], at = 1; g < tgptr[t + 1]; ++g)
          if (gdst[g] < 0) {  // -(slot + 1)
            ++nd;
            na += gdst[g] + 1 == at;
            at = gdst[g];
          }
        const int32_t ng = tgptr[t + 1] - tgptr[t], nm = tmptr[t + 1] - tmptr[t];
        const uint32_t m = nm ? gmul[tmptr[t + 1] - 1] : (uint32_t)ng;  // the last accumulators
        tmeta[4 * t]     = tgptr[t];
        tmeta[4 * t + 1] = tmptr[t];
        tmeta[4 * t + 2] = tns[t] | (ng - nm) << 10 | nm << 20;
        tmeta[4 * t + 3] = (int32_t)((m & 0xFFFFu) + (m >> 16)) | (int32_t)tmaxr[t] << 16;
        // node of corner q of slot s (padding slots repeat slot 0): what the kernel's lanes load first
        for (int s = 0; s < kTileElems; ++s) {
          const int32_t e = tileElem[t * kTileElems + s];
          std::copy_n(conn + (int64_t)(e >= 0 ? e : tileElem[t * kTileElems]) * 8, 8,
                      &tileNode[(t * kTileElems + s) * 8]);
        }
      }
      direct += nd;
      adjacent += na;
    });
    h->adjacent = direct ? (double)adjacent / (double)direct : 0.0;
    h->tmeta.upload(tmeta.data(), tmeta.size(), h->stream);
    h->tileNode.upload(tileNode.data(), tileNode.size(), h->stream);
    h->gmul.upload(gmul.data(), gmul.size(), h->stream);
    h->tgptr = std::move(tgptr);
    h->tmaxr = std::move(tmaxr);
    h->maxGroups = maxGroups;
    h->maxAcc    = maxAcc;
  }
  // the gather's upper blocks: the gathered ones in gather order (chunkQ[c]: first one of chunk c), placed by
  // a prefix count over qord; each one's segment must start where the previous one's ends
  {
    HostVec<int64_t> at;
    parallelPrefix(nup, [&](int64_t k) { return (int64_t)gathered[qord[k]]; }, at);
    const int64_t ng = at[nup];
    HostVec<int32_t> cup(ng), cupT(ng), cseg(ng + 1);
    HostVec<uint16_t> cmask(ng);
    cseg[0] = 0;
    parallelChunks(nup, [&](int64_t k0, int64_t k1, int64_t) {
      for (int64_t k = k0; k < k1; ++k) {
        const int32_t q = qord[k];
        if (!gathered[q]) continue;
        const int64_t i = at[k];
        cup[i]          = h->hpos[up[q]];
        cupT[i]         = h->hpos[upT[q]];
        cmask[i]        = mask[q];
        cseg[i + 1]     = segBeg[q] + segCnt[q];
      }
    });
    parallelChunks(nup, [&](int64_t k0, int64_t k1, int64_t) {
      for (int64_t k = k0; k < k1; ++k)
        if (gathered[qord[k]])
          require(segBeg[qord[k]] == cseg[at[k]], IK_EINVAL, "internal error: gather segments not contiguous");
    });
    h->chunkQ.assign(nchunks + 1, 0);
    for (int64_t c = 0; c < nchunks; ++c) h->chunkQ[c + 1] = at[qchunk[c + 1]];
    h->upMask.upload(cmask.data(), cmask.size(), h->stream);
    h->upBlk.upload(cup.data(), cup.size(), h->stream);
    h->upT.upload(cupT.data(), cupT.size(), h->stream);
    h->segptr.upload(cseg.data(), cseg.size(), h->stream);
  }
  std::vector<int32_t> ncnt(nn + 1, 0);
  for (int64_t i = 0; i <= nn; ++i) ncnt[i] = (int32_t)cnt[i];
  h->rowptr.upload(h->hrowptr.data(), h->hrowptr.size(), h->stream);  // colidx: uploaded when ik_matrix_bsr asks
  {
    std::vector<int32_t> dslot(nn);
    for (int64_t i = 0; i < nn; ++i) dslot[i] = h->hpos[h->hdiag[i]];
    h->diagBlk.upload(dslot.data(), dslot.size(), h->stream);
  }
  // residual staging slot of every element corner (residualSlot of its rank in the node's incidence list)
  HostVec<int32_t> rdest((size_t)ne * 8);
  const int64_t tail = residualTail(nn);
  std::atomic<bool> anyTail{false};
  parallelChunks(nn, [&](int64_t i0, int64_t i1, int64_t) {
    bool any = false;
    for (int64_t i = i0; i < i1; ++i)
      for (int64_t j = cnt[i]; j < cnt[i + 1]; ++j) {
        const int64_t rank = j - cnt[i];
        any |= rank >= kResidualRanks;
        rdest[nlist[j]] = (int32_t)(rank < kResidualRanks ? residualSlot(i, rank) : tail + j);
      }
    if (any) anyTail = true;
  });
  h->rslots = tail + (anyTail ? ne * 8 : 0);
  require(h->rslots <= INT32_MAX, IK_EINVAL, "internal error: too many residual staging slots");
  h->ncptr.upload(ncnt.data(), ncnt.size(), h->stream);
  h->rdest.upload(rdest.data(), rdest.size(), h->stream);
  IK_HIP(hipStreamSynchronize(h->stream));
  h->patternBuilt = true;
}

}  // namespace ik
