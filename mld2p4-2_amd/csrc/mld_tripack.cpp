// Packed triangular factors (see mld_tripack.hpp): formed on the host.
#include <omp.h>

#include <algorithm>
#include <cstring>

#include "mld_tripack_host.hpp"

namespace mld {
namespace tp {

// The line in tp_pack: a stream at the 90 GB/s of one CU against the sync-free
// form, which spends 1.3 to 1.65 us on a level set of these widths and spreads
// the bytes over the whole GPU, so it lies at 1.2 us of stream per level set
// (the first coarse level of a 256^3 grid, 905 rows of 15 entries per level
// set, stays sync-free: 3.3 ms of stream against 3.7 ms).
// Level sets, then slices, are shared among the host threads: both factors of
// 105 692 rows of 15 entries (20.7 MB each), with their upload, 29 -> 9 ms
// against one thread per factor.
template <typename V>
bool tp_pack(const HCsr& f, const std::vector<int>& ptr, const std::vector<int>& srows, const double* d,
             Packed<V>& out) {
  const int n = f.nr, nlev = (int)ptr.size() - 1;
  constexpr int W = tp_w<V>();
  if (n <= 0 || nlev <= 0) return false;
  const double us = ((double)f.nnz() * (sizeof(V) + 2) * 1.2 + (double)n * (2 * sizeof(V))) / 90e3;
  if (us > 1.2 * nlev) return false;
  auto len = [&](int r) { return (int)(f.irp[r + 1] - f.irp[r]); };
  // inside a level set the longest rows first, others in their order
  std::vector<int> pos(n);
  std::vector<int64_t> key(n);
  out.rows.resize(n);
  const int* rows = out.rows.data();
  const int nt = std::max(1, std::min(omp_get_max_threads(), n / 4096));
  bool bad = false;
#pragma omp parallel for schedule(static) num_threads(nt) reduction(|| : bad)
  for (int l = 0; l < nlev; ++l) {
    for (int p = ptr[l]; p < ptr[l + 1]; ++p) {
      bad = bad || len(srows[p]) > 1000;
      key[p] = -(int64_t)len(srows[p]) * ((int64_t)1 << 32) + p;
    }
    std::sort(key.begin() + ptr[l], key.begin() + ptr[l + 1]);
    for (int p = ptr[l]; p < ptr[l + 1]; ++p) {
      const int r = srows[(int)(key[p] & 0xffffffff)];
      out.rows[p] = r;
      pos[r] = p;
    }
  }
  if (bad) return false;
  // the window: a row reads slots of positions that no row of its level set,
  // or of an earlier one, has taken since
#pragma omp parallel for schedule(static) num_threads(nt) reduction(|| : bad)
  for (int l = 0; l < nlev; ++l)
    for (int p = ptr[l]; p < ptr[l + 1] && !bad; ++p) {
      const int r = rows[p];
      for (int64_t k = f.irp[r]; k < f.irp[r + 1]; ++k)
        bad = bad || pos[f.ja[k]] >= ptr[l] || ptr[l + 1] - 1 - pos[f.ja[k]] >= W;
    }
  if (bad) return false;
  // slices and groups: where each begins
  struct Slice {
    size_t base;
    int p, m, g;
  };
  std::vector<Slice> sl;
  std::vector<int> gg(n);  // position -> group
  size_t bytes = 0;
  int G = -1;
  for (int l = 0; l < nlev; ++l) {
    int ingroup = TP_NW;
    for (int p = ptr[l]; p < ptr[l + 1];) {
      if (ingroup == TP_NW) {
        ++G;
        ingroup = 0;
      }
      const int m = std::min(64, ptr[l + 1] - p);
      if (bytes / 16 > 0xf0000000ull) return false;
      sl.push_back({bytes, p, m, G});
      bytes += tp_slice_bytes<V>(m, len(rows[p]));
      std::fill(gg.begin() + p, gg.begin() + p + m, G);
      ++ingroup;
      p += m;
    }
  }
  const int64_t ns = (int64_t)sl.size();
  std::vector<std::vector<SliceHdr>> list(TP_NW);
  for (int t = 0; t < TP_NW; ++t) list[t].resize((size_t)((ns - t + TP_NW - 1) / TP_NW));
  out.bytes.resize(bytes + 64);  // (an ending header's row is read, and not used)
  std::memset(out.bytes.data() + bytes, 0, 64);
#pragma omp parallel for schedule(static) num_threads(nt)
  for (int64_t q = 0; q < ns; ++q) {
    const size_t base = sl[q].base;
    const int p = sl[q].p, m = sl[q].m, g = sl[q].g;
    const int w = len(rows[p]), nc = (w + 3) / 4, nq = nc * 4 / tp_vpc<V>();
    // leading chunks of 4 entries without one from the group before
    int ke = std::min(nc, TP_KE / 4);
    for (int i = p; i < p + m; ++i) {
      const int64_t k0 = f.irp[rows[i]];
      for (int k = 0; k < std::min(4 * ke, len(rows[i])); ++k)
        if (gg[pos[f.ja[k0 + k]]] >= g - 1) ke = k / 4;
    }
    std::memset(out.bytes.data() + base, 0, tp_slice_bytes<V>(m, w));
    uint16_t* col = (uint16_t*)(out.bytes.data() + base);
    V* val = (V*)(out.bytes.data() + base + ((size_t)nc * m * 8 + 15) / 16 * 16);
    V* dd = val + (size_t)nq * m * tp_vpc<V>();
    for (int i = 0; i < m; ++i) {
      const int r = rows[p + i], ln = len(r);
      const int64_t k0 = f.irp[r];
      // padding: -0 times the zero slot is -0, and acc + (-0) = acc
      for (int k = 0; k < nc * 4; ++k) {
        col[((size_t)(k / 4) * m + i) * 4 + k % 4] = (uint16_t)(k < ln ? pos[f.ja[k0 + k]] % W : W);
        val[((size_t)(k / tp_vpc<V>()) * m + i) * tp_vpc<V>() + k % tp_vpc<V>()] = k < ln ? (V)f.val[k0 + k] : (V)-0.0;
      }
      if (d) dd[i] = (V)d[r];
    }
    list[q % TP_NW][(size_t)(q / TP_NW)] = {
        (uint32_t)(base / 16), p, g,
        (uint32_t)(p % W) | (uint32_t)(m - 1) << 15 | (uint32_t)ke << 21 | (uint32_t)nc << 24};
  }
  out.ngroups = G + 1;
  out.hdr.clear();
  out.first.clear();
  for (const auto& q : list) {
    out.first.push_back((int)out.hdr.size());
    out.hdr.insert(out.hdr.end(), q.begin(), q.end());
    for (int e = 0; e < 2; ++e) out.hdr.push_back({0, 0, out.ngroups, 0});
  }
  out.first.push_back((int)out.hdr.size());
  return true;
}


template bool tp_pack<float>(const HCsr&, const std::vector<int>&, const std::vector<int>&, const double*,
                             Packed<float>&);
template bool tp_pack<double>(const HCsr&, const std::vector<int>&, const std::vector<int>&, const double*,
                              Packed<double>&);

}  // namespace tp
}  // namespace mld
