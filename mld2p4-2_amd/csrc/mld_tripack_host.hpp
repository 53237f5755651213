// The packed triangular factors of mld_tripack.hpp: their layout, and the host
// code that forms them.
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

#include "mld_host.hpp"

namespace mld {
namespace tp {

constexpr int TP_NW = 12;                 // wavefronts
constexpr int TP_T = 64 * TP_NW;
constexpr int TP_KE = 16;                 // entries of a row in registers that are summed ahead of its group
constexpr int TP_KL = 24;                 // and behind the barrier
constexpr int TP_LDS = 160 * 1024;        // the whole LDS of a CU

// Rows whose solution the LDS window holds; behind them a constant zero, which
// padding entries point to, and a slot that nobody reads.
template <typename V>
constexpr int tp_w() { return (TP_LDS - 64) / (int)sizeof(V) < 32766 ? (TP_LDS - 64) / (int)sizeof(V) : 32766; }
template <typename V>
constexpr int tp_vpc() { return 16 / (int)sizeof(V); }  // values of a 16-byte chunk

struct SliceHdr {
  uint32_t off;   // data offset, 16-byte units
  int32_t p;      // first position
  int32_t g;      // group
  uint32_t shape; // 15 bits: p mod window; 6: rows - 1; 3: chunks of 4 entries summed ahead; 8: chunks
};

template <typename V>
struct Packed {
  bigvec<unsigned char> bytes;       // slice data
  std::vector<SliceHdr> hdr;         // slices of wavefront 0, of wavefront 1, ...; each list ends with two of group ngroups
  std::vector<int> first;            // TP_NW + 1 starts in hdr
  std::vector<int> rows;             // position -> row
  int ngroups = 0;
};

// Data bytes of a slice: columns (slots) in chunks of 4, values in 16-byte
// chunks (rows padded to 4 entries), both chunk-major over the rows, then the
// diagonal.
template <typename V>
static inline size_t tp_slice_bytes(int m, int w) {
  const size_t c = (w + 3) / 4, q = c * 4 / tp_vpc<V>();
  return (c * m * 8 + 15) / 16 * 16 + q * m * 16 + (sizeof(V) * m + 15) / 16 * 16;
}

// The packed form of factor f (level sets ptr / rows), diagonal d (null: none
// is read).  False when a dependency lies outside the window, a row is too
// long, or the stream takes longer than the waits it saves.
template <typename V>
bool tp_pack(const HCsr& f, const std::vector<int>& ptr, const std::vector<int>& srows, const double* d,
             Packed<V>& out);
extern template bool tp_pack<float>(const HCsr&, const std::vector<int>&, const std::vector<int>&, const double*,
                                    Packed<float>&);
extern template bool tp_pack<double>(const HCsr&, const std::vector<int>&, const std::vector<int>&, const double*,
                                     Packed<double>&);

}  // namespace tp
}  // namespace mld
