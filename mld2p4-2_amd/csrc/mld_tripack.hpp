// Triangular substitution by one workgroup over a packed stream.  The level
// sets of a factor are narrow (tens to a few hundred rows) and depend on each
// other, so the time of a solve is its chain, not its bytes.  Here the chain
// stays inside one CU: the solution of the last tp_w() rows lives in LDS, and
// a level set costs an LDS round trip, a few additions and a barrier.
//
// Rows are taken in level-schedule order (inside a level set the longest
// first) and cut into slices of at most 64 rows, one row per lane.  A group is
// what happens between two barriers: the slices of a level set, each on a
// wavefront of its own.  Slices go to the TP_NW wavefronts in turn, so every
// wavefront has the time of several groups to bring its next slice's entries
// from memory into registers (12 wavefronts with up to 10 KB each in flight),
// and to sum, in order, the leading entries that no row of the group before
// theirs is gathered for (a row's latest neighbours are mostly its last ones).
// Between two barriers stand only the remaining gathers, products and additions
// and one LDS store.
//
// FP64 on MI355X, per level set: Gauss-Seidel on a 301 x 301 grid (150 rows of
// 2 entries) 1.65 -> 0.34 us, its first coarse level (32 rows of 4) 1.35 ->
// 0.28 us; ILU(0) on the first coarse level of a 96^3 grid (127 rows of 15)
// 1.53 -> 0.70 us forward and 0.50 backward, and of a 64^2 grid in one workgroup
// with row lists (trsv_run_kernel) 1.0 -> 0.28 us.  What is left is the chain: an
// LDS store, barrier and read take 134-176 cycles, an addition 8, a division 76;
// the wavefronts wait for 82 % of their cycles.  Not the bytes: 20.7 MB of that
// factor pass at 35-50 GB/s, where one CU streams 95-117.  The sums ahead gain
// nothing there (forward 588 us with 7.6 of 18.8 entries per row ahead, 418 with
// none) nor on the 2-D grids (1 %).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mld_kernels.hpp"
#include "mld_tripack_host.hpp"

namespace mld {
namespace tp {

// --------------------------------------------------------------- kernels
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// A barrier that waits for no load or store in flight to memory, as
// __syncthreads would: lds_arrive after an LDS store that the others read
// next, lds_pass where this wavefront has none.
__device__ __forceinline__ void lds_arrive() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void lds_pass() { asm volatile("s_barrier" ::: "memory"); }

// One packed solve in place: bt holds the right-hand side in position order
// and receives the solution.  SC as in tri_row: 0 unit diagonal, 1 t = d b -
// acc, 2 t = (b - acc) / d; per row the products are added in stored order,
// so the values are those of the other substitutions bit for bit.
template <typename V, int SC>
__global__ __launch_bounds__(TP_T, 1) void tripack_kernel(int ngroups, const unsigned char* __restrict__ pk,
                                                          const SliceHdr* __restrict__ hdr,
                                                          const int* __restrict__ first, V* bt) {
  constexpr int W = tp_w<V>();
  constexpr int VPC = tp_vpc<V>();
  constexpr int CPQ = 4 / VPC;  // value chunks of 4 entries
  typedef V vchunk __attribute__((ext_vector_type(VPC)));
  __shared__ __align__(16) V ring[W + 2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) ring[W] = (V)0;

  const u32x4* hp = (const u32x4*)hdr + first[wave];
  // this wavefront's next slice: its entries in registers, those summed ahead
  // (ev, ec) apart from those that wait for the group before (lv, lc)
  int p = 0, m = 0, ke = 0, nc = 0, slot0 = 0, sg = 0;
  unsigned off = 0;
  vchunk ev[TP_KE / VPC] = {}, lv[TP_KL / VPC] = {};
  u32x2 ec[TP_KE / 4] = {}, lc[TP_KL / 4] = {};
  V dcur = (V)1, bcur = (V)0, acc = (V)0;
  u32x4 nh = hp[0];
  auto load_slice = [&]() __attribute__((always_inline)) {
    off = __builtin_amdgcn_readfirstlane(nh.x);
    p = __builtin_amdgcn_readfirstlane(nh.y);
    sg = __builtin_amdgcn_readfirstlane(nh.z);
    const unsigned shape = __builtin_amdgcn_readfirstlane(nh.w);
    slot0 = (int)(shape & 0x7fffu);
    m = (int)((shape >> 15) & 63u) + 1;
    ke = (int)((shape >> 21) & 7u);
    nc = (int)(shape >> 24);
    nh = *++hp;
    const unsigned l = (unsigned)min(lane, m - 1);
    const unsigned char* c = pk + (size_t)off * 16;
    const unsigned char* v = c + (nc * m * 8 + 15) / 16 * 16;
    if constexpr (SC > 0) dcur = *(const V*)(v + nc * CPQ * m * 16 + l * (unsigned)sizeof(V));
    bcur = *(const V*)((const unsigned char*)(bt + p) + l * (unsigned)sizeof(V));
#pragma unroll
    for (int q = 0; q < TP_KE / 4; ++q) {
      if (q >= ke) break;
      ec[q] = *(const u32x2*)(c + l * 8);
      c += m * 8;
#pragma unroll
      for (int e = 0; e < CPQ; ++e) {
        ev[q * CPQ + e] = *(const vchunk*)(v + l * 16);
        v += m * 16;
      }
    }
#pragma unroll
    for (int q = 0; q < TP_KL / 4; ++q) {
      if (q >= nc - ke) break;
      lc[q] = *(const u32x2*)(c + l * 8);
      c += m * 8;
#pragma unroll
      for (int e = 0; e < CPQ; ++e) {
        lv[q * CPQ + e] = *(const vchunk*)(v + l * 16);
        v += m * 16;
      }
    }
  };
  // acc = the C leading entries of every row, in order
  auto ahead = [&](auto cc) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    V t[C + 1];
#pragma unroll
    for (int q = 0; q < C / 4; ++q) {
      t[4 * q] = ring[ec[q].x & 0xffffu];
      t[4 * q + 1] = ring[ec[q].x >> 16];
      t[4 * q + 2] = ring[ec[q].y & 0xffffu];
      t[4 * q + 3] = ring[ec[q].y >> 16];
    }
    acc = (V)0;
#pragma unroll
    for (int k = 0; k < C; ++k) acc = acc + ev[k / VPC][k % VPC] * t[k];
    // keeps the cases of the switch apart: with their common ends merged the
    // compiler (ROCm 7.2) has left columns of the longer case undefined
    // (tests/test_gpu_packed_cases.py runs every pair of cases)
    asm volatile("; ahead %0" ::"n"(C));
  };
  // The rest of the slice: what can be done before the barrier is, so that
  // behind it stand the gathers of the C late entries, the additions and the
  // store.  wait: the group before this one is still open.
  auto finish = [&](auto cc, bool wait) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    unsigned ad[C + 1];
#pragma unroll
    for (int q = 0; q < C / 4; ++q) {
      ad[4 * q] = (lc[q].x & 0xffffu) * (unsigned)sizeof(V);
      ad[4 * q + 1] = (lc[q].x >> 16) * (unsigned)sizeof(V);
      ad[4 * q + 2] = (lc[q].y & 0xffffu) * (unsigned)sizeof(V);
      ad[4 * q + 3] = (lc[q].y >> 16) * (unsigned)sizeof(V);
    }
    int so = slot0 + lane;
    if (so >= W) so -= W;
    so = (lane < m) ? so : W + 1;  // (lanes without a row store behind the zero slot)
    const V bi = (SC == 1) ? dcur * bcur : bcur;
    V s = acc;
    if (wait) lds_pass();
    V t[C + 1];
#pragma unroll
    for (int k = 0; k < C; ++k) t[k] = *(const V*)((const char*)ring + ad[k]);
#pragma unroll
    for (int k = 0; k < C; ++k) s = s + lv[k / VPC][k % VPC] * t[k];
    if constexpr (C == TP_KL) {  // the rest of longer rows, from memory
      const unsigned l = (unsigned)min(lane, m - 1);
      const unsigned char* c = pk + (size_t)off * 16;
      const unsigned char* v = c + (nc * m * 8 + 15) / 16 * 16;
      for (int q = ke + TP_KL / 4; q < nc; ++q) {
        const u32x2 x = *(const u32x2*)(c + q * m * 8 + l * 8);
        V u[4];
        u[0] = ring[x.x & 0xffffu];
        u[1] = ring[x.x >> 16];
        u[2] = ring[x.y & 0xffffu];
        u[3] = ring[x.y >> 16];
#pragma unroll
        for (int e = 0; e < CPQ; ++e) {
          const vchunk z = *(const vchunk*)(v + (q * CPQ + e) * m * 16 + l * 16);
#pragma unroll
          for (int k = 0; k < VPC; ++k) s = s + z[k] * u[e * VPC + k];
        }
      }
    }
    V ti;
    if constexpr (SC == 2) ti = (bi - s) / dcur;
    else ti = bi - s;
    ring[so] = ti;
    lds_arrive();
    if (lane < m) bt[p + lane] = ti;
    asm volatile("; late %0" ::"n"(C));
  };
  static_assert(TP_KE == 16 && TP_KL == 24, "the cases below");
  load_slice();
  lds_arrive();
  int g = 0;  // groups closed
  while (sg < ngroups) {
    const bool wait = (g < sg);
    for (; g + 1 < sg; ++g) lds_pass();
    switch (ke) {
      case 0: ahead(std::integral_constant<int, 0>()); break;
      case 1: ahead(std::integral_constant<int, 4>()); break;
      case 2: ahead(std::integral_constant<int, 8>()); break;
      case 3: ahead(std::integral_constant<int, 12>()); break;
      default: ahead(std::integral_constant<int, 16>()); break;
    }
    switch (min(nc - ke, TP_KL / 4)) {
      case 0: finish(std::integral_constant<int, 0>(), wait); break;
      case 1: finish(std::integral_constant<int, 4>(), wait); break;
      case 2: finish(std::integral_constant<int, 8>(), wait); break;
      case 3: finish(std::integral_constant<int, 12>(), wait); break;
      case 4: finish(std::integral_constant<int, 16>(), wait); break;
      case 5: finish(std::integral_constant<int, 20>(), wait); break;
      default: finish(std::integral_constant<int, 24>(), wait); break;
    }
    g = sg + 1;
    load_slice();
  }
  for (; g < ngroups; ++g) lds_pass();
}

// b in position order: o[p] = b[idx[p]]
template <typename V>
__global__ __launch_bounds__(256) void tripack_in(int n, const int* __restrict__ idx, const V* __restrict__ b,
                                                  V* __restrict__ o) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p < n) o[p] = b[idx[p]];
}
// the solution back in row order: t (when not null) and y = s, y += s
template <typename V, int BETA>
__global__ __launch_bounds__(256) void tripack_out(int n, const int* __restrict__ pos, const V* __restrict__ s,
                                                   V* __restrict__ t, V* __restrict__ y) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const V v = s[pos[i]];
  if (t) t[i] = v;
  if (BETA == 1) y[i] = y[i] + v;
  else if (BETA == 0) y[i] = v;
}

}  // namespace tp
}  // namespace mld
