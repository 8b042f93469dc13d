// Transfers between localisation regions and the global region, in the
// compressed form: psi_to_locreg2 (locregs/locreg_operations.f90:2143-2318)
// and Lpsi_to_global2 (locreg_operations.f90:1665-1837).  The reference walks
// the local segments (shifted into the global box, shift_locreg_indexes,
// :2321-2380) against the global segments; here every local compressed point
// is located through the region map (local grid point + box offset -> global
// grid point -> global compressed index through the inverse map of the
// global region), and every coefficient is one thread: a coarse point moves
// one value, a fine point's seven values are moved by seven consecutive
// threads, so loads and stores of a wave cover contiguous ranges of both
// orbitals.  Same elements, same values, no floating-point arithmetic.
#include "bdft_internal.h"

namespace bdft {

constexpr int XT = 256;        // threads per tile
constexpr int XU = 8;          // coefficients per thread
constexpr int XC = XT * XU;    // coefficients per tile

__device__ __forceinline__ int xfer_find(const XferArgs& A, int tile) {
  int lo = 0, hi = A.nd - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (A.d[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ int xfer_div(int n, unsigned q, int s) {
  return q ? (int)(__umulhi((unsigned)n, q) >> s) : n;
}

// one tile of the coarse (FINE false) or the fine part: coefficient e (fine:
// point e / 7, wavelet t) per thread, XU of them, each of the three dependent
// loads issued for all of them before the next.  A load and a store per
// coefficient, one map and one inverse-map value per point: bound by memory
// once the grid index is split without divisions (two 32-bit divisions per
// coefficient: 24 us instead of 18 for 128 spheres of 42 k coefficients, 86 MB
// moved).
template <bool FINE>
__device__ __forceinline__ void xfer_tile(const XferArgs& A, const XferDesc& D, int e0) {
  const int ne = FINE ? 7 * D.nvctr_f : D.nvctr_c;
  const int* map = FINE ? D.fmap : D.cmap;
  const int* inv = FINE ? A.gfinv : A.gcinv;
  int lin[XU], gi[XU];
#pragma unroll
  for (int u = 0; u < XU; ++u) {
    const int e = min(e0 + u * XT, ne - 1);
    lin[u] = map[FINE ? e / 7 : e];
  }
#pragma unroll
  for (int u = 0; u < XU; ++u) {
    const int r = xfer_div(lin[u], D.q1, D.s1), i3 = xfer_div(r, D.q2, D.s2);
    const int g1 = lin[u] - r * D.m1 + D.ns[0], g2 = r - i3 * D.m2 + D.ns[1],
              g3 = i3 + D.ns[2];
    const bool in = (unsigned)g1 < (unsigned)A.g1 && (unsigned)g2 < (unsigned)A.g2 &&
                    (unsigned)g3 < (unsigned)A.g3;
    gi[u] = -1;
    if (in) {
      const int g = g1 + A.g1 * (g2 + A.g2 * g3);
      gi[u] = inv ? inv[g] : g;
    }
  }
  double* dst = A.dst;
  const long long lb = D.loff + (FINE ? D.nvctr_c : 0), gb = D.goff + (FINE ? A.gnvctr_c : 0);
  double v[XU];
#pragma unroll
  for (int u = 0; u < XU; ++u) {
    const int e = min(e0 + u * XT, ne - 1), t = FINE ? e % 7 : 0;
    v[u] = 0.0;
    if (gi[u] >= 0) v[u] = A.src[A.to_local ? gb + (FINE ? 7LL * gi[u] + t : gi[u]) : lb + e];
  }
#pragma unroll
  for (int u = 0; u < XU; ++u) {
    const int e = e0 + u * XT, t = FINE ? e % 7 : 0;
    if (e >= ne) continue;
    if (A.to_local) dst[lb + e] = v[u];
    else if (gi[u] >= 0) dst[gb + (FINE ? 7LL * gi[u] + t : gi[u])] = v[u];
    else if (t == 0) {   // once per point
      atomicAdd(A.miss, 1);
      __hip_atomic_store(A.flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

__global__ __launch_bounds__(XT) void k_xfer(XferArgs A) {
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const XferDesc D = A.d[xfer_find(A, tile)];
  const int lt = tile - D.tile0;
  const int ctiles = (D.nvctr_c + XC - 1) / XC;
  if (lt < ctiles) xfer_tile<false>(A, D, lt * XC + threadIdx.x);
  else xfer_tile<true>(A, D, (lt - ctiles) * XC + threadIdx.x);
}

hipError_t launch_xfer(const XferArgs& A, int ntiles, hipStream_t s) {
  if (ntiles > 0) k_xfer<<<ntiles, XT, 0, s>>>(A);
  return hipGetLastError();
}

long long xfer_tiles(int nvctr_c, int nvctr_f) {
  return ((long long)nvctr_c + XC - 1) / XC + (7LL * nvctr_f + XC - 1) / XC;
}

}  // namespace bdft
