// Plane-fused kernels of the FP32 sequence (and of the matrix-core ones'
// backward pass on the vector units): one work-group holds a whole x-y plane of
// one box in LDS and applies both in-plane axes there.
//
//   k_plane_fwd  plane j3 of W (wavelet x,y at wavelet z index j3):
//                K  = K_x W + K_y W              (kinetic, + ekin partial)
//                T2 = G_y G_x W                  (real x,y at wavelet z)
//   k_plane_bwd  plane j3 of T2 after the z pass (G_z^T V G_z):
//                out = G_x^T G_y^T T2 + K        -> hpsi += compress(out)
//
// Together with the z-line kernels (k_zpot, k_kin<2>) this replaces the
// x/y line passes and the compress pass: the (L1,2N2,2N3) intermediate and
// the separate wavelet output volume never reach memory.  Operators and
// filters are those of the line kernels (growshrink.f90 comb_grow/comb_shrink,
// convolut_ib_optim.f90 ConvolkineticT).  Chunks whose stencil lies inside
// the line read it directly; the forward pass's other chunks read through a
// per-box line map (periodic wrap, or a zero slot for free padding), the
// backward pass's apply the wrap or padding by index arithmetic.
#include "bdft_internal.h"
#include "bdft_stencil.h"

namespace bdft {

// threads per plane work-group: two to four work-groups of 8 waves run per CU
constexpr int NTP = 512;

// A contiguous n1 x n2 plane (x fastest) from memory into LDS rows of
// stride rs > n1: element i = tid + k NTP of the plane, its row carried from
// step to step (no division per element), UR loads in flight per thread.
// TRANS: stored transposed, x = j of row ch at j rs + ch (rs >= n2, odd).
template <bool TRANS = false>
__device__ __forceinline__ void plane_load(float* dst, int rs, const float* __restrict__ src,
                                           int n1, int n2) {
  constexpr int UR = 8;
  const int tot = n1 * n2;
  ItDiv d(threadIdx.x, n1, NTP);
  for (int base = threadIdx.x; base < tot; base += NTP * UR) {
    float v[UR];
    int a[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const int i = base + u * NTP;
      v[u] = i < tot ? src[i] : 0.0f;
      // row r, column i - r n1 at r rs + i - r n1 (transposed: (i - r n1) rs + r)
      a[u] = TRANS ? d.j * rs + d.ch : i + d.ch * (rs - n1);
      d.next(n1);
    }
#pragma unroll
    for (int u = 0; u < UR; ++u)
      if (base + u * NTP < tot) dst[a[u]] = v[u];
  }
}

// the reverse: LDS rows of stride rs into a contiguous n1 x n2 plane
__device__ __forceinline__ void plane_store(float* __restrict__ dst, const float* src, int rs,
                                            int n1, int n2) {
  const int tot = n1 * n2;
  ItDiv d(threadIdx.x, n1, NTP);
  for (int i = threadIdx.x; i < tot; i += NTP) {
    dst[i] = src[i + d.ch * (rs - n1)];
    d.next(n1);
  }
}

__device__ __forceinline__ double block_sum_p(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < NTP / 64; ++i) s += red[i];
  return s;
}

// LDS layout of the forward plane kernel: the W plane A
// (W2 rows of stride RA = W1 + 1, then a zero row; column W1 of every row is
// zero: the free lines' zero slots), the second plane C (W2 + 1 rows of
// stride RC), then the line maps (x on the rows of A, y on the columns of A,
// y on the columns of C).  Byte offset of the maps:
__host__ __device__ inline size_t plane_maps_off(int N1, int N2, int RC) {
  const size_t rows = 2 * N2 + 1, RA = 2 * N1 + 1;
  return ((rows * RA + rows * RC) * sizeof(float) + 7) & ~(size_t)7;
}

// zero slots: column W1 and row W2 of A, row W2 of C (stride RC)
__device__ __forceinline__ void plane_zero_slots(float* A, int RA, int W1, int W2, float* C,
                                                 int RC) {
  for (int i = threadIdx.x; i < W2; i += NTP) A[i * RA + W1] = 0.0f;
  for (int i = threadIdx.x; i < RA; i += NTP) A[W2 * RA + i] = 0.0f;
  for (int i = threadIdx.x; i < RC; i += NTP) C[W2 * RC + i] = 0.0f;
}

// ---------------------------------------------------------------------------
// forward plane kernel; KIN = false: T2 only (the density's x and y grow,
// daub_to_isf in sumrho.f90:377-469), no kinetic, no K, no ekin.  tt: the
// launch's tiles (all boxes, or one group of them); ft: the table over all
// boxes whose tile numbers index the kinetic partials
// ---------------------------------------------------------------------------
template <bool KIN = true>
__global__ __launch_bounds__(NTP) void k_plane_fwd(Batch B, TileTable tt, TileTable ft,
                                                   double* part) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[NTP / 64];
  const int tile = tile_of(tt);
  const int lb = find_box(tt, tile);
  const int b = table_box(tt, lb);
  const BoxDesc bd = B.box[b];
  const int j3 = tile - box_first_tile(tt, lb);
  const int N1 = bd.N[0], N2 = bd.N[1], L1 = bd.L[0], L2 = bd.L[1], per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * N2;
  const int RA = W1 + 1;            // row stride of the wavelet plane
  const int RB = odd_stride(L1);    // row stride of the G_x output
  const int RC = max(RA, RB);
  float* A = (float*)smem;              // W plane: A[j2*RA + j1]
  float* C = A + (W2 + 1) * RA;         // kinetic accumulator, later G_x output
  int2* mx = (int2*)(smem + plane_maps_off(N1, N2, RC));
  int2* mya = mx + map_len(N1);
  int2* myc = mya + map_len(N2);
  const float* src = (const float*)B.W + bd.w_off + (long long)W1 * W2 * j3;
  const int tid = threadIdx.x;
  // load the plane (contiguous), UNR loads in flight per thread
  plane_load(A, RA, src, W1, W2);
  build_map(mx, N1, per, sizeof(float), W1, tid, NTP);
  build_map(mya, N2, per, RA * sizeof(float), W2, tid, NTP);
  build_map(myc, N2, per, RB * sizeof(float), W2, tid, NTP);
  plane_zero_slots(A, RA, W1, W2, C, RB);
  __syncthreads();
  if constexpr (KIN) {
  // K_x: rows j2, chunks of 4 coarse x positions -> C
  const float kx = (float)bd.kscale[0], ky = (float)bd.kscale[1];
  const int cx = (N1 + 3) >> 2;
  for (ItDiv d(tid, W2, NTP); d.ch < cx; d.next(W2)) {
    const int ch = d.ch, j2 = d.j;
    const int i0 = 4 * ch;
    float oc[4], od[4];
    kin4_any(PLine<float>{A + j2 * RA, 1}, mx, N1, i0, oc, od);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (i0 + r < N1) {
        C[j2 * RA + i0 + r] = oc[r] * kx;
        C[j2 * RA + N1 + i0 + r] = od[r] * kx;
      }
  }
  __syncthreads();
  // K_y: columns j1, chunks of 4 coarse y positions, accumulated into C
  double ek = 0.0;
  const int cy = (N2 + 3) >> 2;
  for (ItDiv d(tid, W1, NTP); d.ch < cy; d.next(W1)) {
    const int ch = d.ch, j1 = d.j;
    const int i0 = 4 * ch;
    float oc[4], od[4];
    kin4_any(PLine<float>{A + j1, RA}, mya, N2, i0, oc, od);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (i0 + r < N2) {
        const int a = (i0 + r) * RA + j1, d = (N2 + i0 + r) * RA + j1;
        const float vc = C[a] + oc[r] * ky, vd = C[d] + od[r] * ky;
        C[a] = vc;
        C[d] = vd;
        ek += (double)vc * (double)A[a] + (double)vd * (double)A[d];
      }
  }
  const double eks = block_sum_p(ek, red);
  if (tid == 0) part[box_first_tile(ft, b) + j3] = eks;
  __syncthreads();
  // K plane -> memory (contiguous)
  {
    float* kd = (float*)B.K + bd.w_off + (long long)W1 * W2 * j3;
    plane_store(kd, C, RA, W1, W2);
  }
  __syncthreads();
  }
  // G_x: rows j2 -> C as (W2 rows) x (L1 cols), row stride RB
  const int gx = (L1 + 7) >> 3;
  for (ItDiv d(tid, W2, NTP); d.ch < gx; d.next(W2)) {
    const int ch = d.ch, j2 = d.j;
    const int p0 = 8 * ch;
    float o[8];
    grow8_any(PLine<float>{A + j2 * RA, 1}, mx, N1, grow_k0(p0, per), o);
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (p0 + r < L1) C[j2 * RB + p0 + r] = o[r];
  }
  __syncthreads();
  // G_y: columns p1 of C -> T2 plane (real x,y at wavelet z j3)
  float* dst = (float*)B.T2 + bd.t2_off + (long long)L1 * L2 * j3;
  const int gy = (L2 + 7) >> 3;
  for (ItDiv d(tid, L1, NTP); d.ch < gy; d.next(L1)) {
    const int ch = d.ch, p1 = d.j;
    const int p0 = 8 * ch;
    float o[8];
    grow8_any(PLine<float>{C + p1, RB}, myc, N2, grow_k0(p0, per), o);
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (p0 + r < L2) dst[p1 + (long long)L1 * (p0 + r)] = o[r];
  }
}

// ---------------------------------------------------------------------------
// backward plane kernel with compress-accumulate
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NTP) void k_plane_bwd(Batch B, TileTable tt) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int tile = tile_of(tt);
  const int lb = find_box(tt, tile);   // tables over a subset carry a box map
  const BoxDesc bd = B.box[table_box(tt, lb)];
  const int j3 = tile - box_first_tile(tt, lb);
  const int N1 = bd.N[0], N2 = bd.N[1], N3 = bd.N[2], L1 = bd.L[0], L2 = bd.L[1],
            per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * N2;
  // odd row strides: a free box's fine extents are odd already, so its rows
  // take no padding (with the periodic maps, the plane takes no more LDS
  // than with untransposed rows of L1 + 1)
  const int RU = L2 | 1;            // T2 plane, transposed: y lines as rows
  const int RQ = L1 | 1;            // G_y^T output rows (read by rows)
  const int RO = W1 + 1;
  float* U = (float*)smem;            // T2 plane: U[p1*RU + p2], later output O
  float* Bq = U + max(L1 * RU, W2 * RO);  // G_y^T output: Bq[j2*RQ + p1]
  int* fmx = (int*)(Bq + W2 * RQ);     // periodic fine-line maps (x: rows of Bq,
  int* fmy = fmx + fmap_len(N1);       // y: rows of U)
  const int tid = threadIdx.x;
  const float* src = (const float*)B.T2 + bd.t2_off + (long long)L1 * L2 * j3;
  // the compress's first point per thread (indices, K, old hpsi) is loaded
  // before the plane, so that its latency overlaps the plane load and the
  // two passes (one point: more registers held through the passes cost
  // occupancy); later steps take UC points each
  constexpr int UC = 2, UP = 1;
  const float* Kp = (const float*)B.K + bd.w_off + (long long)W1 * W2 * j3;
  CompressStep<float, UP> st0;
  compress_load<UP, NTP>(bd, j3, Kp, B.hpsi, tid, st0);
  plane_load<true>(U, RU, src, L1, L2);
  if (per) {
    build_fmap(fmx, N1, L1, sizeof(float), tid, NTP);
    build_fmap(fmy, N2, L2, sizeof(float), tid, NTP);
  }
  __syncthreads();
  // G_y^T: y lines p1 (rows of U) -> Bq rows (c: i2, d: N2+i2), NOY coarse outputs
  // per work item (NOX for G_x^T): two, so that the last round of items leaves
  // fewer lanes idle between the barriers than with four (1024 spheres, 3.41 ->
  // 3.22 ms)
  constexpr int NOY = 2, NOX = NOY;
  const int cy = (N2 + NOY - 1) / NOY;
  for (ItDiv d(tid, L1, NTP); d.ch < cy; d.next(L1)) {
    const int ch = d.ch, p1 = d.j;
    const int i0 = NOY * ch;
    float oc[NOY], od[NOY];
    shrink4_any<float, NOY>(U + p1 * RU, fmy, L2, i0, per, oc, od);
#pragma unroll
    for (int r = 0; r < NOY; ++r)
      if (i0 + r < N2) {
        Bq[(i0 + r) * RQ + p1] = oc[r];
        Bq[(N2 + i0 + r) * RQ + p1] = od[r];
      }
  }
  __syncthreads();
  // G_x^T: rows j2 of Bq -> output plane O (reuses U), row stride RO
  float* O = U;
  const int cx = (N1 + NOX - 1) / NOX;
  for (ItDiv d(tid, W2, NTP); d.ch < cx; d.next(W2)) {
    const int ch = d.ch, j2 = d.j;
    const int i0 = NOX * ch;
    float oc[NOX], od[NOX];
    shrink4_any<float, NOX>(Bq + j2 * RQ, fmx, L1, i0, per, oc, od);
#pragma unroll
    for (int r = 0; r < NOX; ++r)
      if (i0 + r < N1) {
        O[j2 * RO + i0 + r] = oc[r];
        O[j2 * RO + N1 + i0 + r] = od[r];
      }
  }
  __syncthreads();
  // out = O + K, accumulated into hpsi at the compressed positions of the
  // plane's four components (s3 fixed by j3), compress_and_accumulate_mixed
  // (un-compress.f90:2174-2238)
  compress_store<float, UP, NTP>(bd, j3, O, RO, B.hpsi, tid, st0);
  for (int i0 = tid + NTP * UP; i0 < N1 * N2; i0 += NTP * UC) {
    CompressStep<float, UC> st;
    compress_load<UC, NTP>(bd, j3, Kp, B.hpsi, i0, st);
    compress_store<float, UC, NTP>(bd, j3, O, RO, B.hpsi, i0, st);
  }
}

// LDS bytes of the two plane kernels for the largest box extents
size_t plane_lds_fwd(int N1, int N2, int L1) {
  const int RA = 2 * N1 + 1, RB = odd_stride(L1);
  return plane_maps_off(N1, N2, RA > RB ? RA : RB) +
         8 * (size_t)(map_len(N1) + 2 * map_len(N2));
}
size_t plane_lds_bwd(int N1, int N2, int L1, int L2) {
  const size_t RU = L2 | 1, RQ = L1 | 1, RO = 2 * N1 + 1;
  const size_t u = (size_t)L1 * RU > 2 * N2 * RO ? (size_t)L1 * RU : 2 * N2 * RO;
  const bool per = L1 == 2 * N1;
  return (u + 2 * N2 * RQ) * sizeof(float) +
         (per ? 4 * (size_t)(fmap_len(N1) + fmap_len(N2)) : 0);
}

static hipError_t plane_setup(int bytes) {
  const void* k[] = {(const void*)k_plane_fwd<true>, (const void*)k_plane_fwd<false>,
                     (const void*)k_plane_bwd};
  for (const void* f : k) {
    const hipError_t e =
        hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// LDS bytes one work-group may use on the current device; the plane kernels'
// dynamic-LDS limit is raised to it where the runtime asks for that.
size_t plane_attributes() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) !=
          hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  if (plane_setup(v) != hipSuccess)
    (void)hipGetLastError();  // not required on this runtime; clear the error
  return (size_t)v;
}

hipError_t launch_plane_fwd(const Batch& B, const TileTable& t, const TileTable& ft,
                            int ntiles, size_t lds, double* part, hipStream_t s) {
  k_plane_fwd<true><<<ntiles, NTP, lds, s>>>(B, t, ft, part);
  return hipGetLastError();
}
hipError_t launch_plane_grow(const Batch& B, const TileTable& t, int ntiles, size_t lds,
                             hipStream_t s) {
  k_plane_fwd<false><<<ntiles, NTP, lds, s>>>(B, t, t, nullptr);
  return hipGetLastError();
}
hipError_t launch_plane_bwd(const Batch& B, const TileTable& t, int ntiles, size_t lds,
                            hipStream_t s) {
  k_plane_bwd<<<ntiles, NTP, lds, s>>>(B, t);
  return hipGetLastError();
}

}  // namespace bdft
