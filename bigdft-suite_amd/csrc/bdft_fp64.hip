// FP64 sequence of the local-Hamiltonian apply.
//
//   k_zgrow    psi -> TZ = G_z W            64 z lines of 16 coarse columns
//   k_xykin    psi -> K  = K_x W + K_y W    one x-y plane of W
//   k_xypot    TZ <- G_x^T G_y^T V G_y G_x TZ   one x-y plane at a fine z point
//   k_zback    hpsi += compress(G_z^T TZ + K + K_z W)   64 z lines
//
// The wavelet volume W never reaches memory: the kernels that need it gather
// it from the compressed coefficients (every 56-byte fine record read whole
// by the z kernels, by two neighbouring planes in k_xykin), and V is applied
// between the two halves of one plane's work, so the only grids are TZ
// (2 N1 x 2 N2 x L3) and K.  88 bytes move per point of a periodic box where
// the x-y-z order with W, K and (L1, L2, 2 N3) grids moved 112; a free box's
// TZ is also (2 N1 2 N2 L3) / (L1 L2 2 N3) of that grid (0.66 at 28 coarse
// points an axis).  Operators and filters are those of the line kernels
// (growshrink.f90 comb_grow / comb_shrink, convolut_ib_optim.f90
// ConvolkineticT); sums run in another order of the axes.
//
// Measured on 128 orbitals of a periodic 40^3 box (6.6e7 fine points), the
// x-y-z order's kernels before: uncompress 183 us, forward planes 1085, z
// kinetic 553, z potential 413, backward planes 689, an apply 2.65 ms; now,
// each the fastest of five launches under the tracer, k_zgrow 0.24 ms (16 B per
// point: 4.5 TB/s, a large copy runs at 4.9), k_xykin 0.46 and k_xypot 0.47
// (three times the time of their FMAs at the FP64 peak; a quarter of their
// vector instructions are addresses, the rest waits at barriers and LDS
// loads), k_zback 0.57 (40 B per point: 4.6 TB/s); an apply without the tracer
// 1.68 ms.  48 orbitals of a 64^3 box, whose pairs of planes did not fit in LDS
// (line passes): 4.54 -> 2.80 ms; 256 free boxes of 16 to 40 points an axis
// 2.66 -> 2.02 ms.
//
// Grid TZ of a box (tz_off): plane p3 = 0 .. L3 - 1, in it the wavelet plane
// [j1 + 2 N1 j2]; K (w_off): the wavelet volume.
#include <algorithm>

#include "bdft_internal.h"
#include "../../include/bigdft_hip.h"
#include "bdft_stencil.h"

namespace bdft {

// ---------------------------------------------------------------------------
// z-line tiles: C = 16 coarse columns q = i1 + N1 i2 of a box, each with its
// four z lines (s1, s2): line l = col + C (s1 + 2 s2), one lane per line.  A wave
// works on one chunk of outputs of all 64 lines, so the chunk's rows are
// uniform over the wave: LDS rows are read without bank conflicts at
// immediate offsets, and a line end costs scalar instructions only.
//
// Lines whose 64-line tile does not fit in LDS (beyond 159 periodic, 145 free
// points): C = 8 columns, 32 lines, and each half of a wave takes a chunk of
// its own (up to the library's 256 points, 138 KB).  The longer lines of a
// batch have launches of their own.  16 orbitals of 24 x 24 x 200 points: 0.51
// ms, on the line passes of bdft_pass.hip 2.04 (density 0.27 and 1.09 ms,
// four preconditioner steps 1.86 and 5.12).
// ---------------------------------------------------------------------------
constexpr int CC = CCOL;
constexpr int NL = 4 * CC;      // lines of a tile of 16 columns
static_assert(NL == 64, "one lane per line");

// this lane's line and its chunk among the SUB a wave takes at a time
template <int C>
struct ZLane {
  static constexpr int NLC = 4 * C, SUB = CC / C;
  int line, sub;
  __device__ __forceinline__ ZLane() {
    const int lane = threadIdx.x & 63;
    line = SUB == 1 ? lane : lane & (NLC - 1);
    sub = SUB == 1 ? 0 : lane / NLC;
  }
};

// W of the tile's columns into LDS: row s3 N3 + i3 (wavelet z index),
// lane l.  Thread e = tid mod 8 C moves element e of every (tid / 8 C)-th coarse
// z: columns' scaling coefficients for e < C, else component (e - C) mod 7
// of column (e - C) / 7, the order the records have in memory.
template <int C = CC>
struct RecElem {
  int col, t;                   // column and component 0..7
  __device__ __forceinline__ explicit RecElem(int e) {
    if (e < C) {
      col = e;
      t = 0;
    } else {
      col = (e - C) / 7;
      t = e - C - 7 * col + 1;
    }
  }
};

// AX = 1: the y lines of 16 coarse x of one coarse z instead, rows s2 N2 +
// i2, lines col + CC (s1 + 2 s3).  lin0: linear index of the first column's
// first point.
template <int NT, int AX = 2, int C = CC>
__device__ __forceinline__ void load_columns(double* lds, const BoxDesc& bd, const double* psi,
                                             int first, int nq) {
  constexpr int NL = 4 * C, EL = 8 * C, ZS = NT / EL, UR = 8;
  const int n = bd.N[AX], step = AX == 2 ? bd.N[0] * bd.N[1] : bd.N[0];
  const RecElem<C> re(threadIdx.x & (EL - 1));
  const int z0 = threadIdx.x / EL;
  const bool on = re.col < nq;
  const int lin0 = first + (on ? re.col : 0);
  const char* src = (const char*)(psi + bd.psi_off);
  const unsigned off = re.t == 0 ? 0u : 8u * (unsigned)(bd.nvctr_c + re.t - 1);
  const unsigned mul = re.t == 0 ? 8u : 56u;
  const int sec = AX == 2 ? re.t >> 2 : (re.t >> 1) & 1;
  const int ln = AX == 2 ? re.t & 3 : (re.t & 1) + 2 * (re.t >> 2);
  double* dst = lds + sec * n * NL + re.col + C * ln;
  if (!bd.cinv && !bd.finv) {
    for (int zb = z0; zb < n; zb += ZS * UR) {
      double v[UR];
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        const int z = min(zb + u * ZS, n - 1);
        v[u] = *(const double*)(src + (off + mul * (unsigned)(lin0 + step * z)));
      }
#pragma unroll
      for (int u = 0; u < UR; ++u)
        if (zb + u * ZS < n) dst[(zb + u * ZS) * NL] = on ? v[u] : 0.0;
    }
  } else {
    const int* inv = re.t == 0 ? bd.cinv : bd.finv;
    for (int zb = z0; zb < n; zb += ZS * UR) {
      int r[UR];
      double v[UR];
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        const int z = zb + u * ZS, lin = lin0 + step * z;
        r[u] = -1;
        if (on && z < n) r[u] = inv ? inv[lin] : lin;
      }
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        v[u] = 0.0;
        if (r[u] >= 0) v[u] = *(const double*)(src + (off + mul * (unsigned)r[u]));
      }
#pragma unroll
      for (int u = 0; u < UR; ++u)
        if (zb + u * ZS < n) dst[(zb + u * ZS) * NL] = v[u];
    }
  }
}

// The taps of rows k0 .. k0 + NK - 1 of a line, k0 uniform over the lanes of a
// chunk: tap(kk, k) with k a valid row.  Rows past a line end wrap (periodic) or
// are left out (free: they hold zeros).
template <int NK, int SUB = 1, typename F>
__device__ __forceinline__ void line_taps(int k0, int n, int per, F tap) {
  // (SUB > 1: the chunks of the whole wave)
  if (SUB == 1 ? k0 >= 0 && k0 + NK <= n : (bool)__all(k0 >= 0 && k0 + NK <= n)) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) tap(kk, k0 + kk);
  } else if (per) {
    int k = k0;
    while (k < 0) k += n;
    while (k >= n) k -= n;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      tap(kk, k);
      k = k + 1 == n ? 0 : k + 1;
    }
  } else {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      if (k0 + kk >= 0 && k0 + kk < n) tap(kk, k0 + kk);
  }
}

// The 32 taps of a kinetic chunk from both ends inwards: tap 31 - kk has the
// mirror of tap kk's coefficients (the filters are symmetric or each other's
// mirror), so each pair shares its constants.  In ascending order they stay
// live from one half to the other, more than the scalar registers hold, and
// a tenth of the vector instructions are their spills.
template <typename F>
__device__ __forceinline__ void kin_order(F tap) {
#pragma unroll
  for (int kk = 0; kk < 16; ++kk) {
    tap(kk);
    tap(31 - kk);
  }
}
// ... on a line of n values from k0 (as line_taps)
template <int SUB = 1, typename F>
__device__ __forceinline__ void kin_taps(int k0, int n, int per, F tap) {
  if (SUB == 1 ? k0 >= 0 && k0 + 32 <= n : (bool)__all(k0 >= 0 && k0 + 32 <= n)) {
    kin_order([&](int kk) { tap(kk, k0 + kk); });
  } else if (per) {
    int ka = k0, kb = k0 + 31;
    while (ka < 0) ka += n;
    while (ka >= n) ka -= n;
    while (kb < 0) kb += n;
    while (kb >= n) kb -= n;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      tap(kk, ka);
      tap(31 - kk, kb);
      ka = ka + 1 == n ? 0 : ka + 1;
      kb = kb == 0 ? n - 1 : kb - 1;
    }
  } else {
    kin_order([&](int kk) {
      if (k0 + kk >= 0 && k0 + kk < n) tap(kk, k0 + kk);
    });
  }
}

// a tile's lines: first column, columns, and this lane's line
template <int C = CC>
struct ColTile {
  int q0, nq;
  bool on;       // this lane's column is one of the box
  unsigned at;   // its line in a wavelet plane, j1 + 2 N1 j2
  __device__ __forceinline__ ColTile(const BoxDesc& bd, int lt) {
    const int N1 = bd.N[0], N2 = bd.N[1];
    q0 = lt * C;
    nq = min(C, N1 * N2 - q0);
    const int line = ZLane<C>().line, col = line & (C - 1), s = line / C;
    on = col < nq;
    const int q = q0 + (on ? col : 0);
    const int i2 = qdiv(q, N1, 1.0f / (float)N1), i1 = q - i2 * N1;
    at = (unsigned)(i1 + N1 * (s & 1) + 2 * N1 * (i2 + N2 * (s >> 1)));
  }
};

// ---------------------------------------------------------------------------
// TZ = G_z W
// ---------------------------------------------------------------------------
template <int ZG_NT, int C = CC>
__device__ __forceinline__ void zgrow_tile(const Batch& B, const TileTable& tt, int tile,
                                           unsigned char* smem) {
  constexpr int NL = 4 * C, SUB = CC / C;
  double* lds = (double*)smem;
  const int lb = find_box(tt, tile);
  const BoxDesc bd = B.box[table_box(tt, lb)];
  const int N3 = bd.N[2], L3 = bd.L[2], per = bd.per;
  const ColTile<C> ct(bd, tile - box_first_tile(tt, lb));
  load_columns<ZG_NT, 2, C>(lds, bd, B.psi, ct.q0, ct.nq);
  __syncthreads();
  const ZLane<C> zl;
  const double* c = lds + zl.line;
  const double* d = c + N3 * NL;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t ps = 4 * (size_t)(bd.N[0] * bd.N[1]);
  double* out = (double*)B.TZ + bd.tz_off + ct.at;
  for (int pw = 8 * SUB * w; pw < L3; pw += 8 * SUB * (ZG_NT / 64)) {
    const int p0 = pw + 8 * zl.sub;
    double o[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) o[r] = 0.0;
    line_taps<19, SUB>(grow_k0(p0, per), N3, per,
                       [&](int kk, int k) { grow_tap(kk, c[k * NL], d[k * NL], o); });
    if (ct.on) {
      double* q = out + ps * p0;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (p0 + r < L3) q[ps * r] = o[r];
    }
  }
}
template <int ZG_NT, int C = CC>
__global__ __launch_bounds__(ZG_NT) void k_zgrow(Batch B, TileTable tt) {
  extern __shared__ __align__(16) unsigned char smem[];
  zgrow_tile<ZG_NT, C>(B, tt, tile_of(tt), smem);
}

// ---------------------------------------------------------------------------
// hpsi += compress(G_z^T TZ + K + K_z W), ekin partial.  MI: chunks of four
// coarse z per wave, their sums held in registers while the LDS rows change
// from W to TZ to the records of hpsi.  The
// first loads of K and TZ are issued before the passes ahead of them.
// ---------------------------------------------------------------------------
template <int ZB_NT, int MI, int WPE, int C = CC>
__global__ __launch_bounds__(ZB_NT, WPE) void k_zback(Batch B, TileTable tt, TileTable ft,
                                                 double* part) {
  constexpr int NW = ZB_NT / 64, NL = 4 * C, SUB = CC / C;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  __shared__ double red[NW];
  const int tile = tile_of(tt);
  const int lb = find_box(tt, tile);
  const int b = table_box(tt, lb);
  const BoxDesc bd = B.box[b];
  const int lt = tile - box_first_tile(tt, lb);
  const int N3 = bd.N[2], L3 = bd.L[2], per = bd.per;
  const ColTile<C> ct(bd, lt);
  const ZLane<C> zl;
  const int lane = zl.line;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t ps = 4 * (size_t)(bd.N[0] * bd.N[1]);
  // chunk (row) j of this wave's
  auto mine = [&](int j) { return SUB == 1 ? j : SUB * j + zl.sub; };
  // K of a chunk; the lines of TZ, TR rows of this wave at a time
  const double* K = (const double*)B.K + bd.w_off + ct.at;
  auto load_k = [&](int i0, double k[8]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int z = min(i0 + r, N3 - 1);
      k[r] = K[ps * z];
      k[4 + r] = K[ps * (N3 + z)];
    }
  };
  constexpr int TR = 8;
  const double* tz = (const double*)B.TZ + bd.tz_off + ct.at;
  auto load_tz = [&](int pb, double v[TR]) {
#pragma unroll
    for (int u = 0; u < TR; ++u) v[u] = tz[ps * min(mine(pb + u * NW), L3 - 1)];
  };
  double k0[8], tv[TR];
  load_k(4 * mine(w), k0);
  load_columns<ZB_NT, 2, C>(lds, bd, B.psi, ct.q0, ct.nq);
  __syncthreads();
  load_tz(w, tv);
  double o[MI][8];   // c, then d
  double ek = 0.0;
  {
    const double* c = lds + lane;
    const double* d = c + N3 * NL;
    const double ks = bd.kscale[2];
#pragma unroll
    for (int m = 0; m < MI; ++m) {
      const int i0 = 4 * mine(w + m * NW);
      if (i0 < N3) {
        double k[8];
        if (m > 0) load_k(i0, k);
#pragma unroll
        for (int r = 0; r < 8; ++r) o[m][r] = 0.0;
        kin_taps<SUB>(i0 - 14, N3, per, [&](int kk, int z) {
          kin_tap(kk, c[z * NL], d[z * NL], o[m], o[m] + 4);
        });
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          o[m][r] = fma(o[m][r], ks, m > 0 ? k[r] : k0[r]);
          o[m][4 + r] = fma(o[m][4 + r], ks, m > 0 ? k[4 + r] : k0[4 + r]);
          if (i0 + r < N3) {   // lanes off the box hold W = 0
            ek = fma(o[m][r], c[(i0 + r) * NL], ek);
            ek = fma(o[m][4 + r], d[(i0 + r) * NL], ek);
          }
        }
      }
    }
  }
  __syncthreads();
  for (int pb = w; SUB * pb < L3; pb += NW * TR) {
    if (pb > w) load_tz(pb, tv);
#pragma unroll
    for (int u = 0; u < TR; ++u)
      if (mine(pb + u * NW) < L3) lds[mine(pb + u * NW) * NL + lane] = tv[u];
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * mine(w + m * NW);
    if (i0 < N3) {
      // summed by itself: on top of the larger kinetic term every tap would
      // round at its size
      double g[8] = {};
      line_taps<37, SUB>(per ? 2 * i0 - 14 : 2 * i0, L3, per, [&](int qq, int p) {
        shrink_tap<double, 4>(qq, lds[p * NL + lane], g, g + 4);
      });
#pragma unroll
      for (int r = 0; r < 8; ++r) o[m][r] += g[r];
    }
  }
  const double eks = block_sum_rt(ek, red);   // starts with a barrier
  if (threadIdx.x == 0) part[box_first_tile(ft, b) + lt] = eks;
  // the sums as records: row i3, element e of RecElem (lane's component
  // s + 4 s3, s = lane / CC; component 0 is the scaling coefficient)
  {
    const int col = lane & (C - 1), s = lane / C;
    const int ec = s == 0 ? col : C + 7 * col + s - 1, ed = C + 7 * col + s + 3;
#pragma unroll
    for (int m = 0; m < MI; ++m) {
      const int i0 = 4 * mine(w + m * NW);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (i0 + r < N3) {
          lds[(i0 + r) * 2 * NL + ec] = o[m][r];
          lds[(i0 + r) * 2 * NL + ed] = o[m][4 + r];
        }
    }
  }
  __syncthreads();
  {
    constexpr int EL = 8 * C, ZS = ZB_NT / EL, UR = 8;
    const int e = threadIdx.x & (EL - 1), npl = bd.N[0] * bd.N[1];
    const RecElem<C> re(e);
    if (re.col < ct.nq) {
      char* dst = (char*)(B.hpsi + bd.psi_off);
      const unsigned off = re.t == 0 ? 0u : 8u * (unsigned)(bd.nvctr_c + re.t - 1);
      const unsigned mul = re.t == 0 ? 8u : 56u;
      const int lin0 = ct.q0 + re.col;
      const int* inv = re.t == 0 ? bd.cinv : bd.finv;
      for (int zb = threadIdx.x / EL; zb < N3; zb += ZS * UR) {
        int rec[UR];
        double v[UR];
#pragma unroll
        for (int u = 0; u < UR; ++u) {
          const int z = zb + u * ZS, lin = lin0 + npl * z;
          rec[u] = -1;
          if (z < N3) rec[u] = inv ? inv[lin] : lin;
        }
#pragma unroll
        for (int u = 0; u < UR; ++u)
          v[u] = rec[u] >= 0 ? *(const double*)(dst + (off + mul * (unsigned)rec[u])) : 0.0;
#pragma unroll
        for (int u = 0; u < UR; ++u)
          if (rec[u] >= 0)
            *(double*)(dst + (off + mul * (unsigned)rec[u])) =
                v[u] + lds[(zb + u * ZS) * 2 * NL + e];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Preconditioner, first half of A v = S (K + c) S v: K = c W + K_z W, W = S v.
// MODE 0: v = x; 1: v = d; 2: v = d after the step's updates of the compressed
// vectors, x += alpha d and d = r + beta d (the only kernel that reads whole
// records of all three, so both updates ride on it: a conjugate-gradient step
// moves 96 bytes per coefficient, in kernels of their own 128).  64 orbitals
// of a periodic 48^3 box, six steps: 13.1 ms with the volumes W and K scattered
// and gathered by kernels of their own, 8.3 now; this kernel 0.53 ms (48 bytes
// per coefficient, 5.2 TB/s: bound by memory), k_xykin 0.53, the update of r
// 0.23.
// ---------------------------------------------------------------------------
template <int MODE, int PZ_NT, int WPE, int C = CC>
__global__ __launch_bounds__(PZ_NT, WPE) void k_pcz(Batch B, TileTable tt, PcArgs P) {
  constexpr int NW = PZ_NT / 64, NL = 4 * C, SUB = CC / C, EL = 8 * C, ZS = PZ_NT / EL,
                UR = MODE == 2 ? 4 : 8;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  const int tile = tile_of(tt);
  const int lb = find_box(tt, tile);
  const int b = table_box(tt, lb);
  const BoxDesc bd = B.box[b];
  const int N3 = bd.N[2], per = bd.per, npl = bd.N[0] * bd.N[1];
  const ColTile<C> ct(bd, tile - box_first_tile(tt, lb));
  {
    const RecElem<C> re(threadIdx.x & (EL - 1));
    const bool on = re.col < ct.nq;
    const int lin0 = ct.q0 + (on ? re.col : 0);
    const int* inv = re.t == 0 ? bd.cinv : bd.finv;
    const unsigned off = re.t == 0 ? 0u : 8u * (unsigned)(bd.nvctr_c + re.t - 1);
    const unsigned mul = re.t == 0 ? 8u : 56u;
    char *x = (char*)(P.x + bd.psi_off), *d = (char*)(P.d + bd.psi_off);
    const char* r = (const char*)(P.r + bd.psi_off);
    const double sc = P.pc[9 * b + 1 + re.t];
    const double alpha = MODE == 2 ? P.sc[4 * b + 1] : 0.0;
    const double beta = MODE == 2 ? P.sc[4 * b + 2] : 0.0;
    double* dst = lds + (re.t >> 2) * N3 * NL + re.col + C * (re.t & 3);
    for (int zb = threadIdx.x / EL; zb < N3; zb += ZS * UR) {
      int e[UR];
      double v[UR], rv[UR], xv[UR];
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        const int z = zb + u * ZS, lin = lin0 + npl * z;
        e[u] = -1;
        if (on && z < N3) e[u] = inv ? inv[lin] : lin;
      }
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        const unsigned at = off + mul * (unsigned)e[u];
        v[u] = e[u] >= 0 ? *(const double*)((MODE == 0 ? x : d) + at) : 0.0;
        if (MODE == 2) {
          rv[u] = e[u] >= 0 ? *(const double*)(r + at) : 0.0;
          xv[u] = e[u] >= 0 ? *(const double*)(x + at) : 0.0;
        }
      }
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        if (MODE == 2 && e[u] >= 0) {
          const unsigned at = off + mul * (unsigned)e[u];
          *(double*)(x + at) = fma(alpha, v[u], xv[u]);
          v[u] = fma(beta, v[u], rv[u]);
          *(double*)(d + at) = v[u];
        }
        if (zb + u * ZS < N3) dst[(zb + u * ZS) * NL] = sc * v[u];
      }
    }
  }
  __syncthreads();
  const ZLane<C> zl;
  const double* c = lds + zl.line;
  const double* d = c + N3 * NL;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t ps = 4 * (size_t)npl;
  const double ks = bd.kscale[2], cp = P.pc[9 * b];
  double* K = (double*)B.K + bd.w_off + ct.at;
  for (int iw = 4 * SUB * w; iw < N3; iw += 4 * SUB * NW) {
    const int i0 = iw + 4 * zl.sub;
    double o[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) o[h] = 0.0;
    kin_taps<SUB>(i0 - 14, N3, per,
                  [&](int kk, int z) { kin_tap(kk, c[z * NL], d[z * NL], o, o + 4); });
    if (ct.on) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
        if (i0 + h < N3) {
          K[ps * (i0 + h)] = fma(cp, c[(i0 + h) * NL], o[h] * ks);
          K[ps * (N3 + i0 + h)] = fma(cp, d[(i0 + h) * NL], o[4 + h] * ks);
        }
    }
  }
}

// ---------------------------------------------------------------------------
// in-plane passes.  One of a thread's work items is one chunk of a line, lanes along the
// lines.  A pass keeps its items' outputs in registers (at most MI items of 8
// values a thread) and writes them over the plane after a barrier, transposed
// where the next pass runs along the other axis: the lines are LDS rows of
// odd stride (taps at immediate offsets, 64 lanes on 64 rows meet no bank
// twice) and one plane of LDS serves all passes, two work-groups per CU up to
// 49 periodic or 36 free coarse points (two planes, 150 KB at 48, allow one,
// whose load, passes and store run one after the other).  Two chunks of a
// line per item (half the LDS reads, half the coefficients) and coefficients
// from scalar loads (half the scalar instructions) were both slower: 0.60 and
// 0.65 ms for k_xypot on the batch above when it took 0.59.
//
// Line ends: a wave whose chunks all lie inside their lines reads them
// directly.  Otherwise, periodic: through a line map in LDS (any N); free:
// the taps past the line are masked out per lane (they read whatever lies
// next to the row, PAD values around the plane keep that inside the
// allocation) and cost nothing where the whole wave is past the line.
// ---------------------------------------------------------------------------
constexpr int PAD = 16, PADE = 8;   // rows are read at most 15 values before, 5 past their end

// NK taps from value k0 of a line of n values: load(kk) reads tap kk's
// input(s) from the row, mapped(kk) through the line map, apply(kk, x) adds
// it to the outputs
template <int NK, typename FL, typename FM, typename FA>
__device__ __forceinline__ void row_taps(int k0, int n, int per, FL load, FM mapped, FA apply) {
  if (__all(k0 >= 0 && k0 + NK <= n)) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) apply(kk, load(kk));
  } else if (per) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) apply(kk, mapped(kk));
  } else {
    // loads run two taps ahead of the masked sums
    auto x0 = load(0), x1 = load(1);
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const auto x = x0;
      x0 = x1;
      if (kk + 2 < NK) x1 = load(kk + 2);
      if ((unsigned)(k0 + kk) < (unsigned)n) apply(kk, x);
    }
  }
}

__device__ __forceinline__ double2 at2(const double* ln, int2 e) {
  return make_double2(*(const double*)((const char*)ln + e.x),
                      *(const double*)((const char*)ln + e.y));
}

// G of a wavelet row [c; d] of N + N values: 8 fine outputs from k = k0 ..
// k0 + 18; m: the axis's coarse line map
__device__ __forceinline__ void grow_row(const double* ln, const int2* m, int N, int k0, int per,
                                         double o[8]) {
#pragma unroll
  for (int r = 0; r < 8; ++r) o[r] = 0.0;
  const double *c = ln + k0, *d = ln + N + k0;
  const int2* mm = m + (k0 + MOFF);
  row_taps<19>(
      k0, N, per, [&](int kk) { return make_double2(c[kk], d[kk]); },
      [&](int kk) { return at2(ln, mm[kk]); },
      [&](int kk, double2 x) { grow_tap(kk, x.x, x.y, o); });
}

// G^T of a fine row of L values: coarse outputs i0 .. i0 + 3; m: fine line
// map (periodic)
__device__ __forceinline__ void shrink_row(const double* ln, const int* m, int L, int i0,
                                           int per, double o[8]) {
#pragma unroll
  for (int r = 0; r < 8; ++r) o[r] = 0.0;
  const int p0 = per ? 2 * i0 - 14 : 2 * i0;
  const double* x = ln + p0;
  const int* mm = m + 2 * i0;
  row_taps<37>(
      p0, L, per, [&](int qq) { return x[qq]; },
      [&](int qq) { return *(const double*)((const char*)ln + mm[qq]); },
      [&](int qq, double v) { shrink_tap<double, 4>(qq, v, o, o + 4); });
}

// line maps of a periodic axis: coarse entry e (k = e - MOFF, up to N + 20):
// byte offsets of c and d at k modulo N; fine entry e (up to 2 N + 42): that
// of fine index e - 14 modulo 2 N
__host__ __device__ constexpr int cmap_len(int N) { return N + MOFF + 21; }
__host__ __device__ constexpr int smap_len(int N) { return 2 * N + 44; }
__device__ __forceinline__ void build_maps(int2* mc, int* mf, int N, int tid, int nt) {
  for (int e = tid; e < cmap_len(N); e += nt) {
    int k = e - MOFF;
    while (k < 0) k += N;
    while (k >= N) k -= N;
    mc[e] = make_int2(8 * k, 8 * (N + k));
  }
  if (mf)
    for (int e = tid; e < smap_len(N); e += nt) {
      int p = e - 14;
      while (p < 0) p += 2 * N;
      while (p >= 2 * N) p -= 2 * N;
      mf[e] = 8 * p;
    }
}

// items (chunk ch, line j) of a pass over nch chunks of n lines; d: the
// thread's first item
template <int MI, typename F>
__device__ __forceinline__ void each_item(ItDiv d, int n, int nch, F f) {
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    if (d.ch < nch) f(m, d.ch, d.j);
    d.next(n);
  }
}

// ---------------------------------------------------------------------------
// K = K_x W + K_y W of one x-y plane (wavelet z index i3 + N3 s3; the two
// planes of a coarse z are neighbouring tiles: they read the same fine
// records).
//
// Eight lanes take the 64 values of a 4 x 4 block of coarse points: for K_x
// a lane per row (o, s2), its results the eight columns (o1, s1); for K_y a
// lane per column, its results the eight rows.  An 8 x 8 transposition between
// lanes and registers brings K_x into K_y's layout and the sum goes to memory
// once, 16 neighbouring columns per half-row of lanes.  The plane in LDS is
// only read, so its one barrier is after the load, and K makes no second trip:
// K_y written, read back and added to K_x moved 32 B per point in place of 16
// (50 in place of 26 with PC), at 4.2 to 4.8 TB/s.  40^3 x 128 (65 M points):
// 0.50 -> 0.47 ms, 64^3 x 48: 0.96 -> 0.80, PC 2 of 48^3 x 64: 0.63 -> 0.53;
// bound by the vector units, three quarters of whose instructions are the
// stencils.
//
// LDS: rows j2, c and d of a coarse x side by side (one 16-byte read per tap
// of K_x), a stride of an odd number of such pairs.  Lane bits: o 0-1, s 4,
// blocks 2, 3, 5: 16 lanes of K_x read four rows of four neighbouring blocks,
// 32 lanes of K_y 32 neighbouring values, all in distinct banks.
//
// PC: the last half of the preconditioner's A v = S (K + c) S v, W = S v of
// the compressed vector v and c W + K_z W in K (k_pcz): S (K + K_x W + K_y W)
// goes to the compressed vectors.  1, v = x: r = b - A x, d = r, partial
// |r|^2; 2, v = d: q = A d, partial q d = (K + K_x W + K_y W) W.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int pair_stride(int N) { return 2 * ((N + 1) | 1); }

// register pair (a, b) <-> lane bit 0 or 1 (CTRL: the quad_perm of that
// exchange), bit: this lane's value of it
template <int CTRL>
__device__ __forceinline__ unsigned quad_lane(unsigned x) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ void swap_quad(double& a, double& b, bool bit) {
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  // every lane takes part in the exchange, then chooses
  const uint2 u = make_uint2(quad_lane<CTRL>(x.x), quad_lane<CTRL>(x.y));
  const uint2 w = make_uint2(quad_lane<CTRL>(y.x), quad_lane<CTRL>(y.y));
  const uint2 p = make_uint2(bit ? w.x : x.x, bit ? w.y : x.y);
  const uint2 q = make_uint2(bit ? y.x : u.x, bit ? y.y : u.y);
  a = __builtin_bit_cast(double, p);
  b = __builtin_bit_cast(double, q);
}
// ... <-> lane bit 4
__device__ __forceinline__ void swap_row16(double& a, double& b) {
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  const auto lo = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
  a = __builtin_bit_cast(double, make_uint2(lo[0], hi[0]));
  b = __builtin_bit_cast(double, make_uint2(lo[1], hi[1]));
}
// v[4 s + o] of lane (s', o') <-> v[4 s' + o'] of lane (s, o)
__device__ __forceinline__ void transpose8(double v[8]) {
  const bool o0 = threadIdx.x & 1, o1 = threadIdx.x & 2;
#pragma unroll
  for (int r = 0; r < 4; ++r) swap_row16(v[r], v[4 + r]);
#pragma unroll
  for (int r = 0; r < 8; r += 2) swap_quad<0xb1>(v[r], v[r + 1], o0);
#pragma unroll
  for (int r = 0; r < 8; r += 4) {
    swap_quad<0x4e>(v[r], v[r + 2], o1);
    swap_quad<0x4e>(v[r + 1], v[r + 3], o1);
  }
}

// Component t = s1 + 2 s2 + 4 s3 of the compressed vectors: index of a grid
// point's record (t = 0: scaling coefficient), -1 where it has none, and the
// byte offset of its value
struct Comp {
  const int* inv;
  unsigned off, mul;
  __device__ __forceinline__ Comp(const BoxDesc& bd, int t)
      : inv(t == 0 ? bd.cinv : bd.finv), off(t == 0 ? 0u : 8u * (unsigned)(bd.nvctr_c + t - 1)),
        mul(t == 0 ? 8u : 56u) {}
  __device__ __forceinline__ int index(int lin) const { return inv ? inv[lin] : lin; }
  __device__ __forceinline__ unsigned at(int i) const { return off + mul * (unsigned)i; }
};

template <int NTM, int PC>
__device__ __forceinline__ void xykin_tile(const Batch& B, const TileTable& tt,
                                           const TileTable& ft, const PcArgs& P, int tile,
                                           unsigned char* smem) {
  const int lb = find_box(tt, tile);
  const int b = table_box(tt, lb);
  const BoxDesc bd = B.box[b];
  const int lt = tile - box_first_tile(tt, lb);
  const int N1 = bd.N[0], N2 = bd.N[1], N3 = bd.N[2], per = bd.per;
  const int s3 = lt & 1, i3 = lt >> 1;
  const int W1 = 2 * N1, W2 = 2 * N2, RA = pair_stride(N1), npl = N1 * N2;
  double* A = (double*)smem;
  int2* my = (int2*)(A + (W2 + 1) * RA);
  int* mx = (int*)(my + map_len(N2));
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lin0 = npl * i3;
  const int st = nt >> 2;
  {
    // gather: thread's component c = s1 + 2 s2 of every (nt / 4)-th point
    constexpr int UR = 8;
    const int c = tid & 3;
    const Comp cp(bd, c + 4 * s3);
    const double sc = PC ? P.pc[9 * b + 1 + c + 4 * s3] : 1.0;
    const char* src = (const char*)((PC == 0 ? B.psi : PC == 1 ? P.x : P.d) + bd.psi_off);
    const bool dense = !bd.cinv && !bd.finv;
    double* base = A + (c >> 1) * N2 * RA + (c & 1);
    ItDiv d(tid >> 2, N1, st);
    for (int pb = tid >> 2; pb < npl; pb += st * UR) {
      double v[UR];
      if (dense) {
#pragma unroll
        for (int u = 0; u < UR; ++u)
          v[u] = *(const double*)(src + cp.at(lin0 + min(pb + u * st, npl - 1)));
      } else {
        int r[UR];
#pragma unroll
        for (int u = 0; u < UR; ++u) {
          const int p = pb + u * st;
          r[u] = -1;
          if (p < npl) r[u] = cp.index(lin0 + p);
        }
#pragma unroll
        for (int u = 0; u < UR; ++u)
          v[u] = r[u] >= 0 ? *(const double*)(src + cp.at(r[u])) : 0.0;
      }
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        if (pb + u * st < npl) base[d.ch * RA + 2 * d.j] = PC ? sc * v[u] : v[u];
        d.next(N1);
      }
    }
  }
  build_map(my, N2, per, RA * sizeof(double), W2, tid, nt);
  for (int e = tid; e < map_len(N1); e += nt) {
    int k = e - MOFF;
    if (per) {
      while (k < 0) k += N1;
      while (k >= N1) k -= N1;
    } else if ((unsigned)k >= (unsigned)N1) {
      k = N1;   // a pair of zeros
    }
    mx[e] = 16 * k;
  }
  for (int i = tid; i < W2; i += nt) *(double2*)(A + i * RA + W1) = make_double2(0.0, 0.0);
  for (int i = tid; i < RA; i += nt) A[W2 * RA + i] = 0.0;
  __syncthreads();
  const double kx = bd.kscale[0], ky = bd.kscale[1];
  const int cx = (N1 + 3) >> 2, nblk = cx * ((N2 + 3) >> 2);
  const float icx = 1.0f / (float)cx;
  double* K = (double*)B.K + bd.w_off + (long long)W1 * W2 * (i3 + N3 * s3);
  double sum = 0.0;
  for (int b0 = 8 * __builtin_amdgcn_readfirstlane(tid >> 6); b0 < nblk; b0 += nt >> 3) {
    int l = tid;   // opaque: what follows from it is not held over the loop
    asm volatile("" : "+v"(l));
    const int o = l & 3, s = (l >> 4) & 1, g = ((l >> 2) & 3) + 4 * ((l >> 5) & 1);
    const int blk = min(b0 + g, nblk - 1);
    const int chy = qdiv(blk, cx, icx), i1 = 4 * (blk - chy * cx), i2 = 4 * chy;
    const int x = min(i1 + o, N1 - 1);                     // lane's column
    const int row = s * N2 + min(i2 + o, N2 - 1);          // and row
    // results of this lane: rows i2 + r (s2 = 0: h = r, 1: h = 4 + r)
    const int nrow = b0 + g < nblk && i1 + o < N1 ? N2 - i2 : 0;
    // byte offset of the first of them from the plane's K (uniform base)
    const unsigned at = 8u * (unsigned)(x + N1 * s + W1 * i2);
    auto kp = [&](int h) {
      return (double*)((char*)K + (at + 8u * (unsigned)(W1 * ((h & 3) + (h >> 2) * N2))));
    };
    double vx[8], vy[8];
#pragma unroll
    for (int h = 0; h < 8; ++h) vx[h] = vy[h] = 0.0;
    {
      const char* a = (const char*)(A + row * RA);
      const int* m = mx + (i1 - 14 + MOFF);
      kin_order([&](int kk) {
        const double2 w = *(const double2*)(a + m[kk]);
        kin_tap(kk, w.x, w.y, vx, vx + 4);
      });
    }
    transpose8(vx);
    const double* col = A + 2 * x + s;
    if (__all(i2 >= 14 && i2 + 17 < N2)) {
      const double *yc = col + (i2 - 14) * RA, *yd = yc + N2 * RA;
      kin_order([&](int kk) { kin_tap(kk, yc[kk * RA], yd[kk * RA], vy, vy + 4); });
    } else {
      const int2* m = my + (i2 - 14 + MOFF);
      kin_order([&](int kk) {
        const double2 w = at2(col, m[kk]);
        kin_tap(kk, w.x, w.y, vy, vy + 4);
      });
    }
    if (PC) {
#pragma unroll
      for (int h = 0; h < 8; ++h) vx[h] = fma(vy[h], ky, vx[h] * kx);
      double k[8];
#pragma unroll
      for (int h = 0; h < 8; ++h) k[h] = (h & 3) < nrow ? *kp(h) : 0.0;
#pragma unroll
      for (int h = 0; h < 8; ++h) vx[h] += k[h];
    } else {
#pragma unroll
      for (int h = 0; h < 8; ++h) vx[h] = fma(vy[h], ky, vx[h] * kx);
    }
    if (PC < 2) {
#pragma unroll
      for (int h = 0; h < 8; ++h)
        if ((h & 3) < nrow) *kp(h) = vx[h];
    } else {
      char* q = (char*)(P.q + bd.psi_off);
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const int r = h & 3, s2 = h >> 2, t = s + 2 * s2 + 4 * s3;
        const Comp cp(bd, t);
        int i = -1;
        if (r < nrow) i = cp.index(lin0 + x + N1 * (i2 + r));
        if (i >= 0) {
          *(double*)(q + cp.at(i)) = P.pc[9 * b + 1 + t] * vx[h];
          sum = fma(vx[h], col[(s2 * N2 + i2 + r) * RA], sum);
        }
      }
    }
  }
  if constexpr (PC == 1) {
    // r and d in the order of the records: three streams of single values from
    // the blocks' lanes took 0.89 ms, K through memory 0.66
    __syncthreads();
    constexpr int UR = 4;
    int to = tid;   // opaque, as in the loop
    asm volatile("" : "+v"(to));
    const int c = to & 3;
    const Comp cp(bd, c + 4 * s3);
    const double sc = P.pc[9 * b + 1 + c + 4 * s3];
    const char* y = (const char*)(P.b + bd.psi_off);
    char* rr = (char*)(P.r + bd.psi_off);
    char* dd = (char*)(P.d + bd.psi_off);
    const double* kc = K + (size_t)((c >> 1) * N2) * W1 + (c & 1) * N1;
    ItDiv d(to >> 2, N1, st);
    for (int pb = to >> 2; pb < npl; pb += st * UR) {
      int r[UR];
      double k[UR], v[UR];
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        const int p = pb + u * st;
        r[u] = -1;
        if (p < npl) r[u] = cp.index(lin0 + p);
        k[u] = p < npl ? kc[d.ch * W1 + d.j] : 0.0;
        d.next(N1);
      }
#pragma unroll
      for (int u = 0; u < UR; ++u) v[u] = r[u] >= 0 ? *(const double*)(y + cp.at(r[u])) : 0.0;
#pragma unroll
      for (int u = 0; u < UR; ++u)
        if (r[u] >= 0) {
          const double rv = v[u] - sc * k[u];
          *(double*)(rr + cp.at(r[u])) = rv;
          *(double*)(dd + cp.at(r[u])) = rv;
          sum = fma(rv, rv, sum);
        }
    }
  }
  if constexpr (PC != 0) {
    __shared__ double red[NTM / 64];
    const double v = block_sum_rt(sum, red);
    if (tid == 0) P.part[box_first_tile(ft, b) + lt] = v;
  }
}

template <int NTM, int WPE, int PC>
__global__ __launch_bounds__(NTM, WPE) void k_xykin(Batch B, TileTable tt, TileTable ft,
                                                    PcArgs P) {
  extern __shared__ __align__(16) unsigned char smem[];
  xykin_tile<NTM, PC>(B, tt, ft, P, tile_of(tt), smem);
}

// Both kernels that read psi alone in one launch: nx planes of k_xykin, then
// the tiles of k_zgrow.
template <int NTM>
__global__ __launch_bounds__(NTM, 6) void k_zgrow_xykin(Batch B, TileTable tz, TileTable tx,
                                                        int nx) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int b = blockIdx.x;
  if (b < nx)
    xykin_tile<NTM, 0>(B, tx, tx, PcArgs{}, tx.xcd ? xcd_tile(b, nx) : b, smem);
  else
    zgrow_tile<NTM>(B, tz, tz.xcd ? xcd_tile(b - nx, gridDim.x - nx) : b - nx, smem);
}

// ---------------------------------------------------------------------------
// A plane of TZ (2 N1 x 2 N2) in LDS: x lines as rows (stride RX) for G_x and
// G_x^T, y lines as rows (RY) in between.
// ---------------------------------------------------------------------------
struct Plane {
  int N1, N2, L1, L2, per, W1, W2, RX, RY;
  double* A;
  int2 *mx, *my;   // line maps, one pair for both axes of a square plane
  int *sx, *sy;
  ItDiv dn, dw, dl;   // first pair of values, first x and y items
  __device__ __forceinline__ Plane(const BoxDesc& bd, unsigned char* smem)
      : N1(bd.N[0]), N2(bd.N[1]), L1(bd.L[0]), L2(bd.L[1]), per(bd.per), W1(2 * N1),
        W2(2 * N2), RX(L1 | 1), RY(L2 | 1), A((double*)smem + PAD),
        dn(threadIdx.x, N1, blockDim.x), dw(threadIdx.x, W2, blockDim.x),
        dl(threadIdx.x, L1, blockDim.x) {
    const bool sq = N1 == N2;
    mx = (int2*)(A + max(W2 * RX, L1 * RY) + PADE);
    my = mx + (sq ? 0 : cmap_len(N1));
    sx = (int*)(my + cmap_len(N2));
    sy = sx + (sq ? 0 : smap_len(N1));
    if (per) {
      build_maps(mx, sx, N1, threadIdx.x, blockDim.x);
      if (!sq) build_maps(my, sy, N2, threadIdx.x, blockDim.x);
    }
  }
  // the thread's items, opaque: addresses and line-end masks made from them
  // are neither moved out of a loop over planes nor shared between passes
  // (either way they spill; a kernel that uses scratch memory starts 0.13 ms
  // late on a queue that has run none: the first apply on a new stream of one
  // 16^3 orbital took 0.32 to 0.45 ms in place of 0.20)
  __device__ __forceinline__ void opaque() {
    asm volatile("" : "+v"(dn.ch), "+v"(dn.j));
    opaque_xy();
  }
  __device__ __forceinline__ void opaque_xy() {
    asm volatile("" : "+v"(dw.ch), "+v"(dw.j), "+v"(dl.ch), "+v"(dl.j));
  }
  // T's plane into the x rows, two values at a time (rows of 2 N1, planes of
  // 4 N1 N2 values: 16-byte aligned)
  __device__ __forceinline__ void load(const double* T) const {
    constexpr int UR = 4;
    const int tot = N1 * W2, nt = blockDim.x;
    const double2* src = (const double2*)T;
    ItDiv d = dn;
    for (int i = threadIdx.x; i < tot; i += nt * UR) {
      double2 v[UR];
#pragma unroll
      for (int u = 0; u < UR; ++u) v[u] = src[min(i + u * nt, tot - 1)];
#pragma unroll
      for (int u = 0; u < UR; ++u) {
        if (i + u * nt < tot) {
          double* a = A + d.ch * RX + 2 * d.j;
          a[0] = v[u].x;
          a[1] = v[u].y;
        }
        d.next(N1);
      }
    }
  }
  // G_x on the rows j2, written as columns of the y rows (barriers: the plane
  // is loaded before, the y rows are complete after)
  template <int MI>
  __device__ __forceinline__ void grow_x(double o[MI][8]) const {
    const int gx = (L1 + 7) >> 3;
    __syncthreads();
    each_item<MI>(dw, W2, gx, [&](int m, int ch, int j2) {
      grow_row(A + j2 * RX, mx, N1, grow_k0(8 * ch, per), per, o[m]);
    });
    __syncthreads();
    each_item<MI>(dw, W2, gx, [&](int m, int ch, int j2) {
      double* a = A + 8 * ch * RY + j2;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        if (8 * ch + r < L1) a[r * RY] = o[m][r];
    });
    __syncthreads();
  }
  __device__ __forceinline__ void grow_y(int ch, int p1, double o[8]) const {
    grow_row(A + p1 * RY, my, N2, grow_k0(8 * ch, per), per, o);
  }
};

// ---------------------------------------------------------------------------
// TZ <- G_x^T G_y^T V G_y G_x TZ of the plane at fine z point p3, epot
// partial
// ---------------------------------------------------------------------------
template <int NTM, int MI, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_xypot(Batch B, TileTable tt, TileTable ft,
                                                    double* part) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[NTM / 64];
  const int tile = tile_of(tt);
  const int lb = find_box(tt, tile);
  const int b = table_box(tt, lb);
  const BoxDesc bd = B.box[b];
  const int p3 = tile - box_first_tile(tt, lb);
  Plane P(bd, smem);
  const int N1 = P.N1, N2 = P.N2, L1 = P.L1, L2 = P.L2, per = P.per;
  const int W2 = P.W2, RX = P.RX, RY = P.RY;
  double* A = P.A;
  double* T = (double*)B.TZ + bd.tz_off + (long long)P.W1 * W2 * p3;
  P.load(T);
  double o[MI][8];
  P.grow_x<MI>(o);
  P.opaque_xy();
  const int gy = (L2 + 7) >> 3;
  // G_y and V on the rows p1.  V outside the potential box is zero, the
  // zeroing of psir there (potential.f90:874-947); those points read a value
  // of the box and discard it, so all loads of a chunk are in flight together
  // while its stencil runs.
  const int q3 = p3 - bd.ishift[2];
  const bool in3 = q3 >= 0 && q3 < bd.potdim[2];
  const unsigned pd1 = (unsigned)bd.potdim[0];
  const double* pot = B.pot + bd.pot_off +
                      (size_t)pd1 * (unsigned)bd.potdim[1] *
                          (unsigned)min(max(q3, 0), bd.potdim[2] - 1);
  const double cz = bd.conf_on ? conf_axis2(bd, 2, p3) : 0.0;
  double ep = 0.0;
  each_item<MI>(P.dl, L1, gy, [&](int m, int ch, int p1) {
    const int q1 = p1 - bd.ishift[0], q20 = 8 * ch - bd.ishift[1];
    // rows of the chunk inside the box and the potential box
    const bool in13 = in3 && q1 >= 0 && q1 < bd.potdim[0];
    const int rlo = -q20, rhi = in13 ? min(L2 - 8 * ch, bd.potdim[1] - q20) : 0;
    double v[8];
    const bool whole = __all(rlo <= 0 && rhi >= 8);
    if (whole) {
      const unsigned v0 = 8u * ((unsigned)q1 + pd1 * (unsigned)q20);
#pragma unroll
      for (int r = 0; r < 8; ++r)
        v[r] = *(const double*)((const char*)(pot + r * (size_t)pd1) + v0);
    } else {
      const unsigned v0 = (unsigned)min(max(q1, 0), bd.potdim[0] - 1);
#pragma unroll
      for (int r = 0; r < 8; ++r)
        v[r] = pot[v0 + pd1 * (unsigned)min(max(q20 + r, 0), bd.potdim[1] - 1)];
    }
    P.grow_y(ch, p1, o[m]);
    if (bd.conf_on || !whole) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const bool ok = r >= rlo && r < rhi;
        v[r] = ok ? v[r] : 0.0;
        if (bd.conf_on && ok)
          v[r] += conf_term(bd, cz + conf_axis2(bd, 0, p1) + conf_axis2(bd, 1, 8 * ch + r));
      }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const double vp = v[r] * o[m][r];
      ep = fma(vp, o[m][r], ep);
      o[m][r] = vp;
    }
  });
  __syncthreads();
  each_item<MI>(P.dl, L1, gy, [&](int m, int ch, int p1) {
    double* a = A + p1 * RY + 8 * ch;
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (8 * ch + r < L2) a[r] = o[m][r];
  });
  __syncthreads();
  P.opaque_xy();
  // G_y^T on the rows p1, written as columns of the x rows
  const int cy = (N2 + 3) >> 2, cx = (N1 + 3) >> 2;
  each_item<MI>(P.dl, L1, cy, [&](int m, int ch, int p1) {
    shrink_row(A + p1 * RY, P.sy, L2, 4 * ch, per, o[m]);
  });
  __syncthreads();
  each_item<MI>(P.dl, L1, cy, [&](int m, int ch, int p1) {
    double* a = A + 4 * ch * RX + p1;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * ch + r < N2) {
        a[r * RX] = o[m][r];
        a[(N2 + r) * RX] = o[m][4 + r];
      }
  });
  __syncthreads();
  P.opaque_xy();
  // G_x^T on the rows j2
  each_item<MI>(P.dw, W2, cx, [&](int m, int ch, int j2) {
    shrink_row(A + j2 * RX, P.sx, L1, 4 * ch, per, o[m]);
  });
  __syncthreads();
  each_item<MI>(P.dw, W2, cx, [&](int m, int ch, int j2) {
    double* a = A + j2 * RX + 4 * ch;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * ch + r < N1) {
        a[r] = o[m][r];
        a[N1 + r] = o[m][4 + r];
      }
  });
  const double eps = block_sum_rt(ep, red);   // has the barriers
  if (threadIdx.x == 0) part[box_first_tile(ft, b) + p3] = eps;
  {
    const int tot = N1 * W2;
    double2* dst = (double2*)T;
    int tid = threadIdx.x;   // opaque: counted anew, not held through the passes
    asm volatile("" : "+v"(tid));
    ItDiv d(tid, N1, blockDim.x);
    for (int i = tid; i < tot; i += (int)blockDim.x) {
      const double* a = A + d.ch * RX + 2 * d.j;
      dst[i] = make_double2(a[0], a[1]);
      d.next(N1);
    }
  }
}

// ---------------------------------------------------------------------------
// Boxes whose planes do not fit in LDS (beyond 70 periodic, 55 or 70 free
// coarse points on x and y): the x and y passes on tiles of 64 lines, a lane
// per line and a wave per chunk as in the z kernels.
//   k_xlines_grow    TX = G_x TZ, TX[p3][p1][j2] (y fastest: the lanes' lines
//                    j2 are neighbours, and the y lines are rows again)
//   k_ylines_pot     TX <- G_y^T V G_y TX in place, epot partial
//   k_xlines_shrink  TZ = G_x^T TX
//   k_xlines_kin     K = K_x W,  k_ylines_kin  K += K_y W
// Rows of memory go through LDS as columns of stride LR (odd: neither side
// meets a bank twice).  77x93x131, 8 orbitals (60 M points): 0.21, 0.42, 0.22,
// 0.30 and 0.36 ms, 16 to 24 B per point at 2.2 to 4.8 TB/s; the apply 2.34 ms,
// 5.50 ms on the line passes of bdft_pass.hip.  Per point the planes move
// less (20 ps, these 25), so boxes whose planes fit keep them.
// Work-groups of 12 or 16 waves, two on a CU while the lines leave LDS and
// registers for two; the outputs that replace a tile's inputs are held in
// registers, MI chunks per wave (with 8 waves and five chunks each the three
// code paths of every chunk did not fit the instruction cache: k_xlines_kin
// 0.64 ms).
// ---------------------------------------------------------------------------
constexpr int LR = NL + 1;

// nr rows of n values (n even, 16-byte aligned) <-> LDS [x LR + row]
template <bool STORE>
__device__ __forceinline__ void rows_move(double* lds, double* mem, int nr, int n) {
  constexpr int UR = 4;
  const int h = n >> 1, tot = nr * h, nt = blockDim.x;
  double2* m2 = (double2*)mem;
  ItDiv d(threadIdx.x, h, nt);
  for (int i = threadIdx.x; i < tot; i += nt * UR) {
    double2 v[UR];
    if (!STORE) {
#pragma unroll
      for (int u = 0; u < UR; ++u) v[u] = m2[min(i + u * nt, tot - 1)];
    }
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      double* a = lds + 2 * d.j * LR + d.ch;
      if (i + u * nt < tot) {
        if (STORE) {
          m2[i + u * nt] = make_double2(a[0], a[LR]);
        } else {
          a[0] = v[u].x;
          a[LR] = v[u].y;
        }
      }
      d.next(h);
    }
  }
}

template <int NTM, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_xlines_grow(Batch B, TileTable tt) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  const int tile = tile_of(tt);
  const int b = find_box(tt, tile);
  const BoxDesc bd = B.box[b];
  const int N1 = bd.N[0], L1 = bd.L[0], L3 = bd.L[2], per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * bd.N[1];
  const int r0 = (tile - box_first_tile(tt, b)) * NL, nr = min(NL, W2 * L3 - r0);
  rows_move<false>(lds, (double*)B.TZ + bd.tz_off + (long long)r0 * W1, nr, W1);
  __syncthreads();
  const int lane = threadIdx.x & 63, r = r0 + min(lane, nr - 1);
  const int p3 = r / W2, j2 = r - p3 * W2;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* out = (double*)B.T2 + bd.t2_off + (long long)p3 * L1 * W2 + j2;
  const double *c = lds + lane, *d = c + N1 * LR;
  for (int p0 = 8 * w; p0 < L1; p0 += 8 * (NTM / 64)) {
    double o[8] = {};
    line_taps<19>(grow_k0(p0, per), N1, per,
                  [&](int kk, int k) { grow_tap(kk, c[k * LR], d[k * LR], o); });
    if (lane < nr) {
#pragma unroll
      for (int h = 0; h < 8; ++h)
        if (p0 + h < L1) out[(size_t)W2 * (unsigned)(p0 + h)] = o[h];
    }
  }
}

template <int NTM, int MI, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_ylines_pot(Batch B, TileTable tt, double* part) {
  constexpr int NW = NTM / 64;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  __shared__ double red[NW];
  const int tile = tile_of(tt);
  const int b = find_box(tt, tile);
  const BoxDesc bd = B.box[b];
  const int L1 = bd.L[0], N2 = bd.N[1], L2 = bd.L[1], L3 = bd.L[2], per = bd.per;
  const int W2 = 2 * N2;
  const int r0 = (tile - box_first_tile(tt, b)) * NL, nr = min(NL, L1 * L3 - r0);
  double* T = (double*)B.T2 + bd.t2_off + (long long)r0 * W2;
  rows_move<false>(lds, T, nr, W2);
  __syncthreads();
  const int lane = threadIdx.x & 63, r = r0 + min(lane, nr - 1);
  const int p3 = r / L1, p1 = r - p3 * L1;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (lanes past the tile walk its last line again and store nothing)
  const bool on = lane < nr;
  double* col = lds + min(lane, nr - 1);
  // V outside the potential box is zero; lanes off it read a value of the box
  // and discard it
  const int q1 = p1 - bd.ishift[0], q3 = p3 - bd.ishift[2];
  const bool in13 = on && q1 >= 0 && q1 < bd.potdim[0] && q3 >= 0 && q3 < bd.potdim[2];
  const unsigned pd1 = (unsigned)bd.potdim[0], pd2 = (unsigned)bd.potdim[1];
  const unsigned v0 = in13 ? (unsigned)q1 + pd1 * pd2 * (unsigned)q3 : 0u;
  const double* pot = B.pot + bd.pot_off;
  const double cxz = bd.conf_on ? conf_axis2(bd, 0, p1) + conf_axis2(bd, 2, p3) : 0.0;
  double o[MI][8];
  double ep = 0.0;
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int p0 = 8 * (w + m * NW);
    if (p0 < L2) {
      double v[8];
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const int q2 = p0 + h - bd.ishift[1];
        v[h] = pot[v0 + pd1 * (unsigned)min(max(q2, 0), bd.potdim[1] - 1)];
        o[m][h] = 0.0;
      }
      line_taps<19>(grow_k0(p0, per), N2, per, [&](int kk, int k) {
        grow_tap(kk, col[k * LR], col[(N2 + k) * LR], o[m]);
      });
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        const int q2 = p0 + h - bd.ishift[1];
        const bool ok = in13 && p0 + h < L2 && q2 >= 0 && q2 < bd.potdim[1];
        double vr = ok ? v[h] : 0.0;
        if (bd.conf_on && ok) vr += conf_term(bd, cxz + conf_axis2(bd, 1, p0 + h));
        const double vp = vr * o[m][h];
        ep = fma(vp, o[m][h], ep);
        o[m][h] = vp;
      }
    }
  }
  const double eps = block_sum_rt(ep, red);   // starts with a barrier
  if (threadIdx.x == 0) part[tile] = eps;
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int p0 = 8 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 8; ++h)
      if (on && p0 + h < L2) col[(p0 + h) * LR] = o[m][h];
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 8; ++h) o[m][h] = 0.0;
    if (i0 < N2)
      line_taps<37>(per ? 2 * i0 - 14 : 2 * i0, L2, per, [&](int qq, int p) {
        shrink_tap<double, 4>(qq, col[p * LR], o[m], o[m] + 4);
      });
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (on && i0 + h < N2) {
        col[(i0 + h) * LR] = o[m][h];
        col[(N2 + i0 + h) * LR] = o[m][4 + h];
      }
  }
  __syncthreads();
  rows_move<true>(lds, T, nr, W2);
}

template <int NTM, int MI, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_xlines_shrink(Batch B, TileTable tt) {
  constexpr int NW = NTM / 64, UR = 8;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  const int tile = tile_of(tt);
  const int b = find_box(tt, tile);
  const BoxDesc bd = B.box[b];
  const int N1 = bd.N[0], L1 = bd.L[0], L3 = bd.L[2], per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * bd.N[1];
  const int r0 = (tile - box_first_tile(tt, b)) * NL, nr = min(NL, W2 * L3 - r0);
  const int lane = threadIdx.x & 63, r = r0 + min(lane, nr - 1);
  const int p3 = r / W2, j2 = r - p3 * W2;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double* src = (const double*)B.T2 + bd.t2_off + (long long)p3 * L1 * W2 + j2;
  double* col = lds + lane;
  for (int pb = w; pb < L1; pb += NW * UR) {
    double v[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) v[u] = src[(size_t)W2 * (unsigned)min(pb + u * NW, L1 - 1)];
#pragma unroll
    for (int u = 0; u < UR; ++u)
      if (pb + u * NW < L1) col[(pb + u * NW) * LR] = v[u];
  }
  __syncthreads();
  double o[MI][8];
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 8; ++h) o[m][h] = 0.0;
    if (i0 < N1)
      line_taps<37>(per ? 2 * i0 - 14 : 2 * i0, L1, per, [&](int qq, int p) {
        shrink_tap<double, 4>(qq, col[p * LR], o[m], o[m] + 4);
      });
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (i0 + h < N1) {
        col[(i0 + h) * LR] = o[m][h];
        col[(N1 + i0 + h) * LR] = o[m][4 + h];
      }
  }
  __syncthreads();
  rows_move<true>(lds, (double*)B.TZ + bd.tz_off + (long long)r0 * W1, nr, W1);
}

// x lines of 16 rows q = i2 + N2 i3 of coarse points: line row + 16 (s2 + 2
// s3), gathered a row per wave (its records are contiguous)
template <int NTM, int MI, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_xlines_kin(Batch B, TileTable tt) {
  constexpr int NW = NTM / 64, UR = 8, ZS = NTM / 128;
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  const int tile = tile_of(tt);
  const int b = find_box(tt, tile);
  const BoxDesc bd = B.box[b];
  const int N1 = bd.N[0], N2 = bd.N[1], N3 = bd.N[2], per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * N2;
  const int q0 = (tile - box_first_tile(tt, b)) * CC, nq = min(CC, N2 * N3 - q0);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // 128 threads per 16 records of a row, as load_columns
  const RecElem<> re(threadIdx.x & 127);
  const int z0 = threadIdx.x >> 7, nit = CC * ((N1 + CC - 1) / CC);
  const char* src = (const char*)(B.psi + bd.psi_off);
  const unsigned off = re.t == 0 ? 0u : 8u * (unsigned)(bd.nvctr_c + re.t - 1);
  const unsigned mul = re.t == 0 ? 8u : 56u;
  const int* inv = re.t == 0 ? bd.cinv : bd.finv;
  double* dst = lds + (re.t & 1) * N1 * LR + CC * (re.t >> 1);
  for (int ib = z0; ib < nit; ib += ZS * UR) {
    double v[UR];
    int r[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const int it = ib + u * ZS, row = it & (CC - 1), x = (it & -CC) + re.col;
      r[u] = -1;
      if (row < nq && x < N1) {
        const int lin = (q0 + row) * N1 + x;
        r[u] = inv ? inv[lin] : lin;
      }
    }
#pragma unroll
    for (int u = 0; u < UR; ++u)
      v[u] = r[u] >= 0 ? *(const double*)(src + (off + mul * (unsigned)r[u])) : 0.0;
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const int it = ib + u * ZS, row = it & (CC - 1), x = (it & -CC) + re.col;
      if (it < nit && x < N1) dst[x * LR + row] = v[u];
    }
  }
  __syncthreads();
  double* col = lds + lane;
  const double ks = bd.kscale[0];
  double o[MI][8];
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 8; ++h) o[m][h] = 0.0;
    if (i0 < N1)
      kin_taps(i0 - 14, N1, per, [&](int kk, int k) {
        kin_tap(kk, col[k * LR], col[(N1 + k) * LR], o[m], o[m] + 4);
      });
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int i0 = 4 * (w + m * NW);
#pragma unroll
    for (int h = 0; h < 4; ++h)
      if (i0 + h < N1) {
        col[(i0 + h) * LR] = o[m][h] * ks;
        col[(N1 + i0 + h) * LR] = o[m][4 + h] * ks;
      }
  }
  __syncthreads();
  for (int l = w; l < NL; l += NW) {
    const int row = l & (CC - 1), s = l / CC, q = q0 + row;
    if (row < nq) {
      const int i3 = q / N2, i2 = q - i3 * N2;
      double* k = (double*)B.K + bd.w_off +
                  (long long)W1 * (i2 + N2 * (s & 1) + W2 * (i3 + N3 * (s >> 1)));
      for (int x = lane; x < W1; x += 64) k[x] = lds[x * LR + l];
    }
  }
}

// y lines of 16 coarse x of one coarse z: line col + 16 (s1 + 2 s3)
template <int NTM, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_ylines_kin(Batch B, TileTable tt) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* lds = (double*)smem;
  const int tile = tile_of(tt);
  const int b = find_box(tt, tile);
  const BoxDesc bd = B.box[b];
  const int N1 = bd.N[0], N2 = bd.N[1], N3 = bd.N[2], per = bd.per;
  const int W1 = 2 * N1, W2 = 2 * N2, nx = (N1 + CC - 1) / CC;
  const int lt = tile - box_first_tile(tt, b), i3 = lt / nx, x0 = (lt - i3 * nx) * CC;
  const int nq = min(CC, N1 - x0);
  load_columns<NTM, 1>(lds, bd, B.psi, x0 + N1 * N2 * i3, nq);
  __syncthreads();
  const int lane = threadIdx.x & 63, cl = lane & (CC - 1), s = lane / CC;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool on = cl < nq;
  double* K = (double*)B.K + bd.w_off + (x0 + (on ? cl : 0) + N1 * (s & 1)) +
              (long long)W1 * W2 * (i3 + N3 * (s >> 1));
  const double *c = lds + lane, *d = c + N2 * NL;
  const double ks = bd.kscale[1];
  for (int i0 = 4 * w; i0 < N2; i0 += 4 * (NTM / 64)) {
    double k[8], o[8] = {};
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int i = min(i0 + h, N2 - 1);
      k[h] = K[W1 * i];
      k[4 + h] = K[W1 * (N2 + i)];
    }
    kin_taps(i0 - 14, N2, per,
                  [&](int kk, int i) { kin_tap(kk, c[i * NL], d[i * NL], o, o + 4); });
    if (on) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
        if (i0 + h < N2) {
          K[W1 * (i0 + h)] = fma(o[h], ks, k[h]);
          K[W1 * (N2 + i0 + h)] = fma(o[4 + h], ks, k[4 + h]);
        }
    }
  }
}

// ---------------------------------------------------------------------------
// density (local_partial_density, sumrho.f90:377-469): the planes p3 of TZ of
// one group's orbitals (orbitals order[0 ..] of one spin, one box) in turn,
// psir = G_y G_x, and sum hfac psir^2 kept in registers, written once as the
// group's partial density.  Three items per thread (128 VGPRs) on 8 waves, two
// work-groups per CU: with the sums beside the passes' outputs, two items at
// 80 VGPRs spill (0.42 against 0.49 ms for 96 orbitals of a periodic 48^3
// box).  That batch, 8.5e7 points: unpack 0.23, x-y planes 0.51, z lines 0.43
// ms before, k_zgrow 0.27 and k_xyden 0.42 now (24 bytes per point for 40).
// ---------------------------------------------------------------------------
template <int NTM, int MI, int WPE>
__global__ __launch_bounds__(NTM, WPE) void k_xyden(Batch B, DenArgs D) {
  extern __shared__ __align__(16) unsigned char smem[];
  const BoxDesc bd = B.box[0];
  const int L3 = bd.L[2];
  const int g = blockIdx.x / L3, p3 = blockIdx.x - g * L3;
  Plane P(bd, smem);
  const long long plane = (long long)P.W1 * P.W2;
  const int gy = (P.L2 + 7) >> 3;
  double acc[MI][8];
#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[m][r] = 0.0;
  const int o1 = D.gstart[g + 1];
  for (int k = D.gstart[g]; k < o1; ++k) {
    const double hf = D.hfac[k];
    P.opaque();
    P.load((const double*)B.TZ + B.box[D.order[k]].tz_off + plane * p3);
    double o[MI][8];
    P.grow_x<MI>(o);
    each_item<MI>(P.dl, P.L1, gy, [&](int m, int ch, int p1) {
      double v[8];
      P.grow_y(ch, p1, v);
#pragma unroll
      for (int r = 0; r < 8; ++r) acc[m][r] += hf * (v[r] * v[r]);
    });
    __syncthreads();
  }
  double* dst = D.part + (long long)g * D.nisf + (long long)P.L1 * P.L2 * p3;
  each_item<MI>(P.dl, P.L1, gy, [&](int m, int ch, int p1) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
      if (8 * ch + r < P.L2) dst[p1 + P.L1 * (8 * ch + r)] = acc[m][r];
  });
}

// rho += sum of the group partials of a spin, groups in order
__global__ __launch_bounds__(256) void k_xyden_sum(DenArgs D) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= D.nisf) return;
  const int s = blockIdx.y;
  double a = 0.0;
  for (int g = s ? D.gspin : 0; g < (s ? D.ngroups : D.gspin); ++g) a += D.part[g * D.nisf + i];
  D.rho[s * D.nisf + i] += a;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// LDS bytes of the kernels for a box
constexpr size_t LDS_STATIC = 128;   // the kernels' static LDS (reductions)
// rows of W; of W or of TZ
static size_t lds_w(int N3, int cols = CC) { return (size_t)4 * cols * 2 * N3 * 8; }
size_t fp64_lds_z(const BoxDesc& b, int cols) {
  return (size_t)4 * cols * std::max(b.L[2], 2 * b.N[2]) * 8;
}
int fp64_zcols(const BoxDesc& b, size_t plane_lds) {
  for (int cols : {CC, CC / 2})
    if (fp64_lds_z(b, cols) + LDS_STATIC <= plane_lds) return cols;
  return 0;
}
static size_t fp64_lds_kin(int N1, int N2) {
  return 8 * ((size_t)(2 * N2 + 1) * pair_stride(N1) + map_len(N2)) + 4 * map_len(N1);
}
static size_t fp64_lds_pot(int N1, int N2, int L1, int L2) {
  const size_t x = (size_t)2 * N2 * (L1 | 1), y = (size_t)L1 * (L2 | 1);
  size_t maps = 0;
  if (L1 == 2 * N1) {
    maps = 8 * (size_t)cmap_len(N2) + 4 * (size_t)smap_len(N2);
    if (N1 != N2) maps += 8 * (size_t)cmap_len(N1) + 4 * (size_t)smap_len(N1);
  }
  return 8 * ((x > y ? x : y) + PAD + PADE) + maps;
}
// Launch shapes of the in-plane kernels by items (8 values) of a plane's
// largest pass and by the work-groups whose LDS fits a CU; work-groups of 4,
// 8, 12 or 16 waves, as many on each SIMD (work-groups of 7 and 13 waves ran
// 20 to 40 % slower, and two of 13 do not share a CU).  2 to 4: at least that
// many work-groups per CU, two items per thread (80 VGPRs: 24 waves per CU);
// 1: one, three items.
constexpr int S2_NT = 768, S1_NT = 1024;
static PlaneFit plane_fit(size_t lds, int items, size_t plane_lds) {
  plane_lds -= std::min(plane_lds, LDS_STATIC);
  if (items <= 512 && lds <= plane_lds / 4) return {4, items <= 256 ? 128 : 256, lds};
  if (items <= 1024 && lds <= plane_lds / 3) return {3, 512, lds};
  if (items <= 2 * S2_NT && lds <= plane_lds / 2) return {2, items <= 1024 ? 512 : 768, lds};
  if (items <= 3 * S1_NT && lds <= plane_lds) return {1, items <= 1536 ? 768 : 1024, lds};
  return {0, 0, lds};
}
static int chunks(int n, int len) { return (n + len - 1) / len; }
// do the line kernels hold a box's x and y lines?
static size_t lds_rows(int n) { return 8 * (size_t)LR * n; }
bool fp64_kin_lines_ok(const BoxDesc& b, size_t plane_lds) {
  return std::max(lds_rows(2 * b.N[0]), lds_w(b.N[1])) <= plane_lds;
}
// (K, TZ and TX of a flat free box can take more than the grids of the line
// passes, by which the fixed device array's entry admits it: half that array
// or the line passes' bytes bound them)
bool fp64_pot_lines_ok(const BoxDesc& b, size_t plane_lds) {
  const size_t n1 = 2 * b.N[0], n2 = 2 * b.N[1], n3 = 2 * b.N[2];
  const size_t l1 = b.L[0], l2 = b.L[1], l3 = b.L[2];
  return lds_rows(std::max(b.L[0], b.L[1])) + LDS_STATIC <= plane_lds &&
         n1 * n2 * (n3 + l3) + n2 * l1 * l3 <=
             std::max<size_t>(BDFT_FIXED_BYTES / 16,
                              2 * n1 * n2 * n3 + l1 * n2 * n3 + l1 * l2 * n3);
}
PlaneFit fp64_fit_kin(const BoxDesc& b, size_t plane_lds) {
  // a wave takes eight blocks of 4 x 4 points, any number of times
  const int nblk = chunks(b.N[0], 4) * chunks(b.N[1], 4);
  const size_t lds = fp64_lds_kin(b.N[0], b.N[1]);
  plane_lds -= std::min(plane_lds, LDS_STATIC);
  if (lds <= plane_lds / 4) return {4, nblk <= 32 ? 128 : 256, lds};
  if (lds <= plane_lds / 3) return {3, 512, lds};
  if (lds <= plane_lds / 2) return {2, S2_NT, lds};
  return {lds <= plane_lds ? 1 : 0, S1_NT, lds};
}
PlaneFit fp64_fit_pot(const BoxDesc& b, size_t plane_lds) {
  const int N1 = b.N[0], N2 = b.N[1], L1 = b.L[0], L2 = b.L[1];
  return plane_fit(fp64_lds_pot(N1, N2, L1, L2),
                   std::max(std::max(2 * N2 * chunks(L1, 8), L1 * chunks(L2, 8)),
                            std::max(L1 * chunks(N2, 4), 2 * N2 * chunks(N1, 4))),
                   plane_lds);
}

// the z kernels over the boxes of each tile width (shape 2: 16 columns, 1: 8):
// f(table, tiles, shape, longest line, LDS of the back pass)
template <typename F>
static hipError_t z_pass(const PassTables& PT, F f) {
  if (PT.n_zg == 0)
    return PT.ntiles[P_CZ] <= 0 ? hipSuccess
                                : f(PT.t[P_CZ], PT.ntiles[P_CZ], PT.shape_zg[0], PT.len_zg[0],
                                    PT.lds_zg[0]);
  hipError_t e = hipSuccess;
  for (int k = 0; k < PT.n_zg && e == hipSuccess; ++k)
    e = f(PT.zg[k], PT.nt_zg[k], PT.shape_zg[k], PT.len_zg[k], PT.lds_zg[k]);
  return e;
}
// 256 threads; more where long lines leave LDS for few work-groups per CU
static hipError_t launch_zgrow(const Batch& B, const PassTables& PT, hipStream_t s) {
  return z_pass(PT, [&](const TileTable& t, int n, int shape, int n3, size_t) {
    const size_t lds = lds_w(n3);
    if (shape == 1) k_zgrow<1024, CC / 2><<<n, 1024, lds_w(n3, CC / 2), s>>>(B, t);
    else if (n3 <= 64) k_zgrow<256><<<n, 256, lds, s>>>(B, t);
    else if (n3 <= 80) k_zgrow<512><<<n, 512, lds, s>>>(B, t);
    else k_zgrow<1024><<<n, 1024, lds, s>>>(B, t);
    return hipGetLastError();
  });
}
// The launch shape says which chunks of a line a wave adds to its ekin sum, so
// it follows the longest line of the whole batch (zb_n3, of the boxes in tiles
// of 16 columns): a part of a chunked batch that chose by its own lines summed
// 33 to 64 points in another order.  (Up to 32 points every shape has one chunk
// per wave.)
//
// Lines of at most 16 points keep one to four waves busy; the idle ones of a
// work-group of eight hold its CU's wave slots.  Two or four waves from two
// work-groups per CU on: free boxes of 44 x 44 x 2, 128 of them 217 -> 106 us,
// 20 x 20 x 1 x 256 90 -> 35 us, periodic 44 x 44 x 16 x 64 185 -> 140 us; a
// single box loads faster with eight (16^3: 10.5 against 11.7 us).
static hipError_t launch_zback(const Batch& B, const PassTables& PT, hipStream_t s) {
  const TileTable& ft = PT.t[P_CZ];
  double* part = PT.part[0];
  return z_pass(PT, [&](const TileTable& t, int n, int shape, int, size_t lds) {
    if (shape == 1) k_zback<1024, 2, 4, CC / 2><<<n, 1024, lds, s>>>(B, t, ft, part);
    else if (PT.zb_n3 <= 8 && n > 512) k_zback<128, 1, 4><<<n, 128, lds, s>>>(B, t, ft, part);
    else if (PT.zb_n3 <= 16 && n > 512) k_zback<256, 1, 4><<<n, 256, lds, s>>>(B, t, ft, part);
    else if (PT.zb_n3 <= 32) k_zback<512, 1, 4><<<n, 512, lds, s>>>(B, t, ft, part);
    else if (PT.zb_n3 <= 48) k_zback<768, 1, 6><<<n, 768, lds, s>>>(B, t, ft, part);
    else if (PT.zb_n3 <= 64) k_zback<512, 2, 4><<<n, 512, lds, s>>>(B, t, ft, part);
    else k_zback<1024, 3, 4><<<n, 1024, lds, s>>>(B, t, ft, part);
    return hipGetLastError();
  });
}
template <int PC>
static hipError_t launch_xykin(const Batch& B, const TileTable& t, const TileTable& ft,
                               int ntiles, size_t lds, int nt, int shape, const PcArgs& P,
                               hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  if (shape >= 2) k_xykin<S2_NT, 6, PC><<<ntiles, nt, lds, s>>>(B, t, ft, P);
  else k_xykin<S1_NT, 4, PC><<<ntiles, nt, lds, s>>>(B, t, ft, P);
  return hipGetLastError();
}
// the x-y kinetic pass: one launch per group of boxes, or one over all
template <int PC>
static hipError_t xykin_pass(const Batch& B, const PassTables& PT, const PcArgs& P,
                             hipStream_t s) {
  const TileTable& ft = PT.t[P_PF];
  if (PT.n_pfg == 0)
    return launch_xykin<PC>(B, ft, ft, PT.ntiles[P_PF], PT.lds_pfg[0], PT.nthr_pfg[0],
                            PT.shape_pfg[0], P, s);
  hipError_t e = hipSuccess;
  for (int k = 0; k < PT.n_pfg && e == hipSuccess; ++k)
    e = launch_xykin<PC>(B, PT.pfg[k], ft, PT.nt_pfg[k], PT.lds_pfg[k], PT.nthr_pfg[k],
                         PT.shape_pfg[k], P, s);
  return e;
}
static hipError_t launch_xypot(const Batch& B, const TileTable& t, const TileTable& ft,
                               int ntiles, size_t lds, int nt, int shape, double* part,
                               hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  if (shape >= 2) k_xypot<S2_NT, 2, 6><<<ntiles, nt, lds, s>>>(B, t, ft, part);
  else k_xypot<S1_NT, 3, 4><<<ntiles, nt, lds, s>>>(B, t, ft, part);
  return hipGetLastError();
}

// the x-y kinetic and potential passes of boxes whose planes do not fit
static hipError_t kin_lines_pass(const Batch& B, const PassTables& PT, hipStream_t s) {
  const size_t lx = lds_rows(2 * PT.maxN1), ly = lds_w(PT.maxN2);
  const int nx = PT.ntiles[P_XK], ny = PT.ntiles[P_YK];
  if (nx <= 0) return hipSuccess;
  if (PT.maxN1 <= 96) k_xlines_kin<768, 2, 6><<<nx, 768, lx, s>>>(B, PT.t[P_XK]);
  else k_xlines_kin<1024, 3, 4><<<nx, 1024, lx, s>>>(B, PT.t[P_XK]);
  if (PT.maxN2 <= 80) k_ylines_kin<768, 6><<<ny, 768, ly, s>>>(B, PT.t[P_YK]);
  else k_ylines_kin<1024, 4><<<ny, 1024, ly, s>>>(B, PT.t[P_YK]);
  return hipGetLastError();
}
static hipError_t pot_lines_pass(const Batch& B, const PassTables& PT, hipStream_t s) {
  const size_t lg = lds_rows(2 * PT.maxN1), ly = lds_rows(PT.maxL2), lx = lds_rows(PT.maxL1);
  const int nx = PT.ntiles[P_XR], ny = PT.ntiles[P_YL];
  if (nx <= 0) return hipSuccess;
  k_xlines_grow<1024, 8><<<nx, 1024, lg, s>>>(B, PT.t[P_XR]);
  if (PT.maxL2 <= 256) k_ylines_pot<1024, 2, 4><<<ny, 1024, ly, s>>>(B, PT.t[P_YL], PT.part[3]);
  else k_ylines_pot<1024, 3, 4><<<ny, 1024, ly, s>>>(B, PT.t[P_YL], PT.part[3]);
  if (PT.maxN1 <= 96) k_xlines_shrink<768, 2, 6><<<nx, 768, lx, s>>>(B, PT.t[P_XR]);
  else k_xlines_shrink<1024, 3, 4><<<nx, 1024, lx, s>>>(B, PT.t[P_XR]);
  return hipGetLastError();
}

// ev: null, or 2 S_COUNT events recorded before / after each stage
hipError_t launch_fp64_seq(const Batch& B, const PassTables& PT, hipStream_t s,
                           hipEvent_t* ev) {
  auto mark = [&](int stage, int end) {
    if (ev) (void)hipEventRecord(ev[2 * stage + end], s);
  };
  hipError_t e = hipSuccess;
  // k_zgrow and k_xykin share a launch, unless stages are timed: it saves a
  // launch and the first kernel's last, partly empty wave of work-groups, 6 to
  // 10 us for one orbital of 16^3 to 40^3 (60 of 66, 84 of 94 us), 15 to 25 us
  // for ten to sixty (32^3 x 60: 420 of 445 us; 40^3 x 40: 584 of 607).  From
  // FP64_JOIN work-groups on the gain is lost in the mix of two kinds of
  // work-group on a CU (32^3 x 300: 1.955 of 1.960 ms, 40^3 x 128: 1.760 of
  // 1.745).
  const int nz = PT.ntiles[P_CZ], nx = PT.ntiles[P_PF];
  if (!ev && !PT.kin_lines && PT.n_pfg == 0 && PT.shape_pfg[0] >= 2 && nz + nx <= FP64_JOIN &&
      PT.n_zg == 0 && PT.shape_zg[0] == 2) {
    const size_t lds = std::max(lds_w(PT.len_zg[0]), PT.lds_pfg[0]);
    const TileTable &tz = PT.t[P_CZ], &tx = PT.t[P_PF];
    if (nz + nx <= 0) return hipSuccess;
    if (PT.nthr_pfg[0] <= 256) k_zgrow_xykin<256><<<nz + nx, 256, lds, s>>>(B, tz, tx, nx);
    else if (PT.nthr_pfg[0] <= 512) k_zgrow_xykin<512><<<nz + nx, 512, lds, s>>>(B, tz, tx, nx);
    else k_zgrow_xykin<S2_NT><<<nz + nx, S2_NT, lds, s>>>(B, tz, tx, nx);
    e = hipGetLastError();
  } else {
    mark(S_ZG, 0);
    e = launch_zgrow(B, PT, s);
    mark(S_ZG, 1);
    // one launch per group of boxes, or one over all of them
    mark(S_KXY, 0);
    if (e == hipSuccess)
      e = PT.kin_lines ? kin_lines_pass(B, PT, s) : xykin_pass<0>(B, PT, PcArgs{}, s);
    mark(S_KXY, 1);
  }
  mark(S_XYP, 0);
  if (e == hipSuccess && PT.pot_lines) e = pot_lines_pass(B, PT, s);
  else if (e == hipSuccess && PT.n_pbg == 0)
    e = launch_xypot(B, PT.t[P_RP], PT.t[P_RP], PT.ntiles[P_RP], PT.lds_pbg[0],
                     PT.nthr_pbg[0], PT.shape_pbg[0], PT.part[3], s);
  for (int k = 0; k < PT.n_pbg && e == hipSuccess; ++k)
    e = launch_xypot(B, PT.pbg[k], PT.t[P_RP], PT.nt_pbg[k], PT.lds_pbg[k], PT.nthr_pbg[k],
                     PT.shape_pbg[k], PT.part[3], s);
  mark(S_XYP, 1);
  mark(S_ZB, 0);
  if (e == hipSuccess)
    e = launch_zback(B, PT, s);
  mark(S_ZB, 1);
  if (e != hipSuccess) return e;
  EnergyTables et;
  et.t[0] = PT.t[P_CZ];
  et.p[0] = PT.part[0];
  et.t[1] = PT.t[PT.pot_lines ? P_YL : P_RP];
  et.p[1] = PT.part[3];
  et.nk = 1;
  et.n = 2;
  mark(S_ENERGY, 0);
  launch_energy(et, B, s);
  mark(S_ENERGY, 1);
  if (ev)
    for (int st : {S_ZERO, S_UNC, S_XF, S_YF, S_KY, S_KZ, S_ZP, S_YB, S_XB, S_COMP, S_PF, S_PB}) {
      mark(st, 0);
      mark(st, 1);
    }
  return hipGetLastError();
}

static int den_threads(const PassTables& PT) {
  return PT.shape_pbg[0] >= 2 ? std::min(512, PT.nthr_pbg[0]) : PT.nthr_pbg[0];
}
// work-groups of k_xyden that 256 CUs hold at a time: 16 waves of 128 VGPRs and
// plane_lds bytes of LDS each
int fp64_den_resident(const PassTables& PT, size_t plane_lds) {
  const size_t lds = std::max(PT.lds_pbg[0], (size_t)1);
  return 256 * std::max(1, std::min(1024 / den_threads(PT), (int)(plane_lds / lds)));
}
hipError_t launch_fp64_density(const Batch& B, const PassTables& PT, const DenArgs& D, int L3,
                               hipStream_t s) {
  hipError_t e = launch_zgrow(B, PT, s);
  if (e != hipSuccess) return e;
  const int n = D.ngroups * L3, nt = den_threads(PT);
  const size_t lds = PT.lds_pbg[0];
  if (PT.shape_pbg[0] >= 2) k_xyden<512, 3, 4><<<n, nt, lds, s>>>(B, D);
  else k_xyden<S1_NT, 3, 4><<<n, nt, lds, s>>>(B, D);
  k_xyden_sum<<<dim3((unsigned)((D.nisf + 255) / 256), D.nspin), 256, 0, s>>>(D);
  return hipGetLastError();
}

template <int MODE>
static hipError_t launch_pcz(const Batch& B, const PassTables& PT, const PcArgs& P,
                             hipStream_t s) {
  return z_pass(PT, [&](const TileTable& t, int n, int shape, int n3, size_t) {
    if (shape == 1)
      k_pcz<MODE, 1024, 4, CC / 2><<<n, 1024, lds_w(n3, CC / 2), s>>>(B, t, P);
    else
      k_pcz<MODE, 512, 6><<<n, 512, lds_w(n3), s>>>(B, t, P);
    return hipGetLastError();
  });
}

// c W + K_z W + K_x W + K_y W of W = S v and the compressed sums that follow
// (mode 0: v = x, r = d = b - A x; 1: v = d; 2: x and d of the step first)
hipError_t launch_fp64_pc_apply(const Batch& B, const PassTables& PT, const PcArgs& P, int mode,
                                hipStream_t s) {
  const hipError_t e = mode == 0   ? launch_pcz<0>(B, PT, P, s)
                       : mode == 1 ? launch_pcz<1>(B, PT, P, s)
                                   : launch_pcz<2>(B, PT, P, s);
  if (e != hipSuccess) return e;
  return mode == 0 ? xykin_pass<1>(B, PT, P, s) : xykin_pass<2>(B, PT, P, s);
}

// raise the dynamic-LDS limit of the kernels to lds bytes
void fp64_attributes(size_t lds) {
  const void* k[] = {(const void*)k_zgrow<256>,      (const void*)k_zgrow<512>,
                     (const void*)k_zgrow<1024>,     (const void*)k_zgrow_xykin<256>,
                     (const void*)k_zgrow_xykin<512>, (const void*)k_zgrow_xykin<S2_NT>,
                     (const void*)k_xlines_grow<1024, 8>,
                     (const void*)k_ylines_pot<1024, 2, 4>,  (const void*)k_ylines_pot<1024, 3, 4>,
                     (const void*)k_xlines_shrink<768, 2, 6>,
                     (const void*)k_xlines_shrink<1024, 3, 4>,
                     (const void*)k_xlines_kin<768, 2, 6>, (const void*)k_xlines_kin<1024, 3, 4>,
                     (const void*)k_ylines_kin<768, 6>, (const void*)k_ylines_kin<1024, 4>, (const void*)k_zback<512, 1, 4>,
                     (const void*)k_zback<128, 1, 4>,   (const void*)k_zback<256, 1, 4>,
                     (const void*)k_zback<768, 1, 6>,   (const void*)k_zback<512, 2, 4>,
                     (const void*)k_zback<1024, 3, 4>,
                     (const void*)k_xyden<512, 3, 4>, (const void*)k_xyden<S1_NT, 3, 4>,
                     (const void*)k_xykin<S2_NT, 6, 0>, (const void*)k_xypot<S2_NT, 2, 6>,
                     (const void*)k_xykin<S2_NT, 6, 1>, (const void*)k_xykin<S2_NT, 6, 2>,
                     (const void*)k_xykin<S1_NT, 4, 1>, (const void*)k_xykin<S1_NT, 4, 2>,
                     (const void*)k_pcz<0, 512, 6>, (const void*)k_pcz<1, 512, 6>,
                     (const void*)k_pcz<2, 512, 6>, (const void*)k_pcz<0, 1024, 4, CC / 2>,
                     (const void*)k_pcz<1, 1024, 4, CC / 2>,
                     (const void*)k_pcz<2, 1024, 4, CC / 2>,
                     (const void*)k_zgrow<1024, CC / 2>, (const void*)k_zback<1024, 2, 4, CC / 2>,
                     (const void*)k_xykin<S1_NT, 4, 0>, (const void*)k_xypot<S1_NT, 3, 4>};
  for (const void* f : k)
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
        hipSuccess)
      (void)hipGetLastError();
}

}  // namespace bdft
