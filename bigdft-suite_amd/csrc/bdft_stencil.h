// Stencil pieces shared by the plane kernels (bdft_plane.hip) and the FP64
// kernels (bdft_fp64.hip): the taps of G, G^T and the wavelet-basis kinetic
// on register-held output chunks, the line maps of a plane in LDS, and the
// work-item counter of the in-plane passes.
#pragma once
#include "bdft_internal.h"

namespace bdft {

template <typename T>
struct PLine {
  const T* p;  // element 0 of the line
  int es;      // element stride
};

// Work item it = tid + k step (k = 0, 1, ...) of a loop over ch * n + j
// (0 <= j < n): one division per thread, then a carry per step.
struct ItDiv {
  int ch, j, dch, dj;
  __device__ __forceinline__ ItDiv(int tid, int n, int step) {
    ch = tid / n;
    j = tid - ch * n;
    dch = __builtin_amdgcn_readfirstlane(step / n);   // n, step: the same in all threads
    dj = step - dch * n;
  }
  __device__ __forceinline__ void next(int n) {
    ch += dch;
    j += dj;
    if (j >= n) {
      j -= n;
      ++ch;
    }
  }
};

// LDS row stride for rows of n values: odd (n + 1 or n + 2), so that the
// lanes of a wave that each walk their own row hit distinct banks
__host__ __device__ constexpr int odd_stride(int n) { return (n + 1) | 1; }

// G on a wavelet line [c(0..N-1); d(0..N-1)]: the taps of coarse input
// k = k0 + kk on the 8 fine outputs of a chunk (k0 = first coarse index)
template <typename T>
__device__ __forceinline__ void grow_tap(int kk, T c, T d, T o[8]) {
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int j = r + 16 - 2 * kk;
    if (j >= -14 && j <= 16) {
      o[r] = fma((T)Fil::F2S[j + 14], c, o[r]);
      o[r] = fma((T)Fil::F2W[j + 14], d, o[r]);
    }
  }
}

// first coarse index of the grow chunk starting at fine output p0
__device__ __forceinline__ int grow_k0(int p0, int per) {
  return per ? (p0 >> 1) - 8 : (p0 >> 1) - 15;
}

// wavelet-basis kinetic (unscaled): the taps of coarse input k = i0-14+kk
// (kk < 32) on the 4 coarse outputs i0..i0+3 (c and d)
template <typename T>
__device__ __forceinline__ void kin_tap(int kk, T c, T d, T oc[4], T od[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int l = kk - 14 - r;
    if (l >= -14 && l <= 14) {
      const int al = l < 0 ? -l : l;
      oc[r] = fma((T)Fil::KA[al], c, oc[r]);
      oc[r] = fma((T)Fil::KC[-l + 14], d, oc[r]);
      od[r] = fma((T)Fil::KC[l + 14], c, od[r]);
      od[r] = fma((T)Fil::KE[al], d, od[r]);
    }
  }
}

// Line map of one axis of a box's plane in LDS: entry k + MOFF, for coarse
// index k = -MOFF .. N + 17, holds the byte offsets from the line's element
// 0 of c(k) and d(k): k taken modulo N on a periodic line; on a free line a
// k outside 0..N-1 gives, for both, the offset of a slot that holds zero.
// The stencil chunks that reach past a line end read through it, one map
// entry per tap in place of wrap or bounds arithmetic.  Every tap of the
// grow (k0 >= -15, k0 + 18 <= N + 17 for L <= 2N + 29) and kinetic chunks
// (i0 - 14 >= -14, i0 + 17 <= N + 16) lies in that range.
constexpr int MOFF = 15;
__host__ __device__ constexpr int map_len(int N) { return N + MOFF + 18; }

// es: byte stride of the line's elements; zero: element index of the zero slot
__device__ __forceinline__ void build_map(int2* m, int N, int per, int es, int zero, int tid,
                                          int nt) {
  for (int e = tid; e < map_len(N); e += nt) {
    const int k = e - MOFF;
    int c, d;
    if (per) {
      int kw = k;
      while (kw < 0) kw += N;
      while (kw >= N) kw -= N;
      c = kw;
      d = N + kw;
    } else if ((unsigned)k < (unsigned)N) {
      c = k;
      d = N + k;
    } else {
      c = d = zero;
    }
    m[e] = make_int2(c * es, d * es);
  }
}

// G on a wavelet line: 8 fine outputs from k = k0 .. k0+18, read directly
// where the chunk lies inside the line, else through the line map m
template <typename T>
__device__ __forceinline__ void grow8_any(PLine<T> ln, const int2* m, int N, int k0, T o[8]) {
#pragma unroll
  for (int r = 0; r < 8; ++r) o[r] = (T)0;
  if (k0 >= 0 && k0 + 18 < N) {
#pragma unroll
    for (int kk = 0; kk < 19; ++kk)
      grow_tap(kk, ln.p[(k0 + kk) * ln.es], ln.p[(N + k0 + kk) * ln.es], o);
  } else {
    const int2* mm = m + (k0 + MOFF);
    const char* p = (const char*)ln.p;
#pragma unroll
    for (int kk = 0; kk < 19; ++kk) {
      const int2 e = mm[kk];
      grow_tap(kk, *(const T*)(p + e.x), *(const T*)(p + e.y), o);
    }
  }
}

// wavelet-basis kinetic (unscaled) on a wavelet line: 4 coarse outputs
// i0..i0+3 (c and d) from k = i0-14 .. i0+17, direct or through the map
template <typename T>
__device__ __forceinline__ void kin4_any(PLine<T> ln, const int2* m, int N, int i0, T oc[4],
                                         T od[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    oc[r] = (T)0;
    od[r] = (T)0;
  }
  if (i0 - 14 >= 0 && i0 + 17 < N) {
#pragma unroll
    for (int kk = 0; kk < 32; ++kk) {
      const int k = i0 - 14 + kk;
      kin_tap(kk, ln.p[k * ln.es], ln.p[(N + k) * ln.es], oc, od);
    }
  } else {
    const int2* mm = m + (i0 - 14 + MOFF);
    const char* p = (const char*)ln.p;
#pragma unroll
    for (int kk = 0; kk < 32; ++kk) {
      const int2 e = mm[kk];
      kin_tap(kk, *(const T*)(p + e.x), *(const T*)(p + e.y), oc, od);
    }
  }
}

// G^T on a real line of L points (periodic: fine index p, L = 2N; free: fine
// index p-14): the taps of fine input I = 2i0-14+qq (qq < 2 NO + 29) on the
// NO coarse outputs i0..i0+NO-1 (c and d)
template <typename T, int NO>
__device__ __forceinline__ void shrink_tap(int qq, T x, T oc[NO], T od[NO]) {
#pragma unroll
  for (int r = 0; r < NO; ++r) {
    const int j = qq - 2 * r - 14;
    if (j >= -14 && j <= 16) {
      oc[r] = fma((T)Fil::F2S[j + 14], x, oc[r]);
      od[r] = fma((T)Fil::F2W[j + 14], x, od[r]);
    }
  }
}

// Fine-line map of a periodic line for the backward pass: entry e = 2 i0 + qq
// of a shrink chunk holds the byte offset of its input, fine index e - 14
// modulo L.  Every chunk's entries lie below 2 N + 2 NO + 27 <= fmap_len(N).
__host__ __device__ constexpr int fmap_len(int N) { return 2 * N + 40; }
__device__ __forceinline__ void build_fmap(int* m, int N, int L, int es, int tid, int nt) {
  for (int e = tid; e < fmap_len(N); e += nt) {
    int p = (e - 14) % L;
    p += p < 0 ? L : 0;
    m[e] = p * es;
  }
}

// G^T on a fine line stored as an LDS row: NO coarse outputs, read directly
// where the chunk's inputs lie inside the line; else, periodic, through the
// map m, free (only the line's last chunk), with fine points past L as zero
template <typename T, int NO = 4>
__device__ __forceinline__ void shrink4_any(const T* ln, const int* m, int L, int i0, int per,
                                            T oc[NO], T od[NO]) {
#pragma unroll
  for (int r = 0; r < NO; ++r) {
    oc[r] = (T)0;
    od[r] = (T)0;
  }
  const bool in = per ? (2 * i0 - 14 >= 0 && 2 * i0 + 2 * NO + 14 < L)
                      : (2 * i0 + 2 * NO + 28 < L);
  if (in) {
    const T* q = ln + 2 * i0 - (per ? 14 : 0);
#pragma unroll
    for (int qq = 0; qq < 2 * NO + 29; ++qq) shrink_tap<T, NO>(qq, q[qq], oc, od);
  } else if (per) {
    const int* mm = m + 2 * i0;
    const char* p = (const char*)ln;
#pragma unroll
    for (int qq = 0; qq < 2 * NO + 29; ++qq)
      shrink_tap<T, NO>(qq, *(const T*)(p + mm[qq]), oc, od);
  } else {
#pragma unroll
    for (int qq = 0; qq < 2 * NO + 29; ++qq) {
      const int p = 2 * i0 + qq;
      const bool v = p < L;
      const T x = ln[v ? p : 0];
      shrink_tap<T, NO>(qq, v ? x : (T)0, oc, od);
    }
  }
}

// Sum of one double per thread over a work-group of blockDim.x / 64 waves
// (red: one entry per wave), in thread 0.  Starts with a barrier.
__device__ __forceinline__ double block_sum_rt(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)blockDim.x >> 6; ++i) s += red[i];
  return s;
}

}  // namespace bdft
