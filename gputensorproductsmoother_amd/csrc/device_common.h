// device_common.h - shared device-side definitions for the gfx950 kernels.
//
// Table layout: every degree K owns one packed array of 1D data per
// precision (built once per context by setup.hip), passed to kernels as a
// `const T* __restrict__` so that uniform, compile-time-indexed reads become
// scalar loads.  Offsets are compile-time functions of K.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace gtps
{
  constexpr int MAX_DEGREE = 7;
  constexpr int MAX_QUAD   = 16;  // quadrature points per direction (error norms)
  constexpr int MAX_DENSE_COARSE = 4096;  // interior DoFs of a tabulated level-2 V-cycle

  template <int K>
  struct Tab
  {
    static constexpr int N  = K + 1;      // cell DoFs per direction
    static constexpr int NP = 2 * K + 1;  // patch box per direction
    static constexpr int NI = 2 * K - 1;  // patch interior per direction
    static constexpr int W  = 2 * K + 1;  // width of a global 1D matrix row
    // reference-cell mass and stiffness [N*N]
    static constexpr int cellM = 0;
    static constexpr int cellK = cellM + N * N;
    // 2-cell patch mass and stiffness [NP*NP]
    static constexpr int patchM = cellK + N * N;
    static constexpr int patchK = patchM + NP * NP;
    // M-orthonormal interior eigenvectors S[i*NI+j] (vector j) and values
    static constexpr int S   = patchK + NP * NP;
    static constexpr int lam = S + NI * NI;
    // embedding (prolongation) matrix E[q*N+a], q in [0,2K], a in [0,K]
    static constexpr int E = lam + NI;
    // rows of the assembled global 1D matrices, by node position p in its
    // cell (p = 0: vertex row), band[p*W + off + K] for off in [-K, K]
    static constexpr int bandM = E + NP * N;
    static constexpr int bandK = bandM + K * W;
    // 1 / (l_i + l_j + l_k), [k][j][i], and 1 / (l_i + l_j), [j][i]
    static constexpr int lamInv3 = bandK + K * W;
    static constexpr int lamInv2 = lamInv3 + NI * NI * NI;
    // Even/odd split of the eigenbasis.  The interior pencil is invariant
    // under the reflection i -> NI-1-i, so every eigenvector is even or odd.
    // With MH = K-1 the middle index, the K even vectors are stored by their
    // rows 0..MH (SE[i*K+e]) and the K-1 odd ones by rows 0..MH-1
    // (SO[i*(K-1)+o]); eigen coordinates are renumbered even first, then
    // odd, and lamInv3p holds 1/(l_a+l_b+l_c) in that numbering [c][b][a].
    static constexpr int MH      = K - 1;
    static constexpr int NE = K, NO = K - 1;
    static constexpr int SE      = lamInv2 + NI * NI;
    static constexpr int SO      = SE + (MH + 1) * NE;
    static constexpr int lamInv3p = SO + (MH > 0 ? MH * NO : 0);
    // Face form of the patch solve (even/odd numbering).  IE/IO hold S^T M
    // of the interior (the map nodal -> eigen coordinates, S^{-1}) by folded
    // node rows like SE/SO; mv = S^T M e_0 couples the left end node (the
    // right end has the same entry for an even vector, the opposite one for
    // an odd vector) and at = S^T K e_0 - lambda mv its stiffness once the
    // end's basis function is made M-orthogonal to the interior.
    // (lamInv3p, mv and at are contiguous: one block of per-lane operands.)
    static constexpr int mv   = lamInv3p + NI * NI * NI;
    static constexpr int at   = mv + NI;
    static constexpr int IE   = at + NI;
    static constexpr int IO   = IE + (MH + 1) * NE;
    // 1/(l_a+l_b) in the even/odd numbering, [b][a]
    static constexpr int lamInv2p = IO + (MH > 0 ? MH * NO : 0);
    static constexpr int size     = lamInv2p + NI * NI;
  };

  // packed DG table offsets (NN = k+1, PD = 2 NN)
  template <int K>
  struct DTab
  {
    static constexpr int NN = K + 1, PD = 2 * NN;
    static constexpr int M  = 0;              // cell mass [NN][NN]
    static constexpr int Lm = M + NN * NN;    // block (c, c-1)
    static constexpr int Lp = Lm + NN * NN;   // block (c, c+1)
    static constexpr int Lc = Lp + NN * NN;   // 3 diagonal blocks:
                                              // interior, first, last cell
    static constexpr int S   = Lc + 3 * NN * NN;  // 4 patch variants [PD][PD]
    static constexpr int lam = S + 4 * PD * PD;   // 4 x [PD]
    static constexpr int E   = lam + 4 * PD;      // child embedding [2][NN][NN]
    // Off-diagonal blocks in face form: the left neighbour cell w couples to
    // the patch as e_0 (AR.w) - d0 w(1) / 2 (d0: derivatives of the first
    // cell's basis at its left end), the right one as e_last (AL.w) + d1 w(0)
    // / 2.  MS = M S per variant [node][i] (S^T M: nodal -> eigen), EL and ER
    // the S^T of d0 and d1 on the first and last cell per variant.
    static constexpr int MS   = E + 2 * NN * NN;
    static constexpr int EL   = MS + 4 * PD * PD;
    static constexpr int ER   = EL + 4 * PD;
    static constexpr int AR   = ER + 4 * PD;
    static constexpr int AL   = AR + NN;
    static constexpr int size = AL + NN;
  };

  // Column range of row r of a 2-cell patch matrix (block sparsity: rows
  // inside cell 0 couple to nodes 0..K, rows inside cell 1 to K..2K, the
  // shared vertex row to all).
  template <int K>
  __host__ __device__ constexpr int
  prow_lo(int r)
  {
    return r <= K ? 0 : K;
  }
  template <int K>
  __host__ __device__ constexpr int
  prow_hi(int r)
  {
    return r < K ? K : 2 * K;
  }
  // Column offsets of a global 1D row for node position p within its cell.
  template <int K>
  __host__ __device__ constexpr int
  band_lo(int p)
  {
    return p == 0 ? -K : -p;
  }
  template <int K>
  __host__ __device__ constexpr int
  band_hi(int p)
  {
    return p == 0 ? K : K - p;
  }

  template <typename T>
  __device__ __forceinline__ T
  wave_sum(T v)
  {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      v += __shfl_xor(v, off, 64);
    return v;
  }

  // Sum over the block; result valid in thread 0.  `red` holds >= NT/64
  // doubles of LDS.
  template <int NT>
  __device__ __forceinline__ double
  block_sum(double v, double *red)
  {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
      red[wid] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
      {
#pragma unroll
        for (int w = 0; w < NT / 64; ++w)
          s += red[w];
      }
    return s;
  }

  // division by an invariant divisor d >= 1 for 0 <= n < 2^31:
  // n / d = (umulhi(n, m) + n) >> s with s = ceil(log2 d),
  // m = floor(2^32 (2^s - d) / d) + 1 (set up on the host by make_fastdiv)
  struct FastDiv
  {
    unsigned d, m;
    int      s;
  };
  inline FastDiv
  make_fastdiv(unsigned d)
  {
    int s = 0;
    while ((1ull << s) < d)
      ++s;
    const unsigned long long m = ((1ull << 32) * ((1ull << s) - d)) / d + 1;
    return FastDiv{d, (unsigned)m, s};
  }
  __device__ __forceinline__ unsigned
  fastdiv(unsigned n, const FastDiv &f)
  {
    return (__umulhi(n, f.m) + n) >> f.s;
  }

  // Fast-diagonalisation transforms in the even/odd eigenbasis (tables
  // Tab::SE, Tab::SO): t = S^T v with t numbered even vectors first, and
  // its inverse v = S t.  The reflection symmetry of the eigenvectors
  // halves the products: K(K) + (K-1)^2 multiply-adds and 2(K-1)
  // additions instead of (2K-1)^2.
  template <int K, typename T>
  __device__ __forceinline__ void
  fd_fwd(const T *SE, const T *SO, const T (&v)[2 * K - 1], T (&t)[2 * K - 1])
  {
    constexpr int NI = 2 * K - 1, MH = K - 1, NE = K, NO = K - 1;
    T e[MH + 1], o[MH > 0 ? MH : 1];
#pragma unroll
    for (int i = 0; i < MH; ++i)
      {
        e[i] = v[i] + v[NI - 1 - i];
        o[i] = v[i] - v[NI - 1 - i];
      }
    e[MH] = v[MH];
#pragma unroll
    for (int q = 0; q < NE; ++q)
      {
        T s = 0;
#pragma unroll
        for (int i = 0; i <= MH; ++i)
          s += SE[i * NE + q] * e[i];
        t[q] = s;
      }
#pragma unroll
    for (int q = 0; q < NO; ++q)
      {
        T s = 0;
#pragma unroll
        for (int i = 0; i < MH; ++i)
          s += SO[i * NO + q] * o[i];
        t[NE + q] = s;
      }
  }

  template <int K, typename T>
  __device__ __forceinline__ void
  fd_inv(const T *SE, const T *SO, const T (&t)[2 * K - 1], T (&v)[2 * K - 1])
  {
    constexpr int NI = 2 * K - 1, MH = K - 1, NE = K, NO = K - 1;
#pragma unroll
    for (int i = 0; i < MH; ++i)
      {
        T pe = 0, po = 0;
#pragma unroll
        for (int q = 0; q < NE; ++q)
          pe += SE[i * NE + q] * t[q];
#pragma unroll
        for (int q = 0; q < NO; ++q)
          po += SO[i * NO + q] * t[NE + q];
        v[i]          = pe + po;
        v[NI - 1 - i] = pe - po;
      }
    T pm = 0;
#pragma unroll
    for (int q = 0; q < NE; ++q)
      pm += SE[MH * NE + q] * t[q];
    v[MH] = pm;
  }

  // table address hidden from the optimiser: the entries are loaded (scalar)
  // for this use instead of being kept live and spilled
  template <typename T>
  using ConstP = const T __attribute__((address_space(4))) *;
  template <typename T>
  __device__ __forceinline__ ConstP<T>
  here(const T *p)
  {
    ConstP<T> c = (ConstP<T>)p;
    asm volatile("" : "+s"(c));
    return c;
  }

  __device__ __forceinline__ int
  linear_block_id()
  {
    return blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  }

  // MI355X dispatches consecutive work-group ids round-robin over its 8
  // XCDs, each with a private L2.  This bijection maps the hardware id to a
  // logical id such that every XCD works through one contiguous range of
  // logical ids, so neighbouring tiles (which share halo / face data) run
  // on the same XCD and hit the same L2.
  constexpr int N_XCD = 8;
  __host__ __device__ __forceinline__ int
  xcd_logical_id(int hw, int n)
  {
    // unsigned: the divisions by 8 are shifts and masks
    const unsigned un = (unsigned)n, uh = (unsigned)hw;
    const unsigned q = un / N_XCD, r = un % N_XCD;
    const unsigned xcd = uh % N_XCD, slot = uh / N_XCD;
    return (int)((xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot);
  }
} // namespace gtps
