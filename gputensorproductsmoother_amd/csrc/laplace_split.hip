// laplace_split.hip - the 3D constant-coefficient operator in two launches:
// per z-plane a = M_y M_x u and c = (K_y M_x + M_y K_x) u, then per (x, y)
// column y = scale (K_z a + M_z c).
//
// The z-marching kernel (laplace.hip) moves fewer bytes but keeps windows of
// 2k+1 planes of 1 to 5 columns per thread in registers: from k = 4 on two or
// three wavefronts a SIMD stay resident and it waits.  Here every thread owns
// one cell's line, 6 vectors cross the memory instead of 2 (residual 3), much
// of it within the 256 MB last-level cache.
#include "gtps_internal.h"

#include <type_traits>

namespace gtps
{
  namespace
  {
    constexpr int ZNT = 256;

    template <int K, typename T>
    struct XY
    {
      static constexpr int CY   = 2;             // cells along y per work-group
      static constexpr int ROWS = K * (CY + 1) + 1;
      // 768: one pass of the lines along x at k = 7 (704); FP32 and k = 5 do
      // better with more work-groups a CU (Q7 32^3 FP64 160 us with 768, 179
      // with 512; FP32 91 and 89)
      static constexpr int NT   = sizeof(T) == 8 && K >= 6 ? 768 : 512;
      static size_t lds(int n) { return (size_t)2 * ROWS * ((K * n + 1) | 1) * sizeof(T); }
    };

    // a = M_y M_x u, c = (K_y M_x + M_y K_x) u on the rows 0 < y < N1 - 1 of
    // plane blockIdx.y; work-group = CY cells along y, whole rows in LDS.
    // n lanes of one wavefront share a row (n <= 64), so the row's products
    // along x replace it without a barrier.
    template <int K, typename T>
    __global__ void __launch_bounds__((XY<K, T>::NT))
    laplace_xy_kernel(const T *__restrict__ x, T *__restrict__ a, T *__restrict__ c,
                      const T *__restrict__ tab, const int n, const int log_n)
    {
      using C         = XY<K, T>;
      using TB        = Tab<K>;
      constexpr int W = 2 * K + 1, NT = C::NT, CY = C::CY;
      static_assert(CY == 2, "the products along y pick one of two cells");
      extern __shared__ double smem_raw[];
      T              *sm  = reinterpret_cast<T *>(smem_raw);
      const int       N1  = K * n + 1, RS = N1 | 1;
      const int       tid = threadIdx.x;
      const long long P   = (long long)N1 * N1;
      const int       cy0 = blockIdx.x * CY;
      // row r of the window is y = K (cy0 - 1) + r
      const int       y0  = K * (cy0 - 1);
      const int       r0 = cy0 == 0 ? K : 0;
      const int       r1 = K * ((cy0 + CY < n ? cy0 + CY : n) - cy0 + 1);
      T              *sM = sm, *sK = sm + C::ROWS * RS;
      const T        *xp = x + blockIdx.y * P + (long long)y0 * N1;
      for (int r = r0 + (tid >> 6); r <= r1; r += NT / 64)
        for (int i = tid & 63; i < N1; i += 64)
          sM[r * RS + i] = xp[(long long)r * N1 + i];
      __syncthreads();
      // products along x: lane (row, cell), K outputs, the vertex row with
      // the left cell's nodes
      const T *bM = tab + TB::bandM, *bK = tab + TB::bandK;
      for (int t = tid; t < ((r1 - r0 + 1) << log_n); t += NT)
        {
          const int r = r0 + (t >> log_n), cx = t & (n - 1);
          T        *d = sM + r * RS + K * cx, *e = sK + r * RS + K * cx;
          T         v[W], m[K], k[K];
#pragma unroll
          for (int i = 0; i < K; ++i)
            v[i] = cx > 0 ? d[i - K] : T(0);
#pragma unroll
          for (int i = K; i < W; ++i)
            v[i] = d[i - K];
#pragma unroll
          for (int q = 0; q < K; ++q)
            {
              const ConstP<T> M = here(bM + q * W), L = here(bK + q * W);
              T               sm_ = 0, sk = 0;
#pragma unroll
              for (int o = band_lo<K>(q); o <= band_hi<K>(q); ++o)
                {
                  sm_ += M[o + K] * v[K + q + o];
                  sk += L[o + K] * v[K + q + o];
                }
              m[q] = sm_;
              k[q] = sk;
            }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
          for (int q = 0; q < K; ++q)
            {
              d[q] = m[q];
              e[q] = k[q];
            }
        }
      __syncthreads();
      // products along y: lane (cell, x) - interior columns
      const long long o0 = blockIdx.y * P + (long long)K * cy0 * N1;
      for (int t = tid; t < CY * N1; t += NT)
        {
          const int cl = t >= N1 ? 1 : 0, xx = t - (cl ? N1 : 0);
          if (xx == 0 || xx == N1 - 1 || cy0 + cl >= n)
            continue;
          const T *m0 = sM + K * (cl + 1) * RS + xx, *k0 = sK + K * (cl + 1) * RS + xx;
          const bool low = cy0 + cl > 0;  // y = 0 is a Dirichlet row
          T          m[W], k[W];
#pragma unroll
          for (int i = 0; i < K; ++i)
            {
              m[i] = low ? m0[(i - K) * RS] : T(0);
              k[i] = low ? k0[(i - K) * RS] : T(0);
            }
#pragma unroll
          for (int i = K; i < W; ++i)
            {
              m[i] = m0[(i - K) * RS];
              k[i] = k0[(i - K) * RS];
            }
#pragma unroll
          for (int q = 0; q < K; ++q)
            {
              const ConstP<T> M = here(bM + q * W), L = here(bK + q * W);
              T               sa = 0, sc = 0;
#pragma unroll
              for (int o = band_lo<K>(q); o <= band_hi<K>(q); ++o)
                {
                  sa += M[o + K] * m[K + q + o];
                  sc += L[o + K] * m[K + q + o];
                  sc += M[o + K] * k[K + q + o];
                }
              if (q > 0 || low)
                {
                  const long long g = o0 + (long long)(K * cl + q) * N1 + xx;
                  a[g]              = sa;
                  c[g]              = sc;
                }
            }
        }
    }

    // y = scale (K_z a + M_z c) (RESID: b - that), Dirichlet rows copied;
    // thread = column, blockIdx.y = chunk of cz cells
    template <int K, typename T, bool RESID, bool DOT>
    __global__ void __launch_bounds__(ZNT)
    laplace_z_kernel(const T *__restrict__ a, const T *__restrict__ c, const T *x, const T *b,
                     T *y, const T *__restrict__ tab, const int n, const int cz,
                     const T scale, double *__restrict__ partial)
    {
      using TB        = Tab<K>;
      constexpr int W = 2 * K + 1;
      __shared__ double sred[ZNT / 64];
      const int       N1 = K * n + 1;
      const long long P  = (long long)N1 * N1;
      const int       col = blockIdx.x * ZNT + threadIdx.x;
      const int       c0 = blockIdx.y * cz, c1 = c0 + cz < n ? c0 + cz : n;
      const T *bM = tab + TB::bandM, *bK = tab + TB::bandK;
      double   dot = 0.0;
      if (col < N1 * N1)
        {
          const int  yy = col / N1, xx = col - yy * N1;
          const bool rim = xx == 0 || yy == 0 || xx == N1 - 1 || yy == N1 - 1;
          auto       copy = [&](int z) {
            const long long g = col + z * P;
            const T         xv = x[g], yv = RESID ? b[g] - xv : xv;
            y[g]               = yv;
            if (DOT)
              dot += (double)xv * (double)yv;
          };
          if (rim)
            {
              for (int z = K * c0; z < K * c1; ++z)
                copy(z);
              if (c1 == n)
                copy(N1 - 1);
            }
          else
            {
              if (c0 == 0)
                copy(0);
              if (c1 == n)
                copy(N1 - 1);
              // planes K (cl - 1) .. K (cl + 1)
              T va[W], vc[W];
#pragma unroll
              for (int i = 0; i <= K; ++i)
                {
                  const int z = K * (c0 - 1) + i;
                  va[K + i]   = z >= 0 ? a[col + z * P] : T(0);
                  vc[K + i]   = z >= 0 ? c[col + z * P] : T(0);
                }
              for (int cl = c0; cl < c1; ++cl)
                {
#pragma unroll
                  for (int i = 0; i <= K; ++i)
                    {
                      va[i] = va[K + i];
                      vc[i] = vc[K + i];
                    }
#pragma unroll
                  for (int i = 1; i <= K; ++i)
                    {
                      const long long g = col + (long long)(K * cl + i) * P;
                      va[K + i]         = a[g];
                      vc[K + i]         = c[g];
                    }
#pragma unroll
                  for (int q = 0; q < K; ++q)
                    {
                      const ConstP<T> M = here(bM + q * W), L = here(bK + q * W);
                      T               s = 0;
#pragma unroll
                      for (int o = band_lo<K>(q); o <= band_hi<K>(q); ++o)
                        {
                          s += L[o + K] * va[K + q + o];
                          s += M[o + K] * vc[K + q + o];
                        }
                      s *= scale;
                      if (q > 0 || cl > 0)
                        {
                          const long long g = col + (long long)(K * cl + q) * P;
                          const T         yv = RESID ? b[g] - s : s;
                          if (DOT)
                            dot += (double)x[g] * (double)yv;
                          y[g] = yv;
                        }
                    }
                }
            }
        }
      if (DOT)
        {
          const double s = block_sum<ZNT>(dot, sred);
          if (threadIdx.x == 0)
            partial[blockIdx.x + gridDim.x * blockIdx.y] = s;
        }
    }

    template <int K, typename T>
    int
    split_k(const gtps_level *lvl, T *y, const T *x, const T *b, bool dot)
    {
      using C             = XY<K, T>;
      const int   n       = lvl->n, N1 = lvl->N1;
      const T    *tab     = (const T *)lvl->dtab();
      T          *a       = (T *)lvl->split, *c = a + lvl->N;
      hipStream_t s       = lvl->ctx->stream;
      const size_t lds    = C::lds(n);
      int          log_n  = 0;
      while ((1 << log_n) < n)
        ++log_n;
      auto xy = laplace_xy_kernel<K, T>;
      if (lds > 65536)
        GTPS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(xy),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      // the planes z = 0 and N1 - 1 too: their values enter interior rows
      hipLaunchKernelGGL(xy, dim3((n + C::CY - 1) / C::CY, N1), dim3(C::NT), lds, s, x, a, c,
                         tab, n, log_n);
      const int  cz = 4;  // 8: too few wavefronts (Q7 32^3 FP64 191 instead of 179 us)
      const dim3 grid((N1 * N1 + ZNT - 1) / ZNT, (n + cz - 1) / cz);
      const int  nb = (int)(grid.x * grid.y);
      if (dot)
        GTPS_REQUIRE(nb <= lvl->ctx->ws.capacity, "too many blocks for partials");
      double *pt = lvl->ctx->ws.partials;
      const T sc = (T)lvl->scale;
#define GTPS_Z(R, D)                                                                  \
  hipLaunchKernelGGL((laplace_z_kernel<K, T, R, D>), grid, dim3(ZNT), 0, s, a, c, x, b, y, \
                     tab, n, cz, sc, pt)
      if (b && dot)
        GTPS_Z(true, true);
      else if (b)
        GTPS_Z(true, false);
      else if (dot)
        GTPS_Z(false, true);
      else
        GTPS_Z(false, false);
#undef GTPS_Z
      GTPS_LAUNCH_CHECK();
      return nb;
    }

    template <typename F>
    auto
    split_dispatch(int k, F f)
    {
      switch (k)
        {
          case 5: return f(std::integral_constant<int, 5>{});
          case 6: return f(std::integral_constant<int, 6>{});
          default: return f(std::integral_constant<int, 7>{});
        }
    }
  } // namespace

  // Measured on MI355X, us, two launches / z-marching (vmult, residual): Q5
  // 32^3 FP32 40 / 40, 46 / 81, FP64 57 / 93, 65 / 108; Q6 32^3 65 / 67, 72 /
  // 84, 90 / 148, 115 / 189; Q7 32^3 90 / 104, 100 / 204, 160 / 204, 190 /
  // 252; Q5 64^3 FP32 280 / 364, 309 / 749.  Not: k <= 4 (Q4 32^3 FP32 36 /
  // 20), 16^3 (Q7 FP32 29 / 25), larger rows in LDS (Q5 64^3 FP64 626 / 540,
  // Q6 64^3 FP32 581 / 490).
  bool
  laplace_split_fits(int dim, int k, int n, int prec)
  {
    if (dim != 3 || k < 5 || n < 32 || n > 64)
      return false;
    const size_t lds = split_dispatch(k, [&](auto kk) {
      constexpr int K = decltype(kk)::value;
      return prec == GTPS_FP32 ? XY<K, float>::lds(n) : XY<K, double>::lds(n);
    });
    return lds <= (n == 32 ? 80 : 48) * 1024;
  }

  int
  launch_laplace_split(const gtps_level *lvl, void *y, const void *x, const void *b, bool dot)
  {
    return split_dispatch(lvl->k, [&](auto kk) {
      constexpr int K = decltype(kk)::value;
      return lvl->prec == GTPS_FP32
               ? split_k<K>(lvl, (float *)y, (const float *)x, (const float *)b, dot)
               : split_k<K>(lvl, (double *)y, (const double *)x, (const double *)b, dot);
    });
  }
} // namespace gtps
