// smoother_add2d.hip - additive vertex-patch smoothing in 2D, residual and
// every patch in one launch:  c = w sum_P R_P^T A_P^{-1} R_P (b - A u).
//
// A work-group owns TC x TC cells and solves the (TC + 1)^2 patches that touch
// their nodes from u and b on one more cell all round (the residual on a
// patch's interior needs the patch's own cells only), then every node sums
// its one, two or four patches in a fixed order.  A sweep was a residual and
// four colour launches, each a few us of latency on these small levels (Q2
// 128^2 FP64: 7 + 4 x 3 us, and 5 us from zero now).
#include "gtps_internal.h"

namespace gtps
{
  namespace
  {
    constexpr int A2NT = 256;

    template <int K>
    struct A2
    {
      static constexpr int TC = K == 1 ? 8 : (K <= 3 ? 4 : 2);
      static constexpr int NI = 2 * K - 1;
      static constexpr int WR = K * (TC + 2) + 1, RS = WR | 1;  // window
      static constexpr int NP = TC + 1, PS = NI * NI;           // patches
      static constexpr int R  = 0;                              // residual
      static constexpr int U  = WR * RS;  // u, then M_y u; the patches later
      static constexpr int V  = U + WR * RS;                    // K_y u
      static constexpr int size = V + WR * RS > U + NP * NP * PS ? V + WR * RS
                                                                 : U + NP * NP * PS;
    };

    // ZERO: u = 0 (not read), out = c everywhere.  Otherwise out = c, zero on
    // the Dirichlet nodes.
    template <int K, typename T, bool ZERO>
    __global__ void __launch_bounds__(A2NT)
    additive2d_kernel(const T *__restrict__ u, const T *__restrict__ b, T *__restrict__ out,
                      const T *__restrict__ tab, const int n, const T relax)
    {
      using C          = A2<K>;
      using TB         = Tab<K>;
      constexpr int NI = C::NI, WR = C::WR, RS = C::RS, TC = C::TC, NP = C::NP, W = 2 * K + 1;
      __shared__ T  sm[C::size];
      const int     N1 = K * n + 1, tid = threadIdx.x;
      const int     nt = (n + TC - 1) / TC;
      const int     bx = blockIdx.x % nt, by = blockIdx.x / nt;
      // window origin: node K (first owned cell - 1)
      const int x0 = K * (bx * TC - 1), y0 = K * (by * TC - 1);
      T        *R = sm + C::R, *U = sm + C::U, *V = sm + C::V;
      for (int t = tid; t < WR * WR; t += A2NT)
        {
          const int  j = t / WR, i = t - j * WR, x = x0 + i, y = y0 + j;
          const bool in = x >= 0 && y >= 0 && x < N1 && y < N1;
          const long long g = x + (long long)y * N1;
          R[j * RS + i] = in ? b[g] : T(0);
          if (!ZERO)
            U[j * RS + i] = in ? u[g] : T(0);
        }
      __syncthreads();
      if (!ZERO)
        {
          // one cell's K rows (columns) per task, the vertex one with the
          // cell before; band rows as in the operator
          const T *bM = tab + TB::bandM, *bK = tab + TB::bandK;
          constexpr int L = WR * (TC + 2);
          constexpr int PP = (L + A2NT - 1) / A2NT;
          T             m[PP][K], k[PP][K];
#pragma unroll
          for (int pp = 0; pp < PP; ++pp)
            {
              const int t = tid + A2NT * pp, c = t / WR, i = t - c * WR;
              if (t < L)
                {
                  T v[W];
#pragma unroll
                  for (int a = 0; a < W; ++a)
                    v[a] = c > 0 || a >= K ? U[(K * (c - 1) + a) * RS + i] : T(0);
#pragma unroll
                  for (int q = 0; q < K; ++q)
                    {
                      T s0 = 0, s1 = 0;
#pragma unroll
                      for (int o = band_lo<K>(q); o <= band_hi<K>(q); ++o)
                        {
                          s0 += bM[q * W + o + K] * v[K + q + o];
                          s1 += bK[q * W + o + K] * v[K + q + o];
                        }
                      m[pp][q] = s0;
                      k[pp][q] = s1;
                    }
                }
            }
          __syncthreads();
#pragma unroll
          for (int pp = 0; pp < PP; ++pp)
            {
              const int t = tid + A2NT * pp, c = t / WR, i = t - c * WR;
              if (t < L)
                {
#pragma unroll
                  for (int q = 0; q < K; ++q)
                    {
                      U[(K * c + q) * RS + i] = m[pp][q];
                      V[(K * c + q) * RS + i] = k[pp][q];
                    }
                }
            }
          __syncthreads();
          for (int t = tid; t < L; t += A2NT)
            {
              const int c = t / WR, j = t - c * WR;
              T         v[W], w[W];
#pragma unroll
              for (int a = 0; a < W; ++a)
                {
                  v[a] = c > 0 || a >= K ? U[j * RS + K * (c - 1) + a] : T(0);
                  w[a] = c > 0 || a >= K ? V[j * RS + K * (c - 1) + a] : T(0);
                }
#pragma unroll
              for (int q = 0; q < K; ++q)
                {
                  T s = 0;
#pragma unroll
                  for (int o = band_lo<K>(q); o <= band_hi<K>(q); ++o)
                    {
                      s += bK[q * W + o + K] * v[K + q + o];
                      s += bM[q * W + o + K] * w[K + q + o];
                    }
                  R[j * RS + K * c + q] -= s;
                }
            }
          __syncthreads();
        }
      // the patches: S^T along x, then y with the scaling and back, S along x
      const T *SE = tab + TB::SE, *SO = tab + TB::SO;
      T       *Q = U;
      for (int t = tid; t < NP * NP * NI; t += A2NT)
        {
          const int p = t / NI, j = t - p * NI, py = p / NP, px = p - py * NP;
          const T  *r = R + (K * py + 1 + j) * RS + K * px + 1;
          T         v[NI], w[NI];
#pragma unroll
          for (int i = 0; i < NI; ++i)
            v[i] = r[i];
          fd_fwd<K>(SE, SO, v, w);
#pragma unroll
          for (int i = 0; i < NI; ++i)
            Q[t * NI + i] = w[i];
        }
      __syncthreads();
      for (int t = tid; t < NP * NP * NI; t += A2NT)
        {
          const int p = t / NI, i = t - p * NI;
          T        *q = Q + p * NI * NI + i;
          const T  *li = tab + TB::lamInv2p + i;
          T         v[NI], w[NI];
#pragma unroll
          for (int j = 0; j < NI; ++j)
            v[j] = q[j * NI];
          fd_fwd<K>(SE, SO, v, w);
#pragma unroll
          for (int j = 0; j < NI; ++j)
            w[j] *= li[j * NI] * relax;
          fd_inv<K>(SE, SO, w, v);
#pragma unroll
          for (int j = 0; j < NI; ++j)
            q[j * NI] = v[j];
        }
      __syncthreads();
      for (int t = tid; t < NP * NP * NI; t += A2NT)
        {
          T v[NI], w[NI];
#pragma unroll
          for (int i = 0; i < NI; ++i)
            v[i] = Q[t * NI + i];
          fd_inv<K>(SE, SO, v, w);
#pragma unroll
          for (int i = 0; i < NI; ++i)
            Q[t * NI + i] = w[i];
        }
      __syncthreads();
      // owned nodes: K TC per direction, the last tile's far end as well
      constexpr int O = K * TC + 1;
      for (int t = tid; t < O * O; t += A2NT)
        {
          const int jj = t / O, ii = t - jj * O;
          const int x = x0 + K + ii, y = y0 + K + jj;
          if (x >= N1 || y >= N1 || (ii == O - 1 && x != N1 - 1) || (jj == O - 1 && y != N1 - 1))
            continue;
          T s = 0;
          if (x > 0 && y > 0 && x < N1 - 1 && y < N1 - 1)
            {
              // patch index m (window cells m, m + 1) and node in it; vertex
              // nodes are inside the patch centred there only
              const int cx = ii / K, qx = ii - cx * K, cy = jj / K, qy = jj - cy * K;
#pragma unroll
              for (int dy = 0; dy < 2; ++dy)
#pragma unroll
                for (int dx = 0; dx < 2; ++dx)
                  {
                    // patch (px, py): global vertex bx TC + px
                    const int px = cx + dx, py = cy + dy;
                    const int gx = bx * TC + px, gy = by * TC + py;
                    const int i = K * (1 - dx) + qx - 1, j = K * (1 - dy) + qy - 1;
                    if (gx > 0 && gx < n && gy > 0 && gy < n && i >= 0 && j >= 0)
                      s += Q[((py * NP + px) * NI + j) * NI + i];
                  }
            }
          out[x + (long long)y * N1] = s;
        }
    }

    template <typename T>
    __global__ void __launch_bounds__(A2NT)
    add_kernel(T *__restrict__ u, const T *__restrict__ c, const long long n)
    {
      const long long i = (long long)blockIdx.x * A2NT + threadIdx.x;
      if (i < n)
        u[i] += c[i];
    }

    template <typename T>
    void
    add2d_t(const gtps_level *lvl, T *u, const T *b, T *c, bool zero, double relax)
    {
      hipStream_t s   = lvl->ctx->stream;
      const T    *tab = (const T *)lvl->dtab();
      auto        go  = [&](auto kk) {
        constexpr int   K  = decltype(kk)::value;
        const int       nt = (lvl->n + A2<K>::TC - 1) / A2<K>::TC;
        const long long nb = (long long)nt * nt;
        GTPS_REQUIRE(nb < (1LL << 31), "too many work-groups");
        if (zero)
          hipLaunchKernelGGL((additive2d_kernel<K, T, true>), dim3((unsigned)nb), dim3(A2NT), 0,
                             s, u, b, u, tab, lvl->n, (T)relax);
        else
          hipLaunchKernelGGL((additive2d_kernel<K, T, false>), dim3((unsigned)nb), dim3(A2NT),
                             0, s, u, b, c, tab, lvl->n, (T)relax);
      };
      switch (lvl->k)
        {
          case 1: go(std::integral_constant<int, 1>{}); break;
          case 2: go(std::integral_constant<int, 2>{}); break;
          case 3: go(std::integral_constant<int, 3>{}); break;
          case 4: go(std::integral_constant<int, 4>{}); break;
          case 5: go(std::integral_constant<int, 5>{}); break;
          case 6: go(std::integral_constant<int, 6>{}); break;
          default: go(std::integral_constant<int, 7>{}); break;
        }
      GTPS_LAUNCH_CHECK();
      if (!zero)
        {
          hipLaunchKernelGGL((add_kernel<T>), dim3((unsigned)((lvl->N + A2NT - 1) / A2NT)),
                             dim3(A2NT), 0, s, u, c, lvl->N);
          GTPS_LAUNCH_CHECK();
        }
    }
  } // namespace

  // The tiles recompute the patches and nodes they share, which costs more than
  // the launches saved once a level fills the GPU; FP64 gains all the same
  // where the per-colour kernel is slow (degree 3 and from 5 on, not 4, whose
  // tile of 2 x 2 cells recomputes 9 patches for 4).  Measured on MI355X in a
  // graph, us per sweep, this / per colour (from zero): Q2 128^2 FP32 6.5 / 17
  // (4.5 / 20), 512^2 29 / 22 (18 / 27), Q5 128^2 18.9 / 27.9 (10.9 / 31),
  // 512^2 172 / 112 (106 / 125), 1024^2 699 / 383 (414 / 403), Q4 512^2 from
  // zero 79.2 / 76.9; FP64 Q2 512^2 33 / 28 (20 / 36), Q3 512^2 55 / 69 (31 /
  // 80), 2048^2 812 / 977, Q4 256^2 49 / 48 (27 / 56), 512^2 157 / 134 (85 /
  // 145), 1024^2 645 / 502 (329 / 526), 4096^2 10253 / 8395 (6368 / 8801), Q5
  // 1024^2 966 / 1014, 2048^2 3858 / 3909, Q7 512^2 485 / 775 (306 / 797).
  bool
  additive2d_pays(const gtps_level *lvl, bool zero)
  {
    const bool f64 = lvl->prec == GTPS_FP64;
    if (zero)
      return f64 || lvl->N <= (lvl->k == 4 ? 2000000 : 10000000);
    return lvl->N <= 600000 || (f64 && lvl->k >= 3 && lvl->k != 4);
  }

  void
  launch_additive2d(const gtps_level *lvl, void *u, const void *b, void *c, bool zero,
                    double relax)
  {
    if (lvl->prec == GTPS_FP32)
      add2d_t(lvl, (float *)u, (const float *)b, (float *)c, zero, relax);
    else
      add2d_t(lvl, (double *)u, (const double *)b, (double *)c, zero, relax);
  }
} // namespace gtps
