// dg_row.hip - SIPG-DG vertex-patch sweep, three colours per launch: one
// work-group owns one x-row of patches (fixed y and z patch index) and smooths
// its patches p = 0, 1, 2 (mod 3) one class after the other.
//
// Rows of one (y, z) colour touch disjoint cells, and the y- and z-neighbour
// cells of a row belong to no row of the same colour, so the three x-classes
// of a row need no exchange between work-groups.
//
// Face form of the local solve u_P = A_PP^{-1}(b_P - A_P,ext u_ext).  The
// off-diagonal blocks of L have rank two: a neighbour cell enters through its
// trace and one combination of trace and normal derivative on the shared
// face.  With y and z in the eigen coordinates of the row (S^T of the
// right-hand side, S^T M of u) every pair (k, j) is an independent 1D problem
// along x, g = S_z^T S_y^T b / scale - M_x (faces normal to y and z), which
// the patches of the row solve in turn:
//   w = S_x [S_x^T g - (faces normal to x)] / (l_i + l_j + l_k) ;
// a patch hands the two traces of one of its cells to the later classes.
// Everything along y and z is done once per row instead of once per patch.
#include "gtps_internal.h"

#include <type_traits>

namespace gtps
{
  namespace
  {
    template <int K>
    struct DR
    {
      static constexpr int NN = K + 1, NI = 2 * NN, N2 = NI * NI;
      // LDS, in values, for n cells: G [k][j] rows of RS; face arrays F
      // [4 y faces][k] and [4 z faces][j] rows of RS, which the traces of
      // class A take over; traces O and of one special cell [4][k][j]; per
      // lane constants
      __host__ __device__ static int rs(int n) { return (n * NN) | 1; }
      __host__ __device__ static int slots(int n) { return (n + 2) / 3; }
      __host__ __device__ static int F(int n) { return N2 * rs(n); }
      __host__ __device__ static int O(int n) { return F(n) + 8 * NI * rs(n); }
      __host__ __device__ static int SP(int n) { return O(n) + slots(n) * 4 * N2; }
      __host__ __device__ static int CT(int n) { return SP(n) + 4 * N2; }
      __host__ __device__ static int size(int n) { return CT(n) + 10 * NI; }
    };

    // t_q = sum_a A[a][q] v_a, and v_a = sum_q A[a][q] t_q
    template <int NI, typename T>
    __device__ __forceinline__ void
    dense_t(const T *A_, const T (&v)[NI], T (&t)[NI])
    {
      const ConstP<T> A = here(A_);
#pragma unroll
      for (int a = 0; a < NI; ++a)
#pragma unroll
        for (int q = 0; q < NI; ++q)
          t[q] = a == 0 ? A[q] * v[0] : t[q] + A[a * NI + q] * v[a];
    }
    template <int NI, typename T>
    __device__ __forceinline__ void
    dense_n(const T *A_, const T (&t)[NI], T (&v)[NI])
    {
      const ConstP<T> A = here(A_);
#pragma unroll
      for (int a = 0; a < NI; ++a)
        {
          T s = A[a * NI] * t[0];
#pragma unroll
          for (int q = 1; q < NI; ++q)
            s += A[a * NI + q] * t[q];
          v[a] = s;
        }
    }

    template <int K, typename T, int NT>
    __global__ void __launch_bounds__(NT)
    dg_rows_kernel(T *__restrict__ u_, const T *__restrict__ b_, const T *__restrict__ tab,
                   const int n, const int cy, const int cz, const int rev, const T scale,
                   const FastDiv div_y, const FastDiv div_n1)
    {
      using C          = DR<K>;
      using TB         = DTab<K>;
      constexpr int NN = C::NN, NI = C::NI, N2 = C::N2;
      extern __shared__ double smem_raw[];
      T              *sm  = reinterpret_cast<T *>(smem_raw);
      const int       tid = threadIdx.x;
      const int       N1 = n * NN, RS = C::rs(n);
      const long long P = (long long)N1 * N1;
      const int       row = xcd_logical_id(blockIdx.x, gridDim.x);
      const int       qz = (int)fastdiv((unsigned)row, div_y);
      const int       py = cy + 3 * (row - qz * (int)div_y.d), pz = cz + 3 * qz;
      const long long org = (long long)py * NN * N1 + (long long)pz * NN * P;
      T       *ug = u_ + (long long)blockIdx.y * P * N1 + org;
      const T *bg = b_ + (long long)blockIdx.y * P * N1 + org;
      const int vy = (py == 0 ? 1 : 0) + (py + 2 == n ? 2 : 0);
      const int vz = (pz == 0 ? 1 : 0) + (pz + 2 == n ? 2 : 0);
      const T  *Sy = tab + TB::S + vy * N2, *Sz = tab + TB::S + vz * N2;
      const T  *My = tab + TB::MS + vy * N2, *Mz = tab + TB::MS + vz * N2;
      T *G = sm, *F = sm + C::F(n), *O = sm + C::O(n), *SP = sm + C::SP(n), *CT = sm + C::CT(n);
      T *A = F;  // once the face arrays are used up

      // per-lane constants: couplings of the y (0..3) and z (4..7) faces to
      // the eigenvectors, then the eigenvalues
      static_assert(10 * NI <= NT, "one constant per thread");
      T ctv = 0;
      if (tid < 10 * NI)
        {
          const int  f = tid / NI, j = tid - f * NI;
          const bool z = f >= 4 && f != 8;
          const int  v = z ? vz : vy, e = f & 3;
          const int  o = f >= 8   ? TB::lam + v * NI
                         : e == 0 ? TB::S + v * N2
                         : e == 1 ? TB::EL + v * NI
                         : e == 2 ? TB::S + v * N2 + (NI - 1) * NI
                                  : TB::ER + v * NI;
          ctv          = tab[o + j];
        }

      // stage 1: along z for the right-hand side and the y faces and x
      // traces, along y for the z faces.  Tasks: [faces | x traces | b]
      const int r0 = rev ? 1 : 2;  // class whose original traces come first
      // the cell of class 0 that no patch covers before class 1 reads it
      const int sp  = rev ? 0 : ((n - 1) % 3 == 0 ? n - 1 : -1);
      const int nO  = (n - r0 + 2) / 3;
      // Whole wavefronts per kind of task, so that the tables are uniform.
      const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
      const int wF = (2 * N1 + 63) / 64, wX = ((nO + 1) * NI + 63) / 64;
      const int tB = NI * N1, wB = (tB + 63) / 64;
      // face and trace waves: lane -> cell line w (normal stride sn, other
      // stride so), its end and the destination; everything else uniform
      for (int w = wave; w < 2 * wF + 2 * wX + wB; w += NT / 64)
        {
          if (w < 2 * wF + 2 * wX)
            {
              const bool zf = w >= wF, tr = w >= 2 * wF, t1 = w >= 2 * wF + wX;
              const int  t  = (w - (t1 ? 2 * wF + wX : tr ? 2 * wF : zf ? wF : 0)) * 64 + lane;
              const long long sn = tr ? 1 : (zf ? P : N1), so = tr || !zf ? P : N1;
              const T  *Mo = tr || !zf ? Mz : My;
              const int st = tr ? NI : RS;       // destination stride
              const int sb = tr ? N2 : NI * RS;  // second value
              bool      on, use, hi;
              const T  *p = ug;
              T        *d;
              if (tr)
                {
                  // traces of an original cell: right end (the cell is a
                  // left neighbour) or left end
                  const int s = t / NI, y = t - s * NI, c = s < nO ? r0 + 3 * s : sp;
                  hi = t1;
                  on = use = s <= nO && c >= 0;
                  p += c * NN + (long long)y * N1;
                  d = (s < nO ? O + s * 4 * N2 : SP) + (t1 ? 2 * N2 : 0) + y;
                }
              else
                {
                  const int q = zf ? pz : py;
                  hi          = t >= N1;
                  const int x = hi ? t - N1 : t;
                  use         = t < 2 * N1;
                  on          = use && (hi ? q + 2 < n : q > 0);
                  p += x + (hi ? NI * sn : -NN * sn);
                  d = F + (zf ? 4 * NI * RS : 0) + (hi ? 2 : 0) * NI * RS + x;
                }
              T v[NI][NN], ga[NI], gb[NI], tt[NI];
              if (on)
                {
#pragma unroll
                  for (int a = 0; a < NI; ++a)
#pragma unroll
                    for (int i = 0; i < NN; ++i)
                      v[a][i] = p[a * so + i * sn];
                }
              else
                {
#pragma unroll
                  for (int a = 0; a < NI; ++a)
#pragma unroll
                    for (int i = 0; i < NN; ++i)
                      v[a][i] = 0;
                }
              const ConstP<T> al = here(tab + TB::AL), ar = here(tab + TB::AR);
              T               cf[NN];
#pragma unroll
              for (int i = 0; i < NN; ++i)
                cf[i] = hi ? al[i] : ar[i];
#pragma unroll
              for (int a = 0; a < NI; ++a)
                {
                  T s = 0;
#pragma unroll
                  for (int i = 0; i < NN; ++i)
                    s += cf[i] * v[a][i];
                  ga[a] = s;
                  gb[a] = hi ? T(0.5) * v[a][0] : T(-0.5) * v[a][NN - 1];
                }
              dense_t<NI>(Mo, ga, tt);
              if (use)
                {
#pragma unroll
                  for (int k = 0; k < NI; ++k)
                    d[k * st] = tt[k];
                }
              dense_t<NI>(Mo, gb, tt);
              if (use)
                {
#pragma unroll
                  for (int k = 0; k < NI; ++k)
                    d[sb + k * st] = tt[k];
                }
            }
          else
            {
              const int m = (w - 2 * wF - 2 * wX) * 64 + lane;
              if (m < tB)
                {
                  const int y = (int)fastdiv((unsigned)m, div_n1), x = m - y * N1;
                  const T  *g = bg + x + (long long)y * N1;
                  T         v[NI], tt[NI];
#pragma unroll
                  for (int z = 0; z < NI; ++z)
                    v[z] = g[z * P];
                  dense_t<NI>(Sz, v, tt);
                  T *d = G + y * RS + x;
#pragma unroll
                  for (int k = 0; k < NI; ++k)
                    d[k * NI * RS] = tt[k];
                }
            }
        }
      if (tid < 10 * NI)
        CT[tid] = ctv;
      __syncthreads();
      // stage 2: along y for the right-hand side and the x traces
      const int tO = (nO + 1) * 4 * NI, wO = (tO + 63) / 64;
      for (int w = wave; w < wO + wB; w += NT / 64)
        {
          const bool o = w < wO;
          const int  m = (o ? w : w - wO) * 64 + lane;
          if (m < (o ? tO : tB))
            {
              T  v[NI], tt[NI];
              T *d;
              if (o)
                d = (m < nO * 4 * NI ? O : SP - nO * 4 * N2) + m * NI;
              else
                {
                  const int k = (int)fastdiv((unsigned)m, div_n1);
                  d           = G + k * NI * RS + (m - k * N1);
                }
              const int st = o ? 1 : RS;
#pragma unroll
              for (int y = 0; y < NI; ++y)
                v[y] = d[y * st];
              dense_t<NI>(o ? My : Sy, v, tt);
#pragma unroll
              for (int j = 0; j < NI; ++j)
                d[j * st] = tt[j];
            }
        }
      __syncthreads();
      // g = b^ / scale - M_x (y and z faces), cell by cell
      const T inv_scale = T(1) / scale;
      for (int t = tid; t < n * N2; t += NT)
        {
          const int c = t / N2, r = t - c * N2, k = r / NI, j = r - k * NI;
          T        *d  = G + r * RS + c * NN;
          const T  *fy = F + k * RS + c * NN, *fz = F + (4 * NI + j) * RS + c * NN;
          T         q[NN];
#pragma unroll
          for (int i = 0; i < NN; ++i)
            q[i] = 0;
#pragma unroll
          for (int f = 0; f < 4; ++f)
            {
              const T a = CT[f * NI + j], b = CT[(4 + f) * NI + k];
#pragma unroll
              for (int i = 0; i < NN; ++i)
                q[i] += a * fy[f * NI * RS + i] + b * fz[f * NI * RS + i];
            }
          const ConstP<T> M = here(tab + TB::M);
#pragma unroll
          for (int i = 0; i < NN; ++i)
            {
              T s = d[i] * inv_scale;
#pragma unroll
              for (int a = 0; a < NN; ++a)
                s -= M[i * NN + a] * q[a];
              d[i] = s;
            }
        }
      __syncthreads();
      // the 1D problems, class after class.  Wavefronts take whole blocks of
      // lines of one boundary variant: the interior patches of the class
      // packed, then the patch at the left and the one at the right end
      constexpr int WP = (N2 + 63) / 64;
      for (int ph = 0; ph < 3; ++ph)
        {
          const int  cl = rev ? 2 - ph : ph;  // patch class
          const bool hasL = cl == 0, hasR = (n - 2) % 3 == cl;
          const int  first = hasL ? 3 : cl;                      // first interior patch
          const int  endI  = hasR ? n - 2 : n - 1;               // interior: p < endI
          const int  nInt  = first < endI ? (endI - 1 - first) / 3 + 1 : 0;
          const int  wI    = (nInt * N2 + 63) / 64;
          const int  wT    = wI + (hasL ? WP : 0) + (hasR ? WP : 0);
          for (int w = wave; w < wT; w += NT / 64)
            {
              const bool inner = w < wI, left = !inner && hasL && w < wI + WP;
              const int  v     = inner ? 0 : (left ? 1 : 2);
              const int  t     = (inner ? w : w - wI - (!left && hasL ? WP : 0)) * 64 + lane;
              const int  ip = t / N2, r = t - ip * N2;
              if (inner ? ip >= nInt : ip >= 1)
                continue;
              const int p = inner ? first + 3 * ip : (left ? 0 : n - 2);
              const int k = r / NI, j = r - k * NI;
              T        *d = G + r * RS + p * NN;
              const T  *Sx = tab + TB::S + v * N2;
              T         x[NI], tt[NI];
#pragma unroll
              for (int i = 0; i < NI; ++i)
                x[i] = d[i];
              dense_t<NI>(Sx, x, tt);
              // traces of the neighbours: class 0 cells in A, the others
              // in O; the special one apart
              auto tr = [&](int c) -> const T * {
                return c == sp && ph == 1 ? SP + r
                       : ph == 1          ? A + (c / 3) * 4 * N2 + r
                                          : O + (c / 3) * 4 * N2 + r;
              };
              if (!left)
                {
                  const T        *q  = tr(p - 1);
                  const T         ga = q[0], gb = q[N2];
                  const ConstP<T> el = here(tab + TB::EL + v * NI), s0 = here(Sx);
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    tt[i] -= s0[i] * ga + el[i] * gb;
                }
              if (inner || left)
                {
                  const T        *q  = tr(p + 2);
                  const T         ha = q[2 * N2], hb = q[3 * N2];
                  const ConstP<T> er = here(tab + TB::ER + v * NI),
                                  s1 = here(Sx + (NI - 1) * NI);
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    tt[i] -= s1[i] * ha + er[i] * hb;
                }
              const T         ljk = CT[8 * NI + j] + CT[9 * NI + k];
              const ConstP<T> lam = here(tab + TB::lam + v * NI);
#pragma unroll
              for (int i = 0; i < NI; ++i)
                {
                  // FP32: hardware reciprocal (1 ulp), FP64: IEEE division
                  const T den = lam[i] + ljk;
                  if constexpr (sizeof(T) == 4)
                    tt[i] *= __builtin_amdgcn_rcpf(den);
                  else
                    tt[i] /= den;
                }
              dense_n<NI>(Sx, tt, x);
              // a cell's right-hand side stays until its last patch
              const int  cp = p % 3;  // = cl
              const bool lastL = p == 0 || (rev ? (cp + 2) % 3 > cp : (cp + 2) % 3 < cp);
              const bool lastR = p == n - 2 || (rev ? (cp + 1) % 3 > cp : (cp + 1) % 3 < cp);
              if (lastL)
                {
#pragma unroll
                  for (int i = 0; i < NN; ++i)
                    d[i] = x[i];
                }
              if (lastR)
                {
#pragma unroll
                  for (int i = NN; i < NI; ++i)
                    d[i] = x[i];
                }
              if (ph < 2)
                {
                  // traces of the left cell (right cell when reversed)
                  const ConstP<T> al = here(tab + TB::AL), ar = here(tab + TB::AR);
                  T              *q  = (ph == 0 ? A : O) + ((p + rev) / 3) * 4 * N2 + r;
                  T               ga = 0, ha = 0;
#pragma unroll
                  for (int i = 0; i < NN; ++i)
                    {
                      const T xi = rev ? x[NN + i] : x[i];
                      ga += ar[i] * xi;
                      ha += al[i] * xi;
                    }
                  q[0]      = ga;
                  q[N2]     = T(-0.5) * (rev ? x[NI - 1] : x[NN - 1]);
                  q[2 * N2] = ha;
                  q[3 * N2] = T(0.5) * (rev ? x[NN] : x[0]);
                  if (!rev && ph == 0 && p == n - 2 && n % 3 == 2)
                    {
                      // the last cell is the left cell of no patch: its left
                      // end goes to the third class from here
                      T *qe = O + ((n - 1) / 3) * 4 * N2 + r, he = 0;
#pragma unroll
                      for (int i = 0; i < NN; ++i)
                        he += al[i] * x[NN + i];
                      qe[2 * N2] = he;
                      qe[3 * N2] = T(0.5) * x[NN];
                    }
                }
            }
          __syncthreads();
        }
      // back along y, then along z with the store
      for (int t = tid; t < tB; t += NT)
        {
          const int k = (int)fastdiv((unsigned)t, div_n1), x = t - k * N1;
          T        *d = G + k * NI * RS + x;
          T         v[NI], o[NI];
#pragma unroll
          for (int j = 0; j < NI; ++j)
            v[j] = d[j * RS];
          dense_n<NI>(Sy, v, o);
#pragma unroll
          for (int y = 0; y < NI; ++y)
            d[y * RS] = o[y];
        }
      __syncthreads();
      for (int t = tid; t < tB; t += NT)
        {
          const int y = (int)fastdiv((unsigned)t, div_n1), x = t - y * N1;
          const T  *d = G + y * RS + x;
          T        *w = ug + x + (long long)y * N1;
          T         v[NI], o[NI];
#pragma unroll
          for (int k = 0; k < NI; ++k)
            v[k] = d[k * NI * RS];
          dense_n<NI>(Sz, v, o);
#pragma unroll
          for (int z = 0; z < NI; ++z)
            w[z * P] = o[z];
        }
    }

    template <int K, typename T>
    void
    rows_k(const gtps_dg_level *lvl, T *u, const T *b, bool reverse, int nvec)
    {
      constexpr int NT   = 1024;
      const int     n    = lvl->n;
      const size_t  lds  = DR<K>::size(n) * sizeof(T);
      auto          kern = dg_rows_kernel<K, T, NT>;
      if (lds > 65536)
        GTPS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      for (int cc = 0; cc < 9; ++cc)
        {
          const int c = reverse ? 8 - cc : cc, cy = c % 3, cz = c / 3;
          if (cy >= n - 1 || cz >= n - 1)
            continue;
          const int npy = (n - 1 - cy + 2) / 3, npz = (n - 1 - cz + 2) / 3;
          hipLaunchKernelGGL(kern, dim3((unsigned)(npy * npz), nvec), dim3(NT), lds,
                             lvl->ctx->stream, u, b, (const T *)lvl->tab, n, cy, cz,
                             reverse ? 1 : 0, (T)lvl->scale, make_fastdiv((unsigned)npy),
                             make_fastdiv((unsigned)lvl->N1));
          GTPS_LAUNCH_CHECK();
        }
    }

    template <typename F>
    auto
    row_dispatch(int k, F f)
    {
      switch (k)
        {
          case 1: return f(std::integral_constant<int, 1>{});
          case 2: return f(std::integral_constant<int, 2>{});
          case 3: return f(std::integral_constant<int, 3>{});
          case 4: return f(std::integral_constant<int, 4>{});
          case 5: return f(std::integral_constant<int, 5>{});
          case 6: return f(std::integral_constant<int, 6>{});
          case 7: return f(std::integral_constant<int, 7>{});
          default: throw Error(GTPS_EINVAL, "degree must be in 1..7");
        }
    }
  } // namespace

  // Where three colours per launch are the faster form for nvec vectors at
  // once.  A row is one work-group whose time grows with n, while a colour
  // takes the time of one patch as long as its work-groups fit the 256 CUs at
  // once; with the cheaper local solve of low degrees the launches saved decide
  // on every mesh.  Measured on MI355X in a graph, us per sweep, rows /
  // colours, one vector (four): FP32 k = 1 5^3 58 / 96, 24^3 64 / 109 (67 /
  // 162), k = 2 24^3 91 / 136 (97 / 211), k = 3 12^3 111 / 136, 20^3 135 / 152,
  // k = 4 6^3 140 / 170 (141 / 173), 10^3 169 / 171, 12^3 180 / 171 (184 /
  // 182), 14^3 189 / 178 (197 / 235), 16^3 209 / 179 (215 / 256), 19^3 230 /
  // 184 (241 / 431), 24^3 267 / 251 (289 / 717), 28^3 297 / 350, k = 5 11^3 247
  // / 253, 14^3 293 / 254 (306 / 428), 19^3 348 / 265 (368 / 956), 24^3 420 /
  // 503, k = 6 9^3 323 / 358, 12^3 415 / 367; FP64 k = 1 24^3 74 / 121, k = 2
  // 12^3 107 / 132, k = 3 12^3 154 / 160, 16^3 179 / 162 (184 / 233), 19^3 188
  // / 165 (197 / 376), 24^3 210 / 229 (231 / 628), k = 4 8^3 211 / 209, 12^3
  // 249 / 213, k = 5 7^3 361 / 365, 8^3 393 / 366.
  bool
  dg_rows_fit(int k, int prec, int n, int nvec)
  {
    const bool   f32  = prec == GTPS_FP32;
    const size_t size = row_dispatch(k, [&](auto kk) {
      return (size_t)DR<decltype(kk)::value>::size(n) * (f32 ? 4 : 8);
    });
    const int largest = f32 ? (k <= 5 ? n : 9) : (k <= 3 ? n : k == 4 ? 8 : 7);
    if (n < 5 || size > 160 * 1024 || n > largest)
      return false;
    // degrees and meshes on which the colours win while they fit the chip
    const int from = f32 ? (k == 4 ? 11 : k == 5 ? 12 : n + 1) : (k == 3 ? 15 : n + 1);
    if (n < from)
      return true;
    const long long side = (n + 1) / 3;  // of the largest colour
    const bool one_round = side * side * side * nvec <= 256 ||
                           (nvec == 1 && n <= (f32 && k == 4 ? 24 : 20));
    return !one_round;
  }

  void
  launch_dg_rows(const gtps_dg_level *lvl, void *u, const void *b, bool reverse, int nvec)
  {
    row_dispatch(lvl->k, [&](auto kk) {
      constexpr int K = decltype(kk)::value;
      if (lvl->prec == GTPS_FP32)
        rows_k<K>(lvl, (float *)u, (const float *)b, reverse, nvec);
      else
        rows_k<K>(lvl, (double *)u, (const double *)b, reverse, nvec);
      return 0;
    });
  }
} // namespace gtps
