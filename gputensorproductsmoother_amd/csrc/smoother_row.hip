// smoother_row.hip - multiplicative vertex-patch sweep, two colours per
// launch: one work-group owns one x-row of patches (fixed patch index along
// y and z) and smooths its even-x and its odd-x patches one after the other.
//
// Patches of one (y, z) parity in different rows never read each other's
// interiors, and within a row the second x-parity reads of the first one
// only the middle plane of each patch, so the pair of colours needs no
// exchange between work-groups.
//
// Face form of the local solve u_I = w A_II^{-1}(b_I - A_IB u_B).  Per
// direction let the two end functions of the patch box be made M-orthogonal
// to its interior functions ("tilde" coordinates: S^T M of the whole line;
// "plain" coordinates: S^T M of its interior, i.e. S^{-1}; they differ by
// mv times the end values).  In that basis M has no interior-boundary
// entries, so the box enters only through its six faces in tilde
// coordinates.  With y and z transformed first, every eigen pair (j, k) is
// left with one 1D problem along x per patch,
//   S_x^T b^_kj / scale - at_j S_x^T M Y_kj - at_k S_x^T M Z_kj - at_i X_kj
//     = (l_i + l_j + l_k) w~_i ,
// Y and Z the faces normal to y and z (transformed in z respectively y, at
// every x), X the tilde coordinates of the two faces normal to x, and the
// plain coordinates of the result follow from
//   w = (S_x (w~ - mv_i X)) - mv_j Y_plain - mv_k Z_plain
// (the telescoped product of the three 1D changes of basis: Y tilde in z and
// nodal in x, Z plain in y and nodal in x).  The faces of a direction enter
// as sum (even eigenvectors) and difference (odd ones).  All transforms in y
// and z are shared by both x-parities, and the second parity takes its X
// from the plain coordinates of the first one's middle planes without
// leaving LDS.
#include "gtps_internal.h"

#include <type_traits>

namespace gtps
{
  namespace
  {
    // CP patches of the first parity per chunk of a row; longer rows are
    // walked chunk by chunk, carrying the last K + 1 columns.
    template <int K, int CP>
    struct RowCfg
    {
      static constexpr int NP = 2 * K + 1, NI = 2 * K - 1;
      static constexpr int WX = K * (2 * CP + 1) + 1;  // columns of a chunk
      static constexpr int RS = WX | 1;                // row stride (odd: banks)
      // LDS, in values: interior rows [k][j], then per row of faces
      static constexpr int FD = 0;                      // NI * NI rows
      static constexpr int Y  = FD + NI * NI * RS;      // [sum, diff][k]
      static constexpr int ZT = Y + 2 * NI * RS;        // [sum, diff][j], tilde
      static constexpr int ZP = ZT + 2 * NI * RS;       // [sum, diff][j], plain
      static constexpr int NR = NI * NI + 6 * NI;       // rows in all
      // x faces of the first parity, plain: CP + 1 positions and the two
      // domain ends, [pos][k][j]
      static constexpr int NPOS = CP + 3;
      static constexpr int XP   = NR * RS;
      // S_x^T M of Y and ZT per patch: [patch][row][NI]
      static constexpr int NF = 4 * NI;
      static constexpr int FS = NI;
      static constexpr int F  = XP + NPOS * NI * NI;
      static constexpr int LM = F + 2 * CP * NF * FS;   // 1 / (l_i + l_j + l_k), mv, at
      static constexpr int size = LM + NI * NI * NI + 2 * NI;
    };

    // Even/odd transforms like fd_fwd / fd_inv with the table's address hidden
    // from the optimiser once per call (even part, odd part): the entries are
    // loaded (scalar) for this call and not kept live across the stages.
    // Kept live, both tables exceed the scalar registers and every use is a
    // lane read of a spilled one: k = 7 FP64 has 5.2k VALU instructions a
    // thread instead of 4.0k, k = 5 FP64 2.3k instead of 1.9k.  Below that
    // the repeated loads cost more (k = 3 FP32 122 instead of 106 us a
    // sweep at 64^3).
    template <int K, typename T>
    constexpr bool LAUNDER = sizeof(T) == 8 ? K >= 5 : K >= 6;
    template <int K, typename T>
    __device__ __forceinline__ void
    row_fwd(const T *E_, const T *O_, const T (&v)[2 * K - 1], T (&t)[2 * K - 1])
    {
      constexpr int NI = 2 * K - 1, MH = K - 1, NE = K, NO = K - 1;
      if constexpr (!LAUNDER<K, T>)
        {
          fd_fwd<K>(E_, O_, v, t);
          return;
        }
      const ConstP<T> E = here(E_);
#pragma unroll
      for (int i = 0; i <= MH; ++i)
        {
          const T e = i < MH ? v[i] + v[NI - 1 - i] : v[MH];
#pragma unroll
          for (int q = 0; q < NE; ++q)
            t[q] = i == 0 ? E[q] * e : t[q] + E[i * NE + q] * e;
        }
      const ConstP<T> O = here(O_);
#pragma unroll
      for (int i = 0; i < MH; ++i)
        {
          const T o = v[i] - v[NI - 1 - i];
#pragma unroll
          for (int q = 0; q < NO; ++q)
            t[NE + q] = i == 0 ? O[q] * o : t[NE + q] + O[i * NO + q] * o;
        }
    }
    template <int K, typename T>
    __device__ __forceinline__ void
    row_inv(const T *E_, const T *O_, const T (&t)[2 * K - 1], T (&v)[2 * K - 1])
    {
      constexpr int NI = 2 * K - 1, MH = K - 1, NE = K, NO = K - 1;
      if constexpr (!LAUNDER<K, T>)
        {
          fd_inv<K>(E_, O_, t, v);
          return;
        }
      const ConstP<T> E = here(E_);
      T pe[MH + 1];
#pragma unroll
      for (int i = 0; i <= MH; ++i)
        {
          pe[i] = E[i * NE] * t[0];
#pragma unroll
          for (int q = 1; q < NE; ++q)
            pe[i] += E[i * NE + q] * t[q];
        }
      v[MH] = pe[MH];
      const ConstP<T> O = here(O_);
#pragma unroll
      for (int i = 0; i < MH; ++i)
        {
          T po = 0;
#pragma unroll
          for (int q = 0; q < NO; ++q)
            po += O[i * NO + q] * t[NE + q];
          v[i]          = pe[i] + po;
          v[NI - 1 - i] = pe[i] - po;
        }
    }

    // p[i] with a uniform p: scalar base, 32-bit lane offset
    template <typename T>
    __device__ __forceinline__ T &
    off32(T *p, unsigned i)
    {
      using B = std::conditional_t<std::is_const_v<T>, const char, char>;
      return *reinterpret_cast<T *>(reinterpret_cast<B *>(p) +
                                    (size_t)(unsigned)(i * (unsigned)sizeof(T)));
    }

    // ZERO: u = 0 on entry (first pair of a forward sweep): no face is read
    // and the row's share of the skeleton is set to zero.
    template <int K, typename T, bool ZERO, int CP, int NT>
    __global__ void __launch_bounds__(NT, sizeof(T) == 8 && K <= 3 ? 4 : 1)
    patch_rows3d_kernel(T *__restrict__ u, const T *__restrict__ src,
                        const T *__restrict__ tab, const int n, const int py,
                        const int pz, const int first, const T inv_scale,
                        const T relax, const FastDiv div_y)
    {
      using TB         = Tab<K>;
      using C          = RowCfg<K, CP>;
      constexpr int NP = C::NP, NI = C::NI, RS = C::RS, WX = C::WX, NE = TB::NE;
      constexpr int NPOS = C::NPOS;
      extern __shared__ double smem_raw[];
      T        *sm  = reinterpret_cast<T *>(smem_raw);
      const int tid = threadIdx.x;
      const int N1  = K * n + 1;
      const long long P = (long long)N1 * N1;
      const int npy = (n - py) / 2;
      const int row = xcd_logical_id(blockIdx.x, gridDim.x);
      const int qz  = (int)fastdiv((unsigned)row, div_y), qy = row - qz * npy;
      // first DoF of the row's box
      const long long org = (long long)K * (2 * qy + py) * N1 + (long long)K * (2 * qz + pz) * P;
      T       *ug = u + org;
      const T *sg = src + org;
      const T *SE = tab + TB::SE;
      const T *SO = tab + TB::SO;
      const T *IE = tab + TB::IE;
      const T *IO = tab + TB::IO;
      const T *mv = tab + TB::mv;
      constexpr int LV = C::LM, LA = C::LM + NI * NI * NI;  // contiguous in the table
      for (int i = tid; i < NI * NI * NI + 2 * NI; i += NT)
        sm[LV + i] = tab[TB::lamInv3p + i];
      if constexpr (ZERO)
        {
          // box rows on a y or z face, and the domain ends of the others
          for (int t = tid; t < NP * NP * N1; t += NT)
            {
              const int  r = t / N1, x = t - r * N1;
              const int  iz = r / NP, iy = r - iz * NP;
              const bool face = iz == 0 || iz == NP - 1 || iy == 0 || iy == NP - 1;
              if (face || x == 0 || x == N1 - 1)
                ug[x + iy * N1 + iz * P] = T(0);
            }
        }

      // tilde coordinates of a line
      auto tilde = [&](const T (&v)[NI], T e0, T e1, T (&w)[NI], bool plain) {
        row_fwd<K>(IE, IO, v, w);
        const T es = plain ? T(0) : e0 + e1, eo = plain ? T(0) : e0 - e1;
#pragma unroll
        for (int q = 0; q < NI; ++q)
          w[q] += mv[q] * (q < NE ? es : eo);
      };

      // The right-hand side at the domain's ends and the x face positions that
      // are no face reach no result; read with the rest (inside the box) or
      // zero, the former set where it is loaded (EARLY) or used.  No form
      // suits every degree: zero Q3 64^3 FP32 95.7 instead of 93.4 us a sweep,
      // read Q7 32^3 FP64 598 instead of 562, zero where loaded 575; Q7 32^3
      // FP32, two sweeps among those of other streams, 415 us zero where
      // loaded, 427 where used.
      constexpr bool ENDS  = !LAUNDER<K, T>;
      constexpr bool EARLY = K == 7 && sizeof(T) == 4;
      constexpr int NB = NI * WX;                       // interior lines by column
      constexpr int TF = 2 * WX + NPOS * NI;            // first face direction
      constexpr int PB = (NB + NT - 1) / NT, PF = (TF + NT - 1) / NT;
      constexpr int ROT = NB % NT;                      // face tasks start on idle lanes
      constexpr int NCY = C::NR * (K + 1), PCY = (NCY + NT - 1) / NT;
      int C0 = 0, C1 = 2 * CP + first < n ? 2 * CP + first : n;
      while (true)
        {
          const bool lead = C0 == 0, last = C1 == n;
          const int  Cw  = lead ? 0 : C0 - 1;  // first cell of the window
          const int  x0  = K * Cw;             // its first column
          const int  cn0 = lead ? 0 : K + 1, cE = K * (C1 - Cw);  // new columns
          // first-parity patches: centre vertices mA0, mA0 + 2, ...; second:
          // mB0, ...; the one that straddles C1 waits for the next chunk
          const int mA0 = C0 + 1 + (lead ? first : 0);
          const int nA  = mA0 < C1 ? (C1 - 1 - mA0) / 2 + 1 : 0;
          const int mB0 = lead ? 2 - first : C0;
          const int nB  = mB0 < C1 ? (C1 - 1 - mB0) / 2 + 1 : 0;

          // positions that are a face of the first parity
          auto x_on = [&](int pos) {
            return pos <= CP ? nA > 0 && pos <= nA
                             : first == 1 && (pos == CP + 1 ? lead : last);
          };

          // every global load first
          T rb[PB][NI];
#pragma unroll
          for (int pp = 0; pp < PB; ++pp)
            {
              const int t = tid + NT * pp, y = t / WX, col = cn0 + t - y * WX;
              const int x = x0 + col;
              if (y < NI && col <= cE && (ENDS || (x > 0 && x < N1 - 1)))
                {
                  const T *p = sg + x + (y + 1) * N1 + P;
#pragma unroll
                  for (int z = 0; z < NI; ++z)
                    rb[pp][z] = p[z * P];
                }
              else if (EARLY)
                {
#pragma unroll
                  for (int z = 0; z < NI; ++z)
                    rb[pp][z] = 0;
                }
            }
          T fl[ZERO ? 1 : PF][NP], fr[ZERO ? 1 : PF][NP];
          if constexpr (!ZERO)
            {
#pragma unroll
              for (int pp = 0; pp < PF; ++pp)
                {
                  const int t = (tid >= ROT ? tid - ROT : tid - ROT + NT) + NT * pp;
                  if (t < 2 * WX)
                    {
                      // y faces: lines along z; z faces: lines along y
                      const bool yf  = t < WX;
                      const int  col = cn0 + t - (yf ? 0 : WX);
                      if (col <= cE)
                        {
                          const long long st = yf ? P : N1;
                          const T        *p  = ug + x0 + col;
                          const T        *q  = p + (NP - 1) * (yf ? (long long)N1 : P);
#pragma unroll
                          for (int i = 0; i < NP; ++i)
                            {
                              fl[pp][i] = p[i * st];
                              fr[pp][i] = q[i * st];
                            }
                        }
                    }
                  else if (t < TF)
                    {
                      const int  m = t - 2 * WX, y = m / NPOS, pos = m - y * NPOS;
                      const int x = K * (pos <= CP ? mA0 - 1 + 2 * pos : (pos == CP + 1 ? 0 : n));
                      if (ENDS || x_on(pos))
                        {
                          const unsigned o = (unsigned)((x < N1 ? x : N1 - 1) + (y + 1) * N1);
#pragma unroll
                          for (int z = 0; z < NI; ++z)
                            fl[pp][z] = off32(ug + (z + 1) * P, o);
                        }
                    }
                }
            }

          // stage 1: along z for the right-hand side and the x faces; first
          // direction of the y and z faces
#pragma unroll
          for (int pp = 0; pp < PB; ++pp)
            {
              const int t = tid + NT * pp, y = t / WX, col = cn0 + t - y * WX;
              if (y < NI && col <= cE)
                {
                  const int x = x0 + col;
                  T        *d = sm + C::FD + y * RS + col;
                  T         tt[NI];
                  if (ENDS || EARLY || (x > 0 && x < N1 - 1))
                    row_fwd<K>(SE, SO, rb[pp], tt);
                  else
                    {
#pragma unroll
                      for (int k = 0; k < NI; ++k)
                        tt[k] = 0;
                    }
#pragma unroll
                  for (int k = 0; k < NI; ++k)
                    d[k * NI * RS] = tt[k];
                }
            }
          if constexpr (!ZERO)
            {
#pragma unroll
              for (int pp = 0; pp < PF; ++pp)
                {
                  const int t = (tid >= ROT ? tid - ROT : tid - ROT + NT) + NT * pp;
                  if (t < 2 * WX)
                    {
                      const bool yf  = t < WX;
                      const int  col = cn0 + t - (yf ? 0 : WX);
                      if (col <= cE)
                        {
                          T *d = sm + (yf ? C::Y : C::ZT) + col;
#pragma unroll
                          for (int sd = 0; sd < 2; ++sd)
                            {
                              T v[NI], p[NI];
#pragma unroll
                              for (int i = 0; i < NI; ++i)
                                v[i] = sd == 0 ? fl[pp][i + 1] + fr[pp][i + 1]
                                               : fl[pp][i + 1] - fr[pp][i + 1];
                              const T e0 = sd == 0 ? fl[pp][0] + fr[pp][0]
                                                   : fl[pp][0] - fr[pp][0];
                              const T e1 = sd == 0 ? fl[pp][NP - 1] + fr[pp][NP - 1]
                                                   : fl[pp][NP - 1] - fr[pp][NP - 1];
                              const T es = e0 + e1, eo = e0 - e1;
                              row_fwd<K>(IE, IO, v, p);
#pragma unroll
                              for (int q = 0; q < NI; ++q)
                                {
                                  if (!yf)
                                    d[C::ZP - C::ZT + (sd * NI + q) * RS] = p[q];
                                  d[(sd * NI + q) * RS] = p[q] + mv[q] * (q < NE ? es : eo);
                                }
                            }
                        }
                    }
                  else if (t < TF)
                    {
                      const int m = t - 2 * WX, y = m / NPOS, pos = m - y * NPOS;
                      T         v[NI], p[NI];
                      T        *d = sm + C::XP + pos * NI * NI + y;
#pragma unroll
                      for (int i = 0; i < NI; ++i)
                        v[i] = ENDS || x_on(pos) ? fl[pp][i] : T(0);
                      row_fwd<K>(IE, IO, v, p);
#pragma unroll
                      for (int k = 0; k < NI; ++k)
                        d[k * NI] = p[k];
                    }
                }
            }
          __syncthreads();

          // stage 2: along y for the right-hand side and the x faces; along
          // x for the y and z faces of every patch of the chunk
          for (int t = tid; t < NB; t += NT)
            {
              const int k = t / WX, col = cn0 + t - k * WX;
              if (col <= cE)
                {
                  T *d = sm + C::FD + k * NI * RS + col;
                  T  v[NI], tt[NI];
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    v[i] = d[i * RS];
                  row_fwd<K>(SE, SO, v, tt);
#pragma unroll
                  for (int j = 0; j < NI; ++j)
                    d[j * RS] = tt[j];
                }
            }
          if constexpr (!ZERO)
            {
              const int rt = tid >= ROT ? tid - ROT : tid - ROT + NT;
              for (int t = rt; t < NPOS * NI + 2 * CP * C::NF; t += NT)
                {
                  if (t < NPOS * NI)
                    {
                      T *d = sm + C::XP + t * NI;
                      T  v[NI], p[NI];
#pragma unroll
                      for (int i = 0; i < NI; ++i)
                        v[i] = d[i];
                      row_fwd<K>(IE, IO, v, p);
#pragma unroll
                      for (int j = 0; j < NI; ++j)
                        d[j] = p[j];
                    }
                  else
                    {
                      const int  s = t - NPOS * NI, pb = s / C::NF, rr = s - pb * C::NF;
                      const bool A = pb < CP;
                      const int  q = A ? pb : pb - CP;
                      if (q < (A ? nA : nB))
                        {
                          const int m = (A ? mA0 : mB0) + 2 * q;
                          const T  *v0 = sm + C::Y + rr * RS + K * (m - 1 - Cw);
                          T        *d  = sm + C::F + s * C::FS;
                          T         v[NI], p[NI];
#pragma unroll
                          for (int i = 0; i < NI; ++i)
                            v[i] = v0[i + 1];
                          tilde(v, v0[0], v0[NP - 1], p, false);
#pragma unroll
                          for (int i = 0; i < NI; ++i)
                            d[i] = p[i];
                        }
                    }
                }
            }
          __syncthreads();

          // stage 3: the 1D problems along x, first parity, then second
          T carry[PCY];
#pragma unroll
          for (int ph = 0; ph < 2; ++ph)
            {
              const int np = ph == 0 ? nA : nB, m0 = ph == 0 ? mA0 : mB0;
              for (int t = tid; t < np * NI * NI; t += NT)
                {
                  const int p = t / (NI * NI), r = t - p * (NI * NI);
                  const int k = r / NI, j = r - k * NI;
                  const int m = m0 + 2 * p, c0 = K * (m - 1 - Cw);
                  T        *d = sm + C::FD + r * RS + c0;
                  const T  *y = sm + C::Y + ((j < NE ? 0 : NI) + k) * RS + c0;
                  const T  *z = sm + C::ZP + ((k < NE ? 0 : NI) + j) * RS + c0;
                  const T   my = sm[LA + j], mz = sm[LA + k];
                  const T  *lv = sm + LV + r * NI;
                  T         v[NI], tt[NI];
                  T xl = 0, xr = 0;
                  if (ph == 0)
                    {
                      if (!ZERO)
                        {
                          xl = sm[C::XP + p * NI * NI + r];
                          xr = sm[C::XP + (p + 1) * NI * NI + r];
                        }
                    }
                  else
                    {
                      if (m > 1)
                        xl = d[0];
                      else if (!ZERO)
                        xl = sm[C::XP + (CP + 1) * NI * NI + r];
                      if (m < n - 1)
                        xr = d[2 * K];
                      else if (!ZERO)
                        xr = sm[C::XP + (CP + 2) * NI * NI + r];
                    }
                  if (!ZERO)
                    {
                      xl += my * y[0] + mz * z[0];
                      xr += my * y[2 * K] + mz * z[2 * K];
                    }
                  const T fe = xl + xr, fo = xl - xr;
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    v[i] = d[i + 1];
                  row_fwd<K>(SE, SO, v, tt);
                  const T  ay = sm[LA + NI + j], az = sm[LA + NI + k];
                  const auto ma = [&] { if constexpr (LAUNDER<K, T>) return here(mv); else return mv; }();
                  const T *fy = sm + C::F + ((ph * CP + p) * C::NF + (j < NE ? 0 : NI) + k) * C::FS;
                  const T *fz = sm + C::F +
                                ((ph * CP + p) * C::NF + 2 * NI + (k < NE ? 0 : NI) + j) * C::FS;
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    {
                      const T x  = i < NE ? fe : fo;
                      T       c1 = tt[i] * inv_scale;
                      c1 -= ma[NI + i] * x;
                      if (!ZERO)
                        {
                          c1 -= ay * fy[i];
                          c1 -= az * fz[i];
                        }
                      tt[i] = c1 * lv[i] - ma[i] * x;
                    }
                  row_inv<K>(SE, SO, tt, v);
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    {
                      // the first parity's columns off the middle plane stay
                      // right-hand side for the second one, but for the two
                      // half patches at the domain's ends
                      const bool keep = ph == 1 || i == K - 1 || (i < K - 1 && m == 1) ||
                                        (i > K - 1 && m == n - 1);
                      T w = v[i];
                      if (!ZERO)
                        w -= my * y[i + 1] + mz * z[i + 1];
                      if (keep)
                        d[i + 1] = relax * w;
                    }
                }
              if (ph == 1 && !last)
                {
#pragma unroll
                  for (int pp = 0; pp < PCY; ++pp)
                    {
                      const int t = tid + NT * pp;
                      if (t < NCY)
                        carry[pp] = sm[(t / (K + 1)) * RS + K * (C1 - 1 - Cw) + t % (K + 1)];
                    }
                }
              __syncthreads();
            }

          // stages 4 and 5: back along y, then along z, for the columns that
          // are final
          const int cO = last ? cE - 1 : cE - K;
          for (int t = tid; t < NB; t += NT)
            {
              const int k = t / WX, col = 1 + t - k * WX;
              if (col <= cO)
                {
                  T *d = sm + C::FD + k * NI * RS + col;
                  T  v[NI], o[NI];
#pragma unroll
                  for (int j = 0; j < NI; ++j)
                    v[j] = d[j * RS];
                  row_inv<K>(SE, SO, v, o);
#pragma unroll
                  for (int i = 0; i < NI; ++i)
                    d[i * RS] = o[i];
                }
            }
          __syncthreads();
          for (int t = tid; t < NB; t += NT)
            {
              const int y = t / WX, col = 1 + t - y * WX;
              if (col <= cO)
                {
                  const T *d = sm + C::FD + y * RS + col;
                  T        v[NI], o[NI];
                  const unsigned g = (unsigned)(x0 + col + (y + 1) * N1);
#pragma unroll
                  for (int k = 0; k < NI; ++k)
                    v[k] = d[k * NI * RS];
                  row_inv<K>(SE, SO, v, o);
#pragma unroll
                  for (int z = 0; z < NI; ++z)
                    off32(ug + (z + 1) * P, g) = o[z];
                }
            }
          if (last)
            break;
          __syncthreads();
#pragma unroll
          for (int pp = 0; pp < PCY; ++pp)
            {
              const int t = tid + NT * pp;
              if (t < NCY)
                sm[(t / (K + 1)) * RS + t % (K + 1)] = carry[pp];
            }
          C0 = C1;
          C1 = C0 + 2 * CP < n ? C0 + 2 * CP : n;
        }
    }

    template <int K, typename T, int CP, int NT>
    void
    launch_cfg(const gtps_level *lvl, T *u, const T *src, int py, int pz, int first, bool zero,
               double relax)
    {
      using C             = RowCfg<K, CP>;
      const int     n     = lvl->n;
      const int     npy   = (n - py) / 2, npz = (n - pz) / 2;
      const size_t  lds   = C::size * sizeof(T);
      static_assert(C::size * sizeof(T) <= 160 * 1024, "row chunk exceeds the LDS");
      const T      *tab   = reinterpret_cast<const T *>(lvl->dtab());
      const FastDiv dy    = make_fastdiv((unsigned)npy);
      auto          go    = [&](auto kern) {
        if (lds > 65536)
          GTPS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kern, dim3((unsigned)((long long)npy * npz)), dim3(NT), lds,
                           lvl->ctx->stream, u, src, tab, n, py, pz, first,
                           (T)(1.0 / lvl->scale), (T)relax, dy);
      };
      if (zero)
        go(patch_rows3d_kernel<K, T, true, CP, NT>);
      else
        go(patch_rows3d_kernel<K, T, false, CP, NT>);
      GTPS_LAUNCH_CHECK();
    }

    template <typename T>
    void
    launch_t(const gtps_level *lvl, T *u, const T *src, int py, int pz, int first, bool zero,
             double relax)
    {
      // Chunk length and lanes per row: one pass of the NI (2K CP + K + 1)
      // interior lines per stage where registers and LDS leave at least two
      // work-groups a CU.  Measured on MI355X, us per sweep: k = 3 FP32 at
      // 64^3 98 with (16, 256) and 106 with (16, 512), at 32^3 36 and 27
      // (a quarter of the rows: latency; in a graph 93 and 25 as they are
      // now); k = 4 32^3 55 with (8, 512), 94 with (4, 256); k = 7 FP32 32^3
      // 262 with (4, 1024), 298 with
      // (4, 512), FP64 568 with (3, 512), 683 with (2, 512), 908 with
      // (3, 1024) (spills).
      constexpr bool d = sizeof(T) == 8;
#define GTPS_ROW(K, CP, NT) return launch_cfg<K, T, CP, NT>(lvl, u, src, py, pz, first, zero, relax)
      switch (lvl->k)
        {
          case 1: GTPS_ROW(1, 64, 256);
          case 2: GTPS_ROW(2, 32, 512);
          case 3:
            if (!d && lvl->n >= 64)
              GTPS_ROW(3, 16, 256);
            GTPS_ROW(3, 16, 512);
          case 4: GTPS_ROW(4, 8, 512);
          case 5: GTPS_ROW(5, (d ? 5 : 6), 512);
          case 6: GTPS_ROW(6, 4, 512);
          case 7: GTPS_ROW(7, (d ? 3 : 4), (d ? 512 : 1024));
          default: throw Error(GTPS_EINVAL, "degree must be in 1..7");
        }
#undef GTPS_ROW
    }
  } // namespace

  // colours (first, py, pz) and (1 - first, py, pz) of the multiplicative
  // sweep, in this order
  void
  launch_patch_rows(const gtps_level *lvl, void *u, const void *src, int py, int pz, int first,
                    bool zero, double relax)
  {
    if (lvl->n - py < 2 || lvl->n - pz < 2)
      return;
    if (lvl->prec == GTPS_FP32)
      launch_t(lvl, (float *)u, (const float *)src, py, pz, first, zero, relax);
    else
      launch_t(lvl, (double *)u, (const double *)src, py, pz, first, zero, relax);
  }
} // namespace gtps
