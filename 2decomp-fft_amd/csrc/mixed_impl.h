// mixed_impl.h -- axis stages of any length with factors 2-17 (gfx950).
//
// The specialised kernels (fast_impl.h) fix the length at compile time and
// the general kernel (fft_kernels.hip) calls one non-inlined function per
// pass, which costs it 248 VGPRs (2 waves per SIMD) and callee-saved
// registers spilled around every call.  Here the radix of a pass is a
// compile-time case of a uniform switch and everything else (length, tile,
// rows) is read from the descriptor, so one kernel serves every length
// without calls.  In FP64 the lengths with factors 2-7 and the chirps hold up to
// 128 VGPRs (4 waves per SIMD), factors up to 17 up to 183 (2-3 waves); FP32 58-109
// (4-8 waves).  Only packed columns (60 bytes a lane in FP64, 52 in FP32), the FP64
// real-to-real lines of factors up to 17 (36) and some of the chirps (8-68) use
// scratch.
//
// A workgroup owns a tile of TX columns of n points; `rows` threads share a
// column and take butterflies row, row + rows, ... of every pass, about 10
// values each (mx_nb; up to 20 in FP32 columns).  Strided columns put
// consecutive threads on consecutive tile columns (one run of 128 bytes or more
// per point); contiguous lines put them on consecutive points of a line.  The
// first pass reads HBM, the last writes HBM, those in between exchange through
// LDS; real transforms pair two real columns as the general kernel does.
//
// Measured against the general kernel on 0.8 GB stages, FP64 TB/s of the bytes
// read and written once (columns c2c / lines r2c / lines c2r):
//   n = 100  2.0 / 2.7 / 2.3 -> 5.2 / 5.5 / 5.1
//   n = 405  1.9 / 3.0 / 2.4 -> 4.4 / 4.7 / 4.6
//   n = 1000 1.3 / 2.0 / 1.6 -> 3.9 / 4.9 / 4.9
// Class 2 ("chirp") runs lengths with a prime factor above 17 by Bluestein's
// algorithm over a length m >= 2n - 1 (mixed_length), in place (the general kernel
// sweeps the LDS tile twelve times at n = 382): columns of 101 / 191 / 382 / 1021
// points 1.0 / 0.8 / 0.8 / 0.9 -> 2.4 / 2.1 / 1.9 / 1.8 TB/s.  It is bound by latency and
// by the loads of twiddles, chirp and spectrum: on the 382-point columns of a
// 450 x 405 grid waves wait 49 % of their time, the address units are busy 61 %
// of the launch, the vector units half of the time that a workgroup is on the
// CU.  Its radices are those of its convolution lengths, up to 12, where FP64 still
// fits 128 VGPRs with a pass's twiddles loaded ahead.
// Real-to-real stages (columns / lines, the general kernel -> here): DCT-II of
// 300 points 1.2 / 1.3 -> 3.9 / 3.7 TB/s, DCT-I 0.9 / 0.9 -> 2.8 / 2.9, DCT-IV 0.3 /
// 0.3 -> 3.3 / 3.5; on 513-point grids the compiled DCT-I tiles run at 2.0 / 2.1
// where these reach 2.5 / 2.7, the DCT-IV ones at 2.7 / 2.8 against 3.7 / 3.9 (on
// small pencils the tiles are ahead: dtt_choice, plan.cpp).
// What bounds the Stockham classes: up to 600 points the HBM rate of the access
// pattern; longer columns the workgroups per CU, since a tile of 8 columns takes
// over half of the LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include "codelets.h"
#include "fast_kernels.h"
#include "internal.h"

namespace d2dhip {

namespace {

// Butterflies of radix r that a lane takes per pass: one, or as many as make
// 10 values, 20 of FP32 columns (at most 4).  (20 FP32 values: columns of 450
// points 4.7 -> 5.2 TB/s, 675 3.4 -> 5.1; lines of 405 points 4.3 -> 3.5.)
constexpr int mx_nb(int r, int rb, bool lines) {
  const int per = (rb == 4 && !lines ? 20 : 10) / r;
  return per < 1 ? 1 : (per < 4 ? per : 4);
}

// Radices by kernel class: 0 the codelets that fit 128 VGPRs in FP64 at 1024
// threads (real-to-real stages only those up to 12: set 2), 1 the large primes too
// (512 threads), 2 (chirp) those of the convolution lengths: set 3.
constexpr int mx_set(int cls, int io) { return cls == 2 ? 3 : cls == 0 && io == IO_R2R ? 2 : cls; }
template <int SET, class F>
__device__ __forceinline__ void radix_case(int r, F &&f) {
  switch (r) {
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    default:
      if constexpr (SET != 3) {
        if (r == 3) f(std::integral_constant<int, 3>{});
        else if (r == 5) f(std::integral_constant<int, 5>{});
        else if (r == 6) f(std::integral_constant<int, 6>{});
        else if (r == 7) f(std::integral_constant<int, 7>{});
        else if (r == 9) f(std::integral_constant<int, 9>{});
      }
      if constexpr (SET < 2) {
        if (r == 15) f(std::integral_constant<int, 15>{});
        else if (r == 16) f(std::integral_constant<int, 16>{});
      }
      if constexpr (SET == 1) {
        if (r == 11) f(std::integral_constant<int, 11>{});
        else if (r == 13) f(std::integral_constant<int, 13>{});
        else if (r == 17) f(std::integral_constant<int, 17>{});
      }
  }
}

// w / n and w % n by the reciprocal, corrected to exact (0 <= w < 2^23).
__device__ __forceinline__ void est_divmod(int w, int n, float inv, int &q, int &r) {
  q = (int)((float)w * inv);
  r = w - q * n;
  if (r < 0) {
    --q;
    r += n;
  } else if (r >= n) {
    ++q;
    r -= n;
  }
}

// (a + b + c + d) sqrt(1/2), rounded once: the split of an odd DCT-IV, whose four
// roundings would make it less accurate than the general kernel's longer DFT
// (27 points in FP32 9.7e-8 there, 1.00e-7 with them).
template <typename T>
__device__ __forceinline__ T sum4_sqrt_half(T a, T b, T c, T d) {
  constexpr double h = kRootCos[kRootOff[8] + 1];
  if constexpr (sizeof(T) == 4) {
    return (T)((((double)a + (double)b) + ((double)c + (double)d)) * h);
  } else {
    T err = T(0);
    auto sum = [&](T x, T y) __attribute__((always_inline)) {  // Knuth's two-sum
      const T s = x + y, v = s - x;
      err += (x - (s - v)) + (y - v);
      return s;
    };
    const T s = sum(sum(a, b), sum(c, d));
    constexpr double l = -4.833646656726457e-17;
    return s * h + (s * l + err * h);
  }
}

// VAR = 1: c2c columns in the packed order of an exchange; real-to-real stages of
// types 4 and 8 of even length; 2: those of odd length (in one kernel with the others
// they cost registers and scratch: FP32 columns of 300 points 202 -> 245 us).
template <typename T, int IO, bool LINES, int CLS, int VAR>
__device__ __forceinline__ void mixed_tile(DescPtr d, const void *in, void *out, int conj,
                                           long long tile) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  cpx<T> *lds = reinterpret_cast<cpx<T> *>(lds_raw);
  constexpr bool R2R = IO == IO_R2R;
  constexpr int SET = mx_set(CLS, IO);
  constexpr int LO = R2R && sizeof(T) == 8 ? 2 : 1;  // form of the butterflies (codelets.h)
  // real-to-real stages: the transform, and which of its ends are not the
  // points of the DFT themselves (types 3 and 7 merge the line into a Hermitian
  // sequence first, 2, 6 and odd-length 4, 8 split the result afterwards);
  // types 4 and 8 of even length take one real line per tile column, those of odd
  // length a DFT of as many points of signed permuted ones (odd48)
  const int type = R2R ? d->dtt : 0, Lr = R2R ? d->dtt_len : 0;
  constexpr bool PK = VAR == 1 && !R2R, single = VAR == 1 && R2R, odd48 = VAR == 2;
  const bool pre = VAR == 0 && (type == 3 || type == 7), post = odd48 || (VAR == 0 && (type == 2 || type == 6));
  const bool alt = type >= 6;  // 6, 7, 8: signs (-1)^j
  const bool PAIRED = IO == IO_R2C || IO == IO_C2R || (R2R && !single);
  constexpr bool CHIRP = CLS == 2;
  // n: points of a line; m: points of the transform
  const int m = d->n, n = CHIRP ? d->nblue : m, TX = d->TX, lg = d->log2TX, rows = d->rows, np = d->npass;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const long long tiles0 = d->tiles0;
  const long long c1 = tile / tiles0;
  const long long c0b = (tile - c1 * tiles0) * TX;
  int t, row;
  if constexpr (LINES) {
    est_divmod(tid, rows, 1.0f / (float)rows, t, row);
  } else {
    t = tid & (TX - 1);
    row = tid >> lg;
  }
  const long long c0 = c0b + t;
  const long long ca = PAIRED ? 2 * c0 : c0;  // first (real) column of the lane
  // lanes without a column or a row take no butterfly (they keep to the barriers)
  if (t >= TX || row >= rows || ca >= (PAIRED ? d->C0r : d->C0)) row = 1 << 24;
  const bool two = !PAIRED || ca + 1 < d->C0r;
  const bool full = 2 * (c0b + TX) <= d->C0r;  // every pair of the tile is whole
  const long long sji = d->in_sj, sjo = d->out_sj;
  const long long f0 = R2R ? d->dtt_first : 0;
  const long long in_base = (IO == IO_R2C || R2R ? ca : c0) * d->in_s0 + c1 * d->in_s1 + f0 * sji +
                            (IO == IO_C2C && !LINES ? (c0 >> d->bsh) * d->in_b0 : 0);
  const long long out_base = (IO == IO_C2R || R2R ? ca : c0) * d->out_s0 + c1 * d->out_s1 + f0 * sjo +
                             (IO == IO_C2C && !LINES ? (c0 >> d->bsh) * d->out_b0 : 0);
  // LDS: [point][column] for strided columns; [line][point] with one pad
  // point in 17 for contiguous lines, whose first exchange writes with the
  // stride of the first radix
  const int ldt = d->ldt;
  auto A = [&](int j, int tt) __attribute__((always_inline)) {
    return LINES ? j + (j >> 4) + tt * ldt : (j << lg) + tt;
  };

  const bool adj_in = !LINES && d->in_s0 == 1, adj_out = !LINES && d->out_s0 == 1;

  // ---- pieces of a pass ------------------------------------------------------
  // values of the first pass (and whole transforms of one pass) from HBM
  auto load = [&](auto rc, auto &v) __attribute__((always_inline)) {
    constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
    const int nb = m / R;
    const long long step = (long long)nb * sji;
    if constexpr (R2R) {
      // point J of the sequence that the DFT takes, types 1, 2, even 4, 5, 6, even 8:
      // +- x_src (zero where src is no point of the line), src piecewise linear in J:
      //   2, 6  x_0 x_2 x_4 ... x_5 x_3 x_1       1  e[j] = e[n-j] = x_j
      //   5     e[j+1] = -e[n-j-1] = x_j
      // and (x_2J, x_{L-1-2J}) for even 4, 8.  All loads first, then the signs.
      const int h = (type == 2 || type == 6) ? (n + 1) / 2 : type == 1 ? Lr : type == 5 ? Lr + 1 : n;
      const int a1 = (type == 2 || type == 6 || single) ? 2 : 1, b1 = type == 5 ? -1 : 0;
      const int a2 = (type == 2 || type == 6) ? -2 : -1, b2 = (type == 2 || type == 6) ? 2 * n - 1 : type == 1 ? n : n - 1;
      auto src = [&](int J) __attribute__((always_inline)) {
        return J < h ? a1 * J + b1 : (CHIRP && J >= n ? -1 : a2 * J + b2);
      };
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = row + q * rows;
        if (b < nb) {
          auto off = [&](int s) __attribute__((always_inline)) {
            const int j = src(b + s * nb);
            return in_base + (long long)((unsigned)j < (unsigned)Lr ? j : 0) * sji;
          };
          if (odd48) {
            // J = 2j + 1 mod L for one j.  With r = 2j + 1 in [0, 2L), the residue of r
            // mod 8 decides between x_j and x_{L-1-j} and the sign (get_dtt4_odd_table)
            auto at = [&](int s, bool &neg) __attribute__((always_inline)) {
              const int J = b + s * nb, r = J & 1 ? J : J + n;
              const int j = r & 2 ? n - 1 - (r >> 1) : r >> 1;
              neg = (((r >> 2) ^ ((r & n) >> 1) ^ (alt ? j : 0)) & 1) != 0;
              return !CHIRP || J < n ? j : -1;
            };
#pragma unroll
            for (int s = 0; s < R; ++s) {
              bool neg;
              const int j = at(s, neg);
              const long long o = in_base + (long long)(j < 0 ? 0 : j) * sji;
              if (adj_in && full) {
                v[q * R + s] = gload_pair<T>(in, o);
              } else {
                v[q * R + s].x = gload_r<T>(in, o);
                v[q * R + s].y = two ? gload_r<T>(in, o + d->in_s0) : T(0);
              }
            }
#pragma unroll
            for (int s = 0; s < R; ++s) {
              bool neg;
              if (at(s, neg) < 0) v[q * R + s] = cpx<T>{T(0), T(0)};
              else if (neg) v[q * R + s] = cpx<T>{-v[q * R + s].x, -v[q * R + s].y};
            }
            continue;
          }
          if (single) {
#pragma unroll
            for (int s = 0; s < R; ++s) {
              v[q * R + s].x = gload_r<T>(in, off(s));
              const int j = src(b + s * nb);
              v[q * R + s].y = gload_r<T>(in, in_base + (long long)((unsigned)j < (unsigned)Lr ? 2 * n - 1 - j : 0) * sji);
            }
          } else if (adj_in && full) {
#pragma unroll
            for (int s = 0; s < R; ++s) v[q * R + s] = gload_pair<T>(in, off(s));
          } else {
#pragma unroll
            for (int s = 0; s < R; ++s) {
              v[q * R + s].x = gload_r<T>(in, off(s));
              v[q * R + s].y = two ? gload_r<T>(in, off(s) + d->in_s0) : T(0);
            }
          }
          if (single) {
            if (alt) {
#pragma unroll
              for (int s = 0; s < R; ++s) v[q * R + s].y = -v[q * R + s].y;
            }
          } else if (alt) {
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (src(b + s * nb) & 1) v[q * R + s] = cpx<T>{-v[q * R + s].x, -v[q * R + s].y};
          } else if (type == 5) {
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (b + s * nb >= h) v[q * R + s] = cpx<T>{-v[q * R + s].x, -v[q * R + s].y};
          }
          if (CHIRP || type == 5) {
#pragma unroll
            for (int s = 0; s < R; ++s)
              if ((unsigned)src(b + s * nb) >= (unsigned)Lr) v[q * R + s] = cpx<T>{T(0), T(0)};
          }
          if (single) {  // exp(-i pi (4J+1) / 4L)
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (b + s * nb < n) v[q * R + s] = cmul(v[q * R + s], gload<T>(d->dtw, b + s * nb));
          }
        }
      }
    } else if constexpr (IO == IO_R2C) {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = row + q * rows;
        if (b < nb) {
          const long long o = in_base + (long long)b * sji;
          if (adj_in && full) {  // adjacent columns: one load per pair
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (!CHIRP || b + s * nb < n) v[q * R + s] = gload_pair<T>(in, o + s * step);
          } else {
#pragma unroll
            for (int s = 0; s < R; ++s) {
              if (CHIRP && b + s * nb >= n) continue;
              v[q * R + s].x = gload_r<T>(in, o + s * step);
              v[q * R + s].y = two ? gload_r<T>(in, o + s * step + d->in_s0) : T(0);
            }
          }
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = row + q * rows;
        if (b < nb) {
          const long long o = in_base + (long long)b * sji;
          if (PK && d->packj >= 2) {
#pragma unroll
            for (int s0 = 0; s0 < R; s0 += 4) {  // four table reads, then their loads
              long long off[4];
#pragma unroll
              for (int s = s0; s < R && s < s0 + 4; ++s)
                if (!CHIRP || b + s * nb < n) off[s - s0] = packj_offset(d, b + s * nb, c1);
#pragma unroll
              for (int s = s0; s < R && s < s0 + 4; ++s)
                if (!CHIRP || b + s * nb < n) v[q * R + s] = gload<T>(in, o + s * step + off[s - s0]);
            }
          } else {
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (!CHIRP || b + s * nb < n) v[q * R + s] = gload<T>(in, o + s * step);
          }
          if (conj) {
#pragma unroll
            for (int s = 0; s < R; ++s) v[q * R + s].y = -v[q * R + s].y;
          }
        }
      }
    }
  };
  // outputs j = b + s * (n / R) of the last pass to HBM
  auto store = [&](auto rc, auto &v) __attribute__((always_inline)) {
    constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
    const int nb = m / R;
    const long long step = (long long)nb * sjo;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int b = row + q * rows;
      if (b < nb) {
        const long long o = out_base + (long long)b * sjo;
        if constexpr (R2R) {  // types 1, 3, 4 and 8 (even length), 5, 7
          if (single) {  // u_k = V_k exp(-i pi k / L): Y_2k = 2 Re u_k, Y_{L-1-2k} = -2 Im u_k
#pragma unroll
            for (int s = 0; s < R; ++s) {
              const int J = b + s * nb;
              if (CHIRP && J >= n) continue;
              const cpx<T> u = cmul(v[q * R + s], gload<T>(d->dtw, n + J));
              const int ie = alt ? 2 * n - 1 - 2 * J : 2 * J, io = 2 * n - 1 - ie;
              gstore_r<T>(out, out_base + (long long)ie * sjo, T(2) * u.x);
              gstore_r<T>(out, out_base + (long long)io * sjo, T(-2) * u.y);
            }
          } else {
            // 3, 7: z = conj(result) = v_a + i v_b, y_2n = v_n, y_{2n+1} = v_{L-1-n};
            // 1: the real DFT of an even extension; 5: the imaginary one of an odd
#pragma unroll
            for (int s = 0; s < R; ++s) {
              const int J = b + s * nb;
              const cpx<T> z = v[q * R + s];
              const int kk = pre ? (2 * J < n ? 2 * J : 2 * n - 1 - 2 * J) : type == 1 ? J : J - 1;
              cpx<T> y = pre ? cconj(z) : type == 1 ? z : cpx<T>{-z.y, z.x};
              if (pre && alt && (kk & 1)) y = cpx<T>{-y.x, -y.y};
              if ((unsigned)kk >= (unsigned)Lr || (CHIRP && J >= n)) continue;
              const long long ok = out_base + (long long)kk * sjo;
              if (adj_out && full) {
                gstore_pair<T>(out, ok, y);
              } else {
                gstore_r<T>(out, ok, y.x);
                if (two) gstore_r<T>(out, ok + d->out_s0, y.y);
              }
            }
          }
        } else if constexpr (IO == IO_C2R) {  // the pre-phase stored conj(Z): z = conj(result)
#pragma unroll
          for (int s = 0; s < R; ++s) {
            if (CHIRP && b + s * nb >= n) continue;
            if (adj_out && full) {
              gstore_pair<T>(out, o + s * step, cconj(v[q * R + s]));
            } else {
              gstore_r<T>(out, o + s * step, v[q * R + s].x);
              if (two) gstore_r<T>(out, o + s * step + d->out_s0, -v[q * R + s].y);
            }
          }
        } else {
          if (conj) {
#pragma unroll
            for (int s = 0; s < R; ++s) v[q * R + s].y = -v[q * R + s].y;
          }
          if (PK && (d->packj & 1)) {
            const long long *tab = d->packj == 1 ? d->pack : d->pack2;
#pragma unroll
            for (int s0 = 0; s0 < R; s0 += 4) {
              long long off[4];
#pragma unroll
              for (int s = s0; s < R && s < s0 + 4; ++s)
                if (!CHIRP || b + s * nb < n) off[s - s0] = packj_offset_in(tab, b + s * nb, c1);
#pragma unroll
              for (int s = s0; s < R && s < s0 + 4; ++s)
                if (!CHIRP || b + s * nb < n) gstore<T>(out, o + s * step + off[s - s0], v[q * R + s]);
            }
          } else {
#pragma unroll
            for (int s = 0; s < R; ++s)
              if (!CHIRP || b + s * nb < n) gstore<T>(out, o + s * step, v[q * R + s]);
          }
        }
      }
    }
  };
  // inputs j = b + s * (n / R) of a pass from LDS
  auto lds_read = [&](auto rc, auto &v, int nb, int row_, int rows_, int t_) __attribute__((always_inline)) {
    constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int b = row_ + q * rows_;
      if (b < nb) {
#pragma unroll
        for (int s = 0; s < R; ++s) v[q * R + s] = lds[A(b + s * nb, t_)];
      }
    }
  };

  // the points outside [dtt_first, dtt_first + dtt_len) of a real-to-real stage
  auto copy_through = [&]() __attribute__((always_inline)) {
    if constexpr (R2R) {
      const int npt = d->dtt_n - Lr, fi = d->dtt_first, per = single ? 1 : 2;
      for (int w = tid; w < TX * npt; w += nthr) {
        const int tt = LINES ? w / npt : w & (TX - 1), i = LINES ? w % npt : w >> lg;
        const int k = i < fi ? i : i + Lr;
        for (int e = 0; e < per; ++e) {
          const long long cc = per * (c0b + tt) + e;
          if (cc < d->C0r)
            gstore_r<T>(out, cc * d->out_s0 + c1 * d->out_s1 + (long long)k * d->out_sj,
                        gload_r<T>(in, cc * d->in_s0 + c1 * d->in_s1 + (long long)k * d->in_sj));
        }
      }
    }
  };

  // ---- inputs ------------------------------------------------------------------
  const int nh = d->nh;
  const float inv_nh = 1.0f / (float)nh;
  if constexpr (IO == IO_C2R) {
    // conj(Z) of the merged half spectra, all n points, into LDS; the loads
    // of four points of both columns are in flight together
    constexpr int U = 4;
    const int total = TX * nh;
    for (int w0 = tid; w0 < total; w0 += U * nthr) {
      cpx<T> a[U], b[U];
      int kk[U], tt[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int w = w0 + u * nthr;
        kk[u] = -1;
        tt[u] = 0;
        a[u] = b[u] = cpx<T>{T(0), T(0)};
        if (w < total) {
          if constexpr (LINES) {
            est_divmod(w, nh, inv_nh, tt[u], kk[u]);
          } else {
            tt[u] = w & (TX - 1);
            kk[u] = w >> lg;
          }
          const long long cc = 2 * (c0b + tt[u]);
          long long ia = cc * d->in_s0 + c1 * d->in_s1 + (long long)kk[u] * sji;
          long long ib = ia + d->in_s0;
          if (LINES && d->npack) {  // receive-buffer order, or the blocked layout
            ia = pack_index(d, kk[u], cc + c1 * d->pack_l1);
            ib = pack_index(d, kk[u], cc + 1 + c1 * d->pack_l1);
          }
          if (cc < d->C0r) a[u] = gload<T>(in, ia);
          if (cc + 1 < d->C0r) b[u] = gload<T>(in, ib);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = kk[u];
        if (k >= 0) {
          if (k == 0 || 2 * k == n) a[u].y = b[u].y = T(0);
          lds[A(k, tt[u])] = cpx<T>{a[u].x - b[u].y, -(a[u].y + b[u].x)};
          if (k > 0 && 2 * k < n) lds[A(n - k, tt[u])] = cpx<T>{a[u].x + b[u].y, a[u].y - b[u].x};
        }
      }
    }
    __syncthreads();
  }

  if constexpr (R2R) {
    if (pre) {
      // conj(Z_j) = w_j conj(u_j), u_j = (Xa_j + Xb_{L-j}, Xb_j - Xa_{L-j}) (X_L =
      // 0; DST-III reads X backwards), for j and L - j together
      constexpr int U = 4;
      const int nj = n / 2 + 1, total = TX * nj;
      const float inv_nj = 1.0f / (float)nj;
      for (int w0 = tid; w0 < total; w0 += U * nthr) {
        cpx<T> a[U], b[U];
        int jj[U], tt[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int w = w0 + u * nthr;
          jj[u] = -1;
          tt[u] = 0;
          a[u] = b[u] = cpx<T>{T(0), T(0)};
          if (w < total) {
            if constexpr (LINES) {
              est_divmod(w, nj, inv_nj, tt[u], jj[u]);
            } else {
              tt[u] = w & (TX - 1);
              jj[u] = w >> lg;
            }
            const int j = jj[u];
            const long long cc = 2 * (c0b + tt[u]);
            const long long base = cc * d->in_s0 + c1 * d->in_s1 + f0 * sji;
            const long long o1 = base + (long long)(alt ? n - 1 - j : j) * sji;
            const long long o2 = base + (long long)(alt ? j - 1 : n - j) * sji;
            if (cc + 1 < d->C0r && adj_in) {
              a[u] = gload_pair<T>(in, o1);
              if (j > 0) b[u] = gload_pair<T>(in, o2);
            } else if (cc < d->C0r) {
              a[u].x = gload_r<T>(in, o1);
              if (j > 0) b[u].x = gload_r<T>(in, o2);
              if (cc + 1 < d->C0r) {
                a[u].y = gload_r<T>(in, o1 + d->in_s0);
                if (j > 0) b[u].y = gload_r<T>(in, o2 + d->in_s0);
              }
            }
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int j = jj[u], jm = n - j;
          if (j >= 0) {
            const cpx<T> cs = gload<T>(d->dtw, j);
            const T ux = a[u].x + b[u].y, uy = a[u].y - b[u].x;
            lds[A(j, tt[u])] = cpx<T>{cs.x * ux - cs.y * uy, -(cs.x * uy + cs.y * ux)};
            if (j > 0 && j < jm) {
              const cpx<T> cm = gload<T>(d->dtw, jm);
              const T vx = b[u].x + a[u].y, vy = b[u].y - a[u].x;
              lds[A(jm, tt[u])] = cpx<T>{cm.x * vx - cm.y * vy, -(cm.x * vy + cm.y * vx)};
            }
          }
        }
      }
      __syncthreads();
    }
  }

  // ---- passes --------------------------------------------------------------------
  const bool HBM_IN = IO != IO_C2R && !pre, HBM_OUT = IO != IO_R2C && !post;
  if constexpr (!CHIRP) {
    if (HBM_IN && HBM_OUT && np == 1) {
      radix_case<SET>(d->pass[0].r, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
        cpx<T> v[NB * R];
        load(rc, v);
        if (row < rows) dft<T, R, LO>(v);  // n == R: one butterfly per column
        store(rc, v);
      });
      copy_through();
      return;
    }
  }
  const void *tw = d->tw;
  if constexpr (CHIRP) {
    // y_k = c_k sum_j (x_j c_j) w_{k-j}: the first transform runs its passes
    // from the last to the first by decimation in frequency, the inverse one
    // (as conj(DFT(conj(.)))) from the first to the last by decimation in time,
    // all in place: a lane writes a butterfly back to the points it read.  So
    // an exchange takes one barrier, both transforms share one twiddle table,
    // and the spectrum stays in the first one's order (bhat is stored in it, over
    // m).
    // The twiddles of a pass are loaded before its points.
    const int tw_last = d->pass[np - 1].tw_off;
    radix_case<SET>(d->pass[np - 1].r, [&](auto rc) __attribute__((always_inline)) {
      constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
      const int nb = m / R;
      cpx<T> v[NB * R];
#pragma unroll
      for (int i = 0; i < NB * R; ++i) v[i] = cpx<T>{T(0), T(0)};
      if (HBM_IN) {
        load(rc, v);
      } else {  // the merged spectra, already in LDS
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int b = row + q * rows;
#pragma unroll
          for (int s = 0; s < R; ++s)
            if (b < nb && b + s * nb < n) v[q * R + s] = lds[A(b + s * nb, t)];
        }
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = row + q * rows;
        if (b < nb) {
#pragma unroll
          for (int s = 0; s < R; ++s)
            if (b + s * nb < n) v[q * R + s] = cmul(v[q * R + s], gload<T>(d->chirp, b + s * nb));
          dft<T, R, LO>(&v[q * R]);
          lds[A(b, t)] = v[q * R];
#pragma unroll
          for (int s = 1; s < R; ++s)
            lds[A(b + s * nb, t)] = cmul(v[q * R + s], gload<T>(tw, tw_last + b * (R - 1) + (s - 1)));
        }
      }
    });
    __syncthreads();
    for (int w = 0; w < 2 * np - 3; ++w) {
      // w < np - 2: passes np - 2 .. 1 of the first transform; w = np - 2:
      // pass 0 of both; then passes 1 .. np - 2 of the second
      const int turn = np - 2, p = w < turn ? turn - w : w - turn;
      const int L = d->pass[p].L, tw_off = d->pass[p].tw_off;
      const float invL = d->pass[p].invL;
      // a zero the compiler cannot see through: it would otherwise hoist the
      // loop-invariant address parts of every radix's case out of the loop,
      // far more than there are registers
      int zero;
      asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
      const int m_ = m + zero, rows_ = rows + zero, row_ = row + zero, t_ = t + zero;
      radix_case<SET>(d->pass[p].r, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
        const int nb = m_ / R;
        if (w == turn) {
#pragma unroll
          for (int q = 0; q < NB; ++q) {
            const int b = row_ + q * rows_;
            if (b < nb) {
              cpx<T> v[R], f[R];
#pragma unroll
              for (int s = 0; s < R; ++s) f[s] = gload<T>(d->bhat, b * R + s);
#pragma unroll
              for (int s = 0; s < R; ++s) v[s] = lds[A(b * R + s, t_)];
              dft<T, R, LO>(v);
#pragma unroll
              for (int s = 0; s < R; ++s) v[s] = cconj(cmul(v[s], f[s]));
              dft<T, R, LO>(v);
#pragma unroll
              for (int s = 0; s < R; ++s) lds[A(b * R + s, t_)] = v[s];
            }
          }
        } else {
#pragma unroll
          for (int q = 0; q < NB; ++q) {
            const int b = row_ + q * rows_;
            if (b < nb) {
              int g, k;
              est_divmod(b, L, invL, g, k);
              const int jb = g * L * R + k;
              cpx<T> v[R], f[R];
#pragma unroll
              for (int s = 1; s < R; ++s) f[s] = gload<T>(tw, tw_off + k * (R - 1) + (s - 1));
#pragma unroll
              for (int s = 0; s < R; ++s) v[s] = lds[A(jb + s * L, t_)];
              if (w > turn) {
#pragma unroll
                for (int s = 1; s < R; ++s) v[s] = cmul(v[s], f[s]);
              }
              dft<T, R, LO>(v);
              if (w < turn) {
#pragma unroll
                for (int s = 1; s < R; ++s) v[s] = cmul(v[s], f[s]);
              }
#pragma unroll
              for (int s = 0; s < R; ++s) lds[A(jb + s * L, t_)] = v[s];
            }
          }
        }
      });
      __syncthreads();
    }
    radix_case<SET>(d->pass[np - 1].r, [&](auto rc) __attribute__((always_inline)) {
      constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
      const int nb = m / R;
      cpx<T> v[NB * R];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = row + q * rows;
        if (b < nb) {
          cpx<T> f[R];
#pragma unroll
          for (int s = 1; s < R; ++s) f[s] = gload<T>(tw, tw_last + b * (R - 1) + (s - 1));
          v[q * R] = lds[A(b, t)];
#pragma unroll
          for (int s = 1; s < R; ++s) v[q * R + s] = cmul(lds[A(b + s * nb, t)], f[s]);
          dft<T, R, LO>(&v[q * R]);
#pragma unroll
          for (int s = 0; s < R; ++s)
            if (b + s * nb < n) {
              v[q * R + s] = cmul(cconj(v[q * R + s]), gload<T>(d->chirp, b + s * nb));
              if (!HBM_OUT) lds[A(b + s * nb, t)] = v[q * R + s];
            }
        }
      }
      if (HBM_OUT) store(rc, v);
    });
    if (!HBM_OUT) __syncthreads();
  } else {
    int p = 0;
    if (HBM_IN) {
      radix_case<SET>(d->pass[0].r, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
        const int nb = n / R;
        cpx<T> v[NB * R];
        load(rc, v);
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int b = row + q * rows;
          if (b < nb) {
            dft<T, R, LO>(&v[q * R]);
#pragma unroll
            for (int s = 0; s < R; ++s) lds[A(b * R + s, t)] = v[q * R + s];
          }
        }
      });
      __syncthreads();
      p = 1;
    }
    const int pmid = HBM_OUT ? np - 1 : np;
    for (; p < pmid; ++p) {
      const int L = d->pass[p].L, tw_off = d->pass[p].tw_off;
      const float invL = d->pass[p].invL;
      // (an opaque zero, as above: 430 bytes of spill per lane without it)
      int zero;
      asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
      const int n_ = n + zero, rows_ = rows + zero, row_ = row + zero, t_ = t + zero;
      radix_case<SET>(d->pass[p].r, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
        const int nb = n_ / R;
        cpx<T> v[NB * R];
        lds_read(rc, v, nb, row_, rows_, t_);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int b = row_ + q * rows_;
          if (b < nb) {
            int g, k;
            est_divmod(b, L, invL, g, k);
            if (L > 1) {
#pragma unroll
              for (int s = 1; s < R; ++s)
                v[q * R + s] = cmul(v[q * R + s], gload<T>(tw, tw_off + k * (R - 1) + (s - 1)));
            }
            dft<T, R, LO>(&v[q * R]);
            const int jb = g * L * R + k;
#pragma unroll
            for (int s = 0; s < R; ++s) lds[A(jb + s * L, t_)] = v[q * R + s];
          }
        }
      });
      __syncthreads();
    }
    if (HBM_OUT) {
      const int tw_off = d->pass[np - 1].tw_off;
      radix_case<SET>(d->pass[np - 1].r, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value, NB = mx_nb(R, sizeof(T), LINES);
        const int nb = n / R;  // = L: every butterfly of the last pass is its own k
        cpx<T> v[NB * R];
        lds_read(rc, v, nb, row, rows, t);
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const int b = row + q * rows;
          if (b < nb) {
            if (nb > 1) {
#pragma unroll
              for (int s = 1; s < R; ++s)
                v[q * R + s] = cmul(v[q * R + s], gload<T>(tw, tw_off + b * (R - 1) + (s - 1)));
            }
            dft<T, R, LO>(&v[q * R]);
          }
        }
        store(rc, v);
      });
    }
  }
  if constexpr (R2R) {
    if (post) {
      // Z in LDS.  Types 2, 6: Y_k = 2 Re(w_q V_q) of each line of the pair, V
      // split from Z as in a real-to-complex transform, q = k (DCT-II) or
      // L-1-k (DST-II).  Types 4, 8 of odd L: the same with q = (2k+1) / 8 mod L and
      // w_k = (+-1 -+ i) / sqrt 2, the signs from the table
      const int total = TX * Lr;
      const float inv_L = 1.0f / (float)Lr;
      for (int w = tid; w < total; w += nthr) {
        int tt, k;
        if constexpr (LINES) {
          est_divmod(w, Lr, inv_L, tt, k);
        } else {
          tt = w & (TX - 1);
          k = w >> lg;
        }
        const long long cc = 2 * (c0b + tt);
        if (cc < d->C0r) {
          const int kk = alt ? Lr - 1 - k : k;
          int q = kk;
          if (odd48) {
            int turns;
            est_divmod(d->dtt_q0 + kk * d->dtt_q1, Lr, inv_L, turns, q);
          }
          const cpx<T> zk = lds[A(q, tt)], zm = lds[A(q == 0 ? 0 : n - q, tt)];
          const cpx<T> cs = gload<T>(d->dtw, kk);
          const cpx<T> y = odd48 ? cpx<T>{sum4_sqrt_half(cs.x * zk.x, cs.x * zm.x, cs.y * zk.y, -cs.y * zm.y),
                                          sum4_sqrt_half(cs.x * zk.y, cs.x * zm.y, cs.y * zm.x, -cs.y * zk.x)}
                                 : cpx<T>{cs.x * (zk.x + zm.x) + cs.y * (zk.y - zm.y),
                                          cs.x * (zk.y + zm.y) + cs.y * (zm.x - zk.x)};
          const long long o = cc * d->out_s0 + c1 * d->out_s1 + (f0 + k) * sjo;
          if (cc + 1 < d->C0r && adj_out) {
            gstore_pair<T>(out, o, y);
          } else {
            gstore_r<T>(out, o, y.x);
            if (cc + 1 < d->C0r) gstore_r<T>(out, o + d->out_s0, y.y);
          }
        }
      }
    }
    copy_through();
  } else if constexpr (IO == IO_R2C) {
    // A[k] = (Z[k] + conj Z[n-k]) / 2 and B[k] = (Z[k] - conj Z[n-k]) / (2i)
    const T half = T(0.5);
    const int total = TX * nh;
    for (int w = tid; w < total; w += nthr) {
      int tt, k;
      if constexpr (LINES) {
        est_divmod(w, nh, inv_nh, tt, k);
      } else {
        tt = w & (TX - 1);
        k = w >> lg;
      }
      const long long cc = 2 * (c0b + tt);
      if (cc < d->C0r) {
        const cpx<T> zk = lds[A(k, tt)], zm = lds[A(k == 0 ? 0 : n - k, tt)];
        long long oa = cc * d->out_s0 + c1 * d->out_s1 + (long long)k * sjo;
        long long ob = oa + d->out_s0;
        if (LINES && d->npack) {  // send-buffer order, or the blocked layout
          oa = pack_index(d, k, cc + c1 * d->pack_l1);
          ob = pack_index(d, k, cc + 1 + c1 * d->pack_l1);
        }
        gstore<T>(out, oa, cpx<T>{(zk.x + zm.x) * half, (zk.y - zm.y) * half});
        if (cc + 1 < d->C0r) gstore<T>(out, ob, cpx<T>{(zk.y + zm.y) * half, (zm.x - zk.x) * half});
      }
    }
  }
}

// Threads a workgroup may have, and the waves per SIMD its registers leave
// room for.
constexpr int mx_threads(int cls) { return cls == 1 ? 512 : 1024; }
template <typename T>
constexpr int mx_wpe(int cls, int io) {
  if (io == IO_R2R && cls == 1 && sizeof(T) == 8) return 3;  // (143-point DCT-I lines 580 -> 415 us)
  return cls != 1 ? (sizeof(T) == 8 ? 4 : 6) : (sizeof(T) == 8 ? 2 : 4);
}

// One grid (ng = 0: the stage of the arguments), or the tiles of several
// grids (the same code, so that a batch's results equal the plans' own).
template <typename T, int IO, bool LINES, int CLS, int VAR>
__global__ void __launch_bounds__(mx_threads(CLS)) __attribute__((amdgpu_waves_per_eu(mx_wpe<T>(CLS, IO))))
    mixed_kernel(const AxisDesc *__restrict__ d, const void *in, void *out, int conj,
                 const MultiGroup *__restrict__ g, int ng, long long tiles) {
  long long it = xcd_tile((long long)blockIdx.x + (long long)blockIdx.y * gridDim.x, tiles);
  if (it >= tiles) return;  // whole block, before any barrier
  if (ng > 0) {
    const int gi = find_multi_group(g, ng, it);
    d = g[gi].d;
    in = g[gi].in;
    out = g[gi].out;
    conj = g[gi].conj;
    it -= g[gi].tile0;
  }
  mixed_tile<T, IO, LINES, CLS, VAR>(desc_ptr(d), in, out, conj, it);
}

template <typename T, int IO, bool LINES, int CLS, int VAR>
int mixed_go(const AxisDesc *dd, const AxisIo &io, const MultiGroup *g, int ng, long long tiles, int nt,
             size_t lds, hipStream_t st) {
  const long long nb = xcd_grid(tiles);
  if (nb <= 0) return D2DHIP_SUCCESS;
  const long long gx = nb < (1LL << 20) ? nb : (1LL << 20);
  const long long gy = (nb + gx - 1) / gx;
  if (gy > 65535) return set_error(D2DHIP_ERR_UNSUPPORTED, "axis stage has too many tiles");
  hipLaunchKernelGGL((mixed_kernel<T, IO, LINES, CLS, VAR>), dim3((unsigned)gx, (unsigned)gy), dim3(nt), lds,
                     st, dd, io.in, io.out, io.conj, g, ng, tiles);
  return hip_check(hipGetLastError(), "mixed_kernel launch");
}

template <typename T, int IO, bool LINES, int CLS>
int mixed_launch(const AxisDesc *dd, const AxisDesc &h, const AxisIo &io, hipStream_t st) {
  const long long tiles = (long long)h.tiles0 * h.C1;
  auto go = [&](auto var) {
    return mixed_go<T, IO, LINES, CLS, decltype(var)::value>(dd, io, nullptr, 0, tiles, h.nthreads, h.lds_bytes, st);
  };
  if constexpr (IO == IO_C2C && !LINES) {
    if (h.packj) return go(std::integral_constant<int, 1>{});
  }
  if constexpr (IO == IO_R2R) {
    if (h.dtt == 4 || h.dtt == 8)
      return h.dtt_len % 2 ? go(std::integral_constant<int, 2>{}) : go(std::integral_constant<int, 1>{});
  }
  return go(std::integral_constant<int, 0>{});
}

template <typename T, int IO, bool LINES, int CLS>
int mixed_launch_multi(const MultiGroup *g, int ng, long long tiles, int nt, size_t lds, hipStream_t st) {
  const AxisIo io = {nullptr, nullptr, 0};
  return mixed_go<T, IO, LINES, CLS, 0>(nullptr, io, g, ng, tiles, nt, lds, st);
}

constexpr int kMaxLds = 160 * 1024;

// The LDS limit of the kernels, raised once per device (a bit of `done`).
template <typename T, int IO, bool LINES, int CLS>
hipError_t mixed_prepare() {
  static std::atomic<unsigned long long> done{0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
  if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
  auto raise = [&](auto var) {
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void *)mixed_kernel<T, IO, LINES, CLS, decltype(var)::value>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
  };
  raise(std::integral_constant<int, 0>{});
  if constexpr ((IO == IO_C2C && !LINES) || IO == IO_R2R) raise(std::integral_constant<int, 1>{});
  if constexpr (IO == IO_R2R) raise(std::integral_constant<int, 2>{});
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}

template <typename T, int IO, bool LINES, int CLS>
FastVariant mixed_variant(const char *name) {
  FastVariant v;
  v.rb = (int)sizeof(T);
  v.io = IO;
  v.lines = LINES ? 1 : 0;
  v.mixed = 1 + CLS;
  v.launch = &mixed_launch<T, IO, LINES, CLS>;
  v.prepare = &mixed_prepare<T, IO, LINES, CLS>;
  v.launch_multi = &mixed_launch_multi<T, IO, LINES, CLS>;
  v.prepare_multi = &mixed_prepare<T, IO, LINES, CLS>;
  v.name = name;
  return v;
}

// c2c, r2c, c2r and r2r of one class, strided columns and contiguous lines
#define D2D_MIXED_ALL(T, CLS, TAG)                                            \
  mixed_variant<T, IO_C2C, false, CLS>(#T " mixed c2c" TAG),                  \
      mixed_variant<T, IO_C2C, true, CLS>(#T " mixed c2c" TAG),               \
      mixed_variant<T, IO_R2C, false, CLS>(#T " mixed r2c" TAG),              \
      mixed_variant<T, IO_R2C, true, CLS>(#T " mixed r2c" TAG),               \
      mixed_variant<T, IO_C2R, false, CLS>(#T " mixed c2r" TAG),              \
      mixed_variant<T, IO_C2R, true, CLS>(#T " mixed c2r" TAG),               \
      mixed_variant<T, IO_R2R, false, CLS>(#T " mixed dct" TAG),              \
      mixed_variant<T, IO_R2R, true, CLS>(#T " mixed dct" TAG)

}  // namespace

}  // namespace d2dhip
