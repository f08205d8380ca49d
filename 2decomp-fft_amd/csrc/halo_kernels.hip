// halo_kernels.hip -- halo cells of one rank's pencil (update_halo,
// halo_exchange; src/halo.f90, src/halo_common.f90,
// src/halo_exchange_{x,y,z}_body.f90).
//
// A halo array has the pencil's local extents plus `level` cells on both
// sides of the two distributed axes (y, z for an x-pencil; x, z for a
// y-pencil; x, y for a z-pencil).  update_halo copies the pencil into its
// interior, then halo_exchange fills the halo slabs axis by axis: for an
// x-pencil y then z, for a y-pencil x then z, for a z-pencil x then y.  Each
// step moves, over the whole extent of the other two axes (their halo cells
// included), the `level` interior slabs next to each side into the
// neighbour's opposite halo.  At one rank the neighbour along an axis is
// the rank itself when that axis is periodic (MPI_CART_SHIFT of a periodic
// communicator of size 1) and none otherwise, so the low halo takes the
// last `level` interior slabs, the high halo the first ones, and a
// non-periodic axis leaves its halo cells as they were.  Doing the axes in
// the reference's order with the same slab extents gives the same corner
// cells.
#include <hip/hip_runtime.h>

#include "internal.h"

namespace d2dhip {

// (a vector, not a struct: arrays of a struct went to scratch memory, 80 bytes a
// lane)
using H16 = unsigned long long __attribute__((ext_vector_type(2)));

// 16 bytes of adjacent cells, aligned as one cell is.
template <typename E>
struct Cells {
  static constexpr int V = 16 / (int)sizeof(E);
  using Q = E __attribute__((ext_vector_type(V), aligned(sizeof(E))));
};
template <>
struct Cells<H16> {
  static constexpr int V = 1;
  using Q = H16;
};

// Extents s of the pencil and n of the halo array, offset o of the pencil in
// it, and whether an axis's halo cells are filled (w).
struct HaloArgs {
  int s[3], n[3], o[3], w[3];
};

// update_halo in one pass over the halo array.  Folding every filled axis into
// the pencil gives the cell that the axis-by-axis exchange would have copied:
// a cell of the pencil, or, where the other axis is not periodic and the cell
// lies in its halo, a cell of the array that nothing writes.  2^lg threads
// share a row (i fastest): 16 bytes of the pencil's part each, two loads (of whole
// 16-byte cells: one) ahead of their stores, and one cell of the two ends, loaded with
// them; so a row that the threads fill takes one round whatever its ends.
//
// Bound by HBM, against a copy of the pencil by rows and a launch per filled axis,
// all axes periodic, level 2, 512^3: FP64 x-pencil 366 -> 343 us (6.4 TB/s of cells
// read and written once), y-pencil 403 -> 344, FP32 z-pencil 311 -> 176; complex FP64
// 256^3 y-pencil 100 -> 88.  Small arrays are bound by the launch (64^3 13.7 -> 8.4 us),
// short rows by the lanes that a block per row left idle (27 x 700 x 600 152 -> 24
// us).  Without periodic axes there is one copy on either side: level with it but for
// complex FP64, which is 2 to 6 % slower on rows that leave threads idle.
template <typename E>
__global__ void __launch_bounds__(256) halo_update_kernel(const E *__restrict__ in, E *arr, HaloArgs a,
                                                          int lg) {
  using Q = typename Cells<E>::Q;
  constexpr int V = Cells<E>::V, U = V == 1 ? 1 : 2;
  const int lanes = 1 << lg, lane = threadIdx.x & (lanes - 1), n1 = a.n[0], s1 = a.s[0], o1 = a.o[0];
  const int nv = s1 / V, ne = n1 - s1;
  const long long rows = (long long)a.n[1] * a.n[2], step = (long long)gridDim.x * (256 >> lg);
  for (long long row = (long long)blockIdx.x * (256 >> lg) + (threadIdx.x >> lg); row < rows; row += step) {
    const int k = rows >> 31 ? (int)(row / a.n[1]) : (int)((unsigned)row / (unsigned)a.n[1]);
    int c[2] = {(int)(row - (long long)k * a.n[1]) - a.o[1], k - a.o[2]};
    bool moved = false, open = false;  // open: in the halo of an axis that is not filled
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int n = a.s[d + 1];
      if (c[d] >= 0 && c[d] < n) continue;
      if (a.w[d + 1]) {
        c[d] += c[d] < 0 ? n : -n;
        moved = true;
      } else {
        open = true;
      }
    }
    // cell i of the source row is arow[i] or, within the pencil, src[i - o1]
    const E *arow = arr + ((long long)(c[1] + a.o[2]) * a.n[1] + c[0] + a.o[1]) * n1;
    const E *src = open ? arow + o1 : in + ((long long)c[1] * a.s[1] + c[0]) * s1;
    E *dst = arr + row * n1;
    const bool copy = moved || !open;
    // end cell e (those below the pencil's part, then those above) and where it
    // comes from, if it is written
    auto end_source = [&](int e) -> const E * {
      if (e >= ne) return nullptr;
      if (a.w[0]) return src + (e < o1 ? e + s1 - o1 : e - o1);
      return moved ? arow + (e < o1 ? e : e + s1) : nullptr;
    };
    const E *from = end_source(lane);
    E end{};
    if (from) end = *from;
    if (copy) {
      for (int b = lane; b < nv; b += U * lanes) {
        Q v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (b + u * lanes < nv) v[u] = *reinterpret_cast<const Q *>(src + (b + u * lanes) * V);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (b + u * lanes < nv) *reinterpret_cast<Q *>(dst + o1 + (b + u * lanes) * V) = v[u];
      }
      for (int i = nv * V + lane; i < s1; i += lanes) dst[o1 + i] = src[i];
    }
    if (from) dst[lane < o1 ? lane : lane + s1] = end;
    for (int e = lane + lanes; e < ne; e += lanes)
      if (const E *f = end_source(e)) dst[e < o1 ? e : e + s1] = *f;
  }
}

// The 2 * level halo slabs of axis d of arr (n1, n2, n3) from the slabs on
// the other side of the interior.
template <typename E>
__global__ void __launch_bounds__(256) halo_wrap_kernel(E *arr, int n1, int n2, int n3, int d,
                                                        int level) {
  const int m1 = d == 0 ? 2 * level : n1, m2 = d == 1 ? 2 * level : n2;
  const int m3 = d == 2 ? 2 * level : n3;
  const int nd = d == 0 ? n1 : (d == 1 ? n2 : n3);
  const long long total = (long long)m1 * m2 * m3;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    const long long r = t / m1;
    int c[3];
    c[0] = (int)(t - r * m1);
    c[2] = (int)(r / m2);
    c[1] = (int)(r - (long long)c[2] * m2);
    const int q = c[d];
    int s[3] = {c[0], c[1], c[2]};
    if (q < level) {  // low halo <- last interior slabs
      s[d] = nd - 2 * level + q;
    } else {  // high halo <- first interior slabs
      c[d] = nd - level + (q - level);
      s[d] = q;
    }
    arr[c[0] + (long long)c[1] * n1 + (long long)c[2] * n1 * n2] =
        arr[s[0] + (long long)s[1] * n1 + (long long)s[2] * n1 * n2];
  }
}

static long long halo_grid(long long total) {
  long long g = (total + 255) / 256;
  return g < 1 ? 1 : (g > 65536 ? 65536 : g);
}

template <typename E>
static int halo_run(const void *in, void *arr, const int s[3], const int n[3], const int o[3],
                    const int order[2], const int wrap[2], int level, hipStream_t st) {
  if (in && s[0] > 0 && s[1] > 0 && s[2] > 0) {  // the exchange included
    HaloArgs a = {};
    for (int e = 0; e < 3; ++e) {
      a.s[e] = s[e];
      a.n[e] = n[e];
      a.o[e] = o[e];
    }
    for (int q = 0; q < 2; ++q) a.w[order[q]] = wrap[q];
    // The power of two of threads to a row that fills them best: as many as the
    // pencil's row has 16-byte groups, or half of that where the last round would be
    // less than an eighth full.  us with 256 / 128 / 64 / 32 threads, level 2: FP64
    // rows of 512 cells 344 / 381 / 380 / 402, FP32 ones 216 / 171 / 191 / 189, of 150
    // 102 / 56 / 35 / 24; complex FP64 rows of 150 132 / 112 / 117 / 133.
    const int nv = (s[0] + Cells<E>::V - 1) / Cells<E>::V;
    int lg = 0;
    while (lg < 8 && (2LL << lg) <= nv) ++lg;
    if (lg && (nv - 1) % (1 << lg) + 1 <= (1 << lg) / 8) --lg;
    const long long per = 256 >> lg, g = ((long long)n[1] * n[2] + per - 1) / per;
    hipLaunchKernelGGL(halo_update_kernel<E>, dim3((unsigned)(g < (1LL << 20) ? g : 1LL << 20)), dim3(256), 0, st,
                       (const E *)in, (E *)arr, a, lg);
    return hip_check(hipGetLastError(), "halo kernel launch");
  }
  for (int a = 0; a < 2; ++a) {
    if (!wrap[a] || level == 0) continue;
    const int d = order[a];
    long long total = 2LL * level;
    for (int e = 0; e < 3; ++e)
      if (e != d) total *= n[e];
    if (total > 0)
      hipLaunchKernelGGL(halo_wrap_kernel<E>, dim3((unsigned)halo_grid(total)), dim3(256), 0, st,
                         (E *)arr, n[0], n[1], n[2], d, level);
  }
  return hip_check(hipGetLastError(), "halo kernel launch");
}

int launch_halo(int esize, const void *in, void *arr, int s1, int s2, int s3, int level,
                int ipencil, const int periodic[3], hipStream_t st) {
  // halo axes and their order (src/halo_exchange_{x,y,z}_body.f90)
  int order[2];
  if (ipencil == 1) {
    order[0] = 1;
    order[1] = 2;
  } else if (ipencil == 2) {
    order[0] = 0;
    order[1] = 2;
  } else {
    order[0] = 0;
    order[1] = 1;
  }
  const int s[3] = {s1, s2, s3};
  int n[3] = {s1, s2, s3}, o[3] = {0, 0, 0};
  int wrap[2];
  for (int a = 0; a < 2; ++a) {
    n[order[a]] += 2 * level;
    o[order[a]] = level;
    wrap[a] = periodic[order[a]] ? 1 : 0;
  }
  switch (esize) {
    case 4: return halo_run<unsigned int>(in, arr, s, n, o, order, wrap, level, st);
    case 8: return halo_run<unsigned long long>(in, arr, s, n, o, order, wrap, level, st);
    default: return halo_run<H16>(in, arr, s, n, o, order, wrap, level, st);
  }
}

}  // namespace d2dhip
