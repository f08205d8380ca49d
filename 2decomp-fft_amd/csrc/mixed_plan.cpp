// mixed_plan.cpp -- the tile and radix schedule that a kernel of any length
// (mixed_impl.h) takes for a length, and the list of those kernels.
#include <algorithm>

#include "mixed_impl.h"

namespace d2dhip {

namespace {

constexpr int kRadices[4][15] = {{16, 15, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2},
                                 {17, 16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2},
                                 {12, 10, 9, 8, 7, 6, 5, 4, 3, 2},
                                 {12, 10, 8, 4, 2}};

// Least rows per column of a schedule (every pass within its butterflies per
// lane), and the work of its passes in lanes, idle ones counted.
int least_rows(int n, const std::vector<int> &r, const FastVariant &v) {
  int rows = 1;
  for (int x : r) rows = std::max(rows, (n / x + mx_nb(x, v.rb, v.lines) - 1) / mx_nb(x, v.rb, v.lines));
  return rows;
}
double sched_cost(int n, int rows, const std::vector<int> &r) {
  double c = 0;
  for (int x : r) c += (double)rows * ((n / x + rows - 1) / rows) * x / n;
  return c + (double)r.size();
}

// Schedules of n over non-increasing radices, at most 5 passes; keeps the
// cheapest.
void search(int n, int left, int from, int set, const FastVariant &v, std::vector<int> &cur, std::vector<int> &best, int &rows,
            double &cost) {
  if (left == 1) {
    // the least rows, or up to half as many again where they divide a pass evenly,
    // within a workgroup's threads
    const int r0 = least_rows(n, cur, v);
    auto take = [&](int r) {
      if (r < r0 || r > r0 + r0 / 2 || r > mx_threads(v.mixed - 1)) return;
      const double c = sched_cost(n, r, cur);
      if (c < cost - 1e-9 || (c < cost + 1e-9 && best == cur && r < rows)) {
        cost = c;
        best = cur;
        rows = r;
      }
    };
    take(r0);
    for (int x : cur)
      for (int q = 1; q <= 4; ++q) take((n / x + q - 1) / q);
    return;
  }
  if (cur.size() == 5) return;
  for (int i = from; i < 15 && kRadices[set][i]; ++i) {
    const int x = kRadices[set][i];
    if (left % x) continue;
    cur.push_back(x);
    search(n, left / x, i, set, v, cur, best, rows, cost);
    cur.pop_back();
  }
}

// Passes of the cheapest schedule of m.
int passes(int m, const FastVariant &v) {
  std::vector<int> cur, best;
  int rows = 0;
  double cost = 1e30;
  search(m, m, 0, mx_set(v.mixed - 1, v.io), v, cur, best, rows, cost);
  return rows ? (int)best.size() : 99;
}

// A class takes the lengths that the lighter one does not, up to six points
// per thread of a block (the fewest a lane may have in a pass) and one
// column per tile.
bool takes_length(const FastVariant &v, int n) {
  const int cls = v.mixed - 1;
  int left = n;
  for (int x : {2, 3, 5, 7}) while (left > 0 && left % x == 0) left /= x;
  const bool smooth = left == 1;
  for (int x : {11, 13, 17}) while (left > 0 && left % x == 0) left /= x;
  if (n < 2 || cls != (smooth ? 0 : left == 1 ? 1 : 2)) return false;
  const int m = mixed_length(v, n);
  return m <= 6 * mx_threads(cls) && (size_t)m * 17 / 16 * 2 * v.rb + 64 <= (size_t)kMaxLds;
}

}  // namespace

// A length of the kernel's class that some schedule fits into a workgroup; the
// others keep the general kernel.
bool mixed_runs(const FastVariant &v, int n) {
  std::vector<int> radices;
  AxisShape s;
  return mixed_shape(v, n, 1, radices, s);
}

// Length of the transform: n itself, or for a chirp the least power of two m >=
// 2n - 1, or 15/16 of it where that saves a pass (960 = 12 10 8 for 1024 = 8 8 8 2:
// 382-point columns 1.6 -> 1.9 TB/s in FP64, 1.0 -> 1.2 in FP32).  The rounding errors
// of a convolution grow as the square root of (2n - 1) / m: 3/4 of the power of
// two (768 for 382 points, 2.0 TB/s) is up to 12 % further from the exact
// transform than the general kernel, which takes the power of two.  (120 for
// 128 would save a pass too, and be 2 to 7 % further off in FP64.)  Lengths whose
// power of two does not fit a workgroup take the least 2^k times 3, 5 or 9; they
// run on the general kernel unless chosen (mixed_short).
int mixed_length(const FastVariant &v, int n) {
  if (v.mixed != 3) return n;
  int m = 16;
  while (m < 2 * n - 1) m *= 2;
  if (m <= 6 * mx_threads(2)) {
    const int q = m / 16 * 15;
    return m >= 512 && q >= 2 * n - 1 && passes(q, v) < passes(m, v) ? q : m;
  }
  int best = m;
  for (int f : {3, 5, 9}) {
    m = f;
    while (m < 2 * n - 1) m *= 2;
    best = std::min(best, m);
  }
  return best;
}

bool mixed_short(const FastVariant &v, int n) {
  if (v.mixed != 3) return false;
  int m = 16;
  while (m < 2 * n - 1) m *= 2;
  return m > 6 * mx_threads(2);
}

// Columns: the widest rows (256 bytes at most) that leave room for two
// workgroups on a CU, and more columns while the block stays below 256
// threads and 40 KB.  FP64 columns, 16 / 8 / 4 wide, TB/s: 270 points 5.0 /
// 4.7 / 4.7, 512 points 4.7 / 4.7 / 4.2, 720 points 3.7 / 3.7 / 3.9, 1024
// points 3.7 / 3.8 / 4.1.  Lines: as many as make 256 threads (64 to 512
// threads lie within 5 %).
bool mixed_shape(const FastVariant &v, int n, long long C0, std::vector<int> &radices, AxisShape &s) {
  const int cls = v.mixed - 1, cb = 2 * v.rb;
  if (!takes_length(v, n)) return false;
  n = mixed_length(v, n);
  std::vector<int> cur;
  double cost = 1e30;
  int rows = 0;
  search(n, n, 0, mx_set(cls, v.io), v, cur, radices, rows, cost);
  if (!rows) return false;
  if (v.lines)  // an odd first radix: its stride spreads the first exchange over the banks
    std::stable_partition(radices.begin(), radices.end(), [](int x) { return x % 2 == 1; });
  const int ldt = v.lines ? ((n - 1) + ((n - 1) >> 4) + 1) | 1 : n;
  const int maxt = mx_threads(cls);
  auto lds = [&](int tx) { return (size_t)tx * ldt * cb; };
  int tx = v.lines ? 1 : (cls == 2 ? 128 : 256) / cb;
  while (tx > 1 && (tx * rows > maxt || lds(tx) > (size_t)kMaxLds / 2)) tx >>= 1;
  if (tx * rows > maxt || lds(tx) > (size_t)kMaxLds) return false;
  while (tx < C0 && tx < 64 && 2 * tx * rows <= 256 && lds(2 * tx) <= 40 * 1024) tx *= 2;
  // chirps wait on their barriers: blocks of a multiple of four waves load the
  // four SIMDs alike (m = 768, 4 columns: 1.96 TB/s with 512 threads, 1.85
  // with 384)
  if (cls == 2 && tx * rows > 256)
    while (tx * rows % 256 && tx * (rows + 1) <= maxt) ++rows;
  s.TX = tx;
  s.rows = rows;
  s.nthreads = (tx * rows + 63) / 64 * 64;
  s.lds_bytes = lds(tx);
  s.ldj = v.lines ? 1 : tx;
  s.ldt = v.lines ? ldt : 1;
  return true;
}

// compiled in mixed_f64.hip, mixed_f64_chirp.hip, mixed_f32.hip and
// mixed_f32_chirp.hip
std::vector<FastVariant> mixed_variants_f64();
std::vector<FastVariant> mixed_variants_f64_chirp();
std::vector<FastVariant> mixed_variants_f32();
std::vector<FastVariant> mixed_variants_f32_chirp();

std::vector<FastVariant> mixed_variants() {
  std::vector<FastVariant> v;
  for (auto part : {mixed_variants_f64, mixed_variants_f64_chirp, mixed_variants_f32,
                    mixed_variants_f32_chirp}) {
    const std::vector<FastVariant> q = part();
    v.insert(v.end(), q.begin(), q.end());
  }
  return v;
}

}  // namespace d2dhip
