// Every length that a kernel of any length says it runs has a launch shape,
// and the shape keeps the kernel's limits.  Prints "name n what" for each
// length that does not, then "checked <count>"; with arguments "rb io lines n"
// prints the shape of that length.
#include <cstdio>
#include <cstdlib>

#include "fast_kernels.h"

using namespace d2dhip;

static const char *check(const FastVariant &v, int n, long long C0) {
  std::vector<int> r;
  AxisShape s;
  if (!mixed_shape(v, n, C0, r, s)) return "no shape";
  const int m = mixed_length(v, n);
  long long prod = 1;
  for (int x : r) {
    prod *= x;
    // a lane takes 10 values of a pass, 20 of FP32 columns, at most four
    // butterflies and at least one
    const int room = (v.rb == 4 && !v.lines ? 20 : 10) / x;
    const int per = room < 1 ? 1 : room > 4 ? 4 : room;
    if ((long long)s.rows * per < m / x) return "too few rows";
  }
  if (prod != m || (m == n) != (v.mixed != 3) || (m != n && m < 2 * n - 1)) return "radices";
  if ((int)r.size() > kMaxPass) return "passes";
  if (s.nthreads < s.TX * s.rows || s.nthreads > (v.mixed == 2 ? 512 : 1024) || s.nthreads % 64) return "threads";
  const int last = v.lines ? (s.TX - 1) * s.ldt + (m - 1) + ((m - 1) >> 4) : (m - 1) * s.ldj + s.TX - 1;
  if (s.lds_bytes > 160 * 1024 || (size_t)(last + 1) * 2 * v.rb > s.lds_bytes) return "LDS";
  return nullptr;
}

int main(int argc, char **argv) {
  long long checked = 0;
  for (const FastVariant &v : fast_registry()) {
    if (!v.mixed) continue;
    if (argc == 5) {
      const int n = std::atoi(argv[4]);
      if (v.rb == std::atoi(argv[1]) && v.io == std::atoi(argv[2]) && v.lines == std::atoi(argv[3]) && mixed_runs(v, n))
        std::printf("%s %d runs\n", v.name, n);
      continue;
    }
    for (int n = 1; n <= 7000; ++n) {
      if (!mixed_runs(v, n)) continue;
      for (long long C0 : {1ll, 3ll, 1000ll}) {
        const char *e = check(v, n, C0);
        if (e) std::printf("%s lines=%d n=%d C0=%lld: %s\n", v.name, v.lines, n, C0, e);
        ++checked;
      }
    }
  }
  if (argc != 5) std::printf("checked %lld\n", checked);
  return 0;
}
