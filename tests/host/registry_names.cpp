// Prints "lines name" of every kernel in the library's registry.
#include <cstdio>

#include "fast_kernels.h"

int main() {
  for (const d2dhip::FastVariant &v : d2dhip::fast_registry()) std::printf("%d %s\n", v.lines, v.name);
  return 0;
}
