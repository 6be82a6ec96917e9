// Prints brick_extent's record for every line "first own total threads cap" of
// the standard input.
#include <stdio.h>

#include "../../moldy_amd/csrc/mdk_brick.h"

int main() {
  int a0, own, total, threads, cap;
  while (scanf("%d %d %d %d %d", &a0, &own, &total, &threads, &cap) == 5) {
    const int4 r = brick_extent(a0, own, total, threads, cap);
    printf("%d %d %d\n", r.x, r.y, r.z);
  }
  return 0;
}
