// The emulated wave (rt.cpp).
#pragma once

#include "hip/hip_runtime.h"

#undef asm
#undef volatile
#include <stdio.h>

namespace emu {
void watch(void *lds, size_t bytes);      // the memory whose accesses are checked
void leave_out(void *p, size_t bytes);    // ... but for this part
// runs f(arg) in n lanes; `seed` picks the order in which they run
void run(int n, unsigned seed, long limit, void (*f)(void *), void *arg);
int report(FILE *f);  // kinds of unordered exchange seen
}  // namespace emu
