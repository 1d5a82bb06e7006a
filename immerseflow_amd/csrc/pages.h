// Host memory helpers (no device code).
#pragma once
#include <cstddef>

namespace iff {

// Fault in the pages of n bytes at p for writing; what they hold stays.  One
// locked read-modify-write a page, which faults once, as a write (a load and a
// store would fault a fresh page twice).
inline void touch_pages(void *p, size_t n)
{
    char *c = (char *)p;
    auto touch = [](char *q) { asm volatile("lock orb $0, %0" : "+m"(*q) : : "cc"); };
    for (size_t b = 0; b < n; b += 4096) touch(c + b);
    if (n > 0) touch(c + n - 1);
}

}  // namespace iff
