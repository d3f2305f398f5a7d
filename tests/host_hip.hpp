// Stand-in for the device built-ins that the library's headers name, for host
// builds of its sources by a plain C++ compiler (tests/host_memory.cpp).
#pragma once
#include <stdint.h>
static inline unsigned int __umulhi(unsigned int a, unsigned int b) { return (unsigned int)(((uint64_t)a * b) >> 32); }
