/* Loaded with RTLD_GLOBAL before libfa_rocm.so, its hipMalloc comes first:
 * while fail_from is not 0, requests of at least that many bytes find no
 * memory (hipErrorOutOfMemory); the others, and all while it is 0, are the
 * runtime's. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

size_t fail_from = 0;
int failed = 0;

int hipMalloc(void** ptr, size_t size) {
  static int (*real)(void**, size_t);
  if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipMalloc");
  if (fail_from && size >= fail_from) {
    failed++;
    return 2;
  }
  return real(ptr, size);
}
