/* hipMalloc with a limit, for tests of calls that meet a full device: loaded
 * with RTLD_GLOBAL before the library under test, whose hipMalloc then resolves
 * here. Sizes from the limit up, and the sizes listed, fail as the runtime's own
 * call does when memory is short; the rest goes to the runtime. */
#include <dlfcn.h>
#include <stddef.h>

static size_t limit = (size_t)-1;
static size_t listed[8];
static int refusals = 0;

void alloc_limit(size_t bytes) { limit = bytes; }
void alloc_refuse(int slot, size_t bytes) { listed[slot & 7] = bytes; }
int alloc_refusals(void) { return refusals; }

int hipMalloc(void** ptr, size_t bytes) {
  static int (*real)(void**, size_t) = NULL;
  if (!real) {
    void* rt = dlopen("libamdhip64.so.7", RTLD_NOW);
    real = rt ? (int (*)(void**, size_t))dlsym(rt, "hipMalloc") : NULL;
  }
  int full = !real || bytes >= limit;
  for (int k = 0; k < 8; ++k) full |= bytes > 0 && bytes == listed[k];
  if (full) {
    ++refusals;
    *ptr = NULL;
    return 2; /* hipErrorOutOfMemory */
  }
  return real(ptr, bytes);
}
