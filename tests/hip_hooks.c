/* HIP entry points put in front of the runtime's for a test's child process
 * (loaded with RTLD_GLOBAL before the library under test): each counts its
 * calls and passes them on, except where the environment asks for
 *   HOOK_NO_PINNED  pinned allocations that fail as for want of memory
 *   HOOK_DEFER      copies to the device that read their source in stream
 *                   order and not before the call returns, as copies from
 *                   pinned memory may */
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

static void *next(const char *name) {
  static void *lib;
  if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW);
  return dlsym(lib, name);
}

enum { N_PINNED, N_MALLOC, N_MEMCPY, N_MEMSET, N_COUNT };
static long count[N_COUNT];
long hook_count(int which) { return count[which]; }

int hipHostMalloc(void **p, size_t n, unsigned flags) {
  int (*f)(void **, size_t, unsigned) = next("hipHostMalloc");
  count[N_PINNED]++;
  if (getenv("HOOK_NO_PINNED")) {
    f(NULL, n, flags); /* refused by the runtime, which keeps the error */
    return 2;
  }
  return f(p, n, flags);
}

int hipMalloc(void **p, size_t n) {
  int (*f)(void **, size_t) = next("hipMalloc");
  count[N_MALLOC]++;
  return f(p, n);
}

int hipMemcpy(void *d, const void *s, size_t n, int kind) {
  int (*f)(void *, const void *, size_t, int) = next("hipMemcpy");
  count[N_MEMCPY]++;
  return f(d, s, n, kind);
}

int hipMemset(void *d, int v, size_t n) {
  int (*f)(void *, int, size_t) = next("hipMemset");
  count[N_MEMSET]++;
  return f(d, v, n);
}

struct late { void *to; const void *from; size_t n; };
static void read_source(void *p) {
  struct late *l = p;
  memcpy(l->to, l->from, l->n);
  free(l);
}

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream) {
  int (*f)(void *, const void *, size_t, int, void *) = next("hipMemcpyAsync");
  int (*pinned)(void **, size_t, unsigned) = next("hipHostMalloc");
  int (*host)(void *, void (*)(void *), void *) = next("hipLaunchHostFunc");
  struct late *l;
  if (kind != 1 || !getenv("HOOK_DEFER")) return f(d, s, n, kind, stream);
  l = malloc(sizeof *l);
  l->from = s;
  l->n = n;
  if (!l || pinned(&l->to, n, 0)) return 2; /* kept until the process ends */
  void *to = l->to;
  int e = host(stream, read_source, l);
  return e ? e : f(d, to, n, kind, stream);
}
