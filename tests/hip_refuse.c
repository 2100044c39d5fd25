/* hipMalloc and hipFree of the real runtime with a limit on the bytes held:
 * what goes beyond it is refused by the host, before the runtime sees it. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static struct {
  void *p;
  size_t n;
} held[4096];
static size_t used = 0, limit = (size_t)-1;

static void *real(const char *name)
{
  static void *lib = NULL;
  if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL); /* the one the library links */
  return lib ? dlsym(lib, name) : NULL;
}

void hh_limit(size_t bytes) { limit = bytes; }
size_t hh_used(void) { return used; }

int hipMalloc(void **p, size_t n)
{
  int (*f)(void **, size_t) = (int (*)(void **, size_t))real("hipMalloc");
  int rc, i;
  *p = NULL;
  if (!f) return 1;                  /* hipErrorInvalidValue */
  if (used + n > limit) return 2;    /* hipErrorOutOfMemory */
  rc = f(p, n);
  if (rc) return rc;
  for (i = 0; i < 4096; ++i)
    if (!held[i].p) {
      held[i].p = *p;
      held[i].n = n;
      used += n;
      break;
    }
  return 0;
}

int hipFree(void *p)
{
  int (*f)(void *) = (int (*)(void *))real("hipFree");
  int i;
  for (i = 0; p && i < 4096; ++i)
    if (held[i].p == p) {
      used -= held[i].n;
      held[i].p = NULL;
      break;
    }
  return f ? f(p) : 1;
}
