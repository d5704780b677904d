/* hipMalloc for a process that loads this library before the runtime's
 * callers: once armed, `count` calls after the next `skip` ones find no memory. */
#include <stddef.h>

enum { out_of_memory = 2 }; /* hipErrorOutOfMemory */

static int (*real)(void**, size_t);
static long skip, count, refused, calls;

void refuse_real(void* f) { real = (int (*)(void**, size_t))f; }

void refuse_arm(long s, long n)
{
  skip = s;
  count = n;
  refused = calls = 0;
}

long refuse_refused(void) { return refused; }
long refuse_calls(void) { return calls; }

int hipMalloc(void** p, size_t bytes)
{
  const long k = calls++;
  if (k >= skip && refused < count) {
    ++refused;
    return out_of_memory;
  }
  return real(p, bytes);
}
