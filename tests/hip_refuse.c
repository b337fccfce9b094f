/* hipMalloc that refuses requests of lo to hi bytes and passes the others on,
 * for tests of what happens when device memory runs out.  Loaded with
 * RTLD_GLOBAL before the library. */
#include <dlfcn.h>
#include <stddef.h>

static size_t lo = 1, hi = 0;
static int refused = 0;

void refuse(size_t a, size_t b) { lo = a; hi = b; }
int refusals(void) { return refused; }

int hipMalloc(void **p, size_t n)
{
	static int (*real)(void **, size_t);
	if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipMalloc");
	if (n >= lo && n <= hi) {
		refused++;
		return 2; /* hipErrorOutOfMemory */
	}
	return real ? real(p, n) : 2;
}
