// build_weight_list (imageworsener_amd/csrc/iw_tables.cpp) when memory or
// threads run out, built by tests/test_tables_memory.py.  Operator new is
// replaced: it counts, records the largest request and fails from a chosen one
// on.  Arguments: the scenario.  Exit status 0: all checks passed.
#include "iw_tables.h"
#include "iw_ctx.h"

#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

static std::atomic<long> g_count{0}, g_fail_at{-1}, g_fail_len{0};
static std::atomic<size_t> g_largest{0};

void *operator new(size_t n)
{
	const long k = g_count++;
	size_t m = g_largest.load();
	while (n > m && !g_largest.compare_exchange_weak(m, n)) {}
	const long at = g_fail_at.load();
	if (at >= 0 && k >= at && k < at + g_fail_len.load()) throw std::bad_alloc();
	void *p = malloc(n ? n : 1);
	if (!p) throw std::bad_alloc();
	return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

// What iw_tables.cpp takes from the rest of the library.
double iwx_x_to_linear(double v, const struct iw_csdescr *) { return v; }
double iwx_linear_to_x(double v, const struct iw_csdescr *) { return v; }

static iwamd_resize resize(int family, double blur, int in, int out)
{
	iwamd_resize r;
	memset(&r, 0, sizeof(r));
	r.family = family;
	r.blur_factor = blur;
	r.param1 = 3.0;
	r.num_in = in;
	r.num_out = out;
	r.out_true_size = out;
	r.edge_policy = IW_EDGE_POLICY_STANDARD;
	return r;
}

// Every allocation of a list built by several threads fails in turn, alone and
// with all that follow it: the caller gets the list or std::bad_alloc.
static int threads()
{
	const iwamd_resize r = resize(IW_RESIZETYPE_LANCZOS, 1.0, 4000, 1000);
	const iwx::WeightList want = iwx::build_weight_list(r, 0, 0.0);
	g_count = 0;
	iwx::build_weight_list(r, 0, 0.0);
	const long n = g_count;
	int failed = 0;
	for (long len : {1L, 1000000L})
		for (long k = 0; k < n + 4; k++) {
			g_count = 0;
			g_fail_len = len;
			g_fail_at = k;
			try {
				const iwx::WeightList got = iwx::build_weight_list(r, 0, 0.0);
				g_fail_at = -1;
				if (got.w != want.w || got.src != want.src || got.start != want.start) return 1;
			} catch (const std::bad_alloc &) {
				g_fail_at = -1;
				failed++;
			}
		}
	printf("%ld allocations, %d lists refused\n", n, failed);
	return failed >= n ? 0 : 2;
}

// Blurs up to the widest: what is asked for at once is no more than the list
// itself could come to (its entries lie inside the image).
static int reserve()
{
	for (double blur : {1.0, 30.0, 1000.0, 10000.0})
		for (int out : {1, 40, 1000}) {
			const iwamd_resize r = resize(IW_RESIZETYPE_LANCZOS, blur, 1000, out);
			g_largest = 0;
			const iwx::WeightList l = iwx::build_weight_list(r, 0, 0.0);
			const size_t most = sizeof(double) * (size_t)out * (1000 + 2);
			printf("blur %g, %d outputs: %zu entries, largest request %zu\n", blur, out, l.w.size(), g_largest.load());
			if (g_largest > most) return 1;
		}
	return 0;
}

int main(int argc, char **argv)
{
	if (argc == 2 && !strcmp(argv[1], "threads")) return threads();
	if (argc == 2 && !strcmp(argv[1], "reserve")) return reserve();
	return 3;
}
