/* A HIP runtime of host memory, for tests of the library's host side where
 * there is no GPU: device memory is calloc'd, copies are memcpy, kernel
 * launches are logged by name and grid and do nothing, events read the times
 * a test sets.  Loaded with RTLD_GLOBAL before the library, so that the
 * library's HIP calls bind here (tests/test_host_side.py).  mock_*: what a
 * test sets and reads. */
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned int x, y, z; } dim3;
enum { SUCCESS = 0, OUT_OF_MEMORY = 2, UNKNOWN = 999 };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;

/* ---- controls ---- */
static size_t fail_lo = 1, fail_hi = 0;
static int sync_errors = 0, copy_errors = 0;
static int streams_made = 0, streams_freed = 0;
static double (*event_ms)(int) = NULL;
static size_t symbol_bytes = 0;

void mock_fail_malloc(size_t lo, size_t hi) { fail_lo = lo; fail_hi = hi; }
void mock_sync_errors(int n) { sync_errors = n; }
void mock_copy_errors(int n) { copy_errors = n; }
int mock_streams_made(void) { return streams_made; }
int mock_streams_freed(void) { return streams_freed; }
void mock_event_ms(double (*f)(int)) { event_ms = f; }
size_t mock_symbol_bytes(void) { return symbol_bytes; }

/* ---- kernels: host stub -> name, and the log of launches ---- */
#define MAXK 4096
static const void *kptr[MAXK];
static char *kname[MAXK];
static int nk = 0;
#define MAXLOG 65536
static struct { const char *name; dim3 grid, block; size_t shmem; void *arg[2]; int n; } lg[MAXLOG];
static int nlog = 0;

int mock_launches(void) { return nlog; }
void mock_clear_log(void) { nlog = 0; }
const char *mock_launch(int i, unsigned int *grid3)
{
	memcpy(grid3, &lg[i].grid, sizeof(dim3));
	return lg[i].name;
}
/* The work items of a band_kernel launch (plan, first row), and their number. */
const void *mock_launch_items(int i) { return lg[i].arg[1]; }
int mock_launch_count(int i) { return lg[i].n; }

void **__hipRegisterFatBinary(const void *data) { static void *h; (void)data; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *host, char *dev, const char *name, unsigned int lim, void *a, void *b,
	void *c, void *d, int *w)
{
	(void)h; (void)dev; (void)lim; (void)a; (void)b; (void)c; (void)d; (void)w;
	if (nk < MAXK) {
		kptr[nk] = host;
		kname[nk++] = strdup(name);
	}
}
static const void *vptr[64];
static size_t vsize[64];
static int nv = 0;
void __hipRegisterVar(void **h, void *var, char *host, char *dev, int ext, size_t size, int constant, int global)
{
	(void)h; (void)host; (void)dev; (void)ext; (void)constant; (void)global;
	if (nv < 64) {
		vptr[nv] = var;
		vsize[nv++] = size;
	}
}

static __thread struct { dim3 grid, block; size_t shmem; void *st; } cfg;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, void *st)
{
	cfg.grid = grid;
	cfg.block = block;
	cfg.shmem = shmem;
	cfg.st = st;
	return SUCCESS;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, void **st)
{
	*grid = cfg.grid;
	*block = cfg.block;
	*shmem = cfg.shmem;
	*st = cfg.st;
	return SUCCESS;
}
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shmem, void *st)
{
	(void)st;
	pthread_mutex_lock(&mu);
	for (int i = 0; i < nk; i++)
		if (kptr[i] == f && nlog < MAXLOG) {
			lg[nlog].name = kname[i];
			lg[nlog].grid = grid;
			lg[nlog].block = block;
			lg[nlog].arg[0] = lg[nlog].arg[1] = NULL;
			lg[nlog].n = 0;
			if (strstr(kname[i], "11band_kernel")) {
				for (int k = 0; k < 2; k++) lg[nlog].arg[k] = *(void **)args[k];
				lg[nlog].n = *(int *)args[2];
			}
			lg[nlog++].shmem = shmem;
			break;
		}
	pthread_mutex_unlock(&mu);
	return SUCCESS;
}

/* ---- the runtime ---- */
int hipGetDeviceCount(int *n) { *n = 1; return SUCCESS; }
int hipGetDevice(int *d) { *d = 0; return SUCCESS; }
int hipSetDevice(int d) { return d == 0 ? SUCCESS : UNKNOWN; }
int hipDeviceGetAttribute(int *v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return SUCCESS; }
int hipDeviceSynchronize(void) { return SUCCESS; }
int hipGetLastError(void) { return SUCCESS; }
const char *hipGetErrorString(int e) { return e ? "mock error" : "no error"; }
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f; (void)a; (void)v; return SUCCESS; }
int hipMalloc(void **p, size_t n)
{
	if (n >= fail_lo && n <= fail_hi) return OUT_OF_MEMORY;
	*p = calloc(1, n ? n : 1);
	return *p ? SUCCESS : OUT_OF_MEMORY;
}
int hipFree(void *p) { free(p); return SUCCESS; }
int hipHostMalloc(void **p, size_t n, unsigned int f) { (void)f; return hipMalloc(p, n); }
int hipHostFree(void *p) { free(p); return SUCCESS; }
int hipHostGetDevicePointer(void **d, void *h, unsigned int f) { (void)f; *d = h; return SUCCESS; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return SUCCESS; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st)
{
	(void)kind; (void)st;
	if (copy_errors > 0) {
		copy_errors--;
		return UNKNOWN;
	}
	memcpy(d, s, n);
	return SUCCESS;
}
int hipGetSymbolAddress(void **p, const void *sym)
{
	for (int i = 0; i < nv; i++)
		if (vptr[i] == sym) {
			symbol_bytes = vsize[i];
			*p = calloc(1, vsize[i]);
			return *p ? SUCCESS : OUT_OF_MEMORY;
		}
	return UNKNOWN;
}
int hipStreamCreateWithFlags(void **s, unsigned int f)
{
	(void)f;
	*s = malloc(8);
	streams_made++;
	return SUCCESS;
}
int hipStreamDestroy(void *s) { free(s); streams_freed++; return SUCCESS; }
int hipStreamSynchronize(void *s)
{
	(void)s;
	if (sync_errors > 0) {
		sync_errors--;
		return UNKNOWN;
	}
	return SUCCESS;
}
int hipEventCreate(void **e) { *e = malloc(8); return SUCCESS; }
int hipEventCreateWithFlags(void **e, unsigned int f) { (void)f; return hipEventCreate(e); }
int hipEventDestroy(void *e) { free(e); return SUCCESS; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return SUCCESS; }
int hipEventSynchronize(void *e) { (void)e; return SUCCESS; }
int hipEventQuery(void *e) { (void)e; return SUCCESS; }
int hipEventElapsedTime(float *ms, void *a, void *b)
{
	(void)a; (void)b;
	*ms = event_ms ? (float)event_ms(nlog) : 0.01f;
	return SUCCESS;
}
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return SUCCESS; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = malloc(8); return SUCCESS; }
int hipGraphInstantiate(void **e, void *g, void **n, char *log, size_t size)
{
	(void)g; (void)n; (void)log; (void)size;
	*e = malloc(8);
	return SUCCESS;
}
int hipGraphLaunch(void *e, void *s) { (void)e; (void)s; return SUCCESS; }
int hipGraphDestroy(void *g) { free(g); return SUCCESS; }
int hipGraphExecDestroy(void *e) { free(e); return SUCCESS; }
