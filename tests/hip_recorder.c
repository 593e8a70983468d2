/*
 * A HIP runtime without a GPU, for tests of the engine's host side on the CPU: the entry points that
 * alis_amd/libalis.so uses, over host memory.  Device memory is zeroed host memory and copies are
 * made at once; kernels do not run, but every launch, wait and copy is recorded in order:
 *
 *     launch <kernel> <workgroups> <stream>
 *     wait <stream> <stream the event was recorded on>
 *
 * Loaded (RTLD_GLOBAL) before the library, whose references then bind here.  There are two devices;
 * an event may be recorded only on a stream of its own device.  A box that k_unpack would write
 * outside its allocation is counted (hipRecOutside), and so is a launch of k_mirror from a thread
 * whose current device is not the stream's (hipRecForeign).
 */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3;
typedef struct { int device, id, held; } stream;
typedef struct { int device; stream *on; } event;

enum { OK = 0, INVALID_VALUE = 1, INVALID_HANDLE = 400, NOT_READY = 600 };

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t changed = PTHREAD_COND_INITIALIZER;

/* ---- record ---- */

static char *text;
static size_t used, room;
static int nstreams, waiting, nevents, npinned, pinnedNow;
static long outside, foreign;

static void say(const char *what, const char *name, long n, int s)
{
	char line[400];
	const int k = snprintf(line, sizeof line, "%s %s %ld %d\n", what, name, n, s);
	pthread_mutex_lock(&lock);
	if (used + k + 1 > room) text = realloc(text, room = 2 * room + 4096);
	memcpy(text + used, line, k + 1);
	used += k;
	pthread_mutex_unlock(&lock);
}

const char *hipRecLog(void) { return text ? text : ""; }
void hipRecClear(void) { if (text) text[used = 0] = 0; }
long hipRecOutside(void) { return outside; }
long hipRecForeign(void) { return foreign; }
int hipRecStreamOf(void *s) { return ((stream *)s)->id; }
int hipRecPinned(void) { return npinned; }              /* pinned allocations made, and held now */
int hipRecPinnedNow(void) { return pinnedNow; }

/* The next wait for an event blocks until hipRecLetGo (once): hipRecWaiting tells that one does. */
static int hold;
void hipRecHold(void) { pthread_mutex_lock(&lock), hold = 1, pthread_mutex_unlock(&lock); }
int hipRecWaiting(void) { pthread_mutex_lock(&lock); const int w = waiting; pthread_mutex_unlock(&lock); return w; }
void hipRecLetGo(void) { pthread_mutex_lock(&lock), hold = waiting = 0, pthread_cond_broadcast(&changed), pthread_mutex_unlock(&lock); }

/* ---- devices ---- */

static __thread int current;

int hipGetDeviceCount(int *n) { *n = 2; return OK; }
int hipGetDevice(int *d) { *d = current; return OK; }
int hipSetDevice(int d) { if (d < 0 || d > 1) return INVALID_VALUE; current = d; return OK; }
int hipDeviceSynchronize(void) { return OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorString(int e) { return e == INVALID_HANDLE ? "event and stream of different devices" : "error"; }

/* ---- memory ---- */

typedef struct { char *at; size_t n; } block;
static block *blocks;
static int nblocks, capblocks;

int hipMalloc(void **p, size_t n)
{
	*p = calloc(1, n);
	pthread_mutex_lock(&lock);
	if (nblocks == capblocks) blocks = realloc(blocks, (capblocks = 2 * capblocks + 64) * sizeof *blocks);
	blocks[nblocks++] = (block){*p, n};
	pthread_mutex_unlock(&lock);
	return OK;
}

int hipFree(void *p)
{
	pthread_mutex_lock(&lock);
	for (int b = 0; b < nblocks; b++) if (blocks[b].at == p) { blocks[b] = blocks[--nblocks]; break; }
	pthread_mutex_unlock(&lock);
	free(p);
	return OK;
}

int hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n); npinned++, pinnedNow++; return OK; }
int hipHostFree(void *p) { free(p); pinnedNow--; return OK; }
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *s) { (void)kind, (void)s; memcpy(dst, src, n); return OK; }
int hipMemsetAsync(void *dst, int v, size_t n, void *s) { (void)s; memset(dst, v, n); return OK; }

/* ---- streams and events ---- */

int hipStreamCreateWithFlags(void **s, unsigned flags)
{
	stream *S = calloc(1, sizeof *S);
	(void)flags;
	S->device = current;
	pthread_mutex_lock(&lock), S->id = nstreams++, pthread_mutex_unlock(&lock);
	*s = S;
	return OK;
}
int hipStreamDestroy(void *s) { (void)s; return OK; }       /* (their number stays valid) */
int hipStreamSynchronize(void *s) { (void)s; return OK; }

int hipEventCreateWithFlags(void **e, unsigned flags)
{
	event *E = calloc(1, sizeof *E);
	(void)flags;
	E->device = current;
	nevents++;
	*e = E;
	return OK;
}
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { free(e); return OK; }

static int record(event *E, stream *S)
{
	if (E->device != S->device) return INVALID_HANDLE;
	E->on = S;
	return OK;
}
int hipEventRecord(void *e, void *s) { return record(e, s); }
int hipEventQuery(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a, (void)b; *ms = 1; return OK; }
int hipEventSynchronize(void *e)
{
	(void)e;
	pthread_mutex_lock(&lock);
	if (hold && !waiting) {
		waiting = 1;
		while (hold) pthread_cond_wait(&changed, &lock);
	}
	pthread_mutex_unlock(&lock);
	return OK;
}
int hipStreamWaitEvent(void *s, void *e, unsigned flags)
{
	event *E = e;
	(void)flags;
	say("wait", "-", ((stream *)s)->id, E->on ? E->on->id : -1);
	return OK;
}

/* ---- kernels ---- */

static struct { const void *f; char name[200]; } kernels[512];
static int nkernels;
static char handle[8];

void **__hipRegisterFatBinary(const void *data) { (void)data; return (void **)handle; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int ext, size_t n, int constant, int global) { (void)m, (void)v, (void)h, (void)d, (void)ext, (void)n, (void)constant, (void)global; }
int hipGetSymbolAddress(void **p, const void *v) { (void)v; *p = calloc(1, 4 << 20); return OK; }
void __hipRegisterFunction(void **m, const void *f, char *h, const char *name, unsigned limit, void *a, void *b, void *c, void *d, int *w)
{
	(void)m, (void)h, (void)limit, (void)a, (void)b, (void)c, (void)d, (void)w;
	if (nkernels == 512) return;
	kernels[nkernels].f = f;
	snprintf(kernels[nkernels++].name, sizeof kernels[0].name, "%s", name);
}

static __thread struct { dim3 grid, block; size_t lds; void *s; } call;
int __hipPushCallConfiguration(dim3 grid, dim3 blk, size_t lds, void *s) { call.grid = grid, call.block = blk, call.lds = lds, call.s = s; return OK; }
int __hipPopCallConfiguration(dim3 *grid, dim3 *blk, size_t *lds, void **s) { *grid = call.grid, *blk = call.block, *lds = call.lds, *s = call.s; return OK; }

/* k_unpack(src, index map, box, dst): the places of the box's corners against dst's allocation. */
static void checkUnpack(const char *name, void **args)
{
	const struct { int i0, j0, k0, koff; long si, sj; } *L = args[1];
	const int *b = args[2];
	char *dst = *(char **)args[3];
	const long size = strstr(name, "k_unpackId") ? 8 : 4;
	const long lo = (b[0] - L->i0) * L->si + (b[2] - L->j0) * L->sj + b[4] - L->k0 + L->koff;
	const long hi = (b[1] - L->i0) * L->si + (b[3] - L->j0) * L->sj + b[5] - L->k0 + L->koff;
	pthread_mutex_lock(&lock);
	int in = 0;
	for (int x = 0; x < nblocks; x++)
		if (dst >= blocks[x].at && dst < blocks[x].at + blocks[x].n)
			in = dst + lo * size >= blocks[x].at && dst + (hi + 1) * size <= blocks[x].at + blocks[x].n;
	outside += !in;
	pthread_mutex_unlock(&lock);
}

static int launch(const void *f, dim3 grid, void **args, stream *S)
{
	const char *name = "?";
	for (int k = 0; k < nkernels; k++) if (kernels[k].f == f) name = kernels[k].name;
	if (strstr(name, "k_unpack")) checkUnpack(name, args);
	if (strstr(name, "k_mirror") && S->device != current) __atomic_fetch_add(&foreign, 1, __ATOMIC_RELAXED);
	say("launch", name, (long)grid.x * grid.y * grid.z, S->id);
	return OK;
}
int hipLaunchKernel(const void *f, dim3 grid, dim3 blk, void **args, size_t lds, void *s)
{
	(void)blk, (void)lds;
	return launch(f, grid, args, s);
}
int hipExtLaunchKernel(const void *f, dim3 grid, dim3 blk, void **args, size_t lds, void *s, void *e0, void *e1, int flags)
{
	(void)blk, (void)lds, (void)flags;
	if ((e0 && record(e0, s)) || (e1 && record(e1, s))) return INVALID_HANDLE;
	return launch(f, grid, args, s);
}
