/*
 * host_check.c - the library's host code on the CPU, with the GPU runtime and
 * the kernel launches it needs replaced by the few lines below: device memory
 * is ordinary memory, copies are done at once, and every pointer handed to a
 * copy or a launch has to lie in a live allocation.  One check per argument;
 * exit status 0 when it holds, and why not on stderr.
 */
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#define float3 zpic_float3 /* the runtime's headers have a type of that name */
#include "zpic_internal.h"

static int failed;
#define CHECK(c)                                                                                                       \
    do {                                                                                                               \
        if (!(c)) {                                                                                                    \
            fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c);                                                    \
            failed = 1;                                                                                                \
        }                                                                                                              \
    } while (0)

/* ---- device memory ---- */

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static struct {
    char *p;
    size_t n;
} block[256];

static int live(const void *p, size_t n)
{
    int ok = 0;
    pthread_mutex_lock(&lock);
    for (int k = 0; k < 256; k++)
        ok |= block[k].p && (const char *)p >= block[k].p && (const char *)p + n <= block[k].p + block[k].n;
    pthread_mutex_unlock(&lock);
    return ok;
}

hipError_t hipMalloc(void **p, size_t n)
{
    *p = calloc(1, n);
    pthread_mutex_lock(&lock);
    int k = 0;
    while (block[k].p) k++;
    block[k].p = *p;
    block[k].n = n;
    pthread_mutex_unlock(&lock);
    return hipSuccess;
}

hipError_t hipFree(void *p)
{
    pthread_mutex_lock(&lock);
    for (int k = 0; k < 256; k++)
        if (block[k].p == p) block[k].p = NULL;
    pthread_mutex_unlock(&lock);
    free(p);
    return hipSuccess;
}

hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t s)
{
    const int ok = kind == hipMemcpyHostToDevice   ? live(dst, n)
                   : kind == hipMemcpyDeviceToHost ? live(src, n)
                                                   : live(dst, n) && live(src, n);
    CHECK(ok);
    if (ok) memcpy(dst, src, n);
    return hipSuccess;
}

/* ---- the rest of the runtime ---- */

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
static __thread int device; /* current device of the thread; streams are on device 0 */
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipSetDevice(int d) { return device = d, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }
static int pinned;   /* allocations of page-locked memory and of events */
static int nopinned; /* page-locked memory has run out */
hipError_t hipHostMalloc(void **p, size_t n, unsigned f)
{
    pinned++;
    *p = nopinned ? NULL : malloc(n);
    return nopinned ? hipErrorOutOfMemory : hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) 
{
    CHECK(device == 0); /* an event belongs to the device it is made on */
    pinned++;
    *e = (hipEvent_t)1;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    CHECK(device == 0);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return "error"; }

/* ---- launches ---- */

int zk_fill_f32(float *p, size_t n, float v, zk_stream_t s)
{
    CHECK(live(p, 4 * n));
    if (live(p, 4 * n))
        for (size_t k = 0; k < n; k++) p[k] = v;
    return 0;
}

int zk_unpack(const void *aos, int n, const zk_parts *dst, int64_t id0, zk_spec_ctr *ctr, int append, zk_stream_t s)
{
    CHECK(live(aos, 28 * (size_t)n) && live(dst->cell, 4 * (size_t)n));
    ctr->np_total = n;
    return 0;
}

int zk_sort(const zk_parts *src, const zk_parts *dst, zk_spec_ctr *ctr, int *cnt, int *off, int *cursor, int *tile_n,
            const zk_tiles *t, int np_upper, int spread, int slack, int cap_slots, zk_stream_t s)
{
    ctr->n_sorted = ctr->np_total;
    return 0;
}

int zk_charge(zk_charge_args a, int tail_upper, zk_stream_t s)
{
    CHECK(live(a.rho, 4 * (size_t)(a.t.nx + 1) * (a.t.ny + 1)));
    return 0;
}

int zk_noalloc_scratch(float **p)
{
    static void *scratch;
    if (!scratch) hipMalloc(&scratch, 8 * (size_t)ZK_NOALLOC_CHARGE_MAX);
    *p = scratch;
    return 0;
}

int zk_add_f32(float *acc, const float *v, size_t n, zk_stream_t s)
{
    for (size_t k = 0; k < n; k++) acc[k] += v[k];
    return 0;
}

/* ---- checks ---- */

static void species(t_species *s, int nx, int ny)
{
    const int n[2] = {nx, ny}, ppc[2] = {1, 1};
    const float u[3] = {0, 0, 0};
    float box[2] = {0.1f * nx, 0.1f * ny};
    spec_new(s, "electrons", -1.0f, ppc, u, u, n, box, 0.07f, NULL);
}

/* the staging buffer is allocated again after the species' device buffers
 * were freed to track ids */
static void staging(void)
{
    t_species s;
    species(&s, 8, 8);
    float rho[81] = {0};
    spec_deposit_charge(&s, rho);
    spec_track_ids(&s);
    CHECK(s.dev->stage == NULL);
    spec_deposit_charge(&s, rho);
    CHECK(live(s.dev->stage, s.dev->stage_cap));
}

/* the charge deposit that allocates nothing, on a grid whose read would
 * otherwise be staged through page-locked memory */
static void noalloc(void)
{
    t_species s;
    species(&s, 1500, 1400);
    zpic_stage_hold(1);
    zpic_species_ensure(&s);
    float *rho = malloc(4 * (size_t)1501 * 1401);
    for (int k = 0; k < 1501 * 1401; k++) rho[k] = 1.0f;
    pinned = 0;
    CHECK(spec_deposit_charge_noalloc(&s, rho) == 0);
    CHECK(pinned == 0);
    CHECK(rho[1600] == 1.0f);
}

/* large reads with and without page-locked memory to stage them in */
static void reads(void)
{
    const size_t n = (size_t)9 << 20;
    char *src = zpic_dmalloc(n), *dst = malloc(n);
    for (size_t k = 0; k < n; k++) src[k] = (char)(k * 7 + k / 4096);
    zpic_stage_hold(1);
    for (nopinned = 1; nopinned >= 0; nopinned--) {
        memset(dst, 0, n);
        zpic_d2h(dst, src, n);
        CHECK(!memcmp(dst, src, n));
    }
    pinned = 0;
    zpic_d2h(dst, src, n);
    CHECK(pinned == 0); /* the chunks are kept */
    zpic_stage_hold(-1);
}

/* a large read by a caller that works on another device */
static void other_device(void)
{
    const size_t n = (size_t)9 << 20;
    char *src = zpic_dmalloc(n), *dst = malloc(n);
    zpic_stage_hold(1);
    device = 1;
    zpic_d2h(dst, src, n);
    CHECK(device == 1);
    zpic_stage_hold(-1);
}

/* a slab on a grid whose cells are not square: its particles fit the buffer */
static void slab(void)
{
    const float dx[3] = {0.05f, 0.1f, 0.2f};
    for (int k = 0; k < 9; k++) {
        const int n[2] = {130, 70}, ppc[2] = {2, 2};
        const float u[3] = {0, 0, 0};
        float box[2] = {dx[k / 3] * n[0], dx[k % 3] * n[1]};
        t_density d;
        memset(&d, 0, sizeof(d));
        d.type = SLAB;
        d.n = 1.0f;
        d.start = 0.2f * box[0];
        d.end = 0.6f * box[0];
        t_species s;
        spec_new(&s, "slab", -1.0f, ppc, u, u, n, box, 0.01f, &d);
        CHECK(s.np == 52 * 70 * 4);
        CHECK(s.np <= s.np_max);
    }
}

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "staging")) staging();
    else if (!strcmp(what, "noalloc")) noalloc();
    else if (!strcmp(what, "reads")) reads();
    else if (!strcmp(what, "device")) other_device();
    else if (!strcmp(what, "slab")) slab();
    else CHECK(!"a known check");
    return failed;
}
