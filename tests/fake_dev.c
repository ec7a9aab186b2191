/* A stand-in for the device layer (libcc_amd/csrc/ccx_dev.h) on host memory, for tests of the C host
 * layer's state without a GPU: device memory is counted against a budget, kernels do nothing
 * (except the input scan, which scans), calls can be made to fail, and the clearing of the scan's
 * flag is queued on its stream and done only when that stream is waited for or used by a scan. */
#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

long long fake_total = 1LL << 40;  /* device memory, bytes */
long long fake_room = 1LL << 40;   /* what can still be had of it */
int fake_fail_zero_flag, fake_fail_scan;   /* how many of the next calls fail */
void (*fake_during_adjoint)(void);         /* called while a gradient's kernels would run */

#define NALLOC 4096
static struct { void *p; size_t n; } g_mem[NALLOC];
static struct { unsigned int *flag; void *stream; } g_clear[64];
static int g_nclear;

static void run_stream(void *stream)
{
    int left = 0;
    for (int q = 0; q < g_nclear; ++q)
        if (g_clear[q].stream == stream) *g_clear[q].flag = 0u;
        else g_clear[left++] = g_clear[q];
    g_nclear = left;
}

int ccx_hip_malloc(void **p, size_t bytes)
{
    *p = NULL;
    if (bytes == 0) return 0;
    if ((long long)bytes > fake_room) return 1;
    for (int q = 0; q < NALLOC; ++q)
        if (!g_mem[q].p) {
            if (!(*p = malloc(bytes))) return 1;
            memset(*p, 0xab, bytes < 4096 ? bytes : 4096);   /* nothing is clear by itself */
            g_mem[q].p = *p;
            g_mem[q].n = bytes;
            fake_room -= (long long)bytes;
            return 0;
        }
    return 1;
}

int ccx_hip_free(void *p)
{
    if (!p) return 0;
    int left = 0;
    for (int q = 0; q < g_nclear; ++q)   /* a free waits for the work on its memory */
        if ((void *)g_clear[q].flag != p) g_clear[left++] = g_clear[q];
    g_nclear = left;
    for (int q = 0; q < NALLOC; ++q)
        if (g_mem[q].p == p) {
            fake_room += (long long)g_mem[q].n;
            g_mem[q].p = NULL;
            free(p);
            return 0;
        }
    abort();   /* freed twice, or never allocated */
}

int ccx_hip_host_malloc(void **p, size_t bytes) { return (*p = malloc(bytes ? bytes : 1)) ? 0 : 1; }
int ccx_hip_host_free(void *p) { free(p); return 0; }
int ccx_hip_sync(void *stream) { run_stream(stream); return 0; }
int ccx_hip_memcpy_h2d(void *dst, const void *src, size_t n, void *stream) { memcpy(dst, src, n); return ccx_hip_sync(stream); }
int ccx_hip_memcpy_d2h(void *dst, const void *src, size_t n, void *stream) { memcpy(dst, src, n); return ccx_hip_sync(stream); }
int ccx_hip_memcpy_d2d(void *dst, const void *src, size_t n, void *stream) { (void)stream; memcpy(dst, src, n); return 0; }
int ccx_hip_memcpy_h2d_queue(void *dst, const void *src, size_t n, void *stream) { (void)stream; memcpy(dst, src, n); return 0; }

int ccx_hip_zero_flag(unsigned int *flag, void *stream)
{
    if (fake_fail_zero_flag > 0) { --fake_fail_zero_flag; return 1; }
    g_clear[g_nclear].flag = flag;
    g_clear[g_nclear++].stream = stream;
    return 0;
}

int ccx_hip_nonfinite(const double *const *p, const size_t *n, int narr, unsigned int *flag, int *nonfinite, void *stream)
{
    run_stream(stream);
    for (int q = 0; q < narr; ++q)
        for (size_t i = 0; i < n[q]; ++i)
            if (!isfinite(p[q][i])) *flag |= 1u;
    if (fake_fail_scan > 0) { --fake_fail_scan; *flag |= 1u; return 1; }   /* the result could not be fetched */
    *nonfinite = *flag != 0u;
    return 0;
}

/* The kernels (declared without parameters, so ccx_dev.h is not included here) */
int ccx_hip_adj_items() { if (fake_during_adjoint) fake_during_adjoint(); return 0; }
int fake_packed_routes;            /* virtual-triple sums that went through the packed copies */
int ccx_hip_w_abc() { return 0; }
int ccx_hip_abc_pack() { ++fake_packed_routes; return 0; }
int ccx_hip_w_abc_packed() { return 0; }
#define KERNEL(name) int name() { return 0; }
KERNEL(ccx_hip_pack) KERNEL(ccx_hip_pack_ax_one) KERNEL(ccx_hip_pack_pairs) KERNEL(ccx_hip_triples)
KERNEL(ccx_hip_pack_split) KERNEL(ccx_hip_pack_f32v) KERNEL(ccx_hip_finalize) KERNEL(ccx_hip_t1wt3)
KERNEL(ccx_hip_x_abc)
KERNEL(ccx_hip_gax) KERNEL(ccx_hip_gbx) KERNEL(ccx_hip_dvoe_reduce) KERNEL(ccx_hip_unpack_grad) KERNEL(ccx_hip_zero)

int ccx_hip_event_create(void **ev) { *ev = NULL; return 0; }
int ccx_hip_event_destroy(void *ev) { (void)ev; return 0; }
int ccx_hip_event_record(void *ev, void *stream) { (void)ev; (void)stream; return 0; }
int ccx_hip_event_ms(void *start, void *stop, float *ms) { (void)start; (void)stop; *ms = 1.0f; return 0; }
int ccx_hip_device_count(int *n) { *n = 1; return 0; }
int ccx_hip_cu_count(int *n) { *n = 4; return 0; }
int ccx_hip_mem_info(size_t *room, size_t *total) { *room = (size_t)fake_room; *total = (size_t)fake_total; return 0; }
int ccx_hip_form_kpad(int form) { return form == 1 ? 48 : form == 3 ? 256 : form >= 2 ? 64 : 4; }
int ccx_hip_split_elem_bytes(int form) { return form == 2 ? 6 : 8; }
size_t ccx_hip_adj_stage_doubles(void) { return 1024; }
size_t ccx_hip_gbx_part_doubles(int nup, int kp, int nent, int nsplit) { return (size_t)nent * nsplit * nup * kp; }
size_t ccx_hip_abc_a_doubles(int no, int nu, int kp) { return (size_t)no * nu * nu * kp; }
size_t ccx_hip_abc_b_doubles(int no, int nu, int kp) { return (size_t)no * no * nu * kp; }
