/* Stand-in for the device layer (csrc/croma_kernels.h) on host memory: the C
 * host runtime links against it and runs on the CPU, so that its routes, its
 * allocations and the device it works on can be tested without a GPU.  Copies
 * are immediate, events are always complete, kernels compute nothing and are
 * recorded.  A stream or event belongs to the device current at its creation;
 * recording an event on another device's stream, and a launch on a stream of
 * a device that is not current, fail as they do in the HIP runtime.  So does
 * the replay of a graph whose contraction writes to memory since freed, which
 * on a device would be a write out of range. */
#include "croma_kernels.h"

#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define STUB_LOG 4096

typedef struct {
    int dev;
    double at; /* events: the clock when recorded */
} Obj;

typedef struct Head {
    size_t bytes;
    int dev, fixed, serial;
    struct Head *next;
} Head; /* before every device allocation */

typedef struct {
    const void *inje; /* what the captured contraction writes, */
    int serial;       /* and the allocation it lay in */
} Graph;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static __thread int cur;
static char err[128] = "stub";
static size_t live, peak, limit = (size_t)1 << 40, free_mem = (size_t)1 << 38;
static int log_mode[STUB_LOG], log_rows[STUB_LOG], log_tasks[STUB_LOG], nlog;
static int dev_streams[8], dev_events[8], dev_allocs[8];
static Head *allocs;
static char fixed_mem[16 << 20];
static size_t fixed_next;
static int fixed_used;
static __thread int capturing;
static __thread const void *captured;
static int nalloc;
static void (*hook_host_alloc)(void);
/* the clock advances with each fused launch of tasks over k snapshots at r
 * rows per lane by launch_ms[r] + k slot_ms[r] */
static double now_ms, launch_ms[17], slot_ms[17];

void stub_reset(void)
{
    peak = live;
    limit = (size_t)1 << 40;
    free_mem = (size_t)1 << 38;
    nlog = 0;
    hook_host_alloc = 0;
    for (int r = 0; r <= 16; r++) launch_ms[r] = 1.0, slot_ms[r] = 0.0;
    memset(dev_streams, 0, sizeof(dev_streams));
    memset(dev_events, 0, sizeof(dev_events));
    memset(dev_allocs, 0, sizeof(dev_allocs));
}
void stub_set_limit(size_t largest, size_t free_bytes)
{
    limit = largest;
    free_mem = free_bytes;
}
void stub_set_cost(int r, double launch, double slot)
{
    launch_ms[r] = launch;
    slot_ms[r] = slot;
}
/* the next device allocation of this size takes the one fixed address, if that
 * is free */
void stub_fix_next(size_t bytes) { fixed_next = bytes; }
void stub_set_host_alloc_hook(void (*f)(void)) { hook_host_alloc = f; }
size_t stub_peak(void) { return peak; }
size_t stub_live(void) { return live; }
int stub_launches(int *mode, int *rows, int *tasks, int cap)
{
    int i;
    for (i = 0; i < nlog && i < cap; i++) mode[i] = log_mode[i], rows[i] = log_rows[i], tasks[i] = log_tasks[i];
    return nlog;
}
/* streams, events and device allocations made on device d since the reset */
void stub_made(int d, int *out)
{
    out[0] = dev_streams[d];
    out[1] = dev_events[d];
    out[2] = dev_allocs[d];
}

static int fail(const char *what)
{
    snprintf(err, sizeof(err), "stub: %s", what);
    return -1;
}
static int on_current(void *s) { return !s || ((Obj *)s)->dev == cur ? 0 : fail("launch on another device's stream"); }

const char *ck_last_error(void) { return err; }
int ck_device_count(void) { return 8; }
int ck_set_device(int d)
{
    if (d < 0 || d >= 8) return fail("device");
    cur = d;
    return 0;
}
int ck_get_device(void) { return cur; }
int ck_device_name(int dev, char *buf, int len) { return snprintf(buf, (size_t)len, "stub %d", dev) < 0; }
int ck_device_cu_count(int dev) { return dev >= 0 ? 256 : 0; }
int ck_mem_info(size_t *f, size_t *t)
{
    *f = free_mem;
    *t = free_mem;
    return 0;
}
void *ck_malloc(size_t bytes)
{
    Head *h;
    const int fix = fixed_next == bytes && !fixed_used && 256 + bytes <= sizeof(fixed_mem);
    if (bytes > limit || !(h = fix ? (Head *)fixed_mem : (Head *)calloc(1, 256 + bytes))) {
        fail("out of memory");
        return 0;
    }
    if (fix) memset(h, 0, 256 + bytes), fixed_next = 0, fixed_used = 1;
    h->bytes = bytes;
    h->dev = cur;
    h->fixed = fix;
    pthread_mutex_lock(&mu);
    h->serial = ++nalloc;
    h->next = allocs;
    allocs = h;
    live += bytes;
    if (live > peak) peak = live;
    dev_allocs[cur]++;
    pthread_mutex_unlock(&mu);
    return (char *)h + 256;
}
int ck_free(void *p)
{
    Head *h = (Head *)((char *)p - 256), **q;
    if (!p) return 0;
    pthread_mutex_lock(&mu);
    live -= h->bytes;
    for (q = &allocs; *q != h; q = &(*q)->next) {}
    *q = h->next;
    pthread_mutex_unlock(&mu);
    if (h->fixed) fixed_used = 0;
    else free(h);
    return 0;
}
void *ck_host_alloc(size_t bytes)
{
    if (hook_host_alloc) hook_host_alloc();
    return calloc(1, bytes + 8);
}
int ck_host_free(void *p)
{
    free(p);
    return 0;
}
static void *make(int *count)
{
    Obj *o = (Obj *)calloc(1, sizeof(*o));
    o->dev = cur;
    pthread_mutex_lock(&mu);
    count[cur]++;
    pthread_mutex_unlock(&mu);
    return o;
}
void *ck_stream_create(void) { return make(dev_streams); }
int ck_stream_destroy(void *s)
{
    free(s);
    return 0;
}
int ck_stream_sync(void *s) { return s ? 0 : 0; }
void *ck_event_create(void) { return make(dev_events); }
int ck_event_destroy(void *e)
{
    free(e);
    return 0;
}
int ck_event_record(void *e, void *s)
{
    ((Obj *)e)->at = now_ms;
    return !s || ((Obj *)e)->dev == ((Obj *)s)->dev ? 0 : fail("event of another device");
}
int ck_event_query(void *e) { return e ? 1 : -1; }
int ck_event_sync(void *e) { return e ? 0 : -1; }
float ck_event_elapsed_ms(void *a, void *b) { return a && b ? (float)(((Obj *)b)->at - ((Obj *)a)->at) : -1.0f; }
int ck_stream_wait_event(void *s, void *e) { return s && e ? 0 : -1; }
int ck_h2d(void *dst, const void *src, size_t bytes, void *s)
{
    (void)s;
    memcpy(dst, src, bytes);
    return 0;
}
int ck_d2h(void *dst, const void *src, size_t bytes, void *s) { return ck_h2d(dst, src, bytes, s); }
int ck_d2d(void *dst, const void *src, size_t bytes, void *s) { return ck_h2d(dst, src, bytes, s); }
int ck_device_sync(void) { return 0; }
static int serial_at(const void *p)
{
    Head *h;
    pthread_mutex_lock(&mu);
    for (h = allocs; h && (char *)h + 256 != (const char *)p; h = h->next) {}
    pthread_mutex_unlock(&mu);
    return h ? h->serial : 0;
}
int ck_graph_begin(void *s)
{
    capturing = 1;
    captured = 0;
    return s ? 0 : -1;
}
void *ck_graph_end(void *s)
{
    Graph *g = (Graph *)calloc(1, sizeof(*g));
    g->inje = captured;
    g->serial = serial_at(captured);
    capturing = 0;
    return s ? g : 0;
}
int ck_graph_launch(void *g, void *s)
{
    return !s || serial_at(((Graph *)g)->inje) != ((Graph *)g)->serial ? fail("graph writes to freed memory") : 0;
}
int ck_graph_destroy(void *g)
{
    free(g);
    return 0;
}

int ck_fill_i32(int *dst, int v, size_t count, void *s)
{
    size_t i;
    if (on_current(s)) return -1;
    for (i = 0; i < count; i++) dst[i] = v;
    return 0;
}
int ck_fill_f64(double *dst, double v, size_t count, void *s)
{
    size_t i;
    if (on_current(s)) return -1;
    for (i = 0; i < count; i++) dst[i] = v;
    return 0;
}
int ck_fill_u8(unsigned char *dst, unsigned char v, size_t count, void *s)
{
    if (on_current(s)) return -1;
    memset(dst, v, count);
    return 0;
}
int ck_fused_supported(int n, int r) { return (r == 2 || r == 4 || r == 8 || r == 16) && n / r >= 4 && n / r <= 64; }
/* the FP32-coefficient instances with the in-kernel contraction are the scarce
 * ones: none at one wave per SIMD here */
int ck_fused_f32_supported(int n, int r, int occ, int mode) { return ck_fused_supported(n, r) && (mode != 1 || occ == 2); }
int ck_launch_fused(int n, int r, int occ, int nblocks, int mode, CkGrid g, const CkSlot *slots, const CkTask *tasks,
                    int ntasks, int *counter, int *e, void *s)
{
    (void)n, (void)occ, (void)nblocks, (void)g, (void)slots, (void)tasks, (void)counter, (void)e;
    if (on_current(s)) return -1;
    pthread_mutex_lock(&mu);
    now_ms += launch_ms[r] + (ntasks > 0 ? tasks[0].nslot : 0) * slot_ms[r];
    if (nlog < STUB_LOG) log_mode[nlog] = mode, log_rows[nlog] = r, log_tasks[nlog] = ntasks, nlog++;
    pthread_mutex_unlock(&mu);
    return 0;
}
/* every tracer takes 8 substeps, all of them on */
int ck_nsub_arrays(CkGrid g, CkParams prm, int ntr, double dt, double lo, double hi, const double *n_gas,
                   const double *kbt, const double *b, const double *divv, const double *lt, const double *dv,
                   int *nsub, int *n_on, void *s)
{
    int i;
    (void)g, (void)prm, (void)dt, (void)lo, (void)hi, (void)n_gas, (void)kbt, (void)b, (void)divv, (void)lt, (void)dv;
    if (on_current(s)) return -1;
    for (i = 0; i < ntr; i++) nsub[i] = n_on[i] = 8;
    return 0;
}

/* the tasks in the tracers' order */
int ck_nsub_order(CkGrid g, const CkSlot *slots, int count, int ntr, int protons, int split, CkTask *tasks, int *key,
                  int *segloc, int *blk, int *hist, unsigned long long *cells, void *s)
{
    int i;
    (void)g, (void)slots, (void)protons, (void)split, (void)key, (void)segloc, (void)blk, (void)hist, (void)cells;
    if (on_current(s)) return -1;
    for (i = 0; i < ntr; i++) tasks[i].slot = 0, tasks[i].tracer = i, tasks[i].nslot = count;
    return 0;
}

/* the remaining launches do nothing but look at their stream, the last argument */
int ck_sec_contract(int n, const double *a, const int *b, const double *c, double *d, long e, const int *f, int g,
                    void *s)
{
    (void)n, (void)a, (void)b, (void)c, (void)e, (void)f, (void)g;
    if (capturing) captured = d;
    return on_current(s);
}
int ck_ic_rows(int n, const double *a, double b, double c, int d, const double *e, double *f, double *g, int *h, void *s)
{
    (void)n, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h;
    return on_current(s);
}
int ck_grid_loss_tables(CkGrid g, double epmax, void *s)
{
    (void)g, (void)epmax;
    return on_current(s);
}
int ck_lerp_f64(size_t n, const double *a, const double *b, double c, double *d, void *s)
{
    (void)n, (void)a, (void)b, (void)c, (void)d;
    return on_current(s);
}
int ck_plain_gather(int n, int c, const int *i, const CkSlot *S, CkPlainWs w, void *s)
{
    (void)n, (void)c, (void)i, (void)S, (void)w;
    return on_current(s);
}
int ck_plain_lerp(int n, int c, const int *i, const CkSlot *S, double a, CkPlainWs w, void *s)
{
    (void)n, (void)c, (void)i, (void)S, (void)a, (void)w;
    return on_current(s);
}
int ck_plain_coeff(int n, int c, CkGrid g, CkParams p, double a, double b, int d, CkPlainWs w, int *e, void *s)
{
    (void)n, (void)c, (void)g, (void)p, (void)a, (void)b, (void)d, (void)w, (void)e;
    return on_current(s);
}
int ck_plain_secondary(int n, int c, const double *a, int j, CkPlainWs w, void *s)
{
    (void)n, (void)c, (void)a, (void)j, (void)w;
    return on_current(s);
}
int ck_plain_thomas(int n, int c, int a, double b, int d, int f, int g, int h, CkPlainWs w, int *e, void *s)
{
    (void)n, (void)c, (void)a, (void)b, (void)d, (void)f, (void)g, (void)h, (void)w, (void)e;
    return on_current(s);
}
int ck_plain_scatter(int n, int c, const int *i, const CkSlot *S, CkPlainWs w, void *s)
{
    (void)n, (void)c, (void)i, (void)S, (void)w;
    return on_current(s);
}
int ck_solve_cc_batch(int n, int m, double dt, const double *a, const double *b, const double *c, const double *q,
                      const double *x, double *y, double *w, int *e, int mark, void *s)
{
    (void)n, (void)m, (void)dt, (void)a, (void)b, (void)c, (void)q, (void)x, (void)y, (void)w, (void)e, (void)mark;
    return on_current(s);
}
int ck_emission_contract(int a, int b, int c, int d, const double *e, const uint16_t *f, const uint16_t *g,
                         const float *h, const double *i, const int *j, const double *k, double *l, int m, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h, (void)i, (void)j, (void)k, (void)l, (void)m;
    return on_current(s);
}
int ck_synch_table(int a, int b, int c, int d, double e, double f, int g, double h, const double *i, const double *j,
                   const double *k, const double *l, const double *m, double *n, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h, (void)i, (void)j, (void)k, (void)l, (void)m,
        (void)n;
    return on_current(s);
}
int ck_synch_mfma_prepare(int a, int b, int c, const double *d, const double *e, uint16_t *f, uint16_t *g, int *h,
                          float *i, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h, (void)i;
    return on_current(s);
}
int ck_synch_mfma_run(int a, int b, int c, int d, double e, double f, const double *g, const uint16_t *h,
                      const uint16_t *i, const int *j, const float *k, int *l, int *m, const double *n, const double *o,
                      const double *p, double *q, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h, (void)i, (void)j, (void)k, (void)l, (void)m,
        (void)n, (void)o, (void)p, (void)q;
    return on_current(s);
}
int ck_secondary_weights(int n, const double *a, const double *b, const double *c, const double *d, double *e, int *f,
                         void *s)
{
    (void)n, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f;
    return on_current(s);
}
int ck_emission_kernel_table(int a, int b, int c, double d, double e, double f, const double *g, double *h, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h;
    return on_current(s);
}
int ck_emission_synch(int a, int b, int c, int d, double e, double f, const double *g, double *h, int *i,
                      const double *j, const double *k, const double *l, double *m, int n, void *s)
{
    (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h, (void)i, (void)j, (void)k, (void)l, (void)m,
        (void)n;
    return on_current(s);
}
