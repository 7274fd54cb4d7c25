/*
 * croma_stage.c -- transfers between pageable host arrays and the device
 * through a pinned ring filled (emptied) by several host threads.
 *
 * The runtime's own pageable copies go through one thread's staging: measured
 * 28 GB/s up and 18 GB/s down, against 57 GB/s for pinned memory either way.
 * Here up to four threads each take every fourth 1 MiB piece of an array, copy
 * it into (out of) one of their two pinned slots and queue the piece's transfer
 * on a stream of their own, between an event that the caller's stream recorded
 * before and one that it waits for after (on one stream the transfers'
 * start-up, 15 us each, kept it to 31 GB/s).  82 MB up 2,781 -> 1,769 us, down
 * 4,633 -> 1,814 us, into untouched memory 8,047 -> 2,502 us.  Arrays below 4
 * MiB, and transfers that find the ring in use by another thread, take the
 * runtime's path.
 *
 * These are the rates of a warm process.  The runtime opens its copy engines one
 * by one, when a copy finds the opened ones busy, and the copy call that opens
 * one takes 6.5 ms: about five of a process's first thirty calls of 40,000 x 256
 * emissivities take 9.6 ms instead of 3.0, and the first 15 to 22 ms (5.9 each
 * and 13 the first with the runtime's copies).  Two streams, or larger pieces,
 * open an engine or two less and run 2 to 5% slower.  A copy kernel of 16 blocks
 * opens none and is as fast, but waits for the end of a persistent kernel that
 * another thread is running (65 ms where an engine takes 2), so the copies stay
 * with the engines.
 *
 * One ring per device, made at the first large transfer and shared by the
 * device's contexts (8 MiB of pinned memory, a millisecond to allocate); it is
 * freed with the last of them.  Its lock is held for a whole transfer; a slot
 * is reused after the event behind its last transfer.  The ring is made and
 * used with its device current, which the calling thread's need not be.
 */
#include "croma_host.h"

#include <pthread.h>
#include <string.h>

#define ST_THREADS 4
#define ST_SLOTS 2
#define ST_PIECE ((size_t)1 << 20)
#define ST_MIN ((size_t)4 << 20)
#define ST_DEVICES 16

typedef struct {
    pthread_mutex_t lock; /* held by the transfer using the ring */
    char *pin;
    void *st[ST_THREADS]; /* streams of the pieces' transfers */
    void *ev_go, *ev_done[ST_THREADS];
    void *ev[ST_THREADS][ST_SLOTS];
    int used[ST_THREADS][ST_SLOTS]; /* the slot's event has been recorded */
} StRing;

static pthread_mutex_t g_refs_lock = PTHREAD_MUTEX_INITIALIZER;
static int g_refs[ST_DEVICES];
static StRing g_ring[ST_DEVICES] = {[0 ... ST_DEVICES - 1] = {.lock = PTHREAD_MUTEX_INITIALIZER}};

static void ring_free(StRing *r)
{
    int t, s;
    for (t = 0; t < ST_THREADS; t++) {
        for (s = 0; s < ST_SLOTS; s++) {
            if (r->ev[t][s]) {
                if (r->used[t][s]) ck_event_sync(r->ev[t][s]);
                ck_event_destroy(r->ev[t][s]);
            }
            r->ev[t][s] = 0;
            r->used[t][s] = 0;
        }
        if (r->ev_done[t]) ck_event_destroy(r->ev_done[t]);
        if (r->st[t]) ck_stream_destroy(r->st[t]);
        r->ev_done[t] = r->st[t] = 0;
    }
    if (r->ev_go) ck_event_destroy(r->ev_go);
    r->ev_go = 0;
    ck_host_free(r->pin);
    r->pin = 0;
}

void ch_stage_ref(int dev)
{
    if (dev < 0 || dev >= ST_DEVICES) return;
    pthread_mutex_lock(&g_refs_lock);
    g_refs[dev]++;
    pthread_mutex_unlock(&g_refs_lock);
}

void ch_stage_unref(int dev)
{
    if (dev < 0 || dev >= ST_DEVICES) return;
    pthread_mutex_lock(&g_refs_lock);
    if (--g_refs[dev] == 0) {
        pthread_mutex_lock(&g_ring[dev].lock);
        ring_free(&g_ring[dev]);
        pthread_mutex_unlock(&g_ring[dev].lock);
    }
    pthread_mutex_unlock(&g_refs_lock);
}

/* The device's ring, locked, or NULL: in use, or no pinned memory. */
static StRing *ring_take(int dev)
{
    StRing *r;
    int t, s, ok = 1;
    if (dev < 0 || dev >= ST_DEVICES) return 0;
    r = &g_ring[dev];
    if (pthread_mutex_trylock(&r->lock)) return 0;
    if (!r->pin) {
        r->pin = (char *)ck_host_alloc(ST_THREADS * ST_SLOTS * ST_PIECE);
        ok = r->pin && (r->ev_go = ck_event_create()) != 0;
        for (t = 0; t < ST_THREADS && ok; t++) {
            ok = (r->st[t] = ck_stream_create()) != 0 && (r->ev_done[t] = ck_event_create()) != 0;
            for (s = 0; s < ST_SLOTS && ok; s++) ok = (r->ev[t][s] = ck_event_create()) != 0;
        }
        if (!ok) {
            ring_free(r);
            pthread_mutex_unlock(&r->lock);
            return 0;
        }
    }
    return r;
}

typedef struct {
    StRing *r;
    int dev, t, nthr, up, rc;
    char *dst;
    const char *src;
    size_t bytes;
} StJob;

static size_t piece_bytes(const StJob *j, size_t k)
{
    return j->bytes - k * ST_PIECE < ST_PIECE ? j->bytes - k * ST_PIECE : ST_PIECE;
}

/* Pieces t, t + nthr, ... of one transfer. */
static void stage_run(StJob *j)
{
    const size_t n = (j->bytes + ST_PIECE - 1) / ST_PIECE;
    size_t k, back = (size_t)j->t;
    int s = 0, sb = 0, rc = 0;
    void *const st = j->r->st[j->t];
    if (ck_stream_wait_event(st, j->r->ev_go)) rc = -1;
    for (k = (size_t)j->t; k < n && !rc; k += (size_t)j->nthr, s ^= 1) {
        char *slot = j->r->pin + (size_t)(j->t * ST_SLOTS + s) * ST_PIECE;
        void *ev = j->r->ev[j->t][s];
        if (j->up) {
            if (j->r->used[j->t][s] && ck_event_sync(ev)) rc = -1;
            if (!rc) {
                memcpy(slot, j->src + k * ST_PIECE, piece_bytes(j, k));
                rc = ck_h2d(j->dst + k * ST_PIECE, slot, piece_bytes(j, k), st) || ck_event_record(ev, st);
            }
        } else {
            /* both slots in flight: empty the older one first */
            if (k >= back + (size_t)(ST_SLOTS * j->nthr)) {
                if (ck_event_sync(ev)) rc = -1;
                else memcpy(j->dst + back * ST_PIECE, slot, piece_bytes(j, back));
                back += (size_t)j->nthr;
                sb ^= 1;
            } else if (j->r->used[j->t][s] && ck_event_sync(ev)) {
                rc = -1; /* an earlier upload from this slot */
            }
            if (!rc)
                rc = ck_d2h(slot, j->src + k * ST_PIECE, piece_bytes(j, k), st) || ck_event_record(ev, st);
        }
        j->r->used[j->t][s] = 1;
    }
    for (; !j->up && back < n && !rc; back += (size_t)j->nthr, sb ^= 1) {
        if (ck_event_sync(j->r->ev[j->t][sb])) rc = -1;
        else memcpy(j->dst + back * ST_PIECE, j->r->pin + (size_t)(j->t * ST_SLOTS + sb) * ST_PIECE, piece_bytes(j, back));
    }
    j->rc = rc || ck_event_record(j->r->ev_done[j->t], st);
}

/* a new thread starts on device 0 */
static void *stage_thread(void *arg)
{
    StJob *j = (StJob *)arg;
    if (ck_set_device(j->dev)) j->rc = -1;
    else stage_run(j);
    return 0;
}

static int stage(int dev, int up, void *dst, const void *src, size_t bytes, void *stream)
{
    StJob jobs[ST_THREADS];
    pthread_t th[ST_THREADS];
    int started[ST_THREADS] = {0}, t, nthr = ch_host_threads(), rc = 0;
    const int prev = bytes >= ST_MIN ? ch_device_enter(dev) : -1;
    StRing *r = prev >= 0 ? ring_take(dev) : 0;
    if (!r) {
        ch_device_leave(prev);
        return up ? ck_h2d(dst, src, bytes, stream) : ck_d2h(dst, src, bytes, stream);
    }
    if (nthr > ST_THREADS) nthr = ST_THREADS;
    if (nthr < 1) nthr = 1;
    if (ck_event_record(r->ev_go, stream)) {
        pthread_mutex_unlock(&r->lock);
        ch_device_leave(prev);
        return -1;
    }
    for (t = 0; t < nthr; t++) {
        const StJob j = {r, dev, t, nthr, up, 0, (char *)dst, (const char *)src, bytes};
        jobs[t] = j;
    }
    for (t = 1; t < nthr; t++) started[t] = pthread_create(&th[t], 0, stage_thread, &jobs[t]) == 0;
    stage_run(&jobs[0]);
    for (t = 1; t < nthr; t++) {
        if (started[t]) pthread_join(th[t], 0);
        else stage_run(&jobs[t]);
    }
    for (t = 0; t < nthr; t++) rc |= jobs[t].rc || ck_stream_wait_event(stream, r->ev_done[t]);
    pthread_mutex_unlock(&r->lock);
    ch_device_leave(prev);
    return rc;
}

/* ck_h2d / ck_d2h for arrays of any size: the host array is free for reuse
 * (up) or filled (down, after a stream sync for small arrays) on return. */
int ch_stage_h2d(int dev, void *dst, const void *src, size_t bytes, void *stream)
{
    return stage(dev, 1, dst, src, bytes, stream);
}

int ch_stage_d2h(int dev, void *dst, const void *src, size_t bytes, void *stream)
{
    return stage(dev, 0, dst, src, bytes, stream);
}
