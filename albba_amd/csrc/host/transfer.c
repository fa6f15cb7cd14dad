/*
 * Copies between the device and the caller's ordinary memory.
 *
 * Above STAGED_MIN bytes a copy goes through the context's pinned stages in
 * pieces: the device's copy engine fills or drains one stage (30 GB/s on this
 * link) while a few threads move another one between pinned and ordinary
 * memory.  What bounds such a copy otherwise is the ordinary memory: a fresh
 * result array is paged in during the copy, by one thread at 4 GB/s (eight:
 * 23), and an upload of memory the runtime has not seen pins it first (7 GB/s
 * for a 250 MB matrix).
 */
#include "internal.h"
#include "device_int.h"

#include <errno.h>
#include <omp.h>
#include <unistd.h>

/* below this the threads' start costs more than they save: 2 x 2 MB of
 * results take 213 us in one thread and 249 staged, 2 x 4 MB 431 and 338,
 * 2 x 64 MB 13.1 ms and 4.7 */
#define STAGED_MIN ((size_t)3 << 20)
#define COPY_THREADS 8

/* pieces of a transfer: at least four, so that the engine's and the threads'
 * parts overlap on small ones too, of 256 KB to a whole stage */
static size_t piece_bytes(size_t bytes)
{
    size_t p = (bytes / 4 + 65535) / 65536 * 65536;
    if (p < ((size_t)256 << 10)) p = (size_t)256 << 10;
    return p > ALBD_STAGE_BYTES ? ALBD_STAGE_BYTES : p;
}

static int copy_threads(void)
{
    const int t = omp_get_max_threads();
    return t < COPY_THREADS ? t : COPY_THREADS;
}

/* thread `id` of `n`: its part of `len` bytes, cut at pages */
static void part_of(size_t len, int id, int n, size_t *lo, size_t *hi)
{
    const size_t per = (len / (size_t)n + 4095) / 4096 * 4096;
    *lo = (size_t)id * per < len ? (size_t)id * per : len;
    *hi = id == n - 1 || *lo + per > len ? len : *lo + per;
}

int albba_d2h(albd_ctx *d, void *dst, const void *src, size_t bytes)
{
    void *stage[ALBD_STAGES];
    if (bytes < STAGED_MIN || albd_stages(d, stage)) return albd_d2h(d, dst, src, bytes);
    const size_t piece = piece_bytes(bytes);
    const int64_t np = (int64_t)((bytes + piece - 1) / piece);
    int rc = 0;
#define PIECE_LEN(i) ((i) + 1 < np ? piece : bytes - (size_t)(i) * piece)
    for (int64_t i = 0; !rc && i < np && i < ALBD_STAGES; ++i)
        rc = albd_d2h_async(d, stage[i], (const char *)src + (size_t)i * piece, PIECE_LEN(i)) || albd_stage_mark(d, (int)i);
    if (!rc) {
#pragma omp parallel num_threads(copy_threads())
        for (int64_t i = 0; i < np; ++i) {
            const int k = (int)(i % ALBD_STAGES);
#pragma omp master
            rc = rc ? rc : albd_stage_wait(d, k);
#pragma omp barrier
            if (rc) break; /* every thread reads the same value */
            size_t lo, hi;
            part_of(PIECE_LEN(i), omp_get_thread_num(), omp_get_num_threads(), &lo, &hi);
            memcpy((char *)dst + (size_t)i * piece + lo, (const char *)stage[k] + lo, hi - lo);
#pragma omp barrier
#pragma omp master
            if (i + ALBD_STAGES < np)
                rc = albd_d2h_async(d, stage[k], (const char *)src + (size_t)(i + ALBD_STAGES) * piece,
                                    PIECE_LEN(i + ALBD_STAGES)) ||
                     albd_stage_mark(d, k);
        }
    }
    /* nothing may still write a stage when it is used next */
    const int rs = albd_sync(d);
    albd_stages_release(d);
    return rc ? ALBBA_EHIP : rs;
}

/* Fill the stages piece by piece (from memory, or from a file when fd >= 0)
 * and send each to the device. */
static int to_device(albd_ctx *d, void *dst, const void *src, int fd, int64_t off, size_t bytes, void *const *stage)
{
    const size_t piece = piece_bytes(bytes);
    const int64_t np = (int64_t)((bytes + piece - 1) / piece);
    /* Every thread has to leave the loop at the same barrier: it leaves on
     * what only the master writes, and not again before each thread has passed
     * another barrier.  (On `bad`, which a thread may set as soon as it reads,
     * a slower one could leave while the others waited for it: a hang.) */
    int rc = 0, bad = 0, waited = 0, stop = 0;
#pragma omp parallel num_threads(copy_threads())
    for (int64_t i = 0; i < np; ++i) {
        const int k = (int)(i % ALBD_STAGES);
#pragma omp master
        if (i >= ALBD_STAGES) waited = albd_stage_wait(d, k);
#pragma omp barrier
        if (waited) break;
        size_t lo, hi;
        part_of(PIECE_LEN(i), omp_get_thread_num(), omp_get_num_threads(), &lo, &hi);
        if (fd < 0) {
            memcpy((char *)stage[k] + lo, (const char *)src + (size_t)i * piece + lo, hi - lo);
        } else {
            while (lo < hi) {
                const ssize_t r = pread(fd, (char *)stage[k] + lo, hi - lo, (off_t)(off + (int64_t)((size_t)i * piece + lo)));
                if (r < 0 && errno == EINTR) continue;
                if (r <= 0) {
#pragma omp atomic write
                    bad = 1;
                    break;
                }
                lo += (size_t)r;
            }
        }
#pragma omp barrier
#pragma omp master
        {
            if (!bad)
                rc = albd_h2d_async(d, (char *)dst + (size_t)i * piece, stage[k], PIECE_LEN(i)) ||
                     albd_stage_mark(d, k);
            stop = rc || bad;
        }
#pragma omp barrier
        if (stop) break;
    }
    const int rs = albd_sync(d);
    if (bad) return ALBBA_EIO;
    return rc || waited ? ALBBA_EHIP : rs;
}

int albba_h2d(albd_ctx *d, void *dst, const void *src, size_t bytes)
{
    void *stage[ALBD_STAGES];
    if (bytes < STAGED_MIN || albd_stages(d, stage)) return albd_h2d(d, dst, src, bytes);
    const int rc = to_device(d, dst, src, -1, 0, bytes, stage);
    albd_stages_release(d);
    return rc;
}

int albba_file_to_device(albd_ctx *d, FILE *f, int64_t off, void *dst, size_t bytes)
{
    void *stage[ALBD_STAGES];
    int rc = bytes ? albd_stages(d, stage) : 0;
    if (rc || !bytes) return rc;
    if (lseek(fileno(f), 0, SEEK_CUR) >= 0) {
        rc = to_device(d, dst, NULL, fileno(f), off, bytes, stage);
    } else {
        /* not seekable: read in order */
        for (size_t done = 0; !rc && done < bytes;) {
            const size_t len = bytes - done < ALBD_STAGE_BYTES ? bytes - done : ALBD_STAGE_BYTES;
            if (fread(stage[0], 1, len, f) != len) rc = ALBBA_EIO;
            if (!rc) rc = albd_h2d_async(d, (char *)dst + done, stage[0], len);
            const int rs = albd_sync(d); /* the stage is filled again */
            rc = rc ? rc : rs;
            done += len;
        }
    }
    albd_stages_release(d);
    return rc;
}

_Static_assert(STAGED_MIN <= ALBD_STAGE_BYTES, "a smaller array fits a stage");

int albba_d2h_pair(albd_ctx *d, void *dst0, const void *src0, void *dst1, const void *src1, size_t bytes)
{
    void *stage[ALBD_STAGES];
    int rc;
    if (!dst0 || !dst1 || bytes >= STAGED_MIN || bytes == 0 || albd_stages(d, stage)) {
        rc = dst0 ? albba_d2h(d, dst0, src0, bytes) : 0;
        return !rc && dst1 ? albba_d2h(d, dst1, src1, bytes) : rc;
    }
    /* one stage each; of larger arrays the first is copied while the second
     * is on its way */
    const int early = bytes >= ((size_t)256 << 10);
    rc = albd_d2h_async(d, stage[0], src0, bytes) || (early && albd_stage_mark(d, 0)) ||
         albd_d2h_async(d, stage[1], src1, bytes);
    if (!rc && early && !(rc = albd_stage_wait(d, 0))) memcpy(dst0, stage[0], bytes);
    const int rs = albd_sync(d);
    if (!rc && !rs) {
        if (!early) memcpy(dst0, stage[0], bytes);
        memcpy(dst1, stage[1], bytes);
    }
    albd_stages_release(d);
    return rc ? ALBBA_EHIP : rs;
}
