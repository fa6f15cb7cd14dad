/* The host objects that own device state, shared by the host sources that
 * drive the device (level loop, batched BFS). */
#ifndef ALBBA_DEVICE_INT_H
#define ALBBA_DEVICE_INT_H

#include "internal.h"
#include "../albd.h"

struct albba_ctx {
    albd_ctx *d;
    int device;
};

struct albba_graph {
    albba_ctx *ctx;
    albd_graph g;
    albd_state st;
    int32_t n;
    int32_t sigma;       /* the layout's sigma as requested */
    int32_t order_flags; /* ALBBA_SELL_* row-order flags of the layout */
    int64_t nnz;
    int64_t device_bytes;
    void *scratch_visited; /* BEST-policy snapshots */
    void *scratch_ctr;
    int64_t *host_log;     /* small-frontier level sizes, 4 per level */
    int64_t *word_entries; /* host: stored entries per position word, made
                            * on the first BFS that accounts swept entries */
    int32_t *list_copy;    /* host: a pull's word list, for that accounting */
    int needs_reset;       /* a BFS failed midway: pmin/pkey may be dirty */
};

/* host/transfer.c: as albd_d2h / albd_h2d, through the context's pinned
 * stages and several threads where the copy is large */
ALBBA_HIDDEN int albba_d2h(albd_ctx *d, void *dst, const void *src, size_t bytes);
ALBBA_HIDDEN int albba_h2d(albd_ctx *d, void *dst, const void *src, size_t bytes);
/* two device arrays of `bytes` each (a null destination: not that one) */
ALBBA_HIDDEN int albba_d2h_pair(albd_ctx *d, void *dst0, const void *src0, void *dst1, const void *src1,
                                size_t bytes);
/* `bytes` of f at offset `off` (where f stands, if it cannot seek) into device
 * memory; ALBBA_EIO when the file is shorter */
ALBBA_HIDDEN int albba_file_to_device(albd_ctx *d, FILE *f, int64_t off, void *dst, size_t bytes);

#endif
