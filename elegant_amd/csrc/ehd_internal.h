/*
 * ehd_internal.h - state of one device context (HIP side only).
 */
#ifndef ELEGANT_AMD_EHD_INTERNAL_H
#define ELEGANT_AMD_EHD_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "eh_program.h"

#define EHD_MAX_COLL 16
/* the no-allocation WAKE step: most wake points (bins) and the size of its
 * static scratch (plan 128 B + histogram and voltage for EHD_NOALLOC_BINS + 16
 * bins + 1,025 fixed-point partials, rounded up) */
#define EHD_ZL_MAX_BINS (1 << 20) /* ZLONGIT bins: the bin optimiser's default cap (ztransverse.c:672-759) */
/* Rows on their way in or out: 4 million of 8 columns at a time, a copy of 5 ms
 * against some 20 us of launch and wait, so that they take this much of the
 * device beside the 64 bytes per particle of the columns, not 140 per particle */
#define EHD_STAGE_BYTES ((int64_t)256 << 20)
#define EHD_PIN_BYTES (1 << 20) /* small results come back through pinned memory */
#define EHD_NOALLOC_BINS 16384
#define EHD_NOALLOC_BYTES (256 * 1024)

typedef struct {
  double *W;          /* WAKE Green function */
  int64_t wpoints;
  double *Z, *tc, *ts; /* ZLONGIT impedance and FFT twiddles */
  int32_t nb;
  int64_t W_cap, Z_cap; /* points the buffers hold: kept between uploads */
  int32_t tw_nb;        /* bins the twiddles are for, 0: none yet */
} ehd_coll_slot;

struct ehd_dev {
  int device;
  hipStream_t stream;
  hipEvent_t ev0, ev1, cev0, cev1;
  double *coord[6];
  int32_t *loss_pass, *loss_code;
  double *ids;         /* particle IDs (column 6 of the rows) */
  int64_t n, cap;
  int64_t upload;      /* counts the uploads: whose particles the columns hold */
  /* rows as the caller holds them, on their way to or from the columns
   * above: at most EHD_STAGE_BYTES each, kept between calls, freed with the
   * context */
  double *rows, *rows2;
  int64_t rows_cap, rows2_cap;   /* doubles */
  int32_t rows_w;                /* columns per row of the last upload */
  int rows_kept;                 /* rows holds all of it */
  int64_t stage_rows;            /* tests: rows at a time */
  int32_t *order;
  int64_t order_cap;
  void *pin;           /* pinned host buffer of EHD_PIN_BYTES */
  eh_op *ops;          /* flat records of the batch kernel's programs */
  int32_t nops;
  int64_t ops_cap;
  /* the tracking kernel's program (ehd_put_program) */
  eh_op *host_prog;    /* flat copy on the host: patches refold it */
  int32_t nflat, host_prog_cap;
  void *pbuf, *pstage; /* the three arrays below in one buffer, and its pinned host copy */
  size_t pbuf_cap;
  hipEvent_t pev;      /* the last copy out of pstage */
  eh_op *tops;         /* run bodies */
  eh_run *runs;
  double *zpos;        /* (z_start, z_end) of each flat position */
  int32_t ntops, nruns;
  int32_t block;
  unsigned long long *counter;
  double track_ms, coll_ms;
  int64_t track_launches, coll_launches;
  /* collective work buffers */
  ehd_coll_slot slot[EHD_MAX_COLL];
  void *cwork;       /* reductions, histogram, voltages */
  void *host_plan;   /* a collective step's plan, pinned */
  int32_t *bunch;    /* bunch index per particle (bunched beams) */
  int64_t bunch_cap;
  void *noalloc;     /* device address of this GPU's static no-allocation scratch */
  int64_t cwork_bytes;
  /* batched variants */
  eh_vdesc *vdesc;
  eh_chunk *chunks;
  int32_t nvar, nchunks, chunk_cap, var_cap;
  unsigned int *queue;
  int32_t *perm;     /* compacted particle indices the chunks refer to (NULL: identity) */
  int64_t perm_cap;
  int use_perm;
  int32_t *dev_nchunks; /* the chunk count the batch kernel reads (inside the queue buffer) */
  int32_t *tile_sum;    /* device compaction: tile prefix sums, then per-variant info */
  int64_t tile_cap;
  int32_t vinfo_cap;
  double *snap[6];
  int32_t *snap_lp, *snap_lc;
  int64_t snap_cap;
  int num_cu;
  char msg[512];
};

#endif
