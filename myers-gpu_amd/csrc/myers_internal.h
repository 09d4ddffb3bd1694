/*
 * Internal entry points shared by the C host files of libmyers_amd.so
 * (not exported in the public headers).
 */
#ifndef MYERS_INTERNAL_H
#define MYERS_INTERNAL_H

#include <stdint.h>

/* 1 if every operation enqueued on the buffer's stream has finished, 0 if
 * work is pending, negative on a HIP error. */
int myers_buffer_ready(void *myersBuffer);

/* The launches of a buffer's last batch, for tests of the dispatch: MYERS_RAN_*
 * bits, and the split launch's words per lane and slots (0 without one). */
enum { MYERS_RAN_BIN = 1,            /* a launch per bin */
       MYERS_RAN_SLICE = 2,          /* sliced kernel, reads up to 1024 bases */
       MYERS_RAN_FIRST_ROWS = 4,     /* their first rows, and the rest of those kept */
       MYERS_RAN_WIDE_SLICE = 8,     /* sliced kernel of longer reads */
       MYERS_RAN_QUEUE = 16,         /* multi-lane queue launch */
       MYERS_RAN_LONG = 32,          /* long-read launch */
       MYERS_RAN_SPLIT = 64,         /* split launch */
       MYERS_RAN_HANDOVERS = 128,    /* ... of several parts per candidate */
       MYERS_RAN_CUT = 256 };        /* cut-off kernel of a bin's launch */
typedef struct {
    uint32_t ran, split_words, split_slots;
} myers_launch_info_t;
int myers_launch_info(void *myersBuffer, myers_launch_info_t *out);

/* What the resident server needs from a library instance: the device, the
 * resident reference, the buffer's threshold, and for every read length in
 * words the variant the resident kernel runs it with (the bin table's
 * choice when that variant can run there, else the cheapest one that can),
 * given as the variant's key (lanes << 8 | words) and its pull rank (0 for
 * the variant with the most words per candidate). */
#define MYERS_SERVE_MAX_WORDS 768u       /* MYERS_MAX_QUERY_SIZE / 32 */
typedef struct {
    int             device;
    int             num_cus;
    const uint32_t *d_ref;
    uint64_t        ref_words;           /* readable words, guard included */
    uint64_t        ref_size;
    float           threshold;           /* < 0: off */
    uint32_t        max_words;           /* longest read the plan covers, in words */
    uint32_t        lds_bytes;           /* largest workspace of the plan's variants */
    uint32_t        num_ranks;
    uint32_t        rank_key[64];        /* key of each rank */
    uint32_t        rank_slots[64];      /* candidates per chunk of each rank */
    uint8_t         rank_of_words[MYERS_SERVE_MAX_WORDS + 1];
} myers_serve_plan_t;
int myers_serve_plan(void *myersBuffer, myers_serve_plan_t *out);

#endif
