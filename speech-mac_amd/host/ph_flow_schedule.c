/* Task list of the one-launch decode step (pgpu_flow_launch, phonon_gpu.h).
 *
 * The order is the launch's dispatch order. Every task comes after the
 * tasks it waits for, so the lowest-numbered unfinished task can always run
 * and the launch cannot deadlock.
 *
 * Within that constraint the list is laid out on a model clock: attention
 * tasks advance the clock by unit_us each (they stream K/V from HBM at a
 * steady rate), and each projection phase of a tile's chain is listed
 * after_us[phase] after the tile's last attention task, i.e. about when its
 * inputs will be ready. A task listed too early holds a work-group slot
 * while it waits; one listed too late delays its chain. The next layer's
 * attention of a tile is never listed before that tile's QKV (a pending
 * chain is flushed first). */
#include "ph_internal.h"

#include <stdlib.h>

typedef struct {
    double at;        /* model time of the entry */
    size_t seq;       /* insertion order (ties) */
    uint32_t kind, layer, tile;
} Pending;

typedef struct {
    Pending *items;
    size_t count, seq;
    int fused;  /* fused MLP: MLP_OUT only after the last layer */
} Queue;

static const uint32_t kChainKinds[4] = {PGPU_FLOW_OUT, PGPU_FLOW_MLP_IN, PGPU_FLOW_MLP_OUT,
                                        PGPU_FLOW_QKV};

/* Tasks of one phase of a (layer, tile); with the fused MLP, MLP_OUT is the
 * last layer's output tasks. */
static uint32_t phase_tasks(uint32_t kind, int fused) {
    switch (kind) {
    case PGPU_FLOW_QKV: return PGPU_FLOW_QKV_TASKS;
    case PGPU_FLOW_OUT: return PGPU_FLOW_OUT_TASKS;
    case PGPU_FLOW_MLP_IN: return PGPU_FLOW_MLP_IN_TASKS;
    default: return fused ? PGPU_FLOW_FUSED_OUT_TASKS : PGPU_FLOW_MLP_OUT_TASKS;
    }
}

/* QKV tasks head by head (q, k, v of head 0, then of head 1, ...): the
 * attention of a head waits only for its own three. */
static void emit_phase(uint32_t *d, size_t *k, uint32_t kind, uint32_t layer, uint32_t tile,
                       int fused) {
    const uint32_t n = phase_tasks(kind, fused);
    for (uint32_t i = 0; i < n; i++) {
        const uint32_t index = kind == PGPU_FLOW_QKV ? (i % 3) * PH_HEADS + i / 3 : i;
        d[(*k)++] = PGPU_FLOW_TASK(kind, layer, tile, index);
    }
}

/* Sorted insert by (at, seq). */
static void push(Queue *q, double at, uint32_t kind, uint32_t layer, uint32_t tile) {
    size_t i = q->count++;
    const Pending e = {at, q->seq++, kind, layer, tile};
    while (i > 0 && q->items[i - 1].at > at) {
        q->items[i] = q->items[i - 1];
        i--;
    }
    q->items[i] = e;
}

static void remove_at(Queue *q, size_t i) {
    for (; i + 1 < q->count; i++)
        q->items[i] = q->items[i + 1];
    q->count--;
}

/* Emits every pending entry, one kind after another (all OUT, then all
 * MLP_IN, ...): with many tiles a tile-major chain would fill the dispatch
 * window with tasks that wait for each other. */
static void flush_by_phase(Queue *q, uint32_t *d, size_t *k) {
    for (int p = 0; p < 4; p++)
        for (size_t i = 0; i < q->count;) {
            const Pending e = q->items[i];
            if (e.kind == kChainKinds[p]) {
                emit_phase(d, k, e.kind, e.layer, e.tile, q->fused);
                remove_at(q, i);
            } else {
                i++;
            }
        }
}

/* Emits every pending entry of `tile` (all tiles if tile < 0), in order. */
static void flush(Queue *q, int tile, uint32_t *d, size_t *k) {
    for (size_t i = 0; i < q->count;) {
        const Pending e = q->items[i];
        if (tile < 0 || e.tile == (uint32_t)tile) {
            emit_phase(d, k, e.kind, e.layer, e.tile, q->fused);
            remove_at(q, i);
        } else {
            i++;
        }
    }
}

pgpu_flow_placement ph_flow_default_placement(int rounds) {
    /* Clock in ATTN tasks (rounds 256-key splits, 128 KB of K/V each): at
     * B = 64 a 16-stream tile's attention is ~640 splits. Swept on MI355X
     * at B = 64 (one split per task) and B = 48, 96, 128, 160 (two), contexts
     * U{1..2048}; a decode step's own placement follows its contexts
     * (ph_flow_step_placement). */
    const pgpu_flow_placement one = {1.0f, {550.0f, 1000.0f, 1450.0f, 1750.0f}};
    const pgpu_flow_placement two = {2.0f, {1150.0f, 1850.0f, 2550.0f, 3050.0f}};
    return rounds > 1 ? two : one;
}

/* One while a step is a latency chain, two (fewer, longer attention tasks, which
 * keep more K/V in flight per work-group slot) once it streams. us per step,
 * one / two, contexts U{1..n}, splits of a layer over all heads: 16 streams n =
 * 1000 (400) 410 / 439; 16, 8000 (2232) 880 / 890; 48, 2048 (2008) 611 / 652; 64,
 * 2048 (2800) 672 / 740; 64, 3000 (3536) 832 / 850; 64, 4000 (4440) 1036 / 997;
 * 64, 6000 (6296) 1468 / 1400. With more tiles the line lies lower, since what
 * the other tiles' tasks leave uncovered is shorter: it is drawn at the number of
 * those (2700, where 3600 splits of four tiles lie). 112, 1000 (2503 of the
 * others) 640 / 651; 72, 2048 (2803) 823 / 807; 96, 1500 (2900) 849 / 794; 192,
 * 300 (2816) 676 / 527; 224, 300 (3328) 722 / 576; 128, 1000 (3087) 790 / 732. Up
 * to two tiles whose contexts fill one task of two splits run those (16 streams,
 * n = 300: 374 / 365), except the smallest batches. */
int ph_flow_step_rounds(size_t streams, size_t splits) {
    enum { ONE_ROUND_STREAMS = 8, ONE_ROUND_SPLITS = 3600, ONE_ROUND_OTHERS = 2700 };
    const size_t tiles = (streams + 15) / 16, all = splits * PH_HEADS;
    if (streams <= ONE_ROUND_STREAMS)
        return 1;
    if (tiles <= 2 && splits <= 2 * streams)
        return PGPU_FLOW_ATTN_ROUNDS;
    return all <= ONE_ROUND_SPLITS && all * (tiles - 1) <= ONE_ROUND_OTHERS * tiles
               ? 1
               : PGPU_FLOW_ATTN_ROUNDS;
}

/* A tile's QKV, the last of its chain's four phases, belongs just before the
 * other tiles' attention tasks of the layer run out, for that is when the
 * tile's next attention can be listed: later and the tile starves, earlier and
 * the waiting tasks hold slots. The other phases come before it in the
 * proportion of the times they take. `last` against the others' tasks was swept
 * on MI355X over 0.58 .. 1.06 of them (one split per task) and 2300 .. 4200
 * (two), and lies on straight lines between the points below: it is nearly all
 * of them for few, when the chain takes longer than they do; 0.82 from 2100 on;
 * from 3700 on less, the chain being long done. It must not jump: at 2022 ..
 * 2100 others (64 streams, contexts U{1..2048}) a step takes 656 .. 672 us at
 * 0.82 of them, 666 .. 678 at 0.88 and 695 .. 707 at 0.94, while 1696 (40
 * streams) take 588 at 0.94 and 609 at 0.82. us per step, contexts U{1..n},
 * against the fixed offsets above: 24 streams n = 6000 760 / 824; 40, 2048 588 /
 * 726; 48, 2048 619 / 719; 64, 300 442 / 592; 64, 6000 1402 / 1533; 128, 300 478
 * / 842; 160, 2048 1575 / 1566; 200, 2048 1870 / 1860. */
pgpu_flow_placement ph_flow_step_placement(size_t tiles, size_t splits, int rounds) {
    /* More than eight tiles leave "nearly all" earlier: 224 streams, n = 100, 578
     * at 0.94 of 1664 others, 481 at 0.82 (fixed offsets 535); 176, 100 484 at 0.94
     * of 1280, 449 at 0.86; 144, 100 434 at 0.94 of 1024, 480 at 0.86; but 128, 240
     * 472 at 0.82 of 1792, 452 at 0.9. */
    const int many = tiles > 8;
    const struct {
        double others, last;
    } at[] = {{0, 0},
              {many ? 1024 : 1700, many ? 0.94 * 1024 : 0.94 * 1700},
              {many ? 1536 : 2100, many ? 0.82 * 1536 : 0.82 * 2100},
              {3700, 0.82 * 3700},
              {4200, 0.75 * 4200},
              {5600, 0.75 * 5600}};
    enum { POINTS = sizeof(at) / sizeof(at[0]) };
    const double others = tiles ? (double)splits * (tiles - 1) / tiles : 0.0;
    double last = at[POINTS - 1].last;
    for (int i = 1; i < POINTS; i++)
        if (others < at[i].others) {
            last = at[i - 1].last + (at[i].last - at[i - 1].last) * (others - at[i - 1].others) /
                                        (at[i].others - at[i - 1].others);
            break;
        }
    const float f = (float)last;
    return (pgpu_flow_placement){(float)rounds, {0.314f * f, 0.571f * f, 0.829f * f, f}};
}

size_t pgpu_flow_schedule(size_t streams, size_t layers, const size_t *units,
                          const pgpu_flow_placement *place, int flags, uint32_t *schedule,
                          size_t capacity) {
    if (!streams || !layers || !units || (flags & ~(PGPU_FLOW_SCHEDULE_PREFILL |
                                                    PGPU_FLOW_SCHEDULE_FUSED_MLP)))
        return 0;
    const int prefill = (flags & PGPU_FLOW_SCHEDULE_PREFILL) != 0;
    const int fused = !prefill && (flags & PGPU_FLOW_SCHEDULE_FUSED_MLP) != 0;
    const size_t tiles = (streams + 15) / 16;
    size_t attn = 0;
    for (size_t s = 0; s < streams; s++)
        attn += units[s];
    const size_t chain = PGPU_FLOW_QKV_TASKS + PGPU_FLOW_OUT_TASKS + PGPU_FLOW_MLP_IN_TASKS;
    const size_t tasks = layers * tiles * chain +
                         (fused ? tiles * PGPU_FLOW_FUSED_OUT_TASKS
                                : layers * tiles * PGPU_FLOW_MLP_OUT_TASKS) +
                         layers * PH_HEADS * attn;
    if (!schedule || capacity < tasks)
        return tasks;
    double after[4] = {0.0, 0.0, 0.0, 0.0}, unit_us = 0.0;
    if (place && !prefill) {
        unit_us = place->unit_us > 0.0f ? place->unit_us : 0.0;
        for (int p = 0; p < 4; p++) {
            const double a = place->after_us[p] > 0.0f ? place->after_us[p] : 0.0;
            after[p] = p && a < after[p - 1] ? after[p - 1] : a;  /* phases in order */
        }
    }
    Queue q = {malloc(4 * tiles * sizeof(Pending)), 0, 0, fused};
    if (!q.items)
        return 0;
    uint32_t *d = schedule;
    size_t k = 0;
    for (size_t t = 0; t < tiles; t++)
        emit_phase(d, &k, PGPU_FLOW_QKV, 0, (uint32_t)t, fused);
    double now = 0.0;
    for (size_t l = 0; l < layers; l++) {
        /* With prefill every ATTN task of layer l waits for the QKV of all
         * tiles: everything pending goes first, phase by phase. */
        if (prefill)
            flush_by_phase(&q, d, &k);
        for (size_t t = 0; t < tiles; t++) {
            flush(&q, (int)t, d, &k);  /* tile t's chain, through its QKV of layer l */
            for (size_t n = 0; n < 16 && t * 16 + n < streams; n++)
                for (size_t j = 0; j < units[t * 16 + n]; j++)
                    for (uint32_t h = 0; h < PH_HEADS; h++) {
                        while (q.count && q.items[0].at <= now) {
                            emit_phase(d, &k, q.items[0].kind, q.items[0].layer,
                                       q.items[0].tile, fused);
                            remove_at(&q, 0);
                        }
                        d[k++] = PGPU_FLOW_TASK(PGPU_FLOW_ATTN, l, t, h | j << 3 | n << 11);
                        now += unit_us;
                    }
            for (int p = 0; p < 4; p++) {
                if (p == 3 && l + 1 == layers)
                    break;
                if (p == 2 && fused && l + 1 < layers)
                    continue; /* the next layer's QKV tasks sum the MLP partials */
                /* prefill: the layer's chains wait for the next layer's flush */
                push(&q, prefill ? 1e300 : now + after[p], kChainKinds[p],
                     (uint32_t)(p == 3 ? l + 1 : l), (uint32_t)t);
            }
        }
    }
    if (prefill)
        flush_by_phase(&q, d, &k);
    else
        flush(&q, -1, d, &k);
    free(q.items);
    return k;
}
