/*
 * uir_plan.c -- work-table construction for the table-driven projectors.
 *
 * FP items: for every subset (a direction run, or one angle) and every
 * detector block of UIRK_FP_DETS, angle blocks of up to the tile's angle
 * count.  An angle block is accepted only if the footprint of its rays over
 * any chunk of UIRK_FP_LINES lines fits the LDS staging window.  Ray
 * positions are affine in the detector index and the line index, so the
 * footprint width over a chunk is a convex function of the chunk's position
 * and attains its maximum at the first or the last chunk; both are evaluated
 * exactly here (with a margin for float stepping).  The line model's ray
 * positions lie half a line step further along than joseph's (`shift`, in
 * line steps).
 */
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "uir_internal.h"

static int fp_push(uirk_fp_vec *v, uirk_fp_item it)
{
    if (v->n == v->cap) {
        size_t cap = v->cap ? 2 * v->cap : 256;
        uirk_fp_item *p = (uirk_fp_item *)realloc(v->v, cap * sizeof *p);
        if (!p)
            return -1;
        v->v = p;
        v->cap = cap;
    }
    v->v[v->n++] = it;
    return 0;
}

static int bp_push(uirk_bp_vec *v, uirk_bp_item it)
{
    if (v->n == v->cap) {
        size_t cap = v->cap ? 2 * v->cap : 256;
        uirk_bp_item *p = (uirk_bp_item *)realloc(v->v, cap * sizeof *p);
        if (!p)
            return -1;
        v->v = p;
        v->cap = cap;
    }
    v->v[v->n++] = it;
    return 0;
}

/* Position steps of an angle's rays per detector and per line. */
typedef struct {
    double det, line;
} ray_step;

/* Footprint width (in staged positions, as the kernel computes it) of the rays
 * of angles ray[0 .. k) and detectors [d0, d0 + 64) over lines [l0, l0 + C). */
static int window_width(int n, int n_dets, double axis, const ray_step *ray, int k, int d0, int l0, double shift)
{
    const int C = UIRK_FP_LINES;
    const int d1 = d0 + UIRK_FP_DETS - 1 < n_dets - 1 ? d0 + UIRK_FP_DETS - 1 : n_dets - 1;
    const int l1 = l0 + C - 1;
    double lo = 1e300, hi = -1e300;
    for (int a = 0; a < k; ++a) {
        const double det_step = ray[a].det, step = ray[a].line;
        const int ds[2] = {d0, d1};
        const int ls[2] = {l0, l1};
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 2; ++j) {
                const double t = (double)ds[i] + 0.5 - axis;
                const double p = t * det_step - 0.5 * n * step + 0.5 * n + ((double)ls[j] + shift) * step;
                if (p < lo) lo = p;
                if (p > hi) hi = p;
            }
    }
    /* kernel: pmin = floor(lo - 0.5) - 1, W = floor(hi - 0.5) + 3 - pmin;
     * +2 margin for the float rounding of stepped coordinates */
    return (int)(floor(hi - 0.5) - floor(lo - 0.5)) + 4 + 2;
}

/* Whether the footprint of angles ray[0 .. k) over detector block d0 fits
 * the staging window in every chunk: the width is convex in the chunk's
 * first line, so the first and the last chunk bound it. */
static int block_fits(int n, int n_dets, float axis, const ray_step *ray, int k, int d0, int wmax, double shift)
{
    const int llast = ((n - 1) / UIRK_FP_LINES) * UIRK_FP_LINES;
    return window_width(n, n_dets, axis, ray, k, d0, 0, shift) <= wmax &&
           window_width(n, n_dets, axis, ray, k, d0, llast, shift) <= wmax;
}

/* Lines [*lo, *hi) outside which no ray of the block (angles ray[0 .. k),
 * detectors [d0, d0 + 64)) samples inside the image.  A sample reads a
 * non-border texel iff its position lies in [-0.5, n + 0.5); positions are
 * affine in the detector and line indices, so each angle's set of lines over
 * the detector block is bounded by its two extreme rays.  A margin of 2
 * positions covers the float rounding of stepped coordinates. */
static void line_range(int n, int n_dets, double axis, const ray_step *ray, int k, int d0, int *lo, int *hi,
                       double shift)
{
    const int d1 = d0 + UIRK_FP_DETS - 1 < n_dets - 1 ? d0 + UIRK_FP_DETS - 1 : n_dets - 1;
    const double plo = -0.5 - 2.0, phi = n + 0.5 + 2.0;
    double lmin = 1e300, lmax = -1e300;
    for (int a = 0; a < k; ++a) {
        const double det_step = ray[a].det, step = ray[a].line;
        const int ds[2] = {d0, d1};
        double p0[2];
        for (int i = 0; i < 2; ++i)
            p0[i] = ((double)ds[i] + 0.5 - axis) * det_step - 0.5 * n * step + 0.5 * n + shift * step;
        for (int i = 0; i < 2; ++i) {
            double l_a, l_b;
            if (fabs(step) < 1e-12) { /* the rays keep their positions: every line if one between the extremes is inside */
                if (fmax(p0[0], p0[1]) < plo || fmin(p0[0], p0[1]) > phi)
                    continue;
                l_a = 0;
                l_b = n;
            } else {
                l_a = (plo - p0[i]) / step;
                l_b = (phi - p0[i]) / step;
                if (l_a > l_b) {
                    const double t = l_a;
                    l_a = l_b;
                    l_b = t;
                }
            }
            if (l_a < lmin) lmin = l_a;
            if (l_b > lmax) lmax = l_b;
        }
    }
    /* Rays between the two extremes are covered: for one angle the entry and
     * exit lines are affine in the detector index, so the union over the
     * block lies within [min, max] of the extreme rays. */
    if (!(lmin <= lmax)) {
        *lo = *hi = 0;
        return;
    }
    double a = floor(lmin) - 1, b = ceil(lmax) + 2;
    if (a < 0) a = 0;
    if (b > n) b = n;
    if (a >= b) {
        *lo = *hi = 0;
        return;
    }
    *lo = (int)a;
    *hi = (int)b;
}

static int plan_fp(uirk_fp_vec *out, int slice, int n, int n_dets, float axis, const float *sin_lut,
                   const float *cos_lut, const uir_subset *subs, uint32_t n_subs, int max_angles, int wmax,
                   double shift)
{
    if (max_angles < 1 || max_angles > UIRK_FP_ANGLES_MAX)
        max_angles = UIRK_FP_ANGLES;
    uint32_t most = 1;
    for (uint32_t si = 0; si < n_subs; ++si)
        most = subs[si].n > most ? subs[si].n : most;
    ray_step *ray = (ray_step *)malloc(sizeof *ray * most);
    if (!ray)
        return -1;
    for (uint32_t si = 0; si < n_subs; ++si) {
        const int off = (int)subs[si].offset, cnt = (int)subs[si].n, dir = subs[si].direction;
        for (int a = 0; a < cnt; ++a) {
            const float s = sin_lut[off + a], c = cos_lut[off + a];
            ray[a].det = dir == 0 ? -1.0 / s : 1.0 / c;
            ray[a].line = dir == 0 ? (double)c / (double)s : (double)s / (double)c;
        }
        /* Angle blocks are cut per detector block: rays far from the axis
         * spread over more positions per angle, so only the outer blocks
         * need fewer angles to fit the window. */
        for (int d0 = 0; d0 < n_dets; d0 += UIRK_FP_DETS) {
            int a = off;
            while (a < off + cnt) {
                /* Shrink in steps of a wave's angle count (a quarter of the
                 * tile's), so that the item's last wave is full: a wave with
                 * no active angle skips the sampling. */
                const int per_wave = max_angles >= 4 ? max_angles / 4 : 1;
                int k = off + cnt - a < max_angles ? off + cnt - a : max_angles;
                while (k > 1 && !block_fits(n, n_dets, axis, ray + (a - off), k, d0, wmax, shift))
                    k = k > per_wave ? ((k - 1) / per_wave) * per_wave : k - 1;
                uirk_fp_item it;
                memset(&it, 0, sizeof it);
                it.slice = slice;
                it.dir = dir;
                it.a0 = a;
                it.na = k;
                it.d0 = d0;
                line_range(n, n_dets, axis, ray + (a - off), k, d0, &it.l_lo, &it.l_hi, shift);
                if (fp_push(out, it)) {
                    free(ray);
                    return -1;
                }
                a += k;
            }
        }
    }
    free(ray);
    return 0;
}

int uirk_plan_fp(uirk_fp_vec *out, int slice, int n, int n_dets, float axis, const float *sin_lut,
                 const float *cos_lut, const uir_subset *subs, uint32_t n_subs, int max_angles, int wmax)
{
    return plan_fp(out, slice, n, n_dets, axis, sin_lut, cos_lut, subs, n_subs, max_angles, wmax, 0.0);
}

int uirk_plan_fp_line(uirk_fp_vec *out, int slice, int n, int n_dets, float axis, const float *sin_unit,
                      const float *cos_unit, const uir_subset *subs, uint32_t n_subs, int max_angles, int wmax)
{
    return plan_fp(out, slice, n, n_dets, axis, sin_unit, cos_unit, subs, n_subs, max_angles, wmax, 0.5);
}

int uirk_plan_bp(uirk_bp_vec *out, int slice, int n, int tile_rows)
{
    if (tile_rows != 32 && tile_rows != UIRK_BP_TILE)
        tile_rows = UIRK_BP_TILE;
    for (int y0 = 0; y0 < n; y0 += tile_rows)
        for (int x0 = 0; x0 < n; x0 += UIRK_BP_TILE) {
            uirk_bp_item it;
            memset(&it, 0, sizeof it);
            it.slice = slice;
            it.x0 = x0;
            it.y0 = y0;
            if (bp_push(out, it))
                return -1;
        }
    return 0;
}

void uirk_plan_trig(const float *sin_lut, const float *cos_lut, uint32_t n, float *trig)
{
    for (uint32_t i = 0; i < n; ++i) {
        trig[2 * i] = sin_lut[i];
        trig[2 * i + 1] = cos_lut[i];
    }
}

int uirk_plan_num_xcd(void)
{
    static int nx = 0;
    if (nx == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeNumberOfXccs, dev) == hipSuccess && v > 0)
            nx = v > UIRK_MAX_XCD ? UIRK_MAX_XCD : v;
        else
            nx = 1;
    }
    return nx;
}

int uirk_plan_device_slots(void)
{
    static int n = 0;
    if (n == 0) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
            n = 4 * cus;
        else
            n = 1024;
    }
    return n;
}

void uirk_plan_bp_count(uirk_bp_counts *c, uint32_t n, uint32_t angles, int rows, int line, int counts_paired)
{
    const int m = line != 0;
    const size_t w = (n + UIRK_BP_TILE - 1) / UIRK_BP_TILE, h32 = (n + 31) / 32;
    const size_t tuned = w * ((n + (uint32_t)rows - 1) / (uint32_t)rows);
    c->all += tuned;
    c->n32[m] += w * h32;
    c->n32_angles[m] += (uint64_t)(w * h32) * angles;
    if (counts_paired) {
        c->p64[m] += tuned;
        c->p32[m] += w * h32;
        c->p32_angles[m] += (uint64_t)(w * h32) * angles;
    }
    c->a_min[m] = c->a_max[m] == 0 || angles < c->a_min[m] ? angles : c->a_min[m];
    c->a_max[m] = angles > c->a_max[m] ? angles : c->a_max[m];
}

/* A pair's item takes 1.4 times the time of one slice's (line model: 1.25), so
 * pairs gain even where they leave CUs idle.  A CU holds 6 unpaired items of 32
 * rows (line model: 4), 3 pair items with 32 staged angles and 4 with 16 (line
 * model: 4).  The tiles are of 32 rows while the paired table is resident at
 * once that way, else of 64; 32 angles are staged while the table is resident at
 * once with them (fewer barriers), else 16.  A slice without a partner runs the
 * pair kernel at a pair's cost, so the slices an item holds count as well.  Items
 * count by their angles, relative to the longest.
 *   Joseph: from more than 4.25 unpaired items of 32 rows a CU on, with at least
 * 1.65 slices an item.  BP in us (f16 sinograms, 200 to 700 angles), unpaired
 * against pairs: 9 x 512 (4.5 a CU) 91 / 83, 4 x 800 229 / 186, 12 x 512 273 /
 * 221, 4 x 1024 259 / 209, 12 x 1024 904 / 738; 7 x 640 (1.75 slices an item)
 * 217 / 211, 5 x 1024 (1.67) 447 / 407, 16 groups of 5 x 512 892 / 840; with 1.5
 * they come out even (10 groups of 3 x 1024 1288 / 1329, 6 of 3 x 417 157 / 165,
 * 6 of 3 x 512 144 / 126).  Images of 16 bits: from 1.5 (3 x 1448 with 90 angles
 * 126 / 109, 4 groups of 3 x 768 127 / 102, 8 of 3 x 512 102 / 75; with 400 angles
 * 390 / 403, 387 / 399, 325 / 294).  Below the line they lose to about 3 a CU (8 x
 * 300 76 / 80, 4 x 512 134 / 142, 6 x 512 199 / 202); from 3 to 4 they would mostly
 * gain (8 x 417 220 / 200, 2 x 1024 163 / 145, 5 x 640 234 / 245), but one or two
 * slices of 1024 are documented to run unpaired in tiles of 32 rows.
 *   Line model: from 2 unpaired items a CU on (5 x 417, 1.9: 137 / 155; 16 x 256
 * 125 / 118, 2 groups of 3 x 417, 2.3: 289 / 261), with at least 1.5 slices an
 * item (3 x 1024 421 / 359, 5 x 800 555 / 430, 10 groups of 3 x 512 499 / 421; at
 * worst even: 2 groups of 3 x 640 383 / 387), or 1.25 if the paired table of 64
 * rows holds 4 items a CU (pairs alternating with two single slices, 1.33: 8 x 4
 * x 512 597 / 543, 2 x 4 x 1024 697 / 650; 1.25: 5 x 5 x 512 973 / 964, 3 x 5 x 640
 * 507 / 536; with fewer 1.33 is even or loses: 3 x 4 x 417 170 / 175).  Up to 5 paired
 * items of 32 rows a CU they keep the 32 rows that the unpaired table would take
 * (3 groups of 3 x 640, 4.7: 191 against 200 with 64; 2 of 3 x 800, 5.1: 376 / 345).
 *   Slices whose angle counts differ by more than a quarter leave the CUs unevenly
 * loaded, where fewer and longer items cost more: pairs from 5.5 items a CU on
 * (line model: 3), 32 rows as in the line model.  Over 365 mixed batches that was
 * 8 % faster than the build that paired from 4 paired items a CU on, and 1 % than
 * 4.25 items of whatever length; one in 25 is slower than the better of both by
 * 5 to 35 % (2 x 1024 of 400 angles beside small slices of 90 to 180: 192 / 131),
 * as the rule does not look at how the items fall on the CUs.  Line model, 200
 * batches: 5 and 3 %. */
uirk_bp_choice uirk_plan_bp_choose(const uirk_bp_counts *n, int line, int half_images)
{
    const int m = line != 0;
    const size_t cu = (size_t)uirk_plan_device_slots() / 4, p64 = n->p64[m], p32 = n->p32[m];
    const uint64_t w = n->n32_angles[m], wp = n->p32_angles[m]; /* w / wp: slices an item */
    const uint64_t full = (uint64_t)cu * n->a_max[m];           /* one of the longest items a CU */
    const int uneven = 4 * (uint64_t)n->a_max[m] > 5 * (uint64_t)n->a_min[m];
    uirk_bp_choice c = {0, n->all <= 4 * cu, 0};
    const char *env = getenv("UIR_PAIR_MIN_ITEMS"); /* override: 0 pairs always */
    if (env && *env) {
        const size_t least = (size_t)atoi(env);
        c.rows32 = n->all <= least;
        c.pairs = (c.rows32 ? p32 : p64) >= least;
        return c;
    }
    const int enough = line ? w >= (uneven ? 3 : 2) * full : 4 * w > (uneven ? 22 : 17) * full;
    const int shared = line ? 2 * w >= 3 * wp || (4 * w >= 5 * wp && p64 >= 4 * cu)
                            : (half_images && !uneven ? 2 * w >= 3 * wp : 20 * w >= 33 * wp);
    if (n->n32[m] && enough && shared) {
        c.pairs = 1;
        c.rows32 = p32 <= 4 * cu || ((line || uneven) && n->all <= 4 * cu && p32 <= 5 * cu);
        c.angles16 = !line && (c.rows32 ? p32 : p64) > 3 * cu;
    }
    return c;
}

uirk_tile uirk_plan_bp_tile(uirk_tile t, uirk_bp_choice c, int line)
{
    const uirk_tile def = UIRK_TILE_DEFAULT;
    if (line)
        t = def;
    if (c.angles16 && !t.bp_tuned)
        t.bp_angles = 16;
    if (c.rows32)
        t.bp_rows = 32;
    return t;
}

double uirk_fp_item_cost(const uirk_fp_item *it)
{
    return (double)it->na * (double)(it->l_hi - it->l_lo) + 16.0; /* + epilogue */
}

void uirk_plan_xcd(const double *cost, int n, int n_xcd, uirk_xcd_part *out)
{
    memset(out, 0, sizeof *out);
    if (n_xcd < 1)
        n_xcd = 1;
    if (n_xcd > UIRK_MAX_XCD)
        n_xcd = UIRK_MAX_XCD;
    out->n_xcd = n_xcd;
    double total = 0;
    for (int i = 0; i < n; ++i)
        total += cost ? cost[i] : 1.0;
    double acc = 0;
    int x = 1;
    out->start[0] = 0;
    for (int i = 0; i < n && x < n_xcd; ++i) {
        acc += cost ? cost[i] : 1.0;
        while (x < n_xcd && acc >= total * x / n_xcd)
            out->start[x++] = i + 1;
    }
    while (x <= n_xcd)
        out->start[x++] = n;
}

/* A bucket per 1/256 of the range's largest cost (a comparison sort took as
 * long as the planning: 0.6 ms for the 4163 items of 1024 / 720 / 1448); the
 * order within one is the table's.  Without memory the table stays as it is. */
void uirk_plan_sort_fp(uirk_fp_item *v, const uirk_xcd_part *part)
{
    enum { BUCKETS = 256 };
    const int n = part->start[part->n_xcd];
    uirk_fp_item *t = (uirk_fp_item *)malloc(sizeof *t * (size_t)(n > 0 ? n : 1));
    uint8_t *bucket = (uint8_t *)malloc((size_t)(n > 0 ? n : 1));
    for (int x = 0; t && bucket && x < part->n_xcd; ++x) {
        const int i0 = part->start[x], i1 = part->start[x + 1];
        int at[BUCKETS] = {0};
        double most = 0;
        for (int i = i0; i < i1; ++i) {
            const double c = uirk_fp_item_cost(&v[i]);
            most = c > most ? c : most;
        }
        const double scale = BUCKETS / most;
        for (int i = i0; i < i1; ++i) { /* bucket 0: the largest costs */
            const int k = (int)((most - uirk_fp_item_cost(&v[i])) * scale);
            bucket[i] = (uint8_t)(k < BUCKETS ? k : BUCKETS - 1);
            ++at[bucket[i]];
        }
        for (int k = 0, sum = i0; k < BUCKETS; ++k) {
            const int c = at[k];
            at[k] = sum;
            sum += c;
        }
        for (int i = i0; i < i1; ++i)
            t[at[bucket[i]]++] = v[i];
        memcpy(v + i0, t + i0, sizeof *v * (size_t)(i1 - i0));
    }
    free(t);
    free(bucket);
}

int uirk_plan_grid_xcd(const uirk_xcd_part *part, int n_items)
{
    if (n_items <= 0)
        return 0;
    if (!part || part->n_xcd <= 1)
        return n_items;
    int most = 0;
    for (int x = 0; x < part->n_xcd; ++x) {
        const int c = part->start[x + 1] - part->start[x];
        most = c > most ? c : most;
    }
    return (most > 0 ? most : 1) * part->n_xcd;
}
