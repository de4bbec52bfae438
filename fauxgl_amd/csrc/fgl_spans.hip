// fgl_spans.hip -- coverage spans.  After binning, every (tile, raster
// triangle) pair is expanded into one span per row the triangle's box
// reaches inside the tile (for a small box, per row whose pixel centers are
// not all surely outside the triangle): the reference's row walk (context.go:184-221) is
// run for that row, with the row recurrence carried from row to row and the
// per-triangle setup (edge values, steps, reciprocals, context.go:162-181)
// done once per pair.  A span records the first covered pixel inside the
// tile, the edge values the reference held there, and how many consecutive
// pixels are covered.  The tile kernel replays the per-pixel additions from
// those edge values, so every barycentric it uses is bit-identical to the
// reference's serial loop.
#include "fgl_internal.h"
#include "fgl_scan.h"
#include "fgl_tiles.h"
#include "fgl_draws.h"

namespace fgl {
namespace FGL_TILE_NS {

FGL_D const PrimRec *prim_rec(const DrawArgs &a, uint32_t ref) {
    return (ref & REF_SIDE) ? a.side_rec + (ref & ~REF_SIDE) : a.rec_main + ref;
}

FGL_D void tile_rect(const DrawArgs &a, uint32_t t, int32_t &cx0, int32_t &cx1, int32_t &cy0, int32_t &cy1) {
    int32_t tx = (int32_t)(t % (uint32_t)a.ntx), ty = (int32_t)(t / (uint32_t)a.ntx);
    cx0 = tx * TILE_W;
    cy0 = ty * TILE_H;
    cx1 = min(cx0 + TILE_W, a.W) - 1;
    cy1 = min(cy0 + TILE_H, a.H) - 1;
}

// The rows of a pair that get spans.  A triangle whose box is at most 24
// pixels square and whose rows in the tile do not wrap (nk == 1, at most 15
// rows) skips every row whose pixel centers inside the tile are all surely
// outside it (edge_margin): a row whose center line misses the triangle's
// vertical extent, and, in a box at most 8 pixels wide, a row whose centers
// each fail the edge test.  Such a row's span would cover nothing.  Bit r
// stands for row ya + r; ROWS_ALL keeps all nY * nk rows.
constexpr uint16_t ROWS_ALL = 0x8000;

FGL_D uint16_t pair_rows(const PrimRec *pr, const ItemGeo &g, int32_t W, int32_t cx0, int32_t cx1) {
    if (g.nk != 1 || g.nY > 15) return ROWS_ALL;
    const double s0x = pr->sx[0], s0y = pr->sy[0], s1x = pr->sx[1], s1y = pr->sy[1], s2x = pr->sx[2],
                 s2y = pr->sy[2];
    const EdgeMargin m = edge_margin(s0x, s0y, s1x, s1y, s2x, s2y, pr->x0, pr->y0, pr->x1, pr->y1, 23);
    if (!m.ok) return ROWS_ALL;
    const double lo = __builtin_fmin(s0y, __builtin_fmin(s1y, s2y));
    const double hi = __builtin_fmax(s0y, __builtin_fmax(s1y, s2y));
    const int32_t kw = g.kmin * W;
    const int32_t xa = pr->x0 > kw + cx0 ? pr->x0 : kw + cx0;
    const int32_t xb = pr->x1 < kw + cx1 ? pr->x1 : kw + cx1;
    const bool narrow = xb - xa <= 7;
    // the three edge functions (signed by sg) at the center of (xa, ya), and
    // their steps per pixel in x and in y; stepping adds at most 40 roundings
    // of values below 700, far inside tol
    const double px = (double)xa + 0.5, py = (double)g.ya + 0.5;
    double e0 = m.sg * ((s2x - px) * (s1y - py) - (s2y - py) * (s1x - px));  // edge(s1, s2, p)
    double e1 = m.sg * ((s0x - px) * (s2y - py) - (s0y - py) * (s2x - px));  // edge(s2, s0, p)
    double e2 = m.sg * ((s1x - px) * (s0y - py) - (s1y - py) * (s0x - px));  // edge(s0, s1, p)
    const double dx0 = m.sg * (s2y - s1y), dx1 = m.sg * (s0y - s2y), dx2 = m.sg * (s1y - s0y);
    const double dy0 = m.sg * (s1x - s2x), dy1 = m.sg * (s2x - s0x), dy2 = m.sg * (s0x - s1x);
    uint16_t rows = 0;
    for (int32_t r = 0; r < g.nY; r++, e0 += dy0, e1 += dy1, e2 += dy2) {
        if (row_surely_outside(m, lo, hi, g.ya + r)) continue;
        bool any = !narrow;
        double f0 = e0, f1 = e1, f2 = e2;
        for (int32_t x = xa; x <= xb && !any; x++, f0 += dx0, f1 += dx1, f2 += dx2)
            any = !(f0 < -m.tol || f1 < -m.tol || f2 < -m.tol);
        if (any) rows |= (uint16_t)(1u << r);
    }
    return rows;
}

// Spans of pair p: the rows pair_rows keeps (times the wraps).
FGL_D uint32_t pair_spans(const DrawArgs &a, const uint32_t *keys, const uint32_t *vals, uint32_t p, uint16_t &rows) {
    int32_t cx0, cx1, cy0, cy1;
    tile_rect(a, keys[p], cx0, cx1, cy0, cy1);
    const PrimRec *pr = prim_rec(a, vals[p]);
    ItemGeo g = item_geo(pr->x0, pr->y0, pr->x1, pr->y1, a.W, cx0, cx1, cy0, cy1);
    rows = pair_rows(pr, g, a.W, cx0, cx1);
    if (rows != ROWS_ALL) return (uint32_t)__builtin_popcount(rows);
    uint64_t n = (uint64_t)g.nY * (uint64_t)g.nk;
    return n > 0xffffffull ? 0xffffffu : (uint32_t)n;
}

// Spans per pair, summed per group of SPAN_GROUP pairs (a wave's; below 2^30)
// and per block of SPAN_THREADS pairs, whose sums alone are scanned (scanning
// the groups' takes k_span_scan 13.1 us instead of 6.7 for the 871,306-triangle
// mesh at 1080p); also the zeroed fragment counts per span block (the whole
// capacity, grid-wide) that k_spans accumulates into where the fragments are
// written out.
template <class G>
FGL_D void span_count_body(const DrawArgs &a, const G &g) {
    __shared__ uint32_t gsum[SPAN_THREADS / 64];
    if (a.ctr->overflow) return;
    const uint64_t nfb = a.zmode && !a.zpick ? 0 : ((uint64_t)a.span_cap + FRAG_BLOCK - 1) / FRAG_BLOCK;
    for (uint64_t k = (uint64_t)g.bid() * SPAN_THREADS + threadIdx.x; k < nfb; k += (uint64_t)g.nblk() * SPAN_THREADS)
        a.frag_blocksum[k] = 0;
    const uint32_t E = a.ctr->npairs;
    const uint32_t *keys = a.keys[a.sorted_buf];
    const uint32_t *vals = a.vals[a.sorted_buf];
    uint32_t p = g.bid() * SPAN_THREADS + threadIdx.x;
    uint16_t rows = ROWS_ALL;
    uint32_t n = p < E ? pair_spans(a, keys, vals, p, rows) : 0u;
    if (p < E) {
        a.pspans[p] = n;
        a.prows[p] = rows;
    }
    if (g.bid() * SPAN_THREADS >= E) return;
    const uint32_t v = wave_sum(n);
    if ((threadIdx.x & 63) == 0) gsum[threadIdx.x / 64] = a.span_groupsum[p / SPAN_GROUP] = v;
    __syncthreads();
    if (threadIdx.x == 0) a.span_blocksum[g.bid()] = ((uint64_t)gsum[0] + gsum[1]) + ((uint64_t)gsum[2] + gsum[3]);
}
static_assert(SPAN_GROUP == 64 && SPAN_THREADS == 4 * SPAN_GROUP, "a wave's pairs are a group, four groups a block");
FGL_DRAW_KERNELS(k_span_count, span_count_body, __launch_bounds__(SPAN_THREADS))

// Exclusive scan of the per-block span sums (one workgroup), total and
// capacity check.
template <class G>
FGL_D void span_scan_body(const DrawArgs &a, const G &) {
    __shared__ uint64_t lds[SCAN_THREADS / 64];
    if (a.ctr->overflow) return;
    const uint32_t E = a.ctr->npairs;
    const int nb = (int)((E + SPAN_THREADS - 1) / SPAN_THREADS);
    const uint64_t total = scan_block_sums(a.span_blocksum, a.span_blockoff, nb, lds);
    if (threadIdx.x == SCAN_THREADS - 1) {
        if (total > a.span_cap) atomicOr(&a.ctr->overflow, 16u);
        a.ctr->nspans = total > a.span_cap ? a.span_cap : (uint32_t)total;
        a.ctr->spans_lo = (uint32_t)total;
        a.ctr->spans_hi = (uint32_t)(total >> 32);
        if (a.zpick) {
            // pairs of one tile that make it crowded, by the spans a pair has on average
            const uint64_t spans = max((uint64_t)a.crowd_min, total / a.crowd_part);
            const uint64_t pairs = total ? spans * E / total : E;
            a.ctr->crowd_pairs = pairs < E ? (uint32_t)pairs : E;
        }
    }
}
FGL_DRAW_KERNELS(k_span_scan, span_scan_body, __launch_bounds__(SCAN_THREADS))

// edge(a, b, c) (context.go:147-149)
FGL_D double edge(double ax, double ay, double bx, double by, double cx, double cy) {
    return (bx - cx) * (ay - cy) - (by - cy) * (ax - cx);
}

// Per-pair setup a wave shares through LDS: the edge values at the first
// row the tile needs (the row recurrence of context.go:275-277 run up to
// it), the steps, the reciprocals of the skip (context.go:185-206) and the
// box.
struct PairSetup {
    double w0, w1, w2;        // edge values at (x0 + 0.5, ya + 0.5)
    double a12, a20, a01;     // per-pixel steps
    double b12, b20, b01;     // per-row steps
    double ra12, ra20, ra01;  // 1 / a12, 1 / a20, 1 / a01
    double ra;                // 1 / edge(s0, s1, s2)
    int32_t x0, x1, ya, kmin, nk;
    int32_t cx0, cx1, cy0, cy1;
    uint32_t ref;
    uint32_t rows;  // pair_rows of the pair
};

FGL_D void pair_setup(const DrawArgs &a, const uint32_t *keys, const uint32_t *vals, uint32_t p, PairSetup &q) {
    const uint32_t ref = vals[p];
    int32_t cx0, cx1, cy0, cy1;
    tile_rect(a, keys[p], cx0, cx1, cy0, cy1);
    const PrimRec *pr = prim_rec(a, ref);
    const int32_t x0 = pr->x0, y0 = pr->y0, x1 = pr->x1, y1 = pr->y1;
    const ItemGeo g = item_geo(x0, y0, x1, y1, a.W, cx0, cx1, cy0, cy1);
    const double s0x = pr->sx[0], s0y = pr->sy[0], s1x = pr->sx[1], s1y = pr->sy[1], s2x = pr->sx[2],
                 s2y = pr->sy[2];
    // forward differencing variables and reciprocals (context.go:162-181)
    const double px = (double)x0 + 0.5, py = (double)y0 + 0.5;
    double w00 = edge(s1x, s1y, s2x, s2y, px, py);
    double w01 = edge(s2x, s2y, s0x, s0y, px, py);
    double w02 = edge(s0x, s0y, s1x, s1y, px, py);
    q.a01 = s1y - s0y;
    q.b01 = s0x - s1x;
    q.a12 = s2y - s1y;
    q.b12 = s1x - s2x;
    q.a20 = s0y - s2y;
    q.b20 = s2x - s0x;
    q.ra = pr->ra;  // 1 / edge(s0, s1, s2), computed with the record
    q.ra12 = 1.0 / q.a12;
    q.ra20 = 1.0 / q.a20;
    q.ra01 = 1.0 / q.a01;
    // rows y0 .. ya-1 of the row recurrence (context.go:275-277)
    for (int32_t y = y0; y < g.ya; y++) {
        w00 += q.b12;
        w01 += q.b20;
        w02 += q.b01;
    }
    q.w0 = w00;
    q.w1 = w01;
    q.w2 = w02;
    q.x0 = x0;
    q.x1 = x1;
    q.ya = g.ya;
    q.kmin = g.kmin;
    q.nk = g.nk;
    q.cx0 = cx0;
    q.cx1 = cx1;
    q.cy0 = cy0;
    q.cy1 = cy1;
    q.ref = ref;
    q.rows = a.prows[p];
}

// Span m of a pair (row yy = m / nk, wrapped column kk = m % nk, or the m-th
// row pair_rows kept): the row's edge values (yy row steps from ya), the skip
// to the first pixel that can be inside, then the pixel walk of the
// reference's row loop (context.go:185-221) through the tile's columns.
// Returns the span and its covered-pixel count.
//
// The coordinates are finite (a record's box lies within BBOX_LIM), so each
// edge value, the running sum of one step, is monotone along the row, and so
// is the sign of its product with ra.  The pixels inside are therefore one
// run, and left of the tile's columns the additions alone reach the same
// values: a run that ended there leaves only pixels outside.  A wide
// triangle's row is walked from its own start in every tile it crosses, so
// that part was most of the kernel there (200,000-triangle soup at 1920x1080:
// 0.67 ms with the tests made, 0.28 without them and with the shared groups
// below).
FGL_D Span pair_span(const PairSetup &q, uint32_t m, int32_t W, uint32_t &cnt_out) {
    int32_t yy = (int32_t)m, kk = 0;
    if (q.rows != ROWS_ALL) {  // the m-th kept row (nk == 1)
        uint32_t r = q.rows;
        for (uint32_t k = 0; k < m; k++) r &= r - 1;
        yy = __builtin_ctz(r);
    } else if (q.nk != 1) {
        yy = (int32_t)(m / (uint32_t)q.nk);
        kk = (int32_t)(m % (uint32_t)q.nk);
    }
    double w00 = q.w0, w01 = q.w1, w02 = q.w2;
    for (int32_t r = 0; r < yy; r++) {
        w00 += q.b12;
        w01 += q.b20;
        w02 += q.b01;
    }
    const int32_t y = q.ya + yy;
    // skip to the first pixel that can be inside (context.go:185-206)
    double d = 0;
    const double d0 = -w00 * q.ra12;
    const double d1 = -w01 * q.ra20;
    const double d2 = -w02 * q.ra01;
    if (w00 < 0 && d0 > d) d = d0;
    if (w01 < 0 && d1 > d) d = d1;
    if (w02 < 0 && d2 > d) d = d2;
    // int(d) and back; a d past int64 converts to its minimum, which the
    // reference replaces by 0, and one past int32 lies right of the box
    if (!(d < 9223372036854775808.0)) d = 0;
    const bool far = d >= 2147483647.0;
    const int32_t id = far ? 0 : (int32_t)d;
    d = (double)id;
    double w0 = w00 + q.a12 * d;
    double w1 = w01 + q.a20 * d;
    double w2 = w02 + q.a01 * d;
    const int32_t xs = (far || id > q.x1 - q.x0) ? q.x1 + 1 : q.x0 + id;
    const int32_t k = q.kmin + kk;
    const int32_t kw = k * W;
    const int32_t pyk = y + k;
    const int32_t xa = q.x0 > kw + q.cx0 ? q.x0 : kw + q.cx0;
    const int32_t xb = q.x1 < kw + q.cx1 ? q.x1 : kw + q.cx1;
    Span sp;
    sp.w[0] = 0;
    sp.w[1] = 0;
    sp.w[2] = 0;
    sp.ref = q.ref;
    sp.pix = 0;
    sp.n = 0;
    uint32_t cnt = 0;
    if (pyk >= q.cy0 && pyk <= q.cy1 && xa <= xb && xs <= xb) {
        const double a12 = q.a12, a20 = q.a20, a01 = q.a01, ra = q.ra;
        const int32_t left = xa - xs;  // pixels left of the tile
#pragma unroll 8
        for (int32_t j = 0; j < left; j++) {
            w0 += a12;
            w1 += a20;
            w2 += a01;
        }
        int32_t x = xs > xa ? xs : xa;
        int32_t first = x;
        for (; x <= xb; x++) {
            // all three products before any branch: testing them one by one
            // costs a third of the kernel (0.28 -> 0.40 ms on the soup)
            const bool o0 = w0 * ra < 0, o1 = w1 * ra < 0, o2 = w2 * ra < 0;
            const bool out = o0 || o1 || o2;
            if (out && cnt) break;
            if (!out) {
                if (cnt == 0) {
                    sp.w[0] = w0;
                    sp.w[1] = w1;
                    sp.w[2] = w2;
                    first = x;
                }
                cnt++;
            }
            w0 += a12;
            w1 += a20;
            w2 += a01;
        }
        if (cnt) sp.pix = (uint16_t)((pyk - q.cy0) * TILE_W + (first - kw - q.cx0));
        sp.n = (uint16_t)(cnt | (k == 0 ? SPAN_INB : 0u));
    }
    cnt_out = cnt;
    return sp;
}

// The spans of a group of SPAN_GROUP pairs, 64 at a time, one span per lane,
// so lanes share the walks evenly however many rows each pair has, and the
// covered pixels of each window added to the fragment counts of the (one or
// two) FRAG_BLOCKs of the span list it lies in.  A lane finds its span's pair
// as the shading kernel finds a fragment's span (each pair marks its first
// span's window position, a max-scan carries the mark) and reads the pair's
// setup from LDS.  The calling wave takes windows w0, w0 + dw, ...; n, excl:
// its lane's pair's spans and their position in the group's T.  Where no
// fragments are written out (zmode) the counts are summed in *frags instead
// (zpick: too).
FGL_D void group_windows(const DrawArgs &a, const PairSetup *setup, uint32_t *ostart, uint64_t gbase, uint32_t n,
                         uint32_t excl, uint32_t T, uint32_t w0, uint32_t dw, uint64_t *frags) {
    const int lane = threadIdx.x & 63;
    for (uint32_t base = w0 * 64; base < T; base += dw * 64) {
        // the pair of the window's first span: the last pair that starts at
        // or before it (pairs without spans start nowhere)
        const uint64_t before = __ballot(n && excl <= base);
        const uint32_t carry = 64u - (uint32_t)__builtin_clzll(before);
        ostart[lane] = 0;
        if (n && excl > base && excl - base < 64) ostart[excl - base] = (uint32_t)lane + 1;
        __builtin_amdgcn_wave_barrier();
        uint32_t om = wave_incl_max(ostart[lane]);
        om = om ? om : carry;
        __builtin_amdgcn_wave_barrier();
        const uint32_t q = base + (uint32_t)lane;
        const int ow = (int)om - 1;
        const uint32_t oexcl = __shfl(excl, ow);
        const uint64_t blk = (gbase + base) / FRAG_BLOCK;
        uint32_t cnt = 0;
        if (q < T) {
            const Span sp = pair_span(setup[ow], q - oexcl, a.W, cnt);
            a.spans[gbase + q] = sp;
        }
        // both blocks' counts (at most 64 * 128 each) in one sum
        if ((gbase + q) / FRAG_BLOCK != blk) cnt <<= 16;
        const uint32_t both = wave_sum(cnt);
        if (a.zmode) {
            *frags += (both & 0xffffu) + (both >> 16);
            if (!a.zpick) continue;
        }
        const uint32_t part = lane == 0 ? both & 0xffffu : both >> 16;
        if (lane < 2 && part) atomicAdd((unsigned long long *)&a.frag_blocksum[blk + lane], (unsigned long long)part);
    }
}

// Groups of SPAN_GROUP pairs, one pair per lane to set up.  A wave takes a
// group to itself where there are many groups of few spans (the small
// triangles of a dense mesh); where pairs average more than SPAN_SHARE spans,
// or the groups are too few to fill the GPU, a workgroup's four waves share a
// group's windows: a 12-triangle cube over four tiles has one group of 640
// spans, which one wave alone took 33 us to walk (now 12; a sphere and a cube
// at 512x512 95 -> 22 us).
constexpr uint32_t SPAN_SHARE = 12;
constexpr uint32_t SPAN_FEW = 2048;       // groups
// Workgroups of a draw, each looping over the groups past the grid; a launch
// for many draws gives each fewer, as most draws have few groups and every
// block costs its dispatch.
constexpr uint32_t SPANS_GRID_MAX = 16384, SPANS_GRID_MANY = 256;

template <class G>
FGL_D void spans_body(const DrawArgs &a, const G &g) {
    __shared__ uint32_t ostart[SPAN_THREADS / 64][64];
    __shared__ PairSetup setup[SPAN_THREADS / 64][64];
    __shared__ uint64_t wfrags[SPAN_THREADS / 64];
    if (a.ctr->overflow) return;
    const uint32_t E = a.ctr->npairs, NS = a.ctr->nspans;
    const uint32_t ngroups = (E + SPAN_GROUP - 1) / SPAN_GROUP;
    const uint32_t *keys = a.keys[a.sorted_buf];
    const uint32_t *vals = a.vals[a.sorted_buf];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr uint32_t WAVES = SPAN_THREADS / 64;
    const bool share = ngroups <= SPAN_FEW || NS / SPAN_SHARE > E;
    const uint32_t wg_first = share ? g.bid() : g.bid() * WAVES;
    const uint32_t first = share ? wg_first : wg_first + (uint32_t)wave;
    const uint32_t step = share ? g.nblk() : g.nblk() * WAVES;
    const int slot = share ? 0 : wave;
    uint64_t frags = 0;
    const uint32_t crowd = a.zpick ? a.ctr->crowd_pairs : E;
    for (uint32_t grp = first; grp < ngroups; grp += step) {
        const uint32_t p = grp * SPAN_GROUP + (uint32_t)lane;
        const uint32_t n = p < E ? a.pspans[p] : 0u;
        uint64_t v = n;
        for (int off = 1; off < 64; off <<= 1) {
            const uint64_t y = __shfl_up(v, off);
            if (lane >= off) v += y;
        }
        const uint4 gs = reinterpret_cast<const uint4 *>(a.span_groupsum)[grp / 4];  // its block's groups
        const uint32_t k = grp % 4;
        const uint64_t gbase = a.span_blockoff[grp / 4] + (k > 0 ? gs.x : 0u) + (k > 1 ? gs.y : 0u) + (k > 2 ? gs.z : 0u);
        const uint32_t excl = (uint32_t)(v - n);
        const uint32_t T = (uint32_t)__shfl(v, 63);
        if (!share || wave == 0) {
            if (p < E) {
                // the first and the last pair of a tile bound its spans
                const uint32_t t = keys[p];
                if (lane == 0 && crowd < E - p && keys[p + crowd] == t) a.ctr->crowded = 1u;
                if (p == 0 || keys[p - 1] != t) a.tstart[t] = (uint32_t)(gbase + excl);
                if (p + 1 == E || keys[p + 1] != t) a.tend[t] = (uint32_t)(gbase + excl) + n;
            }
            if (n) pair_setup(a, keys, vals, p, setup[slot][lane]);
        }
        if (share) __syncthreads();
        else __builtin_amdgcn_wave_barrier();
        group_windows(a, setup[slot], ostart[wave], gbase, n, excl, T, share ? (uint32_t)wave : 0u, share ? WAVES : 1u,
                      &frags);
        if (share) __syncthreads();  // the setups are read before the next group's are written
    }
    if (a.zmode && wg_first < ngroups) {
        // one addition a workgroup: one a wave, all to the same few cache
        // lines, took 8 us of the 871,306-triangle mesh's 34 at 1080p
        if (lane == 0) wfrags[wave] = frags;
        __syncthreads();
        if (threadIdx.x == 0)
            atomicAdd(&a.ctr->ftot[g.bid() % 64], (unsigned long long)((wfrags[0] + wfrags[1]) + (wfrags[2] + wfrags[3])));
    }
}
FGL_DRAW_KERNELS(k_spans, spans_body, __launch_bounds__(SPAN_THREADS))

uint32_t span_blocks(const DrawArgs &a) {
    return (uint32_t)(((uint64_t)a.pair_cap + SPAN_THREADS - 1) / SPAN_THREADS);
}
uint32_t spans_blocks(const DrawArgs &a, bool many) {
    const uint64_t groups = ((uint64_t)a.pair_cap + SPAN_GROUP - 1) / SPAN_GROUP;
    const uint32_t most = many ? SPANS_GRID_MANY : SPANS_GRID_MAX;
    return (uint32_t)(groups < most ? groups : most);
}

hipError_t launch_span_count(const DrawArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_span_count, dim3(span_blocks(a)), dim3(SPAN_THREADS), 0, s, a);
    return hipGetLastError();
}
hipError_t launch_span_scan(const DrawArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_span_scan, dim3(1), dim3(SCAN_THREADS), 0, s, a);
    return hipGetLastError();
}
hipError_t launch_spans(const DrawArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_spans, dim3(spans_blocks(a, false)), dim3(SPAN_THREADS), 0, s, a);
    return hipGetLastError();
}
hipError_t launch_span_count_multi(const MultiArgs &m, uint32_t nb, const DrawArgs &, hipStream_t s) {
    hipLaunchKernelGGL(k_span_count_m, dim3(nb), dim3(SPAN_THREADS), 0, s, m);
    return hipGetLastError();
}
hipError_t launch_span_scan_multi(const MultiArgs &m, uint32_t nb, const DrawArgs &, hipStream_t s) {
    hipLaunchKernelGGL(k_span_scan_m, dim3(nb), dim3(SCAN_THREADS), 0, s, m);
    return hipGetLastError();
}
hipError_t launch_spans_multi(const MultiArgs &m, uint32_t nb, const DrawArgs &, hipStream_t s) {
    hipLaunchKernelGGL(k_spans_m, dim3(nb), dim3(SPAN_THREADS), 0, s, m);
    return hipGetLastError();
}

}  // namespace FGL_TILE_NS
}  // namespace fgl
