// On-chip ("resident") execution of the FDTD steps: the plan that splits a
// unit's padded grid over workgroups and a workgroup's rows over its
// wavefronts.  Plain C++ (host, and the slab geometry on the device).
//
// A unit (one sample's shot) is cut into `slabs` row ranges, one workgroup
// each.  The workgroup keeps p0 and p1 of its rows in LDS for a whole run of
// time steps; neighbouring slabs exchange their edge rows through memory.
// Within a slab the columns fall into
//   * `strips` interior strips of 64 columns (one per lane) over
//     [wl, ntx - wr): never near the left or right absorbing band;
//   * the left and right side blocks, wl and wr columns wide (band + the 4
//     cells its extrapolation reads inward, so a side block never reads
//     another wave's p0), whose points are taken 64 at a time.
// Rows within zt = pml + 4 of the top or bottom edge (the z absorbing band
// and the 4 rows it reads inward) are marched inward from the edge: the new
// field overwrites p0 in place, and a row's inward p0 reads then precede the
// overwrite of those rows.  Where the zone is cut between wavefronts, the
// inner piece holds the results of its first four rows back until every wave
// has computed (ResItem::hold).  All items are dealt to the wavefronts so that the
// four SIMDs carry equal work.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace gpvi {

constexpr int kResWaves = 16;        // wavefronts of a workgroup
constexpr int kResThreads = 64 * kResWaves;
constexpr int kResItems = 7;         // items per wavefront, at most
constexpr int kResZBlock = 2;        // band rows of a strip computed together
constexpr int kResBandSlabs = 3;     // slabs the z band of one edge may span
constexpr int kResTables = kResBandSlabs + 1;
constexpr int kResMaxSlabs = 32;
constexpr int kResCus = 256;         // CUs that plans and their times are made for
constexpr int kResLdsBytes = 160 * 1024;
constexpr unsigned kResGone = 0x80000000u;   // in a cluster's count of arrived workgroups: given up
constexpr int kResLdsFront = 16 + 2 * kResWaves * kResItems + 32;   // words before the first buffer: ticket, items, taper
constexpr int kResLdsBack = 16;      // floats after the last one

enum ResKind : int { kResStrip = 0, kResStripZ = 1, kResSide = 2, kResSideZ = 3 };

// rows start, start + step, ... (count of them, step +-1) of a slab's rows;
// x0: the strip's first column, or the side (0 left, 1 right); hold: the first
// block's results are stored only after every wave has computed.
struct ResItem {
    uint16_t x0;
    int8_t step;
    uint8_t kind : 4, hold : 4;
    uint16_t start, count;
};
static_assert(sizeof(ResItem) == 8, "items travel as kernel arguments");

struct ResPlan {
    int slabs, nband;              // nband: slabs at each edge that hold band rows (explicit heights)
    int band_rows[kResBandSlabs];  // their heights, from the edge
    int strips, wl, wr, zt, hr;    // hr: halo rows exchanged per side
    int mid_rows;                  // height of the tallest other slab
    int lds_bytes;
    int two_phase[kResTables];     // stores that wait for a barrier: held blocks, or p0 read in the halo
    ResItem item[kResTables][kResWaves][kResItems];  // table t < nband: band slab t, nband: the others
};

// Slab g: first row, rows, its table, whether its rows are counted from the
// bottom (flip), and whether it is one row shorter than its table.
struct ResSlab {
    int z0, n, table, flip, shorter;
};

#ifdef __HIPCC__
#define GPVI_RES_FN __host__ __device__ inline
#else
#define GPVI_RES_FN inline
#endif

// Plain rows of a strip computed together (the wider stencils hold more
// neighbours per row in registers).
GPVI_RES_FN constexpr int res_row_block(int lc) { return lc <= 5 ? 4 : 2; }

GPVI_RES_FN ResSlab res_slab(const ResPlan& p, int ntz, int g)
{
    ResSlab s;
    s.flip = 0;
    s.shorter = 0;
    if (p.slabs == 1) {
        s.z0 = 0; s.n = ntz; s.table = 0;
        return s;
    }
    int base = 0;
    for (int i = 0; i < p.nband; ++i) base += p.band_rows[i];
    const int nmid = p.slabs - 2 * p.nband;
    const int below = p.slabs - 1 - g;
    if (g < p.nband || below < p.nband) {
        const int i = g < p.nband ? g : below;
        int off = 0;
        for (int j = 0; j < i; ++j) off += p.band_rows[j];
        s.n = p.band_rows[i];
        s.table = i;
        if (g < p.nband) {
            s.z0 = off;
        } else {
            // without other slabs the two halves meet: an odd grid's lower half is one row shorter
            if (nmid == 0 && i == p.nband - 1 && 2 * base > ntz) { s.n -= 1; s.shorter = 1; }
            s.z0 = ntz - off - s.n;
            s.flip = 1;
        }
        return s;
    }
    const int m = ntz - 2 * base, i = g - p.nband;
    s.z0 = base + i * m / nmid;
    s.n = base + (i + 1) * m / nmid - s.z0;
    s.table = p.nband;
    s.shorter = s.n < p.mid_rows;
    return s;
}

// An item of slab s as absolute slab rows (start, step, count).
GPVI_RES_FN void res_item_rows(const ResSlab& s, const ResItem& it, int* start, int* step, int* count)
{
    int a = it.start, d = it.step, c = it.count;
    if (s.shorter) {
        if (d < 0 && a == s.n) {          // began on the row this slab lacks
            a -= 1;
            c -= 1;
        } else if (d > 0 && a + c == s.n + 1) {
            c -= 1;
        }
    }
    if (c <= 0) {   // the row was the item's only one (its start may lie outside the slab)
        *start = 0; *step = 1; *count = 0;
        return;
    }
    if (s.flip) {
        a = s.n - 1 - a;
        d = -d;
    }
    *start = a; *step = d; *count = c;
}

// An item as the two words that a wavefront reads in every step, and back.
GPVI_RES_FN void res_pack_item(const ResItem& it, int start, int step, int count, unsigned* w0, unsigned* w1)
{
    *w0 = (unsigned)it.x0 | (unsigned)it.kind << 16 | (step < 0 ? 1u << 18 : 0u) | (unsigned)it.hold << 19 |
          (it.count ? 1u << 20 : 0u);
    *w1 = ((unsigned)start & 0xffffu) | (unsigned)count << 16;
}

struct ResWords {
    bool present, hold;
    int x0, kind, step, start, count;
};
GPVI_RES_FN ResWords res_unpack_item(unsigned w0, unsigned w1)
{
    ResWords r;
    r.present = w0 >> 20 & 1;
    r.hold = w0 >> 19 & 1;
    r.step = w0 >> 18 & 1 ? -1 : 1;
    r.kind = (int)(w0 >> 16) & 3;
    r.x0 = (int)(w0 & 0xffff);
    r.start = (int)(w1 & 0xffff);
    r.count = (int)(w1 >> 16);
    return r;
}

// ---------------------------------------------------------------------------
// Host side: building a plan.  Costs are in units of one 64-point interior
// row of one wavefront; the values are the best over 18 batches of a random
// search (within 8 % of the best plan of each).

struct ResGeom {
    int ntx, ntz, lc, pml;
};

namespace res_detail {

constexpr double kRow = 1.0, kRowZ = 2.55, kRowEdge = 0.3, kSide = 3.19, kSideZ = 3.3, kItem = 2.0;
constexpr double kWave = 2.38, kHold = 3.0, kFixed = 4.0, kHalo = 0.9;

struct Work {
    ResItem it;
    double cost;
};
constexpr int kMaxWork = kResWaves * kResItems;   // items of a slab

// Deal the items to the waves (wave w runs on SIMD w % 4): longest first, to
// the least loaded SIMD and its least loaded wave, at most one held item per
// wave.  Returns the makespan (a lone wave fills a third of its SIMD's issue
// slots), < 0: it does not fit.
inline double deal(const Work* w, int n, ResItem (*out)[kResItems])
{
    int order[kMaxWork];
    for (int i = 0; i < n; ++i) order[i] = i;
    std::stable_sort(order, order + n, [&](int a, int b) {
        return w[a].it.hold != w[b].it.hold ? w[a].it.hold > w[b].it.hold : w[a].cost > w[b].cost;
    });
    double simd[4] = {0, 0, 0, 0}, wave[kResWaves] = {0};
    int cnt[kResWaves] = {0};
    bool held[kResWaves] = {false};
    for (int v = 0; v < kResWaves; ++v)
        for (int i = 0; i < kResItems; ++i) out[v][i] = ResItem{0, 1, 0, 0, 0, 0};
    for (int i = 0; i < n; ++i) {
        const Work& x = w[order[i]];
        int best = -1;
        for (int v = 0; v < kResWaves; ++v) {
            if (cnt[v] == kResItems || (x.it.hold && held[v])) continue;
            if (best < 0 || simd[v % 4] < simd[best % 4] || (v % 4 == best % 4 && wave[v] < wave[best]) ||
                (simd[v % 4] == simd[best % 4] && wave[v] < wave[best]))
                best = v;
        }
        if (best < 0) return -1;
        out[best][cnt[best]++] = x.it;
        wave[best] += x.cost;
        simd[best % 4] += x.cost;
        if (x.it.hold) held[best] = true;
    }
    double m = 0;
    for (int s = 0; s < 4; ++s) m = std::max(m, simd[s]);
    for (int v = 0; v < kResWaves; ++v) m = std::max(m, kWave * wave[v]);
    return m;
}

// Cost of `r` rows of a strip's z zone, the first one d rows from the edge.
inline double zone_cost(const ResGeom& g, int d, int r)
{
    double c = 0;
    int e = 0;
    for (; e < r && d + e < g.lc; ++e) c += kRowEdge;
    while (e < r && d + e < g.pml) {
        c += kRowZ * kResZBlock;
        e += std::min(kResZBlock, std::min(r - e, g.pml - d - e));
    }
    const int left = r - e;
    const int rb = res_row_block(g.lc);
    return c + kRow * ((left + rb - 1) / rb * rb);
}

// A slab of n rows, the first one z0 rows from the edge: rows [0, tb) are z
// rows, and so are the last be rows (a whole-grid slab).  Its z items, each
// strip's z rows in `strip` pieces and each side's in `side`, marched inward.
// Pieces after the first hold their first four rows back (all of a shorter
// one), and those lie in the band.  A cut is the one nearest to an equal share
// of the cost or, late, the last one not far past it.  < 0: no such pieces.
// Short pieces matter where few units leave most wavefronts idle and the
// longest item is the step: with at least four rows in every later piece a
// call on 120x200 with 4 shots took 11.8 ms instead of 9.7, 15 units of 61x97
// 4.41 instead of 4.04.
inline int zone_items(const ResGeom& g, const ResPlan& p, int z0, int n, int tb, int be, int strip, int side_pieces,
                      bool late, Work* out, bool* held)
{
    int c = 0;
    *held = false;
    for (int col = 0; col < p.strips + 2; ++col) {
        const bool side = col >= p.strips;
        const int x0 = side ? col - p.strips : p.wl + 64 * col;
        const int wd = side ? (x0 ? p.wr : p.wl) : 64;
        for (int edge = 0; edge < 2; ++edge) {
            const int rows = edge ? be : tb, d0 = edge ? 0 : z0;
            const int want = side ? side_pieces : strip;
            int done = 0;
            for (int i = 0; i < want && done < rows; ++i) {
                int r = rows - done;
                const int at = d0 + done;
                if (i + 1 < want) {
                    const double share = zone_cost(g, at, r) / (want - i);
                    int cut = -1;
                    double off = 0;
                    for (int e = late ? 4 : 1; e < r; ++e) {
                        const int d = at + e, rest = i + 2 == want ? r - e : 2;
                        if (d < g.lc || d + std::min(4, rest) > g.pml || (i > 0 && at + std::min(4, e) > g.pml)) continue;
                        if (!side && (d - std::max(g.lc, at)) % kResZBlock) continue;   // (whole band blocks)
                        const double cost = zone_cost(g, at, e), o = std::abs(cost - share);
                        if (cut < 0 || (late ? cost <= share + kRowZ : o < off)) {
                            cut = e;
                            off = o;
                        }
                    }
                    if (cut > 0) r = cut;
                }
                if (i > 0 && at + std::min(4, r) > g.pml) return -1;
                if (c == kMaxWork) return -1;
                Work& w = out[c++];
                w.it = ResItem{(uint16_t)x0, (int8_t)(edge ? -1 : 1), (uint8_t)(side ? kResSideZ : kResStripZ),
                               (uint8_t)(i > 0), (uint16_t)(edge ? n - 1 - done : done), (uint16_t)r};
                w.cost = kItem + (side ? kSideZ * ((r * wd + 63) / 64) : zone_cost(g, at, r));
                if (i > 0) *held = true;
                done += r;
            }
        }
    }
    return c;
}

// The slab's other items behind the c already there.
inline int plain_items(const ResGeom& g, const ResPlan& p, int n, int tb, int be, int strip, int side_pieces, Work* out,
                       int c)
{
    const int m = n - tb - be;
    if (m <= 0) return c;
    for (int col = 0; col < p.strips + 2; ++col) {
        const bool side = col >= p.strips;
        const int x0 = side ? col - p.strips : p.wl + 64 * col;
        const int wd = side ? (x0 ? p.wr : p.wl) : 64;
        const int unit = side ? 1 : res_row_block(g.lc);      // rows advanced at a time
        const int blocks = (m + unit - 1) / unit;
        const int k = std::min(side ? side_pieces : strip, blocks);
        int done = 0;
        for (int i = 0; i < k; ++i) {
            // the first pieces march down from the top, the last one up from
            // the bottom, so a slab's edge rows are computed (and sent) first
            const int b = (i + 1) * blocks / k - i * blocks / k;
            const int rows = i == k - 1 ? m - done : std::min(m - done, b * unit);
            const bool up = i == k - 1 && k > 1;
            if (c == kMaxWork) return -1;
            Work& w = out[c++];
            w.it = ResItem{(uint16_t)x0, (int8_t)(up ? -1 : 1), (uint8_t)(side ? kResSide : kResStrip), 0,
                           (uint16_t)(up ? tb + done + rows - 1 : tb + done), (uint16_t)rows};
            w.cost = kItem + (side ? kSide * ((rows * wd + 63) / 64) : kRow * ((rows + unit - 1) / unit * unit));
            done += rows;
        }
    }
    return c;
}

// What the items' cost alone makes of a step: equal shares on four SIMDs, and
// the longest item's wavefront.
inline double least_cost(const Work* w, int n)
{
    double sum = 0, top = 0;
    for (int i = 0; i < n; ++i) {
        sum += w[i].cost;
        top = std::max(top, w[i].cost);
    }
    return std::max(sum / 4, kWave * top);
}

// The cheapest dealing of a slab's items; < 0: none costs less than `limit`.
inline double best_table(const ResGeom& g, const ResPlan& p, int z0, int n, int tb, int be,
                         ResItem (*out)[kResItems], int* held, double limit)
{
    double best = -1;
    Work w[kMaxWork];
    ResItem tmp[kResWaves][kResItems];
    const int most = tb + be > 0 ? 5 : 1;
    for (int zs = 1; zs <= most; ++zs)
        for (int zd = 1; zd <= most; ++zd)
            for (int late = 0; late < (zs > 1 || zd > 1 ? 2 : 1); ++late) {
                bool h;
                const int nz = zone_items(g, p, z0, n, tb, be, zs, zd, late != 0, w, &h);
                const double wait = h ? kHold : 0.0;
                if (nz < 0 || least_cost(w, nz) + wait >= limit) continue;
                for (int strip = 1; strip <= 16; strip = strip < 4 ? strip + 1 : strip * 2)
                    for (int side = 1; side <= 8; side *= 2) {
                        const int c = plain_items(g, p, n, tb, be, strip, side, w, nz);
                        if (c < 0 || least_cost(w, c) + wait >= limit) continue;
                        const double d = deal(w, c, tmp), m = d + wait;
                        if (d < 0 || m >= limit) continue;
                        best = limit = m;
                        *held = h ? 1 : 0;
                        for (int v = 0; v < kResWaves; ++v)
                            for (int i = 0; i < kResItems; ++i) out[v][i] = tmp[v][i];
                    }
            }
    return best;
}

}  // namespace res_detail

inline int res_lds_bytes(int ntx, int rows, int hr)
{
    return 4 * (kResLdsFront + kResLdsBack + 2 * (rows + 2 * hr) * ntx);
}

// Column split: widths of the side blocks and the number of strips.  False
// where the grid is too narrow, or its band too wide, for the item kinds.
inline bool res_columns(const ResGeom& g, ResPlan* p)
{
    const int lo = std::max(g.pml + 4, 8);
    double best = -1;
    for (int wl = lo; wl <= 32; ++wl)
        for (int wr = wl; wr <= 32; ++wr) {
            const int inner = g.ntx - wl - wr;
            if (inner < 1) continue;
            const int n = (inner + 63) / 64;
            if (2 * (n + 1) > 2 * kResWaves) continue;   // a wave receives two blocks of halo rows at most
            const double cost = n * res_detail::kRow + res_detail::kSide * (wl + wr) / 64.0;
            if (best < 0 || cost < best - 1e-9) {
                best = cost;
                p->strips = n;
                p->wl = wl;
                p->wr = wr;
            }
        }
    return best >= 0;
}

namespace res_detail {

// Cost of grid row z.
inline double row_cost(const ResGeom& g, const ResPlan& p, int z)
{
    const int d = std::min(z, g.ntz - 1 - z);
    return p.strips * (d < g.lc ? kRowEdge : d < g.pml ? kRowZ : kRow) +
           (p.wl + p.wr) / 64.0 * (d < g.pml + 4 ? kSideZ : kSide);
}

inline double grid_cost(const ResGeom& g, const ResPlan& p)
{
    double t = 0;
    for (int z = 0; z < g.ntz; ++z) t += row_cost(g, p, z);
    return t;
}

}  // namespace res_detail

// Cost of a step of the whole grid (0: no plan).
inline double res_work(const ResGeom& g)
{
    ResPlan p = {};
    return res_columns(g, &p) ? res_detail::grid_cost(g, p) : 0;
}

// What a step costs beside its rows: barriers and bookkeeping, and the halo
// rows sent and awaited (over four SIMDs).
inline double res_fixed(const ResGeom& g, int slabs)
{
    using namespace res_detail;
    return kFixed + (slabs > 1 ? kHalo * 2 * std::max(g.lc - 1, 4) * g.ntx / 256.0 : 0.0);
}

// A plan with `slabs` slabs; its step cost (makespan of the busiest slab), or
// < 0 when it does not fit or cannot cost less than `limit`.
inline double res_make_plan(const ResGeom& g, int slabs, ResPlan* p, double limit = 1e300)
{
    using namespace res_detail;
    p->slabs = slabs;
    p->zt = g.pml + 4;
    p->hr = std::max(g.lc - 1, 4);
    if (g.ntz < 2 * p->zt || slabs < 1 || slabs > kResMaxSlabs || !res_columns(g, p)) return -1;
    const double total = grid_cost(g, *p);
    for (int t = 0; t < kResTables; ++t)
        for (int v = 0; v < kResWaves; ++v)
            for (int i = 0; i < kResItems; ++i) p->item[t][v][i] = ResItem{0, 1, 0, 0, 0, 0};
    for (int t = 0; t < kResTables; ++t) p->two_phase[t] = 0;
    if (slabs == 1) {
        p->nband = 0;
        p->mid_rows = g.ntz;
        p->lds_bytes = res_lds_bytes(g.ntx, g.ntz, p->hr);
        if (p->lds_bytes > kResLdsBytes) return -1;
        return best_table(g, *p, 0, g.ntz, p->zt, p->zt, p->item[0], &p->two_phase[0], limit);
    }
    // Boundaries at equal shares of the rows' cost, from the edge inward.
    const double share = total / slabs;
    const int most = (kResLdsBytes / 4 - kResLdsFront - kResLdsBack) / (2 * g.ntx) - 2 * p->hr;
    const int least = p->hr + 1;   // also for a slab one row shorter
    int z = 0, nband = 0;
    double cum = 0;
    while (z < p->zt) {
        if (nband == kResBandSlabs || 2 * (nband + 1) > slabs) return -1;
        int n = 0;
        const double want = share * (nband + 1);
        while (z + n < g.ntz && (n < least || cum + 0.5 * row_cost(g, *p, z + n) < want)) cum += row_cost(g, *p, z + n++);
        // the last slab of the upper half reaches the middle
        if (2 * (nband + 1) == slabs) n = (g.ntz + 1) / 2 - z;
        if (2 * (z + n) > g.ntz + 1) n = (g.ntz + 1) / 2 - z;
        if (n < least || n > most) return -1;
        p->band_rows[nband++] = n;
        z += n;
        if (2 * nband == slabs && 2 * z < g.ntz) return -1;
    }
    p->nband = nband;
    const int nmid = slabs - 2 * nband, m = g.ntz - 2 * z;
    if (nmid < 0 || (nmid == 0 && m > 0) || (nmid > 0 && m < nmid * least)) return -1;
    p->mid_rows = nmid ? (m + nmid - 1) / nmid : 0;
    if (p->mid_rows > most) return -1;
    int tallest = p->mid_rows;
    double cost = 0;
    int z0 = 0;
    for (int i = 0; i < nband; ++i) {
        const int n = p->band_rows[i], tb = std::max(0, std::min(n, p->zt - z0));
        double c = best_table(g, *p, z0, n, tb, 0, p->item[i], &p->two_phase[i], limit);
        if (c < 0) return -1;
        if (z0 + n < p->zt) p->two_phase[i] = 1;   // its z rows read p0 in the halo
        cost = std::max(cost, c);
        tallest = std::max(tallest, n);
        z0 += n;
    }
    if (nmid) {
        int h;
        const double c = best_table(g, *p, z0, p->mid_rows, 0, 0, p->item[nband], &h, limit);
        if (c < 0) return -1;
        cost = std::max(cost, c);
    }
    p->lds_bytes = res_lds_bytes(g.ntx, tallest, p->hr);
    return p->lds_bytes <= kResLdsBytes ? cost : -1;
}

// Which plans may run.  Launches on different hardware queues run at the same
// time, each with at most one cluster of which only some slabs have a CU: with
// queues (slabs - 1) < cus one is always left for a missing slab.  A stream or
// device with fewer CUs than a plan is made for keeps the step launches: the
// plan's time does not hold there, and streams with a CU mask have hardware
// queues of their own beside the counted ones.
inline bool res_admits(int slabs, int queues, int cus)
{
    return slabs >= 1 && cus >= kResCus && (long long)queues * (slabs - 1) < cus;
}

// The most slabs that are admitted on a whole chip.
inline int res_slab_limit(int queues) { return std::min(kResMaxSlabs, (kResCus - 1) / std::max(1, queues) + 1); }

// Rounds a launch takes over `units` units in `slabs` slabs each on `cus` CUs.
inline double res_rounds(int units, int slabs, int cus)
{
    const int at_once = std::max(1, cus / slabs);
    return (double)((units + at_once - 1) / at_once);
}

// The plan of least time, with at most `most` slabs; its cost (fixed part
// included, all rounds), or < 0: none fits.  Slab counts are tried in the
// order of a lower bound on their time (equal work on every SIMD); the search
// ends where the bound passes the best plan found.
inline double res_select_plan(const ResGeom& g, int units, int cus, int most, ResPlan* plan)
{
    const double work = res_work(g) / 4;
    auto bound = [&](int slabs) { return res_rounds(units, slabs, cus) * (res_fixed(g, slabs) + work / slabs); };
    int order[kResMaxSlabs];
    for (int i = 0; i < kResMaxSlabs; ++i) order[i] = i + 1;
    std::stable_sort(order, order + kResMaxSlabs, [&](int a, int b) { return bound(a) < bound(b); });
    double best = 1e300;
    for (int slabs : order) {
        if (bound(slabs) >= best) break;
        if (slabs > most) continue;
        ResPlan p;
        const double rounds = res_rounds(units, slabs, cus);
        const double c = res_make_plan(g, slabs, &p, best / rounds - res_fixed(g, slabs));
        if (c < 0) continue;
        best = rounds * (res_fixed(g, slabs) + c);
        *plan = p;
    }
    return best < 1e300 ? best : -1;
}

}  // namespace gpvi
