// Resident FDTD steps for gfx950: one launch advances every unit of a batch
// by many time steps of one pass with p0 and p1 of the whole grid on the chip
// (fwi2d_resident.h has the split into slabs and items).
//
// Per step a workgroup computes its rows from p1 (read only) and writes the
// new field over p0, in LDS; one barrier ends the step and the two buffers
// swap roles.  The first and last rows of a slab go to its neighbours as
// 64-bit words {value, step tag} in memory: a relaxed agent-scope atomic
// store, and on the other side a load that is repeated until the tag is this
// step's.  Value and tag travel in one word, so no fence orders them.  Two
// words per point, used by odd and even steps: a slab overwrites a word two
// steps later, which it can only reach after its neighbour has sent a step
// computed from that word.
//
// A workgroup takes its cluster (the slabs of one unit) and slab from a ticket
// counter, in the order in which workgroups start, so at most one cluster of a
// launch has only some of its slabs running; the others always run to the end
// and free their CUs.  Launches of several streams or processes can each hold
// CUs for such a cluster until none is left.  So the workgroups of a cluster
// first wait, for a limited time, until all have arrived; past it the cluster
// gives up as one (one compare-and-swap on its count decides) before it has
// written anything, which frees its CUs, and sits out the next launches too,
// until a kernel behind them does its steps through memory
// (resident_redo_kernel).  A cluster advances units cluster, cluster + clusters,
// ... one after the other (workgroups queued behind a full chip are bound to
// an XCD early and leave others idle: 320 units of 228x428 took two rounds more).
// The waits for a neighbour's rows are bounded in time too (ResArgs::wait,
// though with the whole cluster on CUs they end by themselves); past it the
// halo becomes NaN, nothing waits any more and ResArgs::fault is set.
//
// What bounds it: vector issue, and per step about 2 us of exchange (a word
// takes 0.7 us to a workgroup of the same XCD and up to 1.2 us across), barrier
// and bookkeeping.  A 64-point row costs 83 vector instructions forward and 90
// adjoint on average (320 units of 228x428, Lc 3, counters) where an interior
// row's own block has 39 (157 for four rows); the bands, the bookkeeping of 16
// wavefronts and the exchange are the rest.  They fill 83 and 79 % of the issue
// slots.  Memory is touched by the wavefield store, the gradient and the halo
// only.  One 1024-thread workgroup per CU, as the two
// fields of a slab fill most of its LDS.  Microseconds a step of forward +
// adjoint runs, one launch per step -> resident: 2 units of 52x68 padded points
// 12.7 -> 4.7, 64 of 148x228 16.2 -> 7.4, 20 of 228x428 15.3 -> 8.1, 320 of
// them 124 -> 86.
//
// Arithmetic is the one of fwi2d_step.h, operation by operation.
#include "fwi2d_kernels.h"
#include "fwi2d_step.h"

namespace gpvi {

typedef __attribute__((address_space(3))) float LdsF;
typedef __attribute__((address_space(3))) unsigned LdsU;

// The LDS begins with kResLdsFront words: these, the items, the taper.  (The
// time limit and whether a wait ran out are read in rare cases only; in
// registers they would cost the steps some.)
enum ResFront : int { kFrontTicket = 0, kFrontWait = 1, kFrontFault = 2, kFrontItems = 16 };
__device__ __forceinline__ LdsU* res_front()
{
    extern __shared__ __align__(16) float res_lds[];
    return (LdsU*)(LdsF*)res_lds;
}

// The unit table is not written while a resident kernel runs: reads through
// the constant address space stay scalar.
#ifdef __HIP_DEVICE_COMPILE__
typedef const __attribute__((address_space(4))) UnitDesc* UnitPtr;
#else
typedef const UnitDesc* UnitPtr;   // (the host compiler's pass over this file)
#endif

// Per-workgroup constants (uniform).
struct ResUnit {
    UnitPtr u;
    float dt;
    double ydx, ydz, ydt;   // RN(1/dx), ...: a/b is formed as RN_f(RN_d(a * RN_d(1/b))) (exact, see fwi2d_step.h)
    int P;                  // LDS row length = ntx
    int z0, n;              // slab rows [z0, z0 + n)
    int pml, pitch4;        // pitch4: bytes of a field row
    int rowbase;            // byte offset of slab row 0 in a field
    int x_end;              // strips own columns [wl, x_end)
    int srow, rrow;         // source and receiver row, slab-relative
    int nx4;
    int up_end, dn_begin;   // rows [0, up_end) / [dn_begin, n) go to the slab above / below
    int v2off;              // bytes from a sample's velocities to its (v dt)^2
    int kstep;              // nt_interval
    bool run_fwi;
    Rsrc vel, grad;
    LdsF* taper;            // the absorbing taper (fdtd.c:227-230)
};

// Per-step constants (uniform).
struct ResStep {
    int it;
    bool rec, save_on, first_image, img_pair, has_ck;
    int slot4, fe4;
    Rsrc save, ck;
    unsigned tag;
    unsigned long long *up, *dn;   // where this step's rows 0 and dn_begin go (rows of P words)
};

__device__ __forceinline__ void res_send(unsigned long long* w, float v, unsigned tag)
{
    const unsigned long long x = ((unsigned long long)tag << 32) | __builtin_bit_cast(unsigned, v);
    __hip_atomic_store(G(w), x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread 0 of a workgroup: counts it as arrived and waits until its whole
// cluster is; false where the cluster gave up.  The one word holds
// count and verdict, so all workgroups of a cluster see the same one.
__device__ __forceinline__ bool res_join(const ResJoin& j, unsigned cluster)
{
    unsigned* const arrived = j.arrived + cluster;
    unsigned* const gone = j.gone + cluster;
    const unsigned want = j.want;
    unsigned seen = __hip_atomic_fetch_add(G(arrived), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    // (gave up in an earlier launch: the steps from there on are not this one's)
    if (__hip_atomic_load(G(gone), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
    const unsigned long long t0 = wall_clock64();
    while (!(seen & kResGone) && seen < want) {
        if (wall_clock64() - t0 >= j.ticks) {
            // (a failed exchange loads the word of now)
            if (__hip_atomic_compare_exchange_strong(G(arrived), &seen, seen | kResGone, __ATOMIC_RELAXED,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                __hip_atomic_store(G(gone), j.step + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
        } else {
            __builtin_amdgcn_s_sleep(1);
            seen = __hip_atomic_load(G(arrived), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    return !(seen & kResGone);
}

// LDS-only barrier: global stores may stay in flight across it.
__device__ __forceinline__ void res_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Source or residual injection and the record at one point of the source or
// receiver row (fdtd2D_modelling.c:910-911, 931-937, 949-957).
template <bool ADJ>
__device__ __forceinline__ float res_inject(const ResUnit& k, const ResStep& s, float val, float v, int ix, bool src_row,
                                            bool rec_row, bool ok)
{
    const UnitPtr u = k.u;
    const float dt = k.dt;
    if (!ADJ && src_row && ix == u->s_ix) val = val + G(u->wav)[s.it] * dt * dt * v * v;
    if (rec_row && (ADJ || s.rec)) {
        const int d = ix - u->r_ix0, dr = u->dr, nr = u->nr;
        if (ok && d >= 0 && d % dr == 0 && d / dr < nr) {
            const int ri = s.it * nr + d / dr;
            if (ADJ) {
                const float res = k.run_fwi ? G(u->syn)[ri] - G(u->obs)[ri] : G(u->obs)[ri];
                val = val + res * dt * dt * v * v;
            } else {
                G(u->syn)[ri] = val;
            }
        }
    }
    return val;
}

// The gradient after this step's imaging (and, paired, the one of step
// it + k: see make_step); sv, sv2: the stored wavefields of the two.
__device__ __forceinline__ float res_image(const ResUnit& k, const ResStep& s, float g, float sv, float sv2, float val,
                                           float p0c, float p1c, float v)
{
    const float lam2 = k.kstep == 1 ? p1c : p0c;
    if (k.run_fwi) {
        const double vd = (double)v;
        const float v3 = (float)(vd * vd * vd);
        const double coef = -2.0 / (double)v3;
        if (s.img_pair) g = (float)((double)g + coef * (double)sv2 * (double)lam2 * (double)k.kstep * (double)k.dt);
        g = (float)((double)g + coef * (double)sv * (double)val * (double)k.kstep * (double)k.dt);
    } else {
        if (s.img_pair) g = g + sv2 * lam2 * (float)k.kstep * k.dt;
        g = g + sv * val * (float)k.kstep * k.dt;
    }
    return g;
}

// a*b of the quotient pair (a / dx) / dx + (c / dz) / dz, each division rounded.
__device__ __forceinline__ float res_lap(float a, float c, double ydx, double ydz)
{
    return ddiv(ddiv(a, ydx), ydx) + ddiv(ddiv(c, ydz), ydz);
}

// The second time derivative the forward pass stores (or the field itself).
__device__ __forceinline__ float res_stored(const ResUnit& k, float val, float p1c, float p0c)
{
    return k.run_fwi ? ddiv(ddiv((val - 2.f * p1c) + p0c, k.ydt), k.ydt) : val;
}

// The imaging inputs of R rows of a lane's column: the stored wavefields of
// this step's slot and (paired) the next one, the gradient, the velocity.
template <int R>
struct ResImage {
    float sv[R], sv2[R], g[R], v[R];
};

// A strip being marched: R rows per call, the z neighbours in a register
// window that slides with the march, the x neighbours from LDS.
template <int LC>
struct ResMarch {
    float w[2 * (LC - 1)];   // p1 of the H rows behind and the H rows from the current one
    LdsF *q1, *q0;           // this lane's column, current row
    int ro, go;              // current row's byte offsets in fields and in inner-grid arrays
    int z;                   // current row of the slab
};

template <int R>
__device__ __forceinline__ void res_image_load(const ResUnit& k, const ResStep& s, ResImage<R>& im, int ix, int ro, int go,
                                               int dz)
{
    const unsigned vo = (unsigned)ix * 4u, gvo = (unsigned)(ix - k.pml) * 4u;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int o = go + r * dz * k.nx4;
        im.sv[r] = bload(s.save, gvo, o);
        im.sv2[r] = s.img_pair ? bload(s.save, gvo, o + s.slot4) : 0.f;
        im.g[r] = s.first_image ? 0.f : bload(k.grad, gvo, o);
        im.v[r] = bload(k.vel, vo, ro + r * dz * k.pitch4);
    }
}

// R plain rows, the first m of them (TAIL; else all) in the item: the others
// repeat row m - 1 and are not stored.  IMAGE: an adjoint step with the
// imaging condition (inputs in `im`).
template <int LC, bool ADJ, int R, bool IMAGE, bool TAIL>
__device__ __forceinline__ void res_rows(const ResUnit& k, const ResStep& s, ResMarch<LC>& t, int ix, bool ok, int dz,
                                         const float (&v2)[R], const ResImage<R>& im, int m = R)
{
    constexpr int H = LC - 1;
    const unsigned vo = (unsigned)ix * 4u, gvo = (unsigned)(ix - k.pml) * 4u;   // columns in fields and inner-grid arrays
    const int dP = dz * k.P, dg = dz * k.pitch4, dgo = dz * k.nx4;
    float w[2 * H + R], xl[R][H], xr[R][H], p0c[R], val[R];
#pragma unroll
    for (int j = 0; j < 2 * H; ++j) w[j] = t.w[j];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int rc = TAIL ? min(r, m - 1) : r;
        w[2 * H + r] = t.q1[(rc + H) * dP];
        p0c[r] = t.q0[rc * dP];
        LdsF* x = t.q1 + rc * dP;
#pragma unroll
        for (int j = 0; j < H; ++j) {
            xl[r][j] = x[-1 - j];
            xr[r][j] = x[1 + j];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float p1c = w[r + H];
        const float c = fd_weight(LC, 0) * p1c;
        float dxx = c, dzz = c;
#pragma unroll
        for (int j = 1; j < LC; ++j) {
            dxx = dxx + fd_weight(LC, j) * (xr[r][j - 1] + xl[r][j - 1]);
            dzz = dzz + fd_weight(LC, j) * (w[r + H + j] + w[r + H - j]);
        }
        val[r] = (2.f * p1c - p0c[r]) + v2[r] * res_lap(dxx, dzz, k.ydx, k.ydz);
    }
    // rows that hold the source or the receivers
    const int mm = TAIL ? m : R;
    const int er = (k.rrow - t.z) * dz, es = (k.srow - t.z) * dz;
    if ((unsigned)er < (unsigned)mm || (unsigned)es < (unsigned)mm) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r == er || r == es)
                val[r] = res_inject<ADJ>(k, s, val[r], bload(k.vel, vo, t.ro + r * dg), ix, r == es, r == er, ok);
    }
    if (ok) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (TAIL && r >= m) break;
            t.q0[r * dP] = val[r];
            if (IMAGE)
                bstore(res_image(k, s, im.g[r], im.sv[r], im.sv2[r], val[r], p0c[r], w[r + H], im.v[r]), k.grad, gvo,
                       t.go + r * dgo);
        }
        if (!ADJ && s.save_on) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (TAIL && r >= m) break;
                bstore(res_stored(k, val[r], w[r + H], p0c[r]), s.save, gvo, t.go + r * dgo);
            }
        }
        if (!ADJ && s.has_ck) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (TAIL && r >= m) break;
                bstore(p0c[r], s.ck, vo, t.ro + r * dg);
                bstore(w[r + H], s.ck, vo, t.ro + r * dg + s.fe4);
            }
        }
        // edge rows to the neighbouring slabs
        const int zb = t.z + dz * (mm - 1);
        if (min(t.z, zb) < k.up_end || max(t.z, zb) >= k.dn_begin) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (TAIL && r >= m) break;
                const int z = t.z + dz * r;
                if (z < k.up_end) res_send(s.up + z * k.P + ix, val[r], s.tag);
                if (z >= k.dn_begin) res_send(s.dn + (z - k.dn_begin) * k.P + ix, val[r], s.tag);
            }
        }
    }
    if (TAIL) return;
#pragma unroll
    for (int j = 0; j < 2 * H; ++j) t.w[j] = w[j + R];
    t.q1 += R * dP;
    t.q0 += R * dP;
    t.ro += R * dg;
    t.go += R * dgo;
    t.z += R * dz;
}

// Results held back until every wave has computed: up to four values per
// lane; value r goes to q[r & 1] + (r >> 1) * step (valid: one bit each).
struct ResHeld {
    float val[4];
    LdsF* q[2];
    int step;
    unsigned valid;
};

// A row within LC rows of the top or bottom edge: no stencil, the field stays
// (fdtd2D_modelling.c:756-780 updates from row LC on).
template <int LC, bool ADJ>
__device__ __forceinline__ void res_edge_row(const ResUnit& k, const ResStep& s, LdsF* q1, LdsF* q0, int ix, bool ok,
                                             int z)
{
    const unsigned fo = (unsigned)ix * 4u;
    const int ro = k.rowbase + z * k.pitch4;
    const float p1c = q1[0], p0c = q0[0];
    float val = p1c;
    if (z == k.rrow || z == k.srow)
        val = res_inject<ADJ>(k, s, val, bload(k.vel, fo, ro), ix, z == k.srow, z == k.rrow, ok);
    if (ok) {
        q0[0] = val;
        if (!ADJ && s.has_ck) {
            bstore(p0c, s.ck, fo, ro);
            bstore(p1c, s.ck, fo, ro + s.fe4);
        }
        if (z < k.up_end) res_send(s.up + z * k.P + ix, val, s.tag);
        if (z >= k.dn_begin) res_send(s.dn + (z - k.dn_begin) * k.P + ix, val, s.tag);
    }
}

// Two rows of a strip inside the z absorbing band, marched inward from the
// edge (the first one ec rows from it; m of the two are in the item): the
// extrapolation reads inward along the march, p1 from the window, p0 from LDS.
template <int LC, bool ADJ>
__device__ __forceinline__ void res_zrows(const ResUnit& k, const ResStep& s, LdsF* q1, LdsF* q0, int ix, bool ok,
                                          int z, int dz, int ec, int m, const float (&v)[kResZBlock], int hold,
                                          ResHeld& held)
{
    constexpr int H = LC - 1, R = kResZBlock;
    const int dP = dz * k.P;
    const unsigned vo = (unsigned)ix * 4u;
    const int ro = k.rowbase + z * k.pitch4, dg = dz * k.pitch4;
    float w[2 * H + R], xl[R][H], xr[R][H], a[R + 4], val[R], wt[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wt[r] = k.taper[ec - LC + min(r, m - 1)];
#pragma unroll
    for (int j = 0; j < 2 * H + R; ++j) w[j] = q1[min(j - H, m - 1 + H) * dP];
#pragma unroll
    for (int j = 0; j < R + 4; ++j) a[j] = q0[min(j, m + 3) * dP];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        LdsF* x = q1 + min(r, m - 1) * dP;
#pragma unroll
        for (int j = 0; j < H; ++j) {
            xl[r][j] = x[-1 - j];
            xr[r][j] = x[1 + j];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float p1c = w[r + H];
        const float c = fd_weight(LC, 0) * p1c;
        float dxx = c, dzz = c;
#pragma unroll
        for (int j = 1; j < LC; ++j) {
            dxx = dxx + fd_weight(LC, j) * (xr[r][j - 1] + xl[r][j - 1]);
            dzz = dzz + fd_weight(LC, j) * (w[r + H + j] + w[r + H - j]);
        }
        const float vdt = v[r] * k.dt;
        const float up = (2.f * p1c - a[r]) + (vdt * vdt) * res_lap(dxx, dzz, k.ydx, k.ydz);
        const float sc = ddiv(vdt, k.ydx);
        const float t11 = ((2.f - sc) * (1.f - sc)) / 2.f;
        const float t12 = sc * (2.f - sc);
        const float t13 = (sc * (sc - 1.f)) / 2.f;
        const float h = abc_extrap(p1c, w[r + H + 1], w[r + H + 2], a[r], a[r + 1], a[r + 2], a[r + 3], a[r + 4], t11, t12,
                                   t13);
        val[r] = abc_blend(wt[r], h, up);
    }
    const int er = (k.rrow - z) * dz, es = (k.srow - z) * dz;
    if ((unsigned)er < (unsigned)m || (unsigned)es < (unsigned)m) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r == er || r == es) val[r] = res_inject<ADJ>(k, s, val[r], v[r], ix, r == es, r == er, ok);
    }
    // (the loads above precede the stores: a row's inward p0 is read before
    // any row from it on is overwritten)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const bool here = hold == (r & 2);
        held.val[r] = here ? val[r & 1] : held.val[r];
    }
    if (ok) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r < m) {
                if (hold < 0) q0[r * dP] = val[r];
                if (!ADJ && s.has_ck) {
                    bstore(a[r], s.ck, vo, ro + r * dg);
                    bstore(w[r + H], s.ck, vo, ro + r * dg + s.fe4);
                }
                const int zr = z + dz * r;
                if (zr < k.up_end) res_send(s.up + zr * k.P + ix, val[r], s.tag);
                if (zr >= k.dn_begin) res_send(s.dn + (zr - k.dn_begin) * k.P + ix, val[r], s.tag);
            }
    }
}

// Halo rows to receive, HR words of one column per lane: asked for ahead of
// their use, then awaited.
template <int LC>
struct ResRecv {
    static constexpr int HR = LC - 1 > 4 ? LC - 1 : 4;
    unsigned long long w[HR];
};

// Where they come from and which lanes take part.
struct ResPoll {
    const unsigned long long* src;   // row 0 of this step's words
    int ix;
    bool on, ok;
};

template <int LC>
__device__ __forceinline__ void res_ask(ResRecv<LC>& r, const ResPoll& p, int P, unsigned tag)
{
#pragma unroll
    for (int j = 0; j < ResRecv<LC>::HR; ++j)
        r.w[j] = p.ok ? __hip_atomic_load(G(p.src + j * P) + p.ix, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                      : (unsigned long long)tag << 32;
}

// Repeats the loads until every word carries this step's tag and stores the
// rows at `dst`; false once the wait has run out (the rows are then NaN).  A
// forward kernel notes that in the LDS too, an adjoint one only in `alive`:
// the same outcome, and the better register allocation of each (with the note,
// 20 units of 228x428 take 1.5 % longer in all; without it 48 units of 138x278
// take 2 % longer forward).
template <int LC, bool ADJ>
__device__ __forceinline__ bool res_await(ResRecv<LC>& r, const ResPoll& p, LdsF* dst, int P, unsigned tag, bool alive)
{
    constexpr int HR = ResRecv<LC>::HR;
    auto missing = [&] {
        bool x = false;
#pragma unroll
        for (int j = 0; j < HR; ++j) x |= (unsigned)(r.w[j] >> 32) != tag;
        return any_lane(x);
    };
    if (missing()) {
        const unsigned long long t0 = wall_clock64();
        do {
            if (!alive || wall_clock64() - t0 > (unsigned long long)res_front()[kFrontWait] << 16) {
                alive = false;
                if (!ADJ) res_front()[kFrontFault] = 1;
#pragma unroll
                for (int j = 0; j < HR; ++j) r.w[j] = ((unsigned long long)tag << 32) | 0x7fc00000ull;
            } else {
                res_ask<LC>(r, p, P, tag);
            }
        } while (missing());
    }
    if (p.ok) {
#pragma unroll
        for (int j = 0; j < HR; ++j) dst[j * P + p.ix] = __builtin_bit_cast(float, (unsigned)r.w[j]);
    }
    return alive;
}

// Rows of a strip, marched from `start` (ec rows from the edge if in the z
// zone, else large): rows without a stencil, band rows in pairs, plain rows
// res_row_block at a time.  hold: the first four rows, all in the
// band, are held back.  ask: halfway through the plain rows, ask for the halo
// rows `poll` (the neighbours sent them early in the step); returns whether it
// did.  Lanes past the strip's last column repeat it and store nothing.
template <int LC, bool ADJ>
__device__ __forceinline__ bool res_strip(const ResUnit& k, const ResStep& s, LdsF* f1, LdsF* f0, int x0, int start,
                                          int dz, int cnt, int ec, bool hold, ResHeld& held, bool ask,
                                          const ResPoll& poll, ResRecv<LC>& rx)
{
    constexpr int H = LC - 1, R = res_row_block(LC);
    const int lane = threadIdx.x & 63;
    const bool ok = x0 + lane < k.x_end;
    const int ix = min(x0 + lane, k.x_end - 1);
    int e = 0;
    for (; e < cnt && ec + e < LC; ++e) {
        const int z = start + dz * e;
        res_edge_row<LC, ADJ>(k, s, f1 + z * k.P + ix, f0 + z * k.P + ix, ix, ok, z);
    }
    const unsigned vo = (unsigned)ix * 4u;
    const int dg = dz * k.pitch4;
    if (e < cnt && ec + e < k.pml) {
        // velocities one pair ahead (the margins make every row addressable)
        float vz[kResZBlock];
        int ro = k.rowbase + (start + dz * e) * k.pitch4;
#pragma unroll
        for (int r = 0; r < kResZBlock; ++r) vz[r] = bload(k.vel, vo, ro + r * dg);
        while (e < cnt && ec + e < k.pml) {
            const int z = start + dz * e, m = min(min(cnt - e, k.pml - ec - e), kResZBlock);
            float v[kResZBlock];
            ro += kResZBlock * dg;
#pragma unroll
            for (int r = 0; r < kResZBlock; ++r) {
                v[r] = vz[r];
                vz[r] = bload(k.vel, vo, ro + r * dg);
            }
            res_zrows<LC, ADJ>(k, s, f1 + z * k.P + ix, f0 + z * k.P + ix, ix, ok, z, dz, ec + e, m, v,
                               hold && e < 4 ? e : -1, held);
            e += m;
        }
    }
    if (hold) {
        held.valid = ok ? (1u << min(cnt, 4)) - 1u : 0u;
        held.q[0] = f0 + start * k.P + ix;
        held.q[1] = held.q[0] + dz * k.P;
        held.step = 2 * dz * k.P;
    }
    int left = cnt - e;
    if (left <= 0) return false;
    const int ask_at = ask ? left / 2 : -1;   // rows left when asking
    bool asked = false;
    ResMarch<LC> t;
    t.z = start + dz * e;
    t.q1 = f1 + t.z * k.P + ix;
    t.q0 = f0 + t.z * k.P + ix;
    t.ro = k.rowbase + t.z * k.pitch4;
    t.go = (k.z0 + t.z - k.pml) * k.nx4;
    if (ADJ && s.save_on) {
        // imaging: two rows at a time, every input one block ahead
        constexpr int RI = 2;
        ResImage<RI> nx;
        float vn[RI];
        res_image_load<RI>(k, s, nx, ix, t.ro, t.go, left > 1 ? dz : 0);
#pragma unroll
        for (int r = 0; r < RI; ++r) vn[r] = bload(k.vel, vo, t.ro + k.v2off + r * dg);
#pragma unroll
        for (int j = 0; j < 2 * H; ++j) t.w[j] = t.q1[(j - H) * dz * k.P];
        while (left >= RI) {
            if (!asked && left <= ask_at) {
                res_ask<LC>(rx, poll, k.P, s.tag);
                asked = true;
            }
            const ResImage<RI> im = nx;
            float v2[RI];
#pragma unroll
            for (int r = 0; r < RI; ++r) v2[r] = vn[r];
            left -= RI;
            if (left > 0) {
                // (an odd last row is asked for twice)
                res_image_load<RI>(k, s, nx, ix, t.ro + RI * dg, t.go + RI * dz * k.nx4, left > 1 ? dz : 0);
#pragma unroll
                for (int r = 0; r < RI; ++r) vn[r] = bload(k.vel, vo, t.ro + k.v2off + (RI + r) * dg);
            }
            res_rows<LC, ADJ, RI, true, false>(k, s, t, ix, ok, dz, v2, im);
        }
        if (left > 0) {
            const float v2[1] = {vn[0]};
            const ResImage<1> im = {{nx.sv[0]}, {nx.sv2[0]}, {nx.g[0]}, {nx.v[0]}};
            res_rows<LC, ADJ, 1, true, false>(k, s, t, ix, ok, dz, v2, im);
        }
        return asked;
    }
    float vn[R];
#pragma unroll
    for (int r = 0; r < R; ++r) vn[r] = bload(k.vel, vo, t.ro + k.v2off + r * dg);
#pragma unroll
    for (int j = 0; j < 2 * H; ++j) t.w[j] = t.q1[(j - H) * dz * k.P];
    while (left >= R) {
        if (!asked && left <= ask_at) {
            res_ask<LC>(rx, poll, k.P, s.tag);
            asked = true;
        }
        float v2[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            v2[r] = vn[r];
            vn[r] = bload(k.vel, vo, t.ro + k.v2off + (R + r) * dg);
        }
        res_rows<LC, ADJ, R, false, false>(k, s, t, ix, ok, dz, v2, ResImage<R>());
        left -= R;
    }
    if (left > 0) res_rows<LC, ADJ, R, false, true>(k, s, t, ix, ok, dz, vn, ResImage<R>(), left);
    return asked;
}

// Points of a lane that a side block takes per round (64 units of 148x228 in
// 1000 + 1000 steps take 14.70 ms with one, 15.39 with two; 320 of 228x428 171.1
// and 175.6).
constexpr int kResSideBlock = 1;

// A side block, w columns wide: the item's points in row-major order (columns
// counted inward from the edge), 64 at a time, kResSideBlock of these per
// round, so that every lane has a point whatever the width.  ZB: the rows lie
// in the z zone, the first one e0 rows from its edge, marched inward.  The p0
// reads of the absorbing extrapolations go to later points of that order.
template <int LC, bool ADJ, bool ZB>
__device__ __forceinline__ void res_side(const ResUnit& k, const ResStep& s, LdsF* f1, LdsF* f0, int side, int lanepos,
                                         int w, int start, int dz, int cnt, int e0, bool hold, ResHeld& held)
{
    constexpr int B = kResSideBlock;
    const int P = k.P, pml = k.pml, dP = dz * P;
    const int dx = side ? -1 : 1;
    const int rows64 = 64 / w, cols64 = 64 - rows64 * w;   // 64 points further on
    int row = lanepos >> 8, col = lanepos & 0xff;
    const bool image = ADJ && s.save_on;
    // A point's row and column and its inputs from memory, fetched one round
    // ahead.
    struct Point {
        int row, cl;
        float v, sv, sv2, gr;
    };
    auto place = [&](int r, int c, int* z, int* ix, int* ec, bool* inner, unsigned* go, unsigned* fo) {
        const int rc = min(r, cnt - 1);
        *ix = side ? P - 1 - c : c;
        *z = start + dz * rc;
        *ec = ZB ? e0 + rc : pml;
        *inner = c >= pml && *ec >= pml;
        *go = *inner ? (unsigned)((k.z0 + *z - pml) * k.nx4 + (*ix - pml) * 4) : 0u;
        *fo = (unsigned)(k.rowbase + *z * k.pitch4 + *ix * 4);
    };
    auto fetch = [&] {
        Point p;
        p.row = row;
        p.cl = col;
        row += rows64;
        col += cols64;
        if (col >= w) {
            col -= w;
            ++row;
        }
        int z, ix, ec;
        bool inner;
        unsigned go, fo;
        place(p.row, p.cl, &z, &ix, &ec, &inner, &go, &fo);
        p.v = bload(k.vel, fo, 0);
        p.sv = p.sv2 = p.gr = 0.f;
        if (image && inner) {
            p.sv = bload(s.save, go, 0);
            if (s.img_pair) p.sv2 = bload(s.save, go, s.slot4);
            if (!s.first_image) p.gr = bload(k.grad, go, 0);
        }
        return p;
    };
    Point next[B];
#pragma unroll
    for (int b = 0; b < B; ++b) next[b] = fetch();
    for (int i0 = 0; i0 < cnt * w; i0 += 64 * B) {
        float v[B], p1c[B], p0c[B], val[B], sv[B], sv2[B], gr[B], wz[B], wx[B];
        float xl[B][LC - 1], xr[B][LC - 1], zu[B][LC - 1], zd[B][LC - 1], ax[B][4], az[B][4];
        unsigned go[B], fo[B];
        int z[B], ec[B], cl[B], ix[B];
        LdsF* q0[B];
        bool ok[B], inner[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const Point p = next[b];
            ok[b] = p.row < cnt;
            cl[b] = p.cl;
            v[b] = p.v;
            sv[b] = p.sv;
            sv2[b] = p.sv2;
            gr[b] = p.gr;
            place(p.row, p.cl, &z[b], &ix[b], &ec[b], &inner[b], &go[b], &fo[b]);
            next[b] = fetch();
            wx[b] = k.taper[min(max(cl[b] - LC, 0), pml - LC)];
            if (ZB) wz[b] = k.taper[min(max(ec[b] - LC, 0), pml - LC)];
            LdsF* q1 = f1 + z[b] * P + ix[b];
            q0[b] = f0 + z[b] * P + ix[b];
            p1c[b] = q1[0];
            p0c[b] = q0[b][0];
            // (lanes at the edge of the grid read other words of the buffers
            // and discard the result)
#pragma unroll
            for (int j = 0; j < LC - 1; ++j) {
                xl[b][j] = q1[-1 - j];
                xr[b][j] = q1[1 + j];
                zu[b][j] = q1[(-1 - j) * P];
                zd[b][j] = q1[(1 + j) * P];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ax[b][j] = q0[b][(j + 1) * dx];
                if (ZB) az[b][j] = q0[b][(j + 1) * dP];
            }
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float c = fd_weight(LC, 0) * p1c[b];
            float dxx = c, dzz = c;
#pragma unroll
            for (int j = 1; j < LC; ++j) {
                dxx = dxx + fd_weight(LC, j) * (xr[b][j - 1] + xl[b][j - 1]);
                dzz = dzz + fd_weight(LC, j) * (zd[b][j - 1] + zu[b][j - 1]);
            }
            const float vdt = v[b] * k.dt;
            const float up = (2.f * p1c[b] - p0c[b]) + (vdt * vdt) * res_lap(dxx, dzz, k.ydx, k.ydz);
            float u = cl[b] >= LC && (!ZB || ec[b] >= LC) ? up : p1c[b];
            const float sc = ddiv(vdt, k.ydx);
            const float t11 = ((2.f - sc) * (1.f - sc)) / 2.f;
            const float t12 = sc * (2.f - sc);
            const float t13 = (sc * (sc - 1.f)) / 2.f;
            if (ZB) {
                const float q2 = dz > 0 ? zd[b][0] : zu[b][0], q3 = dz > 0 ? zd[b][1] : zu[b][1];
                const float h = abc_extrap(p1c[b], q2, q3, p0c[b], az[b][0], az[b][1], az[b][2], az[b][3], t11, t12, t13);
                const float t = abc_blend(wz[b], h, u);
                u = ec[b] >= LC && ec[b] < pml ? t : u;
            }
            const float q2 = side ? xl[b][0] : xr[b][0], q3 = side ? xl[b][1] : xr[b][1];
            const float h = abc_extrap(p1c[b], q2, q3, p0c[b], ax[b][0], ax[b][1], ax[b][2], ax[b][3], t11, t12, t13);
            const float t = abc_blend(wx[b], h, u);
            u = cl[b] >= LC && cl[b] < pml ? t : u;
            const bool rec_row = z[b] == k.rrow, src_row = z[b] == k.srow;
            if (rec_row || src_row)
                u = res_inject<ADJ>(k, s, u, v[b], ix[b], src_row, rec_row, ok[b]);
            val[b] = u;
        }
        // (the loads above precede these stores)
        __builtin_amdgcn_wave_barrier();
        // (the first 128 points hold the first four rows: w <= 32)
        const bool hold_now = ZB && hold && i0 < 128;
        if (hold_now) {
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const bool here = i0 + 64 * b == 64 * r;
                    held.val[r] = here ? val[b] : held.val[r];
                    held.q[r] = here ? q0[b] : held.q[r];
                    held.valid |= here && ok[b] ? 1u << r : 0u;
                }
        }
#pragma unroll
        for (int b = 0; b < B; ++b)
            if (ok[b]) {
                if (!hold_now) q0[b][0] = val[b];
                if (s.save_on && inner[b]) {
                    if (ADJ)
                        bstore(res_image(k, s, gr[b], sv[b], sv2[b], val[b], p0c[b], p1c[b], v[b]), k.grad, go[b], 0);
                    else
                        bstore(res_stored(k, val[b], p1c[b], p0c[b]), s.save, go[b], 0);
                }
                if (!ADJ && s.has_ck) {
                    bstore(p0c[b], s.ck, fo[b], 0);
                    bstore(p1c[b], s.ck, fo[b], s.fe4);
                }
                if (z[b] < k.up_end) res_send(s.up + z[b] * P + ix[b], val[b], s.tag);
                if (z[b] >= k.dn_begin) res_send(s.dn + (z[b] - k.dn_begin) * P + ix[b], val[b], s.tag);
            }
    }
}

template <int LC, bool ADJ>
__global__ __launch_bounds__(kResThreads) void resident_kernel(ResArgs a)
{
    constexpr int HR = LC - 1 > 4 ? LC - 1 : 4;
    LdsF* const lds = (LdsF*)res_front();
    const ResPlan& pl = a.plan;
    if (threadIdx.x == 0) {
        res_front()[kFrontWait] = a.wait;
        res_front()[kFrontFault] = 0;
        unsigned t = __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // (expected not taken: the wait's code then stays out of the way of the steps' registers; forward
        // steps of 2 units of 52x68 take 4.58 us, 4.83 without the hint)
        if (__builtin_expect(a.join.slabs != 0, 0) && !res_join(a.join, t / a.join.slabs)) t = kResGone;   // past every unit
        res_front()[kFrontTicket] = t;
    }
    __syncthreads();
    const unsigned ticket = __builtin_amdgcn_readfirstlane(res_front()[kFrontTicket]);
    // readfirstlane: what follows from the cluster and slab stays in scalar registers
    const int cluster = __builtin_amdgcn_readfirstlane((int)(ticket / (unsigned)pl.slabs));
    const int g = (int)ticket - cluster * pl.slabs;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    bool alive = true;
    for (int ui = cluster; ui < a.nunit; ui += a.clusters) {
    const UnitPtr up = (UnitPtr)(uint64_t)(a.units + ui);
    const UnitDesc u = *up;
    const ResSlab sl = res_slab(pl, u.ntz, g);
    const int P = u.ntx, n = sl.n;
    const int64_t margin = (int64_t)kPadRows * u.pitch;

    ResUnit k;
    k.u = up;
    k.dt = u.dt;
    k.ydx = u.ydx; k.ydz = u.ydz; k.ydt = u.ydt;
    k.P = P;
    k.z0 = sl.z0;
    k.n = n;
    k.pml = u.pml;
    k.pitch4 = u.pitch * 4;
    k.rowbase = (sl.z0 + kPadRows) * k.pitch4;
    k.kstep = u.k;
    k.run_fwi = u.run_fwi != 0;
    k.x_end = P - pl.wr;
    k.srow = ADJ ? -1 : u.s_iz - sl.z0;
    k.rrow = u.r_iz - sl.z0;
    k.nx4 = u.nx * 4;
    k.up_end = g > 0 ? HR : 0;
    k.dn_begin = g + 1 < pl.slabs ? n - HR : n;
    k.v2off = a.vdt2_off;
    k.vel = make_rsrc(u.vel - margin);
    k.grad = make_rsrc(u.grad);
    int e0 = 0;   // a band slab's first row, from its edge
    if (pl.slabs > 1)
        for (int i = 0; i < sl.table && i < pl.nband; ++i) e0 += pl.band_rows[i];

    LdsF* const fa = lds + kResLdsFront + HR * P;   // row 0 of the two buffers
    LdsF* const fb = fa + (n + 2 * HR) * P;

    // Initial fields: p1 and p0 of the first step, halo rows included.
    const StepInfo si0 = decode_step(u, a.s0);
    {
        const FieldPtrs fp = step_fields(u, si0);
        for (int z = -HR + wave; z < n + HR; z += kResWaves) {
            const int iz = sl.z0 + z;
            const bool in = iz >= 0 && iz < u.ntz;
            const int64_t o = (int64_t)iz * u.pitch;
            for (int x = lane; x < P; x += 64) {
                fa[z * P + x] = in ? G(fp.p1)[o + x] : 0.f;
                fb[z * P + x] = in ? G(fp.p0)[o + x] : 0.f;
            }
        }
    }
    // The wave's items, decoded, in LDS.
    LdsU* const my_items = (LdsU*)lds + kFrontItems + wave * 2 * kResItems;
    if (lane < kResItems) {
        const ResItem item = pl.item[sl.table][wave][lane];
        int start, dz, cnt;
        res_item_rows(sl, item, &start, &dz, &cnt);
        unsigned w0, w1;
        res_pack_item(item, start, dz, cnt, &w0, &w1);
        my_items[2 * lane] = w0;
        my_items[2 * lane + 1] = w1;
    }
    k.taper = lds + kFrontItems + 2 * kResWaves * kResItems;
    if (wave == 0 && lane < 32 && lane < u.pml0) k.taper[lane] = G(u.wtab)[lane];
    const bool two_phase = pl.two_phase[sl.table] != 0;
    // side blocks: column and row slot of this lane, left and right
    const int pos_l = (lane % pl.wl) | ((lane / pl.wl) << 8);
    const int pos_r = (lane % pl.wr) | ((lane / pl.wr) << 8);

    // halo words: [parity][boundary][direction][HR][P]; boundary b lies below
    // slab b, direction 0 goes down
    const int dir = HR * P, par = (pl.slabs - 1) * 2 * dir;
    unsigned long long* const halo = a.halo + (int64_t)ui * a.halo_stride;
    // Halo rows this wave receives: units of (strip, or both side blocks) x
    // (slab above, slab below), dealt in turn.
    constexpr int kPolls = 2;
    auto poll_unit = [&](int j, const unsigned long long* words, LdsF* f0, LdsF** dst) {
        const int q = wave + kResWaves * j, blk = q >> 1;
        const bool below = q & 1;
        ResPoll p;
        p.on = blk <= pl.strips && (below ? g + 1 < pl.slabs : g > 0);
        p.src = words + (below ? dir : -2 * dir);
        *dst = f0 + (below ? n * P : -HR * P);
        const int side_ix = lane < 32 ? lane : k.x_end + lane - 32;
        p.ix = blk < pl.strips ? pl.wl + 64 * blk + lane : side_ix;
        p.ok = blk < pl.strips ? p.ix < k.x_end : (lane < 32 ? lane < pl.wl : lane - 32 < pl.wr);
        return p;
    };

    // Store slots of the steps (see make_step): slot = it / k within the
    // segment, advanced with the steps; `ph` = it % k.
    const bool rec = si0.mode == kRec, fwd = si0.mode == kFwd;
    const bool stores = ADJ || (u.store && (rec || u.nseg == 1));
    const int seg_it = u.nseg == 1 ? 0 : si0.seg * u.ckpt;
    const int seg_len = u.nseg == 1 ? u.nt : (si0.seg == u.nseg - 1 ? u.last_len : u.ckpt);
    const int nslots = (seg_len + u.k - 1) / u.k;
    const bool pairs = u.k <= 2;
    const int first_slot = pairs ? ((nslots - 1) & ~1) : nslots - 1;
    const bool top_seg = u.grad_init && si0.seg == u.nseg - 1;
    const int64_t slot_elems = (int64_t)u.nx * u.nz;
    int ph = si0.it % u.k;
    int slot = (fwd && u.nseg > 1) ? 0 : (si0.it - seg_it) / u.k + (!ADJ && ph ? 1 : 0);
    const bool cks = fwd && u.nseg > 1;
    int ck_ph = cks ? si0.it % u.ckpt : 1, ck_no = cks ? si0.it / u.ckpt + (ck_ph ? 1 : 0) : 0;

    __syncthreads();
    for (int i = 0; i < a.n; ++i) {
        LdsF* const f1 = (i & 1) ? fb : fa;
        LdsF* const f0 = (i & 1) ? fa : fb;
        ResStep s;
        unsigned long long* const hp = halo + ((a.s0 + i) & 1) * par + 2 * g * dir;   // boundary g, downward
        s.it = ADJ ? si0.it - i : si0.it + i;
        s.rec = fwd;
        const bool image = ADJ && ph == 0 && !(pairs && (slot & 1));
        s.save_on = ADJ ? image : stores && ph == 0;
        s.first_image = image && top_seg && slot == first_slot;
        s.img_pair = image && pairs && slot + 1 < nslots;
        s.slot4 = (int)slot_elems * 4;
        s.fe4 = (int)(u.field_elems * 4);
        if (s.save_on) s.save = make_rsrc(u.save + slot * slot_elems);
        s.has_ck = cks && ck_ph == 0 && ck_no > 0;
        if (s.has_ck) s.ck = make_rsrc(u.ck + (int64_t)(2 * ck_no) * u.field_elems - margin);
        s.tag = (unsigned)(a.s0 + i) + 1u;
        s.up = hp - dir;
        s.dn = hp;
        if (ADJ) {
            if (ph == 0) { ph = u.k - 1; --slot; } else { --ph; }
        } else {
            if (ph == 0) ++slot;
            if (++ph == u.k) ph = 0;
        }
        if (cks) {
            if (ck_ph == 0) ++ck_no;
            if (++ck_ph == u.ckpt) ck_ph = 0;
        }
        ResHeld held;
        held.valid = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) held.val[r] = 0.f;
        ResRecv<LC> rx;
        const bool recv = i + 1 < a.n;
        bool asked = false;
        LdsF* poll_dst;
        const ResPoll poll = poll_unit(0, hp, f0, &poll_dst);
        held.q[0] = held.q[1] = f0;
        held.step = 0;
        unsigned n0 = __builtin_amdgcn_readfirstlane(my_items[0]), n1 = __builtin_amdgcn_readfirstlane(my_items[1]);
        for (int q = 1; n0 >> 20 & 1; ++q) {
            const ResWords d = res_unpack_item(n0, n1);
            const int cnt = d.count, start = d.start, x0 = d.x0, kind = d.kind, dz = d.step;
            const bool hold = d.hold;
            n0 = 0;
            if (q < kResItems) {
                n0 = __builtin_amdgcn_readfirstlane(my_items[2 * q]);
                n1 = __builtin_amdgcn_readfirstlane(my_items[2 * q + 1]);
            }
            if (cnt == 0) continue;   // (the one row of an item that a shorter slab lacks)
            // rows from the edge of the z zone's first row in this item
            const int ec = e0 + (pl.slabs == 1 ? (dz > 0 ? start : n - 1 - start) : (sl.flip ? n - 1 - start : start));
            const int pos = x0 ? pos_r : pos_l, w = x0 ? pl.wr : pl.wl;
            if (kind <= kResStripZ)
                asked = res_strip<LC, ADJ>(k, s, f1, f0, x0, start, dz, cnt, kind == kResStripZ ? ec : 1 << 20, hold, held,
                                           recv && poll.on && !(n0 >> 20 & 1), poll, rx);
            else if (kind == kResSide)
                res_side<LC, ADJ, false>(k, s, f1, f0, x0, pos, w, start, dz, cnt, 0, false, held);
            else
                res_side<LC, ADJ, true>(k, s, f1, f0, x0, pos, w, start, dz, cnt, ec, hold, held);
        }
        if (two_phase) {
            res_barrier();
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (held.valid >> r & 1) held.q[r & 1][(r >> 1) * held.step] = held.val[r];
        }
        // The neighbours' edge rows of this step, into the new field's halo.
        if (recv) {
            if (poll.on) {
                if (!asked) res_ask<LC>(rx, poll, P, s.tag);
                alive = res_await<LC, ADJ>(rx, poll, poll_dst, P, s.tag, alive);
            }
#pragma unroll
            for (int j = 1; j < kPolls; ++j) {
                LdsF* dst;
                const ResPoll p = poll_unit(j, hp, f0, &dst);
                if (p.on) {
                    res_ask<LC>(rx, p, P, s.tag);
                    alive = res_await<LC, ADJ>(rx, p, dst, P, s.tag, alive);
                }
            }
        }
        res_barrier();
    }
    // The last two fields, where the next launch (of any kind) expects them.
    const int ql = si0.q + a.n - 1;
    float* const base = ADJ ? u.adj : u.fwd;
    float* const o1 = base + u.field_elems * (ql & 3);
    float* const o0 = base + u.field_elems * ((ql - 1) & 3);
    LdsF* const l1 = (a.n & 1) ? fb : fa;
    LdsF* const l0 = (a.n & 1) ? fa : fb;
    for (int z = wave; z < n; z += kResWaves) {
        const int64_t o = (int64_t)(sl.z0 + z) * u.pitch;
        for (int x = lane; x < P; x += 64) {
            G(o1)[o + x] = l1[z * P + x];
            if (a.n > 1) G(o0)[o + x] = l0[z * P + x];
        }
    }
    __syncthreads();   // the next unit reuses the buffers
    }
    if (__builtin_expect(ADJ ? !alive : res_front()[kFrontFault] != 0, 0))
        __hip_atomic_store(G(a.fault), a.fault_id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// vdt2[m] = (vel[m] * dt)^2 for fields of n values, in and out fields each
// `stride` apart.
__global__ void vdt2_kernel(const float* __restrict__ vel, float* __restrict__ out, float dt, int64_t n, int64_t stride)
{
    const float* v = vel + blockIdx.y * stride;
    float* o = out + blockIdx.y * stride;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float t = v[i] * dt;
        o[i] = t * t;
    }
}

hipError_t launch_vdt2(hipStream_t st, const float* vel, float* out, float dt, int64_t n, int64_t stride, int nsample)
{
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 65536));
    for (int m = 0; m < nsample; m += 65535) {
        hipLaunchKernelGGL(vdt2_kernel, dim3(grid, std::min(65535, nsample - m)), dim3(256), 0, st, vel + m * stride,
                           out + m * stride, dt, n, stride);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int LC, bool ADJ>
static hipError_t launch_resident_lc(hipStream_t st, const ResArgs& a)
{
    hipLaunchKernelGGL((resident_kernel<LC, ADJ>), dim3(a.clusters * a.plan.slabs), dim3(kResThreads), a.plan.lds_bytes, st,
                       a);
    return hipGetLastError();
}

hipError_t launch_resident(hipStream_t st, int lc, bool adjoint, const ResArgs& a)
{
    switch (lc * 2 + (adjoint ? 1 : 0)) {
    case 8: return launch_resident_lc<4, false>(st, a);
    case 9: return launch_resident_lc<4, true>(st, a);
    case 10: return launch_resident_lc<5, false>(st, a);
    case 11: return launch_resident_lc<5, true>(st, a);
    case 12: return launch_resident_lc<6, false>(st, a);
    case 13: return launch_resident_lc<6, true>(st, a);
    case 14: return launch_resident_lc<7, false>(st, a);
    case 15: return launch_resident_lc<7, true>(st, a);
    default: return hipErrorInvalidValue;
    }
}

template <int LC, bool ADJ>
static int resident_capacity_lc()
{
    const void* f = (const void*)resident_kernel<LC, ADJ>;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kResLdsBytes) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, resident_kernel<LC, ADJ>, kResThreads, kResLdsBytes) !=
        hipSuccess)
        return 0;
    return nb;
}

// Workgroups of the resident kernels the current device holds at once (0:
// they do not run there).
int resident_capacity(int lc)
{
    int nb = 0;
    switch (lc) {
    case 4: nb = std::min(resident_capacity_lc<4, false>(), resident_capacity_lc<4, true>()); break;
    case 5: nb = std::min(resident_capacity_lc<5, false>(), resident_capacity_lc<5, true>()); break;
    case 6: nb = std::min(resident_capacity_lc<6, false>(), resident_capacity_lc<6, true>()); break;
    case 7: nb = std::min(resident_capacity_lc<7, false>(), resident_capacity_lc<7, true>()); break;
    default: return 0;
    }
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return nb * cus;
}

}  // namespace gpvi
