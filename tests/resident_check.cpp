// Checks of the resident steps' plans (fwi2d_resident.h) on the CPU.
#include <vector>

#include "fwi2d_resident.h"

using namespace gpvi;

// 0: no such plan; 1: a sound one; < 0: what is wrong with it.
extern "C" int resident_plan_check(int ntx, int ntz, int lc, int pml, int slabs)
{
    const ResGeom g{ntx, ntz, lc, pml};
    ResPlan p;
    if (res_make_plan(g, slabs, &p) < 0) return 0;
    if (p.lds_bytes > kResLdsBytes || p.wl > 32 || p.wr > 32 || p.wl < pml + 4 || p.wr < pml + 4) return -1;
    if (p.wl + 64 * p.strips < ntx - p.wr || p.strips + 1 > kResWaves) return -2;
    struct Row {
        int cover, order, wave;   // order: place in its item, from the item's first row
        bool hold;
    };
    std::vector<Row> at((size_t)ntx * ntz, Row{0, 0, 0, false});
    std::vector<int> slab_of(ntz, -1);
    int rows = 0;
    for (int s = 0; s < slabs; ++s) {
        const ResSlab sl = res_slab(p, ntz, s);
        if (sl.z0 != rows || (slabs > 1 && sl.n < p.hr)) return -3;
        if (res_lds_bytes(ntx, sl.n, p.hr) > p.lds_bytes) return -4;
        rows += sl.n;
        for (int z = 0; z < sl.n; ++z) slab_of[sl.z0 + z] = s;
        for (int w = 0; w < kResWaves; ++w) {
            int held = 0;
            bool end = false;
            for (int i = 0; i < kResItems; ++i) {
                const ResItem& it = p.item[sl.table][w][i];
                if (it.count == 0) { end = true; continue; }
                if (end) return -5;   // the list ends at its first empty item
                held += it.hold ? 1 : 0;
                int a, d, c;
                res_item_rows(sl, it, &a, &d, &c);
                for (int e = 0; e < c; ++e) {
                    const int r = a + d * e, z = sl.z0 + r;
                    if (r < 0 || r >= sl.n) return -6;
                    const bool zone = z < p.zt || z >= ntz - p.zt;
                    if (zone != (it.kind == kResStripZ || it.kind == kResSideZ)) return -7;
                    if (zone && d != (z < p.zt ? 1 : -1)) return -8;   // marched inward
                    const bool strip = it.kind <= kResStripZ;
                    const int x0 = strip ? it.x0 : (it.x0 ? ntx - p.wr : 0);
                    const int x1 = strip ? std::min(x0 + 64, ntx - p.wr) : (it.x0 ? ntx : p.wl);
                    for (int x = x0; x < x1; ++x) {
                        Row& q = at[(size_t)z * ntx + x];
                        ++q.cover;
                        q.wave = w;
                        q.order = e;
                        q.hold = it.hold && e < 4;
                    }
                }
            }
            if (held > 1) return -9;   // one set of held rows per wave
            if (held && !p.two_phase[sl.table]) return -10;
        }
    }
    if (rows != ntz) return -11;
    for (const Row& q : at)
        if (q.cover != 1) return -12;
    // A band row reads p0 of the four rows further in: they must be computed
    // later by the same item, be held back, or lie in another slab whose copy
    // arrives only after the step (two_phase).
    for (int edge = 0; edge < 2; ++edge)
        for (int d = lc; d < pml; ++d)
            for (int f = 1; f <= 4; ++f)
                for (int x = 0; x < ntx; ++x) {
                    const int z = edge ? ntz - 1 - d : d, y = edge ? z - f : z + f;
                    const Row &r = at[(size_t)z * ntx + x], &q = at[(size_t)y * ntx + x];
                    const ResSlab sl = res_slab(p, ntz, slab_of[z]);
                    if (slab_of[y] != slab_of[z]) {
                        if (!p.two_phase[sl.table]) return -13;
                    } else if (!q.hold && !(q.wave == r.wave && q.order > r.order)) {
                        return -14;
                    }
                }
    return 1;
}
