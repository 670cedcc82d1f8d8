// Checks of the row ranges that the resident steps' wavefronts take from a
// plan (fwi2d_resident.h), as the kernel reads them: packed and unpacked; and
// the rule of which plans may run.
#include <vector>

#include "fwi2d_resident.h"

using namespace gpvi;

// 1: every present item of every slab lies in its slab and every point of the
// grid is computed once; < 0: what is wrong.
static int check_plan(const ResPlan& p, int ntx, int ntz)
{
    std::vector<int> cover((size_t)ntx * ntz, 0);
    for (int s = 0; s < p.slabs; ++s) {
        const ResSlab sl = res_slab(p, ntz, s);
        for (int w = 0; w < kResWaves; ++w)
            for (int i = 0; i < kResItems; ++i) {
                const ResItem& it = p.item[sl.table][w][i];
                int start, step, count;
                res_item_rows(sl, it, &start, &step, &count);
                unsigned w0, w1;
                res_pack_item(it, start, step, count, &w0, &w1);
                const ResWords r = res_unpack_item(w0, w1);
                if (!r.present) continue;
                if (r.x0 != it.x0 || r.kind != it.kind || r.hold != (it.hold != 0)) return -1;
                if (r.count > it.count || r.count + 1 < it.count) return -2;   // a shorter slab lacks one row
                if (r.count == 0) continue;
                const int last = r.start + r.step * (r.count - 1);
                if (r.start < 0 || r.start >= sl.n || last < 0 || last >= sl.n) return -3;
                const bool strip = r.kind <= kResStripZ;
                const int x0 = strip ? r.x0 : (r.x0 ? ntx - p.wr : 0);
                const int x1 = strip ? std::min(x0 + 64, ntx - p.wr) : (r.x0 ? ntx : p.wl);
                for (int e = 0; e < r.count; ++e)
                    for (int x = x0; x < x1; ++x) ++cover[(size_t)(sl.z0 + r.start + r.step * e) * ntx + x];
            }
    }
    for (int c : cover)
        if (c != 1) return -4;
    return 1;
}

// The plan with `slabs` slabs (0: there is none).
extern "C" int resident_items_of_plan(int ntx, int ntz, int lc, int pml, int slabs)
{
    ResPlan p;
    if (res_make_plan(ResGeom{ntx, ntz, lc, pml}, slabs, &p) < 0) return 0;
    return check_plan(p, ntx, ntz);
}

// The plan that a batch of `units` units takes on 256 CUs (0: there is none).
extern "C" int resident_items_of_choice(int ntx, int ntz, int lc, int pml, int units)
{
    ResPlan p;
    if (res_select_plan(ResGeom{ntx, ntz, lc, pml}, units, 256, kResMaxSlabs, &p) < 0) return 0;
    return check_plan(p, ntx, ntz);
}

extern "C" int resident_admits(int slabs, int queues, int cus) { return res_admits(slabs, queues, cus) ? 1 : 0; }
extern "C" int resident_slab_limit(int queues) { return res_slab_limit(queues); }
