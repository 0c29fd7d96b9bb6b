// Host side of the matrix-core resident kernels: the kernel order, the tiles
// and their row lists, the launch.
#include "host_par.h"
#include "units.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <numeric>

namespace swe {

namespace {

// The tables, gathered for one allocation and one copy.
struct Tables {
    std::vector<char> bytes;
    template <typename T>
    size_t add(const std::vector<T> &v)
    {
        const size_t at = (bytes.size() + 255) / 256 * 256;
        bytes.resize(at + sizeof(T) * v.size());
        std::memcpy(bytes.data() + at, v.data(), sizeof(T) * v.size());
        return at;
    }
};

// Place of (node of the unit, slot) in a unit's 512 row numbers: for the FP64
// matrix instructions [group of 4 nodes][slot & 3][node][slot / 4], by node
// (FP32, exact) [slot / 8][node][slot & 7].
int prec_at(bool by_node, int m, int slot)
{
    return by_node ? (slot >> 3) * 128 + m * 8 + (slot & 7)
                : (m >> 2) * 128 + ((slot & 3) * 4 + (m & 3)) * 8 + (slot >> 2);
}

}  // namespace

static void free_records(SweUnits &u)
{
    void *ptrs[] = {u.d_wrec, u.d_grec, u.d_tables};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
}

void units_free(swe_hip_ctx *c)
{
    SweUnits &u = c->units;
    if (u.d_hd)
        (void)hipFree(u.d_hd);
    if (u.shared) {
        std::lock_guard<std::mutex> lock(c->mesh->records_mutex);
        if (--u.shared->refs == 0) {
            std::vector<SweUnitRecords *> &all = c->mesh->unit_records;
            all.erase(std::find(all.begin(), all.end(), u.shared));
            free_records(u.shared->u);
            delete u.shared;
        }
    } else {
        free_records(u);   // of a build that failed
    }
    c->bytes -= u.bytes;
    u = SweUnits{};
}

namespace {

// Reorders ids[first, last) so that consecutive chunks of `chunk` nodes are
// compact on the sphere: recursive bisection along the longest principal
// axis, the left part always whole chunks.  Against a Hilbert curve through
// the nodes a tile reads fewer rows from fewer tiles (N = 40962, 161-node
// tiles: at most 352 rows and 10 tiles against 565 and 18; N = 163842: 1006
// and 10 against 1487 and 17).
void bisect(const double *xyz, int n, std::vector<int> &ids, int first, int last, int chunk)
{
    const int count = last - first, parts = (count + chunk - 1) / chunk;
    if (parts < 2)
        return;
    double mean[3] = {0.0, 0.0, 0.0}, cov[3][3] = {};
    for (int i = first; i < last; ++i)
        for (int d = 0; d < 3; ++d)
            mean[d] += xyz[(size_t)d * n + ids[i]] / count;
    for (int i = first; i < last; ++i) {
        double r[3];
        for (int d = 0; d < 3; ++d)
            r[d] = xyz[(size_t)d * n + ids[i]] - mean[d];
        for (int d = 0; d < 3; ++d)
            for (int e = 0; e < 3; ++e)
                cov[d][e] += r[d] * r[e];
    }
    double v[3] = {1.0, 0.7, 0.4};   // power iteration: the split only needs a long axis
    for (int it = 0; it < 24; ++it) {
        double t[3], len = 0.0;
        for (int d = 0; d < 3; ++d) {
            t[d] = cov[d][0] * v[0] + cov[d][1] * v[1] + cov[d][2] * v[2];
            len += t[d] * t[d];
        }
        if (!(len > 0.0) || !std::isfinite(len))
            break;
        len = std::sqrt(len);
        for (int d = 0; d < 3; ++d)
            v[d] = t[d] / len;
    }
    std::vector<std::pair<double, int>> key(count);
    for (int i = 0; i < count; ++i) {
        const int id = ids[first + i];
        const double k = xyz[id] * v[0] + xyz[(size_t)n + id] * v[1] + xyz[2 * (size_t)n + id] * v[2];
        key[i] = {k == k ? k : 0.0, id};   // a NaN coordinate must not break the order
    }
    const int left = parts / 2 * chunk;
    std::nth_element(key.begin(), key.begin() + left, key.end());
    for (int i = 0; i < count; ++i)
        ids[first + i] = key[i].second;
    key = {};
    auto half = [&](int k) {
        bisect(xyz, n, ids, k ? first + left : first, k ? last : first + left, chunk);
    };
    if (count > 4096) {
        in_parallel(2, half);
    } else {
        half(0);
        half(1);
    }
}

}  // namespace

static int build(swe_hip_ctx *c, std::vector<std::vector<int>> *nbr_tiles, std::string *err)
{
    const int n = c->n, W = c->nnbr;
    SweUnits &u = c->units;
    const bool ensemble = c->B > 1, by_node = c->fp32 || exact(c);
    // ensembles: items of 16 members on tiles of 32 nodes, or 8 on 64
    u.halves = c->B > 8 ? 2 : 1;
    const int tmax = ensemble ? kEnsNodes / u.halves : std::max(16, (n + c->ncu - 1) / c->ncu);
    int nt = (n + tmax - 1) / tmax;
    const std::vector<int> &nbr = c->mesh->h_nbr;
    // kernel order: compact tiles of compact units
    const double *xyz = c->mesh->h_xyz.data();
    std::vector<int> perm(n), inv(n);
    std::iota(perm.begin(), perm.end(), 0);
    bisect(xyz, n, perm, 0, n, tmax);
    parallel_ranges(nt, 1024 / tmax, [&](int a, int b) {
        for (int t = a; t < b; ++t)
            bisect(xyz, n, perm, t * tmax, std::min(n, (t + 1) * tmax), 16);
    });
    for (int i = 0; i < n; ++i)
        inv[perm[i]] = i;
    std::vector<int> tstart(nt + 1), ustart, unit_start, own_row;
    for (int t = 0; t <= nt; ++t)
        tstart[t] = std::min(n, t * tmax);
    // distinct rows of each tile (its own nodes among them), ascending
    std::vector<std::vector<int>> list;
    std::vector<uint4> precq;
    unsigned short *prec = nullptr;
    auto list_rows = [&](int a, int b) {
        std::vector<int> mark(n, -1), where(n);
        for (int t = a; t < b; ++t) {
            std::vector<int> &l = list[t];
            for (int i = tstart[t]; i < tstart[t + 1]; ++i) {
                mark[i] = t;
                l.push_back(i);
            }
            for (int i = tstart[t]; i < tstart[t + 1]; ++i)
                for (int s = 0; s < W; ++s) {
                    const int q = inv[nbr[(size_t)s * n + perm[i]]];
                    if (mark[q] != t) {
                        mark[q] = t;
                        l.push_back(q);
                    }
                }
            std::sort(l.begin(), l.end());
            for (int k = 0; k < (int)l.size(); ++k) {
                where[l[k]] = k;
                const int o = l[k] / tmax;
                if (!ensemble && o != t && ((*nbr_tiles)[t].empty() || (*nbr_tiles)[t].back() != o))
                    (*nbr_tiles)[t].push_back(o);
            }
            own_row[t] = where[tstart[t]];
            for (int i = tstart[t]; i < tstart[t + 1]; ++i) {
                const int m = i - tstart[t];
                unsigned short *p = &prec[(size_t)(unit_start[t] + m / 16) * 512];
                for (int slot = 0; slot < W; ++slot)
                    p[prec_at(by_node, m & 15, slot)] =
                        (unsigned short)where[inv[nbr[(size_t)slot * n + perm[i]]]];
            }
        }
    };
    for (;;) {
        nt = (int)tstart.size() - 1;
        ustart.assign(nt + 1, 0);
        unit_start.assign(nt + 1, 0);
        own_row.assign(nt, 0);
        list.assign(nt, {});
        nbr_tiles->assign(nt, {});
        for (int t = 0; t < nt; ++t)
            unit_start[t + 1] = unit_start[t] + (tstart[t + 1] - tstart[t] + 15) / 16;
        precq.assign((size_t)unit_start[nt] * 64, uint4{});
        prec = reinterpret_cast<unsigned short *>(precq.data());
        parallel_ranges(nt, 1024 / tmax, list_rows);
        if (!ensemble)
            break;
        // a few tiles (icosahedral nodes, N = 163842: one of 5121, 146 rows) may
        // read more rows than an item has room for: each becomes two, of whole units
        std::vector<int> cut;
        for (int t = 0; t < nt; ++t) {
            cut.push_back(tstart[t]);
            if ((int)list[t].size() > ensemble_rows(u.halves) && tstart[t + 1] - tstart[t] > 16)
                cut.push_back(tstart[t] + 16 * ((unit_start[t + 1] - unit_start[t]) / 2));
        }
        if ((int)cut.size() == nt)
            break;
        cut.push_back(n);
        tstart = cut;
    }
    const int units = unit_start[nt];
    int rows = 0;
    for (int t = 0; t < nt; ++t) {
        ustart[t + 1] = ustart[t] + (int)list[t].size();
        rows = std::max(rows, (int)list[t].size());
    }
    std::vector<int> ulist;
    ulist.reserve(ustart[nt]);
    for (int t = 0; t < nt; ++t)
        ulist.insert(ulist.end(), list[t].begin(), list[t].end());
    // FP64 slots past the stencil read the zero row after the last
    if (!by_node)
        for (int k = 0; k < units; ++k)
            for (int slot = W; slot < 32; ++slot)
                for (int m = 0; m < 16; ++m)
                    prec[(size_t)k * 512 + prec_at(false, m, slot)] = (unsigned short)rows;
    u.ntiles = nt;
    u.all_units = units;
    u.nodes = std::min(n, tmax);
    u.units = (u.nodes + 15) / 16;
    u.rows = rows;
    // exact mode: a group of 4 nodes per wave; else the plan's
    u.waves = exact(c) ? std::max(4, (tmax + 3) / 4) : 0;
    if (ensemble)
        for (int &q : ulist)
            q = perm[q];   // rows by device node: stages exchange the state itself
    if (!(ensemble ? ensemble_plan(u)
          : exact(c) ? units_plan_exact(u) : c->fp32 ? units_plan32(u) : units_plan64(u))
        || rows > 65534) {
        *err = "unit kernel: a tile's rows do not fit the LDS";
        return SWE_HIP_EINVAL;
    }
    std::vector<int> unit_tile(units);
    for (int t = 0; t < nt; ++t)
        std::fill(unit_tile.begin() + unit_start[t], unit_tile.begin() + unit_start[t + 1], t);
    Tables tb;
    const size_t at[] = {tb.add(precq),  tb.add(tstart), tb.add(unit_start), tb.add(ustart),
                         tb.add(ulist),  tb.add(own_row), tb.add(perm),      tb.add(unit_tile)};
    int rc = 0;
    if (hipMalloc((void **)&u.d_tables, tb.bytes.size()) != hipSuccess) {
        u.d_tables = nullptr;
        *err = "unit tables: hipMalloc";
        return SWE_HIP_ENOMEM;
    }
    c->bytes += (long long)tb.bytes.size();
    u.bytes += (long long)tb.bytes.size();
    if (hipMemcpy(u.d_tables, tb.bytes.data(), tb.bytes.size(), hipMemcpyHostToDevice)
        != hipSuccess) {
        *err = "unit tables: upload";
        return SWE_HIP_EDEVICE;
    }
    auto ints = [&](int k) { return reinterpret_cast<const int *>(u.d_tables + at[k]); };
    u.d_prec = reinterpret_cast<const uint4 *>(u.d_tables + at[0]);
    u.d_tile_start = ints(1);
    u.d_unit_start = ints(2);
    u.d_ustart = ints(3);
    u.d_ulist = ints(4);
    u.d_own_row = ints(5);
    u.d_perm = ints(6);
    u.d_unit_tile = ints(7);
    if (!rc && !exact(c)) {   // the exact kernel reads the mesh itself
        rc = ensemble ? ensemble_pack(c, units)
                      : c->fp32 ? units_pack32(c, units) : units_pack64(c, units);
        if (rc)
            *err = "unit records: allocation or pack kernel";
    }
    return rc;
}

// The context's form of the records (tiles, plan and contents depend on no more).
static int form_of(const swe_hip_ctx *c)
{
    return c->B > 8 ? 2 : c->B > 1 ? 1 : exact(c) ? 3 : 0;
}

// Contexts of one mesh share the records of the form they run: N = 655362 in
// FP64 holds 0.75 GB of them.
static int share_or_build(swe_hip_ctx *c, std::vector<std::vector<int>> *nbr_tiles,
                          std::string *err)
{
    std::vector<SweUnitRecords *> &all = c->mesh->unit_records;
    std::lock_guard<std::mutex> lock(c->mesh->records_mutex);
    const auto at = std::find_if(all.begin(), all.end(), [&](const SweUnitRecords *r) {
        return r->form == form_of(c);
    });
    if (at == all.end()) {
        if (int rc = build(c, nbr_tiles, err))
            return rc;
        auto r = std::make_unique<SweUnitRecords>();
        r->u = c->units;
        r->reads = *nbr_tiles;
        r->form = form_of(c);
        r->refs = 1;
        all.push_back(r.get());
        c->units.shared = r.release();
    } else {
        c->units = (*at)->u;
        c->units.shared = *at;
        ++(*at)->refs;
        c->bytes += c->units.bytes;
        *nbr_tiles = (*at)->reads;
    }
    c->units.chains = c->fp32 && c->split32 == 2 ? 2 : 1;
    return 0;
}

int units_build(swe_hip_ctx *c, std::vector<std::vector<int>> *nbr_tiles, std::string *err)
{
    try {
        if (int rc = share_or_build(c, nbr_tiles, err))
            return rc;
    } catch (const std::bad_alloc &) {
        *err = "unit tables: out of host memory";
        return SWE_HIP_ENOMEM;
    }
    SweUnits &u = c->units;
    if (c->B == 1 && u.mode == UM_GLOBAL) {   // D of the streamed units is the context's own
        const size_t hb = (c->fp32 ? sizeof(float) : sizeof(double)) * 64 * (size_t)u.all_units;
        if (hipMalloc(&u.d_hd, hb) != hipSuccess) {
            u.d_hd = nullptr;
            *err = "unit records: allocation of D";
            return SWE_HIP_ENOMEM;
        }
        c->bytes += (long long)hb;
        u.bytes += (long long)hb;
    }
    return 0;
}

void units_tables(const swe_hip_ctx *c, int nsteps, const DevResSync &y, DevUnits *p)
{
    const SweUnits &u = c->units;
    p->y = y;
    p->tile_start = u.d_tile_start;
    p->unit_start = u.d_unit_start;
    p->ustart = u.d_ustart;
    p->ulist = u.d_ulist;
    p->own_row = u.d_own_row;
    p->perm = u.d_perm;
    p->prec = u.d_prec;
    p->nsteps = nsteps;
    p->bytes = (int)(state_count(c) * (long)(c->fp32 ? sizeof(float) : sizeof(double)));
    p->lds_rows = u.rows;
    p->lds_pos = u.pos;
    p->lds_geo = u.geo;
}

int units_prepare(swe_hip_ctx *c, std::string *err)
{
    if (c->B > 1)
        return ensemble_prepare(c, err);
    void *fn = exact(c) ? units_kernel_exact()
               : c->fp32 ? units_kernel32(c->units) : units_kernel64(c->units);
    int per_cu = 0;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kUnitsMaxLds)
            != hipSuccess
        || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 64 * c->units.waves,
                                                        c->units.lds) != hipSuccess
        || (long)per_cu * c->ncu < c->units.ntiles) {
        *err = "unit kernel: the launch cannot be co-resident on this device";
        return SWE_HIP_EDEVICE;
    }
    return 0;
}

hipError_t units_launch(swe_hip_ctx *c, int nsteps, const DevResSync &y)
{
    return exact(c) ? units_launch_exact(c, nsteps, y)
           : c->fp32 ? units_launch32(c, nsteps, y) : units_launch64(c, nsteps, y);
}

}  // namespace swe
