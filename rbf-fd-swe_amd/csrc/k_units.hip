// Whole RK4 steps of one single-state FP64 mesh in one cooperative launch,
// stencil sums on the matrix cores (fast mode, 31-point stencils).
//
// The sums.  v_mfma_f64_4x4x4f64 multiplies, for each of 4 nodes b, the 4 x 4
// weights (operator i, slot k; lane 16 k + 4 b + i) by the 4 x 4 neighbour
// states (slot k, variable j; lane 16 k + 4 b + j) into S[i][j] (lane 16 i +
// 4 b + j): exactly the shape of a single state, 8 instructions for 31 slots
// of 4 nodes.  It rounds as four fused multiply-adds in ascending k (checked
// bit for bit over 262144 random products), so the sums are those of
// k_stage_pair's fast mode, slot by slot.  Slot 31 has zero weights and reads
// a zero row.  A unit is 16 nodes, four such groups; a 4 x 4 transpose over
// the lane rows (row swaps 32, then 16 lanes apart) then gives lane (node,
// variable) its four operator sums, and the quad evaluates the RHS by DPP.
// Against two lanes per node with FMAs and DPP weight exchange (60 cycles of
// vector issue per slot and 32 nodes) the matrix cores need 16 per 4 slots
// and 4 nodes and leave the vector unit to addresses and the RHS.
//
// The data.  One workgroup per compute unit and tile, 4 to 12 waves (streaming:
// 8, two per SIMD with 256 registers): every wave keeps R units' weights (64
// registers each) for the whole launch; what the registers do not hold is read again every
// stage (UM_STREAM spills 23 registers, none inside the streamed loop), RING
// 16-byte loads per lane in flight (nothing beyond the L2 moves
// faster than 7.0 TB/s here, last-level cache or HBM, so a stage costs what it
// re-reads).  UM_GLOBAL loads the weights non-temporally: the rest, 330 bytes a
// node, then stays in the last-level cache (N = 655362 170 -> 133 us per stage;
// geometry non-temporal too: 144; UM_STREAM: no change).  Rows, positions, H, D and geometry sit in LDS as far as it goes.
// Every wave's rows of a tile are copied once per stage (res_sync.h).
//
// us per RK stage over 100 to 30 steps, against the pair-mapped resident
// kernel up to 65536 nodes and k_stage_pair above:
//   N = 2562     2.15 against 3.3    exchange latency
//   N = 10242    2.64 against 3.39   exchange latency
//   N = 40962    3.66 against 4.35   exchange latency; 0.6 us of LDS conflicts
//   N = 163842   19.4 against 32.6   111 MB re-read (16 of 41 units per tile stay)
//   N = 302762   59   against 96
//   N = 655362   133  against 197    1.30 KB per node and stage at 6.4 TB/s
#include "units.h"

#include <algorithm>

namespace swe {

struct DevUnits64 : DevUnits {
    const double2 *wrec;        // [units][4 groups][4][64 lanes] pairs of slots
    const double2 *grec;        // [units][kUnitGeo] UnitGeo of its 64 lanes
    double *H;                  // the context's state
    double *X0, *Xa, *Xb;       // exchanged states, kernel order
    double *d;                  // [units][64] D of streamed units (UM_GLOBAL; H is X0's)
    double gh0;
    double c[4];                // K = H + c F (dt/2, dt/2, dt); stage 3: H += c D (dt/6)
    double dcoef[4];            // D += dcoef F (0: D = F, 2, 2, 1)
};

constexpr int kUnitGeo = 136;   // 16-byte pieces of a unit's geometry

// A unit's geometry as its lanes hold it, (node, variable) = (lane / 4,
// lane & 3): variables u, v, w a coordinate (x, y, z) and the projection row
// of that variable, h (f, gradghm); ghm in every lane.
struct UnitGeo {
    double2 a, b;
    double ghm;
};

// G groups of 4 nodes per wave and pass (4 a whole unit; fewer on small tiles,
// RESIDENT only): lane rows 0 .. G - 1 hold nodes after the transpose.
template <int R, int MODE, int G>
__global__ __launch_bounds__(MODE == UM_RESIDENT && R == 1 ? 64 * units_waves(G) : 512)
void k_steps_units(DevUnits64 p)
{
    constexpr bool STREAM = MODE != UM_RESIDENT;
    static_assert(G == 4 || !STREAM, "whole units stream");
    constexpr int N = 4 * G;   // nodes per pass
    constexpr int RING = MODE == UM_GLOBAL ? 16 : 8;   // streamed loads in flight per lane
    extern __shared__ double2 lds[];
    const int tile = (int)blockIdx.x;
    const int t0 = p.tile_start[tile];
    const int tcount = p.tile_start[tile + 1] - t0;
    const int ug = p.unit_start[tile];
    const int nu = (tcount + N - 1) / N;
    const int u0 = p.ustart[tile];
    const int ucount = p.ustart[tile + 1] - u0;
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = (int)blockDim.x >> 6;
    const int j = lane & 3;
    const int own0 = p.own_row[tile];
    const int *ulist = p.ulist + u0;

    // LDS: rows and a zero row, positions, H and D of streamed units,
    // geometry, row ids
    char *rows = reinterpret_cast<char *>(lds);
    uint4 *pos = reinterpret_cast<uint4 *>(lds + 2 * (p.lds_rows + 1));
    double2 *hd = reinterpret_cast<double2 *>(pos + 64 * p.lds_pos);
    double2 *gl = hd + (MODE == UM_STREAM ? 64 * (p.lds_pos - R * nw) : 0);
    int *ids = reinterpret_cast<int *>(gl + kUnitGeo * p.lds_geo);
    if constexpr (MODE != UM_GLOBAL)
        for (int i = tid; i < ucount; i += (int)blockDim.x)
            ids[i] = ulist[i];
    const int n16 = p.unit_start[tile + 1] - ug;
    for (int i = tid; i < 64 * (n16 < p.lds_pos ? n16 : p.lds_pos); i += (int)blockDim.x)
        pos[i] = p.prec[64L * ug + i];
    for (int i = tid; i < kUnitGeo * (n16 < p.lds_geo ? n16 : p.lds_geo); i += (int)blockDim.x)
        gl[i] = p.grec[(long)kUnitGeo * ug + i];
    if (tid < 2)
        lds[2 * p.lds_rows + tid] = make_double2(0.0, 0.0);

    // geometry of the unit at g; l = this lane's place in it
    auto geo_of = [&](const double2 *g, int l) {
        UnitGeo r;
        r.a = g[l];
        r.b = g[64 + l];
        r.ghm = reinterpret_cast<const double *>(g + 128)[l >> 2];
        return r;
    };
    const int first = t0 + (lane >> 2);   // + N u: this lane's node of pass u
    auto mine = [&](int u) { return lane < 16 * G && N * u + (lane >> 2) < tcount; };
    double2 w[R][4 * G];
    UnitGeo gr[STREAM ? 1 : R];
    double H[R], D[R];
    static_for<R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        const int u = wv + r * nw;
        H[r] = D[r] = 0.0;
        if (u < nu) {
            // the record's next group is 256 on, across units too
            const double2 *wp = p.wrec + (long)ug * 1024 + 256L * G * u + lane;
#pragma unroll
            for (int q = 0; q < 4 * G; ++q)
                w[r][q] = wp[64 * q];
            if constexpr (!STREAM) {
                const int l = 16 * G * u + lane;   // past the tile's units: any record
                gr[r] = geo_of(p.grec + (long)kUnitGeo * (ug + (l >> 6 < n16 ? l >> 6 : 0)),
                               l & 63);
            }
            if (mine(u))
                H[r] = p.H[4L * p.perm[first + N * u] + j];
        } else {
#pragma unroll
            for (int q = 0; q < 4 * G; ++q)
                w[r][q] = make_double2(0.0, 0.0);
        }
    });
    double2 ring[STREAM ? RING : 1];
    uint4 pnext[MODE == UM_GLOBAL ? 4 : 1];
    double *const d_mem = p.d + 64L * ug + lane;
    if constexpr (STREAM) {
        for (int u = wv + R * nw; u < nu; u += nw) {
            double h = 0.0;
            if (mine(u))
                h = p.H[4L * p.perm[first + N * u] + j];
            if constexpr (MODE == UM_STREAM)
                hd[64 * (u - R * nw) + lane] = make_double2(h, 0.0);
            else if (mine(u))
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, h),
                                                      state_rsrc(p.X0, p.bytes),
                                                      8 * (4 * t0 + 4 * N * u + lane), 0, kSc1);
        }
        const int u = wv + R * nw;
        if (u < nu) {
            const double2 *wp = p.wrec + (long)(ug + u) * 1024 + lane;
#pragma unroll
            for (int q = 0; q < RING; ++q)
                ring[q] = wp[64 * q];
            if constexpr (MODE == UM_GLOBAL) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    pnext[q] = p.prec[64L * (ug + u) + 16 * q + (lane >> 2)];
            }
        }
    }
    unsigned stage = p.y.stage0;
    bool alive = true;

    // stencil sums of one group of 4 nodes: lane (i, b, x) accumulates
    // operator i of node b, variable x
    auto group = [&](const double2 *wg, uint4 pv) {
        const unsigned pw[4] = {pv.x, pv.y, pv.z, pv.w};
        double acc = 0.0;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const unsigned row = (s & 1) ? (pw[s >> 1] >> 16) : (pw[s >> 1] & 0xffffu);
            const double b = *reinterpret_cast<const double *>(rows + (row << 5 | 8u * j));
            acc = __builtin_amdgcn_mfma_f64_4x4x4f64((s & 1) ? wg[s >> 1].y : wg[s >> 1].x, b,
                                                     acc, 0, 0, 0);
        }
        return acc;
    };
    // RHS of this lane's (node, variable), operation order of rhs_point
    auto rhs = [&](int u, double (&acc)[4], const UnitGeo &g) {
        double x0 = acc[0], x1 = acc[1], x2 = acc[2], x3 = acc[3];
        swap_rows32(x0, x2);
        swap_rows32(x1, x3);
        swap_rows16(x0, x1);
        swap_rows16(x2, x3);
        // x0..x3: Dx, Dy, Dz, L sums of variable j of node N u + lane / 4
        const double2 *own = lds + 2 * (own0 + N * u + (lane >> 2));
        const double2 uv = own[0], wh = own[1];
        const bool k3 = j == 3;
        const double s1 = j == 0 ? wh.x : (j == 1 ? uv.x : uv.y);
        const double s2 = j == 0 ? uv.y : (j == 1 ? wh.x : uv.x);
        const double c1 = quad_perm<1, 2, 0, 3>(g.a.x), c2 = quad_perm<2, 0, 1, 3>(g.a.x);
        const double f = quad_bcast<3>(g.a.x);
        const double dh0 = quad_bcast<3>(x0), dh1 = quad_bcast<3>(x1), dh2 = quad_bcast<3>(x2);
        const double dh = j == 0 ? dh0 : (j == 1 ? dh1 : dh2);
        const double div = (quad_bcast<0>(x0) + quad_bcast<1>(x1)) + quad_bcast<2>(x2);
        const double a0 = k3 ? x0 - g.a.y : x0;
        const double a1 = k3 ? x1 - g.b.x : x1;
        const double a2 = k3 ? x2 - g.b.y : x2;
        const double t = ((uv.x * a0) + (uv.y * a1)) + (wh.x * a2);
        const double cor = f * ((c1 * s1) - (c2 * s2));
        const double hx = (wh.y + p.gh0 - g.ghm) * div;
        const double t1 = t + (k3 ? hx : cor);
        const double t2 = t1 + dh;
        const double r = -(k3 ? t1 : t2);
        const double ru = quad_bcast<0>(r), rv = quad_bcast<1>(r), rw = quad_bcast<2>(r);
        const double pr = ((g.a.y * ru) + (g.b.x * rv)) + (g.b.y * rw);
        return (k3 ? r : pr) + x3;
    };

    for (int step = 0; step < p.nsteps && alive; ++step) {
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (!alive)
                return;
            const double *src = s == 0 ? p.X0 : (s == 2 ? p.Xb : p.Xa);
            double *out = s == 0 ? p.Xa : (s == 1 ? p.Xb : (s == 2 ? p.Xa : p.X0));
            if (!(alive = res_wait(p.y, tile, stage)))   // also: ids written, rows free
                return;
            // 32 rows per wave and instruction, two lanes per row; the first
            // stage gathers the state buffer itself
            const bool head = s == 0 && step == 0;
            const double *b = (head ? p.H : src) + 2 * (lane & 1);
            for (int i0 = 32 * wv; i0 < ucount; i0 += 32 * nw) {
                const int i = i0 + (lane >> 1);
                if (i < ucount) {
                    int id = MODE == UM_GLOBAL ? ulist[i] : ids[i];
                    if (head)
                        id = p.perm[id];
                    dma16_sc1(b + 4L * id, rows + 32L * i0);
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            const bool last = s == 3 && step == p.nsteps - 1;
            auto update = [&](int u, double F, double &Hv, double &Dv) {
                double K;
                if constexpr (s == 0) {
                    Dv = F;
                    K = axpy<false>(Hv, p.c[0], F);
                } else if constexpr (s == 1 || s == 2) {
                    Dv = axpy<false>(Dv, p.dcoef[s], F);
                    K = axpy<false>(Hv, p.c[s], F);
                } else {
                    const double d = axpy<false>(Dv, p.dcoef[3], F);
                    K = Hv = axpy<false>(Hv, p.c[3], d);
                }
                if (mine(u)) {
                    const int e = last ? 4 * p.perm[first + N * u] + j
                                       : 4 * t0 + 4 * N * u + lane;
                    __builtin_amdgcn_raw_buffer_store_b64(
                        __builtin_bit_cast(u32x2, K), state_rsrc(last ? p.H : out, p.bytes),
                        8 * e, 0, kSc1);
                }
            };
            static_for<R>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                const int u = wv + r * nw;
                if (u < nu) {
                    UnitGeo g;
                    if constexpr (!STREAM)
                        g = gr[r];
                    else if (MODE == UM_STREAM && u < p.lds_geo)
                        g = geo_of(gl + kUnitGeo * u, lane);
                    else
                        g = geo_of(p.grec + (long)kUnitGeo * (ug + u), lane);
                    double acc[4] = {0.0, 0.0, 0.0, 0.0};
                    const uint4 *pu = pos + 16 * G * u + (lane >> 2);
#pragma unroll
                    for (int q = 0; q < G; ++q)
                        acc[q] = group(w[r] + 4 * q, pu[16 * q]);
                    update(u, rhs(u, acc, g), H[r], D[r]);
                }
            });
            if constexpr (STREAM) {
#pragma unroll 1
                for (int u = wv + R * nw; u < nu; u += nw) {
                    const int un = u + nw < nu ? u + nw : wv + R * nw;   // next, wrapping
                    const double2 *wc = p.wrec + (long)(ug + u) * 1024 + lane;
                    const double2 *wn = p.wrec + (long)(ug + un) * 1024 + lane;
                    UnitGeo g;
                    uint4 pv[4];
                    double2 hv;
                    if constexpr (MODE == UM_STREAM) {
                        if (u < p.lds_geo)
                            g = geo_of(gl + kUnitGeo * u, lane);
                        else
                            g = geo_of(p.grec + (long)kUnitGeo * (ug + u), lane);
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            pv[q] = pos[64 * u + 16 * q + (lane >> 2)];
                    } else {
                        g = geo_of(p.grec + (long)kUnitGeo * (ug + u), lane);
                        // stage 0 gathers H: it is in the own row
                        if constexpr (s == 0) {
                            hv.x = *reinterpret_cast<const double *>(
                                rows + 32 * (own0 + 16 * u + (lane >> 2)) + 8 * j);
                        } else {
                            hv.x = __builtin_bit_cast(
                                double, __builtin_amdgcn_raw_buffer_load_b64(
                                            state_rsrc(p.X0, p.bytes),
                                            8 * (4 * t0 + 4 * N * u + lane), 0, kSc1));
                            hv.y = d_mem[64L * u];
                        }
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            pv[q] = pnext[q];
                            pnext[q] = p.prec[64L * (ug + un) + 16 * q + (lane >> 2)];
                        }
                    }
                    double acc[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        constexpr int AHEAD = RING / 4;   // groups in flight
                        acc[q] = group(ring + 4 * (q % AHEAD), pv[q]);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const double2 *from = q + AHEAD < 4
                                                      ? wc + 64 * (4 * (q + AHEAD) + i)
                                                      : wn + 64 * (4 * (q + AHEAD - 4) + i);
                            ring[4 * (q % AHEAD) + i] =
                                MODE == UM_GLOBAL ? load_nt(from) : *from;
                        }
                    }
                    if constexpr (MODE == UM_STREAM)
                        hv = hd[64 * (u - R * nw) + lane];
                    update(u, rhs(u, acc, g), hv.x, hv.y);
                    if constexpr (MODE == UM_STREAM)
                        hd[64 * (u - R * nw) + lane] = hv;
                    else if constexpr (s < 3)
                        d_mem[64L * u] = hv.y;
                }
            }
            res_publish(p.y, tile, ++stage);
        });
    }
}

// Packs the weight records: one workgroup per unit, thread = (group and slot
// pair, lane).
__global__ void k_pack_weights(DevMesh m, const int *tile_start, const int *unit_start,
                               const int *unit_tile, const int *perm, double2 *wrec)
{
    const int unit = (int)blockIdx.x;
    const int tile = unit_tile[unit];
    const int lane = (int)threadIdx.x & 63, q = (int)threadIdx.x >> 6;
    const int g = q >> 2, k = lane >> 4, b = (lane >> 2) & 3, x = lane & 3;
    const int node = tile_start[tile] + 16 * (unit - unit_start[tile]) + 4 * g + b;
    double v[2] = {0.0, 0.0};
    for (int c = 0; c < 2; ++c) {
        const int slot = 4 * (2 * (q & 3) + c) + k;
        if (node < tile_start[tile + 1] && slot < m.nnbr)
            v[c] = m.wts[4L * (slot_base<0>(m, perm[node]) + (long)slot * slot_stride(m)) + x];
    }
    wrec[(long)unit * 1024 + 64 * q + lane] = make_double2(v[0], v[1]);
}

// Packs the geometry records: one workgroup per unit, thread = (piece, lane).
__global__ void k_pack_geo(DevMesh m, const int *tile_start, const int *unit_start,
                           const int *unit_tile, const int *perm, double2 *grec)
{
    const int unit = (int)blockIdx.x;
    const int tile = unit_tile[unit];
    const int lane = (int)threadIdx.x & 63, q = (int)threadIdx.x >> 6;
    const int j = lane & 3;
    const int node = tile_start[tile] + 16 * (unit - unit_start[tile])
                     + (q < 2 ? lane >> 2 : lane & 15);
    const int n1 = tile_start[tile + 1];
    const int field[4][4] = {{G_X, G_PU, G_PU + 1, G_PU + 2},
                             {G_Y, G_PV, G_PV + 1, G_PV + 2},
                             {G_Z, G_PW, G_PW + 1, G_PW + 2},
                             {G_F, G_GG, G_GG + 1, G_GG + 2}};
    auto fetch = [&](int f) { return node < n1 ? m.geo[(long)f * m.ld + perm[node]] : 0.0; };
    double2 *gu = grec + (long)kUnitGeo * unit;
    if (q < 2)
        gu[64 * q + lane] = make_double2(fetch(field[j][2 * q]), fetch(field[j][2 * q + 1]));
    else if (lane < 16)
        reinterpret_cast<double *>(gu + 128)[lane] = fetch(G_GHM);
}

void pack_weights64(swe_hip_ctx *c, int units)
{
    const SweUnits &u = c->units;
    k_pack_weights<<<units, 1024, 0, c->stream>>>(mesh_of(c), u.d_tile_start, u.d_unit_start,
                                                  u.d_unit_tile, u.d_perm,
                                                  static_cast<double2 *>(u.d_wrec));
}

// All weights resident: one pass of 1, 2 or 4 groups per wave, the fewest that
// leave one wave per SIMD (what a wave does in a stage is a chain of latencies,
// 1820 cycles for 4 groups alone: N = 2562 2.15 against 2.51 us per stage, 7292
// 2.33 against 2.57; with more waves of fewer groups the RHS, which costs a
// wave the same for 4 nodes as for 16, is what is issued: N = 16002 2.90 on 16
// waves against 2.71 on 4), on at most 12 waves (40962 3.66 against 3.78 with
// two passes on 8), else two passes of a unit on 8.
bool units_plan64(SweUnits &u)
{
    const int groups = (u.nodes + 3) / 4;
    u.groups = groups <= 4 ? 1 : groups <= 8 ? 2 : 4;
    u.waves = std::max(4, (groups + u.groups - 1) / u.groups);
    if (u.waves > units_waves(u.groups))
        u.waves = 8;
    const int kept = u.waves > 8 ? u.waves : 2 * u.waves;
    long lds = 32L * (u.rows + 1);
    if (u.groups < 4 || u.units <= kept) {
        u.mode = UM_RESIDENT;
        u.pos = u.units;
        lds += 1024L * u.pos + 4L * u.rows;
    } else if (lds + 1024L * (2 * u.units - kept) + 4L * u.rows <= kUnitsMaxLds) {
        u.mode = UM_STREAM;
        u.pos = u.units;
        lds += 1024L * (2 * u.units - kept) + 4L * u.rows;
        u.geo = (int)std::min((long)u.units, (kUnitsMaxLds - lds) / (16 * kUnitGeo));
        lds += 16L * kUnitGeo * u.geo;
    } else {
        u.mode = UM_GLOBAL;
        u.pos = u.waves;
        lds += 1024L * u.pos;
    }
    u.lds = (int)lds;
    return lds <= kUnitsMaxLds;
}

void *units_kernel64(const SweUnits &u)
{
    switch (u.mode) {
    case UM_STREAM: return reinterpret_cast<void *>(&k_steps_units<2, UM_STREAM, 4>);
    case UM_GLOBAL: return reinterpret_cast<void *>(&k_steps_units<1, UM_GLOBAL, 4>);
    default: break;
    }
    if (u.groups == 1)
        return reinterpret_cast<void *>(&k_steps_units<1, UM_RESIDENT, 1>);
    if (u.groups == 2)
        return reinterpret_cast<void *>(&k_steps_units<1, UM_RESIDENT, 2>);
    return u.units > u.waves ? reinterpret_cast<void *>(&k_steps_units<2, UM_RESIDENT, 4>)
                             : reinterpret_cast<void *>(&k_steps_units<1, UM_RESIDENT, 4>);
}

int units_pack64(swe_hip_ctx *c, int units)
{
    SweUnits &u = c->units;
    const size_t wb = sizeof(double2) * 1024 * (size_t)units;
    const size_t gb = sizeof(double2) * kUnitGeo * (size_t)units;
    if (hipMalloc(&u.d_wrec, wb) != hipSuccess || hipMalloc(&u.d_grec, gb) != hipSuccess)
        return SWE_HIP_ENOMEM;
    c->bytes += (long long)(wb + gb);
    u.bytes += (long long)(wb + gb);
    pack_weights64(c, units);
    k_pack_geo<<<units, 192, 0, c->stream>>>(mesh_of(c), u.d_tile_start, u.d_unit_start,
                                             u.d_unit_tile, u.d_perm,
                                             static_cast<double2 *>(u.d_grec));
    return hipGetLastError() == hipSuccess && hipStreamSynchronize(c->stream) == hipSuccess
               ? 0 : SWE_HIP_EDEVICE;
}

hipError_t units_launch64(swe_hip_ctx *c, int nsteps, const DevResSync &y)
{
    const SweUnits &u = c->units;
    DevUnits64 p{};
    units_tables(c, nsteps, y, &p);
    p.wrec = static_cast<const double2 *>(u.d_wrec);
    p.grec = static_cast<const double2 *>(u.d_grec);
    p.d = static_cast<double *>(u.d_hd);
    p.H = c->d_H;
    p.X0 = c->d_D;   // D lives in the kernel
    p.Xa = c->d_Ka;
    p.Xb = c->d_Kb;
    p.gh0 = c->gh0;
    const double dt = c->dt;
    p.c[0] = dt / 2.0; p.c[1] = dt / 2.0; p.c[2] = dt; p.c[3] = dt / 6.0;
    p.dcoef[0] = 0.0; p.dcoef[1] = 2.0; p.dcoef[2] = 2.0; p.dcoef[3] = 1.0;
    void *args[] = {&p};
    return hipLaunchCooperativeKernel(units_kernel64(u), dim3(u.ntiles), dim3(64 * u.waves), args,
                                      (unsigned)u.lds, c->stream);
}

}  // namespace swe
