// Ensemble stage kernel on the matrix cores (fast mode, 31-point stencils).
//
// An item is a compact tile (recursive bisection, swe_units.hip) of 32 nodes
// for 16 members, or 64 nodes for 8 where the ensemble has no more; a wave
// takes a 16-node unit for 8 members.  v_mfma_f64_4x4x4f64 multiplies the
// weights of 4 nodes (operator, slot), kept in registers over a tile's member
// blocks, by one variable of their neighbours for 4 members (slot, member):
// one 16-byte LDS read per lane feeds two instructions (members 2 j and
// 2 j + 1).  The instruction rounds as four FMAs in slot order (k_units.hip),
// so every member's bits are those of k_stage_members and of a single run.
// A transpose over the lane rows gives lane (node, two members) all 32 sums;
// the RHS and the update need no exchange.
//
// A tile's distinct rows (4.2 per node at 32 nodes, against 8.9 for the 8-node
// tiles of k_stage_tspec) go straight to LDS; the next member block's are asked
// for before the RHS runs.  What the compiler makes of it overlaps less than that
// order promises: it drains the wave's memory counter before H and D are asked
// for (their addresses and registers depend on loads and branches of the item
// before), so every row copy and store has ended by then, and again before the
// update, since the row copies after H and D are not a fixed number.  Across
// tiles nothing is asked for early.  The two workgroups of a compute unit overlap
// each other.  16 members make every access a whole 128-byte line: with 8 a
// launch fetched 2.5 GB instead of 1.4 at N = 163842 x 64 (531 against 465 us).
//
// us per launch: N = 163842 x 64 461 against 474 (k_stage_tspec, side by side); of
// that the traffic alone takes 354 (2.05 GB), the arithmetic alone 283 (221
// without LDS bank conflicts).  Against k_stage_members, the default before: N = 10242 x
// 2, 8, 16: 9.2, 9.8, 14.5 against 15, 22.6, 41.8; 40962 x 8, 32: 27, 67
// against 80, 257; 642 x 2: 8.7 against 15.
#include "units.h"

#include <algorithm>

namespace swe {

struct DevEnsemble {
    const int *tile_start;      // [ntiles + 1] first node (kernel order)
    const int *ustart;          // [ntiles + 1] offsets into ulist
    const int *ulist;           // distinct rows of each tile, device nodes
    const int *own_row;         // [ntiles] row number of the tile's first node
    const int *perm;            // kernel node -> device node
    const int *unit_start;      // [ntiles + 1]
    const uint4 *prec;          // [units][64] row numbers, as k_steps_units
    const double2 *wrec;        // [units][16][64] weights, as k_steps_units
    const double2 *geo;         // [units][16 nodes][kEnsGeo] geometry
    int ntiles;
    int lds_rows;               // rows the LDS holds; the row after them is zero
};

constexpr int kEnsGeo = 9;       // 16-byte pieces of a node's geometry

// Two row numbers (at most 254) to half the byte offsets of chunk 0 in LDS.
template <int HALVES>
__device__ __forceinline__ unsigned chunk_of(unsigned r)
{
    constexpr unsigned m = 4 * HALVES - 1;
    return (r & 0x00ff00ffu) << (6 + HALVES) | (r & (m << 16 | m)) << 5;
}

// Waits until at most N of this wave's later memory operations are in flight.
template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N < 16, "low four bits of the count");
    __builtin_amdgcn_s_waitcnt(0xf70 | N);
}

template <int STAGE, int HALVES>
__global__ __launch_bounds__(256, 2) void k_stage_ensemble(DevEnsemble p, DevStage st, double gh0)
{
    constexpr int MEMBERS = 8 * HALVES;      // members per item
    constexpr int UNITS = 4 / HALVES;        // units per tile
    constexpr int CHUNKS = 4 * HALVES;       // 64-byte chunks of a row: (variable, half)
    constexpr int ROW = 64 * CHUNKS;         // bytes of a row
    constexpr int PER = 64 / (4 * CHUNKS);   // rows one wave instruction copies
    extern __shared__ double2 lds[];
    // LDS: rows [row][chunk][8 members] and a zero row, positions of the
    // tile's units, geometry, row ids
    char *rows = reinterpret_cast<char *>(lds);
    uint4 *pos = reinterpret_cast<uint4 *>(rows + ROW * (p.lds_rows + 1));
    double2 *geo = reinterpret_cast<double2 *>(pos + 64 * UNITS);
    int *ids = reinterpret_cast<int *>(geo + 16 * UNITS * kEnsGeo);
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int uw = wv % UNITS, half = wv / UNITS;   // this wave's unit and members
    const int j = lane & 3;
    const long B = st.members;
    const int active = c_i32(st.active);
    const int nmb = (active + MEMBERS - 1) / MEMBERS;
    // XCD x (workgroups are dealt round-robin over the 8) owns tiles [x0, x1);
    // its W workgroups take whole tiles W apart, so that the tiles in flight
    // are neighbours and share halo rows in that L2; the tiles left over are
    // shared out by member block.
    const int W = (int)gridDim.x >> 3, me = (int)blockIdx.x >> 3, xcd = (int)blockIdx.x & 7;
    const int x0 = (int)((long)p.ntiles * xcd / 8), x1 = (int)((long)p.ntiles * (xcd + 1) / 8);
    const int rounds = (x1 - x0) / W;
    const int rest = (x1 - x0 - rounds * W) * nmb;       // items left over
    const int share = (rest + W - 1) / W;
    if (tid < ROW / 16)
        lds[ROW / 16 * p.lds_rows + tid] = make_double2(0.0, 0.0);

    double2 w[16];
    const int nl = 16 * uw + (lane >> 2);   // this lane's node of the tile
    int tcount = 0, ucount = 0, own0 = 0, dn = 0;
    auto copy_rows = [&](int mb) {
        // lane (row, chunk, 2 members); row i keeps chunk c at c ^ (i mod
        // CHUNKS): the 16 rows of one stencil read would otherwise share banks
        const int part = lane & 3, at = (lane >> 2) & (CHUNKS - 1), sub = lane / (4 * CHUNKS);
        for (int i0 = PER * wv; i0 < ucount; i0 += 4 * PER) {
            const int i = i0 + sub;
            const int c = at ^ (i & (CHUNKS - 1));
            const int mem = MEMBERS * mb + 8 * (c % HALVES) + 2 * part;
            if (i < ucount && mem < B)
                dma16(st.src + (4L * ids[i] + c / HALVES) * B + mem,
                      reinterpret_cast<double *>(rows + (long)ROW * i0));
        }
    };

    for (int r = 0; r <= rounds; ++r) {
        // this workgroup's items of the round: tile, member blocks [m0, m1)
        int first = me * share, last = min(first + share, rest);
        if (r < rounds) {
            first = me * nmb + r * W * nmb;
            last = first + nmb;
        } else {
            first += rounds * W * nmb;
            last += rounds * W * nmb;
        }
        int have = -1;   // tile whose tables are in LDS
        for (int it = first; it < last; ++it) {
            const int tile = x0 + it / nmb, mb = it - (it / nmb) * nmb;
            if (tile != have) {
                have = tile;
                const int t0 = c_i32(p.tile_start + tile);
                tcount = c_i32(p.tile_start + tile + 1) - t0;
                const int u0 = c_i32(p.ustart + tile);
                ucount = c_i32(p.ustart + tile + 1) - u0;
                own0 = c_i32(p.own_row + tile);
                const int ug = c_i32(p.unit_start + tile);
                const int nu = c_i32(p.unit_start + tile + 1) - ug;
                dn = p.perm[t0 + (nl < tcount ? nl : 0)];
                __syncthreads();   // the previous tile's LDS is free
                if (tid < ucount)   // at most 254 rows
                    ids[tid] = p.ulist[u0 + tid];
                // the missing units of a last or cut tile read the zero row
                const unsigned z = (unsigned)p.lds_rows << 16 | (unsigned)p.lds_rows;
                if (tid < 64 * UNITS) {
                    const uint4 pr =
                        tid < 64 * nu ? p.prec[64L * ug + tid] : make_uint4(z, z, z, z);
                    pos[tid] = make_uint4(chunk_of<HALVES>(pr.x), chunk_of<HALVES>(pr.y),
                                          chunk_of<HALVES>(pr.z), chunk_of<HALVES>(pr.w));
                }
                for (int i = tid; i < 16 * kEnsGeo * nu; i += 256)
                    geo[i] = p.geo[16L * kEnsGeo * ug + i];
                const double2 *wp = p.wrec + (long)(ug + (uw < nu ? uw : 0)) * 1024 + lane;
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    w[q] = wp[64 * q];
                __syncthreads();
                copy_rows(mb);
            }
            const int mem = MEMBERS * mb + 8 * half + 2 * j;   // this lane's two members
            const bool live = nl < tcount && mem < B;
            const long e = 4L * dn * B + (mem < B ? mem : 0);
            // H and D on their way before the rows' barrier
            double2 hv[4], dv[4];
            constexpr int OWN = STAGE == ST_RHS || STAGE == ST_0 ? 0 : 8;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (OWN > 0) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    hv[v] = *reinterpret_cast<const double2 *>(st.h + e + v * B);
                    dv[v] = *reinterpret_cast<const double2 *>(st.d + e + v * B);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // this wave's rows are in LDS: at most the OWN loads after them are
            // still out (the compiler has already waited for all before those)
            wait_vm<OWN>();
            __syncthreads();
            // operator sums: acc[g][v] in lane (operator i, node b of group g,
            // members 2 j and 2 j + 1)
            double acc[4][4][2];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint4 pv = pos[64 * uw + 16 * g + (lane >> 2)];
                const unsigned pw[4] = {pv.x, pv.y, pv.z, pv.w};
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[g][v][0] = acc[g][v][1] = 0.0;
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const unsigned off = (s & 1) ? (pw[s >> 1] >> 16) : (pw[s >> 1] & 0xffffu);
                    const unsigned at = (off << 1 | 16u * j) ^ 64u * half;
                    const double a = (s & 1) ? w[4 * g + (s >> 1)].y : w[4 * g + (s >> 1)].x;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const double2 b =
                            *reinterpret_cast<const double2 *>(
                                rows + (at ^ 64u * HALVES * v));
                        acc[g][v][0] =
                            __builtin_amdgcn_mfma_f64_4x4x4f64(a, b.x, acc[g][v][0], 0, 0, 0);
                        acc[g][v][1] =
                            __builtin_amdgcn_mfma_f64_4x4x4f64(a, b.y, acc[g][v][1], 0, 0, 0);
                    }
                }
            }
            const int nc = nl < tcount ? nl : 0;
            double2 own[4];
#pragma unroll
            for (int v = 0; v < 4; ++v)
                own[v] = *reinterpret_cast<const double2 *>(
                    rows + ROW * (own0 + nc)
                    + 64 * ((HALVES * v + half) ^ ((own0 + nc) & (CHUNKS - 1))) + 16 * j);
            Geo gq;
            {
                const double2 *gp = geo + kEnsGeo * nc;
                const double2 g0 = gp[0], g1 = gp[1], g2 = gp[2], g3 = gp[3], g4 = gp[4],
                              g5 = gp[5], g6 = gp[6], g7 = gp[7], g8 = gp[8];
                gq.x = g0.x; gq.y = g0.y; gq.z = g1.x; gq.f = g1.y; gq.ghm = g2.x;
                gq.pu0 = g2.y; gq.pu1 = g3.x; gq.pu2 = g3.y;
                gq.pv0 = g4.x; gq.pv1 = g4.y; gq.pv2 = g5.x;
                gq.pw0 = g5.y; gq.pw1 = g6.x; gq.pw2 = g6.y;
                gq.gx = g7.x; gq.gy = g7.y; gq.gz = g8.x;
            }
            __syncthreads();   // every wave has read its rows
            if (it + 1 < last && (it + 1) / nmb == it / nmb)
                copy_rows(mb + 1);
            // to lane (node, members): groups against lane rows
            double2 F[4];
#pragma unroll
            for (int m2 = 0; m2 < 2; ++m2) {
                double T[4][4];   // [variable][operator]
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    double a0 = acc[0][v][m2], a1 = acc[1][v][m2], a2 = acc[2][v][m2],
                           a3 = acc[3][v][m2];
                    swap_rows32(a0, a2);
                    swap_rows32(a1, a3);
                    swap_rows16(a0, a1);
                    swap_rows16(a2, a3);
                    T[v][0] = a0; T[v][1] = a1; T[v][2] = a2; T[v][3] = a3;
                }
                Sums S;
                S.dudx = T[0][0]; S.dudy = T[0][1]; S.dudz = T[0][2]; S.lu = T[0][3];
                S.dvdx = T[1][0]; S.dvdy = T[1][1]; S.dvdz = T[1][2]; S.lv = T[1][3];
                S.dwdx = T[2][0]; S.dwdy = T[2][1]; S.dwdz = T[2][2]; S.lw = T[2][3];
                S.dhdx = T[3][0]; S.dhdy = T[3][1]; S.dhdz = T[3][2]; S.lh = T[3][3];
                double f[4];
                rhs_point(S, m2 ? own[0].y : own[0].x, m2 ? own[1].y : own[1].x,
                          m2 ? own[2].y : own[2].x, m2 ? own[3].y : own[3].x, gq, gh0, f);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (m2)
                        F[v].y = f[v];
                    else
                        F[v].x = f[v];
                }
            }
            if (live) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if constexpr (STAGE == ST_0)
                        hv[v] = own[v];   // stage 0 gathers H
                    stage_update_pre_pair<STAGE, false>(st, e + v * B, F[v], hv[v], dv[v]);
                }
            }
        }
    }
}

// Geometry records: [unit][16 nodes][kEnsGeo], the fields in Geo's order.
__global__ void k_pack_ensemble(DevMesh m, const int *tile_start, const int *unit_start,
                                const int *unit_tile, const int *perm, double *geo)
{
    const int unit = (int)blockIdx.x, tile = unit_tile[unit];
    const int nl = (int)threadIdx.x / (2 * kEnsGeo), f = (int)threadIdx.x % (2 * kEnsGeo);
    const int node = tile_start[tile] + 16 * (unit - unit_start[tile]) + nl;
    geo[(16L * unit + nl) * 2 * kEnsGeo + f] =
        node < tile_start[tile + 1] && f < GEO_N ? m.geo[(long)f * m.ld + perm[node]] : 0.0;
}

static int ensemble_lds(int halves, int rows)
{
    const int nodes = kEnsNodes / halves;
    return 256 * halves * (rows + 1) + 64 * nodes + 16 * nodes * kEnsGeo + 4 * rows;
}

int ensemble_rows(int halves)
{
    // two workgroups per compute unit, 16-bit row offsets
    return std::min(254, (kUnitsMaxLds / 2 - ensemble_lds(halves, 0)) / (256 * halves + 4));
}

// Items of 32 nodes x 16 members (64 x 8) of one XCD, and the turns its
// workgroups need for them.
static void ensemble_items(int n, int members, int ncu, long *items, long *turns, long *width)
{
    const int halves = members > 8 ? 2 : 1, nodes = kEnsNodes / halves;
    const long nmb = (members + 8 * halves - 1) / (8 * halves);
    const long tiles = ((n + nodes - 1) / nodes + 7) / 8, W = (2L * ncu + 7) / 8;
    *items = tiles * nmb;
    *turns = tiles / W * nmb + (tiles % W * nmb + W - 1) / W;
    *width = W;
}

// Whether the items of a stage keep the workgroups busy: at least 95 % of the
// turns the longest of them takes.  Members in blocks of 16 on 32 nodes make
// coarse items: against k_stage_tspec (whole calls, all members active) N =
// 4412 x 64 is 0.73 as fast at 54 %, 12252 x 32 0.88 at 75 %, 10242 x 64 0.91 at
// 84 %, 60842 x 32 0.95 at 93 %, but 90252 x 64 1.06 at 96 %, 16002 x 64 1.04 at
// 98 %, 116642 x 96 1.11 at 99 %.  Not before the fourth turn, up to which 12 to 14
// us a turn instead of 11 keep it behind (12252 x 64 0.97 in three full ones,
// 16002 x 32 0.96 in two).
bool ensemble_fills(int n, int members, int ncu)
{
    long items, turns, W;
    ensemble_items(n, members, ncu, &items, &turns, &W);
    return turns >= 4 && 20 * items >= 19 * turns * W;
}

// Whether an ensemble that names no member block runs this kernel.  Against
// k_stage_members, the choice where 64 does not divide the members, it always
// does (1.2 to 4.4 times as fast); k_stage_mpair's items are finer, and it is the
// better one until 80 % of the turns are busy (in the first turn: half of
// them, so that both workgroups of a compute unit are).  Against it, per
// stage: N = 642 x 64 0.94 at 19 %, 1962 x 64 0.95 at 50 %, 5762 x 64 0.87 at 72 %,
// 2562 x 192 0.87 at 69 %, 3242 x 192 1.01 at 81 %, 10242 x 64 1.05 at 85 %, 7842
// x 64 1.09 at 97 %, first turn 2252 x 64 1.06 at 56 %.  Fewer than two tiles per
// XCD are too uneven to tell (362 x 320 0.80).
bool ensemble_default(int n, int members, int ncu)
{
    if (members % 64)
        return true;
    long items, turns, W;
    ensemble_items(n, members, ncu, &items, &turns, &W);
    return n >= 16 * kEnsNodes / 2 && (turns == 1 ? 2 * items > W : 5 * items >= 4 * turns * W);
}

// Whether a launch of a batch context (tiles and records) runs this kernel.  It
// works on blocks of 16 active members, k_stage_tspec on whole slots: measured
// over 642 to 163842 nodes x 32 to 128 slots, the one takes 9 to 14 us in the first
// turn and 11 to 13 per turn beyond, the other 3.5 us and 4.5e-5 per node and slot,
// a tenth less when one block of 32 is active.  N = 10242 x 64: 16, 32, 48 and 64
// active members 14.2, 25.3, 26.8, 37.1 against 32.1, 32.1, 32.7, 32.7; 2562 x 64: 9.1,
// 9.6, 11.3, 13.5 against 11.4, 11.0, 11.7, 11.7; 642 x 64: 9 against 6.  Beside
// other batches the compute units that turns leave idle are not lost, so only the
// floor of a turn counts: two full batches of 64 slots at once take 0.88 of
// k_stage_tspec's time at N = 2562, 10242 and 40962, but 1.36 at 642.
bool ensemble_batch(int n, int slots, int active, bool alone, int ncu)
{
    long items, turns, W;
    ensemble_items(n, std::max(active, 9), ncu, &items, &turns, &W);
    const double mine = !alone ? 9.3 : turns > 1 ? 13.0 * turns : 2 * items > W ? 14.0 : 9.3;
    const double blocks = (double)((active + 31) / 32) / (slots / 32.0);
    return mine <= 3.5 + 4.5e-5 * n * slots * (0.9 + 0.1 * blocks);
}

long long ensemble_bytes(int n)
{
    // tiles of two units: weights, geometry, positions, rows, their owners
    const long long tile = 2 * (16 * 1024 + 16 * 16 * kEnsGeo + 1024) + 4 * 2 * 254 + 64;
    return (n / (kEnsNodes / 2) + 1) * tile + 4LL * n + 8 * 256;
}

bool ensemble_plan(SweUnits &u)
{
    u.mode = UM_RESIDENT;
    u.waves = 4;
    u.lds = ensemble_lds(u.halves, u.rows);
    return u.rows <= ensemble_rows(u.halves);
}

int ensemble_pack(swe_hip_ctx *c, int units)
{
    SweUnits &u = c->units;
    const size_t wb = sizeof(double2) * 1024 * (size_t)units;
    const size_t gb = sizeof(double2) * 16 * kEnsGeo * (size_t)units;
    if (hipMalloc(&u.d_wrec, wb) != hipSuccess || hipMalloc(&u.d_grec, gb) != hipSuccess)
        return SWE_HIP_ENOMEM;
    c->bytes += (long long)(wb + gb);
    u.bytes += (long long)(wb + gb);
    pack_weights64(c, units);
    k_pack_ensemble<<<units, 16 * 2 * kEnsGeo, 0, c->stream>>>(
        mesh_of(c), u.d_tile_start, u.d_unit_start, u.d_unit_tile, u.d_perm,
        static_cast<double *>(u.d_grec));
    return hipGetLastError() == hipSuccess && hipStreamSynchronize(c->stream) == hipSuccess
               ? 0 : SWE_HIP_EDEVICE;
}

template <int HALVES>
static void *ensemble_kernel(int stage)
{
    switch (stage) {
    case ST_0: return reinterpret_cast<void *>(&k_stage_ensemble<ST_0, HALVES>);
    case ST_1: return reinterpret_cast<void *>(&k_stage_ensemble<ST_1, HALVES>);
    case ST_2: return reinterpret_cast<void *>(&k_stage_ensemble<ST_2, HALVES>);
    case ST_3: return reinterpret_cast<void *>(&k_stage_ensemble<ST_3, HALVES>);
    case ST_3D: return reinterpret_cast<void *>(&k_stage_ensemble<ST_3D, HALVES>);
    default: return reinterpret_cast<void *>(&k_stage_ensemble<ST_RHS, HALVES>);
    }
}

int ensemble_prepare(swe_hip_ctx *c, std::string *err)
{
    for (int stage : {ST_0, ST_1, ST_2, ST_3, ST_RHS, ST_3D}) {
        void *fn = c->units.halves == 2 ? ensemble_kernel<2>(stage) : ensemble_kernel<1>(stage);
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kUnitsMaxLds / 2)
            != hipSuccess) {
            *err = "ensemble kernel: LDS budget";
            return SWE_HIP_EDEVICE;
        }
    }
    return 0;
}

void launch_ensemble_stage(const swe_hip_ctx *c, int stage, const DevStage &st)
{
    const SweUnits &u = c->units;
    DevEnsemble p{};
    p.tile_start = u.d_tile_start;
    p.ustart = u.d_ustart;
    p.ulist = u.d_ulist;
    p.own_row = u.d_own_row;
    p.perm = u.d_perm;
    p.unit_start = u.d_unit_start;
    p.prec = u.d_prec;
    p.wrec = static_cast<const double2 *>(u.d_wrec);
    p.geo = static_cast<const double2 *>(u.d_grec);
    p.ntiles = u.ntiles;
    p.lds_rows = u.rows;
    DevStage s = st;
    double gh0 = c->gh0;
    void *args[] = {&p, &s, &gh0};
    // a launch error stays behind for the caller's check, as after <<< >>>
    (void)hipLaunchKernel(u.halves == 2 ? ensemble_kernel<2>(stage) : ensemble_kernel<1>(stage),
                          dim3((unsigned)(2 * c->ncu + 7) / 8 * 8), dim3(256), args,
                          (size_t)u.lds, c->stream);
}

}  // namespace swe
