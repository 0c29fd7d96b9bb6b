// Whole RK4 steps of one small single-state FP64 mesh in one cooperative
// launch, exact mode (31-point stencils, at most 64 nodes per compute unit).
//
// Exact sums round every product and every addition, in slot order, so the
// matrix cores cannot take them; what a stage waits for is the chain of 31
// multiplies and adds.  Here each of a node's 16 sums has a lane of its own:
// lane 16 i + 4 b + x of a wave adds operator i of variable x for node b of a
// group of 4 nodes, weights in 31 register pairs, one 8-byte LDS read per slot
// shared by the four operators -- 2 FP64 instructions per slot, where two lanes
// per node (k_steps_resident) issue 16 and exchange weights by DPP.  A wave
// takes one group, at most 16 waves a tile (126 registers); row swaps give
// lane (node, variable) its four sums, and the RHS and the exchange are those
// of k_units.hip, in exact arithmetic.
//
// us per RK stage over 100 steps against k_steps_resident: N = 642 2.50 against
// 3.76, 2562 2.50 against 3.93, 10242 3.18 against 4.06, 16002 3.58 against
// 4.16; what is left is the exchange (2.4 us with almost no arithmetic).
#include "units.h"

#include <algorithm>

namespace swe {

struct DevUnitsExact : DevUnits {
    DevMesh m;
    double *H;                  // the context's state
    double *X0, *Xa, *Xb;       // exchanged states, kernel order
    double c[4];                // K = H + c F (dt/2, dt/2, dt); stage 3: H += c D (dt/6)
    double dcoef[4];            // D += dcoef F (0: D = F, 2, 2, 1)
};

__global__ __launch_bounds__(1024) void k_steps_exact(DevUnitsExact p)
{
    extern __shared__ double2 lds[];
    const int tile = (int)blockIdx.x;
    const int t0 = p.tile_start[tile];
    const int tcount = p.tile_start[tile + 1] - t0;
    const int ug = p.unit_start[tile];
    const int nu = p.unit_start[tile + 1] - ug;
    const int u0 = p.ustart[tile];
    const int ucount = p.ustart[tile + 1] - u0;
    const int tid = (int)threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = (int)blockDim.x >> 6;
    const int own0 = p.own_row[tile];

    // LDS: rows, positions [unit][slot / 8][node], row ids
    char *rows = reinterpret_cast<char *>(lds);
    uint4 *pos = reinterpret_cast<uint4 *>(lds + 2 * p.lds_rows);
    int *ids = reinterpret_cast<int *>(pos + 64 * p.lds_pos);
    for (int i = tid; i < ucount; i += (int)blockDim.x)
        ids[i] = p.ulist[u0 + i];
    for (int i = tid; i < 64 * nu; i += (int)blockDim.x)
        pos[i] = p.prec[64L * ug + i];

    // sums: operator i, node b of group wv, variable x
    const int i = lane >> 4, b = (lane >> 2) & 3, x = lane & 3;
    const int nl = 4 * wv + b;
    const int nc = nl < tcount ? nl : 0;
    const int dn = p.perm[t0 + nc];
    const bool live = i == 0 && nl < tcount;   // after the transpose
    double w[31];
    {
        const double *wp = p.m.wts + 4L * slot_base<31>(p.m, dn) + i;
        const long ld = slot_stride(p.m);
#pragma unroll
        for (int s = 0; s < 31; ++s)
            w[s] = wp[4L * s * ld];
    }
    const bool k3 = x == 3;
    const double *geo = p.m.geo + dn;
    const long gld = p.m.ld;
    const int pf = k3 ? G_GG : G_PU + 3 * x;
    const double gc = geo[(k3 ? G_F : G_X + x) * gld];
    const double g0 = geo[pf * gld], g1 = geo[(pf + 1) * gld], g2 = geo[(pf + 2) * gld];
    const double ghm = geo[G_GHM * gld];
    const double c1 = quad_perm<1, 2, 0, 3>(gc), c2 = quad_perm<2, 0, 1, 3>(gc);
    const double f = quad_bcast<3>(gc);
    double H = p.H[4L * dn + x], D = 0.0;
    unsigned stage = p.y.stage0;
    bool alive = true;

    for (int step = 0; step < p.nsteps && alive; ++step) {
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (!alive)
                return;
            const double *src = s == 0 ? p.X0 : (s == 2 ? p.Xb : p.Xa);
            double *out = s == 0 ? p.Xa : (s == 1 ? p.Xb : (s == 2 ? p.Xa : p.X0));
            if (!(alive = res_wait(p.y, tile, stage)))   // also: ids written, rows free
                return;
            const bool head = s == 0 && step == 0;
            const double *from = (head ? p.H : src) + 2 * (lane & 1);
            for (int i0 = 32 * wv; i0 < ucount; i0 += 32 * nw) {
                const int k = i0 + (lane >> 1);
                if (k < ucount) {
                    int id = ids[k];
                    if (head)
                        id = p.perm[id];
                    dma16_sc1(from + 4L * id, rows + 32L * i0);
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            double x0 = 0.0;
            // a short last tile has no units, and pos no entries, for the waves
            // past its nodes
            if (4 * wv < tcount) {
                const uint4 *pu = pos + 64 * (wv >> 2) + 4 * (wv & 3) + b;
                unsigned pw[16];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint4 v = pu[16 * q];
                    pw[4 * q] = v.x; pw[4 * q + 1] = v.y;
                    pw[4 * q + 2] = v.z; pw[4 * q + 3] = v.w;
                }
#pragma unroll
                for (int j = 0; j < 31; ++j) {
                    const unsigned row = (j & 1) ? (pw[j >> 1] >> 16) : (pw[j >> 1] & 0xffffu);
                    const double sv =
                        *reinterpret_cast<const double *>(rows + (row << 5 | 8u * x));
                    x0 = madd<true>(x0, w[j], sv);
                }
            }
            // the four operators of lane (b, x) into lanes 0 .. 15
            double x1 = 0.0, x2 = 0.0, x3 = 0.0;
            swap_rows32(x0, x2);
            swap_rows32(x1, x3);
            swap_rows16(x0, x1);
            swap_rows16(x2, x3);
            const double2 *own = lds + 2 * (own0 + nc);
            const double2 uv = own[0], wh = own[1];
            const double s1 = x == 0 ? wh.x : (x == 1 ? uv.x : uv.y);
            const double s2 = x == 0 ? uv.y : (x == 1 ? wh.x : uv.x);
            const double dh0 = quad_bcast<3>(x0), dh1 = quad_bcast<3>(x1), dh2 = quad_bcast<3>(x2);
            const double dh = x == 0 ? dh0 : (x == 1 ? dh1 : dh2);
            const double div = (quad_bcast<0>(x0) + quad_bcast<1>(x1)) + quad_bcast<2>(x2);
            const double a0 = k3 ? x0 - g0 : x0;
            const double a1 = k3 ? x1 - g1 : x1;
            const double a2 = k3 ? x2 - g2 : x2;
            const double t = ((uv.x * a0) + (uv.y * a1)) + (wh.x * a2);
            const double cor = f * ((c1 * s1) - (c2 * s2));
            const double hx = (wh.y + p.m.gh0 - ghm) * div;
            const double t1 = t + (k3 ? hx : cor);
            const double t2 = t1 + dh;
            const double rr = -(k3 ? t1 : t2);
            const double ru = quad_bcast<0>(rr), rv = quad_bcast<1>(rr), rw = quad_bcast<2>(rr);
            const double pr = ((g0 * ru) + (g1 * rv)) + (g2 * rw);
            const double F = (k3 ? rr : pr) + x3;
            double K;
            if constexpr (s == 0) {
                D = F;
                K = axpy<true>(H, p.c[0], F);
            } else if constexpr (s == 1 || s == 2) {
                D = axpy<true>(D, p.dcoef[s], F);
                K = axpy<true>(H, p.c[s], F);
            } else {
                const double d = axpy<true>(D, p.dcoef[3], F);
                K = H = axpy<true>(H, p.c[3], d);
            }
            if (live) {
                const bool last = s == 3 && step == p.nsteps - 1;
                const int e = 4 * (last ? dn : t0 + nl) + x;
                __builtin_amdgcn_raw_buffer_store_b64(
                    __builtin_bit_cast(u32x2, K), state_rsrc(last ? p.H : out, p.bytes), 8 * e, 0,
                    kSc1);
            }
            res_publish(p.y, tile, ++stage);
        });
    }
}

bool units_plan_exact(SweUnits &u)
{
    u.mode = UM_RESIDENT;
    u.pos = u.units;
    u.lds = 32 * u.rows + 1024 * u.pos + 4 * u.rows;
    return u.lds <= kUnitsMaxLds && u.units <= 4;   // 64 nodes: 16 waves
}

void *units_kernel_exact() { return reinterpret_cast<void *>(&k_steps_exact); }

hipError_t units_launch_exact(swe_hip_ctx *c, int nsteps, const DevResSync &y)
{
    const SweUnits &u = c->units;
    DevUnitsExact p{};
    units_tables(c, nsteps, y, &p);
    p.m = mesh_of(c);
    p.H = c->d_H;
    p.X0 = c->d_D;   // D lives in the kernel
    p.Xa = c->d_Ka;
    p.Xb = c->d_Kb;
    const double dt = c->dt;
    p.c[0] = dt / 2.0; p.c[1] = dt / 2.0; p.c[2] = dt; p.c[3] = dt / 6.0;
    p.dcoef[0] = 0.0; p.dcoef[1] = 2.0; p.dcoef[2] = 2.0; p.dcoef[3] = 1.0;
    void *args[] = {&p};
    return hipLaunchCooperativeKernel(units_kernel_exact(), dim3(u.ntiles), dim3(64 * u.waves),
                                      args, (unsigned)u.lds, c->stream);
}

}  // namespace swe
