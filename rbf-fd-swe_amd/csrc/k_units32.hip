// Whole RK4 steps of one single-state FP32 mesh in one cooperative launch,
// stencil sums on the matrix cores (fast mode, 31-point stencils); the scheme
// of k_units.hip with v_mfma_f32_4x4x1f32: 16 nodes (a unit) per instruction,
// weight i of node b in lane 4 b + i, variable j of its neighbour in lane 4 b +
// j, S[i][j] in element i of lane 4 b + j -- the layout the RHS wants.  One
// slot per instruction, so a sum is a chain of fused multiply-adds in slot
// order: CHAINS == 1 the bits of k_stage_lane32, CHAINS == 2 (even and odd
// slots apart, then added) those of k_stage_split32<2>, whichever AUTO used at
// that size; two chains also halve the distance between dependent products.
// A unit's weights take 32 registers: 4 units per wave stay (UM_GLOBAL spills 6
// to 8 registers with them, UM_STREAM none; 5 spill: 11.4 against 7.55 us at N =
// 163842).
//
// us per RK stage over 100 to 30 steps, against one lane per node resident up
// to 65536 nodes and the stage kernels above:
//   N = 2562     2.35 against 3.04   exchange latency
//   N = 40962    3.13 against 3.25   exchange latency (a unit per wave on 11
//                                    waves; 3.25 with two passes on 8)
//   N = 163842   7.5  against 19.7   9 of 41 units per tile re-read, from L2
//   N = 655362   69   against 110    128 of 160 re-read
#include "units.h"

#include <algorithm>

namespace swe {

struct DevUnits32 : DevUnits {
    const float4 *rec;          // [units][kRec32][64]: 31 slots and ghm, geometry
    float *H;                   // the context's state
    float *X0, *Xa, *Xb;        // exchanged states, kernel order
    float *d;                   // [units][64] D of streamed units (UM_GLOBAL; H is X0's)
    float gh0;
    float c[3];                 // K = H + c F: (float)(dt/2.0), (float)(dt/2.0), dt
    double c6;                  // stage 3: H += (dt/6.0) D in double
    float dcoef[4];             // D += dcoef F (0: D = F, 2, 2, 1)
};

// A unit's record: weight x of slots 4 q .. 4 q + 3 in piece q < 8 (lane 4 b +
// x; slot 31 is free and carries ghm), then lane (b, j)'s geometry: the
// coordinate of variable j and its projection row, for h f and gradghm.
constexpr int kRec32 = 9;
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int P0, int P1, int P2, int P3>
__device__ __forceinline__ float quad_perm32(float v)
{
    return dpp32<P0 | P1 << 2 | P2 << 4 | P3 << 6>(v);
}
template <int K>
__device__ __forceinline__ float quad_bcast32(float v)
{
    return dpp32<K * 0x55>(v);
}

template <int R, int MODE, int CHAINS, bool NT = false>
__global__ __launch_bounds__(MODE == UM_RESIDENT ? 1024 : 512) void k_steps_units32(DevUnits32 p)
{
    constexpr bool STREAM = MODE != UM_RESIDENT;
    extern __shared__ float4 lds32[];
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
    const int j = lane & 3;
    const int own0 = p.own_row[tile];
    const int *ulist = p.ulist + u0;

    // LDS: rows, positions, the resident units' geometry, H and D of streamed
    // units, row ids
    char *rows = reinterpret_cast<char *>(lds32);
    uint4 *pos = reinterpret_cast<uint4 *>(lds32 + p.lds_rows);
    float4 *gl = reinterpret_cast<float4 *>(pos + 64 * p.lds_pos);
    float2 *hd = reinterpret_cast<float2 *>(gl + 64 * p.lds_geo);
    int *ids = reinterpret_cast<int *>(
        hd + (MODE == UM_STREAM && p.lds_pos > R * nw ? 64 * (p.lds_pos - R * nw) : 0));
    if constexpr (MODE != UM_GLOBAL)
        for (int i = tid; i < ucount; i += (int)blockDim.x)
            ids[i] = ulist[i];
    for (int i = tid; i < 64 * (nu < p.lds_pos ? nu : p.lds_pos); i += (int)blockDim.x)
        pos[i] = p.prec[64L * ug + i];
    for (int i = tid; i < 64 * (nu < p.lds_geo ? nu : p.lds_geo); i += (int)blockDim.x)
        gl[i] = p.rec[64L * kRec32 * (ug + (i >> 6)) + 64 * 8 + (i & 63)];

    const int first = t0 + (lane >> 2);   // + 16 u: this lane's node of unit u
    float4 w[R][8];
    float4 gr[STREAM ? 1 : R];
    float H[R], D[R];
    static_for<R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        const int u = wv + r * nw;
        H[r] = D[r] = 0.0f;
        if (u < nu) {
            const float4 *wp = p.rec + 64L * kRec32 * (ug + u) + lane;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                w[r][q] = wp[64 * q];
            if constexpr (!STREAM)
                gr[r] = wp[64 * 8];
            if (16 * u + (lane >> 2) < tcount)
                H[r] = p.H[4L * p.perm[first + 16 * u] + j];
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                w[r][q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    });
    float4 ring[STREAM ? kRec32 : 1];   // the next streamed record
    uint4 pnext[MODE == UM_GLOBAL ? 4 : 1];
    float *const d_mem = p.d + 64L * ug + lane;
    if constexpr (STREAM) {
        for (int u = wv + R * nw; u < nu; u += nw) {
            float h = 0.0f;
            if (16 * u + (lane >> 2) < tcount)
                h = p.H[4L * p.perm[first + 16 * u] + j];
            if constexpr (MODE == UM_STREAM)
                hd[64 * (u - R * nw) + lane] = make_float2(h, 0.0f);
            else if (16 * u + (lane >> 2) < tcount)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, h),
                                                      state_rsrc(p.X0, p.bytes),
                                                      4 * (4 * t0 + 64 * u + lane), 0, kSc1);
        }
        const int u = wv + R * nw;
        if (u < nu) {
            const float4 *wp = p.rec + 64L * kRec32 * (ug + u) + lane;
#pragma unroll
            for (int q = 0; q < kRec32; ++q)
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

    // slots 4 q .. 4 q + 3 of a unit into its sums: operator i of (node,
    // variable) = lane in element i, each chain fused multiply-adds in order
    struct Acc {
        f32x4 c[CHAINS];
    };
    auto quarter = [&](Acc acc, int q, float4 w4, unsigned p0, unsigned p1) {
        const float wq[4] = {w4.x, w4.y, w4.z, w4.w};
        const unsigned r[4] = {p0 & 0xffffu, p0 >> 16, p1 & 0xffffu, p1 >> 16};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < 31) {
                const float b = *reinterpret_cast<const float *>(rows + (r[i] << 4 | 4u * j));
                f32x4 &a = acc.c[i % CHAINS];
                a = __builtin_amdgcn_mfma_f32_4x4x1f32(wq[i], b, a, 0, 0, 0);
            }
        return acc;
    };
    // RHS of this lane's (node, variable), operation order of rhs_point32
    auto rhs = [&](int u, const Acc &acc, float4 g, float ghm) {
        f32x4 x = acc.c[0];
        if constexpr (CHAINS == 2)
            x += acc.c[1];
        const float4 o = lds32[own0 + 16 * u + (lane >> 2)];
        const bool k3 = j == 3;
        const float s1 = j == 0 ? o.z : (j == 1 ? o.x : o.y);
        const float s2 = j == 0 ? o.y : (j == 1 ? o.z : o.x);
        const float c1 = quad_perm32<1, 2, 0, 3>(g.x), c2 = quad_perm32<2, 0, 1, 3>(g.x);
        const float f = quad_bcast32<3>(g.x);
        const float dh0 = quad_bcast32<3>(x[0]), dh1 = quad_bcast32<3>(x[1]),
                    dh2 = quad_bcast32<3>(x[2]);
        const float dh = j == 0 ? dh0 : (j == 1 ? dh1 : dh2);
        const float div = (quad_bcast32<0>(x[0]) + quad_bcast32<1>(x[1])) + quad_bcast32<2>(x[2]);
        const float a0 = k3 ? x[0] - g.y : x[0];
        const float a1 = k3 ? x[1] - g.z : x[1];
        const float a2 = k3 ? x[2] - g.w : x[2];
        const float t = ((o.x * a0) + (o.y * a1)) + (o.z * a2);
        const float cor = f * ((c1 * s1) - (c2 * s2));
        const float hx = (o.w + p.gh0 - ghm) * div;
        const float t1 = t + (k3 ? hx : cor);
        const float t2 = t1 + dh;
        const float r = -(k3 ? t1 : t2);
        const float ru = quad_bcast32<0>(r), rv = quad_bcast32<1>(r), rw = quad_bcast32<2>(r);
        const float pr = ((g.y * ru) + (g.z * rv)) + (g.w * rw);
        return (k3 ? r : pr) + x[3];
    };

    for (int step = 0; step < p.nsteps && alive; ++step) {
        static_for<4>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (!alive)
                return;
            const float *src = s == 0 ? p.X0 : (s == 2 ? p.Xb : p.Xa);
            float *out = s == 0 ? p.Xa : (s == 1 ? p.Xb : (s == 2 ? p.Xa : p.X0));
            if (!(alive = res_wait(p.y, tile, stage)))   // also: ids written, rows free
                return;
            // 64 rows per wave and instruction; the first stage gathers the
            // state buffer itself
            const bool head = s == 0 && step == 0;
            const float *b = head ? p.H : src;
            for (int i0 = 64 * wv; i0 < ucount; i0 += 64 * nw) {
                const int i = i0 + lane;
                if (i < ucount) {
                    int id = MODE == UM_GLOBAL ? ulist[i] : ids[i];
                    if (head)
                        id = p.perm[id];
                    dma16_sc1(b + 4L * id, rows + 16L * i0);
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            const bool last = s == 3 && step == p.nsteps - 1;
            auto update = [&](int u, float F, float &Hv, float &Dv) {
                float K;
                if constexpr (s == 0) {
                    Dv = F;
                    K = axpy32<false>(Hv, p.c[0], F);
                } else if constexpr (s == 1 || s == 2) {
                    Dv = axpy32<false>(Dv, p.dcoef[s], F);
                    K = axpy32<false>(Hv, p.c[s], F);
                } else {
                    const float d = axpy32<false>(Dv, p.dcoef[3], F);
                    K = Hv = update_h32<false>(Hv, p.c6, d);
                }
                if (16 * u + (lane >> 2) < tcount) {
                    const int e = last ? 4 * p.perm[first + 16 * u] + j
                                       : 4 * t0 + 64 * u + lane;
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __builtin_bit_cast(unsigned, K), state_rsrc(last ? p.H : out, p.bytes),
                        4 * e, 0, kSc1);
                }
            };
            static_for<R>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                const int u = wv + r * nw;
                if (u < nu) {
                    Acc acc = {};
                    const uint4 *pu = pos + 64 * u + (lane >> 2);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint4 pv = pu[16 * q];
                        acc = quarter(acc, 2 * q, w[r][2 * q], pv.x, pv.y);
                        acc = quarter(acc, 2 * q + 1, w[r][2 * q + 1], pv.z, pv.w);
                    }
                    float4 g;
                    if constexpr (STREAM)
                        g = gl[64 * u + lane];
                    else
                        g = gr[r];
                    update(u, rhs(u, acc, g, w[r][7].w), H[r], D[r]);
                }
            });
            if constexpr (STREAM) {
#pragma unroll 1
                for (int u = wv + R * nw; u < nu; u += nw) {
                    const int un = u + nw < nu ? u + nw : wv + R * nw;   // next, wrapping
                    const float4 *wn = p.rec + 64L * kRec32 * (ug + un) + lane;
                    uint4 pv[4];
                    float2 hv;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if constexpr (MODE == UM_STREAM) {
                            pv[q] = pos[64 * u + 16 * q + (lane >> 2)];
                        } else {
                            pv[q] = pnext[q];
                            pnext[q] = p.prec[64L * (ug + un) + 16 * q + (lane >> 2)];
                        }
                    }
                    if constexpr (MODE == UM_GLOBAL) {
                        // stage 0 gathers H: it is in the own row
                        if constexpr (s == 0) {
                            hv.x = *reinterpret_cast<const float *>(
                                rows + 16 * (own0 + 16 * u + (lane >> 2)) + 4 * j);
                        } else {
                            hv.x = __builtin_bit_cast(
                                float, __builtin_amdgcn_raw_buffer_load_b32(
                                           state_rsrc(p.X0, p.bytes),
                                           4 * (4 * t0 + 64 * u + lane), 0, kSc1));
                            hv.y = d_mem[64L * u];
                        }
                    }
                    Acc acc = {};
                    const float4 g = ring[8];
                    const float ghm = ring[7].w;
                    ring[8] = NT ? load_nt(wn + 64 * 8) : wn[64 * 8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        const uint4 v = pv[q >> 1];
                        acc = (q & 1) ? quarter(acc, q, ring[q], v.z, v.w)
                                      : quarter(acc, q, ring[q], v.x, v.y);
                        ring[q] = NT ? load_nt(wn + 64 * q) : wn[64 * q];
                    }
                    if constexpr (MODE == UM_STREAM)
                        hv = hd[64 * (u - R * nw) + lane];
                    update(u, rhs(u, acc, g, ghm), hv.x, hv.y);
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

// Packs the unit records: one workgroup per unit, thread = (piece, lane).
__global__ void k_pack_units32(DevMesh32 m, const int *tile_start, const int *unit_start,
                               const int *unit_tile, const int *perm, float4 *rec)
{
    const int unit = (int)blockIdx.x;
    const int tile = unit_tile[unit];
    const int lane = (int)threadIdx.x & 63, q = (int)threadIdx.x >> 6;
    const int node = tile_start[tile] + 16 * (unit - unit_start[tile]) + (lane >> 2);
    const int x = lane & 3;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (node < tile_start[tile + 1]) {
        const int dn = perm[node];
        const int field[4][4] = {{G_X, G_PU, G_PU + 1, G_PU + 2},
                                 {G_Y, G_PV, G_PV + 1, G_PV + 2},
                                 {G_Z, G_PW, G_PW + 1, G_PW + 2},
                                 {G_F, G_GG, G_GG + 1, G_GG + 2}};
        const long ld = m.sblk ? 16L : (long)m.ld;
        const long sb = m.sblk ? ((long)(dn >> 4) * m.nnbr << 4) + (dn & 15) : (long)dn;
        for (int c = 0; c < 4; ++c) {
            const int slot = 4 * q + c;
            if (q == 8)
                v[c] = m.geo[(long)field[x][c] * m.ld + dn];
            else if (slot == 31)
                v[c] = m.geo[(long)G_GHM * m.ld + dn];
            else
                v[c] = m.wts[4L * (sb + (long)slot * ld) + x];
        }
    }
    rec[64L * kRec32 * unit + 64 * q + lane] = make_float4(v[0], v[1], v[2], v[3]);
}

constexpr int kUnits32Kept = 4;   // resident units per wave of the streaming modes

bool units_plan32(SweUnits &u)
{
    // up to 16 units one per wave (74 registers), else kUnits32Kept on 8 waves
    const int kept = kUnits32Kept * 8;
    long lds = 16L * u.rows;
    u.waves = u.units <= 16 ? std::max(4, u.units) : 8;
    if (u.units <= u.waves) {
        u.mode = UM_RESIDENT;
        u.pos = u.units;
        lds += 1024L * u.pos + 4L * u.rows;
    } else {
        const long whole = 1024L * u.units + 1024L * std::min(u.units, kept)
                           + 512L * std::max(0, u.units - kept) + 4L * u.rows;
        if (lds + whole <= kUnitsMaxLds) {
            u.mode = UM_STREAM;
            u.pos = u.units;
            u.geo = std::min(u.units, kept);
            lds += whole;
        } else {
            u.mode = UM_GLOBAL;
            // past the 256 MB last-level cache the records are better not kept
            // there at all (N = 605162: 62.2 against 65.7 us per stage, 655362
            // 69 against 77); while they fit they are (576002: 55.5 against
            // 58.9, 349692 27.8 against 34.2)
            u.stream_nt = 1024L * kRec32 * (u.units - kept) * u.ntiles > (256L << 20);
            u.pos = u.geo = kept;
            lds += 2048L * kept;
        }
    }
    u.lds = (int)lds;
    return lds <= kUnitsMaxLds;
}

template <int CHAINS>
static void *streaming32(const SweUnits &u)
{
    // two chains end at 262144 nodes (151 MB of records), before stream_nt
    if constexpr (CHAINS == 1)
        if (u.mode == UM_GLOBAL && u.stream_nt)
            return reinterpret_cast<void *>(&k_steps_units32<kUnits32Kept, UM_GLOBAL, 1, true>);
    return u.mode == UM_STREAM
               ? reinterpret_cast<void *>(&k_steps_units32<kUnits32Kept, UM_STREAM, CHAINS>)
               : reinterpret_cast<void *>(&k_steps_units32<kUnits32Kept, UM_GLOBAL, CHAINS>);
}

void *units_kernel32(const SweUnits &u)
{
    if (u.mode != UM_RESIDENT)
        return u.chains == 2 ? streaming32<2>(u) : streaming32<1>(u);
    return reinterpret_cast<void *>(&k_steps_units32<1, UM_RESIDENT, 1>);
}

int units_pack32(swe_hip_ctx *c, int units)
{
    SweUnits &u = c->units;
    const size_t rb = sizeof(float4) * 64 * kRec32 * (size_t)units;
    if (hipMalloc(&u.d_wrec, rb) != hipSuccess)
        return SWE_HIP_ENOMEM;
    c->bytes += (long long)rb;
    u.bytes += (long long)rb;
    k_pack_units32<<<units, 64 * kRec32, 0, c->stream>>>(mesh32_of(c), u.d_tile_start,
                                                         u.d_unit_start, u.d_unit_tile, u.d_perm,
                                                         static_cast<float4 *>(u.d_wrec));
    return hipGetLastError() == hipSuccess && hipStreamSynchronize(c->stream) == hipSuccess
               ? 0 : SWE_HIP_EDEVICE;
}

hipError_t units_launch32(swe_hip_ctx *c, int nsteps, const DevResSync &y)
{
    const SweUnits &u = c->units;
    DevUnits32 p{};
    units_tables(c, nsteps, y, &p);
    p.rec = static_cast<const float4 *>(u.d_wrec);
    p.d = static_cast<float *>(u.d_hd);
    p.H = c->f_H;
    p.X0 = c->f_D;   // D lives in the kernel
    p.Xa = c->f_Ka;
    p.Xb = c->f_Kb;
    p.gh0 = (float)c->gh0;
    // the constants of the FP32 stage kernels (rk4_rbffd_swe.c:123-186)
    const float dt = (float)c->dt;
    p.c[0] = (float)(dt / 2.0); p.c[1] = (float)(dt / 2.0); p.c[2] = dt;
    p.c6 = dt / 6.0;
    p.dcoef[0] = 0.0f; p.dcoef[1] = 2.0f; p.dcoef[2] = 2.0f; p.dcoef[3] = 1.0f;
    void *args[] = {&p};
    return hipLaunchCooperativeKernel(units_kernel32(u), dim3(u.ntiles), dim3(64 * u.waves), args,
                                      (unsigned)u.lds, c->stream);
}

}  // namespace swe
