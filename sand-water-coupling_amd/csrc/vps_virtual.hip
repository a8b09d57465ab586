// vps_virtual.hip -- virtual particle generation and the fused virtual sums.
//
// Replaces VirtualParticle::generateParticles / computeDensities /
// computeVolumes / calculateVelocity / calculateDiv
// (Cores/Structures/VirtualParticle.cpp:18-62, 136-147, 171-201).
//
// The reference evaluates the weight w_I = sum_j W_h(x_I - x_j) at every node
// of the lattice (6.9M nodes at 1M particles) and keeps the nodes with
// w_I > 1e-6, in x-fastest node order.  Here:
//   1. every real particle flags the 8^D-node bricks its h-ball touches;
//   2. flagged bricks are compacted into slots (ordered by brick id);
//   3. one workgroup per slot evaluates, per node, in ONE walk over the real
//      and boundary neighbours within h: w_I (FP32, with an exact FP64 redo
//      when it lies within 1e-4 relative of the 1e-6 threshold), rho_I,
//      V_I, the smoothed velocity v_I and the divergence D_I (the CG
//      right-hand side).  Folding calculateVelocity/calculateDiv into
//      generation saves a full neighbour walk; project then uses the
//      velocities as of generation, which is also when the reference reads
//      them (nothing changes velocities between generateParticles and
//      project, DualParticleSphLiquid.cpp:118-125);
//   4. the reference order (x-fastest node rank) comes from a lattice bitmask
//      and a popcount scan, so every node knows its index in the reference's
//      virtual list without the list ever being materialised.
#include <algorithm>
#include <cmath>

#include "vps_scan.h"

namespace vps {
namespace {

inline unsigned blocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Marks the bricks within h of each particle and clears the lattice bitmask
// of the previous generation (grid-stride over its words).
template <int D>
__global__ void __launch_bounds__(256) k_mark_bricks(const double4* pos,
                                                     int64_t n, KConst k,
                                                     uint32_t* flag, uint32_t* bits,
                                                     int64_t nwords, int32_t* unit_count) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t w = i; w < nwords; w += (int64_t)gridDim.x * 256) bits[w] = 0u;
    if (i == 0) unit_count[0] = 0;   // the gradient's unit list is rebuilt next
    if (i >= n) return;
    const double4 p = pos[i];
    const double pc[3] = {p.x, p.y, p.z};
    int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
#pragma unroll
    for (int a = 0; a < D; a++) {
        const double inv = 1.0 / k.spacing;
        int l = (int)floor((pc[a] - k.h - k.origin[a]) * inv);
        int u = (int)floor((pc[a] + k.h - k.origin[a]) * inv) + 1;
        l = l < 0 ? 0 : l;
        u = u >= k.ndims[a] ? k.ndims[a] - 1 : u;
        if (l > u) return;  // ball outside the lattice
        lo[a] = l / kBrick;
        hi[a] = u / kBrick;
    }
    for (int bz = lo[2]; bz <= hi[2]; bz++)
        for (int by = lo[1]; by <= hi[1]; by++)
            for (int bx = lo[0]; bx <= hi[0]; bx++)
                flag[((int64_t)bz * k.bdims[1] + by) * k.bdims[0] + bx] = 1u;
}

// Brick compaction: the scan of the flags gives every flagged brick its slot
// (ordered by brick id); the flags are cleared for the next generation.
struct LoadFlag {
    static constexpr bool kWide = false;
    const uint32_t* flag;
    __device__ __forceinline__ int operator()(int64_t b) const { return (int)flag[b]; }
};
struct AssignSlot {
    static constexpr bool kWide = false;
    uint32_t* flag;
    int32_t *slot_of_brick, *brick_of_slot;
    __device__ __forceinline__ void operator()(int64_t b, int flagged, int slot) const {
        slot_of_brick[b] = flagged ? slot : -1;
        if (flagged) {
            brick_of_slot[slot] = (int32_t)b;
            flag[b] = 0u;
        }
    }
};

// Real-neighbour sums of one node: w, sum W_H, sum V^2 W, sum V W (the v
// denominator), sum v W / rho and the divergence terms.  dx = q - x_j.
// Every sum is linear in its spline's constant (c0 of W, c1 of S = -W'/r),
// so the terms are summed without it and finish_node applies c0h, c0H and
// c1h once per node (one multiply fewer per term); the boundary sums alike.
struct RealAcc {
    float w = 0.f, sH = 0.f, sV = 0.f, den = 0.f;
    float nvx = 0.f, nvy = 0.f, nvz = 0.f;   // sum v_j W / rho_j
    float gx = 0.f, gy = 0.f, gz = 0.f;      // sum V_j gradK
    float dr = 0.f;                           // sum V_j v_j . gradK
    // the sums of this lane and of the one `o` away (lanes that share a node)
    __device__ __forceinline__ void add_lanes(int o) {
        for (float* f : {&w, &sH, &sV, &den, &nvx, &nvy, &nvz, &gx, &gy, &gz, &dr})
            *f += __shfl_xor(*f, o, 64);
    }
    template <int D>
    __device__ __forceinline__ void add(const KConst& k, double d2, float dx,
                                        float dy, float dz, float4 vj,
                                        float inv_rhoj) {
        const KW kh = kernel_f32(d2, k.h2, k.hf, k.inv_h, 1.f, 1.f);
        const KW kH = kernel_f32(d2, k.H2, k.Hf, k.inv_H, 1.f, 1.f);
        const float Vj = vj.w;
        const float wr = kh.w * inv_rhoj;
        w += kh.w;
        sH += kH.w;
        sV += Vj * Vj * kh.w;
        den += Vj * kh.w;
        nvx += vj.x * wr;
        nvy += vj.y * wr;
        nvz += vj.z * wr;
        if (kh.r > 0.f) {
            // gradK(q - x_j) = -W'(r) (q - x_j) / r
            const float s = -kh.dw / kh.r;
            const float ex = dx * s, ey = dy * s, ez = D == 3 ? dz * s : 0.f;
            gx += Vj * ex;
            gy += Vj * ey;
            gz += Vj * ez;
            dr += Vj * (vj.x * ex + vj.y * ey + vj.z * ez);
        }
    }
    // The same sums from an FP32 squared distance d2f < h^2 (0 < d2f), with
    // the division-free spline.
    template <int D>
    __device__ __forceinline__ void add_fast(const KConst& k, float d2f, float dx,
                                             float dy, float dz, float4 vj,
                                             float inv_rhoj) {
        const float rinv = __builtin_amdgcn_rsqf(d2f);
        const float r = d2f * rinv;
        const SplineAB sp = spline_ab(r, k.inv_h);
        const float wh = spline_w_ab(sp, 1.f);
        const float sh = spline_s_ab(sp, rinv, 1.f);
        const float Vj = vj.w;
        const float wr = wh * inv_rhoj;
        w += wh;
        sH += spline_w_ab(spline_ab(r, k.inv_H), 1.f);
        const float vw = Vj * wh;
        sV += Vj * vw;
        den += vw;
        nvx += vj.x * wr;
        nvy += vj.y * wr;
        nvz += vj.z * wr;
        const float vs = Vj * sh;
        gx += dx * vs;
        gy += dy * vs;
        gz += D == 3 ? dz * vs : 0.f;
        dr += vs * (vj.x * dx + vj.y * dy + (D == 3 ? vj.z * dz : 0.f));
    }
};

// Boundary sums of one node: sum V_b W, sum v_b W / rho_b, sum V_b gradK,
// sum V_b v_b . gradK (VirtualParticle.cpp:76-107).
struct BAcc {
    float den = 0.f, bnx = 0.f, bny = 0.f, bnz = 0.f;
    float hx = 0.f, hy = 0.f, hz = 0.f, db = 0.f;
    __device__ __forceinline__ void add_lanes(int o) {
        for (float* f : {&den, &bnx, &bny, &bnz, &hx, &hy, &hz, &db}) *f += __shfl_xor(*f, o, 64);
    }
    // boundary particle at pj within h (FP64 test passed): accurate spline
    template <int D>
    __device__ __forceinline__ void add_exact(const KConst& k, double qx, double qy,
                                              double qz, const double4& pj, double d2,
                                              const float4& vj, float rho_b) {
        const KW kh = kernel_f32(d2, k.h2, k.hf, k.inv_h, 1.f, 1.f);
        const float Vj = vj.w;
        const float wr = kh.w / rho_b;
        den += Vj * kh.w;
        bnx += vj.x * wr;
        bny += vj.y * wr;
        bnz += vj.z * wr;
        if (kh.r > 0.f) {
            const float s = -kh.dw / kh.r;
            const float ex = (float)(qx - pj.x) * s;
            const float ey = (float)(qy - pj.y) * s;
            const float ez = D == 3 ? (float)(qz - pj.z) * s : 0.f;
            hx += Vj * ex;
            hy += Vj * ey;
            hz += Vj * ez;
            db += Vj * (vj.x * ex + vj.y * ey + vj.z * ez);
        }
    }
    // the same from an FP32 squared distance 0 < d2f < h^2 and d = q - x_b,
    // division-free (as the real sums)
    __device__ __forceinline__ void add_fast(const KConst& k, float d2f, float dx, float dy,
                                             float dz, const float4& vj, float inv_rho_b) {
        const float rinv = __builtin_amdgcn_rsqf(d2f);
        const SplineAB sp = spline_ab(d2f * rinv, k.inv_h);
        const float wh = spline_w_ab(sp, 1.f);
        const float sh = spline_s_ab(sp, rinv, 1.f);
        const float Vj = vj.w;
        const float wr = wh * inv_rho_b;
        den += Vj * wh;
        bnx += vj.x * wr;
        bny += vj.y * wr;
        bnz += vj.z * wr;
        const float ex = dx * sh, ey = dy * sh, ez = dz * sh;
        hx += Vj * ex;
        hy += Vj * ey;
        hz += Vj * ez;
        db += Vj * (vj.x * ex + vj.y * ey + vj.z * ez);
    }
};

// Boundary walk of one node from the global cell table (FP64 throughout).
struct BoundaryWalkGlobal3 {
    const int32_t* bcstart;
    const double4* bpos;
    __device__ __forceinline__ void operator()(const KConst& k, double qx, double qy,
                                               double qz, const float4* bvel,
                                               const float4* bnrm, BAcc& b) const {
        for_each_candidate<3>(k, bcstart, bpos, qx, qy, qz, [&](int j, const double4& pj) {
            const double d2 = sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz);
            if (d2 < k.h2) b.add_exact<3>(k, qx, qy, qz, pj, d2, bvel[j], bnrm[j].w);
        });
    }
};

// Everything after the real walk: the exact threshold decision, the boundary
// walk, v_I, D_I and the outputs.
// S lanes share a node: the real sums are the node's, the boundary walk is one
// lane's part, and lane 0 writes.
template <int D, int S = 1, typename BW>
__device__ __forceinline__ void finish_node(
    const KConst& k, const RealAcc& a, double qx, double qy, double qz,
    int cx, int cy, int cz, int64_t out, const double4* rpos,
    const int32_t* rcstart, const BW& bwalk, const float4* bvel,
    const float4* bnrm, float* vrho, float* vvol, float* vb, uint32_t* bits) {
    // the sums carry no spline constants (see RealAcc)
    const float aw = a.w * k.c0h;
    bool virt = aw > 1e-6f;
    if (fabsf(aw - 1e-6f) <= 1e-10f) {
        // exact FP64 decision near the threshold (VirtualParticle.cpp:56)
        double w64 = 0;
        for_each_candidate<D>(k, rcstart, rpos, qx, qy, qz, [&](int j, const double4& pj) {
            const double d2 = D == 3 ? sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz)
                                     : sq_dist2(pj.x, pj.y, qx, qy);
            if (d2 < k.h2) w64 += kernel_w64(d2, k.inv_h64, k.c0h64);
        });
        virt = w64 > 1e-6;
    }
    const bool writes = S == 1 || threadIdx.x % S == 0;
    if (!virt) {
        if (writes) vrho[out] = vvol[out] = vb[out] = 0.f;
        return;
    }
    // boundary neighbours within h
    BAcc b;
    if (writes) b.den = a.den;
    bwalk(k, qx, qy, qz, bvel, bnrm, b);
    if constexpr (S > 1) {
#pragma unroll
        for (int o = 1; o < S; o <<= 1) b.add_lanes(o);
    }
    if (!writes) return;
    // v_I = (m sum v_j W/rho_j + m_b sum v_b W/rho_b) / (sum V W + sum V_b W + 1e-6)
    const float inv_den = 1.f / fmaf(b.den, k.c0h, 1e-6f);
    const float mc = k.mass * k.c0h;
    const float ux = (mc * a.nvx + mc * b.bnx) * inv_den;
    const float uy = (mc * a.nvy + mc * b.bny) * inv_den;
    const float uz = (mc * a.nvz + mc * b.bnz) * inv_den;
    const float rho = k.mass * k.c0H * a.sH;
    const float drho = rho - k.rho0;
    const float D_I = k.c1h * (a.dr - (ux * a.gx + uy * a.gy + uz * a.gz) + b.db -
                               (ux * b.hx + uy * b.hy + uz * b.hz)) -
                      k.kappa * (drho > 0.f ? drho : 0.f) / k.rho0;
    vrho[out] = rho;
    vvol[out] = a.sV * k.c0h;
    vb[out] = D_I;
    const int64_t lin = ((int64_t)cz * k.ndims[1] + cy) * k.ndims[0] + cx;
    atomicOr(&bits[lin >> 5], 1u << (lin & 31));
}

// The real walk straight from global memory (bricks whose neighbourhood does
// not fit the LDS stage).
__device__ __forceinline__ void real_walk_global3(const KConst& k,
                                                 const int32_t* rcstart,
                                                 const double4* rpos,
                                                 const float4* rvel,
                                                 const float* rrho, double qx,
                                                 double qy, double qz,
                                                 RealAcc& a) {
    for_each_candidate<3>(k, rcstart, rpos, qx, qy, qz, [&](int j, const double4& pj) {
        const double d2 = sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz);
        if (d2 < k.h2)
            a.add<3>(k, d2, (float)(qx - pj.x), (float)(qy - pj.y), (float)(qz - pj.z), rvel[j],
                     1.f / rrho[j]);
    });
}

// Fused per-node pass in 2D.  One workgroup = one brick, S lanes per node (see
// walk_lanes2), straight from global memory: 36 candidates a node.
template <int S>
__global__ void __launch_bounds__(64 * S) k_virtual_sums2(
    KConst k, const int32_t* brick_of_slot, const int32_t* nslots_p,
    const double4* rpos, const float4* rvel, const float* rrho,
    const int32_t* rcstart, const double4* bpos, const float4* bvel,
    const float4* bnrm, const int32_t* bcstart, float* vrho, float* vvol,
    float* vb, uint32_t* bits) {
    const int nslots = *nslots_p;   // the grid may exceed the slot count
    if ((int)blockIdx.x >= nslots) return;
    const int slot = xcd_remap(blockIdx.x, nslots);
    const int brick = brick_of_slot[slot];
    const int node = threadIdx.x / S, sub = S > 1 ? threadIdx.x % S : 0;
    const int cx = brick % k.bdims[0] * kBrick + (node & 7),
              cy = brick / k.bdims[0] * kBrick + (node >> 3);
    const int64_t out = (int64_t)slot * 64 + node;
    if (cx >= k.ndims[0] || cy >= k.ndims[1]) {
        if (sub == 0) vrho[out] = vvol[out] = vb[out] = 0.f;
        return;   // uniform over the lanes of a node
    }
    const double qx = node_coord(k.origin[0], cx, k.spacing);
    const double qy = node_coord(k.origin[1], cy, k.spacing);
    RealAcc a;
    for_each_candidate2<S>(k, rcstart, rpos, qx, qy, sub, [&](int j, double px, double py) {
        const double d2 = sq_dist2(px, py, qx, qy);
        if (d2 < k.h2)
            a.add<2>(k, d2, (float)(qx - px), (float)(qy - py), 0.f, rvel[j], 1.f / rrho[j]);
    });
    if constexpr (S > 1) {
#pragma unroll
        for (int o = 1; o < S; o <<= 1) a.add_lanes(o);
    }
    auto boundary = [&](const KConst& k, double qx, double qy, double, const float4* bvel,
                        const float4* bnrm, BAcc& b) {
        for_each_candidate2<S>(k, bcstart, bpos, qx, qy, sub, [&](int j, double px, double py) {
            const double d2 = sq_dist2(px, py, qx, qy);
            if (d2 < k.h2)
                b.add_exact<2>(k, qx, qy, 0.0, make_double4(px, py, 0.0, 0.0), d2, bvel[j],
                               bnrm[j].w);
        });
    };
    finish_node<2, S>(k, a, qx, qy, 0.0, cx, cy, 0, out, rpos, rcstart, boundary, bvel, bnrm,
                      vrho, vvol, vb, bits);
}

// 3D with the brick's neighbourhood staged in LDS: one workgroup of 512
// threads per brick, thread = node, or S workgroups of 8 / S z-planes each
// with S lanes per node.  The cells within one cell of the nodes form
// <= kStageRows x-rows of <= kStageCx cells; their particles (contiguous per
// row in the cell-sorted order) are copied once, each as its FP32 offset from
// its own cell corner with 1/rho_j, first the real and behind them the
// boundary ones, and every node walks its 3 x 3 x 3 cells from LDS in the
// order of the global walk.
// q - x_j = (q - C_q) - (x_j - C_j) + (C_q - C_j) with C the FP64 cell
// corners, so the FP32 difference is accurate to a few ulp of h.
// Membership is pre-tested in FP32 with a band around h^2 in which the
// exact FP64 test on the original positions decides (also at r = 0 and for
// particles clamped into a border cell), so the neighbour sets stay exact.
constexpr int kStageCap = 4096;
constexpr int kStageRows = 64;
constexpr int kStageCx = 8;

// The staged neighbourhood.  px is taken from the corner of the row's first
// cell (NaN: exact test only), py and pz from the particle's own cell; pw is
// 1 / rho of a real particle, x from its own cell of a boundary particle.
// Separate arrays: the membership test reads 12 bytes per candidate as three
// 4-byte loads.  Two workgroups per CU, which is also what their registers
// allow.
template <int S>
struct Stage {
    // the scan reads up to 4 S - 1 entries beyond a row
    float px[kStageCap + 4 * S], py[kStageCap + 4 * S], pz[kStageCap + 4 * S],
        pw[kStageCap + 4 * S];
    int cs[kStageRows][kStageCx + 1];    // cell starts of the rows, global
    int bcs[kStageRows][kStageCx + 1];   // the boundary's
    int rg[kStageRows], brg[kStageRows]; // global - staged index of a row
};

// One lane's part (candidates c0, c0 + S, ...) of a staged row's range
// [c0, je): in chunks of 32, the cheap FP32 test near(j) sets a bit per
// candidate not surely outside, then the lane visits only its own bits: fast(j)
// says whether the FP32 test is certain (and then adds the pair), and the
// others go to exact(j) afterwards, the lanes' together.  (A lane has ~15% of
// its candidates within h, so the wave does not run the accumulation for every
// candidate.)  The test appends its bit at the low end, so the highest set bit
// is the next in order; it runs four candidates at a time past the end of the
// range, whose bits are cleared.
template <int S, typename Near, typename Fast, typename Exact>
__device__ __forceinline__ void staged_range(int c0, int je, Near&& near, Fast&& fast,
                                             Exact&& exact) {
    for (; c0 < je; c0 += 32 * S) {
        const int nc = min((je - c0 + S - 1) / S, 32);
        uint32_t m = 0u, mexact = 0u;
        int i = 0;
        for (; i < nc; i += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) m = m + m + near(c0 + (i + u) * S);
        }
        // candidate 0 to bit 31, candidates nc and on cleared
        m = (m << (32 - i)) & (uint32_t)((int32_t)0x80000000 >> (nc - 1));
        while (m) {
            const int b = __builtin_clz(m);
            const uint32_t bit = 0x80000000u >> b;
            m &= ~bit;
            if (!fast(c0 + b * S)) mexact |= bit;
        }
        while (mexact) {
            const int b = __builtin_clz(mexact);
            mexact &= ~(0x80000000u >> b);
            exact(c0 + b * S);
        }
    }
}

// The staged rows around one node: f(jb, je, rg, ty, tz) per row with
// candidates, jb .. je its staged range and q - C its y and z.
// Cells whose nearest point lies beyond h (1 - 2e-6) are skipped: a whole row
// by its y and z distance, the end cells of a row by their x distance.  Only
// interior cells are culled (a border cell may hold particles clamped into it
// from outside its extent).  The margin is twenty times the FP32 error of
// these distances; a member it drops lies within 2.1e-6 h of the cutoff,
// where W and W' are below 1e-17 and 5e-12 of their peaks, far below FP32
// resolution of the sums.  On a lattice aligned with the cell grid (a node
// every half cell) it skips the cells behind a node on a cell face; the nodes
// of a wave share their z, so the rows behind them in z are skipped by the
// whole wave.
struct StagedRows {
    int clo0, clo1, clo2, ncy;
    template <typename F>
    __device__ __forceinline__ void walk(const KConst& k, double qx, double qy, double qz,
                                         const int (*cs)[kStageCx + 1], const int* rgs,
                                         F&& f) const {
        const int cx = cell_coord(qx, k.cell_lo[0], k.cell_inv, k.cdims[0]);
        const int cy = cell_coord(qy, k.cell_lo[1], k.cell_inv, k.cdims[1]);
        const int cz = cell_coord(qz, k.cell_lo[2], k.cell_inv, k.cdims[2]);
        const int xlo = max(cx - 1, 0), xhi = min(cx + 1, k.cdims[0] - 1);
        const int ylo = max(cy - 1, 0), yhi = min(cy + 1, k.cdims[1] - 1);
        const int zlo = max(cz - 1, 0), zhi = min(cz + 1, k.cdims[2] - 1);
        const int i0 = xlo - clo0, i1 = xhi - clo0;
        const float csf = (float)k.cell_size;
        const float h2c = (float)k.h2 * (1.f - 4e-6f);
        auto gap = [csf](float t) { return fmaxf(fmaxf(-t, t - csf), 0.f); };   // q - C -> distance
        const bool cut_l = xlo < xhi && xlo > 0, cut_r = xhi > xlo && xhi < k.cdims[0] - 1;
        const float gl = gap((float)(qx - cell_corner(k, 0, xlo)));
        const float gr = gap((float)(qx - cell_corner(k, 0, xhi)));
        // (0: the cell stays; rem below is positive)
        const float dl2 = cut_l ? gl * gl : 0.f, dr2 = cut_r ? gr * gr : 0.f;
        for (int z = zlo; z <= zhi; z++) {
            const float tz = (float)(qz - cell_corner(k, 2, z));
            const float gz = z > 0 && z < k.cdims[2] - 1 ? gap(tz) : 0.f;
            for (int y = ylo; y <= yhi; y++) {
                const float ty = (float)(qy - cell_corner(k, 1, y));
                const float gy = y > 0 && y < k.cdims[1] - 1 ? gap(ty) : 0.f;
                const float rem = h2c - gy * gy - gz * gz;
                if (!(rem > 0.f)) continue;
                const int r = (z - clo2) * ncy + (y - clo1);
                const int rg = rgs[r];
                const int jb = cs[r][i0 + (dl2 >= rem)] - rg;
                const int je = cs[r][i1 + 1 - (dr2 >= rem)] - rg;
                if (jb < je) f(jb, je, rg, ty, tz);
            }
        }
    }
};

// Lanes per node: the fewest that fill the machine (a brick by itself takes
// 52 us with one lane per node).  By the particles, not the bricks of the last
// generation, so that a state gives the same bits however it was reached.  us
// with 1, 2, 4, 8 lanes:
//   576 particles 51, 31, 26, 21     16,000  53, 34, 28, 27
//   32,000        54, 35, 33, 47     64,800  59, 45, 55, 71
//   212,503       94, 90, 112, 153   300,000 112, 116, 147, 219
//   1,012,500    264, 274, 382, 558
// A launch holds less than 2^32 threads, and the first generation's grid covers
// every brick: the largest lattices take fewer lanes.
inline int sums_lanes(int64_t n, int64_t nbricks) {
    int lanes = n <= 16000 ? 8 : (n <= 32000 ? 4 : (n <= 250000 ? 2 : 1));
    while (nbricks * 512 * lanes > (int64_t)UINT32_MAX) lanes /= 2;
    return lanes;
}

// Bound by instructions and the latency of the walk (of 264 us at 1M:
// staging about 40, candidate tests 100, sums 80, boundary 45).  Before (one lane per node
// for all sizes, the boundary walked in global memory, two masks per test,
// rows staged through a binary search): 70 us at 576 particles, 77 at 64,800,
// 120 at 212,503, 297 at 1,012,500.
template <int S>
__global__ void __launch_bounds__(512, 4) k_virtual_sums3s(
    KConst k, const int32_t* brick_of_slot, const int32_t* nslots_p,
    const double4* rpos, const float4* rvel, const float* rrho, const float* rrinv,
    const float4* rofs, const int32_t* rcstart, const double4* bpos,
    const float4* bofs, const float4* bvel, const float4* bnrm, const int32_t* bcstart,
    float* vrho, float* vvol, float* vb, uint32_t* bits) {
    constexpr int kPlanes = kBrick / S;
    constexpr int kRowsAtOnce = 5;   // rows a wave loads at once (a brick has about 49; with 7: 268 for 263 us at 1M)
    __shared__ Stage<S> st;
    const int nslots = *nslots_p;   // the grid may exceed the slot count
    if ((int)blockIdx.x >= nslots * S) return;
    const int part = xcd_remap(blockIdx.x, nslots * S);
    const int slot = part / S;
    const int brick = brick_of_slot[slot];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // a wave: the 8 x 8 nodes of one z-plane of the brick, or 8 x 8 / S of them
    const int sub = S > 1 ? t % S : 0;
    const int node = (part % S) * (512 / S) + t / S;
    const int bx = brick % k.bdims[0];
    const int by = (brick / k.bdims[0]) % k.bdims[1];
    const int bz = brick / k.bdims[0] / k.bdims[1];
    const int n0[3] = {bx * kBrick, by * kBrick, bz * kBrick + (part % S) * kPlanes};
    const int cx = n0[0] + (node & 7), cy = n0[1] + ((node >> 3) & 7),
              cz = bz * kBrick + (node >> 6);
    const int64_t out = (int64_t)slot * 512 + node;
    if (S > 1 && n0[2] >= k.ndims[2]) {   // no plane of this block is on the lattice
        if (sub == 0) vrho[out] = vvol[out] = vb[out] = 0.f;
        return;
    }
    int clo[3], nc[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const int last = min(n0[a] + (a == 2 ? kPlanes : kBrick) - 1, k.ndims[a] - 1);
        clo[a] = max(cell_coord(node_coord(k.origin[a], n0[a], k.spacing), k.cell_lo[a],
                                k.cell_inv, k.cdims[a]) - 1, 0);
        nc[a] = min(cell_coord(node_coord(k.origin[a], last, k.spacing), k.cell_lo[a],
                               k.cell_inv, k.cdims[a]) + 1, k.cdims[a] - 1) - clo[a] + 1;
    }
    const int ncx = nc[0], ncy = nc[1], nrows = nc[1] * nc[2];
    bool staged = ncx <= kStageCx && nrows <= kStageRows, pooled = false;
    int nboundary = 0;
    if (staged) {
        for (int e = t; e < nrows * (kStageCx + 1); e += 512) {
            const int r = e / (kStageCx + 1), i = e % (kStageCx + 1);
            if (i > ncx) continue;
            const int64_t g = ((int64_t)(clo[2] + r / ncy) * k.cdims[1] + clo[1] + r % ncy) *
                                  k.cdims[0] + clo[0] + i;
            st.cs[r][i] = rcstart[g];
            st.bcs[r][i] = bcstart[g];
        }
        __syncthreads();
        // Every wave scans the rows' lengths for itself (lane = row).
        const int row = min(lane, nrows - 1);
        const int rlen = lane < nrows ? st.cs[row][ncx] - st.cs[row][0] : 0;
        const int blen = lane < nrows ? st.bcs[row][ncx] - st.bcs[row][0] : 0;
        int rend = rlen, bend = blen;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int a = __shfl_up(rend, o, 64), b = __shfl_up(bend, o, 64);
            if (lane >= o) {
                rend += a;
                bend += b;
            }
        }
        const int total = __shfl(rend, 63, 64);
        staged = total <= kStageCap;
        nboundary = __shfl(bend, 63, 64);
        pooled = staged && total + nboundary <= kStageCap;
        if (wave == 0 && lane < nrows) {
            st.rg[lane] = st.cs[lane][0] - (rend - rlen);
            st.brg[lane] = st.bcs[lane][0] - (total + bend - blen);
        }
        // The waves take the rows in turn, kRowsAtOnce of them loading together.
        auto put = [&](int e, const float4& p, int cell, float pw) {
            // x relative to the corner of the row's first cell (C_c - C_clo =
            // c - clo cells), rounded once from FP64; a particle marked for
            // the exact test only gets x = NaN, which no FP32 test passes
            st.px[e] = p.w < 0.f ? __builtin_nanf("")
                                 : (float)((double)p.x + (double)cell * k.cell_size);
            st.py[e] = p.y;
            st.pz[e] = p.z;
            st.pw[e] = pw;
        };
        auto put_real = [&](int e, const float4& p, float rinv) {
            put(e, p, (int)p.w - 1 - clo[0], rinv);
        };
        auto put_boundary = [&](int r, int e, int at, const float4& p) {
            int cell = 0;
            for (int i = 1; i < ncx; i++) cell += st.bcs[r][i] <= st.bcs[r][0] + e;
            put(at + e, p, cell, p.x);
        };
        for (int r0 = wave; staged && r0 < nrows; r0 += 8 * kRowsAtOnce) {
            float4 p[kRowsAtOnce], pb[kRowsAtOnce];
            float ri[kRowsAtOnce];
            int at[kRowsAtOnce], bat[kRowsAtOnce], len[kRowsAtOnce], bl[kRowsAtOnce];
#pragma unroll
            for (int u = 0; u < kRowsAtOnce; u++) {
                const int r = min(r0 + 8 * u, nrows - 1);
                len[u] = r0 + 8 * u < nrows ? __shfl(rlen, r, 64) : 0;
                bl[u] = r0 + 8 * u < nrows && pooled ? __shfl(blen, r, 64) : 0;
                at[u] = __shfl(rend, r, 64) - len[u];
                bat[u] = total + __shfl(bend, r, 64) - bl[u];
                if (lane < len[u]) {
                    p[u] = rofs[st.cs[r][0] + lane];
                    ri[u] = rrinv[st.cs[r][0] + lane];
                }
                if (lane < bl[u]) pb[u] = bofs[st.bcs[r][0] + lane];
            }
#pragma unroll
            for (int u = 0; u < kRowsAtOnce; u++) {
                if (lane < len[u]) put_real(at[u] + lane, p[u], ri[u]);
                const int r = min(r0 + 8 * u, nrows - 1);
                if (lane < bl[u]) put_boundary(r, lane, bat[u], pb[u]);
                for (int e = 64 + lane; e < len[u]; e += 64)
                    put_real(at[u] + e, rofs[st.cs[r][0] + e], rrinv[st.cs[r][0] + e]);
                for (int e = 64 + lane; e < bl[u]; e += 64)
                    put_boundary(r, e, bat[u], bofs[st.bcs[r][0] + e]);
            }
        }
        __syncthreads();
    }
    if (cx >= k.ndims[0] || cy >= k.ndims[1] || cz >= k.ndims[2]) {
        if (sub == 0) vrho[out] = vvol[out] = vb[out] = 0.f;
        return;   // uniform over the lanes of a node
    }
    const double qx = node_coord(k.origin[0], cx, k.spacing);
    const double qy = node_coord(k.origin[1], cy, k.spacing);
    const double qz = node_coord(k.origin[2], cz, k.spacing);
    RealAcc a;
    if (!staged) {
        if (sub != 0) return;
        real_walk_global3(k, rcstart, rpos, rvel, rrho, qx, qy, qz, a);
        finish_node<3>(k, a, qx, qy, qz, cx, cy, cz, out, rpos, rcstart,
                       BoundaryWalkGlobal3{bcstart, bpos}, bvel, bnrm, vrho,
                       vvol, vb, bits);
        return;
    }
    // The membership test and a real member's sums take x relative to the same
    // corner C_clo for all cells of a row (one offset per node, rounded once
    // from FP64: within 2e-7 h for offsets of up to three cells, inside the
    // FP64 band for the test and far below the tolerance of the sums).
    const float tx = (float)(qx - cell_corner(k, 0, clo[0]));
    // h2_min < d2f < h2f_lo as one unsigned test on the bits (NaN fails).
    // Below h2_min (the band's width, far above the error of d2f near 0)
    // the exact test decides, so a fast member's accurate d2f is > 0.
    const uint32_t lo_min = __float_as_uint(k.h2f_hi - k.h2f_lo);
    const uint32_t lo_span = __float_as_uint(k.h2f_lo) - lo_min - 1u;
    auto sq = [](const float3& d) { return d.x * d.x + d.y * d.y + d.z * d.z; };
    auto sure = [&](float d2f) { return __float_as_uint(d2f) - lo_min - 1u < lo_span; };
    const StagedRows rows{clo[0], clo[1], clo[2], ncy};
    rows.walk(k, qx, qy, qz, st.cs, st.rg, [&](int jb, int je, int rg, float ty, float tz) {
        auto offset = [&](int j) {
            return make_float3(tx - st.px[j], ty - st.py[j], tz - st.pz[j]);
        };
        staged_range<S>(
            jb + sub, je, [&](int j) { return !(sq(offset(j)) >= k.h2f_hi); },
            [&](int j) {
                const float3 d = offset(j);
                const float d2f = sq(d);
                const bool in = sure(d2f);
                if (in) a.add_fast<3>(k, d2f, d.x, d.y, d.z, rvel[j + rg], st.pw[j]);
                return in;
            },
            [&](int j) {
                // the reference's FP64 test and the accurate spline
                const int g = j + rg;
                const double4 pj = rpos[g];
                const double d2 = sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz);
                if (d2 < k.h2)
                    a.add<3>(k, d2, (float)(qx - pj.x), (float)(qy - pj.y), (float)(qz - pj.z),
                             rvel[g], st.pw[j]);
            });
    });
    if constexpr (S > 1) {
#pragma unroll
        for (int o = 1; o < S; o <<= 1) a.add_lanes(o);
    }
    // One lane's part of the boundary walk, over the staged rows as well; from
    // global memory where the boundary did not fit the stage.  The sums take x
    // from the particle's own cell.
    auto boundary = [&](const KConst& k, double qx, double qy, double qz, const float4* bvel,
                        const float4* bnrm, BAcc& b) {
        if (!pooled) {
            if (sub == 0) BoundaryWalkGlobal3{bcstart, bpos}(k, qx, qy, qz, bvel, bnrm, b);
            return;
        }
        if (nboundary == 0) return;
        const int xlo = max(cell_coord(qx, k.cell_lo[0], k.cell_inv, k.cdims[0]) - 1, 0);
        float tx0 = (float)(qx - cell_corner(k, 0, xlo));
        float tx1 = (float)(qx - cell_corner(k, 0, xlo + 1));
        float tx2 = (float)(qx - cell_corner(k, 0, xlo + 2));
        const float s1 = (float)((double)(xlo - clo[0]) + 0.5) * (float)k.cell_size;
        rows.walk(k, qx, qy, qz, st.bcs, st.brg, [&](int jb, int je, int rg, float ty, float tz) {
            auto offset = [&](int j) {
                return make_float3(tx - st.px[j], ty - st.py[j], tz - st.pz[j]);
            };
            staged_range<S>(
                jb + sub, je, [&](int j) { return !(sq(offset(j)) >= k.h2f_hi); },
                [&](int j) {
                    float3 d = offset(j);
                    const bool in = sure(sq(d));
                    if (in) {
                        const float own = st.pw[j], c = st.px[j] - own - s1;
                        d.x = (c < 0.f ? tx0 : (c < (float)k.cell_size ? tx1 : tx2)) - own;
                        b.add_fast(k, sq(d), d.x, d.y, d.z, bvel[j + rg], bofs[j + rg].w);
                    }
                    return in;
                },
                [&](int j) {
                    const int g = j + rg;
                    const double4 pj = bpos[g];
                    const double d2 = sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz);
                    if (d2 < k.h2)
                        b.add_exact<3>(k, qx, qy, qz, pj, d2, bvel[g], bnrm[g].w);
                });
        });
    };
    finish_node<3, S>(k, a, qx, qy, qz, cx, cy, cz, out, rpos, rcstart, boundary, bvel, bnrm, vrho,
                      vvol, vb, bits);
}

// Column order of the 3D slots, for the CG iteration's walk up z-runs of
// bricks: the active bricks of every (x, y) column bottom to top, column after
// column.  The scan of the columns' counts gives every column its place.
struct LoadColumn {
    static constexpr bool kWide = false;
    int32_t plane, nz;   // columns, bricks of a column
    const int32_t* slot_of_brick;
    __device__ __forceinline__ int operator()(int64_t col) const {
        int len = 0;
#pragma unroll 8
        for (int z = 0; z < nz; z++) len += slot_of_brick[col + (int64_t)z * plane] >= 0;
        return len;
    }
};
struct StoreColumn {
    static constexpr bool kWide = false;
    int32_t* off;
    __device__ __forceinline__ void operator()(int64_t col, int, int pre) const {
        off[col] = pre;
    }
};

// Tables over the slots of one generation, in one launch: the slots of the
// 3^D neighbour bricks of every slot (zero brick if absent), and in 3D the
// column order, order[off[column] + active bricks below] = slot (by the thread
// of the middle neighbour), and the gradient's units (by the first threads;
// see unit_append).
template <int D>
__global__ void __launch_bounds__(256) k_slot_tables(
    KConst k, const int32_t* brick_of_slot, const int32_t* slot_of_brick, const int32_t* nslots_p,
    int64_t grid, int32_t zero, int32_t* nbr, const int32_t* off, int32_t* order, UnitArgs ua) {
    constexpr int NN = D == 3 ? 27 : 9;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if constexpr (D == 3) unit_append(k, ua, i);
    const int32_t nsl = *nslots_p;
    // the grid may exceed the slot count; a count beyond the grid leaves the
    // tables to the rerun on the exact grid
    if (i >= (int64_t)nsl * NN || nsl > grid) return;
    const int64_t slot = i / NN;
    const int t = (int)(i - slot * NN);
    const int brick = brick_of_slot[slot];
    const int bx = brick % k.bdims[0];
    const int by = (brick / k.bdims[0]) % k.bdims[1];
    const int bz = D == 3 ? brick / k.bdims[0] / k.bdims[1] : 0;
    const int nx = bx + (t % 3) - 1, ny = by + (t / 3) % 3 - 1,
              nz = D == 3 ? bz + t / 9 - 1 : 0;
    int s = zero;
    if (nx >= 0 && ny >= 0 && nz >= 0 && nx < k.bdims[0] && ny < k.bdims[1] &&
        nz < k.bdims[2]) {
        const int sl = slot_of_brick[((int64_t)nz * k.bdims[1] + ny) * k.bdims[0] + nx];
        if (sl >= 0) s = sl;
    }
    nbr[slot * 27 + t] = s;
    if (D == 3 && t == 13) {
        const int32_t plane = k.bdims[0] * k.bdims[1];
        const int32_t col = brick - bz * plane;
        int d = 0;
#pragma unroll 8
        for (int z = 0; z < bz; z++) d += slot_of_brick[col + (int64_t)z * plane] >= 0;
        order[off[col] + d] = (int32_t)slot;
    }
}

// Words of the lattice bitmask before each word, for the node ranks.
struct LoadPopc {
    static constexpr bool kWide = true;
    __device__ __forceinline__ int4 four(int64_t i) const {
        const uint4 w = *(const uint4*)(bits + i);
        return make_int4(__popc(w.x), __popc(w.y), __popc(w.z), __popc(w.w));
    }
    const uint32_t* bits;
    __device__ __forceinline__ int operator()(int64_t i) const { return __popc(bits[i]); }
};
struct StorePrefix {
    static constexpr bool kWide = true;
    __device__ __forceinline__ void four(int64_t i, int4 pre) const { *(int4*)(prefix + i) = pre; }
    int32_t* prefix;
    __device__ __forceinline__ void operator()(int64_t i, int, int pre) const { prefix[i] = pre; }
};

template <int D, int NB>
__global__ void __launch_bounds__(NB) k_node_rank(KConst k,
                                                  const int32_t* brick_of_slot,
                                                  const int32_t* nslots_p,
                                                  const float* vvol,
                                                  const uint32_t* bits,
                                                  const int32_t* prefix,
                                                  int32_t* rank) {
    const int slot = blockIdx.x;
    if (slot >= *nslots_p) return;
    const int64_t out = (int64_t)slot * NB + threadIdx.x;
    if (!(vvol[out] > 0.f)) {
        rank[out] = -1;
        return;
    }
    const int brick = brick_of_slot[slot];
    const int t = threadIdx.x;
    const int bx = brick % k.bdims[0];
    const int by = (brick / k.bdims[0]) % k.bdims[1];
    const int bz = D == 3 ? brick / k.bdims[0] / k.bdims[1] : 0;
    const int cx = bx * kBrick + (t & 7), cy = by * kBrick + ((t >> 3) & 7),
              cz = D == 3 ? bz * kBrick + (t >> 6) : 0;
    const int64_t lin = ((int64_t)cz * k.ndims[1] + cy) * k.ndims[0] + cx;
    const uint32_t word = bits[lin >> 5];
    const uint32_t below = word & ((1u << (lin & 31)) - 1u);
    rank[out] = prefix[lin >> 5] + __popc(below);
}

// CG initial guess for every node of the active bricks (0 off the set): x0
// for the residual, and the solution in its two parts (base x0, correction
// 0; see k_fold_x in vps_stencil.hip).
template <int D, int NB>
__global__ void __launch_bounds__(NB) k_warm_start(
    int mode, KConst k, const int32_t* brick_of_slot, const float* vvol,
    const int32_t* rank, const float* p_rank_prev, int64_t nprev,
    const int32_t* prev_slot_of_brick, const float* x_prev, StartOut so) {
    const int slot = blockIdx.x;
    const int64_t out = (int64_t)slot * NB + threadIdx.x;
    float v = 0.f;
    if (vvol[out] > 0.f) {
        if (mode == VPS_WARM_INDEX_CARRY) {
            const int r = rank[out];
            if (r < nprev) v = p_rank_prev[r];
        } else if (mode == VPS_WARM_NODE_KEYED || mode == VPS_WARM_LEARNED) {
            if (prev_slot_of_brick) {
                const int ps = prev_slot_of_brick[brick_of_slot[slot]];
                if (ps >= 0) v = x_prev[(int64_t)ps * NB + threadIdx.x];
            }
        }
    }
    so.put(out, v);
}

// After the solve: pressures by reference rank (index-carry warm start of
// the next step) and q = V p for the pressure gradient.  With xb, the
// solution's two parts are folded into the pressures on the way.
__global__ void __launch_bounds__(256) k_after_solve(int64_t nnode,
                                                     const float* vvol,
                                                     float* x, const double* xb,
                                                     const int32_t* rank,
                                                     float* p_rank, float* q,
                                                     SolveGuard guard) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nnode || !solve_accepted(guard)) return;
    const float V = vvol[i];
    float p = x[i];
    if (xb) {
        p = (float)(xb[i] + p);
        x[i] = p;
    }
    q[i] = V * p;
    if (V > 0.f) p_rank[rank[i]] = p;
}

}  // namespace

// Slot-indexed passes of one generation on a grid of `grid` blocks (slots);
// blocks at or beyond the device-side slot count return at once.  first: not a
// rerun on the exact grid (the gradient's units are appended once).
static int generate_slots(vps_context* c, int w, int64_t grid, bool first) {
    const int D = c->dim;
    const int rs = c->cur;
    const int32_t* nsl = (const int32_t*)c->counters.p;   // slot count
    int64_t* dcnt = c->counters.p;
    if (D == 3) {
        auto run = [&](auto kern, int s) {
            hipLaunchKernelGGL(kern, dim3((unsigned)(grid * s)), dim3(512), 0, c->stream, c->k,
                               c->slot_brick[w].p, nsl, c->rpos[rs].p, c->rvel[rs].p, c->rrho.p,
                               c->rrinv.p, c->rofs.p, c->cell_start.p, c->bpos.p, c->bofs.p,
                               c->bvel.p, c->bnrm.p, c->bcell_start.p, c->vrho.p, c->vvol.p,
                               c->vb.p, c->bits.p);
        };
        const int lanes = sums_lanes(c->n, c->nbricks);
        if (lanes == 8) run(k_virtual_sums3s<8>, 8);
        else if (lanes == 4) run(k_virtual_sums3s<4>, 4);
        else if (lanes == 2) run(k_virtual_sums3s<2>, 2);
        else run(k_virtual_sums3s<1>, 1);
    } else {
        auto run = [&](auto kern, int s) {
            hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * s), 0, c->stream, c->k,
                               c->slot_brick[w].p, nsl, c->rpos[rs].p, c->rvel[rs].p, c->rrho.p,
                               c->cell_start.p, c->bpos.p, c->bvel.p, c->bnrm.p,
                               c->bcell_start.p, c->vrho.p, c->vvol.p, c->vb.p, c->bits.p);
        };
        if (walk_lanes2(c->n) == 4) run(k_virtual_sums2<4>, 4);
        else run(k_virtual_sums2<1>, 1);
    }
    // the column order and the tables, on the grid (before the read-back
    // below, so that they run while the host waits)
    const int32_t* bos = c->slot_brick[w].p;
    const int32_t* sob = c->brick_slot[w].p;
    if (D == 3) {
        const int32_t plane = c->k.bdims[0] * c->k.bdims[1];
        // (one column per thread: each is a loop of its own)
        VPS_TRY(scan_launch_as<1>(c, LoadColumn{plane, c->k.bdims[2], sob},
                                  StoreColumn{c->col_off.p}, plane, nullptr));
        const UnitArgs ua = gradient_units(c, first);
        hipLaunchKernelGGL(k_slot_tables<3>, dim3(blocks(std::max(grid * 27, ua.total), 256)),
                           dim3(256), 0, c->stream, c->k, bos, sob, nsl, grid,
                           (int32_t)c->nbricks, c->nbr_slot.p, c->col_off.p, c->col_order.p, ua);
    } else
        hipLaunchKernelGGL(k_slot_tables<2>, dim3(blocks(grid * 9, 256)), dim3(256), 0, c->stream,
                           c->k, bos, sob, nsl, grid, (int32_t)c->nbricks, c->nbr_slot.p,
                           (const int32_t*)nullptr, (int32_t*)nullptr, UnitArgs{});
    VPS_TRY(scan_launch(c, LoadPopc{c->bits.p}, StorePrefix{(int32_t*)c->word_prefix.p}, c->nwords,
                        (int32_t*)(dcnt + 1)));
    if (D == 3)
        hipLaunchKernelGGL((k_node_rank<3, 512>), dim3((unsigned)grid),
                           dim3(512), 0, c->stream, c->k, c->slot_brick[w].p,
                           nsl, c->vvol.p, c->bits.p,
                           (const int32_t*)c->word_prefix.p, c->vrank.p);
    else
        hipLaunchKernelGGL((k_node_rank<2, 64>), dim3((unsigned)grid),
                           dim3(64), 0, c->stream, c->k, c->slot_brick[w].p,
                           nsl, c->vvol.p, c->bits.p,
                           (const int32_t*)c->word_prefix.p, c->vrank.p);
    VPS_HIP(c, hipGetLastError());
    // slot, virtual and gradient-unit counts in one read-back
    VPS_HIP(c, hipMemcpyAsync(c->host_counters, dcnt, 24, hipMemcpyDeviceToHost,
                              c->stream));
    VPS_HIP(c, hipStreamSynchronize(c->stream));
    return VPS_OK;
}

__global__ void __launch_bounds__(256) k_fill_u32(uint32_t* p, int64_t n, uint32_t v) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

int virtual_generate(vps_context* c) {
    // The new slot map goes into the buffer that does NOT hold the last solved
    // pressures, so both warm starts can still read them.
    const int w = c->last_solve_buf >= 0 ? 1 - c->last_solve_buf : 0;
    const int D = c->dim;
    const int s = c->cur;
    // brick flags are zero on entry (cleared by AssignSlot)
    const unsigned mb = blocks(c->n, 256) > 0 ? blocks(c->n, 256) : 1;
    if (D == 3)
        hipLaunchKernelGGL(k_mark_bricks<3>, dim3(mb), dim3(256),
                           0, c->stream, c->rpos[s].p, c->n, c->k,
                           c->brick_flag.p, c->bits.p, c->nwords,
                           (int32_t*)(c->counters.p + 2));
    else
        hipLaunchKernelGGL(k_mark_bricks<2>, dim3(mb), dim3(256),
                           0, c->stream, c->rpos[s].p, c->n, c->k,
                           c->brick_flag.p, c->bits.p, c->nwords,
                           (int32_t*)(c->counters.p + 2));
    int64_t* dcnt = c->counters.p;
    VPS_TRY(scan_launch(c, LoadFlag{c->brick_flag.p},
                        AssignSlot{c->brick_flag.p, c->brick_slot[w].p, c->slot_brick[w].p},
                        c->nbricks, (int32_t*)dcnt));
    // The slot count stays on the device: the slot passes run on a grid
    // sized from the last generation's count (the first time by the bricks
    // that the particles can mark at most, see k_mark_bricks), and again on
    // the exact grid in the rare step where it grew past that.
    double most = (double)c->n;
    for (int a = 0; a < D; a++) most *= std::floor((2 * c->k.h / c->k.spacing + 2) / kBrick) + 2;
    if (c->nslots > 0) most = (double)(c->nslots + c->nslots / 8 + 64);
    const int64_t grid = (int64_t)std::min(most, (double)c->nbricks);
    VPS_TRY(generate_slots(c, w, grid, true));
    int64_t nslots = *(int32_t*)c->host_counters;
    if (nslots > grid) {
        hipLaunchKernelGGL(k_fill_u32, dim3(blocks(c->nwords, 256)), dim3(256), 0,
                           c->stream, c->bits.p, c->nwords, 0u);
        VPS_TRY(generate_slots(c, w, nslots, false));
        nslots = *(int32_t*)c->host_counters;
    }
    c->nslots = nslots;
    c->which = w;
    c->nvirt = nslots ? *(int32_t*)(c->host_counters + 1) : 0;
    c->grad_nunits = *(int32_t*)(c->host_counters + 2);
    return VPS_OK;
}

int warm_start(vps_context* c, int mode) {
    const int w = c->which;
    const int lb = c->last_solve_buf;
    const int32_t* prev_map = lb >= 0 ? c->brick_slot[lb].p : nullptr;
    const float* p_prev = lb >= 0 ? c->p_by_rank[lb].p : nullptr;
    const int64_t nprev = lb >= 0 ? c->last_solve_nvirt : 0;
    const float* x_prev = lb >= 0 ? c->vx[lb].p : nullptr;
    if (c->dim == 3)
        hipLaunchKernelGGL((k_warm_start<3, 512>), dim3((unsigned)c->nslots),
                           dim3(512), 0, c->stream, mode, c->k,
                           c->slot_brick[w].p, c->vvol.p, c->vrank.p, p_prev,
                           nprev, prev_map, x_prev, start_out(c));
    else
        hipLaunchKernelGGL((k_warm_start<2, 64>), dim3((unsigned)c->nslots),
                           dim3(64), 0, c->stream, mode, c->k,
                           c->slot_brick[w].p, c->vvol.p, c->vrank.p, p_prev,
                           nprev, prev_map, x_prev, start_out(c));
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

int after_solve(vps_context* c, SolveGuard g, bool fold) {
    const int w = c->which;
    const int64_t nn = c->nslots * c->brick_nodes;
    if (nn == 0) return VPS_OK;
    hipLaunchKernelGGL(k_after_solve, dim3(blocks(nn, 256)), dim3(256), 0,
                       c->stream, nn, c->vvol.p, c->vx[w].p, fold ? c->vxb.p : nullptr, c->vrank.p,
                       c->p_by_rank[w].p, c->vq.p, g);
    VPS_HIP(c, hipGetLastError());
    if (g.mode == 0) after_solve_commit(c);
    return VPS_OK;
}

void after_solve_commit(vps_context* c) {
    if (c->nslots * c->brick_nodes == 0) return;
    c->last_solve_buf = c->which;
    c->last_solve_nvirt = c->nvirt;
}

}  // namespace vps
