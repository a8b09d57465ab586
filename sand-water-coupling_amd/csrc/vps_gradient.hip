// vps_gradient.hip -- pressure gradient + velocity update, advection, and the
// neighbour query used by tests.
//
// Replaces VirtualParticle::applyPressureGradient
// (Cores/Structures/VirtualParticle.cpp:110-134):
//   v_i += sum_{J in N_H(i)} V_J p_J gradK_H(x_i - x_J)
//        - sum_{b in N_h(i)} V_b min(n_b.(v_i - v_b), 0) n_b W_h(x_i - x_b)
// (no dt, no 1/rho; v_i on the right is the pre-update velocity).
// Virtual particles are lattice nodes, so the virtual neighbours of x_i are
// found by scanning the node box around x_i: the node coordinates of each
// axis are formed once per particle (origin + c * spacing, as
// Grid::dataPosition rounds them) and the exact FP64 test
// ((dx^2 + dy^2) + dz^2) < H^2 decides membership.  The brick map gives
// q_J = V_J p_J (zero on non-virtual nodes).
#include <algorithm>
#include <cmath>

#include "vps_internal.h"

namespace vps {
namespace {

inline unsigned blocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

constexpr int kBox = 10;   // max node candidates per axis (2H/s + 2)

// Boundary part of the update: -sum_b V_b min(n_b.(v_i - v_b), 0) n_b W_h.
// L lanes share a particle, each taking every L-th candidate of a row.
template <int D, int L = 1>
__device__ __forceinline__ void boundary_term(const KConst& k, const double4& q,
                                              const float4& vi, const double4* bpos,
                                              const float4* bvel, const float4* bnrm,
                                              const int32_t* bcstart, float& fx,
                                              float& fy, float& fz, int sub = 0) {
    auto visit = [&](int j, const double4& pj) {
        const double d2 = D == 3 ? sq_dist3(pj.x, pj.y, pj.z, q.x, q.y, q.z)
                                 : sq_dist2(pj.x, pj.y, q.x, q.y);
        if (d2 < k.h2) {
            // W from the select-free spline (no division): r and 1/r from one rsq
            const float d2f = (float)d2;
            const float rinv = d2f > 0.f ? __builtin_amdgcn_rsqf(d2f) : 0.f;
            const float w = spline_w_ab(spline_ab(d2f * rinv, k.inv_h), k.c0h);
            const float4 vb = bvel[j];
            float4 nb = bnrm[j];
            if (nb.x == 0.f && nb.y == 0.f && (D == 2 || nb.z == 0.f)) {
                // a grain: the unit vector from the grain to the particle
                // (none when they coincide)
                nb.x = (float)(q.x - pj.x) * rinv;
                nb.y = (float)(q.y - pj.y) * rinv;
                nb.z = D == 3 ? (float)(q.z - pj.z) * rinv : 0.f;
            }
            const float dn = nb.x * (vi.x - vb.x) + nb.y * (vi.y - vb.y) +
                             (D == 3 ? nb.z * (vi.z - vb.z) : 0.f);
            const float m = dn < 0.f ? dn : 0.f;
            const float sc = vb.w * m * w;
            fx -= sc * nb.x;
            fy -= sc * nb.y;
            if (D == 3) fz -= sc * nb.z;
        }
    };
    if constexpr (L == 1) {
        for_each_candidate<D>(k, bcstart, bpos, q.x, q.y, q.z, visit);
    } else if constexpr (D == 2) {
        for_each_candidate2<L>(k, bcstart, bpos, q.x, q.y, sub, [&](int j, double px, double py) {
            visit(j, make_double4(px, py, 0.0, 0.0));
        });
    } else {
        const int cx = cell_coord(q.x, k.cell_lo[0], k.cell_inv, k.cdims[0]);
        const int cy = cell_coord(q.y, k.cell_lo[1], k.cell_inv, k.cdims[1]);
        const int cz = cell_coord(q.z, k.cell_lo[2], k.cell_inv, k.cdims[2]);
        for_each_row<L>(k, bcstart, q, cy, cz, max(cx - 1, 0), min(cx + 1, k.cdims[0] - 1),
                        [&](float, float, int b, int e) {
            for (int j = b + sub; j < e; j += 2 * L) {
                const double4 p0 = bpos[j], p1 = bpos[min(j + L, e - 1)];
                visit(j, p0);
                if (j + L < e) visit(j + L, p1);
            }
        });
    }
}

// Virtual part of the update from global memory: the node box around x_i,
// exact FP64 membership, brick map lookups.  L lanes share a particle, each
// taking every L-th row.
template <int D, int L = 1>
__device__ __forceinline__ void virtual_term_global(const KConst& k, const double4& q,
                                                    const int32_t* slot_of_brick,
                                                    const float* vq, float& fx,
                                                    float& fy, float& fz, int sub = 0) {
    const double qc[3] = {q.x, q.y, q.z};
    const double inv = 1.0 / k.spacing;
    int lo[3] = {0, 0, 0}, cnt[3] = {1, 1, 1};
    bool empty = false;
#pragma unroll
    for (int a = 0; a < D; a++) {
        int l = (int)floor((qc[a] - k.H - k.origin[a]) * inv);
        int u = (int)floor((qc[a] + k.H - k.origin[a]) * inv) + 1;
        l = l < 0 ? 0 : l;
        u = u >= k.ndims[a] ? k.ndims[a] - 1 : u;
        if (u - l + 1 > kBox) u = l + kBox - 1;  // cannot happen for H = 4s
        lo[a] = l;
        cnt[a] = u - l + 1;
        if (cnt[a] <= 0) empty = true;
    }
    if (!empty) {
        // x-axis differences and squares, kept in registers
        double dx2[kBox];
        float dxf[kBox];
#pragma unroll
        for (int c = 0; c < kBox; c++) {
            const double nx = node_coord(k.origin[0], lo[0] + c, k.spacing);
            const double dxs = dsub(nx, q.x);
            dx2[c] = dsq(dxs);
            dxf[c] = (float)dxs;
        }
        const int bx0 = lo[0] >> 3;
        int64_t brow_cached = -1;
        int s3[3] = {-1, -1, -1};
        for (int iz = 0; iz < cnt[2]; iz++) {
            const int cz = lo[2] + iz;
            double dz = 0, dz2 = 0;
            if (D == 3) {
                dz = dsub(node_coord(k.origin[2], cz, k.spacing), q.z);
                dz2 = dsq(dz);
                if (!(dz2 < k.H2)) continue;   // no node of this plane within H
            }
            for (int iy = sub; iy < cnt[1]; iy += L) {
                const int cy = lo[1] + iy;
                const double dy = dsub(node_coord(k.origin[1], cy, k.spacing), q.y);
                const double dy2 = dsq(dy);
                // dx^2 >= 0, so (dx^2 + dy^2) + dz^2 >= dy^2 + dz^2 in FP64
                // as well: a row with dy^2 + dz^2 >= H^2 has no member
                if (!(dadd(dy2, dz2) < k.H2)) continue;
                const int64_t brow = ((int64_t)(D == 3 ? cz >> 3 : 0) * k.bdims[1] +
                                      (cy >> 3)) * k.bdims[0];
                const int lrow = 8 * ((cy & 7) + (D == 3 ? 8 * (cz & 7) : 0));
                constexpr int NB = D == 3 ? 512 : 64;
                // the row's <= 10 nodes lie in at most 3 bricks along x; the
                // slots change only when the row crosses into another brick row
                if (brow != brow_cached) {
                    brow_cached = brow;
#pragma unroll
                    for (int u = 0; u < 3; u++)
                        s3[u] = bx0 + u < k.bdims[0] ? slot_of_brick[brow + bx0 + u] : -1;
                }
                // issue the q loads of every node inside the sphere at once
                float qv[kBox], d2f[kBox];
#pragma unroll
                for (int c = 0; c < kBox; c++) {
                    const double d2 = D == 3 ? dadd(dadd(dx2[c], dy2), dz2)
                                             : dadd(dx2[c], dy2);
                    d2f[c] = (float)d2;
                    const int cx = lo[0] + c;
                    const int u = (cx >> 3) - bx0;
                    const int s = u == 0 ? s3[0] : (u == 1 ? s3[1] : s3[2]);
                    qv[c] = (c < cnt[0] && d2 < k.H2 && s >= 0)
                                ? vq[(int64_t)s * NB + lrow + (cx & 7)] : 0.f;
                }
                const float dyf = (float)dy, dzf = (float)dz;
#pragma unroll
                for (int c = 0; c < kBox; c++) {
                    if (qv[c] == 0.f) continue;
                    // gradK_H(x_i - x_J) = S (x_i - x_J), S = -W'(r) / r; at
                    // r = 0 the difference is zero
                    const float rinv = __builtin_amdgcn_rsqf(d2f[c]);
                    const float r = d2f[c] > 0.f ? d2f[c] * rinv : 0.f;
                    const float S = spline_s(r * k.inv_H, rinv, k.c1H, k.inv_H);
                    const float sc = qv[c] * S;
                    fx -= sc * dxf[c];
                    fy -= sc * dyf;
                    if (D == 3) fz -= sc * dzf;
                }
            }
        }
    }
}

template <int D, int L>
__global__ void __launch_bounds__(256) k_gradient(
    KConst k, int64_t n, const double4* rpos, float4* rvel,
    const int32_t* slot_of_brick, const float* vq, const double4* bpos,
    const float4* bvel, const float4* bnrm, const int32_t* bcstart, SolveGuard guard) {
    const int64_t tid = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    const int64_t i = tid / L;
    const int sub = L > 1 ? (int)(tid % L) : 0;
    if (i >= n || !solve_accepted(guard)) return;   // uniform over the lanes of a particle
    const double4 q = rpos[i];
    float4 vi = rvel[i];
    float fx = 0.f, fy = 0.f, fz = 0.f;
    virtual_term_global<D, L>(k, q, slot_of_brick, vq, fx, fy, fz, sub);
    boundary_term<D, L>(k, q, vi, bpos, bvel, bnrm, bcstart, fx, fy, fz, sub);
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
        fx += __shfl_xor(fx, o, 64);
        fy += __shfl_xor(fy, o, 64);
        if (D == 3) fz += __shfl_xor(fz, o, 64);
    }
    if (sub != 0) return;
    vi.x += fx;
    vi.y += fy;
    if (D == 3) vi.z += fz;
    rvel[i] = vi;
}

// ---- LDS-staged 3D gradient ---------------------------------------------
// Work unit: a block of cells (UnitArgs).  The workgroup stages q = V p of
// the node box that holds every particle's candidates (nodes f-3 .. f+4 per
// axis around f = floor((x - origin) / s): the nodes within H = 4s of x),
// zero off the virtual set and off the lattice, then L lanes sum a
// particle's 8 x 8 x 8 candidates from LDS.  Nodes at or beyond H get S = 0
// from the spline itself; the kernel gradient is continuous and zero at H,
// so the FP32 distance decides membership (a node within rounding of H
// contributes nothing measurable).  A unit whose box exceeds the stage
// (particles far outside their cells) takes the global per-particle path.
// Bound by the candidates' arithmetic where the machine is full (of 164 us at
// 1,012,500 particles about 80; staging 45, the boundary 30), by one
// particle's chain of 350 candidates and 27 boundary cells below.
constexpr int kGradThreads = 256;
constexpr int kGradCap = 7168;   // staged nodes (28 KB: five blocks per CU)
constexpr int kGradBoxBricks = 128;   // bricks a staged box may touch

__device__ __forceinline__ int node_floor(double x, double o, double inv) {
    double f = floor((x - o) * inv);
    f = f < -1.0e9 ? -1.0e9 : (f > 1.0e9 ? 1.0e9 : f);
    return (int)f;
}

// L lanes share a particle: lane `sub` takes x candidates P and 7 - P of every
// row for the pairs P = sub, sub + L, ... of 4 (with 8 lanes: candidate sub).
// CNT (test support): vq holds V_J instead of q_J, and only the number of
// virtual particles whose term enters the sum (V_J > 0, r < H in the FP32
// spline) goes into members[p]; units beyond the stage are left out.
template <int L, bool CNT = false>
__global__ void __launch_bounds__(kGradThreads, 4) k_gradient3s(
    KConst k, UnitArgs ua, int nunits, const double4* rpos, float4* rvel,
    const int32_t* slot_of_brick, const float* vq, const double4* bpos,
    const float4* bvel, const float4* bnrm, const int32_t* bcstart, SolveGuard guard,
    int32_t* members = nullptr) {
    if (!solve_accepted(guard)) return;   // uniform over the block
    __shared__ float s_q[kGradCap];
    __shared__ int s_bslot[kGradBoxBricks];   // slots of the box's bricks
    __shared__ int s_box[6];
    __shared__ int s_walls;   // boundary particles in the cells around the unit
    __shared__ int s_first[kUnitRows];     // first particle of a row - those before
    __shared__ int s_off[kUnitRows + 1];   // particles before row r (rows beyond: all)
    const int unit = ua.units[xcd_remap(blockIdx.x, nunits)];
    const UnitCells uc(k, ua, unit);
    const int t = threadIdx.x;
    if (t < 64) {
        int b = 0, len = 0;
        if (t < uc.rows()) {
            const int64_t row = uc.row(k, t);
            b = ua.cstart[row];
            len = ua.cstart[row + uc.m[0]] - b;
        }
        int end = len;
#pragma unroll
        for (int o = 1; o < kUnitRows; o <<= 1) {
            const int a = __shfl_up(end, o, 64);
            if (t >= o) end += a;
        }
        if (t < kUnitRows) {
            s_first[t] = b - (end - len);
            s_off[t + 1] = end;
        }
        if (t == 0) s_off[0] = 0;
        // the boundary cells that the particles' walks would visit: the
        // unit's cells and those around them, a row per thread
        const int w1 = uc.m[1] + 2, rows = w1 * (uc.m[2] + 2);
        bool walls = false;
        for (int r = t; r < rows; r += 64) {
            const int y = uc.c[1] - 1 + r % w1, z = uc.c[2] - 1 + r / w1;
            if (y < 0 || z < 0 || y >= k.cdims[1] || z >= k.cdims[2]) continue;
            const int64_t row = ((int64_t)z * k.cdims[1] + y) * k.cdims[0];
            const int lo = max(uc.c[0] - 1, 0), hi = min(uc.c[0] + uc.m[0], k.cdims[0] - 1);
            walls |= bcstart[row + hi + 1] > bcstart[row + lo];
        }
        const bool any = __any(walls);
        if (t == 0) s_walls = any;
    } else if (t < 70)
        s_box[t - 64] = t < 67 ? 0x7fffffff : -0x7fffffff;
    __syncthreads();
    const int count = s_off[kUnitRows];
    // particle of task i: the last row with s_off <= i
    auto particle = [&](int i) {
        int r = 0;
#pragma unroll
        for (int o = kUnitRows / 2; o > 0; o >>= 1) r += s_off[r + o] <= i ? o : 0;
        return s_first[r] + i;
    };
    const double inv = 1.0 / k.spacing;
    {
        int mn[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff};
        int mx[3] = {-0x7fffffff, -0x7fffffff, -0x7fffffff};
        for (int i = t; i < count; i += kGradThreads) {
            const double4 q = rpos[particle(i)];
            const double qc[3] = {q.x, q.y, q.z};
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const int f = node_floor(qc[a], k.origin[a], inv);
                mn[a] = min(mn[a], f);
                mx[a] = max(mx[a], f);
            }
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {
            mn[a] = -wave_max<int>(-mn[a]);
            mx[a] = wave_max<int>(mx[a]);
        }
        if ((t & 63) == 0) {
#pragma unroll
            for (int a = 0; a < 3; a++) {
                atomicMin(&s_box[a], mn[a]);
                atomicMax(&s_box[a + 3], mx[a]);
            }
        }
    }
    __syncthreads();
    const int lo0 = s_box[0] - 3, lo1 = s_box[1] - 3, lo2 = s_box[2] - 3;
    const int64_t e0 = (int64_t)s_box[3] - s_box[0] + 8;
    const int64_t e1 = (int64_t)s_box[4] - s_box[1] + 8;
    const int64_t e2 = (int64_t)s_box[5] - s_box[2] + 8;
    // particles far outside their cells: straight from global memory
    auto beyond_stage = [&] {
        if constexpr (CNT) return;
        for (int i = t; i < count; i += kGradThreads) {
            const int p = particle(i);
            const double4 q = rpos[p];
            float4 v = rvel[p];
            float fx = 0.f, fy = 0.f, fz = 0.f;
            virtual_term_global<3>(k, q, slot_of_brick, vq, fx, fy, fz);
            boundary_term<3>(k, q, v, bpos, bvel, bnrm, bcstart, fx, fy, fz);
            v.x += fx;
            v.y += fy;
            v.z += fz;
            rvel[p] = v;
        }
    };
    // (extents one by one first: the product of three may not fit 64 bits)
    const bool over_nodes =
        e0 > kGradCap || e1 > kGradCap || e2 > kGradCap || e0 * e1 * e2 > kGradCap;
    // the bricks the box touches (floor division by 8, also below zero)
    const int bx0 = lo0 >> 3, by0 = lo1 >> 3, bz0 = lo2 >> 3;
    const int nbx = (int)((lo0 + e0 - 1) >> 3) - bx0 + 1;
    const int nby = (int)((lo1 + e1 - 1) >> 3) - by0 + 1;
    const int nbz = (int)((lo2 + e2 - 1) >> 3) - bz0 + 1;
    if (over_nodes || nbx * nby * nbz > kGradBoxBricks) {
        beyond_stage();
        return;
    }
    // their slots (-1 off the virtual set or off the lattice) in one round
    for (int i = t; i < nbx * nby * nbz; i += kGradThreads) {
        const int bx = bx0 + i % nbx, by = by0 + (i / nbx) % nby, bz = bz0 + i / (nbx * nby);
        int sl = -1;
        if (bx >= 0 && by >= 0 && bz >= 0 && bx < k.bdims[0] && by < k.bdims[1] &&
            bz < k.bdims[2])
            sl = slot_of_brick[((int64_t)bz * k.bdims[1] + by) * k.bdims[0] + bx];
        s_bslot[i] = sl;
    }
    __syncthreads();
    const int n0 = (int)e0, n1 = (int)e1;
    {
        // the box's nodes in turn, four loads of a thread issued together (no
        // branch between them: an invalid node reads q[0] and keeps 0); a
        // node's place from its number by two multiplications (m = 2^32 / d
        // rounded up is exact for numbers below 2^16 by divisors below 2^16)
        const int total = n0 * n1 * (int)e2;
        const uint32_t m0 = 0xffffffffu / (uint32_t)n0 + 1u;
        const uint32_t m1 = 0xffffffffu / (uint32_t)n1 + 1u;
        for (int i0 = t; i0 < total; i0 += 4 * kGradThreads) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t i = i0 + u * kGradThreads;
                const uint32_t rw = __umulhi(i, m0), iz = __umulhi(rw, m1);
                const int gx = lo0 + (int)(i - rw * n0), gy = lo1 + (int)(rw - iz * n1),
                          gz = lo2 + (int)iz;
                const bool in = (int)i < total && gx >= 0 && gy >= 0 && gz >= 0 &&
                                gx < k.ndims[0] && gy < k.ndims[1] && gz < k.ndims[2];
                const int bi = in ? (((gz >> 3) - bz0) * nby + ((gy >> 3) - by0)) * nbx +
                                        ((gx >> 3) - bx0)
                                  : 0;
                const int sl = s_bslot[bi];
                const bool ok = in && sl >= 0;
                const int64_t g = ok ? (int64_t)sl * 512 + ((gz & 7) << 6) + ((gy & 7) << 3) +
                                           (gx & 7)
                                     : 0;
                const float q = vq[g];
                v[u] = ok ? q : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (i0 + u * kGradThreads < total) s_q[i0 + u * kGradThreads] = v[u];
        }
    }
    __syncthreads();
    // spline of H (S = -W'(r) / r, q = r / H): with a = max(1 - q, 0) and
    // b = max(1 - 2 q, 0), S = c1 (a^2 - b^2) / r on every piece:
    // c1 (2 - 3 q) / H for q < 1/2, c1 (1 - q)^2 / r up to q = 1, and 0
    // beyond (a = b = 0).  The offsets d are taken in units of H, so that
    // with w = |d|^2 = q^2 and u = 1 / q (one rsq), a = 1 - w u and
    // b = 2 a - 1 (both clamped to [0, 1]: a = 0 beyond q = 1 gives b = 0),
    // and S d = c1 (a^2 - b^2) u (d / H): 9 VALU and the rsq per candidate.
    // The clamps fold into the fmas; c1 is applied once per particle.
    const float c1 = k.c1H;
    const double iHd = 1.0 / k.H;
    constexpr int kC = 8 / L;   // x candidates of a lane
    const int sub = L > 1 ? t % L : 0;
    for (int i = t / L; i < count; i += kGradThreads / L) {   // uniform over the lanes of a particle
        const int p = particle(i);
        const double4 q = rpos[p];
        const float4 vi = rvel[p];
        float fx = 0.f, fy = 0.f, fz = 0.f;
        int32_t nterms = 0;
        {
            const int f0 = node_floor(q.x, k.origin[0], inv);
            const int f1 = node_floor(q.y, k.origin[1], inv);
            const int f2 = node_floor(q.z, k.origin[2], inv);
            // x candidate of this lane's c-th: the pairs (P, 7 - P) in turn
            auto cand = [&](int c) {
                if constexpr (L == 8) return sub;
                const int P = sub + (c >> 1) * L;
                return (c & 1) ? 7 - P : P;
            };
            float dxf[kC], dx2[kC];   // x offsets of the lane's candidates, in units of H
#pragma unroll
            for (int c = 0; c < kC; c++) {
                dxf[c] = (float)(dsub(node_coord(k.origin[0], f0 - 3 + cand(c), k.spacing), q.x) *
                                 iHd);
                // + 1e-30: rsq stays finite at a coincident node (whose
                // direction factors are all zero)
                dx2[c] = dxf[c] * dxf[c] + 1e-30f;
            }
            // y and z offsets of candidate 0; candidate c adds c s (FP32, units of H)
            const float dy0 = (float)(dsub(node_coord(k.origin[1], f1 - 3, k.spacing), q.y) * iHd);
            const float dz0 = (float)(dsub(node_coord(k.origin[2], f2 - 3, k.spacing), q.z) * iHd);
            const float sf = (float)(k.spacing * iHd);
            const float* base = s_q + ((f2 - 3 - lo2) * n1 + (f1 - 3 - lo1)) * n0 + (f0 - 3 - lo0);
            // Candidate c of row (cy, cz) is node f - 3 + c: its offset from x
            // lies in (c - 4, c - 3] s.  With d(c) = the smallest |offset| of
            // index c (3, 2, 1, 0, 0, 1, 2, 3) a row holds members only if
            // d(cy)^2 + d(cz)^2 < 16, and only at |c - 3.5| < sqrt(R2) + 0.5,
            // R2 = 16 - d(cy)^2 - d(cz)^2: all 8 for R2 >= 11, c = 1..6 for
            // R2 = 6..8, c = 2..5 for R2 = 3 (the uniform bounds below; the
            // first pairs of a lane go when no lane's candidate is in).  The
            // whole 8 x 8 row nest is unrolled: the bounds are constants, and
            // the LDS reads are scheduled ahead of the candidates that use them.
#pragma unroll
            for (int cz = 0; cz < 8; cz++) {
                const float dzfc = fmaf((float)cz, sf, dz0), dz2c = dzfc * dzfc;
                const int dzm = cz <= 3 ? 3 - cz : cz - 4;
                const float* plane = base + cz * n1 * n0;
#pragma unroll
                for (int cy = 0; cy < 8; cy++) {
                    const int dym = cy <= 3 ? 3 - cy : cy - 4;
                    const int R2 = 16 - dym * dym - dzm * dzm;
                    if (R2 <= 0) continue;   // uniform: no member in the row
                    const int cut = R2 >= 11 ? 0 : (R2 >= 6 ? 1 : 2);
                    const float dyc = fmaf((float)cy, sf, dy0);
                    const float dyz = fmaf(dyc, dyc, dz2c);
                    if (!(dyz < 1.f)) continue;   // this particle: none within H
                    const float* row = plane + cy * n0;
                    float sx = 0.f, ss = 0.f;
#pragma unroll
                    for (int c = 0; c < kC; c++) {
                        // the largest pair any lane has here: (c / 2) L + L - 1
                        if (L < 8 && (c >> 1) * L + L - 1 < cut) continue;   // uniform
                        const float qv = row[cand(c)];
                        const float w = dx2[c] + dyz;
                        const float u = __builtin_amdgcn_rsqf(w);
                        const float a = __builtin_amdgcn_fmed3f(fmaf(-w, u, 1.f), 0.f, 1.f);
                        const float b = __builtin_amdgcn_fmed3f(fmaf(a, 2.f, -1.f), 0.f, 1.f);
                        const float sc = qv * u * fmaf(a, a, -(b * b));
                        sx = fmaf(sc, dxf[c], sx);
                        ss += sc;
                        if constexpr (CNT) nterms += (a > 0.f) & (qv > 0.f);
                    }
                    fx -= sx;
                    fy -= ss * dyc;
                    fz -= ss * dzfc;
                }
            }
            fx *= c1;
            fy *= c1;
            fz *= c1;
        }
        if constexpr (CNT) {
#pragma unroll
            for (int o = 1; o < L; o <<= 1) nterms += __shfl_xor(nterms, o, 64);
            if (sub == 0) members[p] = nterms;
            continue;
        }
        if (s_walls) boundary_term<3, L>(k, q, vi, bpos, bvel, bnrm, bcstart, fx, fy, fz, sub);
#pragma unroll
        for (int o = 1; o < L; o <<= 1) {
            fx += __shfl_xor(fx, o, 64);
            fy += __shfl_xor(fy, o, 64);
            fz += __shfl_xor(fz, o, 64);
        }
        if (sub != 0) continue;
        float4 v = vi;
        v.x += fx;
        v.y += fy;
        v.z += fz;
        rvel[p] = v;
    }
}

template <int D>
__global__ void __launch_bounds__(256) k_advect(int64_t n, double4* pos,
                                                float4* vel, double dt,
                                                double g) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double4 p = pos[i];
    float4 v = vel[i];
    p.x += (double)v.x * dt;
    p.y += (double)v.y * dt;
    if (D == 3) p.z += (double)v.z * dt;
    v.y -= (float)(g * dt);
    pos[i] = p;
    vel[i] = v;
}

// ---- neighbour query (tests) ---------------------------------------------
template <int D>
__global__ void __launch_bounds__(128) k_query(
    KConst k, int which, int64_t nq, const double* qs, const double4* pos,
    const int32_t* cstart, const int32_t* ids, const int32_t* slot_of_brick,
    const float* vvol, const int32_t* rank, const int64_t* offsets,
    int64_t* out_count, int64_t* out_idx) {
    const int64_t t = (int64_t)blockIdx.x * 128 + threadIdx.x;
    if (t >= nq) return;
    const double qx = qs[D * t], qy = qs[D * t + 1], qz = D == 3 ? qs[D * t + 2] : 0.0;
    int64_t cnt = 0;
    const int64_t base = offsets ? offsets[t] : 0;
    if (which < 2) {
        for_each_candidate<D>(k, cstart, pos, qx, qy, qz, [&](int j, const double4& pj) {
            const double d2 = D == 3 ? sq_dist3(pj.x, pj.y, pj.z, qx, qy, qz)
                                     : sq_dist2(pj.x, pj.y, qx, qy);
            if (d2 < k.h2) {
                if (out_idx) out_idx[base + cnt] = ids[j];
                cnt++;
            }
        });
    } else {
        const double qc[3] = {qx, qy, qz};
        const double inv = 1.0 / k.spacing;
        int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
        for (int a = 0; a < D; a++) {
            int l = (int)floor((qc[a] - k.H - k.origin[a]) * inv);
            int u = (int)floor((qc[a] + k.H - k.origin[a]) * inv) + 1;
            lo[a] = l < 0 ? 0 : l;
            hi[a] = u >= k.ndims[a] ? k.ndims[a] - 1 : u;
        }
        const int NB = D == 3 ? 512 : 64;
        for (int cz = lo[2]; cz <= hi[2]; cz++)
            for (int cy = lo[1]; cy <= hi[1]; cy++)
                for (int cx = lo[0]; cx <= hi[0]; cx++) {
                    const double nx = node_coord(k.origin[0], cx, k.spacing);
                    const double ny = node_coord(k.origin[1], cy, k.spacing);
                    const double nz = D == 3 ? node_coord(k.origin[2], cz, k.spacing) : 0.0;
                    const double d2 = D == 3 ? sq_dist3(nx, ny, nz, qx, qy, qz)
                                             : sq_dist2(nx, ny, qx, qy);
                    if (!(d2 < k.H2)) continue;
                    const int64_t b = ((int64_t)(D == 3 ? cz >> 3 : 0) * k.bdims[1] +
                                       (cy >> 3)) * k.bdims[0] + (cx >> 3);
                    const int s = slot_of_brick[b];
                    if (s < 0) continue;
                    const int64_t g = (int64_t)s * NB + (cx & 7) + 8 * (cy & 7) +
                                      (D == 3 ? 64 * (cz & 7) : 0);
                    if (!(vvol[g] > 0.f)) continue;
                    if (out_idx) out_idx[base + cnt] = rank[g];
                    cnt++;
                }
    }
    if (out_count) out_count[t] = cnt;
}

}  // namespace

// Lanes per particle and cells of a work unit by the number of particles: the
// fewest lanes and the largest unit (least staged per particle: 77, 22 and 10
// nodes) that fill the machine.  us of one launch that updates, 2x2x2 cells
// with 8 lanes, 4x2x2 with 4, 4x4x4 with 1 (before: spans of 25 cells of one
// row, 36 nodes staged per particle, one lane each):
//   500 particles 19, 24, 42 (45)     32,000 23, 24, 41 (44)
//   64,000        34, 29, 43 (50)    100,000 41, 34, 48 (61)
// and by the launches of a run that update and those that do not, 4x2x2 and 4x4x4:
//   212,503 24, 27 (33)    300,000 23, 23 (31)    1,012,500 122, 102 (146)
struct UnitRule {
    int lanes, u[3];
};
static UnitRule unit_rule(int64_t n) {
    if (n <= 32000) return {8, {2, 2, 2}};
    if (n <= 250000) return {4, {4, 2, 2}};
    return {1, {4, 4, 4}};
}

// The rule's unit, shrunk until its node box fits the stage; false if not even
// one cell's does.
static bool unit_shape(const KConst& k, int64_t n, int u[3]) {
    const UnitRule rule = unit_rule(n);
    for (int a = 0; a < 3; a++) u[a] = rule.u[a];
    const double ratio = k.cell_size / k.spacing;
    auto nodes = [&](int m) { return (int64_t)std::floor(m * ratio) + 9; };
    while (nodes(u[0]) * nodes(u[1]) * nodes(u[2]) > kGradCap) {
        int* largest = std::max_element(u, u + 3);
        if (--*largest < 1) return false;
    }
    return true;
}

int gradient_setup(vps_context* c) {
    c->grad_staged = false;
    if (c->dim != 3) return VPS_OK;
    const KConst& k = c->k;
    // candidates f-3 .. f+4 per axis assume H = 4 s
    if (!(std::fabs(k.H - 4.0 * k.spacing) <= 1e-12 * k.H)) return VPS_OK;
    int u[3];
    if (!unit_shape(k, 0, u)) return VPS_OK;
    int64_t total = 1;   // of the smallest units
    for (int a = 0; a < 3; a++) total *= (k.cdims[a] + u[a] - 1) / u[a];
    VPS_TRY(dalloc(c, c->grad_units, (size_t)total));
    c->grad_staged = true;
    return VPS_OK;
}

UnitArgs gradient_units(vps_context* c, bool append) {
    if (!append || !c->grad_staged) return UnitArgs{};
    UnitArgs a{};
    (void)unit_shape(c->k, c->n, a.u);
    a.total = 1;
    for (int d = 0; d < 3; d++) {
        a.nu[d] = (c->k.cdims[d] + a.u[d] - 1) / a.u[d];
        a.total *= a.nu[d];
    }
    a.cstart = c->cell_start.p;
    a.units = c->grad_units.p;
    a.count = (int32_t*)(c->counters.p + 2);
    c->grad_shape = a;
    return a;
}

// The staged gradient on the units of the last generation; CNT: its terms
// instead (q the volumes), into members.
template <bool CNT>
static void gradient3s(vps_context* c, const float* q, SolveGuard g, int32_t* members) {
    if (c->grad_nunits == 0) return;
    auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)c->grad_nunits), dim3(kGradThreads), 0, c->stream,
                           c->k, c->grad_shape, (int)c->grad_nunits, c->rpos[c->cur].p,
                           c->rvel[c->cur].p, c->brick_slot[c->which].p, q, c->bpos.p, c->bvel.p,
                           c->bnrm.p, c->bcell_start.p, g, members);
    };
    const int lanes = unit_rule(c->n).lanes;
    if (lanes == 8) run(k_gradient3s<8, CNT>);
    else if (lanes == 4) run(k_gradient3s<4, CNT>);
    else run(k_gradient3s<1, CNT>);
}

// Terms of the staged gradient's virtual walk per real particle (test
// support, sorted order; -1 stays where a unit exceeds the stage).
int gradient_member_counts(vps_context* c, int32_t* members) {
    if (c->dim != 3 || !c->grad_staged || c->nslots == 0) return VPS_ERR_INVALID_ARG;
    gradient3s<true>(c, c->vvol.p, SolveGuard{}, members);
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

int pressure_gradient(vps_context* c, SolveGuard g) {
    const int64_t n = c->n;
    const int s = c->cur;
    const int w = c->which;
    if (c->dim == 3 && c->grad_staged) {
        gradient3s<false>(c, c->vq.p, g, nullptr);
    } else {
        auto run = [&](auto kern, int lanes) {
            hipLaunchKernelGGL(kern, dim3(blocks(n * lanes, 256)), dim3(256), 0, c->stream, c->k,
                               n, c->rpos[s].p, c->rvel[s].p, c->brick_slot[w].p, c->vq.p,
                               c->bpos.p, c->bvel.p, c->bnrm.p, c->bcell_start.p, g);
        };
        if (c->dim == 3) run(k_gradient<3, 1>, 1);
        else if (walk_lanes2(n) == 4) run(k_gradient<2, 4>, 4);
        else run(k_gradient<2, 1>, 1);
    }
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

int advect(vps_context* c, double dt, double g) {
    const int s = c->cur;
    if (c->dim == 3)
        hipLaunchKernelGGL(k_advect<3>, dim3(blocks(c->n, 256)), dim3(256), 0,
                           c->stream, c->n, c->rpos[s].p, c->rvel[s].p, dt, g);
    else
        hipLaunchKernelGGL(k_advect<2>, dim3(blocks(c->n, 256)), dim3(256), 0,
                           c->stream, c->n, c->rpos[s].p, c->rvel[s].p, dt, g);
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

int query_neighbors(vps_context* c, int which, int64_t nq, const double* q,
                    int64_t* offsets, int64_t* idx, int64_t cap,
                    int64_t* needed) {
    const int D = c->dim;
    DBuf<double> dq;
    DBuf<int64_t> dcnt, doff, didx;
    VPS_TRY(dalloc(c, dq, (size_t)(nq * D)));
    VPS_TRY(dalloc(c, dcnt, (size_t)nq));
    VPS_TRY(dalloc(c, doff, (size_t)nq + 1));
    VPS_HIP(c, hipMemcpyAsync(dq.p, q, (size_t)nq * D * 8, hipMemcpyHostToDevice,
                              c->stream));
    const double4* pos = which == 0 ? c->rpos[c->cur].p : c->bpos.p;
    const int32_t* cs = which == 0 ? c->cell_start.p : c->bcell_start.p;
    const int32_t* ids = which == 0 ? c->rid[c->cur].p : c->bid.p;
    const int32_t* sob = c->brick_slot[c->which].p;
    auto run = [&](const int64_t* off, int64_t* cntp, int64_t* ix) {
        if (D == 3)
            hipLaunchKernelGGL(k_query<3>, dim3(blocks(nq, 128)), dim3(128), 0,
                               c->stream, c->k, which, nq, dq.p, pos, cs, ids,
                               sob, c->vvol.p, c->vrank.p, off, cntp, ix);
        else
            hipLaunchKernelGGL(k_query<2>, dim3(blocks(nq, 128)), dim3(128), 0,
                               c->stream, c->k, which, nq, dq.p, pos, cs, ids,
                               sob, c->vvol.p, c->vrank.p, off, cntp, ix);
    };
    run(nullptr, dcnt.p, nullptr);
    std::vector<int64_t> cnt((size_t)nq);
    VPS_HIP(c, hipMemcpyAsync(cnt.data(), dcnt.p, (size_t)nq * 8,
                              hipMemcpyDeviceToHost, c->stream));
    VPS_HIP(c, hipStreamSynchronize(c->stream));
    offsets[0] = 0;
    for (int64_t i = 0; i < nq; i++) offsets[i + 1] = offsets[i] + cnt[(size_t)i];
    const int64_t total = offsets[nq];
    if (needed) *needed = total;
    int rc = VPS_OK;
    if (!idx) {
        // size query: offsets and *needed only
    } else if (total > cap) {
        rc = VPS_ERR_INVALID_ARG;
        c->err = "vps_query_neighbors: capacity too small";
    } else if (total > 0) {
        VPS_TRY(dalloc(c, didx, (size_t)total));
        VPS_HIP(c, hipMemcpyAsync(doff.p, offsets, (size_t)(nq + 1) * 8,
                                  hipMemcpyHostToDevice, c->stream));
        run(doff.p, nullptr, didx.p);
        VPS_HIP(c, hipMemcpyAsync(idx, didx.p, (size_t)total * 8,
                                  hipMemcpyDeviceToHost, c->stream));
        VPS_HIP(c, hipStreamSynchronize(c->stream));
        for (int64_t i = 0; i < nq; i++) {
            int64_t* b = idx + offsets[i];
            int64_t* e = idx + offsets[i + 1];
            for (int64_t* u = b + 1; u < e; u++) {
                const int64_t v = *u;
                int64_t* w = u - 1;
                while (w >= b && *w > v) {
                    w[1] = w[0];
                    w--;
                }
                w[1] = v;
            }
        }
    }
    VPS_HIP(c, hipStreamSynchronize(c->stream));
    dfree(dq);
    dfree(dcnt);
    dfree(doff);
    dfree(didx);
    return rc;
}

}  // namespace vps
