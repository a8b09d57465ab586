// vps_dem.hip -- GPU step of the DEM sand grains and their coupling to the
// water projection as moving boundary particles.
//
// Replaces DEMParticleSand<Dim>::advance (Cores/Physics/DEMParticleSand.cpp:
// 89-152) with the contact model of DEMParticle<Dim>
// (Cores/Structures/DEMParticle.cpp:13-134):
//   moveParticles        x += v dt
//   applyPressureForce   v += dt * sum_{j: |x_j - x_i| < 2r} F(x_j - x_i, v_j - v_i)
//                          + sum_{b: |x_b - x_i| < 4r} (F_norm + F_tang)
//   applyExternalForces  v.y -= g dt
// with the soft-sphere contact F (penetration 2r - |d| > 0, n = d / max(|d|,
// 1e-4 r), normal K_n pen n, tangential -K_t v_t limited to tan(phi) |F_n|,
// F = -F_n - F_t) and the wall force F_norm = -V_b min(n_b.(v_i - v_b), 0)
// n_b W_4r, F_tang = -K_t (dv - (n_b.dv) n_b) limited to tan(phi) |F_norm|
// (used as is when |F_tang| <= 1e-6).  The grains are the context's real
// particles (kernel radius h = 4r: grain-grain pairs are the h-walk's
// candidates within 2r), the walls its boundary particles.
//
// The capillary bridge force (DEMParticle.cpp:97-125) acts only for gaps
// 1e-6 < |d| - 2r < d_rupture, i.e. beyond the 2r neighbourhood the reference
// searches, so it never contributes there and is not evaluated.  The
// reference updates velocities in place while other threads read them (an
// OpenMP race); here every force uses the velocities at the start of the pass.
#include <algorithm>
#include <cmath>
#include <utility>

#include "vps_internal.h"

namespace vps {
namespace {

inline unsigned blocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <int D>
__global__ void __launch_bounds__(256) k_dem_move(int64_t n, double4* pos,
                                                  const float4* vel, double dt,
                                                  int32_t* near_count) {
#pragma clang fp contract(off)   // x + v dt rounded twice, as the reference
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i == 0) *near_count = 0;   // the list of k_dem_forces is rebuilt
    if (i >= n) return;
    double4 p = pos[i];
    const float4 v = vel[i];
    p.x += (double)v.x * dt;
    p.y += (double)v.y * dt;
    if (D == 3) p.z += (double)v.z * dt;
    pos[i] = p;
}

struct DemK {
    float k_norm, k_tang, tan_phi;
    float two_r;         // contact distance 2r
    float min_dist;      // 1e-4 r
    double two_r2;       // (2r)^2, the searcher's strict radius
    double reach;        // 2r with a margin, for the cells to visit
    float dt, g_dt;
};

__device__ __forceinline__ float fmul_rounded(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

// Whether any wall particle lies in the cells around q (those that the wall
// walk visits).
template <int D>
__device__ __forceinline__ bool near_walls(const KConst& k, const int32_t* bcstart,
                                           const double4& q) {
    int c[3] = {0, 0, 0};
    const double qa[3] = {q.x, q.y, q.z};
#pragma unroll
    for (int a = 0; a < D; a++) c[a] = cell_coord(qa[a], k.cell_lo[a], k.cell_inv, k.cdims[a]);
    const int x0 = max(c[0] - 1, 0), x1 = min(c[0] + 1, k.cdims[0] - 1);
    // nine rows (2D: three), clamped to the border (a row twice does no harm):
    // constant bounds, so that all loads are issued together
    int found = 0;
#pragma unroll
    for (int r = 0; r < (D == 3 ? 9 : 3); r++) {
        const int y = min(max(c[1] + r % 3 - 1, 0), k.cdims[1] - 1);
        const int z = D == 3 ? min(max(c[2] + r / 3 - 1, 0), k.cdims[2] - 1) : 0;
        const int64_t row = ((int64_t)z * k.cdims[1] + y) * k.cdims[0];
        found |= bcstart[row + x1 + 1] - bcstart[row + x0];
    }
    return found != 0;
}

// The (sorted) grains next to a wall, listed and flagged.  The list's order is
// arbitrary; a grain's sums are its own.
template <int D>
__global__ void __launch_bounds__(256) k_dem_prepare(KConst k, int64_t n, const double4* pos,
                                                     const int32_t* bcstart, int32_t* near, int32_t* near_list,
                                                     int32_t* near_count) {
    const int64_t i = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    bool is_near = false;
    if (i < n) {
        is_near = near_walls<D>(k, bcstart, pos[i]);
        near[i] = is_near ? 1 : 0;
    }
    // one atomic per block with any (one per wave, all on one address, bound
    // this kernel: 39 us against 28 at 1,012,500 grains)
    __shared__ int s_cnt[4], s_base;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const unsigned long long m = __ballot(is_near);
    if (lane == 0) s_cnt[wv] = __popcll(m);
    __syncthreads();
    const int total = (s_cnt[0] + s_cnt[1]) + (s_cnt[2] + s_cnt[3]);
    if (total == 0) return;   // uniform over the block
    if (threadIdx.x == 0) s_base = atomicAdd(near_count, total);
    __syncthreads();
    int at = s_base + __popcll(m & ((1ull << lane) - 1ull));
    for (int w = 0; w < wv; w++) at += s_cnt[w];
    if (is_near) near_list[at] = (int32_t)i;
}

// One grain's velocity after the pass, contacts and (WALLS) walls.
template <int D, bool WALLS>
__device__ __forceinline__ void dem_grain(
    const KConst& k, const DemK& dk, int64_t i, const double4* pos, const float4* ofs,
    const float4* vel, const int32_t* cstart, const double4* bpos, const float4* bofs,
    const float4* bvel, const float4* bnrm, const int32_t* bcstart, float4* vout) {
    const double4 q = pos[i];
    const float4 vi = vel[i];
    float cx = 0.f, cy = 0.f, cz = 0.f;   // sum of contact forces
    auto contact = [&](int j, const double4& pj, const float4& vj) {
        const double d2 = D == 3 ? sq_dist3(pj.x, pj.y, pj.z, q.x, q.y, q.z)
                                 : sq_dist2(pj.x, pj.y, q.x, q.y);
        if (!(d2 < dk.two_r2) || j == i) return;   // self: zero force
        // d = x_j - x_i, v = v_j - v_i
        const float dx = (float)(pj.x - q.x), dy = (float)(pj.y - q.y),
                    dz = D == 3 ? (float)(pj.z - q.z) : 0.f;
        float dist = sqrtf((float)d2);
        const float pen = dk.two_r - dist;
        if (!(pen > 0.f)) return;
        if (dist <= dk.min_dist) dist = dk.min_dist;
        const float inv = 1.f / dist;
        const float nx = dx * inv, ny = dy * inv, nz = dz * inv;
        const float wx = vj.x - vi.x, wy = vj.y - vi.y, wz = D == 3 ? vj.z - vi.z : 0.f;
        const float vn = wx * nx + wy * ny + wz * nz;
        const float tx = wx - vn * nx, ty = wy - vn * ny, tz = wz - vn * nz;
        const float fn = dk.k_norm * pen;   // |normal force|
        float sx = -dk.k_tang * tx, sy = -dk.k_tang * ty, sz = -dk.k_tang * tz;
        const float max_fs = fabsf(fn) * dk.tan_phi;
        const float fs = sqrtf(sx * sx + sy * sy + sz * sz);
        if (fs > max_fs) {
            const float s = max_fs / fs;
            sx *= s;
            sy *= s;
            sz *= s;
        }
        cx += -fn * nx - sx;
        cy += -fn * ny - sy;
        cz += -fn * nz - sz;
    };
    auto contact_at = [&](int j, const double4& pj) { contact(j, pj, vel[j]); };
    // the FP32 distances below are usable: no clamping of this grain into a
    // border cell from far outside
    int cc[3] = {0, 0, 0};
    bool qfar = false;
    const double qa[3] = {q.x, q.y, q.z};
    if constexpr (D == 3) {
        const float far = 2.f * (float)k.cell_size;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            cc[a] = cell_coord(qa[a], k.cell_lo[a], k.cell_inv, k.cdims[a]);
            qfar |= !(fabsf((float)(qa[a] - cell_corner(k, a, cc[a]))) <= far);
        }
    }
    if constexpr (D == 3) {
        // The FP32 distance from the cell offsets keeps the candidates within
        // 2r (margin 1e-4 of (2r)^2, far above its error; particles far from
        // their cell always), then the FP64 test and the force for those
        // only, in candidate order.  The cells are 4r wide and contacts reach
        // 2r, so the ball of 2r touches two cells an axis: 8 of the 27 around
        // the grain, about 64 candidates instead of 216.  (cell_coord is
        // monotone, its clamp to the border cells included: a particle within
        // 2r along an axis lies between the cells of the ball's ends; the
        // margin of `reach` covers the rounding of q +- 2r.)
        int lo[3], hi[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            lo[a] = cell_coord(qa[a] - dk.reach, k.cell_lo[a], k.cell_inv, k.cdims[a]);
            hi[a] = cell_coord(qa[a] + dk.reach, k.cell_lo[a], k.cell_inv, k.cdims[a]);
        }
        const float tx0 = (float)(q.x - cell_corner(k, 0, lo[0]));
        const float x0w = (float)(lo[0] + 1), csf = (float)k.cell_size;
        const float thr = (float)(dk.two_r2 * 1.0001);
        // candidate j of a row: the offset's w is its cell x + 1
        auto close = [&](const float4& p, float ty, float tz) {
            const float dx = fmaf(x0w - fabsf(p.w), csf, tx0) - p.x, dy = ty - p.y,
                        dz = tz - p.z;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            return !(d2 >= thr) || p.w < 0.f || qfar;
        };
        // The usual case, up to two rows of cells along y and z with up to 32
        // candidates each: the bounds of the four rows and then the contacts
        // of all four are loaded ahead of their use (the waves wait for
        // memory most of the time), and the contacts of a grain run as one
        // sequence, not row by row (the lanes' counts differ per row).
        const int ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
        int b[4], e[4];
        bool fits = ny <= 2 && nz <= 2;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int y = min(lo[1] + (r & 1), hi[1]), z = min(lo[2] + (r >> 1), hi[2]);
            const int64_t row = ((int64_t)z * k.cdims[1] + y) * k.cdims[0];
            b[r] = cstart[row + lo[0]];
            e[r] = cstart[row + hi[0] + 1];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if ((r & 1) >= ny || (r >> 1) >= nz) e[r] = b[r];
            fits = fits && e[r] - b[r] <= 32;
        }
        if (fits) {
            uint32_t m[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                m[r] = 0u;
                const float ty = (float)(q.y - cell_corner(k, 1, lo[1] + (r & 1)));
                const float tz = (float)(q.z - cell_corner(k, 2, lo[2] + (r >> 1)));
                for (int j0 = b[r]; j0 < e[r]; j0 += 4) {
                    float4 pv[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) pv[u] = ofs[min(j0 + u, e[r] - 1)];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int j = j0 + u;
                        const bool in = close(pv[u], ty, tz) && j < e[r] && j != (int)i;
                        m[r] |= (uint32_t)in << (j - b[r] & 31);
                    }
                }
            }
            auto next = [&]() -> int {   // the next contact in candidate order, -1: none
                int j = -1;
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (j < 0 && m[r]) {
                        j = b[r] + __builtin_ctz(m[r]);
                        m[r] &= m[r] - 1u;
                    }
                return j;
            };
            int j = next();
            double4 pj{};
            float4 vj{};
            if (j >= 0) {
                pj = pos[j];
                vj = vel[j];
            }
            while (j >= 0) {
                const int jn = next();
                const int jl = jn >= 0 ? jn : j;
                const double4 pn = pos[jl];
                const float4 vn = vel[jl];
                contact(j, pj, vj);
                j = jn;
                pj = pn;
                vj = vn;
            }
        } else {
            for (int z = lo[2]; z <= hi[2]; z++)
                for (int y = lo[1]; y <= hi[1]; y++) {
                    const float ty = (float)(q.y - cell_corner(k, 1, y));
                    const float tz = (float)(q.z - cell_corner(k, 2, z));
                    const int64_t row = ((int64_t)z * k.cdims[1] + y) * k.cdims[0];
                    const int je = cstart[row + hi[0] + 1];
                    for (int j = cstart[row + lo[0]]; j < je; j++)
                        if (close(ofs[j], ty, tz)) contact_at(j, pos[j]);
                }
        }
    } else {
        for_each_candidate<D>(k, cstart, pos, q.x, q.y, q.z, contact_at);
    }
    // (rounded here, with and without walls: not fused into the sum below)
    float fx = fmul_rounded(cx, dk.dt), fy = fmul_rounded(cy, dk.dt), fz = fmul_rounded(cz, dk.dt);
    // walls within 4r
    auto wall = [&](int j, const double4& pj) {
        const double d2 = D == 3 ? sq_dist3(pj.x, pj.y, pj.z, q.x, q.y, q.z)
                                 : sq_dist2(pj.x, pj.y, q.x, q.y);
        if (!(d2 < k.h2)) return;
        const KW kh = kernel_f32(d2, k.h2, k.hf, k.inv_h, k.c0h, k.c1h);
        const float4 vb = bvel[j];   // (v_b, V_b)
        const float4 nb = bnrm[j];   // (n_b, rho_b)
        const float ux = vi.x - vb.x, uy = vi.y - vb.y, uz = D == 3 ? vi.z - vb.z : 0.f;
        const float un = nb.x * ux + nb.y * uy + (D == 3 ? nb.z * uz : 0.f);
        const float m = un < 0.f ? un : 0.f;
        const float an = -vb.w * m * kh.w;
        const float Fx = an * nb.x, Fy = an * nb.y, Fz = D == 3 ? an * nb.z : 0.f;
        float Tx = -dk.k_tang * (ux - un * nb.x), Ty = -dk.k_tang * (uy - un * nb.y),
              Tz = D == 3 ? -dk.k_tang * (uz - un * nb.z) : 0.f;
        const float tn = sqrtf(Tx * Tx + Ty * Ty + Tz * Tz);
        if (tn > 1e-6f) {
            const float lim = sqrtf(Fx * Fx + Fy * Fy + Fz * Fz) * dk.tan_phi;
            if (!(lim > tn)) {
                const float s = lim / tn;
                Tx *= s;
                Ty *= s;
                Tz *= s;
            }
        }
        fx += Fx + Tx;
        fy += Fy + Ty;
        fz += Fz + Tz;
    };
    if constexpr (WALLS && D == 3) {
        // the FP32 distance from the boundary's cell offsets keeps the
        // candidates below the band around h^2, the FP64 test decides
        const int x0 = cc[0] > 0 ? cc[0] - 1 : 0;
        const int x1 = cc[0] + 1 < k.cdims[0] ? cc[0] + 1 : k.cdims[0] - 1;
        const int ylo = cc[1] > 0 ? cc[1] - 1 : 0;
        const int yhi = cc[1] + 1 < k.cdims[1] ? cc[1] + 1 : k.cdims[1] - 1;
        const int zlo = cc[2] > 0 ? cc[2] - 1 : 0;
        const int zhi = cc[2] + 1 < k.cdims[2] ? cc[2] + 1 : k.cdims[2] - 1;
        float tx0 = (float)(q.x - cell_corner(k, 0, x0));
        float tx1 = (float)(q.x - cell_corner(k, 0, x0 + 1));
        float tx2 = (float)(q.x - cell_corner(k, 0, x0 + 2));
        asm volatile("" : "+v"(tx0), "+v"(tx1), "+v"(tx2));
        for (int z = zlo; z <= zhi; z++) {
            const float tz = (float)(q.z - cell_corner(k, 2, z));
            for (int y = ylo; y <= yhi; y++) {
                const int64_t row = ((int64_t)z * k.cdims[1] + y) * k.cdims[0];
                const int b = bcstart[row + x0], e = bcstart[row + x1 + 1];
                if (b >= e) continue;
                const float ty = (float)(q.y - cell_corner(k, 1, y));
                const int b1 = x0 + 1 <= x1 ? bcstart[row + x0 + 1] : e;
                const int b2 = x0 + 2 <= x1 ? bcstart[row + x0 + 2] : e;
                for (int c0 = b; c0 < e; c0 += 32) {
                    const int c1 = min(c0 + 32, e);
                    uint32_t m = 0u;
                    for (int j0 = c0; j0 < c1; j0 += 4) {
                        float4 pv[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) pv[u] = bofs[min(j0 + u, c1 - 1)];
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            const int j = j0 + u;
                            const float tx = j < b1 ? tx0 : (j < b2 ? tx1 : tx2);
                            const float dx = tx - pv[u].x, dy = ty - pv[u].y, dz = tz - pv[u].z;
                            const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                            const bool in =
                                j < c1 && (!(d2 >= k.h2f_hi) || pv[u].w < 0.f || qfar);
                            m |= (uint32_t)in << (j - c0 & 31);
                        }
                    }
                    while (m) {
                        const int j = c0 + __builtin_ctz(m);
                        m &= m - 1u;
                        wall(j, bpos[j]);
                    }
                }
            }
        }
    } else if constexpr (WALLS) {
        for_each_candidate<D>(k, bcstart, bpos, q.x, q.y, q.z, wall);
    }
    float4 v = vi;
    v.x += fx;
    v.y += fy;
    if (D == 3) v.z += fz;
    v.y -= dk.g_dt;
    vout[i] = v;
}

// A wall neighbour costs several times a contact (FP64 test, spline, two
// roots), and only the grains next to a wall have any; but with the grains in
// cell order a quarter of the waves hold one, and would run the wall walk for
// all their lanes.  So the first `nlist` blocks take the listed grains, whole
// waves of them, and the others the rest, contacts only; the list goes first
// because its waves are the longest.  1,012,500 grains: 163 us and 28 for
// k_dem_prepare, against 287 and 8 for one kernel over the 27 cells with both
// walks; the block order (neighbouring grains on one L2) takes the L2 misses
// from 5.4M to 1.0M.
template <int D>
__global__ void __launch_bounds__(256) k_dem_forces(
    KConst k, DemK dk, int64_t n, int nlist, const double4* pos, const float4* ofs,
    const float4* vel, const int32_t* cstart, const double4* bpos, const float4* bofs,
    const float4* bvel, const float4* bnrm, const int32_t* bcstart, const int32_t* near,
    const int32_t* near_list, const int32_t* near_count, float4* vout) {
    if ((int)blockIdx.x < nlist) {   // uniform over the block
        const int m = *near_count;
        for (int j = blockIdx.x * 256 + threadIdx.x; j < m; j += nlist * 256)
            dem_grain<D, true>(k, dk, near_list[j], pos, ofs, vel, cstart, bpos, bofs, bvel, bnrm,
                               bcstart, vout);
        return;
    }
    const int64_t i =
        (int64_t)xcd_remap(blockIdx.x - nlist, gridDim.x - nlist) * 256 + threadIdx.x;
    if (i >= n || near[i]) return;
    dem_grain<D, false>(k, dk, i, pos, ofs, vel, cstart, nullptr, nullptr, nullptr, nullptr,
                        nullptr, vout);
}

// Grain positions / velocities as moving boundary particles of a water
// context: the walls first (FP64 AoS from the host copy), then the grains in
// their caller order (boundary index = wall count + grain index) with a zero
// normal (the water side takes the unit vector from the grain to the fluid
// particle).
template <int D>
__global__ void __launch_bounds__(256) k_pack_grains(int64_t n, const double4* gpos,
                                                     const float4* gvel,
                                                     const int32_t* gid, int64_t off,
                                                     double* x, double* nrm, double* v) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double4 p = gpos[i];
    const float4 u = gvel[i];
    const int64_t b = off + gid[i];
    const double pc[3] = {p.x, p.y, p.z};
    const double uc[3] = {(double)u.x, (double)u.y, (double)u.z};
    for (int a = 0; a < D; a++) {
        x[b * D + a] = pc[a];
        nrm[b * D + a] = 0.0;
        v[b * D + a] = uc[a];
    }
}

}  // namespace

int dem_step(vps_context* c, double dt, double g, const vps_dem_params* dp) {
    const int D = c->dim;
    const int64_t n = c->n;
    int s = c->cur;
    int32_t* near_count = (int32_t*)(c->counters.p + 13);
    if (D == 3)
        hipLaunchKernelGGL(k_dem_move<3>, dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                           n, c->rpos[s].p, c->rvel[s].p, dt, near_count);
    else
        hipLaunchKernelGGL(k_dem_move<2>, dim3(blocks(n, 256)), dim3(256), 0, c->stream,
                           n, c->rpos[s].p, c->rvel[s].p, dt, near_count);
    VPS_TRY(cells_sort_real(c));
    s = c->cur;
    if (c->vel_next.n < (size_t)n) {
        dfree(c->vel_next);
        VPS_TRY(dalloc(c, c->vel_next, (size_t)n));
    }
    const double r = c->p.particle_radius;
    DemK dk;
    dk.k_norm = (float)(dp->young * r);                  // K_norm = Young r
    dk.k_tang = (float)(dp->young * r * dp->poisson);    // K_tang = K_norm Poisson
    dk.tan_phi = (float)std::tan(dp->friction_angle);
    dk.two_r = (float)(2 * r);
    dk.min_dist = (float)(1e-4 * r);
    dk.two_r2 = (2 * r) * (2 * r);
    dk.reach = 2 * r * (1 + 1e-6);
    dk.dt = (float)dt;
    dk.g_dt = (float)(g * dt);
    const double4* bp = c->nb ? c->bpos.p : nullptr;
    const int32_t* bcs = c->nb ? c->bcell_start.p : c->cell_start.p;
    // with no walls the boundary walk must see empty cells
    if (c->nb == 0) {
        if (!c->bcell_start.p) VPS_TRY(dalloc(c, c->bcell_start, (size_t)c->ncells + 1));
        VPS_HIP(c, hipMemsetAsync(c->bcell_start.p, 0, ((size_t)c->ncells + 1) * 4,
                                  c->stream));
        bcs = c->bcell_start.p;
    }
    // sort scratch, free until the next sort
    int32_t* near_list = c->perm.p;
    int32_t* near = c->slot_of.p;
    const unsigned nb = blocks(n, 256);
    // (a multiple of 8, so that the other blocks keep their XCDs)
    const unsigned nlist = c->nb > 0 ? std::min(512u, (nb + 7) & ~7u) : 0;
    auto forces = [&](auto prepare, auto kern) {
        hipLaunchKernelGGL(prepare, dim3(nb), dim3(256), 0, c->stream, c->k, n, c->rpos[s].p, bcs,
                           near, near_list, near_count);
        hipLaunchKernelGGL(kern, dim3(nlist + nb), dim3(256), 0, c->stream, c->k, dk, n,
                           (int)nlist, c->rpos[s].p, c->rofs.p, c->rvel[s].p, c->cell_start.p, bp,
                           c->bofs.p, c->bvel.p, c->bnrm.p, bcs, near, near_list, near_count,
                           c->vel_next.p);
    };
    if (D == 3) forces(k_dem_prepare<3>, k_dem_forces<3>);
    else forces(k_dem_prepare<2>, k_dem_forces<2>);
    VPS_HIP(c, hipGetLastError());
    std::swap(c->rvel[s], c->vel_next);   // every grain's velocity was written
    c->generated = false;
    return VPS_OK;
}

// Boundary of the water context = its walls + the grains of the DEM context.
int couple_grains(vps_context* w, vps_context* g) {
    const int D = w->dim;
    const int64_t nw = (int64_t)(w->host_bx.size() / D);
    const int64_t ng = g->n;
    const int64_t nt = nw + ng;
    // staging (x, n, v) kept across calls; the walls are copied once
    const size_t need = (size_t)(3 * nt * D);
    if (w->couple_stage.n != need || w->couple_walls != nw) {
        dfree(w->couple_stage);
        VPS_TRY(dalloc(w, w->couple_stage, need));
        w->couple_walls = -1;
    }
    double* dx = w->couple_stage.p;
    double* dn = dx + nt * D;
    double* dv = dn + nt * D;
    if (w->couple_walls != nw && nw > 0) {
        VPS_HIP(w, hipMemcpyAsync(dx, w->host_bx.data(), (size_t)nw * D * 8,
                                  hipMemcpyHostToDevice, w->stream));
        VPS_HIP(w, hipMemcpyAsync(dn, w->host_bn.data(), (size_t)nw * D * 8,
                                  hipMemcpyHostToDevice, w->stream));
        VPS_HIP(w, hipMemcpyAsync(dv, w->host_bv.data(), (size_t)nw * D * 8,
                                  hipMemcpyHostToDevice, w->stream));
    }
    w->couple_walls = nw;
    // the grains are read on the water stream once the DEM stream is done
    VPS_HIP(g, hipStreamSynchronize(g->stream));
    if (ng > 0) {
        const int s = g->cur;
        if (D == 3)
            hipLaunchKernelGGL(k_pack_grains<3>, dim3(blocks(ng, 256)), dim3(256), 0,
                               w->stream, ng, g->rpos[s].p, g->rvel[s].p, g->rid[s].p,
                               nw, dx, dn, dv);
        else
            hipLaunchKernelGGL(k_pack_grains<2>, dim3(blocks(ng, 256)), dim3(256), 0,
                               w->stream, ng, g->rpos[s].p, g->rvel[s].p, g->rid[s].p,
                               nw, dx, dn, dv);
        VPS_HIP(w, hipGetLastError());
    }
    VPS_TRY(upload_boundary_device(w, nt, dx, dn, dv));
    VPS_HIP(w, hipStreamSynchronize(w->stream));
    return VPS_OK;
}

}  // namespace vps

using namespace vps;

extern "C" {

int vps_dem_step(vps_context* c, double dt, double gravity,
                 const vps_dem_params* dp) {
    if (!c || !dp) return VPS_ERR_INVALID_ARG;
    if (c->n == 0) {
        c->err = "dem step: no grains (vps_set_particles)";
        return VPS_ERR_STATE;
    }
    if (!std::isfinite(dt) || !std::isfinite(gravity) || !(dt >= 0) ||
        !std::isfinite(dp->young) || !std::isfinite(dp->poisson) ||
        !std::isfinite(dp->friction_angle) || !(dp->young > 0)) {
        c->err = "dem step: dt >= 0, finite gravity and parameters, young > 0";
        return VPS_ERR_INVALID_ARG;
    }
    VPS_TRY(dem_step(c, dt, gravity, dp));
    VPS_HIP(c, hipStreamSynchronize(c->stream));
    return VPS_OK;
}

int vps_couple_grains(vps_context* water, vps_context* grains) {
    if (!water || !grains) return VPS_ERR_INVALID_ARG;
    if (water->dim != grains->dim) {
        water->err = "couple grains: dimensions differ";
        return VPS_ERR_INVALID_ARG;
    }
    if (water->device != grains->device) {
        water->err = "couple grains: contexts on different devices";
        return VPS_ERR_INVALID_ARG;
    }
    return couple_grains(water, grains);
}

}  // extern "C"
