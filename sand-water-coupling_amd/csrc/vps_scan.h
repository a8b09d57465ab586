// vps_scan.h -- one-launch device-wide exclusive scan of int32 counts.
//
// Used for the cell counting sort (cell_start), brick compaction (slots), the
// column order and the lattice-bitmask ranks.  Every tile publishes its total
// and then its inclusive prefix in one 64-bit status word; a tile forms its
// own prefix by looking back over the words of the tiles before it (Merrill
// and Garland, single-pass parallel prefix scan with decoupled look-back), the
// whole block reading 1,024 words at a time: a read of another XCD's word goes
// to memory, so the rounds count.
// All integer, so the result is exact and independent of scheduling.
//
// What bounds it: launches (a step runs four scans; tile sums, a scan of the
// sums and a second pass were three launches each, 4 us and a gap apiece), and
// at millions of cells the passes over memory (the input was read twice).  1M
// cells: 10.8 us against 14 and two gaps.
//
// Tiles take their numbers from a ticket, so a tile that waits only waits for
// tiles that are running or done; the last one resets the ticket.  The status
// words carry the epoch of their launch, so they are never cleared.
#pragma once

#include "vps_internal.h"

namespace vps {

constexpr int kScanBS = 256;
constexpr int kScanWindow = 1024;   // tiles of one look-back

__device__ __forceinline__ int scan_block_exclusive(int v, int* total) {
    __shared__ int swave[kScanBS / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int x = v;   // inclusive wave scan
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) swave[wv] = x;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kScanBS / 64; i++) {
        if (i < wv) off += swave[i];
        tot += swave[i];
    }
    *total = tot;
    return off + x - v;
}

// Status word of a tile: epoch << 34 | flag << 32 | value, flag 1 the tile's
// own total, 2 the prefix including it.
__device__ __forceinline__ uint64_t scan_word(uint32_t epoch, uint32_t flag, int value) {
    return ((uint64_t)epoch << 34) | ((uint64_t)flag << 32) | (uint32_t)value;
}

// load(i) gives element i; store(i, v, pre) takes it with its exclusive
// prefix, once per element, after every element of the tile was loaded (so
// the output may alias the input).  kWide functors also take four elements
// from a multiple of 4 on (16-byte aligned).  IPT consecutive elements per
// thread.
template <int IPT, typename Load, typename Store>
__global__ void __launch_bounds__(kScanBS) k_scan(Load load, Store store, int64_t n, int ntiles,
                                                  uint64_t* status, uint32_t epoch,
                                                  uint32_t* ticket, int32_t* total) {
    __shared__ int s_tile;
    int tile = 0;
    if (ntiles > 1) {   // uniform
        if (threadIdx.x == 0) s_tile = (int)atomicAdd(ticket, 1u);
        __syncthreads();
        tile = s_tile;
    }
    const int64_t base = ((int64_t)tile * kScanBS + threadIdx.x) * IPT;
    // full threads load and store 16 bytes at a time where the functors can (a
    // thread's elements lie side by side, so 4-byte accesses of a wave spread
    // over as many lines as it has lanes: 20 us against 10.8 at 1M cells)
    const bool full = base + IPT <= n;
    int v[IPT], s = 0;
    bool loaded = false;
    if constexpr (Load::kWide && IPT % 4 == 0)
        if (full) {
            loaded = true;
#pragma unroll
            for (int k = 0; k < IPT; k += 4) {
                const int4 w = load.four(base + k);
                v[k] = w.x;
                v[k + 1] = w.y;
                v[k + 2] = w.z;
                v[k + 3] = w.w;
            }
        }
    if (!loaded) {
#pragma unroll
        for (int k = 0; k < IPT; k++) v[k] = base + k < n ? load(base + k) : 0;
    }
#pragma unroll
    for (int k = 0; k < IPT; k++) s += v[k];
    int tot;
    int run = scan_block_exclusive(s, &tot);
    if (ntiles > 1) {
        __shared__ int s_nearest[kScanBS / 64], s_sum[kScanBS / 64];
        const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
        if (t == 0)
            __hip_atomic_store(&status[tile], scan_word(epoch, tile == 0 ? 2 : 1, tot),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int prefix = 0;
        bool found = false;
        for (int end = tile; end > 0 && !found; end -= kScanWindow) {   // uniform
            uint64_t w[kScanWindow / kScanBS];
            int nearest = -1;   // the last tile of the window with its prefix known
#pragma unroll
            for (int q = 0; q < kScanWindow / kScanBS; q++) {
                const int j = end - 1 - (t + kScanBS * q);
                w[q] = 0;
                if (j >= 0) {
                    do   // every tile before this one has started, and publishes
                        w[q] = __hip_atomic_load(&status[j], __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
                    while ((uint32_t)(w[q] >> 34) != epoch);
                    if ((w[q] >> 32 & 3) == 2) nearest = max(nearest, j);
                }
            }
            nearest = wave_max(nearest);
            if (lane == 0) s_nearest[wv] = nearest;
            __syncthreads();
            nearest = max(max(s_nearest[0], s_nearest[1]), max(s_nearest[2], s_nearest[3]));
            int sum = 0;
#pragma unroll
            for (int q = 0; q < kScanWindow / kScanBS; q++) {
                const int j = end - 1 - (t + kScanBS * q);
                if (j >= 0 && j >= nearest) sum += (int)(uint32_t)w[q];
            }
            sum = wave_sum(sum);
            if (lane == 0) s_sum[wv] = sum;
            __syncthreads();
            prefix += (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
            found = nearest >= 0;
        }
        if (t == 0) {
            if (tile > 0)
                __hip_atomic_store(&status[tile], scan_word(epoch, 2, prefix + tot),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (tile == ntiles - 1) *ticket = 0;   // every ticket has been taken
        }
        run += prefix;
        tot += prefix;
    }
    if (total && tile == ntiles - 1 && threadIdx.x == 0) *total = tot;
    int pre[IPT];
#pragma unroll
    for (int k = 0; k < IPT; k++) {
        pre[k] = run;
        run += v[k];
    }
    if constexpr (Store::kWide && IPT % 4 == 0)
        if (full) {
#pragma unroll
            for (int k = 0; k < IPT; k += 4)
                store.four(base + k, make_int4(pre[k], pre[k + 1], pre[k + 2], pre[k + 3]));
            return;
        }
#pragma unroll
    for (int k = 0; k < IPT; k++)
        if (base + k < n) store(base + k, v[k], pre[k]);
}

// Workspace of a scan of `tiles` tiles and the epoch of the next launch.
int scan_workspace(vps_context* c, int64_t tiles, uint64_t** status, uint32_t** ticket,
                   uint32_t* epoch);

template <int IPT, typename Load, typename Store>
int scan_launch_as(vps_context* c, Load load, Store store, int64_t n, int32_t* total_dev) {
    const int64_t nt = (n + kScanBS * IPT - 1) / (kScanBS * IPT);
    uint64_t* status;
    uint32_t *ticket, epoch;
    VPS_TRY(scan_workspace(c, nt, &status, &ticket, &epoch));
    hipLaunchKernelGGL((k_scan<IPT, Load, Store>), dim3((unsigned)nt), dim3(kScanBS), 0, c->stream,
                       load, store, n, (int)nt, status, epoch, ticket, total_dev);
    VPS_HIP(c, hipGetLastError());
    return VPS_OK;
}

// Elements per thread: few for the small scans (more waves, one tile up to
// 2,048), more where the tickets, taken one by one, would add up.
template <typename Load, typename Store>
int scan_launch(vps_context* c, Load load, Store store, int64_t n, int32_t* total_dev) {
    if (n > 4096 * 1024) return scan_launch_as<32>(c, load, store, n, total_dev);
    if (n > 512 * 1024) return scan_launch_as<16>(c, load, store, n, total_dev);
    return scan_launch_as<8>(c, load, store, n, total_dev);
}

}  // namespace vps
