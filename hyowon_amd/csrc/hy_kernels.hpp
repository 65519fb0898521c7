// HIP kernels of the MI355X particle-mesh gravity step (gfx950, wave64).
//
// Stage map (reference hot path, file:line relative to the reference tree):
//   k_bucket_key / k_scan_*, k_cap_* / k_scatter  stable bucketing of particles that
//        feeds the deterministic deposit (reference x-plane counting sort,
//        src/mesh/mass_assignment_workspace.inc:264-374, generalised to
//        tile buckets; determinism restored by k_deposit's index sort).
//   k_deposit    CIC deposit + density source, summation order per cell equal
//        to src/mesh/mass_assignment_deposit.inc:193-240 (bin X with weight
//        1-f, then bin X-1 with weight f, particles in index order, oy outer,
//        oz inner), density contrast as src/gravity/pm_solver.cpp:700-759.
//   k_tl_*       (hy_fft_passes.hpp) r2c / Green / c2r Poisson solve (src/mesh/fft_backend.cpp,
//        src/mesh/green_function.cpp:165-241).
//   k_gather_kdk, k_slot_force  centered-gradient CIC gather
//        (src/mesh/mass_assignment_gradient.cpp:117-206); k_gather_kdk with the K2 kick,
//        the next K1 kick and the periodic drift
//        (include/cosmo_nbody/time/particle_update.hpp:20-116).
#pragma once

#include "hy_device.hpp"
#include <type_traits>
#include "hy_fft.hpp"

namespace hy {

// ===========================================================================
// Bucketing
// ===========================================================================

// Deposit bucket of a base cell: tile (edge T) and boundary class
// (bit2/1/0: last cell of the tile along x/y/z).
__device__ __forceinline__ uint32_t bucket_of(int bx, int by, int bz, const Geom& g) {
    // T = 16 (every mesh divisible by 16) takes shifts instead of divisions
    const int tx = g.T == 16 ? bx >> 4 : bx / g.T;
    const int ty = g.T == 16 ? by >> 4 : by / g.T;
    const int tz = g.T == 16 ? bz >> 4 : bz / g.T;
    const uint32_t cls = ((uint32_t)(bx - tx * g.T == g.T - 1) << 2)
                       | ((uint32_t)(by - ty * g.T == g.T - 1) << 1)
                       | (uint32_t)(bz - tz * g.T == g.T - 1);
    return (((uint32_t)tx * g.nT + ty) * g.nT + tz) * 8u + cls;
}

// Cell of a deposit record inside its tile: (lx*T + ly)*T + lz.
__device__ __forceinline__ uint32_t record_cell(int bx, int by, int bz, const Geom& g) {
    const int T = g.T;
    const int lx = T == 16 ? bx & 15 : bx % T, ly = T == 16 ? by & 15 : by % T, lz = T == 16 ? bz & 15 : bz % T;
    return (uint32_t)((lx * T + ly) * T + lz);
}

// Wave-aggregated integer atomic: lanes with equal keys reserve consecutive
// slots.  Groups are found with ballots first; then every group leader issues
// its atomic in the same instruction, so a wave pays one atomic round trip.
// Returns this lane's rank (slot) within its bucket; groups: the wave's number of
// distinct keys.
__device__ __forceinline__ uint32_t aggregated_rank(uint32_t* counts, uint32_t key, bool valid, uint32_t& groups) {
    const uint32_t lane = lane_id();
    uint64_t remaining = __ballot(valid);
    groups = 0;
    int my_leader = (int)lane;
    uint64_t my_mask = 0;
    while (remaining) {
        const int leader = __ffsll((unsigned long long)remaining) - 1;
        const uint32_t lead_key = (uint32_t)__builtin_amdgcn_readlane((int)key, leader);  // uniform lane: a scalar read
        const uint64_t mask = __ballot(valid && key == lead_key) & remaining;
        if ((mask >> lane) & 1ull) {
            my_leader = leader;
            my_mask = mask;
        }
        remaining &= ~mask;
        ++groups;
    }
    uint32_t old = 0;
    if (valid && (int)lane == my_leader) old = atomicAdd(&counts[key], (uint32_t)__popcll(my_mask));
    const uint32_t base = __shfl(old, my_leader);
    return base + (uint32_t)__popcll(my_mask & ((1ull << lane) - 1ull));
}

// mode 0: deposit buckets; mode 1: reference x-plane bins (key = base x).
// shift: positions are routed as x - shift (the interlacing partner of the
// power-spectrum estimator; 0 otherwise, where x - 0 is x exactly).
// PROBE: counts how well the order of the particles keeps to the buckets.
struct OrderProbe {
    uint32_t* groups;   // distinct keys of the probed waves, added up (null: not probed)
    uint32_t* host;     // their sum in pinned host memory, written by the scatter
    uint32_t stride;    // the first wave of every stride-th workgroup is probed
    uint32_t limit;     // groups above it: the order does not keep to the buckets
};

template <bool PROBE>
__global__ void k_bucket_key(uint64_t n, const double* __restrict__ x, const double* __restrict__ y,
                             const double* __restrict__ z, Geom g, int mode,
                             uint32_t* __restrict__ keys, uint32_t* __restrict__ ranks,
                             uint32_t* __restrict__ counts, uint32_t* __restrict__ err, double shift,
                             OrderProbe probe) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = p < n;
    uint32_t key = 0;
    bool ok = false;
    if (in) {
        int bx, by = 0, bz = 0;
        double f;
        ok = cic_axis(x[p] - shift, g, bx, f);
        if (mode == 0) ok = ok && cic_axis(y[p] - shift, g, by, f) && cic_axis(z[p] - shift, g, bz, f);
        if (ok) key = mode == 0 ? box_of(p, g) * buckets_per_box(g) + bucket_of(bx, by, bz, g) : (uint32_t)bx;
        else atomicOr(err, ERR_POSITION_NONFINITE);
    }
    uint32_t groups;
    const uint32_t rank = aggregated_rank(counts, key, in && ok, groups);
    if constexpr (PROBE) {
        if (blockIdx.x % probe.stride == 0 && threadIdx.x == 0) atomicAdd(probe.groups, groups);
    }
    if (in && !ok) key = 0xffffffffu;
    if (in) {
        keys[p] = key;
        ranks[p] = rank;
    }
}

// Exclusive scan of counts[0..nb) into offsets[0..nb], three launches.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh, uint32_t& total) {
    // Hillis-Steele over 256 threads in LDS (deterministic integer sums).
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int off = 1; off < SCAN_THREADS; off <<= 1) {
        const uint32_t add = t >= off ? sh[t - off] : 0u;
        __syncthreads();
        sh[t] += add;
        __syncthreads();
    }
    total = sh[SCAN_THREADS - 1];
    const uint32_t incl = sh[t];
    __syncthreads();
    return incl - v;
}

__global__ void k_scan_reduce(const uint32_t* __restrict__ counts, uint64_t nb,
                              uint32_t* __restrict__ block_sums) {
    __shared__ uint32_t sh[SCAN_THREADS];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        const uint64_t j = base + (uint64_t)i * SCAN_THREADS + threadIdx.x;
        if (j < nb) s += counts[j];
    }
    uint32_t total;
    (void)block_exclusive_scan(s, sh, total);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

__global__ void k_scan_blocks(uint32_t* __restrict__ block_sums, uint32_t nblocks,
                              uint32_t* __restrict__ grand_total) {
    __shared__ uint32_t sh[SCAN_THREADS];
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nblocks; base += SCAN_THREADS) {
        const uint32_t j = base + threadIdx.x;
        const uint32_t v = j < nblocks ? block_sums[j] : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan(v, sh, total);
        if (j < nblocks) block_sums[j] = ex + carry;
        carry += total;
    }
    if (threadIdx.x == 0) *grand_total = carry;
}

__global__ void k_scan_apply(const uint32_t* __restrict__ counts, uint64_t nb,
                             const uint32_t* __restrict__ block_sums,
                             const uint32_t* __restrict__ grand_total,
                             uint32_t* __restrict__ offsets) {
    __shared__ uint32_t sh[SCAN_THREADS];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        v[i] = (base + i < nb) ? counts[base + i] : 0u;
        s += v[i];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan(s, sh, total) + block_sums[blockIdx.x];
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        if (base + i < nb) offsets[base + i] = run;
        run += v[i];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) offsets[nb] = *grand_total;
}

__global__ void k_scatter(uint64_t n, const uint32_t* __restrict__ keys,
                          const uint32_t* __restrict__ ranks, const uint32_t* __restrict__ offsets,
                          uint32_t* __restrict__ order) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) {
        const uint32_t k = keys[p];
        if (k != 0xffffffffu) order[offsets[k] + ranks[p]] = (uint32_t)p;
    }
}

// Deposit record in bucket order: tile-local base cell (lx*T+ly)*T+lz and the
// three CIC fractions (computed in binary64, stored in binary32).
struct DepRecord {
    uint32_t cell;
    float fx, fy, fz;
};

// ---------------------------------------------------------------------------
// Capacity layout of carried deposit records (binary32, uniform mass).
//
// A fused step that drifts the particles writes each particle's deposit
// record for the next step straight into a slot of its bucket: bucket b owns
// cap(c_b) = c_b + c_b/8 + CAP_SLACK slots, c_b its count at this step (the
// particles move little per step), and a record whose rank within its bucket
// reaches the capacity goes to an overflow list instead.  Before the next
// deposit one three-channel scan over the final counts gives
//   ch 0: the exclusive prefix of the counts (dense offsets; its total is the
//         routing identity's grand total),
//   ch 1: the prefix of the overflow counts max(0, c_b - cap_b) of the layout
//         the records were written in (overflow records are placed after the
//         capacity slots, bucket by bucket),
//   ch 2: the prefix of cap(c_b), the layout the next step's records go to.
// The binary32 deposit sums integers, so the order of a bucket's records
// (the ranks come from atomics) leaves every cell sum unchanged.
// ---------------------------------------------------------------------------
constexpr uint32_t CAP_SLACK = 4;

__device__ __forceinline__ uint32_t capacity_of(uint32_t count) { return count + (count >> 3) + CAP_SLACK; }

struct CapScan {
    const uint32_t* counts;  // records per bucket
    uint64_t nb;             // buckets over all boxes
    const uint32_t* cur;     // nb+1 prefix of the layout the records were written in (null: no overflow)
    uint32_t* dense;         // out: nb+1 prefix of the counts (or null)
    uint32_t* ovf_start;     // out: nb+1 prefix of the overflow counts (when cur)
    uint32_t* capn;          // out: nb+1 prefix of the next layout's capacities (or null)
    uint32_t* block_sums;    // 3 per scan block
    uint32_t* grand_total;   // out: total count
};

__device__ __forceinline__ void cap_channels(const CapScan& s, uint64_t b, uint32_t v[3]) {
    const uint32_t c = s.counts[b];
    v[0] = c;
    if (s.cur) {
        const uint32_t cap = s.cur[b + 1] - s.cur[b];
        v[1] = c > cap ? c - cap : 0u;
    } else {
        v[1] = 0u;
    }
    v[2] = capacity_of(c);
}

__global__ void k_cap_reduce(CapScan s) {
    __shared__ uint32_t sh[SCAN_THREADS];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
    uint32_t acc[3] = {0u, 0u, 0u};
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        const uint64_t j = base + (uint64_t)i * SCAN_THREADS + threadIdx.x;
        if (j < s.nb) {
            uint32_t v[3];
            cap_channels(s, j, v);
            for (int ch = 0; ch < 3; ++ch) acc[ch] += v[ch];
        }
    }
    for (int ch = 0; ch < 3; ++ch) {
        uint32_t total;
        (void)block_exclusive_scan(acc[ch], sh, total);
        if (threadIdx.x == 0) s.block_sums[3 * blockIdx.x + ch] = total;
    }
}

// One workgroup: exclusive scan of each channel's block sums; the totals go
// to index nb of each output and the count total to grand_total.
__global__ void k_cap_blocks(CapScan s, uint32_t nblocks) {
    __shared__ uint32_t sh[SCAN_THREADS];
    for (int ch = 0; ch < 3; ++ch) {
        uint32_t carry = 0;
        for (uint32_t base = 0; base < nblocks; base += SCAN_THREADS) {
            const uint32_t j = base + threadIdx.x;
            const uint32_t v = j < nblocks ? s.block_sums[3 * j + ch] : 0u;
            uint32_t total;
            const uint32_t ex = block_exclusive_scan(v, sh, total);
            if (j < nblocks) s.block_sums[3 * j + ch] = ex + carry;
            carry += total;
        }
        if (threadIdx.x == 0) {
            if (ch == 0) {
                *s.grand_total = carry;
                if (s.dense) s.dense[s.nb] = carry;
            } else if (ch == 1 && s.cur) {
                s.ovf_start[s.nb] = carry;
            } else if (ch == 2 && s.capn) {
                s.capn[s.nb] = carry;
            }
        }
    }
}

__global__ void k_cap_apply(CapScan s) {
    __shared__ uint32_t sh[SCAN_THREADS];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS][3];
    uint32_t acc[3] = {0u, 0u, 0u};
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        if (base + i < s.nb) {
            cap_channels(s, base + i, v[i]);
        } else {
            v[i][0] = v[i][1] = v[i][2] = 0u;
        }
        for (int ch = 0; ch < 3; ++ch) acc[ch] += v[i][ch];
    }
    uint32_t run[3];
    for (int ch = 0; ch < 3; ++ch) {
        uint32_t total;
        run[ch] = block_exclusive_scan(acc[ch], sh, total) + s.block_sums[3 * blockIdx.x + ch];
    }
    uint32_t* out[3] = {s.dense, s.cur ? s.ovf_start : nullptr, s.capn};
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        if (base + i < s.nb) {
            for (int ch = 0; ch < 3; ++ch)
                if (out[ch]) out[ch][base + i] = run[ch];
        }
        for (int ch = 0; ch < 3; ++ch) run[ch] += v[i][ch];
    }
}

// The whole scan in one workgroup, for up to SMALL_SCAN_MAX buckets (a 192^3 mesh
// has 13824): one launch and no round trip through block_sums; 16 -> 6 us for
// the 4096 buckets of a 128^3 mesh, even (15 us) at 13824, where it still saves
// two launches.  Each thread owns a run of buckets.
constexpr int SMALL_SCAN_THREADS = 1024;
constexpr uint64_t SMALL_SCAN_MAX = 16 * SMALL_SCAN_THREADS;

__global__ void __launch_bounds__(SMALL_SCAN_THREADS) k_cap_small(CapScan s) {
    __shared__ uint32_t wave_sum[3][SMALL_SCAN_THREADS / 64];
    const uint32_t per = (uint32_t)((s.nb + SMALL_SCAN_THREADS - 1) / SMALL_SCAN_THREADS);
    const uint32_t b0 = threadIdx.x * per;
    const uint32_t b1 = b0 + per < s.nb ? b0 + per : (uint32_t)s.nb;
    uint32_t acc[3] = {0u, 0u, 0u};
    for (uint32_t b = b0; b < b1; ++b) {
        uint32_t v[3];
        cap_channels(s, b, v);
        for (int ch = 0; ch < 3; ++ch) acc[ch] += v[ch];
    }
    uint32_t incl[3];
    const uint32_t lane = lane_id(), wave = threadIdx.x / 64;
    for (int ch = 0; ch < 3; ++ch) {
        incl[ch] = acc[ch];
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl[ch], d);
            if (lane >= d) incl[ch] += o;
        }
        if (lane == 63) wave_sum[ch][wave] = incl[ch];
    }
    __syncthreads();
    uint32_t run[3];
    for (int ch = 0; ch < 3; ++ch) {
        run[ch] = incl[ch] - acc[ch];
        for (uint32_t w = 0; w < wave; ++w) run[ch] += wave_sum[ch][w];
    }
    uint32_t* out[3] = {s.dense, s.cur ? s.ovf_start : nullptr, s.capn};
    for (uint32_t b = b0; b < b1; ++b) {
        uint32_t v[3];
        cap_channels(s, b, v);
        for (int ch = 0; ch < 3; ++ch) {
            if (out[ch]) out[ch][b] = run[ch];
            run[ch] += v[ch];
        }
    }
    if (threadIdx.x == SMALL_SCAN_THREADS - 1) {  // the totals
        *s.grand_total = run[0];
        for (int ch = 0; ch < 3; ++ch)
            if (out[ch]) out[ch][s.nb] = run[ch];
    }
}

__global__ void k_copy_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Overflow records of the carried layout cur: entry i holds its bucket, its
// rank and its record; it goes to cur[nb] + ovf_start[b] + (rank - cap_b), so each
// bucket's overflow records follow the capacity slots contiguously.  Grid
// stride up to the device count the gather left.
__global__ void k_place_overflow(const uint32_t* __restrict__ ovf_count, const uint32_t* __restrict__ ovf_key,
                                 const uint32_t* __restrict__ ovf_rank, const DepRecord* __restrict__ ovf_rec,
                                 const uint32_t* __restrict__ cur, const uint32_t* __restrict__ ovf_start,
                                 uint64_t nb, DepRecord* __restrict__ rec) {
    const uint32_t total = *ovf_count;
    const uint32_t base = cur[nb];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const uint32_t b = ovf_key[i];
        const uint32_t cap = cur[b + 1] - cur[b];
        rec[base + ovf_start[b] + (ovf_rank[i] - cap)] = ovf_rec[i];
    }
}

// Binary64 deposit record: tile-local base cell (12 bits) and above it the tile
// in its box, the particle index (the reference's per-cell summation order is
// by index) and the binary64 fractions; after the slot-order force kernel, the
// force instead of the fractions.
constexpr int REC_CELL_BITS = 12;  // tile edges up to 16; tiles of a 1024^3 box: 18 bits

struct DepRecord64 {
    uint32_t cell;
    uint32_t index;
    double fx, fy, fz;
};

// What the slot-order force kernels need beside a particle's deposit record:
// the lower corner's weights (float)(1 - f), formed from the binary64
// fractions, and the particle's tile (box-major).  After the force kernel the
// record holds the force instead (w = g).
struct ForceRecord {
    float wx, wy, wz;
    uint32_t tile;
};

// Scatter into bucket order, writing the particle index and its deposit
// record (and, where force is set and a probe has not found the particles in
// order, its force record at the same slot).  The bucket is recomputed from the current position and must equal
// the stored key (keys carried over from the previous step are checked here; a
// mismatch also sets stale, a word of pinned host memory, where given).
// R = DepRecord (binary32 fractions, masses / mass unit) or DepRecord64
// (binary64 fractions and particle index, masses as given).
template <typename R, typename MT>
__global__ void k_scatter_records(uint64_t n, const double* __restrict__ x, const double* __restrict__ y,
                                  const double* __restrict__ z, const double* __restrict__ masses,
                                  double inv_mass_unit, Geom g, const uint32_t* __restrict__ keys,
                                  const uint32_t* __restrict__ ranks, const uint32_t* __restrict__ offsets,
                                  uint32_t* __restrict__ order, R* __restrict__ rec,
                                  MT* __restrict__ rec_mass, uint32_t* __restrict__ err, double shift,
                                  ForceRecord* __restrict__ force, uint32_t* __restrict__ stale,
                                  OrderProbe probe) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    if (probe.groups) {
        const uint32_t groups = *probe.groups;
        if (p == 0) __hip_atomic_store(probe.host, groups, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (groups <= probe.limit) force = nullptr;
    }
    const uint32_t k = keys[p];
    int bx, by, bz;
    double fx, fy, fz;
    // The coordinate loads stay behind the short-circuit checks: issued
    // together (cic_axes), the three streams measured 8% slower here.
    const bool ok = cic_axis(x[p] - shift, g, bx, fx) && cic_axis(y[p] - shift, g, by, fy) &&
                    cic_axis(z[p] - shift, g, bz, fz);
    if (!ok) {
        atomicOr(err, ERR_POSITION_NONFINITE);
        return;
    }
    if (k == 0xffffffffu || box_of(p, g) * buckets_per_box(g) + bucket_of(bx, by, bz, g) != k) {
        // one atomic per wave, one store to the host in all (2M of them took 2 ms)
        if (__ffsll((unsigned long long)__ballot(1)) - 1 == (int)lane_id()) {
            const uint32_t old = atomicOr(err, ERR_STALE_KEYS);
            if (stale && !(old & ERR_STALE_KEYS))
                __hip_atomic_store(stale, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        return;
    }
    const uint32_t dst = offsets[k] + ranks[p];
    if (order) order[dst] = (uint32_t)p;
    R r;
    r.cell = record_cell(bx, by, bz, g);
    if constexpr (sizeof(R) == sizeof(DepRecord64)) {
        r.cell |= (k % buckets_per_box(g)) >> 3 << REC_CELL_BITS;
        r.index = (uint32_t)p;
        r.fx = fx;
        r.fy = fy;
        r.fz = fz;
        rec[dst] = r;
        if (masses) rec_mass[dst] = masses[p];
    } else {
        r.fx = (float)fx;
        r.fy = (float)fy;
        r.fz = (float)fz;
        rec[dst] = r;
        if (masses) rec_mass[dst] = (float)(masses[p] * inv_mass_unit);
        if (force) force[dst] = {(float)(1.0 - fx), (float)(1.0 - fy), (float)(1.0 - fz), k >> 3};
    }
}

// ===========================================================================
// Workgroup sort (ascending u64), arbitrary n, any address space.
// Bitonic network in the "flip" form: every comparator is ascending, so
// virtual +inf padding past n never has to move into range.
// ===========================================================================
template <typename P>
__device__ __forceinline__ void wg_sort_u64(P keys, uint32_t n) {
    if (n < 2) return;
    uint32_t np2 = 1;
    while (np2 < n) np2 <<= 1;
    const uint32_t half = np2 >> 1;
    for (uint32_t k = 2; k <= np2; k <<= 1) {
        // flip step: compare i with its mirror inside the block of size k
        for (uint32_t c = threadIdx.x; c < half; c += blockDim.x) {
            const uint32_t blk = c / (k >> 1);
            const uint32_t off = c % (k >> 1);
            const uint32_t i = blk * k + off;
            const uint32_t j = blk * k + k - 1 - off;
            if (j < n) {
                const uint64_t a = keys[i], b = keys[j];
                if (a > b) { keys[i] = b; keys[j] = a; }
            }
        }
        __threadfence_block();
        __syncthreads();
        for (uint32_t d = k >> 2; d >= 1; d >>= 1) {
            for (uint32_t c = threadIdx.x; c < half; c += blockDim.x) {
                const uint32_t i = (c / d) * 2 * d + (c % d);
                const uint32_t j = i + d;
                if (j < n) {
                    const uint64_t a = keys[i], b = keys[j];
                    if (a > b) { keys[i] = b; keys[j] = a; }
                }
            }
            __threadfence_block();
            __syncthreads();
        }
    }
}

// Sort each bucket's particle indices ascending (canonical stable order).
// Small buckets sort in LDS, large ones in place in global memory.
constexpr int CANON_THREADS = 256;
constexpr int CANON_LDS = 4096;

__global__ void __launch_bounds__(CANON_THREADS)
k_canonicalize(uint64_t nb, const uint32_t* __restrict__ offsets, uint32_t* __restrict__ order,
               uint64_t* __restrict__ scratch, uint64_t scratch_cap,
               unsigned long long* __restrict__ scratch_cursor, uint32_t* __restrict__ err) {
    __shared__ uint64_t sh[CANON_LDS];
    for (uint64_t b = blockIdx.x; b < nb; b += gridDim.x) {
        const uint32_t s = offsets[b], e = offsets[b + 1];
        const uint32_t n = e - s;
        if (n < 2) continue;
        if (n <= CANON_LDS) {
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) sh[i] = order[s + i];
            __syncthreads();
            wg_sort_u64(sh, n);
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) order[s + i] = (uint32_t)sh[i];
            __syncthreads();
        } else {
            __shared__ uint64_t base_sh;
            if (threadIdx.x == 0) base_sh = atomicAdd(scratch_cursor, (unsigned long long)n);
            __syncthreads();
            const uint64_t base = base_sh;
            __syncthreads();
            if (base + n > scratch_cap) {
                if (threadIdx.x == 0) atomicOr(err, ERR_SCRATCH);
                continue;
            }
            uint64_t* g = scratch + base;
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) g[i] = order[s + i];
            __threadfence_block();
            __syncthreads();
            wg_sort_u64(g, n);
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) order[s + i] = (uint32_t)g[i];
            __syncthreads();
        }
    }
}

// ===========================================================================
// Deterministic CIC deposit + density source
// ===========================================================================
constexpr int DEP_THREADS = 512;
constexpr int DEP_MAX_T = 16;
constexpr int DEP_NRANGES = 20;

// ---------------------------------------------------------------------------
// Exact deposited mass: the reference sums every cell's mass with
// ExactPositiveDoubleSum (src/gravity/pm_solver.cpp:132-180).  Here each box
// has SA_DIGITS counters, one per 32-bit digit of the binary positions
// 2^-1074 .. 2^1230 (every binary64 bit), each holding its digit's sum with
// the carries in its upper bits, plus a word flagging an input that is not a
// finite non-negative number.  The counters are integers, so the total is
// exact whatever the order of the additions; sa_round rounds it once to
// nearest (ties to even), as the host's exact_sum does.
// ---------------------------------------------------------------------------
constexpr int SA_DIGITS = 72;
constexpr int SA_WORDS = SA_DIGITS + 1;
// Each wave of a binary64 deposit workgroup stores its sum as a window of
// SA_WAVE_WIN counters from a base digit (SA_WAVE_WORDS words: base, window;
// base -1: empty); digits outside the window go to the box's counters
// directly.  k_mass_finish adds the windows up per box.  (Binary32 waves store
// the two digit sums of their fixed-point cells; k_mass_finish_fixed.)
constexpr int SA_WAVE_WIN = 8;
constexpr int SA_WAVE_WORDS = SA_WAVE_WIN + 1;
constexpr int SA_WAVES_PER_TILE = 8;  // deposit workgroups of 512 threads

// Wave-wide integer sum and minimum in the VALU pipe (no LDS permutes): DPP
// row shifts by 1, 2, 4 and 8 lanes leave each 16-lane row's total (minimum)
// in its last lane, and the four rows' last lanes are read as scalars.  Every
// lane of the wave must be active; the result is the same in every lane.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v, uint32_t fill) {
    // lanes whose source lies outside their row keep fill
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, CTRL, 0xf, 0xf, false);
}

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
    return ((uint64_t)dpp_u32<CTRL>((uint32_t)(v >> 32), 0u) << 32) | dpp_u32<CTRL>((uint32_t)v, 0u);
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
    v += dpp_u64<0x111>(v);  // row_shr:1
    v += dpp_u64<0x112>(v);  // row_shr:2
    v += dpp_u64<0x114>(v);  // row_shr:4
    v += dpp_u64<0x118>(v);  // row_shr:8
    uint64_t s = 0;
#pragma unroll
    for (int r = 15; r < 64; r += 16)
        s += ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), r) << 32) |
             (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, r);
    return s;
}

// Inclusive prefix sum over the 64 lanes of a wave (every lane active): the
// DPP row shifts give each lane its 16-lane row's prefix, then the totals of
// the rows below its own (read as scalars) are added.
__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t v) {
    v += dpp_u32<0x111>(v, 0u);  // row_shr:1
    v += dpp_u32<0x112>(v, 0u);  // row_shr:2
    v += dpp_u32<0x114>(v, 0u);  // row_shr:4
    v += dpp_u32<0x118>(v, 0u);  // row_shr:8
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
    const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
    const uint32_t row = lane_id() >> 4;
    return v + (row > 0 ? r0 : 0u) + (row > 1 ? r1 : 0u) + (row > 2 ? r2 : 0u);
}

// Adds x exactly to the counters d (flagging a value that is not finite and
// non-negative).
__device__ __forceinline__ void sa_add_direct(unsigned long long* d, double x) {
    if (x == 0.0) return;
    if (!(x > 0.0) || !isfinite(x)) {
        atomicOr(&d[SA_DIGITS], 1ull);
        return;
    }
    const uint64_t bits = (uint64_t)__double_as_longlong(x);
    const int e = (int)((bits >> 52) & 0x7ff);
    const uint64_t frac = bits & ((1ull << 52) - 1ull);
    const uint64_t mant = e ? (frac | (1ull << 52)) : frac;
    const int shift = e ? e - 1 : 0;
    const int limb = shift >> 5, o = shift & 31;
    const uint64_t l = mant << o, h = o ? mant >> (64 - o) : 0ull;
    if ((uint32_t)l) atomicAdd(&d[limb], (unsigned long long)(uint32_t)l);
    if ((uint32_t)(l >> 32) && limb + 1 < SA_DIGITS) atomicAdd(&d[limb + 1], (unsigned long long)(uint32_t)(l >> 32));
    if (h && limb + 2 < SA_DIGITS) atomicAdd(&d[limb + 2], (unsigned long long)h);
}

// A lane's running sum of cell masses as three binary64 sums of multiples of
// q1 = 2^80 q3, q2 = 2^40 q3 and q3 = 2^(32 base - 1074): adding and
// subtracting 1.5 2^52 q rounds a value to a multiple of q, so a mass splits
// into three parts whose sums stay exact integers of their quantum (parts of at
// most 2^40 quanta, at most 4096 cells per wave).  Fifteen additions per cell
// instead of the 60-odd integer instructions of a 192-bit accumulator.  A
// mass above 2^40 q1 or with bits below q3 (the host places q3 so that this
// leaves at least 2^-29 .. 2^8 mass units) goes to the box's counters.
struct SaQuanta {
    double c1, c2, c3;     // 1.5 2^52 q
    double i1, i2, i3;     // 1 / q
    double max;            // 2^40 q1; negative: every mass goes to the counters
    int base;              // digit of q3
};

struct SaAcc {
    double s1 = 0.0, s2 = 0.0, s3 = 0.0;
};

__device__ __forceinline__ void sa_acc_add(SaAcc& a, const SaQuanta& q, unsigned long long* d, double x) {
    const double t1 = (x + q.c1) - q.c1, r1 = x - t1;
    const double t2 = (r1 + q.c2) - q.c2, r2 = r1 - t2;
    const double t3 = (r2 + q.c3) - q.c3;
    if (x >= 0.0 && x <= q.max && r2 == t3) {
        a.s1 += t1;
        a.s2 += t2;
        a.s3 += t3;
    } else {
        sa_add_direct(d, x);
    }
}

// Wave-wide sum of binary64 values whose sums are exact (integers of one
// quantum below 2^53), the same in every lane; DPP as wave_sum_u64.
__device__ __forceinline__ double wave_sum_exact(double x) {
    auto shifted = [](uint64_t v, auto ctrl) { return __longlong_as_double((long long)dpp_u64<decltype(ctrl)::value>(v)); };
    auto bits = [](double v) { return (uint64_t)__double_as_longlong(v); };
    x += shifted(bits(x), std::integral_constant<int, 0x111>{});
    x += shifted(bits(x), std::integral_constant<int, 0x112>{});
    x += shifted(bits(x), std::integral_constant<int, 0x114>{});
    x += shifted(bits(x), std::integral_constant<int, 0x118>{});
    const int lo = (int)(uint32_t)bits(x), hi = (int)(uint32_t)(bits(x) >> 32);
    double s = 0.0;
#pragma unroll
    for (int r = 15; r < 64; r += 16)
        s += __longlong_as_double((long long)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, r) << 32) |
                                              (uint32_t)__builtin_amdgcn_readlane(lo, r)));
    return s;
}

// The wave's sum as six 32-bit digits from q.base, the same in every lane;
// every lane of the wave calls this.
__device__ __forceinline__ void sa_acc_digits(const SaAcc& a, const SaQuanta& q, uint64_t (&v)[6]) {
    // s1 2^80 + s2 2^40 + s3 in units of q3: parts may be negative, the sum is not
    const double s1 = wave_sum_exact(a.s1), s2 = wave_sum_exact(a.s2), s3 = wave_sum_exact(a.s3);
    const __int128 low = (__int128)(long long)(s3 * q.i3) + ((__int128)(long long)(s2 * q.i2) << 40);
    const __int128 mid = ((__int128)(long long)(s1 * q.i1) << 16) + (low >> 64);
    const uint64_t a0 = (uint64_t)low, a1 = (uint64_t)mid, a2 = (uint64_t)(mid >> 64);
    v[0] = (uint32_t)a0;
    v[1] = a0 >> 32;
    v[2] = (uint32_t)a1;
    v[3] = a1 >> 32;
    v[4] = (uint32_t)a2;
    v[5] = a2 >> 32;
}

// The wave's window (base, SA_WAVE_WIN digits; base -1: no mass) to out, from
// lanes 0..SA_WAVE_WIN.
__device__ __forceinline__ void sa_acc_flush(const SaAcc& a, const SaQuanta& q, unsigned long long* out) {
    uint64_t v[6];
    sa_acc_digits(a, q, v);
    const uint32_t lane = lane_id();
    uint64_t word = 0ull;
    bool any = false;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        any = any || v[j] != 0ull;
        if (lane == (uint32_t)j + 1) word = q.base + j < SA_DIGITS ? v[j] : 0ull;
    }
    if (lane == 0) word = any ? (uint64_t)q.base : ~0ull;
    if (lane <= (uint32_t)SA_WAVE_WIN) out[lane] = word;
}

// Q * unit * 2^-32 exactly as SA_WAVE_WIN 32-bit digits from digit limb, Q =
// (q1 2^64 + q0) an exact integer sum of 32.32 fixed-point cells (q1 < 2^32).
// False when unit is not a normal binary64 of at least 2^-1042 (the sum is
// then flagged invalid).
__device__ __forceinline__ bool sa_fixed_digits(uint64_t q0, uint64_t q1, double unit, int& limb,
                                                uint32_t (&dig)[SA_WAVE_WIN]) {
    const uint64_t bits = (uint64_t)__double_as_longlong(unit);
    const int e = (int)((bits >> 52) & 0x7ff);
    const int shift = e - 1 - 32;
    if (e == 0 || e == 0x7ff || shift < 0) return false;
    const uint64_t m = (bits & ((1ull << 52) - 1ull)) | (1ull << 52);
    // P = Q * m as three 64-bit words
    const uint64_t a_lo = q0 * m, a_hi = __umul64hi(q0, m);
    const uint64_t b_lo = q1 * m, b_hi = __umul64hi(q1, m);
    const uint64_t p1 = a_hi + b_lo;
    const uint64_t p2 = b_hi + (p1 < a_hi ? 1ull : 0ull);
    const uint32_t v[6] = {(uint32_t)a_lo, (uint32_t)(a_lo >> 32), (uint32_t)p1, (uint32_t)(p1 >> 32),
                           (uint32_t)p2, (uint32_t)(p2 >> 32)};
    // the product shifted by `shift` bits: seven 32-bit digits from shift / 32
    limb = shift >> 5;
    const int off = shift & 31;
#pragma unroll
    for (int k = 0; k < SA_WAVE_WIN; ++k) {
        const uint64_t lo = k < 6 ? (uint64_t)v[k] << off : 0ull;
        const uint64_t hi = (k > 0 && k <= 6 && off) ? (uint64_t)v[k - 1] >> (32 - off) : 0ull;
        dig[k] = (uint32_t)((lo | hi) & 0xffffffffull);
    }
    return true;
}

struct DepParams {
    Geom g;
    const double* x;
    const double* y;
    const double* z;
    const double* masses;   // nullptr -> uniform
    double uniform_mass;
    double pos_shift;         // positions are deposited as x - pos_shift (0: as given)
    const uint32_t* offsets;  // bucket offsets (nb+1)
    const DepRecord64* rec64; // binary64 deposit records in bucket order
    const double* rec_mass64; // binary64 masses in bucket order (explicit masses, or signed adjoint values)
    uint64_t n;               // particle count (bound of every record's index)
    double mean_mass;         // M / N_cells
    double inv_volume;        // 1 / dx^3
    double total_mass;        // M (exact input mass)
    double cells_real;        // N_cells as double
    uint64_t norm_mant;       // 1/(N_cells dx^3) as a 64-bit mantissa ...
    int norm_exp;             // ... times 2^norm_exp (the reference holds it in long double)
    int direct;               // 1: (m - mean) * inv_volume ; 0: fma-centred path
    int raw;                  // 1: write the deposited sum itself (adjoint deposits of signed values)
    SaQuanta sa;                      // splitting of the cell masses (binary64)
    unsigned long long* mass_digits;  // per box SA_WORDS counters of the exact deposited mass
    unsigned long long* mass_waves;   // per tile and wave: binary64 its digit window (SA_WAVE_WORDS),
                                      // binary32 the two digit sums of its cells
    unsigned long long* dense_count;  // binary64 jobs of tiles beyond one workgroup's LDS: evenly cut, planned
    uint64_t* dense_list;             // box of the tile (dep_box) << 32 | box-major tile index: even_cap evenly
                                      // cut jobs, then plan_cap planned ones
    uint32_t even_cap, plan_cap;
    uint64_t* scratch;                // record lists of dense jobs (as far as it reaches)
    uint64_t scratch_cap;
    unsigned long long* scratch_cursor;
    uint32_t* err;
};

// |c| * S with S = s_mant * 2^s_exp (64-bit mantissa), rounded first to a
// 64-bit significand and then to binary64: the x87 long-double product and cast
// of the reference's scaled density normalisation, emulated exactly with a
// 128-bit integer product.
__device__ __forceinline__ double scaled_product_ld(double c, uint64_t s_mant, int s_exp) {
    int ea = 0;
    const double fa = frexp(fabs(c), &ea);
    const uint64_t ma = (uint64_t)ldexp(fa, 53);
    const unsigned __int128 q = (unsigned __int128)ma * (unsigned __int128)s_mant;
    const uint64_t qhi = (uint64_t)(q >> 64);
    const int nb = qhi ? 128 - __clzll(qhi) : 64 - __clzll((uint64_t)q);
    int sh = nb - 64;
    uint64_t m64 = (uint64_t)(q >> sh);
    if (sh > 0) {
        const unsigned __int128 rem = q & ((((unsigned __int128)1) << sh) - 1);
        const unsigned __int128 half = ((unsigned __int128)1) << (sh - 1);
        if (rem > half || (rem == half && (m64 & 1ull))) {
            m64 += 1ull;
            if (m64 == 0ull) { m64 = 1ull << 63; sh += 1; }
        }
    }
    uint64_t m53 = m64 >> 11;
    const uint64_t r2 = m64 & 0x7ffull;
    if (r2 > 0x400ull || (r2 == 0x400ull && (m53 & 1ull))) m53 += 1ull;
    return copysign(ldexp((double)m53, (ea - 53) + s_exp + sh + 11), c);
}

template <typename T>
__device__ __forceinline__ T contrast_of(T sum, const DepParams& P) {
    const double m = (double)sum;
    if (P.raw) return (T)m;
    double v;
    if (P.direct) {
        v = (m - P.mean_mass) * P.inv_volume;
    } else {
        const double c = fma(m, P.cells_real, -P.total_mass);
        v = c == 0.0 ? 0.0 : scaled_product_ld(c, P.norm_mant, P.norm_exp);
    }
    return (T)v;
}

// Binary32 deposit: (m - M/N_c) / dx^3 in binary64, rounded to binary32.  It
// differs from the reference's fma-centred form (taken by contrast_of when
// M/N_c is not exact) by about one binary64 ulp, far below the binary32
// rounding of the cell, and avoids that form's 64-bit mantissa arithmetic.
__device__ __forceinline__ float contrast_fp32(double m, const DepParams& P) {
    if (P.raw) return (float)m;
    return (float)((m - P.mean_mass) * P.inv_volume);
}

// Source ranges of a destination tile: range 0 is the own tile (all eight
// classes, contiguous); ranges 1..19 are the boundary classes c of the seven
// lower neighbour tiles at offset d in {0,1}^3 with (c & d) == d, in the order
//   (0,0) (1,1) (1,3) (1,5) (1,7) (2,2) (2,3) (2,6) (2,7) (3,3) (3,7)
//   (4,4) (4,5) (4,6) (4,7) (5,5) (5,7) (6,6) (6,7) (7,7).
// The d and c of range t are 3-bit fields t of two immediates (a per-lane
// table lookup would cost each tile a memory round trip before its offsets).
constexpr uint64_t kRangeD = 0xfb5b248da491248ull;
constexpr uint64_t kRangeC = 0xff7bf59dfcd7ac8ull;
struct RangeSlot { uint8_t d, c; };
__device__ __forceinline__ RangeSlot range_slot(int t) {
    return RangeSlot{(uint8_t)((kRangeD >> (3 * t)) & 7u), (uint8_t)((kRangeC >> (3 * t)) & 7u)};
}

// Fills rs (start in order[]), rc (prefix of counts, rc[20] = total), rd (d),
// rcls (class) with one global round trip per range, in parallel.
__device__ __forceinline__ void load_source_ranges(const uint32_t* __restrict__ offsets, int tx, int ty,
                                                   int tz, int nT, uint32_t* rs, uint32_t* rc,
                                                   uint8_t* rd, uint8_t* rcls) {
    const int t = threadIdx.x;
    if (t < 64) {  // the first wave: one lane per range, then a wave scan of the counts
        uint32_t cnt = 0;
        if (t < 20) {
            const RangeSlot sl = range_slot(t);
            const int d = sl.d;
            const int sx = (tx - ((d >> 2) & 1) + nT) % nT, sy = (ty - ((d >> 1) & 1) + nT) % nT,
                      sz = (tz - (d & 1) + nT) % nT;
            const uint32_t t8 = (((uint32_t)sx * nT + sy) * nT + sz) * 8u;
            const uint32_t lo = d == 0 ? t8 : t8 + sl.c;
            const uint32_t hi = d == 0 ? t8 + 8 : t8 + sl.c + 1;
            const uint32_t a = offsets[lo], b = offsets[hi];
            rs[t] = a;
            cnt = b - a;
            rd[t] = (uint8_t)d;
            rcls[t] = sl.c;
        }
        const uint32_t incl = wave_incl_scan_u32(cnt);
        if (t < 20) rc[t + 1] = incl;
        if (t == 0) rc[0] = 0;
    }
    __syncthreads();
}

// Exclusive scan of a[0..count) in LDS, in place, by all threads of the
// workgroup (each thread owns a contiguous chunk): a scan inside each
// wavefront, then the wavefront totals (part: one word per wavefront).
__device__ __forceinline__ void wg_exclusive_scan_lds(uint32_t* a, int count, uint32_t* part) {
    const int nt = (int)blockDim.x;
    const int per = (count + nt - 1) / nt;
    const int b = (int)threadIdx.x * per;
    const int e = b + per < count ? b + per : count;
    uint32_t s = 0;
    for (int i = b; i < e; ++i) s += a[i];
    const int lane = (int)lane_id(), wave = (int)threadIdx.x / 64;
    const uint32_t incl = wave_incl_scan_u32(s);
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    uint32_t run = incl - s;
    for (int w = 0; w < wave; ++w) run += part[w];
    for (int i = b; i < e; ++i) {
        const uint32_t v = a[i];
        a[i] = run;
        run += v;
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Binary64 deposit in the reference's summation order.
//
// One workgroup per destination tile.  The tile's records (own bucket and the
// boundary classes of the seven lower neighbours) go to LDS, then a counting
// sort by DESTINATION cell gives every cell the list of its contributions
// (record slot, corner): eight LDS counter atomics and eight 2-byte stores per
// record.  A cell's list is put into the reference's order (base x == cell x
// first, then base x == cell x - 1, each by particle index) and summed:
//   - short lists by one thread (a sorting network in registers, for two
//     neighbouring cells at once while they hold at most 8; at 1/8 to 1
//     particle per cell a list holds 1 to 8 entries);
//   - longer lists by one wave: with the records' ranks by particle index, a
//     list is sorted through a bitmap of its (offset, rank) pairs and a prefix of
//     its word counts, in time linear in its length; then the terms are formed
//     64 at a time and added in order with lane reads, so a dense cell costs
//     one addition latency per entry.
// A tile with more than CAP records, or with a list for a wave, becomes jobs
// (boxes of the tile, one workgroup each) of a second launch: as many as the
// plan of its records makes, or 1 to 64 equal ones where it makes none.  A job
// that still exceeds the LDS lists its records in the scratch (when it has
// room) and halves its box along the longest edge until the records fit.  A
// single cell with more than DEP_CAP sources sorts its particle indices by
// themselves, in index ranges that fit the LDS.
//
// Bound by LDS latency (the chain counter -> scan -> entry -> record) and by
// the 150 or so instructions per cell.  CAP = 736 records (the 1/8 particles per
// cell of a mesh twice the lattice give about 614) keep the workgroup's LDS at
// 53 KB, three per CU (59 KB and two with masses); CAP = 1024, 66 KB and two, is
// for loads whose tiles need it (the host's rule): with 736 alone 0.16 to 0.2
// particles per cell went through the second launch and were 5 to 8% slower than
// the kernel that this one replaced.  Measured against one thread per cell
// merging four index-sorted source lists (and a whole-tile sort in global
// memory above 1024 records): 16.8M lattice particles on 512^3 1.33 -> 0.85 ms,
// 3M clustered particles with masses on 192^3 16.8 -> 2.2 ms, 8192 on 32^3
// 162 -> 36 us.
// ---------------------------------------------------------------------------
constexpr int DEP_CAP = 736;        // records of a job, and of a tile in the first launch's narrow kernel
constexpr int DEP_CAP_WIDE = 1024;  // records of a tile in its wide kernel
constexpr int DEP_SERIAL = 16;  // entries one thread sorts (its network's size) in the second launch ...
constexpr int DEP_COMMON = 8;   // ... and in the first, whose 80 registers hold no larger network
constexpr int DEP_JOB_RECORDS = 256;  // a tile of M records is cut evenly into at most M / DEP_JOB_RECORDS jobs
constexpr int DEP_MAX_CELLS = DEP_MAX_T * DEP_MAX_T * DEP_MAX_T;
constexpr int DEP_HEAVY = 8 * DEP_CAP / (DEP_SERIAL + 1) + 1;  // most lists longer than DEP_SERIAL
constexpr int DEP_STACK = 16;                                   // boxes waiting (at most one per halving, 12)
constexpr int DEP_BITS = 2 * ((DEP_CAP + 31) / 32);  // words of a list's bitmap: both x offsets
static_assert(8 * DEP_CAP_WIDE <= 65535, "16-bit list entries");
static_assert(DEP_BITS <= 64 && DEP_CAP % 16 == 0, "one lane per bitmap word; padded index scans");

// LDS of the workgroup as one block (also the key array of a hot cell).
template <int CAP>
struct DepLds {
    double fx[CAP], fy[CAP], fz[CAP];
    uint32_t start[DEP_MAX_CELLS + 1];
    alignas(16) uint32_t idx[CAP];  // particle index
    uint16_t ent[8 * CAP]; // slot * 8 + corner (ox, oy, oz bits 2, 1, 0)
    uint16_t cell[CAP];    // base cell in the tile, each axis + 1 in 5 bits; then ranks by particle index
};
constexpr uint32_t DEP_HOT_LDS = sizeof(DepLds<DEP_CAP>) / sizeof(uint64_t);

// Halvings (x, y, z in turn) of a tile of M > DEP_CAP records: uniform boxes
// then hold 340 to 750 records.
__device__ __forceinline__ int dep_split(uint32_t M) {
    return M <= 1400u ? 1 : M <= 2400u ? 2 : M <= 4096u ? 3 : M <= 8192u ? 4 : M <= 16384u ? 5 : 6;
}

// Box j of the 2^levels boxes of a tile of edge T: x0, y0, z0 and the edges
// minus one, four bits each.
__device__ __forceinline__ uint32_t dep_box(int T, int levels, uint32_t j) {
    uint32_t code = 0;
    for (int a = 0; a < 3; ++a) {
        const int n = (levels + 2 - a) / 3;  // halvings of this axis
        int lo = 0, e = T;
        for (int l = 0; l < n; ++l) {
            const int h = (e + 1) / 2;
            if (j & 1u) {
                lo += h;
                e -= h;
            } else {
                e = h;
            }
            j >>= 1;
        }
        code |= ((uint32_t)lo << (4 * a)) | ((uint32_t)(e - 1) << (12 + 4 * a));
    }
    return code;
}

// Minimum and maximum of ordinary binary64 numbers as the bare instructions
// (fmin and fmax quiet their operands first).
__device__ __forceinline__ double min_f64(double x, double y) {
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
#else
    return x < y ? x : y;
#endif
}
__device__ __forceinline__ double max_f64(double x, double y) {
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
#else
    return x < y ? y : x;
#endif
}

// In-order sum of up to 64 terms held one per lane, added to sum: sum is
// uniform, each step reads one lane's term.  Whole waves run unrolled, so the
// lane reads go ahead of the additions and a term costs one addition latency.
__device__ __forceinline__ double wave_ordered_add(double sum, double term, int count) {
    const uint64_t b = (uint64_t)__double_as_longlong(term);
    const int lo = (int)(uint32_t)b, hi = (int)(uint32_t)(b >> 32);
    auto at = [&](int j) {
        const uint64_t t = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, j) << 32) |
                           (uint32_t)__builtin_amdgcn_readlane(lo, j);
        return __longlong_as_double((long long)t);
    };
    int j = 0;
    for (; j + 8 <= count; j += 8) {
        double t[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) t[k] = at(j + k);
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += t[k];
    }
    for (; j < count; ++j) sum += at(j);
    return sum;
}

// Jobs of a tile of M > DEP_CAP records: a histogram of the records' base cells
// and its 3-D prefix sums give every box's record count in eight lookups; boxes
// are halved level by level until they hold DEP_CAP records or one cell, so a
// clump's core becomes many jobs and the rest of its tile few.  False (no job
// made) when a level or the job count outgrows its LDS array, or the planned
// jobs outgrow their part of the list: the caller then cuts the tile evenly.
// lds: DEP_PLAN_LDS words; counter: one LDS word.  The whole workgroup calls it.
constexpr int DEP_PLAN_EXT = (DEP_MAX_T + 1) * (DEP_MAX_T + 1) * (DEP_MAX_T + 1);
constexpr uint32_t DEP_FRONTIER = 1024, DEP_LEAVES = 2048;
constexpr int DEP_PLAN_LDS = DEP_PLAN_EXT + 2 * (int)DEP_FRONTIER + (int)DEP_LEAVES + 4;
static_assert(DEP_PLAN_LDS * sizeof(uint32_t) <= sizeof(DepLds<DEP_CAP>), "the plan fits the deposit's LDS");

template <typename BaseCell, typename SlotOf>
__device__ __forceinline__ bool dep_plan_jobs(const DepParams& P, int T, uint32_t M, uint32_t gtile,
                                              BaseCell&& base_cell, SlotOf&& slot_of, uint32_t* lds,
                                              uint32_t* reserved) {
    const int tid = (int)threadIdx.x, E = T + 1;
    uint32_t* hist = lds;
    uint32_t* front = lds + DEP_PLAN_EXT;
    uint32_t* next = front + DEP_FRONTIER;
    uint32_t* leaves = next + DEP_FRONTIER;
    uint32_t* counts = leaves + DEP_LEAVES;  // frontier, next frontier, leaves
    for (int i = tid; i < E * E * E; i += DEP_THREADS) hist[i] = 0u;
    if (tid == 0) {
        front[0] = dep_box(T, 0, 0u);
        counts[0] = 1u;
        counts[1] = 0u;
        counts[2] = 0u;
    }
    __syncthreads();
    for (uint32_t v = (uint32_t)tid; v < M; v += DEP_THREADS) {
        int d;
        const uint32_t slot = slot_of(v, d);
        const uint32_t c = base_cell(P.rec64[slot], d);
        const int x = (int)(c >> 10), y = (int)((c >> 5) & 31u), z = (int)(c & 31u);
        if (x < E && y < E && z < E) atomicAdd(&hist[(x * E + y) * E + z], 1u);
    }
    __syncthreads();
    // inclusive sums along z, then y, then x: line l of each axis by one thread
    for (int axis = 0; axis < 3; ++axis) {
        const int step = axis == 0 ? 1 : (axis == 1 ? E : E * E);
        for (int l = tid; l < E * E; l += DEP_THREADS) {
            const int a = l / E, b = l % E;
            int at = axis == 0 ? l * E : (axis == 1 ? a * E * E + b : l);
            uint32_t s = 0;
            for (int i = 0; i < E; ++i, at += step) {
                s += hist[at];
                hist[at] = s;
            }
        }
        __syncthreads();
    }
    auto sum = [&](int x, int y, int z) -> uint32_t {  // records with base below (x, y, z)
        return x > 0 && y > 0 && z > 0 ? hist[((x - 1) * E + (y - 1)) * E + (z - 1)] : 0u;
    };
    for (;;) {
        const uint32_t nf = counts[0];
        for (uint32_t i = (uint32_t)tid; i < nf; i += DEP_THREADS) {
            const uint32_t code = front[i];
            const int lo[3] = {(int)(code & 15u), (int)((code >> 4) & 15u), (int)((code >> 8) & 15u)};
            const int e[3] = {(int)((code >> 12) & 15u) + 1, (int)((code >> 16) & 15u) + 1, (int)((code >> 20) & 15u) + 1};
            // base cells lo - 1 .. lo + e - 1, stored one up: lo .. lo + e
            const int hx = lo[0] + e[0] + 1, hy = lo[1] + e[1] + 1, hz = lo[2] + e[2] + 1;
            const uint32_t m = sum(hx, hy, hz) - sum(lo[0], hy, hz) - sum(hx, lo[1], hz) - sum(hx, hy, lo[2]) +
                               sum(lo[0], lo[1], hz) + sum(lo[0], hy, lo[2]) + sum(hx, lo[1], lo[2]) -
                               sum(lo[0], lo[1], lo[2]);
            if (m <= (uint32_t)DEP_CAP || e[0] * e[1] * e[2] == 1) {
                const uint32_t at = atomicAdd(&counts[2], 1u);
                if (at < DEP_LEAVES) leaves[at] = code;
            } else {
                const int ax = e[0] >= e[1] && e[0] >= e[2] ? 0 : (e[1] >= e[2] ? 1 : 2);
                const int h = (e[ax] + 1) / 2;
                const uint32_t keep = ~((15u << (4 * ax)) | (15u << (12 + 4 * ax)));
                const uint32_t at = atomicAdd(&counts[1], 2u);
                if (at + 1 < DEP_FRONTIER) {
                    next[at] = (code & keep) | ((uint32_t)lo[ax] << (4 * ax)) | ((uint32_t)(h - 1) << (12 + 4 * ax));
                    next[at + 1] = (code & keep) | ((uint32_t)(lo[ax] + h) << (4 * ax)) |
                                   ((uint32_t)(e[ax] - h - 1) << (12 + 4 * ax));
                }
            }
        }
        __syncthreads();
        const uint32_t nn = counts[1], nl = counts[2];
        __syncthreads();
        if (nn > DEP_FRONTIER || nl > DEP_LEAVES) return false;
        if (nn == 0) break;
        if (tid == 0) {
            counts[0] = nn;
            counts[1] = 0u;
        }
        uint32_t* t = front;
        front = next;
        next = t;
        __syncthreads();
    }
    const uint32_t nl = counts[2];
    if (tid == 0) *reserved = (uint32_t)atomicAdd(P.dense_count + 1, (unsigned long long)nl);
    __syncthreads();
    const uint32_t at = *reserved;
    if (at + nl > P.plan_cap) {
        // the tile's part of the list counts as used; jobs there are marked void
        for (uint32_t i = (uint32_t)tid; i < nl && at + i < P.plan_cap; i += DEP_THREADS)
            P.dense_list[P.even_cap + at + i] = ~0ull;
        return false;
    }
    for (uint32_t i = (uint32_t)tid; i < nl; i += DEP_THREADS)
        P.dense_list[P.even_cap + at + i] = ((uint64_t)leaves[i] << 32) | gtile;
    return true;
}

// TE: compile-time tile edge (16) or 0; MASS: explicit (or signed adjoint) masses.
// DENSE = false: one workgroup per tile; tiles that need more go to the job
// list.  DENSE = true: the workgroups walk that list (the box
// splitting and the hot cells in the common kernel would take its registers
// from 80 to 145, three workgroups per CU to one).
template <int TE, bool MASS, bool DENSE, int CAP>
__global__ void __launch_bounds__(DEP_THREADS) __attribute__((amdgpu_waves_per_eu(DENSE || MASS || CAP > DEP_CAP ? 4 : 6)))
k_deposit(DepParams P, double* __restrict__ mesh0) {
    static_assert(!DENSE || CAP == DEP_CAP, "jobs hold DEP_CAP records");
    constexpr int PER = (CAP + DEP_THREADS - 1) / DEP_THREADS;  // records per thread
    __shared__ __align__(16) DepLds<CAP> S;
    __shared__ double sh_m[MASS ? CAP : 1];
    __shared__ uint32_t sh_rs[DEP_NRANGES], sh_rc[DEP_NRANGES + 1];
    __shared__ uint8_t sh_rd[DEP_NRANGES], sh_rcls[DEP_NRANGES];
    __shared__ uint32_t sh_part[DEP_THREADS / 64];
    __shared__ uint16_t sh_heavy[DEP_HEAVY];
    __shared__ uint32_t sh_bits[DEP_THREADS / 64][DEP_BITS];
    __shared__ uint32_t sh_stack[DEP_STACK];  // boxes: x0, y0, z0 (4 bits each), edges - 1 (4 bits each)
    __shared__ uint32_t sh_count, sh_nheavy;
    __shared__ unsigned long long sh_list;
    __shared__ unsigned long long sh_digits[6];  // DENSE: the workgroup's mass digits

    const Geom& g = P.g;
    const int nT = g.nT;
    const uint32_t ntiles = (uint32_t)nT * nT * nT;
    const int TT = TE > 0 ? TE : g.T;
    const int tid = (int)threadIdx.x, lane = (int)lane_id(), wave = tid >> 6;
    // DENSE: the planned jobs, then the evenly cut ones
    const uint32_t planned = DENSE ? min((uint32_t)P.dense_count[1], P.plan_cap) : 0u;
    const uint32_t jobs = DENSE ? planned + (uint32_t)P.dense_count[0] : gridDim.x;
    for (uint32_t job = blockIdx.x; job < jobs; job += gridDim.x) {
    if constexpr (DENSE) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the last tile's LDS
        __syncthreads();
    }
    const uint64_t entry = DENSE ? P.dense_list[job < planned ? P.even_cap + job : job - planned]
                                 : (uint64_t)xcd_block(job, jobs);
    if (DENSE && entry == ~0ull) continue;
    const uint32_t gtile = (uint32_t)entry;  // box-major tile index
    const uint32_t box = gtile / ntiles, tile = gtile % ntiles;
    const int tz = tile % nT, ty = (tile / nT) % nT, tx = tile / (nT * nT);
    double* mesh = mesh0 + (uint64_t)box * g.N * g.N * g.N;
    static_assert(DEP_THREADS / 64 == SA_WAVES_PER_TILE, "one mass window per wave");
    // exact cell-mass sum: each wave's window, plus the box's counters for the rest
    unsigned long long* box_digits = P.mass_digits + (uint64_t)box * SA_WORDS;
    unsigned long long* wave_out =
        P.mass_waves + ((uint64_t)gtile * SA_WAVES_PER_TILE + threadIdx.x / 64) * SA_WAVE_WORDS;
    SaAcc win;

    if (DENSE && tid == 0) sh_stack[0] = (uint32_t)(entry >> 32);
    load_source_ranges(P.offsets + (uint64_t)box * buckets_per_box(g), tx, ty, tz, nT, sh_rs, sh_rc, sh_rd,
                       sh_rcls);
    const uint32_t M = sh_rc[DEP_NRANGES];
    // !DENSE: leaves the tile to 2^levels equal jobs, which also add its mass
    auto leave = [&](int levels) {
        if (tid < 64) {
            uint32_t at = 0;
            if (lane == 0) at = (uint32_t)atomicAdd(P.dense_count, 1ull << levels);
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
            if (lane < (1 << levels))
                P.dense_list[at + (uint32_t)lane] = ((uint64_t)dep_box(TT, levels, (uint32_t)lane) << 32) | gtile;
        }
        if (lane == 0) wave_out[0] = ~0ull;
    };
    // Writes the finished cell (tile coordinates) and adds its mass.
    mesh += ((uint64_t)(tx * TT) * g.N + (uint64_t)(ty * TT)) * g.N + (uint64_t)(tz * TT);
    auto finish = [&](int lx, int ly, int lz, double sum) {
        if (!P.raw) sa_acc_add(win, P.sa, box_digits, sum);
        mesh[(uint64_t)(uint32_t)(lx * g.N + ly) * (uint64_t)g.N + (uint32_t)lz] = contrast_of(sum, P);
    };

    // Base cell of a record in the tile (-1 .. T-1 per axis, each + 1 in 5 bits);
    // DEP_NOWHERE, outside every box, for a record that does not lie where its
    // bucket says (ERR_COORDINATE; also a slot a failed scatter left unwritten).
    constexpr uint32_t DEP_NOWHERE = 0x7fff;
    auto base_cell = [&](const DepRecord64& rec, int d) -> uint32_t {
        const uint32_t c = rec.cell & ((1u << REC_CELL_BITS) - 1u);
        const int cz = (int)(c % (uint32_t)TT), cy = (int)((c / (uint32_t)TT) % (uint32_t)TT),
                  cx = (int)(c / (uint32_t)(TT * TT));
        if (cx >= TT || ((d & 4) && cx != TT - 1) || ((d & 2) && cy != TT - 1) || ((d & 1) && cz != TT - 1) ||
            rec.index >= P.n) {
            atomicOr(P.err, ERR_COORDINATE);
            return DEP_NOWHERE;
        }
        return (uint32_t)((((d & 4) ? 0 : cx + 1) << 10) | (((d & 2) ? 0 : cy + 1) << 5) | ((d & 1) ? 0 : cz + 1));
    };
    auto slot_of = [&](uint32_t v, int& d) -> uint32_t {  // record v of the tile: its slot and neighbour offset
        int lo = 0, hi = DEP_NRANGES - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sh_rc[mid] <= v) lo = mid;
            else hi = mid - 1;
        }
        d = sh_rd[lo];
        return sh_rs[lo] + (v - sh_rc[lo]);
    };

    if constexpr (!DENSE) {
        if (M > (uint32_t)CAP) {
            if (!dep_plan_jobs(P, TT, M, gtile, base_cell, slot_of, reinterpret_cast<uint32_t*>(&S), &sh_nheavy)) leave(dep_split(M));
            if (lane == 0) wave_out[0] = ~0ull;
            return;
        }
    }

    uint64_t* list = nullptr;  // this job's records: slot << 32 | base cell
    uint32_t listed = 0;
    int depth = 1;
    while (depth > 0) {
        // The box stack written at the end of the last trip, and that box's LDS
        // reads.  The wait is explicit: with one thread's LDS write on a path that
        // ended in continue and no barrier behind it, the compiler left the wait
        // of the header's barrier out, and a wave that read the stack ahead of its
        // write went through other barriers than the rest.  Such a write has its
        // barrier before the continue here, and every barrier of the compiled
        // kernels an LDS wait on all paths to it.
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __syncthreads();
        --depth;
        const uint32_t code = DENSE ? sh_stack[depth] : dep_box(TT, 0, 0u);
        const int x0 = (int)(code & 15u), y0 = (int)((code >> 4) & 15u), z0 = (int)((code >> 8) & 15u);
        const int ex = (int)((code >> 12) & 15u) + 1, ey = (int)((code >> 16) & 15u) + 1,
                  ez = (int)((code >> 20) & 15u) + 1;
        const int cells = ex * ey * ez;

        auto in_box = [&](uint32_t bc) {
            const uint32_t bx = bc >> 10, by = (bc >> 5) & 31u, bz = bc & 31u;
            return bx - (uint32_t)x0 <= (uint32_t)ex && by - (uint32_t)y0 <= (uint32_t)ey &&
                   bz - (uint32_t)z0 <= (uint32_t)ez;
        };
        // The records whose corners touch the box: use(s, base cell, slot) for
        // those that want(base cell, slot) takes, s from a counter in LDS (one
        // atomic per wave and four records per thread, their loads in flight
        // together).
        auto each_match = [&](auto&& want, auto&& use) {
            const uint32_t count = list ? listed : M;
            for (uint32_t v0 = 0; v0 < count; v0 += 4 * DEP_THREADS) {
                uint32_t bc[4], slot[4], at[4];
                bool live[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const uint32_t v = v0 + (uint32_t)(h * DEP_THREADS + tid);
                    bc[h] = DEP_NOWHERE;
                    slot[h] = 0u;
                    if (v < count) {
                        if (list) {
                            const uint64_t e = list[v];
                            bc[h] = (uint32_t)e;
                            slot[h] = (uint32_t)(e >> 32);
                        } else {
                            int d;
                            slot[h] = slot_of(v, d);
                            bc[h] = base_cell(P.rec64[slot[h]], d);
                        }
                    }
                }
                uint32_t total = 0;
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    live[h] = in_box(bc[h]) && want(bc[h], slot[h]);
                    const uint64_t mask = __ballot(live[h]);
                    at[h] = total + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
                    total += (uint32_t)__popcll(mask);
                }
                uint32_t base = 0;
                if (total) {  // uniform over the wave
                    if (lane == 0) base = atomicAdd(&sh_count, total);
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                }
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    if (live[h]) use(base + at[h], bc[h], slot[h]);
            }
        };
        auto any = [](uint32_t, uint32_t) { return true; };
        auto keep = [&](uint32_t s, uint32_t slot, const DepRecord64& rc, uint32_t bc) {
            S.fx[s] = rc.fx;
            S.fy[s] = rc.fy;
            S.fz[s] = rc.fz;
            S.idx[s] = rc.index;
            S.cell[s] = (uint16_t)bc;
            if constexpr (MASS) sh_m[s] = P.rec_mass64[slot];
        };

        uint32_t m = M;
        {
            if (tid == 0) {
                sh_count = 0;
                sh_nheavy = 0;
            }
            for (int i = tid; i <= cells; i += DEP_THREADS) S.start[i] = 0u;
            if constexpr (!DENSE) {
                // both records of a thread in flight together
                DepRecord64 rec[PER];
                uint32_t slot[PER];
                int d[PER];
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const uint32_t v = (uint32_t)(tid + j * DEP_THREADS);
                    if (v < M) {
                        slot[j] = slot_of(v, d[j]);
                        rec[j] = P.rec64[slot[j]];
                    }
                }
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const uint32_t v = (uint32_t)(tid + j * DEP_THREADS);
                    if (v < M) keep(v, slot[j], rec[j], base_cell(rec[j], d[j]));
                }
                __syncthreads();
            } else {
                __syncthreads();
                each_match(any, [&](uint32_t s, uint32_t bc, uint32_t slot) {
                    if (s < (uint32_t)DEP_CAP) keep(s, slot, P.rec64[slot], bc);
                });
                __syncthreads();
                m = sh_count;
            }
        }
        if (DENSE && m > (uint32_t)DEP_CAP) {
            if (!list) {
                // first box of the job: its records listed for the boxes inside it
                __syncthreads();
                if (tid == 0) {
                    sh_list = atomicAdd(P.scratch_cursor, (unsigned long long)m);
                    sh_count = 0;
                }
                __syncthreads();
                if (sh_list + m <= P.scratch_cap) {
                    uint64_t* out = P.scratch + sh_list;
                    each_match(any, [&](uint32_t s, uint32_t bc, uint32_t slot) {
                        if (s < m) out[s] = ((uint64_t)slot << 32) | bc;
                    });
                    __threadfence_block();
                    list = out;
                    listed = m;
                }
            }
            if (cells > 1) {
                // halve the longest edge (x first: its halves are contiguous in the mesh)
                __syncthreads();
                if (tid == 0) {
                    const int hx = ex >= ey && ex >= ez ? (ex + 1) / 2 : 0, hy = !hx && ey >= ez ? (ey + 1) / 2 : 0;
                    const int hz = !hx && !hy ? (ez + 1) / 2 : 0;
                    auto enc = [](int a, int b, int c, int u, int v, int w) {
                        return (uint32_t)(a | (b << 4) | (c << 8) | ((u - 1) << 12) | ((v - 1) << 16) | ((w - 1) << 20));
                    };
                    sh_stack[depth] = enc(x0, y0, z0, hx ? hx : ex, hy ? hy : ey, hz ? hz : ez);
                    sh_stack[depth + 1] = enc(x0 + hx, y0 + hy, z0 + hz, hx ? ex - hx : ex, hy ? ey - hy : ey,
                                              hz ? ez - hz : ez);
                }
                __syncthreads();
                depth += 2;
                continue;
            }
            // One cell with more than DEP_CAP sources: keys (phase, particle index,
            // y and z offset) of the sources whose (phase, index) lies in
            // [lo, hi), a range whose keys fit the LDS, sorted; the terms in
            // place of the keys, then added in order by the first wave.  Range
            // by range, the running sum carried on.
            uint64_t* keys = reinterpret_cast<uint64_t*>(&S);
            const uint64_t end = 2 * P.n;  // keys are phase * n + index
            uint64_t lo = 0, width = m <= DEP_HOT_LDS ? end : (P.n / m + 1) * (DEP_HOT_LDS / 2);
            double sum = 0.0;
            while (lo < end) {
                const uint64_t hi = lo + width;
                __syncthreads();
                if (tid == 0) sh_count = 0;
                __syncthreads();
                // offsets 1 where the base is one below the cell
                auto key = [&](uint32_t bc, uint32_t slot) -> uint64_t {
                    return (((bc >> 10) == (uint32_t)x0 ? P.n : 0ull) + P.rec64[slot].index);
                };
                each_match(
                    [&](uint32_t bc, uint32_t slot) {
                        const uint64_t k = key(bc, slot);
                        return k >= lo && k < hi;
                    },
                    [&](uint32_t s, uint32_t bc, uint32_t slot) {
                        const uint32_t oy = ((bc >> 5) & 31u) == (uint32_t)y0, oz = (bc & 31u) == (uint32_t)z0;
                        if (s < DEP_HOT_LDS) keys[s] = (key(bc, slot) << 2) | (uint64_t)(oy << 1) | (uint64_t)oz;
                    });
                __syncthreads();
                const uint32_t c = sh_count;
                if (c > DEP_HOT_LDS) {
                    width >>= 1;
                    continue;
                }
                wg_sort_u64(keys, c);
                __syncthreads();
                for (uint32_t i = (uint32_t)tid; i < c; i += DEP_THREADS) {
                    const uint64_t k = keys[i];
                    const bool upper = (k >> 2) >= P.n;
                    const uint32_t p = (uint32_t)((k >> 2) - (upper ? P.n : 0ull));
                    int b;
                    double fx, fy, fz;
                    cic_axis(P.x[p] - P.pos_shift, g, b, fx);
                    cic_axis(P.y[p] - P.pos_shift, g, b, fy);
                    cic_axis(P.z[p] - P.pos_shift, g, b, fz);
                    const double mm = MASS ? P.masses[p] : P.uniform_mass;
                    const double term = mm * (upper ? fx : 1.0 - fx) * (k & 2u ? fy : 1.0 - fy) *
                                        (k & 1u ? fz : 1.0 - fz);
                    keys[i] = (uint64_t)__double_as_longlong(term);
                }
                __syncthreads();
                if (wave == 0) {
                    for (uint32_t c0 = 0; c0 < c; c0 += 64) {
                        const double term =
                            c0 + (uint32_t)lane < c ? __longlong_as_double((long long)keys[c0 + (uint32_t)lane]) : 0.0;
                        sum = wave_ordered_add(sum, term, (int)(c - c0 < 64u ? c - c0 : 64u));
                    }
                }
                lo = hi;
                if (c < DEP_HOT_LDS / 4) width <<= 1;
            }
            if (tid == 0) finish(x0, y0, z0, sum);
            continue;
        }

        // counting sort of the contributions by destination cell: corner o of a
        // record is cell c0 + ox sx + oy ez + oz of the box where it lies in it
        const int sx = ey * ez;
        uint32_t rank[PER][4];  // two 16-bit ranks per word (a list holds at most CAP)
        int cell0[PER];
        uint32_t corners[PER];  // bit o: corner o lies in the box
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t s = (uint32_t)(tid + j * DEP_THREADS);
            corners[j] = 0u;
            cell0[j] = 0;
            if (s < m) {
                const uint32_t cc = S.cell[s];
                const int cx = (int)(cc >> 10) - 1 - x0, cy = (int)((cc >> 5) & 31u) - 1 - y0,
                          cz = (int)(cc & 31u) - 1 - z0;
                cell0[j] = (cx * ey + cy) * ez + cz;
                const uint32_t mx = (cx >= 0 && cx < ex ? 0x0fu : 0u) | (cx + 1 < ex ? 0xf0u : 0u),
                               my = (cy >= 0 && cy < ey ? 0x33u : 0u) | (cy + 1 < ey ? 0xccu : 0u),
                               mz = (cz >= 0 && cz < ez ? 0x55u : 0u) | (cz + 1 < ez ? 0xaau : 0u);
                corners[j] = mx & my & mz;
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    const int c = cell0[j] + (o >> 2) * sx + ((o >> 1) & 1) * ez + (o & 1);
                    const uint32_t r = (corners[j] >> o) & 1u ? atomicAdd(&S.start[c], 1u) : 0u;
                    if (!DENSE && r >= (uint32_t)DEP_COMMON) sh_nheavy = 1u;
                    rank[j][o >> 1] = o & 1 ? rank[j][o >> 1] | (r << 16) : r;
                }
            }
        }
        __syncthreads();
        if constexpr (!DENSE) {
            if (sh_nheavy) {  // lists for whole waves
                leave(M > (uint32_t)DEP_CAP ? dep_split(M) : 0);
                return;
            }
        }
        wg_exclusive_scan_lds(S.start, cells + 1, sh_part);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t s = (uint32_t)(tid + j * DEP_THREADS);
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int c = cell0[j] + (o >> 2) * sx + ((o >> 1) & 1) * ez + (o & 1);
                if ((corners[j] >> o) & 1u)
                    S.ent[S.start[c] + ((rank[j][o >> 1] >> (16 * (o & 1))) & 0xffffu)] =
                        (uint16_t)(s * 8u + (uint32_t)o);
            }
        }
        __syncthreads();
        auto term_of = [&](uint16_t e) -> double {
            const uint32_t s = min((uint32_t)e >> 3, (uint32_t)CAP - 1u);  // empty network entries: any record
            const double fx = S.fx[s], fy = S.fy[s], fz = S.fz[s];
            double mm = P.uniform_mass;
            if constexpr (MASS) mm = sh_m[s];
            // weight f or 1 - f as |c - f| with c = 0 or 1 (exact alike)
            auto one_unless = [](uint32_t bit) {
                return __longlong_as_double((long long)((uint64_t)((bit - 1u) & 0x3ff00000u) << 32));
            };
            return mm * fabs(one_unless((e >> 2) & 1u) - fx) * fabs(one_unless((e >> 1) & 1u) - fy) *
                   fabs(one_unless(e & 1u) - fz);
        };
        // box cell -> tile coordinates (edges are powers of two when TE is)
        const int lgz = __ffs(ez) - 1, lgy = __ffs(ey) - 1;
        auto finish_cell = [&](int c, double sum) {
            if constexpr (TE > 0 && (TE & (TE - 1)) == 0)
                finish(x0 + (c >> (lgz + lgy)), y0 + ((c >> lgz) & (ey - 1)), z0 + (c & (ez - 1)), sum);
            else
                finish(x0 + c / (ey * ez), y0 + (c / ez) % ey, z0 + c % ez, sum);
        };
        // Two neighbouring cells per thread: their lists are adjacent, so one
        // network orders both (the cell as the key's top bit) and the chain of
        // dependent LDS reads is paid once for the pair.
#pragma unroll 1
        for (int p0 = 64 * wave; 2 * p0 < cells; p0 += DEP_THREADS) {  // whole waves: the ballots below
            const int c = 2 * (p0 + lane);
            uint32_t b0 = 0, b1 = 0, b2 = 0;
            if (c < cells) {
                b0 = S.start[c];
                b1 = S.start[c + 1];
                b2 = c + 1 < cells ? S.start[c + 2] : b1;
            }
            const bool heavy0 = DENSE && b1 - b0 > (uint32_t)DEP_SERIAL, heavy1 = DENSE && b2 - b1 > (uint32_t)DEP_SERIAL;
            if (heavy0) sh_heavy[atomicAdd(&sh_nheavy, 1u)] = (uint16_t)c;
            if (heavy1) sh_heavy[atomicAdd(&sh_nheavy, 1u)] = (uint16_t)(c + 1);
            const uint32_t first = heavy0 ? b1 : b0, n = (heavy1 ? b1 : b2) - first;
            double sum0 = 0.0, sum1 = 0.0;
            // entries [at0, at0 + n) of a list, at most N in every lane, the first
            // n0 of the pair's first cell: network of N keys (cell of the pair,
            // phase, index, entry; empty ones last), held as the bits of positive
            // normal binary64 numbers, which order alike and compare and exchange
            // in two instructions
            auto network = [&](auto size, uint32_t at0, uint32_t n) {
                constexpr int N = decltype(size)::value;
                const uint32_t n0 = at0 < b1 ? min(n, b1 - at0) : 0u;
                double k[N];
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    // read whether or not the entry exists (within the arrays): the
                    // reads of all entries go out together
                    const uint32_t at = at0 + (uint32_t)i;
                    const uint32_t v = S.ent[min(at, 8u * CAP - 1u)];
                    const uint32_t index = S.idx[min(v >> 3, (uint32_t)CAP - 1u)];
                    const uint32_t top = 0x00100000u | (at >= b1 ? 1u << 18 : 0u) | ((v & 4u) << 14) | (index >> 16);
                    const uint64_t key = ((uint64_t)((uint32_t)i < n ? top : 0x7fe00000u) << 32) | (index << 16) | v;
                    k[i] = __longlong_as_double((long long)key);
                }
                // Batcher's odd-even merge sort
#pragma unroll
                for (int p = 1; p < N; p *= 2)  // any N: comparators past it fall away
#pragma unroll
                    for (int q = p; q >= 1; q /= 2)
#pragma unroll
                        for (int j = q % p; j + q < N; j += 2 * q)
#pragma unroll
                            for (int i = 0; i < q; ++i)
                                if (i + j + q < N && (i + j) / (2 * p) == (i + j + q) / (2 * p)) {
                                    const double x = k[i + j], y = k[i + j + q];
                                    k[i + j] = min_f64(x, y);
                                    k[i + j + q] = max_f64(x, y);
                                }
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    // + 0.0 leaves a sum as it is (no sum is -0.0)
                    const double t = term_of((uint16_t)__double_as_longlong(k[i]));
                    sum0 += (uint32_t)i < n0 ? t : 0.0;
                    sum1 += (uint32_t)i >= n0 && (uint32_t)i < n ? t : 0.0;
                    // two records' fractions in registers at a time
                    if (i & 1) __builtin_amdgcn_sched_barrier(0);
                }
            };
            using I2 = std::integral_constant<int, 2>;
            using I4 = std::integral_constant<int, 4>;
            using I6 = std::integral_constant<int, 6>;
            using I8 = std::integral_constant<int, 8>;
            using I16 = std::integral_constant<int, DEP_SERIAL>;
            if (!__ballot(n > 2)) {
                network(I2{}, first, n);
            } else if (!__ballot(n > 4)) {
                network(I4{}, first, n);
            } else if (!__ballot(n > 6)) {
                network(I6{}, first, n);
            } else if (!__ballot(n > 8)) {
                network(I8{}, first, n);
            } else {
#pragma unroll 1
                for (int h = 0; h < 2; ++h) {  // one cell at a time
                    const uint32_t at = h ? b1 : first, nh = h ? first + n - b1 : b1 - first;
                    if (!DENSE || !__ballot(nh > 8)) network(I8{}, at, nh);
                    else if constexpr (DENSE) network(I16{}, at, nh);
                }
            }
            if constexpr (!DENSE) {
                // an even edge: the pair lies in one row and c < cells throughout
                if (!P.raw) {
                    sa_acc_add(win, P.sa, box_digits, sum0);
                    sa_acc_add(win, P.sa, box_digits, sum1);
                }
                typedef double D2 __attribute__((ext_vector_type(2), aligned(16)));
                const D2 out = {contrast_of(sum0, P), contrast_of(sum1, P)};
                const int lx = c / (TT * TT), ly = (c / TT) % TT, lz = c % TT;
                if (c < cells)
                    *reinterpret_cast<D2*>(&mesh[(uint64_t)(uint32_t)(lx * g.N + ly) * (uint64_t)g.N + (uint32_t)lz]) = out;
            } else {
                if (c < cells && !heavy0) finish_cell(c, sum0);
                if (c + 1 < cells && !heavy1) finish_cell(c + 1, sum1);
            }
        }
        __syncthreads();
        const uint32_t nheavy = DENSE ? sh_nheavy : 0u;
        if (nheavy) {
            // Rank of every record by particle index (the base cells are done
            // with): each thread's records against all, sixteen indices per
            // trip in flight, padded with the largest.
            const uint32_t m16 = (m + 15u) & ~15u;
            if ((uint32_t)tid < m16 - m) S.idx[m + (uint32_t)tid] = 0xffffffffu;
            __syncthreads();
            uint32_t mine[PER], r[PER];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const uint32_t s = (uint32_t)(tid + j * DEP_THREADS);
                mine[j] = s < m ? S.idx[s] : 0u;
                r[j] = 0u;
            }
            typedef uint32_t U4 __attribute__((ext_vector_type(4)));
            const U4* all = reinterpret_cast<const U4*>(S.idx);
            for (uint32_t t = 0; t < m16 / 4u; t += 4) {
                const U4 q[4] = {all[t], all[t + 1], all[t + 2], all[t + 3]};
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int j = 0; j < PER; ++j)
                        r[j] += (q[k].x < mine[j] ? 1u : 0u) + (q[k].y < mine[j] ? 1u : 0u) +
                                (q[k].z < mine[j] ? 1u : 0u) + (q[k].w < mine[j] ? 1u : 0u);
            }
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const uint32_t s = (uint32_t)(tid + j * DEP_THREADS);
                if (s < m) S.cell[s] = (uint16_t)r[j];
            }
            __syncthreads();
        }
        for (uint32_t h = (uint32_t)wave; h < nheavy; h += DEP_THREADS / 64) {
            const int c = sh_heavy[h];
            const uint32_t b = S.start[c], n = S.start[c + 1] - b;  // at most DEP_CAP: one corner per record
            uint32_t* bits = sh_bits[wave];
            auto place = [&](uint16_t e) -> uint32_t {
                return (e & 4 ? 32u * (DEP_BITS / 2) : 0u) + S.cell[e >> 3];
            };
            if (lane < DEP_BITS) bits[lane] = 0u;
            __threadfence_block();
            __builtin_amdgcn_wave_barrier();
            uint16_t mine[(DEP_CAP + 63) / 64];
#pragma unroll
            for (int q = 0; q < (DEP_CAP + 63) / 64; ++q) {
                const uint32_t i = (uint32_t)(lane + 64 * q);
                if (i < n) {
                    mine[q] = S.ent[b + i];
                    const uint32_t at = place(mine[q]);
                    atomicOr(&bits[at >> 5], 1u << (at & 31u));
                }
            }
            __threadfence_block();
            __builtin_amdgcn_wave_barrier();
            const uint32_t word = lane < DEP_BITS ? bits[lane] : 0u;
            const uint32_t below = wave_incl_scan_u32((uint32_t)__popc(word)) - (uint32_t)__popc(word);
#pragma unroll
            for (int q = 0; q < (DEP_CAP + 63) / 64; ++q) {
                if (64u * q >= n) break;  // uniform
                const bool have = (uint32_t)(lane + 64 * q) < n;
                const uint32_t at = have ? place(mine[q]) : 0u;
                const uint32_t w = __shfl(word, (int)(at >> 5)), w0 = __shfl(below, (int)(at >> 5));
                if (have) S.ent[b + w0 + (uint32_t)__popc(w & ((1u << (at & 31u)) - 1u))] = mine[q];
            }
            __threadfence_block();
            __builtin_amdgcn_wave_barrier();
            double sum = 0.0;
            for (uint32_t c0 = 0; c0 < n; c0 += 64) {
                const double term = c0 + (uint32_t)lane < n ? term_of(S.ent[b + c0 + (uint32_t)lane]) : 0.0;
                sum = wave_ordered_add(sum, term, (int)(n - c0 < 64u ? n - c0 : 64u));
            }
            if (lane == 0) finish_cell(c, sum);
        }
        if constexpr (!DENSE) break;
    }
    if constexpr (DENSE) {
        // the workgroup's digits summed in LDS, one atomic per digit and job
        if (tid < 6) sh_digits[tid] = 0ull;
        __syncthreads();
        uint64_t v[6];
        sa_acc_digits(win, P.sa, v);
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (v[j]) atomicAdd(&sh_digits[j], (unsigned long long)v[j]);
        }
        __syncthreads();
        if (tid < 6 && P.sa.base + tid < SA_DIGITS && sh_digits[tid])
            atomicAdd(&box_digits[P.sa.base + tid], sh_digits[tid]);
    } else {
        sa_acc_flush(win, P.sa, wave_out);
        return;  // one tile per workgroup
    }
    }
}

// ---------------------------------------------------------------------------
// Binary32 deposit: fixed-point accumulation in LDS.
//
// Each CIC contribution m*wx*wy*wz is converted to an unsigned integer in
// units of 2^-32 of the mass unit (the uniform particle mass, or the largest
// explicit mass) and added with an integer LDS atomic.  Integer addition is
// associative, so every cell sum is bit-identical whatever the scheduling: the
// deposit is deterministic without a per-cell order and without float
// atomics.  The resolution (2^-32 of a particle mass per contribution) is far
// below binary32 rounding; a cell holds up to 2^31 particle masses.
// ---------------------------------------------------------------------------
constexpr int DEPFX_THREADS = 512;
constexpr int DEPFX_MAX_CELLS = DEP_MAX_T * DEP_MAX_T * DEP_MAX_T;

struct DepFxParams {
    DepParams base;
    double mass_unit;               // uniform mass, or max explicit mass
    double fixed_to_mass;           // mass_unit * 2^-32
    const DepRecord* rec;           // deposit records by bucket
    const float* rec_mass;          // explicit masses / mass_unit, as rec (or null)
    const uint32_t* start;          // nb+1: first slot of each bucket (dense offsets or a capacity layout)
    const uint32_t* counts;         // records per bucket
    const uint32_t* ovf_start;      // nb+1 prefix of the overflow records (or null: none)
    uint64_t nb;                    // buckets over all boxes (start[nb] = first overflow slot)
};

// The 27 buckets that feed a tile: its own eight classes, then the 19
// neighbour (d, c) slots 1..19 of range_slot.  Each gives a main range (its
// slots, at most its capacity) and an overflow range.
constexpr int DEPFX_BUCKETS = 27;
constexpr int DEPFX_NRANGES = 2 * DEPFX_BUCKETS;
static_assert(DEPFX_NRANGES <= 64, "one lane per range");

// The non-empty ranges in order: rs their first slot, rc the prefix of their
// counts (rc[DEPFX_NRANGES] = total), rd the neighbour offset d, *nranges
// their number; one global round trip, the first wave.
__device__ __forceinline__ void load_fx_ranges(const DepFxParams& Q, uint32_t box_base, int tx, int ty, int tz,
                                               int nT, uint32_t* rs, uint32_t* rc, uint8_t* rd,
                                               uint32_t* nranges) {
    const int t = threadIdx.x;
    if (t < 64) {
        uint32_t cnt = 0, rs_lane = 0;
        uint8_t rd_lane = 0;
        if (t < DEPFX_NRANGES) {
            const int j = t % DEPFX_BUCKETS;
            const bool ovf = t >= DEPFX_BUCKETS;
            int d = 0, cls = j;
            if (j >= 8) {
                const RangeSlot sl = range_slot(j - 7);
                d = sl.d;
                cls = sl.c;
            }
            const int sx = (tx - ((d >> 2) & 1) + nT) % nT, sy = (ty - ((d >> 1) & 1) + nT) % nT,
                      sz = (tz - (d & 1) + nT) % nT;
            const uint32_t b = box_base + (((uint32_t)sx * nT + sy) * nT + sz) * 8u + (uint32_t)cls;
            uint32_t first = 0;
            if (!ovf) {
                const uint32_t a = Q.start[b], e = Q.start[b + 1], c = Q.counts[b];
                first = a;
                cnt = c < e - a ? c : e - a;
            } else if (Q.ovf_start) {
                const uint32_t a = Q.ovf_start[b], e = Q.ovf_start[b + 1];
                first = Q.start[Q.nb] + a;
                cnt = e - a;
            }
            rs_lane = first;
            rd_lane = (uint8_t)d;
        }
        // the non-empty ranges, compacted in order: rc[0..R] is their count
        // prefix and rc[R..DEPFX_NRANGES] repeats the total
        const uint64_t live = __ballot(cnt != 0u);
        const uint32_t at = (uint32_t)__popcll(live & ((1ull << t) - 1ull));
        const uint32_t R = (uint32_t)__popcll(live);
        const uint32_t incl = wave_incl_scan_u32(cnt);
        if (cnt != 0u) {
            rs[at] = rs_lane;
            rd[at] = rd_lane;
            rc[at + 1] = incl;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        if (t == 0) rc[0] = 0;
        if ((uint32_t)t > R && t <= DEPFX_NRANGES) rc[t] = total;
        if (t == 0) *nranges = R;
    }
    __syncthreads();
}

// The range of record v: the last r < R with rc[r] <= v (binary search).
__device__ __forceinline__ int fx_range_of(const uint32_t* rc, uint32_t R, uint32_t v) {
    int lo = 0, hi = (int)R - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (rc[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// TE: compile-time tile edge (16, the edge of every mesh divisible by 16:
// cell index arithmetic becomes shifts), or 0 to read it from the geometry.
template <int TE>
__global__ void __launch_bounds__(DEPFX_THREADS) k_deposit_fixed(DepFxParams Q, float* __restrict__ mesh) {
    const DepParams& P = Q.base;
    __shared__ unsigned long long acc[DEPFX_MAX_CELLS];
    __shared__ uint32_t sh_rs[DEPFX_NRANGES], sh_rc[DEPFX_NRANGES + 1];
    __shared__ uint8_t sh_rd[DEPFX_NRANGES];
    __shared__ uint32_t sh_nr;

    const Geom& g = P.g;
    const int nT = g.nT;
    const int T = TE > 0 ? TE : g.T;
    const uint32_t ntiles = (uint32_t)nT * nT * nT;
    const uint32_t gtile = xcd_block(blockIdx.x, gridDim.x);  // box-major tile index
    if (gtile >= ntiles * g.nbox) return;
    const uint32_t box = gtile / ntiles, tile = gtile % ntiles;
    const int tz = tile % nT, ty = (tile / nT) % nT, tx = tile / (nT * nT);
    const int cells = T * T * T;
    mesh += (uint64_t)box * g.N * g.N * g.N;

    for (int c = threadIdx.x; c < cells; c += blockDim.x) acc[c] = 0ull;
    load_fx_ranges(Q, box * buckets_per_box(g), tx, ty, tz, nT, sh_rs, sh_rc, sh_rd, &sh_nr);
    const uint32_t M = sh_rc[DEPFX_NRANGES];
    const uint32_t nr = sh_nr;
    int r = threadIdx.x < M ? fx_range_of(sh_rc, nr, threadIdx.x) : 0;
    bool bad = false;
    // records in pairs: both loads are issued before the first atomic, so a
    // thread with two records waits for one memory round trip, not two
    for (uint32_t v0 = threadIdx.x; v0 < M; v0 += 2 * blockDim.x) {
        DepRecord recs[2];
        float ms[2];
        int ds[2];
        bool have[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t v = v0 + (uint32_t)h * blockDim.x;
            have[h] = v < M;
            if (have[h]) {
                while (sh_rc[r + 1] <= v) ++r;
                const uint32_t slot = sh_rs[r] + (v - sh_rc[r]);
                recs[h] = Q.rec[slot];
                ms[h] = Q.rec_mass ? Q.rec_mass[slot] : 1.0f;
                ds[h] = sh_rd[r];
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (!have[h]) continue;
            const DepRecord rec = recs[h];
            const int d = ds[h];
            const int c = (int)rec.cell;
            const int cz_ = c % T, cy_ = (c / T) % T, cx_ = c / (T * T);
            // a neighbour record sits just below this tile along its shifted axes
            const int lx = (d & 4) ? -1 : cx_;
            const int ly = (d & 2) ? -1 : cy_;
            const int lz = (d & 1) ? -1 : cz_;
            if (((d & 4) && cx_ != T - 1) || ((d & 2) && cy_ != T - 1) || ((d & 1) && cz_ != T - 1)) {
                bad = true;
                continue;
            }
            const float m = ms[h];
            const float wx[2] = {1.0f - rec.fx, rec.fx};
            const float wy[2] = {1.0f - rec.fy, rec.fy};
            const float wz[2] = {1.0f - rec.fz, rec.fz};
#pragma unroll
            for (int ox = 0; ox < 2; ++ox) {
                const int cx = lx + ox;
                if (cx < 0 || cx >= T) continue;
#pragma unroll
                for (int oy = 0; oy < 2; ++oy) {
                    const int cy = ly + oy;
                    if (cy < 0 || cy >= T) continue;
                    const float mxy = m * wx[ox] * wy[oy];
#pragma unroll
                    for (int oz = 0; oz < 2; ++oz) {
                        const int cz = lz + oz;
                        if (cz < 0 || cz >= T) continue;
                        const float w = mxy * wz[oz];
                        // signed 32.32 fixed point (two's complement sums wrap consistently)
                        const unsigned long long q = (unsigned long long)__float2ll_rn(w * 4294967296.0f);
                        atomicAdd(&acc[(cx * T + cy) * T + cz], q);
                    }
                }
            }
        }
    }
    if (bad) atomicOr(P.err, ERR_COORDINATE);
    __syncthreads();

    // the tile's exact mass: its cells' 32.32 integers summed as two 32-bit digit sums
    uint64_t dig0 = 0, dig1 = 0;
    if constexpr (TE > 0 && TE % 4 == 0) {
        // four z-adjacent cells per lane, one 16-byte store (a tile's z-runs
        // start at multiples of TE cells)
        typedef float F4 __attribute__((ext_vector_type(4)));
        for (int c4 = threadIdx.x; c4 < cells / 4; c4 += blockDim.x) {
            const int c = 4 * c4;
            const int lz = c % T, ly = (c / T) % T, lx = c / (T * T);
            float o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const long long q = (long long)acc[c + j];
                dig0 += (uint64_t)q & 0xffffffffull;
                dig1 += (uint64_t)q >> 32;
                o[j] = contrast_fp32((double)q * Q.fixed_to_mass, P);
            }
            const uint64_t gx = (uint64_t)(tx * T + lx), gy = (uint64_t)(ty * T + ly), gz = (uint64_t)(tz * T + lz);
            *reinterpret_cast<F4*>(&mesh[(gx * g.N + gy) * g.N + gz]) = F4{o[0], o[1], o[2], o[3]};
        }
    } else {
        for (int c = threadIdx.x; c < cells; c += blockDim.x) {
            const long long q = (long long)acc[c];
            dig0 += (uint64_t)q & 0xffffffffull;
            dig1 += (uint64_t)q >> 32;
            const double mcell = (double)q * Q.fixed_to_mass;
            const int lz = c % T, ly = (c / T) % T, lx = c / (T * T);
            const uint64_t gx = (uint64_t)(tx * T + lx), gy = (uint64_t)(ty * T + ly), gz = (uint64_t)(tz * T + lz);
            mesh[(gx * g.N + gy) * g.N + gz] = contrast_fp32(mcell, P);
        }
    }
    // each wave's two digit sums (below 2^41), for k_mass_finish_fixed
    static_assert(DEPFX_THREADS / 64 == SA_WAVES_PER_TILE, "one mass pair per wave");
    if (P.raw) dig0 = dig1 = 0;  // signed cells: no mass identity
    const uint64_t s0 = wave_sum_u64(dig0), s1 = wave_sum_u64(dig1);
    if (lane_id() == 0) {
        typedef unsigned long long U2 __attribute__((ext_vector_type(2)));
        *reinterpret_cast<U2*>(P.mass_waves + ((uint64_t)gtile * SA_WAVES_PER_TILE + threadIdx.x / 64) * 2) =
            U2{s0, s1};
    }
}

// Zero fill (used instead of memset nodes in code that callers may capture
// into a HIP graph).
__global__ void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t value) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

// Step factors written on the stream ahead of a graph replay.
__global__ void k_set_factors(double* __restrict__ f, double k_prev, double k_next, double d_next) {
    if (threadIdx.x == 0) {
        f[0] = k_prev;
        f[1] = k_next;
        f[2] = d_next;
    }
}

// The exact sum held by the digit counters d (LDS, SA_DIGITS + 2 words, each
// below 2^62), rounded once to nearest with ties to even; the first wave calls
// it, d is normalised in place and lane 0 holds the result.  The carry chain
// runs over the digits in use only (a handful: the masses of a box lie within
// a few binary orders of each other).
__device__ __forceinline__ double sa_round(unsigned long long* d) {
    constexpr int ND = SA_DIGITS + 2;
    const int lane = (int)lane_id();
    const uint64_t m0 = __ballot(d[lane] != 0ull);
    const uint64_t m1 = __ballot(lane < SA_DIGITS - 64 && d[64 + lane] != 0ull);
    if (!(m0 | m1)) return 0.0;
    double out = 0.0;
    if (lane == 0) {
        const int first = m0 ? __ffsll((unsigned long long)m0) - 1 : 64 + __ffsll((unsigned long long)m1) - 1;
        const int last = m1 ? 127 - __clzll(m1) : 63 - __clzll(m0);
        d[SA_DIGITS] = d[SA_DIGITS + 1] = 0ull;
        uint64_t carry = 0;
        int end = first;  // one past the highest digit written
        for (int i = first; i < ND && (i <= last || carry); ++i) {
            const uint64_t sum = d[i] + carry;
            d[i] = sum & 0xffffffffull;
            carry = sum >> 32;
            end = i + 1;
        }
        int top = -1;
        for (int i = end - 1; i >= first && top < 0; --i)
            if (d[i]) top = i * 32 + (31 - __clz((uint32_t)d[i]));
        auto digit = [&](int i) -> uint64_t { return i >= first && i < end ? d[i] : 0ull; };
        // bits [lo, lo + 64) of the sum
        auto bits64 = [&](int lo) -> uint64_t {
            const int i = lo >> 5, o = lo & 31;
            const uint64_t v = digit(i) >> o | digit(i + 1) << (32 - o);
            return o ? v | digit(i + 2) << (64 - o) : v;
        };
        if (top < 53) {
            out = ldexp((double)(bits64(0) & ((1ull << 53) - 1ull)), -1074);
        } else {
            const int lo = top - 52, r = lo - 1;  // r: the rounding bit
            uint64_t m = bits64(lo) & ((1ull << 53) - 1ull);
            const uint32_t rd = (uint32_t)digit(r >> 5);
            bool sticky = (rd & ((1u << (r & 31)) - 1u)) != 0u;
            for (int i = first; i < (r >> 5) && !sticky; ++i) sticky = d[i] != 0ull;
            if (((rd >> (r & 31)) & 1u) && (sticky || (m & 1ull))) ++m;
            out = ldexp((double)m, lo - 1074);
        }
    }
    return out;
}

// Last workgroup of a grid row to arrive at ticket (reset for the next launch);
// its later reads see what the others wrote before arriving.
__device__ __forceinline__ bool last_block(uint32_t* ticket) {
    __shared__ uint32_t arrived;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        arrived = atomicAdd(ticket, 1u);
        if (arrived == gridDim.x - 1) atomicExch(ticket, 0u);
    }
    __syncthreads();
    const bool last = arrived == gridDim.x - 1;
    if (last) __threadfence();
    return last;
}

// Takes a box's digit counters (SA_WORDS words) into LDS and clears them for the
// next deposit; the flag word's value to flag.  The whole workgroup.
__device__ __forceinline__ void sa_take(unsigned long long* d, unsigned long long* cnt, unsigned long long* flag) {
    for (int w = threadIdx.x; w < SA_WORDS; w += blockDim.x) {
        const unsigned long long v = atomicExch(&d[w], 0ull);
        if (w < SA_DIGITS) cnt[w] = v;
        else *flag = v;
    }
    __syncthreads();
}

// Deposit status on the device, so that calls which do not synchronise stay
// fail-closed: the routing-count identity of the x-plane bins
// (src/mesh/mass_assignment_deposit.inc:269-284: every particle routed exactly
// once) and the mass-conservation bound of src/math/cic_mass_conservation.cpp:
// 25-63 per box, |deposited - input| <= tol_factor * max(input, deposited)
// with a finite positive deposited mass.
struct DepositCheck {
    const uint32_t* grand_total;  // routed particles
    uint64_t n;
    double input_per_box, tol_factor;
    int check;                    // 0: sums only
    uint32_t* err;
};

__device__ __forceinline__ void deposit_check(const DepositCheck& c, uint32_t box, double dep) {
    if (!c.check) return;
    uint32_t bits = 0;
    if (box == 0 && (uint64_t)*c.grand_total != c.n) bits |= ERR_ROUTING;
    const double scale = dep > c.input_per_box ? dep : c.input_per_box;
    if (!isfinite(dep) || !(dep > 0.0) || fabs(dep - c.input_per_box) > c.tol_factor * scale)
        bits |= ERR_MASS_CONSERVATION;
    if (bits) atomicOr(c.err, bits);
}

// Per box (grid row): the deposit's mass records added up, the box's exact mass
// rounded (NaN when a cell was not a finite non-negative number) and checked
// by the row's last workgroup.  One launch in place of the former reduction,
// one-thread rounding (15 to 40 us over a private digit array) and status
// kernels.  Integer sums: exact whatever the order.
// Binary64: the waves' digit windows, those of nearby bases in a thread's
// registers first, then LDS counters, then one atomic per non-zero counter
// and workgroup.
__global__ void __launch_bounds__(256) k_mass_finish(const unsigned long long* __restrict__ waves,
                                                     uint64_t waves_per_box, unsigned long long* digits,
                                                     uint32_t* tickets, double* __restrict__ mass_total,
                                                     DepositCheck chk) {
    __shared__ unsigned long long cnt[SA_DIGITS + 2];
    __shared__ unsigned long long flag;
    const uint64_t box = blockIdx.y;
    for (int w = threadIdx.x; w < SA_DIGITS; w += blockDim.x) cnt[w] = 0ull;
    __syncthreads();
    constexpr int AW = SA_WAVE_WIN + 2;
    long long tb = -1;
    uint64_t acc[AW];
#pragma unroll
    for (int j = 0; j < AW; ++j) acc[j] = 0ull;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < waves_per_box;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const unsigned long long* ww = waves + (box * waves_per_box + t) * SA_WAVE_WORDS;
        const long long b = (long long)ww[0];
        if (b < 0) continue;
        if (tb < 0) tb = b;
        const long long k = b - tb;
        if (k >= 0 && k <= 2) {
#pragma unroll
            for (int j = 0; j < SA_WAVE_WIN; ++j) {
                const uint64_t v = ww[1 + j];
#pragma unroll
                for (int o = 0; o <= 2; ++o)
                    if (k == o) acc[j + o] += v;
            }
        } else {
            for (int j = 0; j < SA_WAVE_WIN; ++j) {
                const unsigned long long v = ww[1 + j];
                if (v && b + j < SA_DIGITS) atomicAdd(&cnt[b + j], v);
            }
        }
    }
    if (tb >= 0) {
#pragma unroll
        for (int j = 0; j < AW; ++j)
            if (acc[j] && tb + j < SA_DIGITS) atomicAdd(&cnt[tb + j], (unsigned long long)acc[j]);
    }
    __syncthreads();
    unsigned long long* d = digits + box * SA_WORDS;
    for (int w = threadIdx.x; w < SA_DIGITS; w += blockDim.x)
        if (cnt[w]) atomicAdd(&d[w], cnt[w]);
    if (!last_block(&tickets[box])) return;
    sa_take(d, cnt, &flag);
    if (threadIdx.x >= 64) return;
    const double total = sa_round(cnt);
    if (threadIdx.x == 0) {
        const double dep = flag ? __builtin_nan("") : total;
        mass_total[box] = dep;
        deposit_check(chk, (uint32_t)box, dep);
    }
}

// Binary32: the waves' digit-sum pairs (s0, s1) added up per workgroup (a 1024^3
// mesh has 2^21 waves of under 2^41 each, so any grid's sums stay below 2^62), and
// the workgroup's exact total (s0 + s1 2^32) * unit * 2^-32 added to the box's counters
// as digits.
__global__ void __launch_bounds__(256) k_mass_finish_fixed(const unsigned long long* __restrict__ waves,
                                                           uint64_t waves_per_box, double unit,
                                                           unsigned long long* digits, uint32_t* tickets,
                                                           double* __restrict__ mass_total, DepositCheck chk) {
    __shared__ uint64_t part[2][4];
    __shared__ unsigned long long cnt[SA_DIGITS + 2];
    __shared__ unsigned long long flag;
    const uint64_t box = blockIdx.y;
    typedef unsigned long long U2 __attribute__((ext_vector_type(2)));
    uint64_t s0 = 0, s1 = 0;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < waves_per_box;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const U2 v = *reinterpret_cast<const U2*>(waves + (box * waves_per_box + t) * 2);
        s0 += v.x;
        s1 += v.y;
    }
    s0 = wave_sum_u64(s0);
    s1 = wave_sum_u64(s1);
    if (lane_id() == 0) {
        part[0][threadIdx.x / 64] = s0;
        part[1][threadIdx.x / 64] = s1;
    }
    __syncthreads();
    unsigned long long* d = digits + box * SA_WORDS;
    if (threadIdx.x == 0) {
        uint64_t a0 = 0, a1 = 0;
        for (int w = 0; w < (int)blockDim.x / 64; ++w) {
            a0 += part[0][w];
            a1 += part[1][w];
        }
        const uint64_t q0 = a0 + (a1 << 32);
        const uint64_t q1 = (a1 >> 32) + (q0 < a0 ? 1ull : 0ull);
        int limb = 0;
        uint32_t dig[SA_WAVE_WIN];
        if (!sa_fixed_digits(q0, q1, unit, limb, dig)) {
            atomicOr(&d[SA_DIGITS], 1ull);
        } else {
            for (int k = 0; k < SA_WAVE_WIN; ++k)
                if (dig[k] && limb + k < SA_DIGITS) atomicAdd(&d[limb + k], (unsigned long long)dig[k]);
        }
    }
    if (!last_block(&tickets[box])) return;
    sa_take(d, cnt, &flag);
    if (threadIdx.x >= 64) return;
    const double total = sa_round(cnt);
    if (threadIdx.x == 0) {
        const double dep = flag ? __builtin_nan("") : total;
        mass_total[box] = dep;
        deposit_check(chk, (uint32_t)box, dep);
    }
}

// Exact sum and maximum of explicit particle masses (out[0], out[1]; the sum
// is NaN when a mass is not a finite non-negative number): the input-mass
// identity of src/gravity/pm_solver.cpp:120-130, rounded once.  Each mass is
// three 32-bit digits from its limb; a thread keeps six digit sums from one
// limb below its first mass, which takes masses within a factor 2^64 of each
// other, and other masses go to LDS counters.  Bound by the atomics, not by the
// read: 256 threads meet at the same few LDS words after about eleven masses each,
// and the workgroups at the same few global ones (3M masses 75 us, 0.32 TB/s; the
// host pass that it replaces copied them and took 9.4 ms).
__global__ void __launch_bounds__(256) k_input_mass(uint64_t n, const double* __restrict__ m,
                                                    unsigned long long* digits, unsigned long long* max_bits,
                                                    uint32_t* ticket, double* __restrict__ out) {
    __shared__ unsigned long long cnt[SA_DIGITS + 2];
    __shared__ unsigned long long flag;
    for (int w = threadIdx.x; w < SA_DIGITS + 2; w += blockDim.x) cnt[w] = 0ull;
    __syncthreads();
    constexpr int AW = 6;
    uint64_t acc[AW];
#pragma unroll
    for (int j = 0; j < AW; ++j) acc[j] = 0ull;
    int tb = -1;
    double mx = 0.0;
    bool bad = false;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const double x = m[i];
        if (!isfinite(x) || x < 0.0) {
            bad = true;
            continue;
        }
        if (x == 0.0) continue;
        mx = x > mx ? x : mx;
        const uint64_t bits = (uint64_t)__double_as_longlong(x);
        const int e = (int)((bits >> 52) & 0x7ff);
        const uint64_t frac = bits & ((1ull << 52) - 1ull);
        const uint64_t mant = e ? (frac | (1ull << 52)) : frac;
        const int shift = e ? e - 1 : 0, limb = shift >> 5, off = shift & 31;
        const uint64_t lo = mant << off, hi = off ? mant >> (64 - off) : 0ull;
        if (tb < 0) tb = limb > 0 ? limb - 1 : 0;
        const int k = limb - tb;
        if (k >= 0 && k <= 3) {
#pragma unroll
            for (int o = 0; o <= 3; ++o) {
                if (k == o) {
                    acc[o] += (uint32_t)lo;
                    acc[o + 1] += lo >> 32;
                    acc[o + 2] += hi;
                }
            }
        } else {
            atomicAdd(&cnt[limb], (unsigned long long)(uint32_t)lo);
            if (limb + 1 < SA_DIGITS) atomicAdd(&cnt[limb + 1], (unsigned long long)(lo >> 32));
            if (limb + 2 < SA_DIGITS) atomicAdd(&cnt[limb + 2], (unsigned long long)hi);
        }
    }
    if (tb >= 0) {
#pragma unroll
        for (int j = 0; j < AW; ++j)
            if (acc[j] && tb + j < SA_DIGITS) atomicAdd(&cnt[tb + j], (unsigned long long)acc[j]);
    }
    // non-negative binary64 numbers order as their bits do
    if (mx > 0.0) atomicMax(&cnt[SA_DIGITS], (unsigned long long)__double_as_longlong(mx));
    if (bad) atomicOr(&cnt[SA_DIGITS + 1], 1ull);
    __syncthreads();
    for (int w = threadIdx.x; w < SA_DIGITS; w += blockDim.x)
        if (cnt[w]) atomicAdd(&digits[w], cnt[w]);
    if (threadIdx.x == 0) {
        if (cnt[SA_DIGITS + 1]) atomicOr(&digits[SA_DIGITS], 1ull);
        atomicMax(max_bits, cnt[SA_DIGITS]);
    }
    if (!last_block(ticket)) return;
    sa_take(digits, cnt, &flag);
    if (threadIdx.x >= 64) return;
    const double total = sa_round(cnt);
    if (threadIdx.x == 0) {
        out[0] = flag ? __builtin_nan("") : total;
        out[1] = __longlong_as_double((long long)atomicExch(max_bits, 0ull));
    }
}

// ===========================================================================
// Fused centered-gradient gather + kick/drift
// ===========================================================================
// Block schedule for particle arrays stored in Lagrangian lattice order
// p = (ix*S + iy)*S + iz (the order of lattice initial conditions, which
// particles keep for the whole run).  Consecutive logical blocks walk a
// TX x TY column of lattice rows (all z) before the next column, so the blocks
// resident on one XCD touch a compact region of the potential that stays in
// its L2.  S == 0: identity.  S a multiple of 256: a block is one 256-particle
// chunk of a z-row (ZC of them per row, TX and TY divide S).  Otherwise (WC > 0) a
// wave is one 64-particle chunk (WC per row, the last one short) and the
// columns at the upper edges are narrower.
struct LatticeTiling {
    uint32_t S, TX, TY, ZC;  // lattice side, column tile, 256-chunks per z-row
    int lS, lTX, lTY, lZC;   // log2 of each when all four are powers of two, else lS < 0
    uint32_t WC;             // 64-chunks per z-row, or 0
};

// Particle of this thread (256-thread blocks) under the wave-chunk schedule;
// past the row or the lattice: n.
__device__ __forceinline__ uint64_t lattice_wave_particle(uint32_t block, const LatticeTiling& t, uint64_t n) {
    const uint32_t unit = block * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (unit >= t.S * t.S * t.WC) return n;
    const uint32_t strip = t.TX * t.S * t.WC;
    const uint32_t tx = unit / strip, u = unit % strip;
    const uint32_t wx = t.S - tx * t.TX < t.TX ? t.S - tx * t.TX : t.TX;
    const uint32_t tile = wx * t.TY * t.WC;
    const uint32_t ty = u / tile, w = u % tile;
    const uint32_t wy = t.S - ty * t.TY < t.TY ? t.S - ty * t.TY : t.TY;
    const uint32_t row = w / t.WC;
    const uint32_t iz = (w - row * t.WC) * 64u + lane_id();
    if (iz >= t.S) return n;
    const uint32_t ix = tx * t.TX + row / wy, iy = ty * t.TY + row % wy;
    return ((uint64_t)ix * t.S + iy) * t.S + iz;
}

__device__ __forceinline__ uint32_t lattice_block(uint32_t L, const LatticeTiling& t) {
    if (t.S == 0) return L;
    if (t.lS >= 0) {  // powers of two: shifts and masks
        const int lper = t.lTX + t.lTY + t.lZC;
        const uint32_t tile = L >> lper, w = L & ((1u << lper) - 1u);
        const int ltiles_y = t.lS - t.lTY;
        const uint32_t tx = tile >> ltiles_y, ty = tile & ((1u << ltiles_y) - 1u);
        const uint32_t zc = w & ((1u << t.lZC) - 1u), dy = (w >> t.lZC) & ((1u << t.lTY) - 1u);
        const uint32_t dx = w >> (t.lZC + t.lTY);
        const uint32_t ix = (tx << t.lTX) + dx, iy = (ty << t.lTY) + dy;
        return (((ix << t.lS) + iy) << t.lZC) + zc;
    }
    // every quantity is below S^2 * ZC = n / 256 < 2^32
    const uint32_t per_tile = t.TX * t.TY * t.ZC;
    const uint32_t tile = L / per_tile, w = L % per_tile;
    const uint32_t tiles_y = t.S / t.TY;
    const uint32_t tx = tile / tiles_y, ty = tile % tiles_y;
    const uint32_t zc = w % t.ZC, dy = (w / t.ZC) % t.TY, dx = w / (t.ZC * t.TY);
    const uint32_t ix = tx * t.TX + dx, iy = ty * t.TY + dy;
    return (ix * t.S + iy) * t.ZC + zc;
}

template <typename T, typename PT>
struct GatherArgs {
    Geom g;
    uint64_t n;
    const T* phi;               // R after the c2r pass
    const double* x_in;
    const double* y_in;
    const double* z_in;
    double* x_out;
    double* y_out;
    double* z_out;
    const PT* px_in;
    const PT* py_in;
    const PT* pz_in;
    PT* px_out;
    PT* py_out;
    PT* pz_out;
    double* acc_x;              // optional: acc += g (force mode)
    double* acc_y;
    double* acc_z;
    T* g_x;                     // optional: g written (transactional force mode)
    T* g_y;
    T* g_z;
    LatticeTiling lat;          // block schedule over the Lagrangian lattice (or identity)
    uint32_t* next_counts;      // optional: bucket counts/ranks of the drifted positions
    uint32_t* next_keys;        // keys and ranks per particle, or with rec_out the overflow
    uint32_t* next_ranks;       // list's bucket and rank per entry
    const uint32_t* rec_start;  // (binary32) the drifted positions' deposit records are written into
    DepRecord* rec_out;         // the capacity layout rec_start (nb+1 prefix); those past a bucket's
    uint32_t* ovf_count;        // capacity are appended to the overflow list (ovf_rec, next_keys,
    DepRecord* ovf_rec;         // next_ranks)
    const double* dfac;         // optional: k_prev, k_next, d_next read from device memory
                                // (graph replays take new factors without re-capture)
    double k_prev;              // K2 of the previous step
    double k_next;              // K1 of the next step
    double d_next;              // drift factor of the next step
    int has_prev;
    int has_next;
    uint32_t* err;
    const uint32_t* gate;       // do nothing where this word is set (another than err), or null
};

// Potential values of the 8 corners' centred differences around base cell
// (ix, iy, iz).  O32: the box's mesh spans at most 2^32 bytes, so the stencil uses
// 32-bit byte offsets from phi (a scalar base where phi is wave-uniform).
template <typename T, bool O32>
__device__ __forceinline__ void load_stencil(const T* phi, int N, int ix, int iy, int iz, T (&X)[4][2][2],
                                             T (&Y)[2][2][2], T (&Z)[2][2][2]) {
    // The 8 corners' centred differences touch 32 distinct potential
    // values: the x stencil X[k][b][c] at (ix-1+k, iy+b, iz+c), and the
    // y / z stencil ends Y[j][a][c] at (ix+a, iy-1 / iy+2, iz+c) and
    // Z[j][a][b] at (ix+a, iy+b, iz-1 / iz+2).  All 32 loads are
    // issued before any arithmetic.
    using Off = typename std::conditional<O32, uint32_t, uint64_t>::type;
    const Off NN = (Off)N * (Off)N;
    const Off es = O32 ? (Off)sizeof(T) : (Off)1;  // offsets in bytes (O32) or elements
    auto ld = [&](Off o) -> T {
        if constexpr (O32) return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(phi) + o);
        else return phi[o];
    };
    Off xo[4], yo[4], zo[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        xo[k] = (Off)wrap_cell(ix - 1 + k, N) * NN * es;
        yo[k] = (Off)wrap_cell(iy - 1 + k, N) * (Off)N * es;
        zo[k] = (Off)wrap_cell(iz - 1 + k, N) * es;
    }
    // The stencil as 12 z-contiguous runs: the (ix+a, iy+b) lines hold
    // iz-1..iz+2 (x and z stencils), the x-end and y-end lines
    // iz..iz+1.  A run that does not wrap in z is one vector load.
    typedef T V4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    auto run = [&](Off xy, int z0, T* dst, int cnt) {
        if (z0 >= 0 && z0 + cnt <= N) {
            const Off o = xy + (Off)z0 * es;
            const char* src = O32 ? reinterpret_cast<const char*>(phi) + o
                                  : reinterpret_cast<const char*>(phi + o);
            if (cnt == 4) {
                const V4 v = *reinterpret_cast<const V4*>(src);
                dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
            } else {
                const V2 v = *reinterpret_cast<const V2*>(src);
                dst[0] = v.x; dst[1] = v.y;
            }
        } else {
            for (int c = 0; c < cnt; ++c) dst[c] = ld(xy + (Off)wrap_cell(z0 + c, N) * es);
        }
    };
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            T q[4];
            run(xo[u + 1] + yo[b + 1], iz - 1, q, 4);
            Z[0][u][b] = q[0];
            X[u + 1][b][0] = q[1];
            X[u + 1][b][1] = q[2];
            Z[1][u][b] = q[3];
        }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        run(xo[0] + yo[b + 1], iz, X[0][b], 2);
        run(xo[3] + yo[b + 1], iz, X[3][b], 2);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int u = 0; u < 2; ++u) run(xo[u + 1] + yo[j * 3], iz, Y[j][u], 2);
}

// Centred-gradient force at one particle: base cell (ix, iy, iz), corner weights
// w[0] = 1 - f, w[1] = f per axis, phi its box's potential (load_stencil).
// Returns whether a non-zero product was lost.
template <typename T, bool O32>
__device__ __forceinline__ bool stencil_force(const T* phi, const Geom& g, int ix, int iy, int iz,
                                              const T (&wx)[2], const T (&wy)[2], const T (&wz)[2], T& gx, T& gy,
                                              T& gz) {
    T X[4][2][2], Y[2][2][2], Z[2][2][2];
    load_stencil<T, O32>(phi, g.N, ix, iy, iz, X, Y, Z);
    // -(f+ - f-) / (2 dx); when dx is a power of two the quotient equals
    // the product with the exact reciprocal bit for bit
    const T two_dx = (T)(2.0 * g.dx);
    const T inv_two_dx = (T)(0.5 * g.inv_dx);
    const bool exact = g.inv_exact != 0;
    auto cdiff = [&](T d) -> T { return exact ? (-d) * inv_two_dx : -d / two_dx; };
    gx = gy = gz = 0;
    // Lost non-zero products (src/mesh/mass_assignment_gradient.cpp:157-196):
    // a weight whose three factors are non-zero, a gradient of a non-zero
    // difference, or a contribution of a non-zero weight and gradient,
    // that rounds to zero.  The reference's corner condition
    //   ((w != 0 || w_lost) && g_lost) || (w_lost && g_nonzero) || (w != 0 && c_lost)
    // equals, for the finite weights here, "all three factors non-zero and
    // some axis with d != 0 and (c == 0 or w == 0)": with w == 0 it asks
    // for a non-zero difference (g_lost || g_nonzero), with w != 0 for a
    // non-zero difference whose contribution w * g is zero (g lost, or
    // g != 0 and the product lost).
    const bool nzx[2] = {wx[0] != (T)0, wx[1] != (T)0};
    const bool nzy[2] = {wy[0] != (T)0, wy[1] != (T)0};
    const bool nzz[2] = {wz[0] != (T)0, wz[1] != (T)0};
    bool lost = false;
#pragma unroll
    for (int ox = 0; ox < 2; ++ox) {
#pragma unroll
        for (int oy = 0; oy < 2; ++oy) {
#pragma unroll
            for (int oz = 0; oz < 2; ++oz) {
                const T w = wx[ox] * wy[oy] * wz[oz];
                const T ypl = oy == 0 ? X[ox + 1][1][oz] : Y[1][ox][oz];
                const T ymi = oy == 0 ? Y[0][ox][oz] : X[ox + 1][0][oz];
                const T zpl = oz == 0 ? X[ox + 1][oy][1] : Z[1][ox][oy];
                const T zmi = oz == 0 ? Z[0][ox][oy] : X[ox + 1][oy][0];
                const T dxv = X[ox + 2][oy][oz] - X[ox][oy][oz];
                const T dyv = ypl - ymi;
                const T dzv = zpl - zmi;
                const T cx = w * cdiff(dxv), cy = w * cdiff(dyv), cz = w * cdiff(dzv);
                const bool wz0 = w == (T)0;
                const bool any = (dxv != (T)0 && (cx == (T)0 || wz0)) || (dyv != (T)0 && (cy == (T)0 || wz0)) ||
                                 (dzv != (T)0 && (cz == (T)0 || wz0));
                lost |= nzx[ox] && nzy[oy] && nzz[oz] && any;
                gx += cx;
                gy += cy;
                gz += cz;
            }
        }
    }
    return lost;
}

// O32: every wave's particles lie in one box (one box, or a particle count
// per box that is a multiple of 64), whose mesh spans at most 2^32 bytes; the
// stencil then uses 32-bit byte offsets from the box's mesh base (one scalar
// base, no per-lane 64-bit address arithmetic).  REC: the drifted positions' deposit records are
// written into the capacity layout (binary32); otherwise keys and ranks.
// OUT: the force outputs acc and g may be set; without them the kernel keeps
// twelve fewer scalar registers live (8 waves per SIMD instead of 7).
// CHUNK: the wave-chunk lattice schedule.  (CHUNK and the gate as run-time branches
// cost the 512^3 gather on 1024^3 2%: 3.98 -> 4.05 ms.)
template <typename T, typename PT, bool O32, bool REC, bool OUT, bool CHUNK>
__global__ void __launch_bounds__(256) k_gather_kdk(GatherArgs<T, PT> a) {
    if constexpr (!REC) {  // records are carried by asynchronous steps only
        if (a.gate && *a.gate) return;
    }
    // each XCD walks a contiguous particle range (spatially compact for
    // lattice-ordered particles), so potential lines are reused in its L2
    const uint32_t bid = xcd_block(blockIdx.x, gridDim.x);
    const uint64_t p = CHUNK ? lattice_wave_particle(bid, a.lat, a.n)
                             : (uint64_t)lattice_block(bid, a.lat) * blockDim.x + threadIdx.x;
    const Geom& g = a.g;
    const int N = g.N;
    uint32_t fail = 0;
    bool live = p < a.n;
    uint32_t next_key = 0;
    bool key_ok = false;
    DepRecord next_rec{0u, 0.0f, 0.0f, 0.0f};
    if (live) {
        int ix = 0, iy = 0, iz = 0;
        double fx = 0.0, fy = 0.0, fz = 0.0;
        // the whole particle state is loaded up front: one memory round trip
        // for it, then one for the potential stencil
        const double xp = __builtin_nontemporal_load(&a.x_in[p]), yp = __builtin_nontemporal_load(&a.y_in[p]),
                     zp = __builtin_nontemporal_load(&a.z_in[p]);
        const bool kick = a.has_prev || a.has_next;
        PT qx0 = 0, qy0 = 0, qz0 = 0;
        if (kick) {
            qx0 = __builtin_nontemporal_load(&a.px_in[p]);
            qy0 = __builtin_nontemporal_load(&a.py_in[p]);
            qz0 = __builtin_nontemporal_load(&a.pz_in[p]);
        }
        if (!(cic_axis(xp, g, ix, fx) && cic_axis(yp, g, iy, fy) && cic_axis(zp, g, iz, fz))) {
            fail = ERR_POSITION_NONFINITE;
        } else {
            const T wx[2] = {(T)(1.0 - fx), (T)fx};
            const T wy[2] = {(T)(1.0 - fy), (T)fy};
            const T wz[2] = {(T)(1.0 - fz), (T)fz};
            // O32: the wave's box, read from its first active lane, gives a scalar base
            const uint64_t box = O32 ? (uint64_t)__builtin_amdgcn_readfirstlane(box_of(p, g)) : (uint64_t)box_of(p, g);
            T gx, gy, gz;
            const bool lost = stencil_force<T, O32>(a.phi + box * (uint64_t)N * (uint64_t)N * (uint64_t)N, g, ix, iy,
                                                    iz, wx, wy, wz, gx, gy, gz);
            if (lost) {
                fail = ERR_GATHER_UNDERFLOW;
            } else if (!isfinite(gx) || !isfinite(gy) || !isfinite(gz)) {
                fail = ERR_FORCE_NONFINITE;
            } else {
                if constexpr (OUT) {
                    if (a.acc_x) {
                        a.acc_x[p] += (double)gx;
                        a.acc_y[p] += (double)gy;
                        a.acc_z[p] += (double)gz;
                    }
                    if (a.g_x) {
                        a.g_x[p] = gx;
                        a.g_y[p] = gy;
                        a.g_z[p] = gz;
                    }
                }
                if (kick) {
                    PT qx = qx0, qy = qy0, qz = qz0;
                    if (!isfinite(qx) || !isfinite(qy) || !isfinite(qz)) {
                        fail = ERR_MOMENTUM_NONFINITE;
                    } else {
                        if (a.has_prev) {
                            const PT k = (PT)(a.dfac ? a.dfac[0] : a.k_prev);
                            qx = qx + (PT)gx * k;
                            qy = qy + (PT)gy * k;
                            qz = qz + (PT)gz * k;
                        }
                        double nx = xp, ny = yp, nz = zp;
                        if (a.has_next) {
                            const PT k = (PT)(a.dfac ? a.dfac[1] : a.k_next);
                            qx = qx + (PT)gx * k;
                            qy = qy + (PT)gy * k;
                            qz = qz + (PT)gz * k;
                            const double D = a.dfac ? a.dfac[2] : a.d_next;
                            const double L = g.L;
                            const double ddx = (double)qx * D, ddy = (double)qy * D, ddz = (double)qz * D;
                            nx = wrap_pos(wrap_pos(xp, L) + minimum_image(ddx, L), L);
                            ny = wrap_pos(wrap_pos(yp, L) + minimum_image(ddy, L), L);
                            nz = wrap_pos(wrap_pos(zp, L) + minimum_image(ddz, L), L);
                        }
                        if (!isfinite(qx) || !isfinite(qy) || !isfinite(qz) || !isfinite(nx)
                            || !isfinite(ny) || !isfinite(nz)) {
                            fail = ERR_UPDATE_NONFINITE;
                        } else {
                            // the particle streams are read and written once per step:
                            // non-temporal, so they do not evict the potential stencil
                            __builtin_nontemporal_store(qx, &a.px_out[p]);
                            __builtin_nontemporal_store(qy, &a.py_out[p]);
                            __builtin_nontemporal_store(qz, &a.pz_out[p]);
                            __builtin_nontemporal_store(nx, &a.x_out[p]);
                            __builtin_nontemporal_store(ny, &a.y_out[p]);
                            __builtin_nontemporal_store(nz, &a.z_out[p]);
                            if (a.next_counts) {
                                // bucket of the drifted position for the next deposit
                                int bx, by, bz;
                                double fxn, fyn, fzn;
                                key_ok = cic_axis(nx, g, bx, fxn) && cic_axis(ny, g, by, fyn)
                                         && cic_axis(nz, g, bz, fzn);
                                if (key_ok) {
                                    next_key = box_of(p, g) * buckets_per_box(g) + bucket_of(bx, by, bz, g);
                                    if constexpr (REC) {  // the record k_scatter_records would write
                                        next_rec.cell = record_cell(bx, by, bz, g);
                                        next_rec.fx = (float)fxn;
                                        next_rec.fy = (float)fyn;
                                        next_rec.fz = (float)fzn;
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
        if (fail) atomicOr(a.err, fail);
    }
    if (a.next_counts) {  // uniform across the grid: every lane reaches the ballots
        const bool have = live && key_ok;
        if constexpr (REC) {
            // the bucket's capacity slots are loaded ahead of the rank atomic, so
            // the two round trips overlap
            uint32_t s0 = 0, s1 = 0;
            if (have) {
                s0 = a.rec_start[next_key];
                s1 = a.rec_start[next_key + 1];
            }
            uint32_t groups;
            const uint32_t rank = aggregated_rank(a.next_counts, next_key, have, groups);
            uint32_t slot = 0;
            bool over = false;
            if (have) {
                if (rank < s1 - s0) slot = s0 + rank;
                else over = true;
            }
            const uint64_t om = __ballot(over);
            uint32_t obase = 0;
            if (om) {  // one atomic per wave for its overflow records
                const int leader = __ffsll((unsigned long long)om) - 1;
                if ((int)lane_id() == leader) obase = atomicAdd(a.ovf_count, (uint32_t)__popcll(om));
                obase = (uint32_t)__builtin_amdgcn_readlane((int)obase, leader);
            }
            if (have) {
                if (!over) {
                    a.rec_out[slot] = next_rec;
                } else {
                    const uint32_t o = obase + (uint32_t)__popcll(om & ((1ull << lane_id()) - 1ull));
                    a.ovf_rec[o] = next_rec;
                    a.next_keys[o] = next_key;
                    a.next_ranks[o] = rank;
                }
            }
        } else {
            uint32_t groups;
            const uint32_t rank = aggregated_rank(a.next_counts, next_key, have, groups);
            if (live) {
                __builtin_nontemporal_store(key_ok ? next_key : 0xffffffffu, &a.next_keys[p]);
                __builtin_nontemporal_store(rank, &a.next_ranks[p]);
            }
        }
    }
}

// The 8 mesh values around base cell (ix, iy, iz).  O32: 32-bit byte offsets from f.
template <typename T, bool O32>
__device__ __forceinline__ void load_cube(const T* f, int N, int ix, int iy, int iz, T (&F)[2][2][2]) {
    using Off = typename std::conditional<O32, uint32_t, uint64_t>::type;
    const Off es = O32 ? (Off)sizeof(T) : (Off)1;
    const Off NN = (Off)N * (Off)N;
    const Off xo[2] = {(Off)ix * NN * es, (Off)wrap_cell(ix + 1, N) * NN * es};
    const Off yo[2] = {(Off)iy * (Off)N * es, (Off)wrap_cell(iy + 1, N) * (Off)N * es};
    const bool zrun = iz + 1 < N;
    const Off z0 = (Off)iz * es, z1 = (Off)wrap_cell(iz + 1, N) * es;
    typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    auto at = [&](Off o) -> const char* {
        return O32 ? reinterpret_cast<const char*>(f) + o : reinterpret_cast<const char*>(f + o);
    };
#pragma unroll
    for (int ox = 0; ox < 2; ++ox)
#pragma unroll
        for (int oy = 0; oy < 2; ++oy) {
            const Off o = xo[ox] + yo[oy];
            if (zrun) {
                const V2 v = *reinterpret_cast<const V2*>(at(o + z0));
                F[ox][oy][0] = v.x;
                F[ox][oy][1] = v.y;
            } else {
                F[ox][oy][0] = *reinterpret_cast<const T*>(at(o + z0));
                F[ox][oy][1] = *reinterpret_cast<const T*>(at(o + z1));
            }
        }
}

// CIC interpolation of mesh f at base cell (ix, iy, iz), corner weights w[0] =
// 1 - f, w[1] = f per axis (src/mesh/mass_assignment_gather.inc:95-181,
// 402-451): the sum over the x, y, z corner offsets, in that order, of
// f * ((wx * wy) * wz).  lost is set where a product of non-zero factors
// rounds to zero.
template <typename T, bool O32>
__device__ __forceinline__ T interp_mesh(const T* f, int N, int ix, int iy, int iz, const T (&wx)[2],
                                         const T (&wy)[2], const T (&wz)[2], bool& lost) {
    T F[2][2][2];
    load_cube<T, O32>(f, N, ix, iy, iz, F);
    T v = (T)0;
#pragma unroll
    for (int ox = 0; ox < 2; ++ox)
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
#pragma unroll
            for (int oz = 0; oz < 2; ++oz) {
                const T xy = wx[ox] * wy[oy];
                const T w = xy * wz[oz];
                const T fv = F[ox][oy][oz];
                if (wx[ox] != (T)0 && wy[oy] != (T)0 && wz[oz] != (T)0 && w == (T)0 && fv != (T)0) lost = true;
                const T c = fv * w;
                if (fv != (T)0 && w != (T)0 && c == (T)0) lost = true;
                v += c;
            }
    return v;
}

// Interpolation of up to three meshes of one box at particle positions.  A
// lost product raises ERR_INTERP_UNDERFLOW, as the reference's
// underflow_error.  out[m] receives v (force mode, a non-finite v raises
// ERR_FORCE_NONFINITE); add[m] receives += v.
template <typename T>
struct InterpArgs {
    Geom g;
    uint64_t n;
    const double* x;
    const double* y;
    const double* z;
    const T* f[3];
    T* out[3];
    double* add[3];
    int meshes;
    uint32_t* err;
};

template <typename T, bool O32>
__global__ void __launch_bounds__(256) k_interp(InterpArgs<T> a) {
    const uint64_t p = (uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (p >= a.n) return;
    const Geom& g = a.g;
    int ix, iy, iz;
    double fx, fy, fz;
    if (!cic_axes(a.x[p], a.y[p], a.z[p], g, ix, iy, iz, fx, fy, fz)) {
        atomicOr(a.err, ERR_POSITION_NONFINITE);
        return;
    }
    const T wx[2] = {(T)(1.0 - fx), (T)fx};
    const T wy[2] = {(T)(1.0 - fy), (T)fy};
    const T wz[2] = {(T)(1.0 - fz), (T)fz};
    bool lost = false, bad = false;
    for (int m = 0; m < a.meshes; ++m) {
        const T v = interp_mesh<T, O32>(a.f[m], g.N, ix, iy, iz, wx, wy, wz, lost);
        if (a.out[m]) {
            if (!isfinite(v)) bad = true;
            a.out[m][p] = v;
        }
        if (a.add[m]) a.add[m][p] += (double)v;
    }
    if (lost) atomicOr(a.err, ERR_INTERP_UNDERFLOW);
    if (bad) atomicOr(a.err, ERR_FORCE_NONFINITE);
}

// Force of the particles in deposit-record order (slot s of the bucket layout),
// the result over the slot's force record (binary64: over the fractions).
// Consecutive slots share a 16^3 tile, so the stencil lines stay in L1 and L2
// whatever the order of the particle arrays; in particle order a shuffled set
// fetches 12 to 16 lines per particle from beyond L2 (20M shuffled particles on
// 512^3: 4.43 ms in particle order, 0.78 here, with 0.28 more in the scatter and
// 0.33 more in the commit; binary64, 3M on 192^3: 0.51 -> 0.12, with 0.03 more in
// the commit).  Where the order keeps to the buckets it is slower (16.8M on 512^3
// near their lattice: 0.42 -> 0.70, with 0.14 and 0.07 more around it); the host
// chooses by a probe of the order (order_probe).  FORCE_SG false: centred gradient of
// f[0] (one potential per box); true: interpolation of the force meshes f[0..2].
template <typename T>
struct SlotForceArgs {
    Geom g;
    uint64_t n;
    const DepRecord* rec;  // binary32
    ForceRecord* force;
    DepRecord64* rec64;    // binary64
    const T* f[3];
    const uint32_t* gate;  // do nothing where this word is set
    uint32_t* err;
};

template <typename T, bool FORCE_SG, bool O32>
__global__ void __launch_bounds__(256) k_slot_force(SlotForceArgs<T> a) {
    const uint64_t s = (uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    // a failed deposit (a particle without a slot) leaves records unwritten
    if (s >= a.n || *a.gate) return;
    const Geom& g = a.g;
    const int E = g.T;
    const uint32_t nT = (uint32_t)g.nT, ntiles = nT * nT * nT;
    uint32_t cell, tile, box;  // O32: one box
    T wx[2], wy[2], wz[2];
    if constexpr (sizeof(T) == 4) {
        const DepRecord r = a.rec[s];
        const ForceRecord q = a.force[s];
        cell = r.cell;
        box = O32 ? 0u : q.tile / ntiles;
        tile = O32 ? q.tile : q.tile % ntiles;
        wx[0] = q.wx; wx[1] = r.fx;
        wy[0] = q.wy; wy[1] = r.fy;
        wz[0] = q.wz; wz[1] = r.fz;
    } else {
        const DepRecord64 r = a.rec64[s];
        cell = r.cell & ((1u << REC_CELL_BITS) - 1u);
        tile = r.cell >> REC_CELL_BITS;
        box = O32 ? 0u : box_of(r.index, g);
        wx[0] = 1.0 - r.fx; wx[1] = r.fx;
        wy[0] = 1.0 - r.fy; wy[1] = r.fy;
        wz[0] = 1.0 - r.fz; wz[1] = r.fz;
    }
    const int cz = E == 16 ? (int)(cell & 15u) : (int)cell % E;
    const int cxy = E == 16 ? (int)(cell >> 4) : (int)cell / E;
    const int cy = E == 16 ? cxy & 15 : cxy % E, cx = E == 16 ? cxy >> 4 : cxy / E;
    const int ix = (int)(tile / (nT * nT)) * E + cx, iy = (int)(tile / nT % nT) * E + cy, iz = (int)(tile % nT) * E + cz;
    T v[3];
    bool lost = false;
    if constexpr (FORCE_SG) {
#pragma unroll
        for (int m = 0; m < 3; ++m) v[m] = interp_mesh<T, O32>(a.f[m], g.N, ix, iy, iz, wx, wy, wz, lost);
    } else {
        const T* phi = a.f[0] + (uint64_t)box * (uint64_t)g.N * (uint64_t)g.N * (uint64_t)g.N;
        lost = stencil_force<T, O32>(phi, g, ix, iy, iz, wx, wy, wz, v[0], v[1], v[2]);
    }
    if (lost) atomicOr(a.err, FORCE_SG ? ERR_INTERP_UNDERFLOW : ERR_GATHER_UNDERFLOW);
    if (!isfinite(v[0]) || !isfinite(v[1]) || !isfinite(v[2])) atomicOr(a.err, ERR_FORCE_NONFINITE);
    if constexpr (sizeof(T) == 4) {
        a.force[s] = {v[0], v[1], v[2], 0u};
    } else {
        a.rec64[s].fx = v[0];
        a.rec64[s].fy = v[1];
        a.rec64[s].fz = v[2];
    }
}

// acc += g for every particle, its force read from its slot, where no error is
// set (status: the error words of the deposit and transform and of the force).
__device__ __forceinline__ void slot_value(const ForceRecord& q, double v[3]) {
    v[0] = q.wx;
    v[1] = q.wy;
    v[2] = q.wz;
}
__device__ __forceinline__ void slot_value(const DepRecord64& q, double v[3]) {
    v[0] = q.fx;
    v[1] = q.fy;
    v[2] = q.fz;
}

template <typename R>
__global__ void __launch_bounds__(256) k_commit_slots(uint64_t n, const uint32_t* __restrict__ keys,
                                                      const uint32_t* __restrict__ ranks,
                                                      const uint32_t* __restrict__ offsets,
                                                      const R* __restrict__ force, double* __restrict__ ax,
                                                      double* __restrict__ ay, double* __restrict__ az,
                                                      const uint32_t* __restrict__ status) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || (status[0] | status[1])) return;
    double v[3];
    slot_value(force[offsets[keys[p]] + ranks[p]], v);
    ax[p] += v[0];
    ay[p] += v[1];
    az[p] += v[2];
}

// Potential-energy diagnostic: sum_p m_p phi(x_p) with phi CIC-interpolated
// (CICMassAssignment::interpolate_mass_weighted_sum_full_mesh,
// src/mesh/mass_assignment_gather.inc:283-399; the caller halves it as
// src/gravity/pm_solver.cpp:817-841 does).  Per particle, in binary64 as the
// reference (its accumulation type is binary64): value = sum over corners
// (x outer, z inner) of phi_c * ((wx wy) wz), then m * value, with the
// reference's lost-product checks (ERR_INTERP_UNDERFLOW).  The summation is the
// reference's deterministic blocked sum (include/cosmo_nbody/math/
// deterministic_sum.hpp:48-104): workgroup b adds the terms of particles
// [b*4096, (b+1)*4096) in index order with Neumaier compensation;
// k_potential_total adds the block sums in order.
constexpr int ENERGY_THREADS = 256;
constexpr int ENERGY_BLOCK = 4096;
constexpr int ENERGY_CHUNK = 2048;  // terms in LDS at a time

// Neumaier's sum over count <= ENERGY_CHUNK terms in LDS, continued from (sum,
// comp) of thread 0, by the whole workgroup.  Only two chains are serial, one
// addition per term each: the running sums, which thread 0 leaves in sums, and
// the compensation; the rounding error of each step needs the two sums around
// it and is formed by all threads (one lane doing it all: 229 cycles per term,
// 0.45 ms for 3M particles).
__device__ __forceinline__ void neumaier_terms(double* terms, double* sums, uint32_t count, double& sum,
                                               double& comp) {
    constexpr uint32_t U = 16;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = sum;
        uint32_t i = 0;
        for (; i + U <= count; i += U) {
            double v[U];
#pragma unroll
            for (uint32_t j = 0; j < U; ++j) v[j] = terms[i + j];
#pragma unroll
            for (uint32_t j = 0; j < U; ++j) {
                sums[i + j] = s;
                s += v[j];
            }
        }
        for (; i < count; ++i) {
            sums[i] = s;
            s += terms[i];
        }
        sums[count] = s;
        sum = s;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < count; i += ENERGY_THREADS) {
        const double s = sums[i], v = terms[i], t = sums[i + 1];
        terms[i] = fabs(s) >= fabs(v) ? (s - t) + v : (v - t) + s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double c = comp;
        uint32_t i = 0;
        for (; i + U <= count; i += U) {
            double v[U];
#pragma unroll
            for (uint32_t j = 0; j < U; ++j) v[j] = terms[i + j];
#pragma unroll
            for (uint32_t j = 0; j < U; ++j) c += v[j];
        }
        for (; i < count; ++i) c += terms[i];
        comp = c;
    }
}

template <typename T>
__global__ void __launch_bounds__(ENERGY_THREADS) k_potential_partials(Geom g, uint64_t n, const double* __restrict__ x,
                                                                      const double* __restrict__ y,
                                                                      const double* __restrict__ z,
                                                                      const double* __restrict__ masses,
                                                                      double uniform_mass, const T* __restrict__ phi,
                                                                      double* __restrict__ partials,
                                                                      uint32_t* __restrict__ err) {
    __shared__ double terms[ENERGY_CHUNK], sums[ENERGY_CHUNK + 1];
    const uint64_t b0 = (uint64_t)blockIdx.x * ENERGY_BLOCK;
    const uint64_t b1 = n < b0 + ENERGY_BLOCK ? n : b0 + ENERGY_BLOCK;
    const int N = g.N;
    const uint64_t NN = (uint64_t)N * (uint64_t)N;
    bool lost = false, bad = false;
    double sum = 0.0, comp = 0.0;
    for (uint64_t c0 = b0; c0 < b1; c0 += ENERGY_CHUNK) {
        const uint64_t c1 = b1 < c0 + ENERGY_CHUNK ? b1 : c0 + ENERGY_CHUNK;
        __syncthreads();
        for (uint64_t p = c0 + threadIdx.x; p < c1; p += ENERGY_THREADS) {
            int ix, iy, iz;
            double fx, fy, fz;
            double weighted = 0.0;
            if (!cic_axes(x[p], y[p], z[p], g, ix, iy, iz, fx, fy, fz)) {
                bad = true;
            } else {
                const double m = masses ? masses[p] : uniform_mass;
                const double wx[2] = {1.0 - fx, fx}, wy[2] = {1.0 - fy, fy}, wz[2] = {1.0 - fz, fz};
                const uint64_t xs[2] = {(uint64_t)ix, (uint64_t)wrap_cell(ix + 1, N)};
                const uint64_t ys[2] = {(uint64_t)iy, (uint64_t)wrap_cell(iy + 1, N)};
                const uint64_t zs[2] = {(uint64_t)iz, (uint64_t)wrap_cell(iz + 1, N)};
                double value = 0.0;
#pragma unroll
                for (int ox = 0; ox < 2; ++ox)
#pragma unroll
                    for (int oy = 0; oy < 2; ++oy)
#pragma unroll
                        for (int oz = 0; oz < 2; ++oz) {
                            const double fv = (double)phi[xs[ox] * NN + ys[oy] * (uint64_t)N + zs[oz]];
                            const double xy = wx[ox] * wy[oy];
                            const double w = xy * wz[oz];
                            if (wx[ox] != 0.0 && wy[oy] != 0.0 && wz[oz] != 0.0 && w == 0.0 && fv != 0.0 && m != 0.0)
                                lost = true;
                            const double c = fv * w;
                            if (fv != 0.0 && w != 0.0 && c == 0.0 && m != 0.0) lost = true;
                            value += c;
                        }
                weighted = m * value;
                if (m != 0.0 && value != 0.0 && weighted == 0.0) lost = true;
            }
            terms[p - c0] = weighted;
        }
        neumaier_terms(terms, sums, (uint32_t)(c1 - c0), sum, comp);
    }
    if (bad) atomicOr(err, ERR_POSITION_NONFINITE);
    if (lost) atomicOr(err, ERR_INTERP_UNDERFLOW);
    if (threadIdx.x == 0) partials[blockIdx.x] = sum + comp;
}

// 0.5 * (Neumaier sum of the workgroup partials, in order) -> out[0]; one workgroup
__global__ void __launch_bounds__(ENERGY_THREADS) k_potential_total(const double* __restrict__ partials, uint64_t count,
                                                                    double* __restrict__ out,
                                                                    uint32_t* __restrict__ err) {
    __shared__ double terms[ENERGY_CHUNK], sums[ENERGY_CHUNK + 1];
    double s = 0.0, c = 0.0;
    for (uint64_t c0 = 0; c0 < count; c0 += ENERGY_CHUNK) {
        const uint32_t m = (uint32_t)(count - c0 < ENERGY_CHUNK ? count - c0 : ENERGY_CHUNK);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < m; i += ENERGY_THREADS) terms[i] = partials[c0 + i];
        neumaier_terms(terms, sums, m, s, c);
    }
    if (threadIdx.x != 0) return;
    const double total = s + c;
    const double half = 0.5 * total;
    if (!isfinite(total) || (total != 0.0 && half == 0.0)) atomicOr(err, ERR_INTERP_UNDERFLOW);
    out[0] = half;
}

// 1LPT displacement spectrum of one axis (src/ic/lpt_displacement.cpp:306-340):
// psi_k = (-Im d, Re d) * k_d / k^2 with k_d = 0 on the Nyquist index of the
// axis and psi_k = 0 where k^2 = 0, times 1/N^3 (the inverse transform's
// normalisation), written into B [kz][ky][kx] from the r2c half spectrum
// dk [x][y][kz] (binary64).
__global__ void __launch_bounds__(256) k_lpt_spectrum(const double2* __restrict__ dk, int axis, int N,
                                                      const double* __restrict__ kc, const double* __restrict__ kd,
                                                      double norm, double2* __restrict__ B) {
    const int NH = N / 2 + 1;
    const uint64_t total = (uint64_t)NH * N * N;
    const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total) return;
    const int kx = (int)(e % (uint64_t)N), ky = (int)((e / (uint64_t)N) % (uint64_t)N), kz = (int)(e / ((uint64_t)N * N));
    const double qx = kc[kx], qy = kc[ky], qz = kc[kz];
    const double k2 = qx * qx + qy * qy + qz * qz;
    double2 out = {0.0, 0.0};
    if (k2 != 0.0) {
        const double dkv = axis == 0 ? kd[kx] : (axis == 1 ? kd[ky] : kd[kz]);
        const double f = dkv / k2;
        const double2 d = dk[((uint64_t)kx * N + ky) * NH + kz];
        out = {-d.y * f * norm, d.x * f * norm};
    }
    B[e] = out;
}

// 1LPT particle update of one axis (src/ic/lpt_displacement.cpp:99-129,
// 341-384; lattice src/ic/initial_conditions.cpp:296-312): particle
// (i, j, k) of the n^3 lattice takes psi at mesh cell (i s, j s, k s),
// position wrap(q + psi) with q = (i, j or k) * dx, momentum p_factor * psi.
__global__ void __launch_bounds__(256) k_lpt_update(const double* __restrict__ psi, int axis, int N, int n, int s,
                                                    double dx, double L, double p_factor, double* __restrict__ pos,
                                                    double* __restrict__ mom, uint32_t* __restrict__ err) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t total = (uint64_t)n * n * n;
    if (p >= total) return;
    const uint64_t i = p / ((uint64_t)n * n), j = (p / (uint64_t)n) % (uint64_t)n, k = p % (uint64_t)n;
    const double v = psi[((i * s) * (uint64_t)N + j * s) * (uint64_t)N + k * s];
    const uint64_t q = axis == 0 ? i : (axis == 1 ? j : k);
    const double disp = 1.0 * v;
    const double inc = p_factor * v;
    const double cand = (double)q * dx + disp;
    const double mcand = 0.0 + inc;
    const double w = wrap_pos(cand, L);
    if (!isfinite(v) || !isfinite(disp) || !isfinite(inc) || !isfinite(cand) || !isfinite(mcand) || !isfinite(w)) {
        atomicOr(err, ERR_UPDATE_NONFINITE);
        return;
    }
    pos[p] = w;
    mom[p] = mcand;
}

// Transactional commit for the reference-shaped force entry: acc += g where no
// error is set.
template <typename T>
__global__ void k_commit_force(uint64_t n, const T* __restrict__ gx, const T* __restrict__ gy,
                               const T* __restrict__ gz, double* __restrict__ ax,
                               double* __restrict__ ay, double* __restrict__ az,
                               const uint32_t* __restrict__ status) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || (status[0] | status[1])) return;
    ax[p] += (double)gx[p];
    ay[p] += (double)gy[p];
    az[p] += (double)gz[p];
}

// ===========================================================================
// Adjoint (vector-Jacobian products) of the fused step.  The forward step is
//   p' = p + (k_prev + k_next) g(x),   x' = wrap(x + d_next p'),
//   g_j(x) = sum_c W(x_j - c) (-D phi)(c),  phi = G s,  s_c = (m_c - M/N_c)/dx^3,
//   m_c = sum_k m W(x_k - c),   D_a f(c) = (f(c + e_a) - f(c - e_a)) / (2 dx).
// For an adjoint vector u (one 3-vector per particle) the product
// J_g(x)^T u has two parts per particle k:
//   (a) through particle k's own gather weights:
//       sum_c dW(x_k - c)/dx_k (u_k . (-D phi)(c)),
//   (b) through the potential: with A_a = sum_j u_j,a W(x_j - c) deposited,
//       chi = G (sum_a D_a A_a) (G symmetric, D_a antisymmetric),
//       (m / dx^3) sum_c chi(c) dW(x_k - c)/dx_k.
// ===========================================================================

// u = lp + d_next lx (the momentum adjoint entering the kick), written over lp.
__global__ void k_adj_kick(uint64_t n, const double* __restrict__ lx, const double* __restrict__ ly,
                           const double* __restrict__ lz, double* __restrict__ lpx, double* __restrict__ lpy,
                           double* __restrict__ lpz, double d_next, int has_next) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n || !has_next) return;
    lpx[p] = lpx[p] + d_next * lx[p];
    lpy[p] = lpy[p] + d_next * ly[p];
    lpz[p] = lpz[p] + d_next * lz[p];
}

// max |q| over particles (per block, then over blocks): the signed deposit unit.
__global__ void k_absmax(uint64_t n, const double* __restrict__ qx, const double* __restrict__ qy,
                         const double* __restrict__ qz, double* __restrict__ out) {
    const double* q = blockIdx.y == 0 ? qx : (blockIdx.y == 1 ? qy : qz);
    __shared__ double sh[256];
    double m = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
        const double v = fabs(q[i]);
        m = v > m ? v : m;
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + k]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.y * gridDim.x + blockIdx.x] = sh[0];
}

// Per-particle values q, scaled by inv_unit, into bucket order for the
// binary32 record deposit (keys/ranks/offsets of the same positions).
template <typename MT>
__global__ void k_scatter_values(uint64_t n, const double* __restrict__ q, double inv_unit,
                                 const uint32_t* __restrict__ keys, const uint32_t* __restrict__ ranks,
                                 const uint32_t* __restrict__ offsets, MT* __restrict__ out) {
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const uint32_t k = keys[p];
    if (k == 0xffffffffu) return;
    if constexpr (sizeof(MT) == sizeof(double)) out[offsets[k] + ranks[p]] = q[p];
    else out[offsets[k] + ranks[p]] = (MT)(q[p] * inv_unit);
}

// out = sum_a D_a A_a (periodic centred differences), one box.
template <typename T>
__global__ void __launch_bounds__(256) k_div_stencil(const T* __restrict__ ax, const T* __restrict__ ay,
                                                     const T* __restrict__ az, T* __restrict__ out, int N,
                                                     double inv_2dx) {
    // four z-adjacent cells per thread (N is a multiple of 4)
    typedef T V4 __attribute__((ext_vector_type(4)));
    const uint64_t NN = (uint64_t)N * N;
    const uint64_t c = 4 * ((uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x);
    if (c >= NN * N) return;
    const int iz = (int)(c % N), iy = (int)((c / N) % N), ix = (int)(c / NN);
    auto at = [&](const T* f, int i, int j) {
        return *reinterpret_cast<const V4*>(f + (uint64_t)wrap_cell(i, N) * NN + (uint64_t)wrap_cell(j, N) * N + iz);
    };
    const V4 xp = at(ax, ix + 1, iy), xm = at(ax, ix - 1, iy), yp = at(ay, ix, iy + 1), ym = at(ay, ix, iy - 1);
    const V4 zc = at(az, ix, iy);
    const T* zrow = az + (uint64_t)ix * NN + (uint64_t)iy * N;
    const T z[6] = {zrow[wrap_cell(iz - 1, N)], zc.x, zc.y, zc.z, zc.w, zrow[wrap_cell(iz + 4, N)]};
    V4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double d = ((double)xp[j] - (double)xm[j]) + ((double)yp[j] - (double)ym[j]) +
                         ((double)z[j + 2] - (double)z[j]);
        o[j] = (T)(d * inv_2dx);
    }
    *reinterpret_cast<V4*>(out + c) = o;
}

template <typename T>
struct AdjGatherArgs {
    Geom g;
    uint64_t n;
    const double* x;
    const double* y;
    const double* z;
    const double* ux;    // adjoint vector per particle (term (a)); null: no term (a)
    const double* uy;
    const double* uz;
    const T* phi;        // forward potential (term (a))
    const T* chi;        // scalar field of term (b)
    double coef_a;       // lambda += coef_a * (a) + coef_b * (b)
    double coef_b;
    double* lx;
    double* ly;
    double* lz;
    const uint32_t* gate;  // do nothing where this word is set
    uint32_t* err;
};

// The potential and chi are read as z-contiguous vector runs, the 32 distinct
// potential values once each (128^3 particles on 256^3, binary32: 196 us with
// eight scalar 7-point stencils, 116 so).
template <typename T, bool O32>
__global__ void __launch_bounds__(256) k_adj_gather(AdjGatherArgs<T> a) {
    const uint64_t p = (uint64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (p >= a.n || *a.gate) return;
    const Geom& g = a.g;
    const int N = g.N;
    int ix, iy, iz;
    double fx, fy, fz;
    if (!cic_axes(a.x[p], a.y[p], a.z[p], g, ix, iy, iz, fx, fy, fz)) {
        atomicOr(a.err, ERR_POSITION_NONFINITE);
        return;
    }
    const double inv_dx = 1.0 / g.dx;
    const double w[3][2] = {{1.0 - fx, fx}, {1.0 - fy, fy}, {1.0 - fz, fz}};
    const double dw[2] = {-inv_dx, inv_dx};
    const bool with_a = a.ux != nullptr;
    const double u[3] = {with_a ? a.ux[p] : 0.0, with_a ? a.uy[p] : 0.0, with_a ? a.uz[p] : 0.0};
    T X[4][2][2], Y[2][2][2], Z[2][2][2], F[2][2][2];
    load_cube<T, O32>(a.chi, N, ix, iy, iz, F);
    if (with_a) load_stencil<T, O32>(a.phi, N, ix, iy, iz, X, Y, Z);
    // -(f+ - f-) / (2 dx); with dx a power of two the product with the exact
    // reciprocal has the quotient's bits
    const double two_dx = 2.0 * g.dx, inv_two_dx = 0.5 * g.inv_dx;
    const bool exact = g.inv_exact != 0;
    auto grad = [&](T hi, T lo) {
        const double d = (double)hi - (double)lo;
        return exact ? -d * inv_two_dx : -d / two_dx;
    };
    double ta[3] = {0.0, 0.0, 0.0}, tb[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int ox = 0; ox < 2; ++ox) {
#pragma unroll
        for (int oy = 0; oy < 2; ++oy) {
#pragma unroll
            for (int oz = 0; oz < 2; ++oz) {
                // derivative of the corner weight along each axis
                const double dwc[3] = {dw[ox] * w[1][oy] * w[2][oz], w[0][ox] * dw[oy] * w[2][oz],
                                       w[0][ox] * w[1][oy] * dw[oz]};
                const double xv = (double)F[ox][oy][oz];
                double s = 0.0;
                if (with_a) {
                    const double gx = grad(X[ox + 2][oy][oz], X[ox][oy][oz]);
                    const double gy = grad(oy == 0 ? X[ox + 1][1][oz] : Y[1][ox][oz],
                                           oy == 0 ? Y[0][ox][oz] : X[ox + 1][0][oz]);
                    const double gz = grad(oz == 0 ? X[ox + 1][oy][1] : Z[1][ox][oy],
                                           oz == 0 ? Z[0][ox][oy] : X[ox + 1][oy][0]);
                    s = u[0] * gx + u[1] * gy + u[2] * gz;
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    ta[d] += dwc[d] * s;
                    tb[d] += dwc[d] * xv;
                }
            }
        }
    }
    a.lx[p] += a.coef_a * ta[0] + a.coef_b * tb[0];
    a.ly[p] += a.coef_a * ta[1] + a.coef_b * tb[1];
    a.lz[p] += a.coef_a * ta[2] + a.coef_b * tb[2];
}

}  // namespace hy
