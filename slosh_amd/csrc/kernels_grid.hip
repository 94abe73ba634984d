// Sparse-grid build for one substep on gfx950: hashed block insertion, the
// block list and neighbour tables, and the particle sort by block.
//
// Replaces WgGrid::launch_sort (src/grid/grid.rs:78-238) and the sort kernels of
// shaders/slosh/grid/{grid,sort}.slang. The active-block set is the reference's
// (primary blocks of every particle plus their 7 "+1" neighbours,
// sort.slang:50-92). A block's header id is the slot of its key in the
// substep's hash table; the order of the block list differs from the
// reference's header order (which depends on atomic order as well).
//
// Steady state: nothing runs here. The previous substep's fused G2P kernel inserted
// every particle's primary block and its +1 neighbours into this substep's table,
// appended the new blocks to the regions' lists, wrote each block's particles
// contiguously and appended the ones that left their block to their new block's list.
// P2G finds each block's range in the previous storage and looks up its neighbours, and
// the grid update gives the blocks their storage. (A launch between G2P and P2G for
// all this took 4-6 us of a substep of a small scene and 21 us of one with 42k blocks.
// Substep without it, before and after: 2k particles 33.5 -> 30.2 us, 131k 45.5 -> 39.9,
// 1M 105 -> 97, 2.1M in 42k blocks 652 -> 616.)
// Full sort (first substep, after host mutations, with hooks), of a table of up to
// INDEX_CAP slots in four launches:
//   k_reset_table      hash slots <- NONE, per-step counters and all counts <- 0
//   k_touch_count      each particle's primary block and its 7 +1 neighbours are
//                      inserted, once per run of equal keys in a wavefront; block totals
//                      and per-(block, cell) ranks via one aggregated atomic per run
//   k_block_list       the block list (occupied slots, workgroup scan and one
//                      atomic per workgroup), each block's +1 / -1 neighbour ids
//                      and its id in the previous table; the scans of the block totals
//                      in slot order and of each block's 64 cell counts
//   k_scatter          sorted slot = block start + cell offset + rank
// of a larger one, where clearing all counts would cost more than the launches:
//   k_reset_table, k_touch_primary (the thread that creates a block clears its
//   counters), k_block_list, k_count (a lookup per run), k_block_scan_tiles / _top / _add
//   (three phases in list order; the first launch's other workgroups scan the cell
//   counts), k_scatter
// (A hooked substep of 30k particles, six launches before and four now, 47.5 -> 42 us; of
// 80k 55 -> 48; with a table of 16384 slots 46 both.)
#include "launch.h"

namespace {

// Tables up to here take the full sort in four launches instead of eight: the reset clears
// every slot's counts (256 bytes of cell counts each, 4 MB at most), the insertion counts
// the particles, and the block list's launch scans the counts.
#define INDEX_CAP 16384u

constexpr int ASSOC[8][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 0}, {0, 1, 1},
                             {1, 0, 0}, {1, 0, 1}, {1, 1, 0}, {1, 1, 1}};

// With `blk_cnt`, the blocks' particle and cell counts are cleared as well.
__global__ __launch_bounds__(256) void k_reset_table(uint32_t *__restrict__ keys, uint32_t cap,
                                                     uint32_t *__restrict__ counters,
                                                     unsigned long long *__restrict__ rsum,
                                                     uint32_t *__restrict__ blk_cnt, uint32_t *__restrict__ cell_cnt) {
    const uint32_t stride = gridDim.x * blockDim.x, t = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t s = t; s < cap; s += stride) {
        keys[s] = SLOSH_NONE;
        if (blk_cnt) blk_cnt[s] = 0u;
    }
    if (blk_cnt)
        for (uint32_t s = t; s < cap * (NODES_PER_BLOCK / 4); s += stride)
            reinterpret_cast<uint4 *>(cell_cnt)[s] = make_uint4(0u, 0u, 0u, 0u);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        counters[CTR_NUM_BLOCKS] = 0u;
        counters[CTR_OVERFLOW] = 0u;
        counters[CTR_ITEMS] = 0u;
    }
    if (blockIdx.x == 0 && threadIdx.x < REGIONS) rsum[threadIdx.x * RSUM_STRIDE] = 0ull;
}

__global__ __launch_bounds__(256) void k_touch_primary(const float4 *__restrict__ pos, uint32_t n, float h,
                                                       uint32_t batched, uint32_t *__restrict__ keys, uint32_t cap,
                                                       uint32_t *__restrict__ counters, BlockInit init) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    uint32_t key = 0u, cell;
    if (valid) key = particle_key(pos[i], h, batched, &cell);
    // One insertion round per run of equal keys: the block and its 7 +1 neighbours.
    const uint64_t heads = run_heads(key, valid) & __ballot(valid);
    ListEntry none;
    insert_blocks(keys, cap, batched, key, heads, counters, init, none);
}

// Neighbour table entry `l` (0..15) of block `hid`: [0..6] the +1 neighbours in
// the reference's associated-block order (grid.slang:362-382), [7] the block's
// id in the previous substep's table, [8..14] the -1 neighbours.
__device__ inline void block_neighbour(uint32_t hid, uint32_t key, uint32_t l, uint32_t *__restrict__ nbr,
                                       const uint32_t *__restrict__ keys, const uint32_t *__restrict__ prev_keys,
                                       uint32_t cap, uint32_t batched) {
    int bx, by, bz;
    uint32_t scene;
    unpack_key(batched, key, &bx, &by, &bz, &scene);
    uint32_t out = SLOSH_NONE;
    if (l < 7) {
        const int *o = ASSOC[l + 1];
        out = hash_find(keys, cap, pack_key(batched, scene, bx + o[0], by + o[1], bz + o[2]));
    } else if (l == NBR_PREV) {
        out = hash_find(prev_keys, cap, key);
    } else if (l >= NBR_MINUS && l < NBR_MINUS + 7) {
        const int *o = ASSOC[l - NBR_MINUS + 1];
        out = hash_find(keys, cap, pack_key(batched, scene, bx - o[0], by - o[1], bz - o[2]));
    }
    nbr[(size_t)hid * NBR_STRIDE + l] = out;
}

// The block list and the neighbour tables of a full sort, one launch of two kinds of
// workgroups: [0, cmp_wgs) the block list: each takes 256 * ITEMS slots and appends
// the occupied ones (workgroup scan, one atomic); the rest the neighbour tables, 16
// lanes per slot, every occupied slot's 15 lookups at once.
// Launched with more workgroups (a table of at most INDEX_CAP slots, whose particles are
// counted before): one scans the blocks' particle counts in slot order, and the rest the
// cell counts of each block, a wave per 16 slots.

struct BlockCounts {
    const uint32_t *blk_cnt, *cell_cnt;
    uint32_t *blk_start, *cell_start;
};

// Exclusive scan of the particle counts of all slots (cap a power of two up to INDEX_CAP)
// by a workgroup of 256 threads, each with consecutive slots.
__device__ inline void scan_slots(const BlockCounts &b, uint32_t cap, uint32_t *wsum) {
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    const uint32_t each = cap > 256u ? cap >> 8 : 1u, lo = tid * each;
    uint32_t sum = 0u;
    if (each >= 4u) {
        const uint4 *v = reinterpret_cast<const uint4 *>(b.blk_cnt + lo);
#pragma unroll 4
        for (uint32_t k = 0; k < each / 4u; k++) sum += v[k].x + v[k].y + v[k].z + v[k].w;
    } else {
        for (uint32_t k = 0; k < each; k++) sum += lo + k < cap ? b.blk_cnt[lo + k] : 0u;
    }
    const uint32_t x = wave_inclusive_scan(sum);
    if (lane == 63u) wsum[wave] = x;
    __syncthreads();
    uint32_t at = x - sum;
    for (uint32_t q = 0; q < wave; q++) at += wsum[q];
    if (each >= 4u) {
        const uint4 *v = reinterpret_cast<const uint4 *>(b.blk_cnt + lo);
        uint4 *out = reinterpret_cast<uint4 *>(b.blk_start + lo);
#pragma unroll 4
        for (uint32_t k = 0; k < each / 4u; k++) {
            const uint4 c = v[k];
            out[k] = make_uint4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
            at += c.x + c.y + c.z + c.w;
        }
    } else {
        for (uint32_t k = 0; k < each && lo + k < cap; k++) {
            b.blk_start[lo + k] = at;
            at += b.blk_cnt[lo + k];
        }
    }
}

template <uint32_t ITEMS>
__global__ __launch_bounds__(256) void k_block_list(const uint32_t *__restrict__ keys,
                                                    const uint32_t *__restrict__ prev_keys, uint32_t cap,
                                                    uint32_t batched, uint32_t *__restrict__ counters,
                                                    uint32_t *__restrict__ blist, uint32_t *__restrict__ nbr,
                                                    uint32_t cmp_wgs, uint32_t nbr_wgs, BlockCounts counts) {
    __shared__ uint32_t wsum[4];
    __shared__ uint32_t wg_base;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    if (blockIdx.x < cmp_wgs) {
        constexpr uint32_t SLOTS = 256u * ITEMS;
        for (uint32_t base = blockIdx.x * SLOTS; base < cap; base += cmp_wgs * SLOTS) {
            uint32_t occ[ITEMS];
            uint32_t mine = 0;
#pragma unroll
            for (uint32_t i = 0; i < ITEMS; i++) {
                const uint32_t s = base + tid * ITEMS + i;
                occ[i] = s < cap && keys[s] != SLOSH_NONE ? 1u : 0u;
                mine += occ[i];
            }
            uint32_t x = mine;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t y = __shfl_up(x, d);
                if ((int)lane >= d) x += y;
            }
            if (lane == 63) wsum[wave] = x;
            __syncthreads();
            uint32_t before = 0, total = 0;
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) {
                before += q < wave ? wsum[q] : 0u;
                total += wsum[q];
            }
            if (tid == 0) wg_base = total ? atomicAdd(&counters[CTR_NUM_BLOCKS], total) : 0u;
            __syncthreads();
            uint32_t o = wg_base + before + x - mine;
#pragma unroll
            for (uint32_t i = 0; i < ITEMS; i++)
                if (occ[i]) blist[o++] = base + tid * ITEMS + i;
            __syncthreads();  // wsum / wg_base are reused by the next run
        }
        return;
    }
    if (blockIdx.x < cmp_wgs + nbr_wgs) {
        for (uint32_t s = (blockIdx.x - cmp_wgs) * 16u + (tid >> 4); s < cap; s += nbr_wgs * 16u) {
            const uint32_t key = keys[s];
            if (key != SLOSH_NONE) block_neighbour(s, key, tid & 15u, nbr, keys, prev_keys, cap, batched);
        }
        return;
    }
    if (blockIdx.x == cmp_wgs + nbr_wgs) {
        scan_slots(counts, cap, wsum);
        return;
    }
    const uint32_t s0 = ((blockIdx.x - cmp_wgs - nbr_wgs - 1u) * 4u + wave) * 16u;
    uint64_t occ = __ballot(lane < 16u && s0 + lane < cap && keys[s0 + lane] != SLOSH_NONE);
    for (; occ; occ &= occ - 1ull) {
        const size_t at = (size_t)(s0 + (uint32_t)__ffsll((unsigned long long)occ) - 1u) * NODES_PER_BLOCK + lane;
        const uint32_t c = counts.cell_cnt[at];
        counts.cell_start[at] = wave_inclusive_scan(c) - c;
    }
}

// Stands for the sort in a timed steady-state substep, so that each pass is counted
// once per substep (its work is done by the kernels around it).
__global__ void k_no_sort() {}

// A particle's block key and cell; whether the block lies in the key space (one outside
// it aliases another one: reported, once per wave).
__device__ inline uint32_t block_of(const float4 *__restrict__ pos, uint32_t i, bool valid, float h, uint32_t batched,
                                    uint32_t *__restrict__ counters, uint32_t *cell) {
    uint32_t key = 0u;
    bool in_range = true;
    *cell = 0u;
    if (valid) {
        const float4 p = pos[i];
        int bx, by, bz;
        assoc_block_cell(h, p.x, p.y, p.z, &bx, &by, &bz, cell);
        key = pack_key(batched, __float_as_uint(p.w) >> 1, bx, by, bz);
        in_range = block_in_key_range(batched, bx, by, bz);
    }
    const uint64_t bad = __ballot(!in_range);
    if (bad && lane_id() == (uint32_t)(__ffsll((unsigned long long)bad) - 1))
        atomicOr(&counters[CTR_ERRORS], ERR_KEY_RANGE);
    return key;
}

// update_block_particle_count (sort.slang:208-246) of the full sort: block
// totals and per-(block, cell) ranks. `hv`: at the head of each run of equal block keys,
// the block's slot.
__device__ inline void count_particle(uint32_t i, bool valid, uint64_t bheads, uint32_t hv, uint32_t cell,
                                      uint32_t *__restrict__ cell_cnt, uint32_t *__restrict__ pslot,
                                      uint32_t *__restrict__ prank, uint32_t *__restrict__ counters,
                                      uint32_t *__restrict__ blk_cnt) {
    const uint32_t lane = lane_id();
    const uint32_t hid = __shfl(hv, run_head_of(bheads));
    const bool ok = valid && hid != SLOSH_NONE;
    // Block totals: one atomic per run of equal block keys.
    if (ok && ((bheads >> lane) & 1ull)) atomicAdd(&blk_cnt[hid], run_length(bheads));
    if (valid && hid == SLOSH_NONE) atomicOr(&counters[CTR_ERRORS], ERR_LOOKUP);
    const uint32_t sk = ok ? hid * NODES_PER_BLOCK + cell : SLOSH_NONE;
    // Per-(block, cell) rank: one atomic per run of equal (block, cell) keys.
    const uint64_t cheads = run_heads(sk, ok);
    uint32_t base = 0u;
    if (ok && ((cheads >> lane) & 1ull)) base = atomicAdd(&cell_cnt[sk], run_length(cheads));
    const int head = run_head_of(cheads);
    base = __shfl(base, head);
    if (valid) {
        pslot[i] = sk;
        prank[i] = base + (lane - (uint32_t)head);
    }
}

__global__ __launch_bounds__(256) void k_count(const float4 *__restrict__ pos, uint32_t n, float h, uint32_t batched,
                                               const uint32_t *__restrict__ keys, uint32_t cap,
                                               uint32_t *__restrict__ cell_cnt, uint32_t *__restrict__ pslot,
                                               uint32_t *__restrict__ prank, uint32_t *__restrict__ counters,
                                               uint32_t *__restrict__ blk_cnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    uint32_t cell;
    const uint32_t key = block_of(pos, i, valid, h, batched, counters, &cell);
    // Hash lookup by the head of each run of equal block keys, all runs at once.
    const uint64_t bheads = run_heads(key, valid);
    uint32_t hv = SLOSH_NONE;
    if (valid && ((bheads >> lane_id()) & 1ull)) hv = hash_find(keys, cap, key);
    count_particle(i, valid, bheads, hv, cell, cell_cnt, pslot, prank, counters, blk_cnt);
}

// k_touch_primary and k_count in one, where the counts of all slots were cleared before
// (so no particle can be counted before its block's counters are): the insertion gives
// each run's slot.
__global__ __launch_bounds__(256) void k_touch_count(const float4 *__restrict__ pos, uint32_t n, float h,
                                                     uint32_t batched, uint32_t *__restrict__ keys, uint32_t cap,
                                                     uint32_t *__restrict__ cell_cnt, uint32_t *__restrict__ pslot,
                                                     uint32_t *__restrict__ prank, uint32_t *__restrict__ counters,
                                                     uint32_t *__restrict__ blk_cnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    uint32_t cell;
    const uint32_t key = block_of(pos, i, valid, h, batched, counters, &cell);
    const uint64_t bheads = run_heads(key, valid);
    ListEntry none;
    const uint32_t hv =
        insert_blocks(keys, cap, batched, key, bheads & __ballot(valid), counters, BlockInit{}, none);
    count_particle(i, valid, bheads, hv, cell, cell_cnt, pslot, prank, counters, blk_cnt);
}

// Per block (one wavefront): exclusive scan of the 64 cell counts (offsets
// relative to the block's first slot). Waves [w0, w0 + nw) of the grid take
// list entries w0, w0 + nw, ...
__device__ inline void cell_starts(const uint32_t *__restrict__ blist, const uint32_t *__restrict__ cell_cnt,
                                   uint32_t *__restrict__ cell_start, uint32_t B, uint32_t w, uint32_t nw) {
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t k = w; k < B; k += nw) {
        const size_t at = (size_t)blist[k] * NODES_PER_BLOCK + lane;
        const uint32_t c = cell_cnt[at];
        cell_start[at] = wave_inclusive_scan(c) - c;
    }
}

// Exclusive scan of v[base, base + 4096) by one workgroup of 1024 threads (4
// consecutive entries per thread), written through `out` with `carry` added;
// returns the tile's total. Entry e is v[e] (list == null) or the block total
// blk_cnt[list[e]] written to out[list[e]]. Every thread must call it.
__device__ inline uint32_t scan_tile(const uint32_t *__restrict__ list, const uint32_t *__restrict__ v,
                                     uint32_t *__restrict__ out, uint32_t base, uint32_t B, uint32_t carry,
                                     uint32_t *wsum) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t idx = base + tid * 4u;
    uint32_t at[4], val[4];
#pragma unroll
    for (int j = 0; j < 4; j++) at[j] = idx + j < B ? (list ? list[idx + j] : idx + j) : 0u;
#pragma unroll
    for (int j = 0; j < 4; j++) val[j] = idx + j < B ? v[at[j]] : 0u;
    const uint32_t t = val[0] + val[1] + val[2] + val[3];
    uint32_t x = t;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(x, d);
        if ((int)lane >= d) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    if (wave == 0) {
        uint32_t w = lane < 16 ? wsum[lane] : 0u;
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) {
            uint32_t y = __shfl_up(w, d);
            if ((int)lane >= d) w += y;
        }
        if (lane < 16) wsum[lane] = w;
    }
    __syncthreads();
    uint32_t e = carry + (wave > 0 ? wsum[wave - 1] : 0u) + x - t;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (idx + j < B) out[at[j]] = e;
        e += val[j];
    }
    const uint32_t total = wsum[15];
    __syncthreads();
    return total;
}

// Exclusive scan of the block totals in block-list order: tiles of 4096 list entries scanned
// in parallel, then the tile totals, then the tile offsets added.
__global__ __launch_bounds__(1024) void k_block_scan_tiles(const uint32_t *__restrict__ blist,
                                                           const uint32_t *__restrict__ blk_cnt,
                                                           uint32_t *__restrict__ blk_start,
                                                           uint32_t *__restrict__ tile_sums,
                                                           const uint32_t *__restrict__ counters,
                                                           uint32_t scan_wgs, const uint32_t *__restrict__ cell_cnt,
                                                           uint32_t *__restrict__ cell_start) {
    __shared__ uint32_t wsum[16];
    const uint32_t B = counters[CTR_NUM_BLOCKS];
    if (blockIdx.x >= scan_wgs) {  // the remaining workgroups compute the cell offsets
        cell_starts(blist, cell_cnt, cell_start, B, (blockIdx.x - scan_wgs) * 16u + (threadIdx.x >> 6),
                    (gridDim.x - scan_wgs) * 16u);
        return;
    }
    for (uint32_t t = blockIdx.x; t * 4096u < B; t += scan_wgs) {
        const uint32_t total = scan_tile(blist, blk_cnt, blk_start, t * 4096u, B, 0u, wsum);
        if (threadIdx.x == 0) tile_sums[t] = total;
    }
}

__global__ __launch_bounds__(1024) void k_block_scan_top(uint32_t *__restrict__ tile_sums,
                                                         const uint32_t *__restrict__ counters) {
    __shared__ uint32_t wsum[16];
    const uint32_t B = counters[CTR_NUM_BLOCKS];
    const uint32_t ntiles = (B + 4095u) / 4096u;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < ntiles; base += 4096u)
        carry += scan_tile(nullptr, tile_sums, tile_sums, base, ntiles, carry, wsum);
}

__global__ __launch_bounds__(256) void k_block_scan_add(const uint32_t *__restrict__ blist,
                                                        uint32_t *__restrict__ blk_start,
                                                        const uint32_t *__restrict__ tile_sums,
                                                        const uint32_t *__restrict__ counters) {
    const uint32_t B = counters[CTR_NUM_BLOCKS];
    for (uint32_t k = 4096u + blockIdx.x * blockDim.x + threadIdx.x; k < B; k += gridDim.x * blockDim.x)
        blk_start[blist[k]] += tile_sums[k >> 12];
}

__global__ __launch_bounds__(256) void k_scatter(const uint32_t *__restrict__ pslot, const uint32_t *__restrict__ prank,
                                                 const uint32_t *__restrict__ cell_start,
                                                 const uint32_t *__restrict__ blk_start, uint32_t *__restrict__ perm,
                                                 uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t s = pslot[i];
    if (s != SLOSH_NONE) perm[blk_start[s / NODES_PER_BLOCK] + cell_start[s] + prank[i]] = i;
}

}  // namespace

// ---------------------------------------------------------------------------
// Host launchers.

static inline uint32_t div_up(uint64_t a, uint32_t b) { return (uint32_t)((a + b - 1) / b); }
static inline uint32_t min_u(uint32_t a, uint32_t b) { return a < b ? a : b; }

// `fast`: the previous substep's fused kernels prepared this table. Otherwise the full
// sort. `ev` (optional) brackets the whole sequence.
hipError_t launch_grid_build(const GridBuffers &g, const float4 *pos, uint32_t n, float h, uint32_t batched,
                             uint32_t cap, bool fast, const PassEvents *ev, hipStream_t stream) {
    if (fast) {
        if (ev) launch_kernel(ev, k_no_sort, dim3(1), dim3(64), 0, stream);
        return hipGetLastError();
    }
    const uint32_t slot_grid = min_u(div_up(cap, 256), 2048);
    const uint32_t part_grid = div_up(n, 256);
    const bool wide = cap > 65536u;
    const uint32_t cmp_wgs = wide ? min_u(div_up(cap, 2048), 2048) : min_u(div_up(cap, 256), 2048);
    const uint32_t nbr_wgs = min_u(div_up(cap, 16), 4096);
    auto list_kernel = wide ? k_block_list<8> : k_block_list<1>;
    PassEvents first, last;
    if (ev) {
        first.start = ev->start;
        last.stop = ev->stop;
    }
    const bool small = cap <= INDEX_CAP;
    launch_kernel(ev ? &first : nullptr, k_reset_table, dim3(slot_grid), dim3(256), 0, stream, g.keys, cap,
                  g.counters, g.rsum, small ? g.blk_cnt : nullptr, g.cell_cnt);
    BlockCounts counts;
    counts.blk_cnt = g.blk_cnt;
    counts.cell_cnt = g.cell_cnt;
    counts.blk_start = g.blk_start;
    counts.cell_start = g.cell_start;
    if (n > 0 && small) {
        launch_kernel(nullptr, k_touch_count, dim3(part_grid), dim3(256), 0, stream, pos, n, h, batched, g.keys, cap,
                      g.cell_cnt, g.pslot, g.prank, g.counters, g.blk_cnt);
    } else if (n > 0) {
        BlockInit init{};
        init.blk_cnt = g.blk_cnt;
        init.cell_cnt = g.cell_cnt;
        launch_kernel(nullptr, k_touch_primary, dim3(part_grid), dim3(256), 0, stream, pos, n, h, batched, g.keys,
                      cap, g.counters, init);
    }
    const PassEvents *sort_ev = n > 0 ? nullptr : (ev ? &last : nullptr);
    const uint32_t scan_wgs = n > 0 && small ? 1u + div_up(cap, 64) : 0u;
    launch_kernel(sort_ev, list_kernel, dim3(cmp_wgs + nbr_wgs + scan_wgs), dim3(256), 0, stream,
                  (const uint32_t *)g.keys, (const uint32_t *)g.prev_keys, cap, batched, g.counters, g.blist, g.nbr,
                  cmp_wgs, nbr_wgs, counts);
    if (n == 0) return hipGetLastError();
    if (!small) {
        launch_kernel(nullptr, k_count, dim3(part_grid), dim3(256), 0, stream, pos, n, h, batched,
                      (const uint32_t *)g.keys, cap, g.cell_cnt, g.pslot, g.prank, g.counters, g.blk_cnt);
        const uint32_t cell_wgs = min_u(div_up(cap, 16), 1024);  // 16 blocks (wavefronts) per workgroup
        const uint32_t tile_wgs = min_u(div_up(cap, 4096), 1024);
        launch_kernel(nullptr, k_block_scan_tiles, dim3(tile_wgs + cell_wgs), dim3(1024), 0, stream,
                      (const uint32_t *)g.blist, (const uint32_t *)g.blk_cnt, g.blk_start, g.tile_sums,
                      (const uint32_t *)g.counters, tile_wgs, (const uint32_t *)g.cell_cnt, g.cell_start);
        launch_kernel(nullptr, k_block_scan_top, dim3(1), dim3(1024), 0, stream, g.tile_sums,
                      (const uint32_t *)g.counters);
        launch_kernel(nullptr, k_block_scan_add, dim3(min_u(div_up(cap, 256), 4096)), dim3(256), 0, stream,
                      (const uint32_t *)g.blist, g.blk_start, (const uint32_t *)g.tile_sums,
                      (const uint32_t *)g.counters);
    }
    launch_kernel(ev ? &last : nullptr, k_scatter, dim3(part_grid), dim3(256), 0, stream, (const uint32_t *)g.pslot,
                  (const uint32_t *)g.prank, (const uint32_t *)g.cell_start, (const uint32_t *)g.blk_start, g.perm, n);
    return hipGetLastError();
}
