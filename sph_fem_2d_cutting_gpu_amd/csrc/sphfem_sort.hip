// Cell list of the locked Green grid (grid.cu:25-42, grid_gpu_green.cu:13-213) for gfx950:
//  * FP64 cell hash with C truncation; blanked particles keep their previous hash;
//  * stable LSD radix sort of (hash, index), 8-bit digits, 4096-key tiles, ranking inside a
//    tile by 64-lane ballot multisplit (stable: wave order, round order, lane order);
//  * cell boundaries from neighbouring sorted keys via a lane shuffle, and the gather of the
//    particle arrays (all 20 for the reference-form sort, or fused with init/predict/EOS/
//    artificial stress for the step).
#include "sphfem_physics.h"
#include "sphfem_rigid.h"

#pragma clang fp contract(off)

namespace sphfem {

constexpr int SORT_BS = 256;
constexpr int SORT_ITEMS = 16;
constexpr int SORT_TILE = SORT_BS * SORT_ITEMS;   // 4096 keys per block
constexpr int RADIX = 256;
constexpr int WAVE = 64;

__device__ __forceinline__ int hash_of(const DevConsts &c, sphfem_double2 pos) {
    int ix = (int)((pos.x - c.geom.bbmin_x) / c.geom.dx);
    int iy = (int)((pos.y - c.geom.bbmin_y) / c.geom.dx);
    return ix * c.geom.ny + iy;
}

// grid.cu:25-42 (blanked particles keep their previous hash)
__global__ void __launch_bounds__(SORT_BS) k_hash(DevConsts c, const double *__restrict__ blanked,
                                                  const sphfem_double2 *__restrict__ pos, int *__restrict__ hash, int N,
                                                  int num_cell, int *__restrict__ flags) {
    const int base = blockIdx.x * SORT_TILE;
    for (int it = 0; it < SORT_ITEMS; it++) {
        int i = base + it * SORT_BS + threadIdx.x;
        if (i >= N) break;
        int h = hash[i];
        if (blanked[i] != 1.) h = hash_of(c, pos[i]);
        if (h < 0 || h >= num_cell) {
            atomicOr(&flags[0], 1);
            h = h < 0 ? 0 : num_cell - 1;
        }
        hash[i] = h;
    }
}

__global__ void __launch_bounds__(SORT_BS) k_upsweep(const int *__restrict__ keys, int N, int shift,
                                                     int *__restrict__ hist, int nblocks) {
    __shared__ int lh[RADIX];
    for (int d = threadIdx.x; d < RADIX; d += SORT_BS) lh[d] = 0;
    __syncthreads();
    const int base = blockIdx.x * SORT_TILE;
    for (int it = 0; it < SORT_ITEMS; it++) {
        int i = base + it * SORT_BS + threadIdx.x;
        if (i >= N) break;
        atomicAdd(&lh[(keys[i] >> shift) & (RADIX - 1)], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < RADIX; d += SORT_BS) hist[d * nblocks + blockIdx.x] = lh[d];
}

// one block per digit: exclusive scan of that digit's per-tile counts, total into digit_tot
__global__ void __launch_bounds__(SORT_BS) k_scan_digits(int *__restrict__ hist, int nblocks,
                                                         int *__restrict__ digit_tot) {
    __shared__ int part[SORT_BS];
    int *row = hist + (long)blockIdx.x * nblocks;
    int per = (nblocks + SORT_BS - 1) / SORT_BS;
    int lo = threadIdx.x * per;
    int hi = min(lo + per, nblocks);
    int s = 0;
    for (int j = lo; j < hi; j++) s += row[j];
    part[threadIdx.x] = s;
    __syncthreads();
    // Hillis-Steele inclusive scan over 256 partials
    for (int off = 1; off < SORT_BS; off <<= 1) {
        int v = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (int j = lo; j < hi; j++) {
        int v = row[j];
        row[j] = run;
        run += v;
    }
    if (threadIdx.x == SORT_BS - 1) digit_tot[blockIdx.x] = part[SORT_BS - 1];
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    const unsigned lane = __lane_id();
    return lane ? ((~0ull) >> (64 - lane)) : 0ull;
}

// stable scatter of one pass; vals_in == nullptr means the values are the input positions.  old_keys
// (pass 0 of the step's sort): the previous sorted keys, whose cells are cleared by the particles that
// left them (a cell that keeps one of its particles gets its start again from the reorder)
__global__ void __launch_bounds__(SORT_BS) k_downsweep(const int *__restrict__ keys_in,
                                                       const int *__restrict__ vals_in,
                                                       int *__restrict__ keys_out, int *__restrict__ vals_out,
                                                       int N, int shift, const int *__restrict__ hist,
                                                       int nblocks, const int *__restrict__ digit_tot,
                                                       int *__restrict__ flags, const int *__restrict__ old_keys,
                                                       int *__restrict__ cell_start, int num_cell) {
    __shared__ int block_off[RADIX];
    __shared__ int wcount[SORT_BS / WAVE][RADIX];
    __shared__ int scan[RADIX];
    const int tid = threadIdx.x;
    const int w = tid / WAVE;
    const int lane = tid % WAVE;
    // digit bases: exclusive scan over the 256 digit totals
    scan[tid] = digit_tot[tid];
    for (int k = 0; k < SORT_BS / WAVE; k++) wcount[k][tid] = 0;
    __syncthreads();
    for (int off = 1; off < RADIX; off <<= 1) {
        int v = tid >= off ? scan[tid - off] : 0;
        __syncthreads();
        scan[tid] += v;
        __syncthreads();
    }
    block_off[tid] = (tid ? scan[tid - 1] : 0) + hist[(long)tid * nblocks + blockIdx.x];
    __syncthreads();

    int key[SORT_ITEMS], val[SORT_ITEMS], rank[SORT_ITEMS];
    const int base = blockIdx.x * SORT_TILE + w * (SORT_ITEMS * WAVE);
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        int i = base + r * WAVE + lane;
        bool valid = i < N;
        int k = valid ? keys_in[i] : 0;
        key[r] = k;
        val[r] = valid ? (vals_in ? vals_in[i] : i) : 0;
        if (valid && old_keys) {
            const int oh = old_keys[i];
            if (oh != k && oh >= 0 && oh < num_cell) cell_start[oh] = -1;
        }
        int d = (k >> shift) & (RADIX - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            uint64_t m = __ballot((d >> b) & 1);
            peers &= ((d >> b) & 1) ? m : ~m;
        }
        int before = __popcll(peers & lt);
        int cnt = __popcll(peers);
        int old = 0;
        if (valid) old = wcount[w][d];
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) wcount[w][d] = old + cnt;
        __builtin_amdgcn_wave_barrier();
        rank[r] = valid ? old + before : -1;
    }
    __syncthreads();
    // prefix of each digit over the waves of this block
    {
        int d = tid;
        int run = 0;
        for (int k = 0; k < SORT_BS / WAVE; k++) {
            int v = wcount[k][d];
            wcount[k][d] = run;
            run += v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        if (rank[r] < 0) continue;
        int d = (key[r] >> shift) & (RADIX - 1);
        int dst = block_off[d] + wcount[w][d] + rank[r];
        if ((unsigned)dst >= (unsigned)N) {   // cannot happen for a consistent histogram
            atomicOr(&flags[0], 2);
            continue;
        }
        keys_out[dst] = key[r];
        vals_out[dst] = val[r];
    }
}

__global__ void k_fill_int(int *p, long n, int v) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long stride = (long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

void launch_fill_int(sphfem_ctx *ctx, int *ptr, long n, int value) {
    if (n <= 0) return;
    int blocks = (int)std::min<long>(nblk(n, 256), 8192);
    KTimer t(ctx, "fill_int");
    k_fill_int<<<blocks, 256, 0, ctx->stream>>>(ptr, n, value);
}

void launch_hash(sphfem_ctx *ctx, sphfem_grid *g, const sphfem_particles &p) {
    // writes into p.hash (the reference's in-place layout)
    int N = (int)p.N;
    int nb = nblk(N, SORT_TILE);
    KTimer t(ctx, "hash");
    k_hash<<<nb, SORT_BS, 0, ctx->stream>>>(ctx->c, p.blanked, p.pos, p.hash, N, g->num_cell, ctx->d_flags);
}

// The passes of the multi-block radix sort from the unsorted keys in `src` to the sorted keys and the
// permutation in (k1, v1), by way of (k2, v2); `src` is k2 for an odd number of passes and k1 for an
// even one.  hist0: pass 0's per-tile histogram is already in g->hist; old_keys: see k_downsweep.
static void launch_radix_passes(sphfem_ctx *ctx, sphfem_grid *g, int N, int *k1, int *v1, int *k2, int *v2, bool hist0,
                                const int *old_keys) {
    const int nb = nblk(N, SORT_TILE);
    const int passes = (g->key_bits + 7) / 8;
    int *kin = passes % 2 ? k2 : k1, *vin = nullptr;
    for (int ps = 0; ps < passes; ps++) {
        const int shift = 8 * ps;
        int *kout = kin == k1 ? k2 : k1, *vout = kin == k1 ? v2 : v1;
        if (ps > 0 || !hist0) {
            KTimer t(ctx, "radix_upsweep");
            k_upsweep<<<nb, SORT_BS, 0, ctx->stream>>>(kin, N, shift, g->hist, nb);
        }
        {
            KTimer t(ctx, "radix_scan");
            k_scan_digits<<<RADIX, SORT_BS, 0, ctx->stream>>>(g->hist, nb, g->digit_tot);
        }
        {
            KTimer t(ctx, "radix_downsweep");
            k_downsweep<<<nb, SORT_BS, 0, ctx->stream>>>(kin, vin, kout, vout, N, shift, g->hist, nb, g->digit_tot,
                                                         ctx->d_flags, ps == 0 ? old_keys : nullptr, g->cell_start,
                                                         g->num_cell);
        }
        kin = kout;
        vin = vout;
    }
}

// Radix sort of (p.hash, index) leaving sorted keys in p.hash and the permutation in p.idx
// (in vals_out when given).
void launch_radix_sort(sphfem_ctx *ctx, sphfem_grid *g, sphfem_particles &p, int *vals_out) {
    const int N = (int)p.N;
    if ((g->key_bits + 7) / 8 % 2)
        (void)hipMemcpyAsync(g->keys_alt, p.hash, sizeof(int) * (size_t)N, hipMemcpyDeviceToDevice, ctx->stream);
    launch_radix_passes(ctx, g, N, p.hash, vals_out ? vals_out : p.idx, g->keys_alt, g->vals_alt, false, nullptr);
}

// ---------------------------------------------------------------------------------------------
// Re-sort of the step.  After a step the particles are stored in the previous sorted order, so the
// previous keys (p.hash) are ascending.  A particle keeps its cell unless it crossed a cell boundary
// (rare at dt ~ 1e-4 of the cell crossing time).  The stable sort of the new keys with the previous
// position as tie-break is then the merge of
//   U: unchanged positions, already in (key, position) order, and
//   C: changed positions sorted by (new key, position):
//   dest(C[r]) = r + P - |{c in C : c < P}|,  P = first p with (old[p], p) >= (key_c, c),
//   and the unchanged positions fill the other destinations in order,
// which is exactly the result of the full stable radix sort (same keys, same order).
// Three launches: the hash pass lists the changed particles (k_hash_mark), one workgroup ranks them
// (k_resort), and the reorder reads each destination's source off the sorted lists (ResortView), so no
// key or index array is written and read back in between.  The full sort runs on the first step and
// whenever more than `cap` particles changed cells: k_resort's workgroups run it in that one launch.
// Where the host knows of it before (force) and N is above SPHFEM_SORT_ONE_LAUNCH_MAX it is the
// multi-block radix sort, whose launches beat the queue's waits there (steps of 400k, 550k, 750k and 1M
// particles 303, 366, 443 and 549 us by the queue, 314, 362, 428 and 511 us by launches).  (Per step with
// the incremental path before: the hash pass, scan, three idle launches per radix pass, compaction, ranking
// and scatter, each a dependent launch of about 4.5 us.)
// Sorted keys and permutation end in (g->keys_alt, p.idx); the caller swaps keys_alt and p.hash.
// ---------------------------------------------------------------------------------------------

// grid.cu:25-42 hash; the changed particles (new hash, position) appended to clist in any order, their
// number counted in sync[RS_COUNT].  KEYS: also the new keys, and their digit-0 histogram per tile, for
// the multi-block sort.  Workgroups past nblocks (tool_blocks of them, when a FEM tool is given) do the
// tool's step start instead (tool_begin_item), which shares no data with the hash pass; a step without
// one clears its counters here, and a rigid tool advances in the first lane past nblocks.
// Bound by HBM: 28 B read per particle.
constexpr int HASH_BS = 1024;                       // 16 wavefronts per tile, 4 items per lane
constexpr int HASH_ITEMS = SORT_TILE / HASH_BS;
// slots of sphfem_grid::sync: changed particles of this step, then the work queue of k_resort
enum { RS_COUNT = 0, RS_TICKET = 1, RS_DONE = 2 };   // RS_DONE + phase: finished items of a phase
constexpr int RS_USED = RS_DONE + 2 * 4;             // at most four passes of two phases
static_assert(RS_USED <= SPHFEM_RESORT_SYNC, "counters");
constexpr int RS_ITEMS = 256;                        // work items of a phase at most, of whole tiles
// changes up to which their ranks are counted (one change a lane, m comparisons), above by a bitonic sort: steps of
// 65k particles with 90, 820, 1890 and 3140 changes 134, 142, 230 and 281 us by counting, 140, 146, 167 and 179
// by the sort
constexpr int RS_COUNTED = 768;

struct StepStart {            // what else begins with the step (see k_hash_mark)
    sphfem_tool tool;
    int tool_blocks;
    double dt;
    RigidTool *rigid;
};

template <bool KEYS>
__global__ void __launch_bounds__(HASH_BS) k_hash_mark(DevConsts c, const double *__restrict__ blanked,
                                                       const sphfem_double2 *__restrict__ pos,
                                                       const int *__restrict__ old_hash, int *__restrict__ hash_out,
                                                       int N, int num_cell, int *__restrict__ hist0, int nblocks,
                                                       int *flags, int *__restrict__ sync, int2 *__restrict__ clist,
                                                       int cap, StepStart st) {
    if ((int)blockIdx.x >= nblocks) {
        const int item = ((int)blockIdx.x - nblocks) * HASH_BS + (int)threadIdx.x;
        if (st.tool_blocks > 0) tool_begin_item(st.tool, 0.5 * st.dt, flags, item);
        else if (item == 0) rigid_move(st.rigid->g, st.dt);
        return;
    }
    __shared__ int lh[KEYS ? RADIX : 1];
    __shared__ int wc[SORT_TILE / 64];
    __shared__ int s_base;
    if constexpr (KEYS) {
        for (int d = threadIdx.x; d < RADIX; d += HASH_BS) lh[d] = 0;
        __syncthreads();
    }
    if (blockIdx.x == 0 && st.tool_blocks == 0 && threadIdx.x == 0) step_counters_clear(flags);
    const int base = blockIdx.x * SORT_TILE;
    // every load of the lane's items first, then the hashes: the pass waits for memory once
    int h[HASH_ITEMS];
    double bls[HASH_ITEMS];
    sphfem_double2 pss[HASH_ITEMS];
#pragma unroll
    for (int it = 0; it < HASH_ITEMS; it++) {
        const int i = base + it * HASH_BS + threadIdx.x;
        h[it] = i < N ? old_hash[i] : 0;
        bls[it] = i < N ? blanked[i] : 1.;
        pss[it] = i < N ? pos[i] : sphfem_double2{0., 0.};
    }
    unsigned long long moved[HASH_ITEMS];
#pragma unroll
    for (int it = 0; it < HASH_ITEMS; it++) {
        const int i = base + it * HASH_BS + threadIdx.x;
        const int oh = h[it];
        bool changed = false;
        if (i < N) {
            if (bls[it] != 1.) h[it] = hash_of(c, pss[it]);
            if (h[it] < 0 || h[it] >= num_cell) {
                atomicOr(&flags[0], 1);
                h[it] = h[it] < 0 ? 0 : num_cell - 1;
            }
            if constexpr (KEYS) {
                hash_out[i] = h[it];
                atomicAdd(&lh[h[it] & (RADIX - 1)], 1);
            }
            changed = h[it] != oh;
        }
        moved[it] = __ballot(changed);
        if (__lane_id() == 0) wc[it * (HASH_BS / 64) + (threadIdx.x >> 6)] = __popcll(moved[it]);
    }
    __syncthreads();
    if constexpr (KEYS)
        for (int d = threadIdx.x; d < RADIX; d += HASH_BS) hist0[d * nblocks + blockIdx.x] = lh[d];
    // one reservation per tile: the prefix over its 64 wavefront rows by the first wavefront
    if (threadIdx.x < 64) {
        const int v = wc[threadIdx.x];
        int incl = v;
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(incl, off);
            if ((int)threadIdx.x >= off) incl += u;
        }
        wc[threadIdx.x] = incl - v;
        if (threadIdx.x == 63) s_base = incl ? atomicAdd(&sync[RS_COUNT], incl) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < HASH_ITEMS; it++) {
        if (!((moved[it] >> __lane_id()) & 1ull)) continue;
        const int k = s_base + wc[it * (HASH_BS / 64) + (threadIdx.x >> 6)] + __popcll(moved[it] & lanemask_lt());
        if (k < cap) clist[k] = make_int2(h[it], base + it * HASH_BS + (int)threadIdx.x);
    }
}

// First position p with (old[p], p) >= (key, c), the old keys ascending.  The previous cell table gives
// the cell's run when it is occupied (checked against the keys: the table may be older than they are);
// else a binary search.
__device__ __forceinline__ int insert_position(const int *__restrict__ old_keys, const int *__restrict__ cell_start,
                                               int N, int key, int c) {
    const int s = cell_start[key];
    int lo = 0, hi = N;
    if (s >= 0 && s < N && old_keys[s] == key && (s == 0 || old_keys[s - 1] != key)) {
        if (c <= s) return s;
        lo = s;                          // the run starts here: gallop along it
        for (int w = 1; lo + w < N; w <<= 1) {
            const int q = lo + w;
            if (old_keys[q] != key || q >= c) { hi = q; break; }
        }
    }
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const int k = old_keys[mid];
        if (k < key || (k == key && mid < c)) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int wave_inclusive(int v) {
    for (int o = 1; o < WAVE; o <<= 1) {
        const int u = __shfl_up(v, o);
        if ((int)__lane_id() >= o) v += u;
    }
    return v;
}

// a store that other workgroups of the same launch read: written through to where every XCD sees it
__device__ __forceinline__ void st_agent(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// waits until `want` items of a phase are done; false (with the error bit set) if that never comes,
// which a queue in order cannot do: an item only waits for items taken before it, by running workgroups
__device__ __forceinline__ bool wait_done(int *counter, int want, int *flags) {
    for (int spin = 0; spin < (1 << 22); spin++) {
        if (__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want) return true;
        __builtin_amdgcn_s_sleep(2);
    }
    atomicOr(&flags[0], 2);
    return false;
}

// The ranking of the changed particles by the first workgroup, or (more than cap of them, or force) the
// full stable LSD radix sort by all of them.  The sort is a queue of items handed out in order by one
// counter: per pass the items' digit counts, then their scatter, each tile put in order in LDS first (tile
// order, and within a tile wavefront, row and lane order, as k_downsweep ranks them, so the permutation is the
// same).  An item is a run of whole tiles, at most RS_ITEMS of them, so that a workgroup meets one or two a
// phase.  Items of a phase wait for every item of the phase before, all of which were taken by workgroups
// that are running: the queue needs no co-resident grid.
// What other workgroups read is written through (st_agent) instead of by a fence that writes the whole L2 back
// per item: with a tile an item, a third phase for the counts' scan and that fence the sort took 122, 274 and
// 810 us at 270k, 1M and 4M particles (above the limit; the multi-block launches with their idle ones before
// 86, 115 and 265), now 41, 107 and 230.
// 72 registers at most: the workgroups that find nothing to do wait for room beside other streams' kernels (84
// registers: a sweep of 16 cases 1297 us against 1283).
// Latency bound: one workgroup on the incremental path (4.5 us at 160k and 5.6 us at 4M particles with 100 to
// 400 changes, where its launches took 46 us and 55 us); per phase of the full sort some 8 us at 131k and 18 us
// at 1M particles.
constexpr int RESORT_BS = 1024;
constexpr int RESORT_ITEMS = SORT_TILE / RESORT_BS;
__global__ void __launch_bounds__(RESORT_BS, 7) k_resort(DevConsts c, const double *__restrict__ blanked,
                                                      const sphfem_double2 *__restrict__ pos,
                                                      const int *__restrict__ old_keys, int *__restrict__ cell_start,
                                                      int N, int num_cell, int nb, int passes, int force, int cap,
                                                      int clear_old, int sort_here, int *k1, int *v1, int *k2, int *v2,
                                                      int *__restrict__ hist, int *flags, int *sync,
                                                      const int2 *__restrict__ clist, int2 *__restrict__ changed,
                                                      int *__restrict__ dests, int *__restrict__ removed) {
    __shared__ unsigned long long comp[SPHFEM_RESORT_CAP];
    __shared__ int gone[SPHFEM_RESORT_CAP];
    // the sort's per-wavefront digit counts and a tile in sorted order, in the bytes of the ranking's lists
    static_assert(sizeof(int) * (RESORT_BS / WAVE) * RADIX <= sizeof(gone) && SORT_TILE <= SPHFEM_RESORT_CAP, "LDS");
    int (*wcount)[RADIX] = reinterpret_cast<int (*)[RADIX]>(gone);
    int (*sums)[RESORT_BS] = reinterpret_cast<int (*)[RESORT_BS]>(gone);
    __shared__ int start[RADIX], cnt[RADIX], part[RADIX / WAVE];
    __shared__ int s_item, s_go;
    const int tid = threadIdx.x;
    const int m = sync[RS_COUNT];
    const bool full = force || m > cap;
    if (blockIdx.x == 0 && tid == 0) {
        flags[3] = full ? 1 : 2;
        flags[4] = m;
    }
    if (!full) {
        if (blockIdx.x != 0) return;
        // the changed particles by (new key, position) and their positions alone, by counting or a bitonic sort
        int np = 64;
        while (np < m) np <<= 1;
        for (int k = tid; k < np; k += RESORT_BS) {
            const int2 e = k < m ? clist[k] : make_int2(-1, INT_MAX);
            comp[k] = ((unsigned long long)(unsigned)e.x << 32) | (unsigned)e.y;
            gone[k] = e.y;
        }
        __syncthreads();
        if (m <= RS_COUNTED) {
            const unsigned long long mine = tid < m ? comp[tid] : 0ull;
            const int at = (int)(unsigned)mine;
            int rank = 0, rp = 0;
            if (tid < m)
                for (int q = 0; q < m; q++) {
                    const unsigned long long other = comp[q];
                    rank += other < mine;
                    rp += (int)(unsigned)other < at;
                }
            __syncthreads();
            if (tid < m) {
                comp[rank] = mine;
                gone[rp] = at;
            }
            __syncthreads();
        } else {
            for (int size = 2; size <= np; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int q = tid; q < np >> 1; q += RESORT_BS) {
                        const int a = 2 * q - (q & (stride - 1)), b = a + stride;
                        const bool up = (a & size) == 0;
                        const unsigned long long ca = comp[a], cb = comp[b];
                        if ((ca > cb) == up) {
                            comp[a] = cb;
                            comp[b] = ca;
                        }
                        const int ga = gone[a], gb = gone[b];
                        if ((ga > gb) == up) {
                            gone[a] = gb;
                            gone[b] = ga;
                        }
                    }
                    __syncthreads();
                }
            }
        }
        int P[SPHFEM_RESORT_CAP / RESORT_BS];
#pragma unroll
        for (int u = 0; u < SPHFEM_RESORT_CAP / RESORT_BS; u++) {
            const int r = tid + u * RESORT_BS;
            if (r < m) P[u] = insert_position(old_keys, cell_start, N, (int)(comp[r] >> 32), (int)(unsigned)comp[r]);
        }
        __syncthreads();                              // before any cell is cleared
#pragma unroll
        for (int u = 0; u < SPHFEM_RESORT_CAP / RESORT_BS; u++) {
            const int r = tid + u * RESORT_BS;
            if (r >= m) continue;
            const int at = (int)(unsigned)comp[r];
            int lo = 0, hi = m;                       // removed positions below P
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (gone[mid] < P[u]) lo = mid + 1;
                else hi = mid;
            }
            dests[r] = r + P[u] - lo;
            changed[r] = make_int2((int)(comp[r] >> 32), at);
            removed[r] = gone[r];
            // a cell that keeps one of its particles gets its start again from the reorder; one that all
            // of them left is cleared by each of them
            const int oh = old_keys[at];
            if (clear_old && oh >= 0 && oh < num_cell) cell_start[oh] = -1;
        }
        return;
    }
    if (!sort_here) return;
    const int w = tid / WAVE, lane = tid % WAVE;
    const uint64_t lt = lanemask_lt();
    const int span = (nb + RS_ITEMS - 1) / RS_ITEMS * SORT_TILE;      // keys of an item
    const int per_phase = (N + span - 1) / span;
    const int items = passes * 2 * per_phase;
    // the item of a turn is taken and published between two barriers and read into a scalar, so that the
    // loop's control flow is uniform for the compiler too: a lane-dependent branch next to the back edge
    // lets it send the other lanes round the loop alone
    if (tid == 0) s_item = atomicAdd(&sync[RS_TICKET], 1);
    __syncthreads();
    int item = __builtin_amdgcn_readfirstlane(s_item);
    while (item < items) {
        // pass, step of the pass (0 counts, 1 scatter) and the item's number in it
        const int phase = item / per_phase, at = item - phase * per_phase, ps = phase >> 1, shift = 8 * ps;
        if (phase > 0) {
            if (tid == 0) {
                s_go = wait_done(&sync[RS_DONE + phase - 1], per_phase, flags) ? 1 : 0;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // the finished items' writes, from any XCD
            }
            __syncthreads();
            if (__builtin_amdgcn_readfirstlane(s_go) == 0) return;
        }
        // pass ps reads (ki, vi) and writes (ko, vo); the last pass ends in (k1, v1)
        const bool to1 = (passes - ps) % 2 != 0;
        int *ki = to1 ? k2 : k1, *ko = to1 ? k1 : k2, *vo = to1 ? v1 : v2;
        const int *vi = to1 ? v2 : v1;
        const int first = at * span, last = first + span < N ? first + span : N;
        if ((phase & 1) == 0) {                       // digit counts of the item
            if (tid < RADIX) cnt[tid] = 0;
            __syncthreads();
            for (int i = first + tid; i < last; i += RESORT_BS) {
                int h;
                if (ps == 0) {                        // the keys themselves, as k_hash_mark computed them
                    const int oh = old_keys[i];
                    h = oh;
                    if (blanked[i] != 1.) h = hash_of(c, pos[i]);
                    h = h < 0 ? 0 : (h >= num_cell ? num_cell - 1 : h);
                    if (clear_old && h != oh && oh >= 0 && oh < num_cell) cell_start[oh] = -1;
                    st_agent(&ki[i], h);
                } else {
                    h = ki[i];
                }
                // nearly sorted keys: most wavefronts hold one value of the higher digits
                const int d = (h >> shift) & (RADIX - 1), d0 = __builtin_amdgcn_readfirstlane(d);
                const uint64_t same = __ballot(d == d0);
                if (d != d0) atomicAdd(&cnt[d], 1);
                else if (__popcll(same & lt) == 0) atomicAdd(&cnt[d0], __popcll(same));
            }
            __syncthreads();
            if (tid < RADIX) st_agent(&hist[(long)at * RADIX + tid], cnt[tid]);
        } else {
            // the item's digits in the output: lower digits of all items, then lower items; the items' counts
            // are summed by a quarter of the lanes each
            int key[RESORT_ITEMS], val[RESORT_ITEMS], next_key[RESORT_ITEMS], next_val[RESORT_ITEMS];
            auto load = [&](int base) {               // of a tile, while the work before it runs
#pragma unroll
                for (int q = 0; q < RESORT_ITEMS; q++) {
                    const int i = base + w * (RESORT_ITEMS * WAVE) + q * WAVE + lane;
                    next_key[q] = i < last ? ki[i] : 0;
                    next_val[q] = i < last ? (ps == 0 ? i : vi[i]) : 0;
                }
            };
            load(first);
            {
                const int d = tid & (RADIX - 1);
                int below = 0, all = 0;
                for (int q0 = tid / RADIX; q0 < per_phase; q0 += 8 * (RESORT_BS / RADIX)) {
                    int v[8];                         // loaded together
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const int q = q0 + u * (RESORT_BS / RADIX);
                        v[u] = q < per_phase ? hist[(long)q * RADIX + d] : 0;
                    }
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        all += v[u];
                        below += q0 + u * (RESORT_BS / RADIX) < at ? v[u] : 0;
                    }
                }
                sums[0][tid] = below;
                sums[1][tid] = all;
            }
            __syncthreads();
            int offset = 0;                           // of digit tid
            if (tid < RADIX) {
                int all = 0;
                for (int q = 0; q < RESORT_BS / RADIX; q++) {
                    offset += sums[0][q * RADIX + tid];
                    all += sums[1][q * RADIX + tid];
                }
                const int incl = wave_inclusive(all);
                if (lane == WAVE - 1) part[w] = incl;
                offset += incl - all;
            }
            __syncthreads();
            if (tid < RADIX)
                for (int k = 0; k < w; k++) offset += part[k];
            for (int base = first; base < last; base += SORT_TILE) {
                int rank[RESORT_ITEMS];
#pragma unroll
                for (int q = 0; q < RESORT_ITEMS; q++) {
                    key[q] = next_key[q];
                    val[q] = next_val[q];
                }
                if (base + SORT_TILE < last) load(base + SORT_TILE);
                for (int k = tid; k < (RESORT_BS / WAVE) * RADIX; k += RESORT_BS) (&wcount[0][0])[k] = 0;
                __syncthreads();
#pragma unroll
                for (int q = 0; q < RESORT_ITEMS; q++) {
                    const bool valid = base + w * (RESORT_ITEMS * WAVE) + q * WAVE + lane < N;
                    const int d = (key[q] >> shift) & (RADIX - 1);
                    uint64_t peers = __ballot(valid);
#pragma unroll
                    for (int b = 0; b < 8; b++) {
                        const uint64_t mm = __ballot((d >> b) & 1);
                        peers &= ((d >> b) & 1) ? mm : ~mm;
                    }
                    const int before = __popcll(peers & lt);
                    int old = 0;
                    if (valid) old = wcount[w][d];
                    __builtin_amdgcn_wave_barrier();
                    if (valid && before == 0) wcount[w][d] = old + __popcll(peers);
                    __builtin_amdgcn_wave_barrier();
                    rank[q] = valid ? old + before : -1;
                }
                __syncthreads();
                // each digit's prefix over the tile's wavefronts, its start in the tile's sorted order, and
                // (cnt) its place in the output less that
                int mine = 0, incl = 0;
                if (tid < RADIX) {
                    for (int k = 0; k < RESORT_BS / WAVE; k++) {
                        const int v = wcount[k][tid];
                        wcount[k][tid] = mine;
                        mine += v;
                    }
                    incl = wave_inclusive(mine);
                    if (lane == WAVE - 1) part[w] = incl;
                }
                __syncthreads();
                if (tid < RADIX) {
                    for (int k = 0; k < w; k++) incl += part[k];
                    start[tid] = incl - mine;
                    cnt[tid] = offset - (incl - mine);
                    offset += mine;
                }
                __syncthreads();
                // the tile in sorted order, so that the output is written in runs
#pragma unroll
                for (int q = 0; q < RESORT_ITEMS; q++) {
                    if (rank[q] < 0) continue;
                    const int d = (key[q] >> shift) & (RADIX - 1);
                    comp[start[d] + wcount[w][d] + rank[q]] =
                        ((unsigned long long)(unsigned)key[q] << 32) | (unsigned)val[q];
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < RESORT_ITEMS; q++) {
                    const int l = q * RESORT_BS + tid;
                    if (base + l >= N) break;
                    const int k = (int)(comp[l] >> 32), v = (int)(unsigned)comp[l];
                    const int dst = cnt[(k >> shift) & (RADIX - 1)] + l;
                    if ((unsigned)dst >= (unsigned)N) {   // cannot happen for consistent counts
                        atomicOr(&flags[0], 2);
                        continue;
                    }
                    st_agent(&ko[dst], k);
                    st_agent(&vo[dst], v);
                }
            }
        }
        stores_done_barrier();                        // this item's writes before it counts as done
        if (tid == 0) {
            atomicAdd(&sync[RS_DONE + phase], 1);
            s_item = atomicAdd(&sync[RS_TICKET], 1);
        }
        __syncthreads();
        item = __builtin_amdgcn_readfirstlane(s_item);
    }
}

// Re-sort of the step: the lists of the incremental path, or the sorted keys and permutation in
// (g->keys_alt, p.idx); what each destination's source is, resort_source tells the reorder.
void launch_resort(sphfem_ctx *ctx, sphfem_grid *g, sphfem_particles &p, sphfem_tool *tool, sphfem_rigid_tool *rt) {
    const int N = (int)p.N;
    const int nb = nblk(N, SORT_TILE);
    int *flags = ctx->d_flags;
    const int cap = std::min(g->resort_limit, SPHFEM_RESORT_CAP);
    const int force = (g->first_sort || cap <= 0) ? 1 : 0;
    const int passes = (g->key_bits + 7) / 8;
    const int clear_old = g->first_sort ? 0 : 1;
    // a full sort known beforehand, and above the size where the multi-block launches win
    const bool launches = force && N > SPHFEM_SORT_ONE_LAUNCH_MAX;
    int *unsorted = passes % 2 ? g->keys_tmp : g->keys_alt;
    StepStart st{};
    if (tool) {
        st.tool = *tool;
        st.tool_blocks = nblk(std::max(std::max(tool->n_nodes, tool->n_seg), 1), HASH_BS);
    }
    st.dt = ctx->c.dt;
    st.rigid = rt ? rt->dev : nullptr;
    const int extra = tool ? st.tool_blocks : (rt ? 1 : 0);
    {
        KTimer t(ctx, tool ? "hash_tool_begin" : "hash");
        if (!launches)
            k_hash_mark<false><<<nb + extra, HASH_BS, 0, ctx->stream>>>(ctx->c, p.blanked, p.pos, p.hash, nullptr, N,
                                                                        g->num_cell, nullptr, nb, flags, g->sync,
                                                                        g->clist, cap, st);
        else
            k_hash_mark<true><<<nb + extra, HASH_BS, 0, ctx->stream>>>(ctx->c, p.blanked, p.pos, p.hash, unsorted, N,
                                                                       g->num_cell, g->hist, nb, flags, g->sync,
                                                                       g->clist, cap, st);
    }
    {
        KTimer t(ctx, "resort");
        const int blocks = launches ? 1 : std::min(nb, 256);
        k_resort<<<blocks, RESORT_BS, 0, ctx->stream>>>(ctx->c, p.blanked, p.pos, p.hash, g->cell_start, N,
                                                        g->num_cell, nb, passes, force, cap, clear_old,
                                                        launches ? 0 : 1, g->keys_alt, p.idx, g->keys_tmp,
                                                        g->vals_alt, g->hist, flags, g->sync, g->clist,
                                                        g->changed, g->dests, g->removed);
    }
    if (launches)
        launch_radix_passes(ctx, g, N, g->keys_alt, p.idx, g->keys_tmp, g->vals_alt, true,
                            clear_old ? p.hash : nullptr);
}

// What the reorder reads of the re-sort: on the incremental path (flags[3] == 2) the sorted destinations
// of the changed particles, the changed particles (key, position) in that order and the removed
// positions, else the sorted keys and sources.  It writes the sorted keys and sources of the incremental
// path, and clears the re-sort's counters for the next step.
struct ResortView {
    const int *old_keys;
    int *keys, *src;                 // sorted keys and sources: read (full sort) or written (incremental)
    const int *dests, *removed;
    const int2 *changed;
    int *sync;
};

// number of entries of the ascending list a[0..m) below x, by the lanes of a wavefront (all 64 of them,
// x uniform): one load per 64-fold step
__device__ __forceinline__ int wave_lower_bound(const int *__restrict__ a, int m, int x) {
    const int lane = (int)__lane_id();
    const int stride = (m + 63) >> 6;
    int first = 0;
    if (stride > 1) {
        const bool below = lane * stride < m && a[lane * stride] < x;
        const int c = __popcll(__ballot(below));
        if (c == 0) return 0;
        first = (c - 1) * stride;
    }
    const int left = m - first < stride ? m - first : stride;
    const int span = stride > 1 ? left : m;
    return first + __popcll(__ballot(lane < span && a[first + (lane < span ? lane : 0)] < x));
}

// the same for entries a[j] - j, by one lane
__device__ __forceinline__ int lower_bound_lane(const int *__restrict__ a, int m, int x, bool minus_j) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] - (minus_j ? mid : 0) < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// source s and key h of sorted position i on the incremental path, by one lane
__device__ __forceinline__ void resort_source_lane(const ResortView &v, int m, int N, int i, int &h, int &s) {
    const int a = lower_bound_lane(v.dests, m, i, false);
    if (a < m && v.dests[a] == i) {
        const int2 e = v.changed[a];
        h = e.x;
        s = e.y;
        return;
    }
    const int k = i - a;                                             // rank among the unchanged
    s = k + lower_bound_lane(v.removed, m, k + 1, true);
    h = (unsigned)s < (unsigned)N ? v.old_keys[s] : -1;
}

// source s and key h of sorted position i = i0 + lane, and the key hp of position i - 1, for a whole
// wavefront (every lane executes this; lanes past N get sources that are not used).  Most wavefronts lie
// between two changes: one shift for all lanes, found by two wavefront-wide searches.
__device__ __forceinline__ void resort_source(const ResortView &v, const int *__restrict__ flags, int N, int i, int &h,
                                              int &s, int &hp) {
    const int lane = (int)__lane_id();
    const int i0 = __builtin_amdgcn_readfirstlane(i);
    const bool in = i < N;
    if (flags[3] != 2) {
        h = in ? v.keys[i] : 0;
        s = in ? v.src[i] : 0;
        hp = __shfl_up(h, 1);
        if (lane == 0 && i > 0) hp = v.keys[i - 1];
        return;
    }
    const int m = flags[4];
    const int lo = i0 > 0 ? i0 - 1 : 0;
    const int last = i0 + 63 < N ? i0 + 63 : N - 1;
    const int a = wave_lower_bound(v.dests, m, lo);
    const int next = a < m ? v.dests[a] : N;
    // removed positions up to the unchanged of rank lo - a: of the ascending removed[j] - j, those <= it
    const int k0 = lo - a;
    int b = 0;
    {
        const int stride = (m + 63) >> 6;
        int first = 0;
        bool none = m == 0;
        if (stride > 1) {
            const int j = lane * stride;
            const int c = __popcll(__ballot(j < m && v.removed[j] - j <= k0));
            none = c == 0;
            first = none ? 0 : (c - 1) * stride;
        }
        const int span = stride > 1 ? (m - first < stride ? m - first : stride) : m;
        const int j = first + (lane < span ? lane : 0);
        const int c = __popcll(__ballot(!none && lane < span && v.removed[j] - j <= k0));
        b = none ? 0 : first + c;
    }
    const int next_gone = b < m ? v.removed[b] - b : N;
    if (next > last && next_gone > last - a) {
        s = i - a + b;
        h = in && (unsigned)s < (unsigned)N ? v.old_keys[s] : -1;
        hp = __shfl_up(h, 1);
        const int sp = i - 1 - a + b;
        if (lane == 0 && i > 0) hp = (unsigned)sp < (unsigned)N ? v.old_keys[sp] : -1;
    } else {
        h = -1;
        s = 0;
        if (in) resort_source_lane(v, m, N, i, h, s);
        hp = __shfl_up(h, 1);
        int sp = 0;
        if (lane == 0 && i > 0) resort_source_lane(v, m, N, i - 1, hp, sp);
    }
    if (in) {
        v.keys[i] = h;
        v.src[i] = s;
    }
}

// grid_gpu_green.cu:13-115: boundaries + gather of the 20 arrays into the buffer
__global__ void __launch_bounds__(256) k_reorder_full(const sphfem_particles p, sphfem_particles b,
                                                      int *__restrict__ cell_start, int *__restrict__ cell_end,
                                                      int num_cell, int *__restrict__ flags) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    int N = (int)p.N;
    if (i >= N) return;
    int h = p.hash[i];
    const int s = p.idx[i];
    if ((unsigned)h >= (unsigned)num_cell || (unsigned)s >= (unsigned)N) {
        atomicOr(&flags[0], 4);
        return;
    }
    int hp = __shfl_up(h, 1);
    if (__lane_id() == 0 && i > 0) hp = p.hash[i - 1];
    if (i == 0 || h != hp) {
        cell_start[h] = i;
        if (i > 0) cell_end[hp] = i;
    }
    if (i == N - 1) cell_end[h] = i + 1;
    b.pos[i] = p.pos[s];
    b.vel[i] = p.vel[s];
    b.fc[i] = p.fc[s];
    b.ft[i] = p.ft[s];
    b.h[i] = p.h[s];
    b.n[i] = p.n[s];
    b.rho[i] = p.rho[s];
    b.S[i] = p.S[s];
    b.eps_pl[i] = p.eps_pl[s];
    b.eps_pl_dot[i] = p.eps_pl_dot[s];
    b.T[i] = p.T[s];
    b.fixed[i] = p.fixed[s];
    b.blanked[i] = p.blanked[s];
    b.tool_particle[i] = p.tool_particle[s];
    b.pos_t[i] = p.pos_t[s];
    b.vel_t[i] = p.vel_t[s];
    b.rho_t[i] = p.rho_t[s];
    b.S_t[i] = p.S_t[s];
    b.T_t[i] = p.T_t[s];
    b.on_seg[i] = p.on_seg[s];
}

void launch_reorder_full(sphfem_ctx *ctx, sphfem_grid *g, const sphfem_particles &p) {
    KTimer t(ctx, "reorder");
    k_reorder_full<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(p, g->buf, g->cell_start, g->cell_end,
                                                            g->num_cell, ctx->d_flags);
}

// ---------------------------------------------------------------------------------------------
// grid_gpu_rothlin.cu:129-249: the stable sort's permutation gathers idx (which therefore keeps
// particle labels), pos, vel, fc, h, rho, S, eps_pl, eps_pl_dot, fixed, blanked, tool_particle, T,
// pos_t, vel_t, rho_t, S_t, T_t and on_seg in place; ft and n are not gathered (as in the
// reference).  The reference's on_seg copy takes the gathered idx buffer (:244-245), which would
// leave particle labels where segment numbers are expected; on_seg is gathered here.  The gather
// writes the buffer and a second pass copies it back, so the particle arrays keep their addresses.
// ---------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_rothlin_gather(const sphfem_particles p, sphfem_particles b,
                                                        const int *__restrict__ perm, int *__restrict__ flags) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = (int)p.N;
    if (i >= N) return;
    const int s = perm[i];
    if ((unsigned)s >= (unsigned)N) {
        atomicOr(&flags[0], 4);
        return;
    }
    b.idx[i] = p.idx[s];
    b.pos[i] = p.pos[s];
    b.vel[i] = p.vel[s];
    b.fc[i] = p.fc[s];
    b.h[i] = p.h[s];
    b.rho[i] = p.rho[s];
    b.S[i] = p.S[s];
    b.eps_pl[i] = p.eps_pl[s];
    b.eps_pl_dot[i] = p.eps_pl_dot[s];
    b.fixed[i] = p.fixed[s];
    b.blanked[i] = p.blanked[s];
    b.tool_particle[i] = p.tool_particle[s];
    b.T[i] = p.T[s];
    b.pos_t[i] = p.pos_t[s];
    b.vel_t[i] = p.vel_t[s];
    b.rho_t[i] = p.rho_t[s];
    b.S_t[i] = p.S_t[s];
    b.T_t[i] = p.T_t[s];
    b.on_seg[i] = p.on_seg[s];
}

__global__ void __launch_bounds__(256) k_rothlin_copy_back(sphfem_particles p, const sphfem_particles b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int)p.N) return;
    p.idx[i] = b.idx[i];
    p.pos[i] = b.pos[i];
    p.vel[i] = b.vel[i];
    p.fc[i] = b.fc[i];
    p.h[i] = b.h[i];
    p.rho[i] = b.rho[i];
    p.S[i] = b.S[i];
    p.eps_pl[i] = b.eps_pl[i];
    p.eps_pl_dot[i] = b.eps_pl_dot[i];
    p.fixed[i] = b.fixed[i];
    p.blanked[i] = b.blanked[i];
    p.tool_particle[i] = b.tool_particle[i];
    p.T[i] = b.T[i];
    p.pos_t[i] = b.pos_t[i];
    p.vel_t[i] = b.vel_t[i];
    p.rho_t[i] = b.rho_t[i];
    p.S_t[i] = b.S_t[i];
    p.T_t[i] = b.T_t[i];
    p.on_seg[i] = b.on_seg[i];
}

// grid_gpu_rothlin.cu:19-126: unique_by_key + |differences| + scatter + inclusive scan with the
// last cell fixed up yields offsets[c] = number of sorted keys below c, so every cell gets
// cell_start[c] = lower_bound(c) and cell_end[c] = lower_bound(c + 1) (start == end when empty).
// One thread per cell, two binary searches over the sorted keys (L2-resident for these sizes).
__device__ __forceinline__ int lower_bound_keys(const int *__restrict__ keys, int N, int c) {
    int lo = 0, n = N;
    while (n > 0) {
        const int half = n >> 1;
        if (keys[lo + half] < c) {
            lo += half + 1;
            n -= half + 1;
        } else {
            n = half;
        }
    }
    return lo;
}

__global__ void __launch_bounds__(256) k_cells_dense(const int *__restrict__ keys, int N, int num_cell,
                                                     int *__restrict__ cell_start, int *__restrict__ cell_end) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= num_cell) return;
    cell_start[c] = lower_bound_keys(keys, N, c);
    cell_end[c] = lower_bound_keys(keys, N, c + 1);
}

void launch_cells_dense(sphfem_ctx *ctx, const int *sorted_keys, int N, int num_cell, int *cell_start, int *cell_end) {
    KTimer t(ctx, "cells_dense");
    k_cells_dense<<<nblk(num_cell, 256), 256, 0, ctx->stream>>>(sorted_keys, N, num_cell, cell_start, cell_end);
}

__global__ void k_iota(int *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

void launch_iota(sphfem_ctx *ctx, int *ptr, int n) {
    k_iota<<<nblk(n, 256), 256, 0, ctx->stream>>>(ptr, n);
}

// grid.cu:88-127: smallest and largest x and y over all particle positions and the largest h
// (blanked particles included, as the reference's min/max_element over the whole arrays).
// Positions are finite; min and max of finite values do not depend on the reduction order.
__device__ __forceinline__ void bbox_combine(double *a, const double *b) {
    a[0] = fmin(a[0], b[0]);
    a[1] = fmin(a[1], b[1]);
    a[2] = fmax(a[2], b[2]);
    a[3] = fmax(a[3], b[3]);
    a[4] = fmax(a[4], b[4]);
}

__device__ void bbox_block_reduce(double *v, double *out) {
    __shared__ double red[5][256 / 64];
    for (int off = 32; off > 0; off >>= 1) {
        double o[5];
        for (int k = 0; k < 5; k++) o[k] = __shfl_xor(v[k], off);
        bbox_combine(v, o);
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0)
        for (int k = 0; k < 5; k++) red[k][wave] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc[5];
        for (int k = 0; k < 5; k++) acc[k] = red[k][0];
        for (int w = 1; w < 256 / 64; w++) {
            double o[5];
            for (int k = 0; k < 5; k++) o[k] = red[k][w];
            bbox_combine(acc, o);
        }
        for (int k = 0; k < 5; k++) out[k] = acc[k];
    }
}

__global__ void __launch_bounds__(256) k_bbox_partial(const sphfem_double2 *__restrict__ pos,
                                                      const double *__restrict__ h, int N, double *__restrict__ part) {
    double v[5] = {INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const sphfem_double2 q = pos[i];
        const double o[5] = {q.x, q.y, q.x, q.y, h[i]};
        bbox_combine(v, o);
    }
    bbox_block_reduce(v, part + 5 * blockIdx.x);
}

__global__ void __launch_bounds__(256) k_bbox_final(const double *__restrict__ part, int nb, double *__restrict__ out) {
    double v[5] = {INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int b = threadIdx.x; b < nb; b += blockDim.x) bbox_combine(v, part + 5 * b);
    bbox_block_reduce(v, out);
}

void launch_bbox(sphfem_ctx *ctx, const sphfem_particles &p, double *part, double *out) {
    const int nb = std::max(1, std::min(nblk(p.N, 256), SPHFEM_BBOX_BLOCKS));
    KTimer t(ctx, "bbox");
    k_bbox_partial<<<nb, 256, 0, ctx->stream>>>(p.pos, p.h, (int)p.N, part);
    k_bbox_final<<<1, 256, 0, ctx->stream>>>(part, nb, out);
}

// p.hash must hold the keys; leaves the sorted keys in p.hash, the gathered arrays in place and
// the dense cell table in the grid
void launch_rothlin_sort(sphfem_ctx *ctx, sphfem_grid *g, sphfem_particles &p) {
    launch_radix_sort(ctx, g, p, g->perm);
    {
        KTimer t(ctx, "rothlin_gather");
        k_rothlin_gather<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(p, g->buf, g->perm, ctx->d_flags);
    }
    {
        KTimer t(ctx, "rothlin_copy_back");
        k_rothlin_copy_back<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(p, g->buf);
    }
    launch_cells_dense(ctx, p.hash, (int)p.N, g->num_cell, g->cell_start, g->cell_end);
}

// a live particle with a non-finite pair input (interactions_gpu.cu:143-379 reads pos, vel, h, rho, p,
// S, R and T of both particles): the pair kernels then evaluate the reference's full 5x5-cell window,
// where such a neighbour turns the sums NaN even outside the kernel support.  A finite sum that
// overflows, or a density or velocity out of the range of pair_inputs_in_range, only sends the step down
// that (exact, slower) path.
__device__ __forceinline__ void flag_nonfinite(int *__restrict__ form, double blanked, sphfem_double2 pos,
                                               sphfem_double2 vel, sphfem_double4 S, double rho, double T, double h,
                                               double pr, sphfem_double4 R) {
    const double s = ((pos.x + pos.y) + (vel.x + vel.y)) + ((S.x + S.y) + (S.z + rho)) + ((T + h) + (pr + R.x)) +
                     (R.y + R.z);
    if (blanked != 1. && !(isfinite(s) && pair_inputs_in_range(rho, vel))) form[0] = 1;      // WINDOW
}

// FP32C neighbour records (RecView) of one sorted particle.  The position is rounded to cell / 2^28 from
// FP64 and wrapped (finer than FP32 relative to the cell corner); the stress terms are the per-particle
// factors of the pair sum, (S - p)/rho^2 and S_xy/rho^2; the temperature is stored as T - T_init, so
// that the FP32 differences T_i - T_j of a nearly uniform field keep ~1e-7 of the deviation instead of
// ~1e-7 of T.
__device__ __forceinline__ void write_records(const DevConsts &c, const RecView &rec, double inv_dx,
                                              int *__restrict__ form, int i, int h, sphfem_double2 pos,
                                              sphfem_double2 vel, sphfem_double4 S, double rho, double T,
                                              double blanked, double tool, double hh, double pr, sphfem_double4 R) {
    const int ny = c.geom.ny;
    const int ix = h / ny, iy = h - ix * ny;
    // cell units from the centre of the particle's cell.  Blanked particles are put 8 cells from it along
    // both axes, where no kernel reaches them from the 5x5 cells.  Above or below the grid a key names a
    // cell of the next or the previous column: those particles see only each other, and keep their place
    // relative to that cell, 8 cells aside in x or in y.  One that lies near neither is put with the blanked
    // ones, and the general form reads its position elsewhere.
    double cx = (pos.x - c.geom.bbmin_x) * inv_dx - (ix + 0.5);
    double cy = (pos.y - c.geom.bbmin_y) * inv_dx - (iy + 0.5);
    const bool live = blanked != 1.;
    bool near = fabs(cx) <= 1.6 && fabs(cy) <= 1.6;
    int turn = 0;
    const double unit = (double)(1 << SPHFEM_POS_BITS);
    if (live && !near) {
        rec.away[i] = make_double2((cx + (ix + 0.5)) * unit, (cy + (iy + 0.5)) * unit);
        turn = cy > 0. ? 1 : -1;
        cx += turn;
        cy -= turn * (double)ny;
        near = fabs(cx) <= 1.6 && fabs(cy) <= 1.6 && ny >= 10;
    }
    const int half = 1 << (SPHFEM_POS_BITS - 1);
    const bool put = live && near;
    unsigned ux = ((unsigned)ix << SPHFEM_POS_BITS) + half, uy = ((unsigned)iy << SPHFEM_POS_BITS) + half;
    if (!put || turn > 0) ux ^= 1u << 31;
    if (!put || turn < 0) uy ^= 1u << 31;
    if (put) {
        ux += (unsigned)(int)rint(cx * unit);
        uy += (unsigned)(int)rint(cy * unit);
    }
    const int2 r0 = make_int2((int)ux, (int)uy);
    // the form of the pair sums: one store per wavefront and word
    const int bits = (__any(live && hh != c.geom.dx) ? SPHFEM_FORM_WIDTH : 0) |
                     (__any(live && !near) ? SPHFEM_FORM_AWAY : 0) |
                     (__any(live && hh > 2. * c.geom.dx) ? SPHFEM_FORM_REACH : 0);
    if (bits != 0 && (int)__lane_id() == __ffsll((long long)__ballot(1)) - 1)
        for (int k = 1; k < SPHFEM_FORM_WORDS; k++)
            if (bits >> k & 1) form[k] = 1;
    const double inv_rho = 1. / rho, rho21 = inv_rho * inv_rho;
    const float vol = (float)(c.phys.mass * inv_rho);
    float4 r1, r2, r3;
    r1.x = (float)vel.x;
    r1.y = (float)vel.y;
    r1.z = tool == 0. ? (float)((S.x - pr) * rho21) : 0.f;
    r1.w = tool == 0. ? (float)(S.y * rho21) : 0.f;
    r2.x = tool == 0. ? (float)((S.z - pr) * rho21) : 0.f;
    r2.y = (float)R.x;
    r2.z = (float)R.y;
    r2.w = (float)R.z;
    r3.x = tool == 1. ? -vol : vol;
    r3.y = (float)rho;
    r3.z = live ? (float)(c.corr.alpha * sqrtf_d(c.phys.K * inv_rho)) : -INFINITY;
    r3.w = (float)(T - c.trml_wp.T_init);    // only differences enter the sums: offset from T_init
    rec.pos[i] = r0;
    rec.r1[i] = r1;
    rec.r2[i] = r2;
    rec.r3[i] = r3;
    rec.h[i] = (float)(hh * inv_dx * unit);
}

// FP32C records of an already sorted state as it stands (no predictor): the inputs of
// interactions_monaghan, with p and R as material_eos and corrector_artificial_stress left them
// (interactions_gpu.cu:143-379 reads them from the particle arrays)
__global__ void __launch_bounds__(256) k_records_state(DevConsts c, const sphfem_particles p, int num_cell,
                                                       int *__restrict__ flags, const RecView rec,
                                                       double inv_dx, int *__restrict__ form,
                                                       int *__restrict__ next_form) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = (int)p.N;
    if (i < SPHFEM_FORM_WORDS) next_form[i] = 0;
    if (i >= N) return;
    int h = p.hash[i];
    if ((unsigned)h >= (unsigned)num_cell) {
        atomicOr(&flags[0], 4);
        h = 0;
    }
    const double tool = p.tool_particle[i];
    const double pr = tool == 0. ? p.p[i] : 0.;
    const sphfem_double4 R = tool == 0. ? p.R[i] : sphfem_double4{0., 0., 0., 0.};
    const sphfem_double2 pos = p.pos[i], vel = p.vel[i];
    const sphfem_double4 S = p.S[i];
    const double rho = p.rho[i], T = p.T[i], blanked = p.blanked[i], hh = p.h[i];
    flag_nonfinite(form, blanked, pos, vel, S, rho, T, hh, pr, R);
    write_records(c, rec, inv_dx, form, i, h, pos, vel, S, rho, T, blanked, tool, hh, pr, R);
}

void launch_records_state(sphfem_ctx *ctx, const sphfem_particles &p, int num_cell, const RecView &rec, int *form,
                          int *next_form) {
    KTimer t(ctx, "records_state");
    k_records_state<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, num_cell, ctx->d_flags, rec,
                                                             1. / ctx->c.geom.dx, form, next_form);
}

// source and key of sorted position i (from the re-sort's lists, or the sorted arrays when there are
// none) and the cell boundaries (grid_gpu_green.cu:13-51); false if the position, the key or the source
// is out of range (flagged).  Every lane of the workgroup calls it.
__device__ __forceinline__ bool cell_bounds(const sphfem_particles &p, const ResortView &rs, int i, int N, int num_cell,
                                            int *__restrict__ cell_start, int *__restrict__ cell_end,
                                            int *__restrict__ flags, int &h, int &s) {
    int hp = -1;
    if (rs.keys) {
        resort_source(rs, flags, N, i, h, s, hp);
        if (i < RS_USED) rs.sync[i] = 0;           // k_resort has read them
    } else {
        h = i < N ? p.hash[i] : 0;
        s = i < N ? p.idx[i] : 0;
        hp = __shfl_up(h, 1);
        if (__lane_id() == 0 && i > 0 && i < N) hp = p.hash[i - 1];
    }
    if (i >= N) return false;
    if ((unsigned)h >= (unsigned)num_cell || (unsigned)s >= (unsigned)N) {
        atomicOr(&flags[0], 4);
        return false;
    }
    if (i == 0 || h != hp) {
        cell_start[h] = i;
        if (i > 0 && (unsigned)hp < (unsigned)num_cell) cell_end[hp] = i;
    }
    if (i == N - 1) cell_end[h] = i + 1;
    return true;
}

// FP64 form, fused: boundaries, gather (state and old derivatives), leap_frog init
// (leap_frog.cu:25-37), predict (:45-69), EOS (actions_gpu.cu:222-232) and artificial stress
// (:234-278).  Reads the unsorted arrays p via idx, writes the sorted predicted state to b.
__global__ void __launch_bounds__(256) k_reorder_predict(DevConsts c, const sphfem_particles p, sphfem_particles b,
                                                         int *__restrict__ cell_start, int *__restrict__ cell_end,
                                                         sphfem_double2 *__restrict__ pos_init,
                                                         sphfem_double2 *__restrict__ vel_init,
                                                         sphfem_double4 *__restrict__ S_init,
                                                         double *__restrict__ rho_init, double *__restrict__ T_init,
                                                         int num_cell, int *__restrict__ flags,
                                                         const PreView pre, ResortView rs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = (int)p.N;
    int *form = flags + SPHFEM_FLAG_FORM;
    int h, s;
    if (!cell_bounds(p, rs, i, N, num_cell, cell_start, cell_end, flags, h, s)) return;
    sphfem_double2 pos = p.pos[s], vel = p.vel[s];
    sphfem_double4 S = p.S[s];
    double rho = p.rho[s], T = p.T[s];
    const double blanked = p.blanked[s], tool = p.tool_particle[s];
    if (blanked != 1.) {
        const double dt = c.dt;
        pos_init[i] = pos;
        vel_init[i] = vel;
        S_init[i] = S;
        rho_init[i] = rho;
        T_init[i] = T;
        const sphfem_double2 pt = p.pos_t[s], vt = p.vel_t[s];
        const sphfem_double4 St = p.S_t[s];
        const double rt = p.rho_t[s], Tt = p.T_t[s];
        pos.x = pos.x + 0.5 * dt * pt.x;
        pos.y = pos.y + 0.5 * dt * pt.y;
        vel.x = vel.x + 0.5 * dt * vt.x;
        vel.y = vel.y + 0.5 * dt * vt.y;
        S.x = S.x + 0.5 * dt * St.x;
        S.y = S.y + 0.5 * dt * St.y;
        S.z = S.z + 0.5 * dt * St.z;
        S.w = S.w + 0.5 * dt * St.w;
        rho = rho + 0.5 * dt * rt;
        T = T + 0.5 * dt * Tt;
    }
    b.pos[i] = pos;
    b.vel[i] = vel;
    b.S[i] = S;
    b.rho[i] = rho;
    b.T[i] = T;
    b.blanked[i] = blanked;
    b.tool_particle[i] = tool;
    b.fc[i] = p.fc[s];
    b.ft[i] = p.ft[s];
    b.h[i] = p.h[s];
    b.n[i] = p.n[s];
    b.eps_pl[i] = p.eps_pl[s];
    b.eps_pl_dot[i] = p.eps_pl_dot[s];
    b.fixed[i] = p.fixed[s];
    b.on_seg[i] = p.on_seg[s];
    // the neighbour fields of interactions_gpu.cu:247-252, 283-285 (m/rho_j in the heat term, :352)
    const bool tool_rec = tool == 1.;
    pre.pos[i] = scan_pos(blanked, pos);
    pre.vr[i] = {c.phys.mass / rho, tool_rec ? -rho : rho};
    if (tool == 0.) {
        const double pr = eos_pressure(c, rho);
        const sphfem_double4 R = artificial_stress(c, rho, pr, S);
        b.p[i] = pr;
        b.R[i] = R;
        const double rho21 = 1. / (rho * rho);
        pre.s1[i] = {(S.x - pr) * rho21, S.y * rho21};
        pre.s2[i] = {(S.z - pr) * rho21, sqrtf_d(c.phys.K / rho)};
        pre.r1[i] = {R.x, R.y};
        pre.r2[i] = {R.z, T};
        flag_nonfinite(form, blanked, pos, vel, S, rho, T, p.h[s], pr, R);
    } else {
        // neither gathered nor computed for tool particles by the reference: they stay in place
        const sphfem_double4 R = p.R[i];
        b.p[i] = p.p[i];
        b.R[i] = R;
        pre.s1[i] = {0., 0.};   // the pair loop skips these terms for tool particles
        pre.s2[i] = {0., 0.};
        pre.r1[i] = {R.x, R.y};
        pre.r2[i] = {R.z, T};
        flag_nonfinite(form, blanked, pos, vel, sphfem_double4{0., 0., 0., 0.}, rho, T, p.h[s], 0.,
                       sphfem_double4{0., 0., 0., 0.});
    }
}

// FP32C form: boundaries, predict, EOS and artificial stress of the sorted particle, written only
// as neighbour records.  The update kernel gathers the pre-step state through idx itself (and
// repeats the predictor for velocity, stress and density), so no sorted copy of the state is
// written here.
__global__ void __launch_bounds__(256) k_reorder_records(DevConsts c, const sphfem_particles p,
                                                         int *__restrict__ cell_start, int *__restrict__ cell_end,
                                                         int num_cell, int *__restrict__ flags,
                                                         const RecView rec, double inv_dx, const RateView rates,
                                                         ResortView rs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = (int)p.N;
    int *form = flags + SPHFEM_FLAG_FORM;
    int h, s;
    if (!cell_bounds(p, rs, i, N, num_cell, cell_start, cell_end, flags, h, s)) return;
    sphfem_double2 pos = ld_stream(&p.pos[s]), vel = ld_stream(&p.vel[s]);
    sphfem_double4 S = ld_stream(&p.S[s]);
    double rho = ld_stream(&p.rho[s]), T = ld_stream(&p.T[s]);
    const double blanked = ld_stream(&p.blanked[s]), tool = ld_stream(&p.tool_particle[s]);
    if (blanked != 1.) {
        const double dt = c.dt;
        // the FP32 derivative carry of the FP32C form, in the order of p
        const float2 pt = ld_stream(&rates.pos_t[s]), vt = ld_stream(&rates.vel_t[s]);
        const float4 St = ld_stream(&rates.S_t[s]);
        const double rt = ld_stream(&rates.rho_t[s]), Tt = ld_stream(&rates.T_t[s]);
        pos.x = pos.x + 0.5 * dt * pt.x;
        pos.y = pos.y + 0.5 * dt * pt.y;
        vel.x = vel.x + 0.5 * dt * vt.x;
        vel.y = vel.y + 0.5 * dt * vt.y;
        S.x = S.x + 0.5 * dt * St.x;
        S.y = S.y + 0.5 * dt * St.y;
        S.z = S.z + 0.5 * dt * St.z;
        S.w = S.w + 0.5 * dt * St.w;
        rho = rho + 0.5 * dt * rt;
        T = T + 0.5 * dt * Tt;
    }
    sphfem_double4 R = {0., 0., 0., 0.};
    double pr = 0.;
    if (tool == 0.) {
        pr = eos_pressure(c, rho);
        R = artificial_stress(c, rho, pr, S);
    }
    const double hh = ld_stream(&p.h[s]);
    flag_nonfinite(form, blanked, pos, vel, tool == 0. ? S : sphfem_double4{0., 0., 0., 0.}, rho, T, hh, pr, R);
    write_records(c, rec, inv_dx, form, i, h, pos, vel, S, rho, T, blanked, tool, hh, pr, R);
}

void launch_reorder_predict(sphfem_ctx *ctx, sphfem_grid *g, const sphfem_particles &p, sphfem_leap_frog *lf,
                            const RateView *rates, bool resorted) {
    ResortView rs{};
    if (resorted) rs = ResortView{p.hash, g->keys_alt, p.idx, g->dests, g->removed, g->changed, g->sync};
    if (lf->precision == SPHFEM_FP32C) {
        KTimer t(ctx, "reorder_records");
        k_reorder_records<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, g->cell_start, g->cell_end,
                                                                   g->num_cell, ctx->d_flags, rec_view(lf->rec, p.N),
                                                                   1. / ctx->c.geom.dx, *rates, rs);
        return;
    }
    KTimer t(ctx, "reorder_predict");
    k_reorder_predict<<<nblk(p.N, 256), 256, 0, ctx->stream>>>(ctx->c, p, g->buf, g->cell_start, g->cell_end,
                                                               lf->pos_init, lf->vel_init, lf->S_init,
                                                               lf->rho_init, lf->T_init, g->num_cell,
                                                               ctx->d_flags, pre_view(lf->pre, p.N), rs);
}

}  // namespace sphfem
