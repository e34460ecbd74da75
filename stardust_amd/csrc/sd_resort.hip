// Sorted order of a step's cell keys from the previous step's order.
//
// The keys a step sorts are key(s) = cell(s) << 32 | s, s being the sphere's
// position in the previous step's sorted order, in which cells were
// non-decreasing. A sphere whose cell did not change (a stayer) keeps the key
// old(s) = old_cell(s) << 32 | s, and old() increases with s: the stayers are
// already in order. The contact kernel lists the spheres whose cell changed
// (movers) with their new and old keys. Every key's place in the sorted order
// is then its rank among all keys:
//   stayer s:  (stayers before s) + (movers whose new key is smaller)
//              = s - (movers before s) + (movers whose new key is smaller)
//   mover x:   (stayers with a smaller key) + (movers whose new key is smaller)
//              stayers with a smaller key = (positions whose old key is smaller)
//                                           - (movers whose old key is smaller),
//              the first read off the previous step's cell starts.
// The result is the same array a stable radix sort of the keys produces, and
// the positions are permuted into that order in the same pass. With more than
// resort_cap(n) changes the step is given up: StepCtl::given_up is set, every later
// kernel of the launch sequence returns at once (the state is untouched), and
// the host redoes that step with the full radix sort.
//
// Replaces nothing in the reference (which re-sorts from scratch every step,
// src/engine/cuda/sh_collision_detection.cu:310-360); the full radix sort runs
// instead whenever more than resort_cap(n) spheres changed cell, and after every
// upload, load or restore.
#include "sd_grid_dev.hpp"
#include "sd_internal.hpp"

namespace sd {

constexpr int RESORT_MERGE_BLOCK = 512;
constexpr int RANK_MOVERS = 64;  // movers ranked by one block
constexpr int RANK_BLOCK = 256;  // four waves share the comparisons of 64 movers
constexpr int MERGE_SLICE = 1024;  // new keys of one merge block held in LDS

// Begins the step's near lists, ranks the movers' new and old keys by counting
// (keys are distinct) and places every mover, 64 movers a block. Counting is M^2 comparisons, so it is spread
// over M / 64 blocks; what remains is the latency of dependent loads that miss
// the cache after the contact kernel (count, keys, cell starts, positions). In
// a 128-scene batch of 1.83M spheres with 900 movers a step one block for all
// of them took 39 us, this form 12; a handful of movers 4.4 us in either.
__global__ __launch_bounds__(RANK_BLOCK) void k_resort_movers(
    const int* __restrict__ mcount, int cap, const uint64_t* __restrict__ mnew, const uint64_t* __restrict__ mold,
    uint64_t* __restrict__ msn, uint64_t* __restrict__ mso, int n, const int* __restrict__ cell_start,
    const float4* __restrict__ pos_state, float4* __restrict__ posB, uint64_t* __restrict__ keys_out,
    StepCtl* __restrict__ ctl, int* __restrict__ newpos, int lists, float list_cell) {
    const int given_up = ctl->given_up, M = *mcount;
    if (given_up) return;  // an earlier step of this launch sequence was given up
    if (M > cap) {  // too many changes: this step is given up (the host redoes it with the full sort)
        if (blockIdx.x == 0 && threadIdx.x == 0) ctl->given_up = GIVEN_UP_SORT;
        return;
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) list_begin_step(ctl, lists, list_cell);
    const int first = blockIdx.x * RANK_MOVERS;
    if (first >= M) return;
    __shared__ uint64_t tn[RANK_BLOCK], to[RANK_BLOCK];
    __shared__ int part[3][RANK_BLOCK];
    const int lane = lane_id(), seg = (int)threadIdx.x >> 6;
    const int i = first + lane;
    const uint64_t x = i < M ? mnew[i] : 0u;
    const uint64_t o = i < M ? mold[i] : 0u;
    // the starts of x's cell and its position, their latency behind the counting
    const uint32_t cell = (uint32_t)(x >> 32);  // < the cell count: written from a clamped cell
    const int c0 = cell_start[cell], c1 = cell_start[cell + 1];
    const float4 px = pos_state[min((uint32_t)x, (uint32_t)(n - 1))];
    int rn = 0, ro = 0, old_less = 0;
    for (int j0 = 0; j0 < M; j0 += RANK_BLOCK) {
        const int j = j0 + (int)threadIdx.x;
        tn[threadIdx.x] = j < M ? mnew[j] : ~0ull;  // (past the end: smaller than no key)
        to[threadIdx.x] = j < M ? mold[j] : ~0ull;
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < RANK_MOVERS; ++k) {
            const uint64_t a = tn[seg * RANK_MOVERS + k], b = to[seg * RANK_MOVERS + k];
            rn += a < x ? 1 : 0;
            ro += b < o ? 1 : 0;
            old_less += b < x ? 1 : 0;
        }
        __syncthreads();
    }
    part[0][threadIdx.x] = rn;
    part[1][threadIdx.x] = ro;
    part[2][threadIdx.x] = old_less;
    __syncthreads();
    if (seg != 0 || i >= M) return;
#pragma unroll
    for (int w = 1; w < RANK_BLOCK / 64; ++w) {
        rn += part[0][w * 64 + lane];
        ro += part[1][w * 64 + lane];
        old_less += part[2][w * 64 + lane];
    }
    msn[rn] = x;
    mso[ro] = o;
    // previous positions with a smaller key: those of the cells before x's
    // cell, and those of x's cell below x's position
    const int sx = (int)(uint32_t)x;
    const int all_less = c0 + (sx < c0 ? 0 : (sx > c1 ? c1 - c0 : sx - c0));
    const int dest = all_less - old_less + rn;
    if (dest >= 0 && dest < n && (uint32_t)x < (uint32_t)n) {  // (always, for consistent keys)
        keys_out[dest] = x;
        if (lists != LIST_USE) posB[dest] = px;
        else newpos[(uint32_t)x] = dest;
    }
}

__device__ __forceinline__ int lower_bound_u64(const uint64_t* a, int lo, int hi, uint64_t key) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Entries of the ascending a[0, M) below key, by a whole wave: 64 probes a
// round, so three dependent loads for up to 262,144 entries. low: the entries'
// low halves (old positions, ascending too) are compared.
template <bool low>
__device__ __forceinline__ int wave_lower_bound(const uint64_t* __restrict__ a, int M, uint64_t key) {
    int lo = 0, hi = M;
    while (hi - lo > 64) {
        const int step = (hi - lo + 63) / 64;
        const int at = lo + (lane_id() + 1) * step - 1;
        bool less = false;
        if (at < hi) less = low ? (uint32_t)a[at] < (uint32_t)key : a[at] < key;
        const int k = __popcll(__ballot(less));
        lo = lo + k * step;
        hi = min(hi, lo + step);
    }
    const int at = lo + lane_id();
    bool less = false;
    if (at < hi) less = low ? (uint32_t)a[at] < (uint32_t)key : a[at] < key;
    return lo + __popcll(__ballot(less));
}

// Every stayer: its place, key and position. Also the new order's cell starts,
// in place: start[c] counts the keys below c << 32, so it changes by the
// movers' new keys below c << 32 minus their old keys below c << 32. Each
// block updates cells_per_block consecutive cells; a run of cells that holds no
// mover key has one change for all its cells (most runs: none). Sets
// *next_count = 0 for the next step's movers, newpos (old position to new, as
// k_resort_movers does for the movers).
//
// A block's positions and cells meet few movers: each wave finds one bound of
// them in the sorted lists, and only that slice is held in LDS (all the movers'
// keys were before, which set their limit and cost 16 KB of LDS a block).
__global__ __launch_bounds__(RESORT_MERGE_BLOCK) void k_resort_merge(
    const int* __restrict__ mcount, int cap, const uint64_t* __restrict__ msn, const uint64_t* __restrict__ mso,
    const uint64_t* __restrict__ keys, int n, const float4* __restrict__ pos_state, float4* __restrict__ posB,
    uint64_t* __restrict__ keys_out, int* __restrict__ cell_start, int n_cells, int cells_per_block,
    int* __restrict__ next_count, const StepCtl* __restrict__ ctl, int* __restrict__ newpos, int lists) {
    const int given_up = ctl->given_up, M = *mcount;
    if (given_up || M > cap) return;
    // a step on lists needs no sorted positions, the others no places of the
    // previous order
    const bool use = lists == LIST_USE, sorted = !use;
    // this thread's key and position, loaded first: their latency overlaps the
    // searches below
    const int s0 = blockIdx.x * RESORT_MERGE_BLOCK;
    const int s = s0 + (int)threadIdx.x;
    uint64_t y = 0u;
    float4 ps = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (s < n) {
        y = keys[s];
        if (sorted) ps = pos_state[s];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *next_count = 0;
    int d = s;
    if (M > 0) {
        constexpr int NW = RESORT_MERGE_BLOCK / 64;
        static_assert(NW == 8, "one search per wave below");
        __shared__ uint64_t so[RESORT_MERGE_BLOCK], sn[MERGE_SLICE];
        __shared__ int bound[NW];
        __shared__ uint64_t ymin[NW], ymax[NW];
        const int w = (int)threadIdx.x >> 6;
        const int c0 = (int)min((long long)blockIdx.x * cells_per_block, (long long)n_cells);
        const int c1 = (int)min((long long)c0 + cells_per_block, (long long)n_cells);
        const uint64_t k0 = (uint64_t)(uint32_t)c0 << 32, k1 = (uint64_t)(uint32_t)c1 << 32;
        int b;
        if (w == 0) b = wave_lower_bound<true>(mso, M, (uint64_t)(uint32_t)s0);
        else if (w == 1) b = wave_lower_bound<true>(mso, M, (uint64_t)(uint32_t)(s0 + RESORT_MERGE_BLOCK));
        else if (w == 2) b = wave_lower_bound<false>(msn, M, k0);
        else if (w == 3) b = wave_lower_bound<false>(msn, M, k1);
        else if (w == 4) b = wave_lower_bound<false>(mso, M, k0);
        else if (w == 5) b = wave_lower_bound<false>(mso, M, k1);
        else b = 0;
        if (lane_id() == 0) bound[w] = b;
        __syncthreads();
        const int olo = bound[0], on = bound[1] - olo;  // at most one old key per position: on <= 512
        const int alo = bound[2], ahi = bound[3], blo = bound[4], bhi = bound[5];
        if ((int)threadIdx.x < on) so[threadIdx.x] = mso[olo + threadIdx.x];
        __syncthreads();
        // cell starts of this block's cells
        if (alo != blo || ahi != alo || bhi != blo) {
            for (int c = c0 + (int)threadIdx.x; c < c1; c += RESORT_MERGE_BLOCK) {
                int dd = alo - blo;
                if (ahi != alo || bhi != blo) {
                    const uint64_t k = (uint64_t)(uint32_t)c << 32;
                    dd = lower_bound_u64(msn, alo, ahi, k) - lower_bound_u64(mso, blo, bhi, k);
                }
                if (dd != 0) cell_start[c] += dd;
            }
        }
        // movers before s: old keys ascend with their positions (the low halves)
        int lo = 0, hi = on;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if ((uint32_t)so[mid] < (uint32_t)s) lo = mid + 1;
            else hi = mid;
        }
        const bool stays = s < n && !(lo < on && (uint32_t)so[lo] == (uint32_t)s);  // (movers are placed already)
        // the stayers' keys ascend: their range, and the new keys inside it
        const uint64_t m = __ballot(stays);
        const int fl = m ? __builtin_ctzll(m) : 0, ll = m ? 63 - __builtin_clzll(m) : 0;
        if (m && lane_id() == fl) ymin[w] = y;
        if (m && lane_id() == ll) ymax[w] = y;
        if (!m && lane_id() == 0) {
            ymin[w] = ~0ull;
            ymax[w] = 0u;
        }
        __syncthreads();
        uint64_t y0 = ~0ull, y1 = 0u;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            y0 = ymin[q] < y0 ? ymin[q] : y0;
            y1 = ymax[q] > y1 ? ymax[q] : y1;
        }
        if (w == 0) b = wave_lower_bound<false>(msn, M, y0);
        else if (w == 1) b = wave_lower_bound<false>(msn, M, y1);
        if (w < 2 && lane_id() == 0) bound[6 + w] = b;
        __syncthreads();
        const int nlo = bound[6], nn = max(bound[7] - nlo, 0);  // new keys in [y0, y1)
        const bool held = nn <= MERGE_SLICE;
        if (held)
            for (int j = threadIdx.x; j < nn; j += RESORT_MERGE_BLOCK) sn[j] = msn[nlo + j];
        __syncthreads();
        if (!stays) return;
        const int a = held ? nlo + lower_bound_u64(sn, 0, nn, y) : lower_bound_u64(msn, nlo, nlo + nn, y);
        d = s - (olo + lo) + a;
    }
    if (s >= n || d < 0 || d >= n) return;  // (d is inside for consistent keys)
    keys_out[d] = y;
    if (sorted) posB[d] = ps;
    if (use) newpos[s] = d;
}

// Cells whose starts one of nblocks merge blocks updates: whole rounds of its
// threads, or all cells (a round more than 2^31 - 1 of them is no int).
constexpr int merge_cells(int n_cells, int nblocks) {
    const long long per = ((long long)n_cells + nblocks - 1) / nblocks;
    const long long rounds = (per + RESORT_MERGE_BLOCK - 1) / RESORT_MERGE_BLOCK * RESORT_MERGE_BLOCK;
    return (int)(rounds < n_cells ? rounds : n_cells);
}
static_assert(merge_cells(0x7fffffff, 1) == 0x7fffffff && merge_cells(0x7ffffe01, 1) == 0x7ffffe01, "no overflow");
static_assert(merge_cells(1025, 2) == 1024 && merge_cells(1024, 2) == 512 && merge_cells(3, 1) == 3, "whole rounds");

sd_status launch_resort_u64(const int* mcount, int cap, const uint64_t* mnew, const uint64_t* mold,
                            uint64_t* msorted_new, uint64_t* msorted_old, const uint64_t* keys, int n,
                            int* cell_start, int n_cells, const float4* pos_state, float4* posB, uint64_t* keys_out,
                            int* next_count, StepCtl* ctl, int* newpos, int lists, float list_cell,
                            hipStream_t s) {
    if (n <= 0) return SD_OK;
    hipLaunchKernelGGL(k_resort_movers, dim3(div_up(cap, RANK_MOVERS)), dim3(RANK_BLOCK), 0, s, mcount, cap, mnew,
                       mold, msorted_new, msorted_old, n, (const int*)cell_start, pos_state, posB, keys_out, ctl,
                       newpos, lists, list_cell);
    SD_LAUNCH_CHECK();
    const int nblocks = div_up(n, RESORT_MERGE_BLOCK);
    const int cells_per_block = merge_cells(n_cells, nblocks);
    hipLaunchKernelGGL(k_resort_merge, dim3(nblocks), dim3(RESORT_MERGE_BLOCK), 0, s, mcount, cap,
                       (const uint64_t*)msorted_new, (const uint64_t*)msorted_old, keys, n, pos_state, posB, keys_out,
                       cell_start, n_cells, cells_per_block, next_count, (const StepCtl*)ctl, newpos, lists);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

}  // namespace sd
