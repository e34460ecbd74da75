// Deterministic per-sphere contact gather and semi-implicit integration.
//
// Replaces computeParticleToParticleCUDA / reactCollisionsCUDA
// (src/engine/cuda/collisions/SAP/sap_reaction.cu:20-160) and, for single-sphere
// bodies, advectParticlesCUDA (src/engine/cuda/physics_update.cu:232-310).
// The reference scatters pair forces into both spheres without atomics; here
// each sphere gathers the forces of all its contacts in a fixed traversal order
// (stencil rows (dz, dy) ascending, sorted positions ascending within a row,
// then walls 0..5), so results do not depend on the launch configuration.
//
// Contact law (per contact, FP32, no fused multiply-add so that the pair force
// seen by each side is the exact negation of the other):
//   n      = (x_i - x_j) / |x_i - x_j|,  delta = r_i + r_j - |x_i - x_j| > 0
//   l_i    = r_i - delta/2 (lever arm to the mid-overlap contact point; the same
//            point for both spheres, so pair torques conserve angular momentum)
//   m_eff  = 1 / (1/m_i + 1/m_j),  c_n = 2 zeta sqrt(k_n m_eff),  c_t = 2 zeta sqrt(k_t m_eff)
//   v_c    = (v_i - v_j) - (l_i w_i + l_j w_j) x n,  v_n = v_c . n,  v_t = v_c - v_n n
//   f_n    = k_n delta - c_n v_n
//   xi_t   = (xi_t - (xi_t . n) n) + v_t dt                (tangential spring history)
//   F_t    = -k_t xi_t - c_t v_t, limited to mu |f_n|; on slip xi_t = -(F_t + c_t v_t) / k_t
//   F_i    = f_n n + F_t,  T_i = -l_i (n x F_t)
// Walls are partners with r = 0, 1/m = 0, v = w = 0 and ids -1..-6.
#include "sd_contact_law.hpp"
#include "sd_grid_dev.hpp"
#include <algorithm>

#include "sd_internal.hpp"

namespace sd {

ContactDev to_dev(const sd_contact_params& c) {
    ContactDev d;
    d.kn = c.kn;
    d.kt = c.kt_ratio * c.kn;
    d.c2z = 2.0f * c.damping_ratio;
    d.mu = c.mu;
    d.dt = c.dt;
    d.gx = c.gravity[0];
    d.gy = c.gravity[1];
    d.gz = c.gravity[2];
    d.walls = c.walls;
    for (int a = 0; a < 3; ++a) {
        d.wlo[a] = c.wall_lo[a];
        d.whi[a] = c.wall_hi[a];
    }
    d.maxc = c.max_contacts;
    return d;
}

sd_status check_contact(const sd_contact_params* c) {
    SD_REQUIRE(c != nullptr, "contact params are NULL");
    SD_REQUIRE(c->kn > 0.0f && c->kt_ratio > 0.0f, "contact: kn and kt_ratio must be positive");
    SD_REQUIRE(c->damping_ratio >= 0.0f && c->mu >= 0.0f, "contact: damping_ratio and mu must be >= 0");
    SD_REQUIRE(c->dt > 0.0f, "contact: dt must be positive");
    SD_REQUIRE(c->max_contacts > 0 && c->max_contacts <= 256, "contact: max_contacts must be in [1, 256]");
    return SD_OK;
}

__device__ __forceinline__ void integrate_sphere(const ContactDev& c, float4& p, float4& v, float4& w, float fx,
                                                 float fy, float fz, float tx, float ty, float tz) {
    if (v.w > 0.0f) {
        v.x = v.x + (fx * v.w + c.gx) * c.dt;
        v.y = v.y + (fy * v.w + c.gy) * c.dt;
        v.z = v.z + (fz * v.w + c.gz) * c.dt;
        p.x = p.x + v.x * c.dt;
        p.y = p.y + v.y * c.dt;
        p.z = p.z + v.z * c.dt;
        w.x = w.x + (tx * w.w) * c.dt;
        w.y = w.y + (ty * w.w) * c.dt;
        w.z = w.z + (tz * w.w) * c.dt;
    }
}

__device__ __forceinline__ int old_slot_of(const ContactArgs& a, int s) {
    if (a.old_slot_i32) return a.old_slot_i32[s];
    return (int)(uint32_t)a.old_slot_u64[s];
}

// Looks up the tangential history stored for partner pid in the old list
// (partner ids in a list are distinct, so the entry found does not depend on
// the search order). The search starts at entry `start`, the position the
// contact has in the new list: contacts are found in the same order step after
// step, so a lasting contact is usually at the same position and the first
// probe finds it.
__device__ __forceinline__ void find_history(const ContactArgs& a, int os, int oc, int pid, int start, float& hx,
                                             float& hy, float& hz) {
    hx = 0.0f;
    hy = 0.0f;
    hz = 0.0f;
    int k = start < oc ? start : 0;
    for (int j = 0; j < oc; ++j) {
        const float4 h = a.hist_old[(size_t)k * a.n + os];
        if (__float_as_int(h.w) == pid) {
            hx = h.x;
            hy = h.y;
            hz = h.z;
            break;
        }
        k = k + 1 < oc ? k + 1 : 0;
    }
}

constexpr int CAND_UNROLL = 4; // candidate positions loaded per batch (loads in flight)
static_assert(CAND_UNROLL - 1 <= CONTACT_POS_PAD, "sorted positions must be padded for a whole batch");
constexpr int CONTACT_ITEMS = 128;  // contacts of a wave handed out at a time (their places in the same LDS)
constexpr int CONTACT_PASS = 12;    // contacts of one sphere spread over the wave
// float4s of LDS per wave: the stage of a search (candidate positions), or only
// what shares it, and the contacts found by each lane. A search of dilute scenes
// needs every wave that its registers allow: with 224 positions staged the LDS
// held fewer. Forces of 1,000,003 dilute spheres 72 us with 224, 69 with 192, 68
// with 160 (in contact 120, 117, 116); a step of 4,194,304 that searches 303, 291,
// 291, but of 250,007, whose runs of candidates are longer, 33, 33, 36.
constexpr int CONTACT_SHARED = CONTACT_ITEMS / 2 + 6 * WAVE / 4;
constexpr int contact_stage(int mode, int lists) {
    return lists == LIST_USE ? CONTACT_SHARED : (mode == CONTACT_FORCES ? 160 : 192);
}
constexpr int contact_lds(int mode, int lists) { return contact_stage(mode, lists) + CONTACT_PASS * WAVE / 4; }
static_assert(LIST_CAP % CAND_UNROLL == 0, "whole batches of a list are read");
static_assert(CONTACT_SHARED <= contact_stage(CONTACT_FORCES, LIST_NONE), "items and results fit the stage");

// Orders one wave's LDS writes and reads (the lanes of a wave only).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Largest of the wave's squared displacements into one of the step's maxima
// (non-negative floats and not-a-numbers order as their bits do). The active
// lanes are a prefix of the wave: DPP steps leave lane i the largest of lanes
// 0 .. i.
__device__ __forceinline__ void note_displacement(StepCtl* L, float d2) {
    uint32_t u = __float_as_uint(d2);
#define SD_STEP(ctrl, rows)                                                                                     \
    {                                                                                                           \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)u, (int)u, ctrl, rows, 0xf, false);       \
        u = o > u ? o : u;                                                                                      \
    }
    SD_STEP(0x111, 0xf) SD_STEP(0x112, 0xf) SD_STEP(0x114, 0xf) SD_STEP(0x118, 0xf)  // row_shr 1, 2, 4, 8
    SD_STEP(0x142, 0xa) SD_STEP(0x143, 0xc)                                          // row_bcast 15, 31
#undef SD_STEP
    const uint64_t m = __ballot(1);
    if (lane_id() == 63 - __builtin_clzll(m)) atomicMax(&L->dmax[((blockIdx.x * 4u + (threadIdx.x >> 6)) & 63u) * 16u], u);
}

// MODE: CONTACT_FORCES writes force/torque; CONTACT_FUSED_* integrates and writes
// the next state and keys. INDIRECT: vel/omg/ids are in the previous step's order
// and are read through old_slot (positions are always in sorted order).
// CONTACT_FUSED_BATCH: the grid, contact law and cell starts come from the
// sphere's scene; the arithmetic is the same code, so a scene stepped in a
// batch is bit-identical to the same scene stepped alone.
// a wave-uniform struct in global memory, word by word into scalar registers
// (the compiler does not use scalar loads for memory the kernel also writes)
template <typename T>
__device__ __forceinline__ T uniform_copy(const T& src) {
    static_assert(sizeof(T) % 4 == 0, "uniform_copy: whole 32-bit words");
    T dst;
    const int* const w = reinterpret_cast<const int*>(&src);
    int* const d = reinterpret_cast<int*>(&dst);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) d[i] = __builtin_amdgcn_readfirstlane(w[i]);
    return dst;
}

// STRADDLE (batch mode only): one 64-thread block per listed wave whose slots
// span more than one scene; every lane then takes its own scene's parameters.
// The work of the 64 consecutive slots of one wave, slot the lane's: everything
// the kernel does once the slot is known.
//
// In three parts. (1) Every lane finds its sphere's contacts, in ascending
// sorted position: among its near list (LISTED), or by a search of the cells
// around it (which also makes the list). (2) The wave's contacts, as one
// sequence, are spread over its lanes, one contact a lane, so that a wave's
// time goes with its number of contacts and not with the largest number of one
// sphere, and the loads of 64 contacts are in flight together. (3) Every lane
// adds up its sphere's forces in order.
//
// A step on lists moves 157 bytes a sphere at rest (state in and out, keys,
// history count, a list row or two; 661 MB by the counters) and is bound by that
// in a dilute scene, at 4.6 TB/s: 4,194,304 spheres 143 us, 181 at 0.5 m/s, where the search of every step took 312 (VALU
// issue, 97 candidate tests a sphere). With 2 to 3 contacts a sphere the chain
// of loads of a contact counts: 1,048,576 spheres 154 us (215 when each lane
// went through its own contacts), 1,000 spheres 18 us (51). A step that makes
// lists takes 416, 222 and 43 us, every 40th step or so.
//
// A kernel for each use of the lists (LISTS): with the search as a branch of one,
// the steps on lists ran at 4 waves a SIMD or with spills (4,194,304 spheres 265
// and 395 us); with the making of lists as a branch of the search, a step that
// only searches lost a wave a SIMD (4,194,304 spheres 318 us, 303 without).
template <int MODE, bool INDIRECT, bool STRADDLE, int LISTS>
__device__ __forceinline__ void contact_wave(const ContactArgs& a, int slot) {
    constexpr bool LISTED = LISTS == LIST_USE, BUILD = LISTS == LIST_BUILD;
    constexpr int STAGE = contact_stage(MODE, LISTS), STAGE_MOST = 3 * STAGE;
    constexpr bool BATCH = MODE == CONTACT_FUSED_BATCH;
    constexpr bool FUSED = MODE != CONTACT_FORCES;
    constexpr bool PADDED = FUSED;  // fused modes read a context's padded buffer
    const int lane = lane_id();
    const bool live = slot < a.n;  // lanes past the end take part in the wave's shared work
    const int first = __builtin_amdgcn_readfirstlane(slot - lane);  // the wave's first slot
    if (first >= a.n) return;
    const int s = min(first + lane, a.n - 1);
    GridDev g;
    ContactDev c;
    const int* ranges;  // CONTACT_FORCES: (start, end) per cell; fused modes: cell starts
    uint32_t cbase = 0u;
    float rmax = 0.0f;
    if constexpr (STRADDLE) {
        const int sid = a.scene_of[s];
        const SceneDev& S = a.scenes[sid];
        g = S.g;
        c = S.c;
        cbase = S.cbase;
        ranges = a.cell_start + cbase;
        rmax = a.scene_rmax[sid];
    } else if constexpr (BATCH) {
        // one scene in the wave (the waves spanning two are in a.straddle and
        // run by the straddle launch): its parameters are wave-uniform
        const int my_scene = a.scene_of[s];
        const int sid = __builtin_amdgcn_readfirstlane(my_scene);
        if (__ballot(my_scene != sid) != 0u) return;
        const SceneDev S = uniform_copy(a.scenes[sid]);
        g = S.g;
        c = S.c;
        cbase = S.cbase;
        ranges = a.cell_start + cbase;
        rmax = a.scene_rmax[sid];
    } else {
        g = a.g;
        c = a.c;
        ranges = MODE == CONTACT_FORCES ? a.ranges : a.cell_start;
        rmax = a.rmax;
    }
    const int os = old_slot_of(a, s);
    const int self = INDIRECT ? os : s;  // the sphere's row: of the previous order, or the sorted one
    const float4* const rowpos = INDIRECT ? a.pos_rows : a.pos;
    // the velocity and spin are read where they are needed, after the
    // contacts: held from here they cost a wave a SIMD
    float4 p = rowpos[self];
    const float inv_m = a.vel[self].w;
    float inv_i = 0.0f;
    if constexpr (FUSED) inv_i = a.omg[self].w;  // (brings the row into the cache)
    const int myid = FUSED ? a.ids[self] : 0;
    int oc = a.hcount_old[os];
    oc = oc < c.maxc ? oc : c.maxc;
    int lcount = 0;      // LISTED: the sphere's list
    float sigma = 0.0f;  // a search that makes lists: their margin
    if constexpr (LISTED) lcount = live ? a.lcount_old[os] : 0;
    else if constexpr (BUILD) sigma = a.ctl->sigma;

    int cx, cy, cz;
    cell_coords(g, p.x, p.y, p.z, cx, cy, cz);
    const uint32_t cell_old = cbase + (uint32_t)((cz * g.ny + cy) * g.nx + cx);
    float fx = 0.0f, fy = 0.0f, fz = 0.0f, tx = 0.0f, ty = 0.0f, tz = 0.0f;
    int nc = 0;

    // LDS of the wave: staged candidates of a search, later the contacts of the
    // wave (row, owning lane and number) and 64 results; the rows of each
    // lane's contacts (entry k of a lane at k * 64 + lane)
    extern __shared__ float4 cstage[];
    float4* const stg = cstage + (threadIdx.x >> 6) * contact_lds(MODE, LISTS);
    int2* const items = reinterpret_cast<int2*>(stg);
    float* const res = reinterpret_cast<float*>(stg + CONTACT_ITEMS / 2);
    int* const pend = reinterpret_cast<int*>(stg + STAGE) + lane;

    // Whether the sphere at row `row`, closer than the radii, (dx, dy, dz) away
    // and not coincident (the sphere itself, too), is a contact: not both
    // static, and in the 27 cells around the sphere. Rounding of the cell of a
    // sphere at a boundary can put a pair as far apart along an axis as the
    // cell is wide two cells apart, which is no contact (nearer pairs cannot
    // be, by far, on grids of up to 65,536 cells a side): a search of the 27
    // cells does not meet it.
    const float near = LISTS != LIST_NONE
                           ? (max(g.nx, max(g.ny, g.nz)) > 65536 ? 0.0f : 0.9f * g.cell)
                           : 3.4e38f;
    auto is_contact = [&](int row, float dx, float dyy, float dzz) -> bool {
        if (fmaxf(fabsf(dx), fmaxf(fabsf(dyy), fabsf(dzz))) > near) {
            const float4 q = rowpos[row];
            int qx, qy, qz;
            cell_coords(g, q.x, q.y, q.z, qx, qy, qz);
            if (abs(qx - cx) > 1 || abs(qy - cy) > 1 || abs(qz - cz) > 1) return false;
        }
        return inv_m > 0.0f || a.vel[row].w > 0.0f;
    };

    int hc = 0;     // contacts found; the first CONTACT_PASS of them are in pend
    int pc = 0;     // contacts in pend
    int after = -1; // LISTED: the place of the last one in pend
    int ln = 0;     // listed neighbours
    if (LISTED) {
        // The listed spheres, in any order; their contacts in ascending
        // new position: the order of the search, so of the sums and of the
        // history. A list made by a search is ascending; only a sphere that
        // changed cell moves in one. Positions come from the previous
        // order's rows, so that the place of a sphere in the new order is
        // off the chain of loads.
        int k0 = 0;
        do {  // (the first batch does not wait for the list's length)
            int t[CAND_UNROLL], tn[CAND_UNROLL];
            float4 q[CAND_UNROLL];
#pragma unroll
            for (int k = 0; k < CAND_UNROLL; ++k) t[k] = a.list_old[(size_t)(k0 + k) * a.n + os];
#pragma unroll
            for (int k = 0; k < CAND_UNROLL; ++k) {
                if (k0 + k >= lcount) t[k] = self;  // (past the list: whatever the row held)
                q[k] = rowpos[t[k]];
                tn[k] = a.newpos[t[k]];
            }
#pragma unroll
            for (int k = 0; k < CAND_UNROLL; ++k) {
                if (k0 + k >= lcount) break;
                const int row = t[k], place = tn[k];
                a.list_new[(size_t)(k0 + k) * a.n + s] = place;
                const float dx = p.x - q[k].x;
                const float dyy = p.y - q[k].y;
                const float dzz = p.z - q[k].z;
                const float d2 = dx * dx + dyy * dyy + dzz * dzz;
                const float rs = p.w + q[k].w;
                if (!(d2 < rs * rs) || d2 == 0.0f ||
                    !is_contact(row, dx, dyy, dzz))
                    continue;
                ++hc;
                const bool full = pc == CONTACT_PASS;
                if (full) {
                    if (place > after) continue;
                    --pc;  // (the furthest one is left out)
                }
                int m = pc++;
                if (place > after) {
                    after = place;
                } else {
                    for (; m > 0; --m) {
                        const int b = pend[(m - 1) * WAVE];
                        if (a.newpos[b] < place) break;
                        pend[m * WAVE] = b;
                    }
                }
                pend[m * WAVE] = row;
                if (full) after = a.newpos[pend[(pc - 1) * WAVE]];
            }
            k0 += CAND_UNROLL;
        } while (k0 < lcount);
    }
    if (!LISTED && live) {
        // Distance test of the candidates at sorted positions t0 .. t0+3
        // (q). Only the distance is tested per candidate; a batch with a
        // possible contact in any lane (rare, and always the batch holding
        // the sphere itself) then drops positions past hi and the sphere
        // itself (position s, without a memory access). While lists are
        // built, the distance is the contact's plus the margin, and every
        // sphere within it is listed.
        const float reach = p.w + sigma;
        // sl: where the candidates are held (position t at sl[t]).
        auto test_batch = [&](const float4 (&q)[CAND_UNROLL], int t0, int hi, const float4* sl) {
            bool h[CAND_UNROLL];
            uint64_t any = 0u;  // lanes with a possible contact (scalar masks)
#pragma unroll
            for (int k = 0; k < CAND_UNROLL; ++k) {
                const float dx = p.x - q[k].x;
                const float dyy = p.y - q[k].y;
                const float dzz = p.z - q[k].z;
                const float d2 = dx * dx + dyy * dyy + dzz * dzz;
                const float rs = reach + q[k].w;
                h[k] = d2 < rs * rs;
                any |= __builtin_amdgcn_ballot_w64(h[k]);
            }
            if (any) {
                uint32_t hit = 0u;
#pragma unroll
                for (int k = 0; k < CAND_UNROLL; ++k) hit |= h[k] ? (1u << k) : 0u;
                while (hit) {
                    const int t = t0 + __builtin_ctz(hit);
                    hit &= hit - 1u;
                    if (t >= hi || t == s) continue;
                    if constexpr (BUILD) {
                        if (ln < LIST_CAP) a.list_new[(size_t)ln * a.n + s] = t;
                        ++ln;
                    }
                    const float4 qt = sl[t];
                    const float dx = p.x - qt.x;
                    const float dyy = p.y - qt.y;
                    const float dzz = p.z - qt.z;
                    const float d2 = dx * dx + dyy * dyy + dzz * dzz;
                    const float rs = p.w + qt.w;
                    if (!(d2 < rs * rs) || d2 == 0.0f) continue;
                    const int row = INDIRECT ? old_slot_of(a, t) : t;
                    if (!is_contact(row, dx, dyy, dzz)) continue;
                    // (the rows past those kept wait where their history will be)
                    if (hc < CONTACT_PASS) pend[hc * WAVE] = row;
                    else if (hc < c.maxc) a.hist_new[(size_t)hc * a.n + s].x = __int_as_float(row);
                    ++hc;
                }
            }
        };

        // Candidate staging. The lanes of a wave are consecutive sorted
        // spheres, so for one stencil row offset (dz, dy) their windows
        // ascend with the lane (rows and cells are in sorted order). The
        // lanes in the first active lane's grid row (segment A) and the
        // others (segment B, normally the next row) each have a compact
        // union of windows. The two unions, each followed by the 3
        // positions a batch may read past a window, form one staged
        // sequence: sorted position t of a lane is entry t + off of it.
        // The wave copies the sequence into its LDS region with coalesced
        // loads (in chunks of STAGE entries; one chunk unless the
        // wave spans several sparse rows) and every lane tests its
        // candidates in the chunk from LDS.
        const uint64_t amask = __ballot(1);  // the searching lanes
        const int arank = __popcll(amask & lanemask_lt());
        const int nact = __popcll(amask);
        const uint32_t rowid = cell_old - (uint32_t)cx;
        const bool segB = rowid != (uint32_t)__builtin_amdgcn_readfirstlane((int)rowid);
        const uint64_t bmask = __ballot(segB);
        constexpr int PAD = CAND_UNROLL - 1;        // a batch reads up to 3 positions past its window
        constexpr int CHUNK = STAGE - PAD;  // sequence entries tested per chunk
        const char* const pos_bytes = reinterpret_cast<const char*>(a.pos);

        // Rows of the search, in ascending order: the 27 cells around the
        // sphere, or, while lists are built, the rows that a sphere within
        // reach of it can lie in (the cell of a coordinate grows with it,
        // so the cells of both ends of the reach bound them): fewer than
        // nine for most spheres, one further out for a sphere near a cell
        // boundary. e: cells on either side in x, the same for the wave
        // (windows ascend with the lane).
        int y0 = max(cy - 1, 0), y1 = min(cy + 1, g.ny - 1), z0 = max(cz - 1, 0), z1 = min(cz + 1, g.nz - 1);
        int e = 1;
        if constexpr (BUILD) {
            const float R = (reach + rmax) * 1.0001f;
            y0 = axis_cell(p.y - R, g.loy, g.cell, g.ny);
            y1 = axis_cell(p.y + R, g.loy, g.cell, g.ny);
            z0 = axis_cell(p.z - R, g.loz, g.cell, g.nz);
            z1 = axis_cell(p.z + R, g.loz, g.cell, g.nz);
            const int x0 = axis_cell(p.x - R, g.lox, g.cell, g.nx);
            const int x1 = axis_cell(p.x + R, g.lox, g.cell, g.nx);
            e = __ballot(cx - x0 > 1 || x1 - cx > 1) ? 2 : 1;
        }
        // row offsets (dz, dy) that some lane of the wave has
        const int dz0 = __ballot(z0 < cz - 1) ? -2 : (__ballot(z0 < cz) ? -1 : 0);
        const int dz1 = __ballot(z1 > cz + 1) ? 2 : (__ballot(z1 > cz) ? 1 : 0);
        const int dy0 = __ballot(y0 < cy - 1) ? -2 : (__ballot(y0 < cy) ? -1 : 0);
        const int dy1 = __ballot(y1 > cy + 1) ? 2 : (__ballot(y1 > cy) ? 1 : 0);
        // window of a row; the next row's window is loaded while a row is
        // copied and tested
        auto window = [&](int dz, int dy, int& lo, int& hi) {
            const int z = cz + dz, y = cy + dy;
            lo = 0;
            hi = 0;
            if (z >= z0 && z <= z1 && y >= y0 && y <= y1) {
                if constexpr (MODE == CONTACT_FORCES) row_range(g, ranges, cx, y, z, lo, hi);
                else row_window(g, ranges, cx, e, y, z, lo, hi);
            }
        };
        int next_lo, next_hi, dz = dz0, dy = dy0;
        window(dz, dy, next_lo, next_hi);
#pragma unroll 1
        while (dz <= dz1) {
            const int lo = next_lo, hi = next_hi;
            if (++dy > dy1) {
                dy = dy0;
                ++dz;
            }
            if (dz <= dz1) window(dz, dy, next_lo, next_hi);
            const uint64_t ne = __ballot(hi > lo);
            if (ne == 0u) continue;
            const uint64_t ma = ne & ~bmask, mb = ne & bmask;
            int la = 0, na = 0, lb = 0, nb = 0;
            if (ma) {
                la = __builtin_amdgcn_readlane(lo, __builtin_ctzll(ma));
                na = __builtin_amdgcn_readlane(hi, 63 - __builtin_clzll(ma)) - la;
            }
            if (mb) {
                lb = __builtin_amdgcn_readlane(lo, __builtin_ctzll(mb));
                nb = __builtin_amdgcn_readlane(hi, 63 - __builtin_clzll(mb)) - lb;
            }
            const int offb = na + PAD;                 // sequence entry of position lb
            const int seq = offb + nb + PAD;           // sequence length
            const int off = segB ? offb - lb : -la;    // sequence entry of sorted position t: t + off
            const int lb_b = lb - offb;                // source of entry e >= offb: lb_b + e
            // A wave of a sparse region beside a dense one (its lanes in many
            // rows of a half-filled layer, the layer below it full): the union of
            // its windows is thousands of positions, of which each lane needs a
            // few, and read chunk by chunk one such wave is all a step waits for
            // (250,007 spheres in contact 227 us, now 51). From three chunks on
            // each lane reads its own window.
            if (seq > STAGE_MOST) {
                for (int t0 = lo; t0 < hi; t0 += CAND_UNROLL) {
                    float4 q[CAND_UNROLL];
#pragma unroll
                    for (int k = 0; k < CAND_UNROLL; ++k) q[k] = a.pos[min(t0 + k, hi - 1)];
                    test_batch(q, t0, hi, a.pos);
                }
                continue;
            }
            for (int e0 = 0; e0 < seq - PAD; e0 += CHUNK) {
                const int m = min(STAGE, seq - e0);
                for (int i = arank; i < m; i += 2 * nact) {
                    const int e1 = e0 + i, e2 = e1 + nact;
                    // sources reach at most n + 2 (3 padding entries past a
                    // window that ends at n): inside a context's padded buffer,
                    // clamped for a caller's unpadded one
                    const int s1 = PADDED ? (e1 < offb ? la : lb_b) + e1 : min((e1 < offb ? la : lb_b) + e1, a.n - 1);
                    const int s2 = PADDED ? (e2 < offb ? la : lb_b) + e2 : min((e2 < offb ? la : lb_b) + e2, a.n - 1);
                    const float4 v1 = *reinterpret_cast<const float4*>(pos_bytes + (size_t)((uint32_t)s1 * 16u));
                    if (i + nact < m) {
                        const float4 v2 = *reinterpret_cast<const float4*>(pos_bytes + (size_t)((uint32_t)s2 * 16u));
                        stg[i + nact] = v2;
                    }
                    stg[i] = v1;
                }
                wave_lds_sync();
                // this lane's positions in the chunk; a batch may read 3 entries
                // past them (still inside the chunk's copy)
                const int tlo = max(lo, e0 - off), thi = min(hi, e0 + CHUNK - off);
                const float4* const sl = stg + (off - e0);
                for (int t0 = tlo; t0 < thi; t0 += CAND_UNROLL) {
                    float4 q[CAND_UNROLL];
#pragma unroll
                    for (int k = 0; k < CAND_UNROLL; ++k) q[k] = sl[t0 + k];
                    test_batch(q, t0, thi, sl);
                }
                wave_lds_sync();  // every lane's reads precede the next copy
            }
        }
    }

    if constexpr (FUSED) asm volatile("" ::"v"(inv_i));  // (the row is in the cache by now; not held further)

    // the wave's contacts: lane l's are [off, off + pc)
    if (!LISTED) pc = min(hc, CONTACT_PASS);
    const int inc = (int)wave_inclusive_scan((uint32_t)pc);
    const int off = inc - pc;
    const int total = __builtin_amdgcn_readlane(inc, 63);
    for (int c0 = 0; c0 < total; c0 += CONTACT_ITEMS) {
        for (int j = max(c0 - off, 0); j < pc && off + j < c0 + CONTACT_ITEMS; ++j)
            items[off + j - c0] = make_int2(pend[j * WAVE], lane | (j << 8));
        wave_lds_sync();
        const int ce = min(total - c0, CONTACT_ITEMS);
        for (int i0 = 0; i0 < ce; i0 += WAVE) {
            const bool on = i0 + lane < ce;
            const int2 it = items[on ? i0 + lane : 0];
            const int row = it.x, ow = it.y & 63;
            // the owner's row, old slot, history entries and entry of this contact
            const int oself = __shfl(self, ow);
            const int oos = INDIRECT ? oself : __shfl(os, ow);
            const int ooc = __shfl(oc, ow);
            const int k = __shfl(nc, ow) + (it.y >> 8);
            ContactDev lc = c;
            if constexpr (STRADDLE) {
                lc.kn = __shfl(c.kn, ow);
                lc.kt = __shfl(c.kt, ow);
                lc.c2z = __shfl(c.c2z, ow);
                lc.mu = __shfl(c.mu, ow);
            }
            if (on) {
                const float4 pi = rowpos[oself], pj = rowpos[row];
                const float4 vi = a.vel[oself], vj = a.vel[row];
                const float4 wi = a.omg[oself], wj = a.omg[row];
                const int pid = a.ids[row];
                const float dx = pi.x - pj.x;
                const float dyy = pi.y - pj.y;
                const float dzz = pi.z - pj.z;
                const float d2 = dx * dx + dyy * dyy + dzz * dzz;
                const float d = sqrtf(d2);
                const float inv_d = 1.0f / d;
                const float nx = dx * inv_d, ny = dyy * inv_d, nz = dzz * inv_d;
                float hx, hy, hz;
                find_history(a, oos, ooc, pid, k, hx, hy, hz);
                const PairForce f =
                    contact_law(lc, nx, ny, nz, (pi.w + pj.w) - d, pi.w, pj.w, vi.w, vj.w, vi.x - vj.x,
                                vi.y - vj.y, vi.z - vj.z, wi.x, wi.y, wi.z, wj.x, wj.y, wj.z, hx, hy, hz);
                res[lane] = f.fx;
                res[64 + lane] = f.fy;
                res[128 + lane] = f.fz;
                res[192 + lane] = f.tx;
                res[256 + lane] = f.ty;
                res[320 + lane] = f.tz;
                if (k < lc.maxc)
                    a.hist_new[(size_t)k * a.n + (first + ow)] = make_float4(hx, hy, hz, __int_as_float(pid));
            }
            wave_lds_sync();
            // this lane's results, in order
            const int f0 = c0 + i0;
            for (int j = max(f0 - off, 0); j < pc && off + j < f0 + WAVE; ++j) {
                const float* const r = res + (off + j - f0);
                fx = fx + r[0];
                fy = fy + r[64];
                fz = fz + r[128];
                tx = tx + r[192];
                ty = ty + r[256];
                tz = tz + r[320];
            }
            wave_lds_sync();
        }
    }
    nc += pc;

    // A sphere with more contacts than that (one large sphere among many small
    // ones): the others one after the other. A second pass of the code above
    // instead, in a loop around it, took 25 registers more. A search has left
    // their rows where their history will be written: searching again made a
    // step with 45 of them 135 us, now 88.
    if (__ballot(hc > CONTACT_PASS) != 0u && hc > CONTACT_PASS) {
        auto add = [&](int row) {
            const float4 q = rowpos[row], vi = a.vel[self], vj = a.vel[row], wi = a.omg[self], wj = a.omg[row];
            const int pid = a.ids[row];
            const float dx = p.x - q.x;
            const float dyy = p.y - q.y;
            const float dzz = p.z - q.z;
            const float d = sqrtf(dx * dx + dyy * dyy + dzz * dzz);
            const float inv_d = 1.0f / d;
            float hx, hy, hz;
            find_history(a, os, oc, pid, nc, hx, hy, hz);
            const PairForce f = contact_law(c, dx * inv_d, dyy * inv_d, dzz * inv_d, (p.w + q.w) - d, p.w, q.w, vi.w,
                                            vj.w, vi.x - vj.x, vi.y - vj.y, vi.z - vj.z, wi.x, wi.y, wi.z, wj.x, wj.y,
                                            wj.z, hx, hy, hz);
            fx = fx + f.fx;
            fy = fy + f.fy;
            fz = fz + f.fz;
            tx = tx + f.tx;
            ty = ty + f.ty;
            tz = tz + f.tz;
            if (nc < c.maxc) a.hist_new[(size_t)nc * a.n + s] = make_float4(hx, hy, hz, __int_as_float(pid));
            ++nc;
        };
        auto touches = [&](int row) -> bool {
            const float4 q = rowpos[row];
            const float dx = p.x - q.x;
            const float dyy = p.y - q.y;
            const float dzz = p.z - q.z;
            const float d2 = dx * dx + dyy * dyy + dzz * dzz;
            const float rs = p.w + q.w;
            return d2 < rs * rs && d2 != 0.0f && is_contact(row, dx, dyy, dzz);
        };
        if constexpr (LISTED) {
            while (nc < hc) {  // the next one in ascending place
                int best = 0x7fffffff, row = 0;
                for (int k = 0; k < lcount; ++k) {
                    const int t = a.list_old[(size_t)k * a.n + os], place = a.newpos[t];
                    if (place > after && place < best && touches(t)) {
                        best = place;
                        row = t;
                    }
                }
                after = best;
                add(row);
            }
        } else {
            const int kept = min(hc, c.maxc);
            int row = nc < kept ? __float_as_int(a.hist_new[(size_t)nc * a.n + s].x) : 0;
            while (nc < kept) {
                const int next = nc + 1 < kept ? __float_as_int(a.hist_new[(size_t)(nc + 1) * a.n + s].x) : 0;
                add(row);
                row = next;
            }
            // more than the history holds (an error, but their forces count): searched again
            int skip = nc;
            for (int r = 0; r < 9 && nc < hc; ++r) {
                const int z = cz + r / 3 - 1, y = cy + r % 3 - 1;
                if (z < 0 || z >= g.nz || y < 0 || y >= g.ny) continue;
                int lo, hi;
                if constexpr (MODE == CONTACT_FORCES) row_range(g, ranges, cx, y, z, lo, hi);
                else row_window(g, ranges, cx, 1, y, z, lo, hi);
                for (int t = lo; t < hi && nc < hc; ++t) {
                    if (t == s) continue;
                    const int at = INDIRECT ? old_slot_of(a, t) : t;
                    if (!touches(at)) continue;
                    if (skip > 0) --skip;
                    else add(at);
                }
            }
        }
    }

    float4 v = a.vel[self];
    float4 w = a.omg[self];

    // walls: the touched ones first, so that the contact-law set-up of a wall
    // contact runs only where some lane of the wave touches a wall
    uint32_t touch = 0u;
    if (c.walls && v.w > 0.0f && live) {
#pragma unroll
        for (int wl = 0; wl < 6; ++wl) {
            const int ax = wl >> 1;
            const bool upper = wl & 1;
            const float pc = ax == 0 ? p.x : (ax == 1 ? p.y : p.z);
            const float dist = upper ? c.whi[ax] - pc : pc - c.wlo[ax];
            touch |= dist < p.w ? (1u << wl) : 0u;
        }
    }
    if (touch) {
#pragma unroll 1
        for (; touch; touch &= touch - 1u) {
            const int wl = __builtin_ctz(touch);
            const int ax = wl >> 1;
            const bool upper = wl & 1;
            const float pc = ax == 0 ? p.x : (ax == 1 ? p.y : p.z);
            const float wlo = ax == 0 ? c.wlo[0] : (ax == 1 ? c.wlo[1] : c.wlo[2]);
            const float whi = ax == 0 ? c.whi[0] : (ax == 1 ? c.whi[1] : c.whi[2]);
            const float dist = upper ? whi - pc : pc - wlo;
            const float sgn = upper ? -1.0f : 1.0f;
            const float nx = ax == 0 ? sgn : 0.0f;
            const float ny = ax == 1 ? sgn : 0.0f;
            const float nz = ax == 2 ? sgn : 0.0f;
            const int pid = -(wl + 1);
            float hx, hy, hz;
            find_history(a, os, oc, pid, nc, hx, hy, hz);
            const PairForce f = contact_law(c, nx, ny, nz, p.w - dist, p.w, 0.0f, v.w, 0.0f, v.x, v.y, v.z, w.x,
                                            w.y, w.z, 0.0f, 0.0f, 0.0f, hx, hy, hz);
            fx = fx + f.fx;
            fy = fy + f.fy;
            fz = fz + f.fz;
            tx = tx + f.tx;
            ty = ty + f.ty;
            tz = tz + f.tz;
            if (nc < c.maxc) a.hist_new[(size_t)nc * a.n + s] = make_float4(hx, hy, hz, __int_as_float(pid));
            ++nc;
        }
    }

    if (live) a.hcount_new[s] = nc < c.maxc ? nc : c.maxc;
    if (nc > c.maxc) atomicMax(a.overflow, nc);

    if (MODE == CONTACT_FORCES) {
        if (live) {
            a.force[s] = make_float4(fx, fy, fz, 0.0f);
            a.torque[s] = make_float4(tx, ty, tz, 0.0f);
        }
    } else {
        if constexpr (LISTED) {
            if (live) a.lcount_new[s] = (uint8_t)lcount;
        } else if constexpr (BUILD) {
            if (live) a.lcount_new[s] = (uint8_t)min(ln, LIST_CAP);
            if (__ballot(live && ln > LIST_CAP) != 0u && lane == 0) a.ctl->over = 1;
        }
        const float ox = p.x, oy = p.y, oz = p.z;
        integrate_sphere(c, p, v, w, fx, fy, fz, tx, ty, tz);
        if (LISTS != LIST_NONE || a.list_new) {  // (a context without lists needs none)
            const float dx = p.x - ox, dyy = p.y - oy, dzz = p.z - oz;
            note_displacement(a.ctl, live ? dx * dx + dyy * dyy + dzz * dzz : 0.0f);
        }
        if (live) {
            a.pos_o[s] = p;
            a.vel_o[s] = v;
            a.omg_o[s] = w;
            a.ids_o[s] = myid;
        }
        {
            const uint32_t cell_new = cbase + cell_id(g, p.x, p.y, p.z);
            const uint64_t key_new = ((uint64_t)cell_new << 32) | (uint64_t)(uint32_t)s;
            if (live) a.keys_o64[s] = key_new;
            // a sphere that left the cell it was sorted in: listed for the next
            // step's re-sort (one atomic per wave)
            const bool moved = a.mcount != nullptr && live && cell_new != cell_old;
            const uint64_t m = __ballot(moved);
            if (moved) {
                const int leader = __ffsll((long long)m) - 1;
                int first = 0;
                if (lane_id() == leader) first = atomicAdd(a.mcount, __popcll(m));
                first = __shfl(first, leader);
                const int i = first + __popcll(m & lanemask_lt());
                if (i < a.mcap) {
                    a.mnew[i] = key_new;
                    a.mold[i] = ((uint64_t)cell_old << 32) | (uint64_t)(uint32_t)s;
                }
            }
        }
    }
}


// Six waves a SIMD for the kernels that only search (a batch's takes 81 registers
// otherwise, one too many: 1.83M spheres of 128 scenes 195 us a step, 187 with one
// spilled; beside a body step 2.00 ms, 1.98).
template <int MODE, bool INDIRECT, bool STRADDLE, int LISTS>
__global__ __launch_bounds__(256, (LISTS == LIST_NONE && !STRADDLE ? 6 : 1)) void k_contacts(ContactArgs a) {
    static_assert(!STRADDLE || MODE == CONTACT_FUSED_BATCH, "k_contacts: straddling waves exist in batch mode only");
    static_assert(LISTS == LIST_NONE || INDIRECT, "k_contacts: only a context's steps have lists");
    if (MODE != CONTACT_FORCES) {
        if (a.ctl->given_up) return;
        if (!STRADDLE && blockIdx.x == 0 && threadIdx.x == 0) a.ctl->ran += 1;
    }
    int s;
    if constexpr (STRADDLE) {
        s = a.straddle[blockIdx.x] * WAVE + (int)threadIdx.x;
    } else {
        const int lb = xcd_logical_block((a.n + (int)blockDim.x - 1) / (int)blockDim.x);
        if (lb < 0) return;
        s = lb * (int)blockDim.x + (int)threadIdx.x;
    }
    contact_wave<MODE, INDIRECT, STRADDLE, LISTS>(a, s);
}

constexpr int PERSIST_CLAIM = 8;    // tiles a wave claims at a time
constexpr int PERSIST_STRIDE = 64;  // ints between the XCDs' counters

// Persistent form of the fused step kernel: a grid of resident blocks whose
// waves claim runs of PERSIST_CLAIM 64-slot tiles from a counter per XCD (tiles of XCD x are the
// x-th eighth of the slots, so an XCD's L2 still holds neighbouring cells)
// until its range is exhausted; the results are those of k_contacts (every
// tile computes the same slots the same way). counters[0..7] start at 0.
template <int MODE, int LISTS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_contacts_persistent(
    ContactArgs a, int* __restrict__ counters) {
    if (a.ctl->given_up) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl->ran += 1;
    const int ntiles = (a.n + WAVE - 1) / WAVE;
    const int per = (ntiles + XCDS - 1) / XCDS;
    const int x = (int)(blockIdx.x % XCDS);
    const int t0 = x * per, t1 = min(ntiles, t0 + per);
    int* const ctr = counters + PERSIST_STRIDE * x;  // one counter per XCD, each on its own 256-byte line
    for (;;) {
        int t = 0;
        if (lane_id() == 0) t = atomicAdd(ctr, PERSIST_CLAIM);
        t = t0 + __shfl(t, 0);
        if (t >= t1) break;
        const int te = min(t + PERSIST_CLAIM, t1);
        for (; t < te; ++t) contact_wave<MODE, true, false, LISTS>(a, t * WAVE + lane_id());
    }
}

__global__ void k_integrate(float4* __restrict__ pos, float4* __restrict__ vel, float4* __restrict__ omg,
                            const float4* __restrict__ f, const float4* __restrict__ t, int n, ContactDev c) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pos[i], v = vel[i], w = omg[i];
    const float4 F = f[i], T = t[i];
    integrate_sphere(c, p, v, w, F.x, F.y, F.z, T.x, T.y, T.z);
    pos[i] = p;
    vel[i] = v;
    omg[i] = w;
}

template <typename F>
static F by_lists(int lists, F use, F build, F none) {
    return lists == LIST_USE ? use : (lists == LIST_BUILD ? build : none);
}

sd_status launch_contacts(int mode, const ContactArgs& a, hipStream_t s, int block) {
    if (a.n <= 0) return SD_OK;
    if (block <= 0) block = 128;
    SD_REQUIRE(block % WAVE == 0 && block <= 256, "contact kernel: block must be a multiple of 64, <= 256");
    const int nblocks = div_up(a.n, block);
    const dim3 grid(div_up(nblocks, XCDS) * XCDS);  // padded for the XCD remap
    const int lists = mode == CONTACT_FORCES ? LIST_NONE : a.lists;
    const size_t lds = (size_t)(block / WAVE) * contact_lds(mode, lists) * sizeof(float4);
    void (*const kernel)(ContactArgs) =
        mode == CONTACT_FORCES      ? &k_contacts<CONTACT_FORCES, false, false, LIST_NONE>
        : mode == CONTACT_FUSED_U64 ? by_lists(lists, &k_contacts<CONTACT_FUSED_U64, true, false, LIST_USE>,
                                               &k_contacts<CONTACT_FUSED_U64, true, false, LIST_BUILD>,
                                               &k_contacts<CONTACT_FUSED_U64, true, false, LIST_NONE>)
                                    : by_lists(lists, &k_contacts<CONTACT_FUSED_BATCH, true, false, LIST_USE>,
                                               &k_contacts<CONTACT_FUSED_BATCH, true, false, LIST_BUILD>,
                                               &k_contacts<CONTACT_FUSED_BATCH, true, false, LIST_NONE>);
    hipLaunchKernelGGL(kernel, grid, dim3(block), lds, s, a);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

sd_status launch_contacts_persistent(int mode, const ContactArgs& a, hipStream_t s, int block, int* counters) {
    if (a.n <= 0) return SD_OK;
    if (block <= 0) block = 128;
    SD_REQUIRE(block % WAVE == 0 && block <= 256, "contact kernel: block must be a multiple of 64, <= 256");
    SD_REQUIRE(mode == CONTACT_FUSED_U64 || mode == CONTACT_FUSED_BATCH,
               "contact kernel: the persistent form is for packed 64-bit keys");
    void (*const kernel)(ContactArgs, int*) =
        mode == CONTACT_FUSED_U64 ? by_lists(a.lists, &k_contacts_persistent<CONTACT_FUSED_U64, LIST_USE>,
                                             &k_contacts_persistent<CONTACT_FUSED_U64, LIST_BUILD>,
                                             &k_contacts_persistent<CONTACT_FUSED_U64, LIST_NONE>)
                                  : by_lists(a.lists, &k_contacts_persistent<CONTACT_FUSED_BATCH, LIST_USE>,
                                             &k_contacts_persistent<CONTACT_FUSED_BATCH, LIST_BUILD>,
                                             &k_contacts_persistent<CONTACT_FUSED_BATCH, LIST_NONE>);
    const size_t lds = (size_t)(block / WAVE) * contact_lds(mode, a.lists) * sizeof(float4);
    int dev = 0, cus = 0, per_cu = 0;
    SD_HIP(hipGetDevice(&dev));
    SD_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    SD_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), block, lds));
    // every resident block, at most one per tile, a multiple of the XCD count
    const int tiles = div_up(a.n, WAVE);
    int nb = std::max(1, per_cu) * std::max(1, cus);
    nb = std::min(nb, div_up(tiles, block / WAVE));
    nb = std::max(XCDS, nb / XCDS * XCDS);
    sd_status st = launch_fill_u32((uint32_t*)counters, 0u, (size_t)PERSIST_STRIDE * XCDS, s);
    if (st != SD_OK) return st;
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(block), lds, s, a, counters);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

sd_status launch_contacts_straddle(const ContactArgs& a, hipStream_t s) {
    if (a.n <= 0 || a.n_straddle <= 0) return SD_OK;
    SD_REQUIRE(a.straddle && a.scenes && a.scene_of, "contact kernel: straddle launch without its lists");
    const size_t lds = (size_t)contact_lds(CONTACT_FUSED_BATCH, a.lists) * sizeof(float4);
    hipLaunchKernelGGL(by_lists(a.lists, &k_contacts<CONTACT_FUSED_BATCH, true, true, LIST_USE>,
                                &k_contacts<CONTACT_FUSED_BATCH, true, true, LIST_BUILD>,
                                &k_contacts<CONTACT_FUSED_BATCH, true, true, LIST_NONE>),
                       dim3(a.n_straddle), dim3(WAVE), lds, s, a);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

sd_status launch_integrate(float4* pos, float4* vel, float4* omg, const float4* f, const float4* t, int n,
                           const ContactDev& c, hipStream_t s) {
    if (n <= 0) return SD_OK;
    hipLaunchKernelGGL(k_integrate, dim3(div_up(n, 256)), dim3(256), 0, s, pos, vel, omg, f, t, n, c);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

}  // namespace sd

using namespace sd;

extern "C" sd_status sd_contact_forces(const float* pos4, const float* vel4, const float* omg4, const int* ids, int n,
                                       const sd_grid* grid, const int* ranges, const sd_contact_params* cp,
                                       const int* old_slot, const int* hist_count_old, const float* hist4_old,
                                       int* hist_count_new, float* hist4_new, float* force4, float* torque4,
                                       int* overflow, void* stream) {
    sd_status st = check_grid(grid);
    if (st != SD_OK) return st;
    st = check_contact(cp);
    if (st != SD_OK) return st;
    SD_REQUIRE(n >= 0, "sd_contact_forces: n < 0");
    if (n == 0) return SD_OK;
    SD_REQUIRE(pos4 && vel4 && omg4 && ids && ranges && old_slot && hist_count_old && hist4_old && hist_count_new &&
                   hist4_new && force4 && torque4 && overflow,
               "sd_contact_forces: null pointer");
    ContactArgs a = {};
    a.pos = (const float4*)pos4;
    a.vel = (const float4*)vel4;
    a.omg = (const float4*)omg4;
    a.ids = ids;
    a.n = n;
    a.g = to_dev(*grid);
    a.ranges = ranges;
    a.c = to_dev(*cp);
    a.old_slot_i32 = old_slot;
    a.hcount_old = hist_count_old;
    a.hist_old = (const float4*)hist4_old;
    a.hcount_new = hist_count_new;
    a.hist_new = (float4*)hist4_new;
    a.overflow = overflow;
    a.force = (float4*)force4;
    a.torque = (float4*)torque4;
    return launch_contacts(CONTACT_FORCES, a, (hipStream_t)stream, 128);
}

extern "C" sd_status sd_integrate_spheres(float* pos4, float* vel4, float* omg4, const float* force4,
                                          const float* torque4, int n, const sd_contact_params* cp, void* stream) {
    sd_status st = check_contact(cp);
    if (st != SD_OK) return st;
    SD_REQUIRE(n >= 0, "sd_integrate_spheres: n < 0");
    if (n == 0) return SD_OK;
    SD_REQUIRE(pos4 && vel4 && omg4 && force4 && torque4, "sd_integrate_spheres: null pointer");
    return launch_integrate((float4*)pos4, (float4*)vel4, (float4*)omg4, (const float4*)force4,
                            (const float4*)torque4, n, to_dev(*cp), (hipStream_t)stream);
}
