// Rigid clumps of spheres: pose, body AABBs, LBVH broadphase, deterministic
// per-body contact gather and semi-implicit quaternion integration.
//
// Replaces updateSphereDataCUDA (src/engine/cuda/physics_update.cu:26-140),
// computeForcesAndTorquesCUDA (:144-228) and advectParticlesCUDA (:232-348)
// with their helpers (src/engine/cuda/cuda_helpers.cuh:65-171). Differences by
// design: the world inverse inertia is R I^-1 R^T (quirk Q11: the reference mixes
// row- and column-major helpers), a singular inertia is not replaced by its input
// (Q10), the quaternion is renormalised every step (Q12), static bodies carry an
// explicit 1/m = 0 instead of mass >= 10 (Q13), and each body gathers the forces
// of its contacts instead of racing scatters (Q7).
//
// Per step: poses (world angular velocity, sphere positions, body boxes), then
// one kernel per body takes its partners, sums its sphere-sphere contacts
// (partners ascending, own spheres ascending, partner spheres ascending) and
// integrates it. Partners come from a list that a step every few tens builds
// (ClumpCtl below), or, for bodies too fast or crowded for lists, from a tree
// that every step builds: global domain, Morton keys, radix sort, LBVH build.
// Every launch has a fixed size, so steps are captured into hipGraphs and
// replayed; the candidate pair list (unique a < b) of the last step's boxes is
// built only when asked for (sd_clump_pairs).
//
// Integration of a body with 1/m > 0 (FP32, fixed operation order):
//   v += (F/m + g) dt;  x += v dt;  L += T dt
//   w  = R I^-1 R^T L (R from the current q);  a = |w| (dt/2)
//   dq = (cos a, w sin(a)/|w|), q = normalise(dq q)
// sin and cos come from fixed Taylor polynomials for a < 0.25 (exact to FP32)
// so the CPU restatement reproduces the bits; larger angles use sinf/cosf.
#include <cstring>
#include <vector>

#include "sd_contact_law.hpp"
#include "sd_gjk_dev.hpp"
#include "sd_internal.hpp"
#include "sd_list_plan.hpp"
#include "sd_rigid_dev.hpp"

extern "C" sd_status sd_global_domain(const float* lo4, const float* hi4, int n, float* domain6, void* scratch,
                                      void* stream);
extern "C" sd_status sd_morton30(const float* lo4, const float* hi4, int n, const float* domain6, uint64_t* keys,
                                 void* stream);
extern "C" sd_status sd_lbvh_build(const uint64_t* sorted_keys, int n, const float* lo4, const float* hi4, int* left,
                                   int* right, int* parent, int* first, int* last, int* rope, float* node_lo4,
                                   float* node_hi4, int* counters, int* error, void* stream);
extern "C" sd_status sd_lbvh_query_scratch_bytes(int n, size_t* bytes);
extern "C" sd_status sd_lbvh_query(const uint64_t* sorted_keys, int n, const int* left, const int* last,
                                   const int* rope, const float* node_lo4, const float* node_hi4, int* pairs,
                                   int capacity, int* n_pairs, int* error, void* scratch, size_t scratch_bytes,
                                   void* stream);

namespace sd {

struct ClumpState {
    const float4* pos;   // (x, y, z, 1/m)
    const float4* vel;   // (vx, vy, vz, 0)
    const float4* quat;  // (w, x, y, z)
    const float4* angm;  // (Lx, Ly, Lz, 0)
};

// Partner lists of a clump context, as the near lists of the sphere contexts: a
// step that builds them inflates the body boxes by a margin, and the steps
// after it take a body's partners from the listed ones whose boxes overlap,
// instead of building and walking a tree. displaced sums the largest movement
// of a box face per step since the build; a pair outside the lists has boxes
// apart while that is below limit (the margin, less what rounding can take). A
// step whose lists have run out is given up and redone with a build.
constexpr int CL_LIST = 16;  // partners listed per body
struct ClumpCtl {
    int given_up;        // != 0: every later kernel of the launch sequence returns at once
    int ran;             // steps that ran
    int error;           // malformed tree
    int over;            // a body had more partners than its list holds
    float displaced[2];  // by buffer parity of the step (written for the next one)
    float limit;
    float last;          // movement of the last step
    float margin;
    int pad[7];
    uint32_t dmax[2][LIST_SLOTS * 16];  // by parity: face movements of the step (float bits)
};
constexpr int CLUMP_CTL_READ = 9;

// Largest face movement of the step, by a whole wave.
__device__ __forceinline__ float step_movement(const uint32_t* dmax) {
    uint32_t u = dmax[lane_id() * 16];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        const uint32_t o = __shfl_xor(u, d);
        u = o > u ? o : u;
    }
    return __uint_as_float(u) * 1.00001f;
}

// A build's margin and limit (domain: of the boxes), the lists' displacement 0.
__global__ __launch_bounds__(64) void k_clump_margin(ClumpCtl* __restrict__ ctl, int par, float size,
                                                     const float* __restrict__ domain) {
    if (ctl->given_up) return;
    const float m = step_movement(ctl->dmax[par]);
    if (threadIdx.x != 0) return;
    float far = 0.0f;
    for (int k = 0; k < 6; ++k) far = fmaxf(far, fabsf(domain[k]));
    const float margin = clump_build_margin(m, size, far);
    ctl->margin = margin;
    ctl->limit = clump_limit(margin, far);
    ctl->over = 0;
}

__global__ void k_clump_inflate(const float4* __restrict__ lo, const float4* __restrict__ hi, int nb,
                                const ClumpCtl* __restrict__ ctl, float4* __restrict__ ilo,
                                float4* __restrict__ ihi) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb || ctl->given_up) return;
    const float m = ctl->margin;
    const float4 l = lo[b], h = hi[b];
    ilo[b] = make_float4(l.x - m, l.y - m, l.z - m, 0.0f);
    ihi[b] = make_float4(h.x + m, h.y + m, h.z + m, 0.0f);
}

// Angular velocity and box of every body, world positions of its spheres, how
// far the box's faces moved since the step before. Bound by the rows it reads
// and writes (36 bytes a sphere, 150 a body: 134 MB at 262,144 bodies of 10
// spheres); POSE_LANES lanes share a body, so that its spheres are read and
// written in runs. Three passes, with the velocity of every sphere written too,
// took 41 us, this one 22.
constexpr int POSE_LANES = 4;
__global__ __launch_bounds__(256) void k_clump_pose(
    ClumpState st, const float4* __restrict__ i0, const float4* __restrict__ i1, const float4* __restrict__ slocal,
    const int* __restrict__ bfirst, const int* __restrict__ bcount, int nb, float4* __restrict__ omega,
    float4* __restrict__ sx, float4* __restrict__ lo4, float4* __restrict__ hi4, ClumpCtl* __restrict__ ctl, int par,
    int track) {
    if (ctl->given_up) return;
    const int at = blockIdx.x * (256 / POSE_LANES) + threadIdx.x / POSE_LANES, sub = threadIdx.x % POSE_LANES;
    const bool mine = at < nb;
    const int b = min(at, nb - 1);  // (past the end: the last body again, nothing written or counted)
    const int k0 = bfirst[b], kn = bcount[b];
    const float4 X = st.pos[b], L = st.angm[b];
    const Rot R = quat_rot(st.quat[b]);
    float lx = 3.402823466e38f, ly = 3.402823466e38f, lz = 3.402823466e38f;
    float hx = -3.402823466e38f, hy = -3.402823466e38f, hz = -3.402823466e38f;
    // 4 spheres a lane with their loads in flight; indices past the last
    // sphere repeat it (min and max do not change)
    for (int k = sub; k < kn; k += 4 * POSE_LANES) {
        float4 l[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) l[j] = slocal[k0 + min(k + j * POSE_LANES, kn - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const V3 r = rot_mul(R, v3(l[j].x, l[j].y, l[j].z));
            const float4 x = make_float4(X.x + r.x, X.y + r.y, X.z + r.z, l[j].w);
            lx = fminf(lx, x.x - x.w);
            ly = fminf(ly, x.y - x.w);
            lz = fminf(lz, x.z - x.w);
            hx = fmaxf(hx, x.x + x.w);
            hy = fmaxf(hy, x.y + x.w);
            hz = fmaxf(hz, x.z + x.w);
            if (mine && k + j * POSE_LANES < kn) sx[k0 + k + j * POSE_LANES] = x;
        }
    }
#pragma unroll
    for (int d = 1; d < POSE_LANES; d <<= 1) {
        lx = fminf(lx, __shfl_xor(lx, d));
        ly = fminf(ly, __shfl_xor(ly, d));
        lz = fminf(lz, __shfl_xor(lz, d));
        hx = fmaxf(hx, __shfl_xor(hx, d));
        hy = fmaxf(hy, __shfl_xor(hy, d));
        hz = fmaxf(hz, __shfl_xor(hz, d));
    }
    if (track) {
        const float4 l = lo4[b], h = hi4[b];
        const float a0 = fabsf(lx - l.x), a1 = fabsf(ly - l.y), a2 = fabsf(lz - l.z);
        const float a3 = fabsf(hx - h.x), a4 = fabsf(hy - h.y), a5 = fabsf(hz - h.z);
        const float sum = ((a0 + a1) + (a2 + a3)) + (a4 + a5);
        const float m = sum < 3.4e38f ? fmaxf(fmaxf(fmaxf(a0, a1), fmaxf(a2, a3)), fmaxf(a4, a5)) : __builtin_inff();
        uint32_t u = mine ? __float_as_uint(m) : 0u;
#pragma unroll
        for (int d = POSE_LANES; d < 64; d <<= 1) {
            const uint32_t o = __shfl_xor(u, d);
            u = o > u ? o : u;
        }
        if (lane_id() == 0) atomicMax(&ctl->dmax[par][((blockIdx.x * 4u + (threadIdx.x >> 6)) & 63u) * 16u], u);
    }
    if (!mine || sub != 0) return;
    const V3 w = inv_inertia_apply(R, i0[b], i1[b], v3(L.x, L.y, L.z));
    omega[b] = make_float4(w.x, w.y, w.z, 0.0f);
    lo4[b] = make_float4(lx, ly, lz, 0.0f);
    hi4[b] = make_float4(hx, hy, hz, 0.0f);
}

// Velocity of the point at l (body frame) of a body.
__device__ __forceinline__ V3 sphere_velocity(float4 quat, float4 V, float4 w, float4 l) {
    const V3 r = rot_mul(quat_rot(quat), v3(l.x, l.y, l.z));
    return v3(V.x + (w.y * r.z - w.z * r.y), V.y + (w.z * r.x - w.x * r.z), V.z + (w.x * r.y - w.y * r.x));
}

constexpr int CL_BLOCK = 128;
constexpr int CL_PCAP = 32;  // partners listed per body and pass
constexpr int CL_SENTINEL = -1;
constexpr int CL_MORTON_DROP = 6;  // lowest Morton code bits not sorted on (24 of 30 kept)

__device__ __forceinline__ bool cl_overlap(float4 al, float4 ah, float4 bl, float4 bh) {
    return al.x <= bh.x && bl.x <= ah.x && al.y <= bh.y && bl.y <= ah.y && al.z <= bh.z && bl.z <= ah.z;
}

// One body per thread: its partners (every body whose AABB overlaps its own),
// visited in ascending body id, then integration. LIST_USE takes them from the
// body's list. Otherwise a pass walks the tree (stackless, ropes) and keeps the
// CL_PCAP smallest partner ids above the last pass's largest, sorted in LDS; a
// body with more partners takes more passes. The walk's bound turns a malformed
// tree into an error flag. LIST_BUILD: the tree is one of inflated boxes, and
// what the walk finds is listed.
//
// Bound by the latency of dependent loads: a node a step of the walk, then
// batches of 4 spheres. 262,144 bodies of 10 spheres: 169 us where every sphere
// of a body is tested against every one of a partner; 162 with the lists alone;
// 46 with the lists and the spheres beyond the partner's box left out (119 for
// the step that builds them). Batches of 8 (157 registers) took 51. The lists
// also save the step the keys, sort and tree (116 us).
template <int LISTS>
__global__ __launch_bounds__(CL_BLOCK) void k_clump_contacts(
    ClumpState st, ClumpState out, const float4* __restrict__ omega, const float4* __restrict__ i0,
    const float4* __restrict__ i1, const float4* __restrict__ sx, const float4* __restrict__ slocal,
    const int* __restrict__ bfirst, const int* __restrict__ bcount, int nb, const float4* __restrict__ blo,
    const float4* __restrict__ bhi, const float4* __restrict__ pnode, ContactDev c, ClumpCtl* __restrict__ ctl,
    int par, uint8_t* __restrict__ lcount, int* __restrict__ list) {
    if (ctl->given_up) return;
    {
        const float m = step_movement(ctl->dmax[par]);
        const float D = LISTS == LIST_USE ? (ctl->displaced[par] + m) * 1.0000002f  // (rounded up)
                                          : (LISTS == LIST_BUILD ? 0.0f : __builtin_inff());
        const bool out_of_margin = LISTS == LIST_USE && (!(D <= ctl->limit) || ctl->over);
        if (blockIdx.x == 0 && threadIdx.x < 64) {
            if (out_of_margin) {
                // (every block sees the same: nothing else is written)
                if (threadIdx.x == 0) ctl->given_up = GIVEN_UP_LIST;
            } else {
                ctl->dmax[1 - par][threadIdx.x * 16] = 0u;
                if (threadIdx.x == 0) {
                    ctl->displaced[1 - par] = D;
                    ctl->last = m;
                    ctl->ran += 1;
                }
            }
        }
        if (out_of_margin) return;
    }
    __shared__ int plist[LISTS == LIST_USE ? 1 : CL_BLOCK][CL_PCAP + 1];  // (+1: rows start in different banks)
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const float4 X = st.pos[b];
    const float4 wb4 = omega[b];
    const int f0 = bfirst[b], fn = bcount[b];
    const float4 ql = blo[b], qh = bhi[b];
    float Fx = 0.0f, Fy = 0.0f, Fz = 0.0f, Tx = 0.0f, Ty = 0.0f, Tz = 0.0f;
    auto partner = [&](int p) {
        const float inv_mp = st.pos[p].w;
        if (X.w + inv_mp == 0.0f) return;  // two static bodies
        const float4 wp4 = omega[p], pl4 = blo[p], ph4 = bhi[p];
        const int g0 = bfirst[p], gn = bcount[p];
        // A sphere beyond the partner's box touches none of its spheres; the
        // slack covers what rounding can take from the sums on both sides.
        const float ex = 1e-6f * (fabsf(pl4.x) + fabsf(ph4.x)), ey = 1e-6f * (fabsf(pl4.y) + fabsf(ph4.y)),
                    ez = 1e-6f * (fabsf(pl4.z) + fabsf(ph4.z));
        auto beyond = [&](float x, float w, float lo, float hi, float e) {
            const float s = e + 1e-6f * (fabsf(x) + w);
            return (x - w) - hi > s || lo - (x + w) > s;
        };
        for (int ib = f0; ib < f0 + fn; ib += 4) {
            uint32_t near = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float4 x = sx[min(ib + u, f0 + fn - 1)];
                const bool out = beyond(x.x, x.w, pl4.x, ph4.x, ex) || beyond(x.y, x.w, pl4.y, ph4.y, ey) ||
                                 beyond(x.z, x.w, pl4.z, ph4.z, ez);
                if (!out && ib + u < f0 + fn) near |= 1u << u;
            }
            while (near) {
                const int i = ib + __builtin_ctz(near);
                near &= near - 1u;
                const float4 xi = sx[i];
                for (int jb = g0; jb < g0 + gn; jb += 4) {
                    uint32_t hit = 0;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float4 xj = sx[min(jb + u, g0 + gn - 1)];
                        const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                        const float d2 = dx * dx + dy * dy + dz * dz;
                        const float rs = xi.w + xj.w;
                        if (d2 < rs * rs && d2 != 0.0f && jb + u < g0 + gn) hit |= 1u << u;
                    }
                    while (hit) {
                        const int j = jb + __builtin_ctz(hit);
                        hit &= hit - 1u;
                        const float4 xj = sx[j];
                        const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                        const float d = sqrtf(dx * dx + dy * dy + dz * dz);
                        const float inv_d = 1.0f / d;
                        const V3 vi = sphere_velocity(st.quat[b], st.vel[b], wb4, slocal[i]);
                        const V3 vj = sphere_velocity(st.quat[p], st.vel[p], wp4, slocal[j]);
                        float hx = 0.0f, hy = 0.0f, hz = 0.0f;  // no tangential history for clumps
                        const PairForce f = contact_law(c, dx * inv_d, dy * inv_d, dz * inv_d, xi.w + xj.w - d, xi.w,
                                                        xj.w, X.w, inv_mp, vi.x - vj.x, vi.y - vj.y, vi.z - vj.z,
                                                        wb4.x, wb4.y, wb4.z, wp4.x, wp4.y, wp4.z, hx, hy, hz);
                        Fx = Fx + f.fx;
                        Fy = Fy + f.fy;
                        Fz = Fz + f.fz;
                        const float ax = xi.x - X.x, ay = xi.y - X.y, az = xi.z - X.z;
                        Tx = Tx + ((ay * f.fz - az * f.fy) + f.tx);
                        Ty = Ty + ((az * f.fx - ax * f.fz) + f.ty);
                        Tz = Tz + ((ax * f.fy - ay * f.fx) + f.tz);
                    }
                }
            }
        }
    };
    if constexpr (LISTS == LIST_USE) {
        const int n = lcount[b];
        for (int k = 0; k < n; ++k) {
            const int p = list[(size_t)k * nb + b];
            if (cl_overlap(ql, qh, blo[p], bhi[p])) partner(p);
        }
    } else {
        int* const pl = plist[threadIdx.x];  // this body's partners
        float4 wl = ql, wh = qh;             // the box that walks
        if (LISTS == LIST_BUILD) {
            const float m = ctl->margin;
            wl = make_float4(ql.x - m, ql.y - m, ql.z - m, 0.0f);
            wh = make_float4(qh.x + m, qh.y + m, qh.z + m, 0.0f);
        }
        int listed = 0;
        for (int lower = -1;;) {
            int np = 0;
            bool more = false;
            int node = nb == 1 ? CL_SENTINEL : 0;
            for (int guard = 0; node != CL_SENTINEL; ++guard) {
                if (guard > 2 * nb + 2 || node < 0 || node >= 2 * nb - 1) {
                    atomicOr(&ctl->error, 4);
                    break;
                }
                // one load step per node: box, the next node if the boxes
                // overlap (left child, or a leaf's body), and the rope
                const float4 nl = pnode[2 * (size_t)node], nh = pnode[2 * (size_t)node + 1];
                if (!cl_overlap(wl, wh, nl, nh)) {
                    node = __float_as_int(nh.w);
                    continue;
                }
                if (node >= nb - 1) {  // a leaf: one body
                    const int p = __float_as_int(nl.w);
                    if (p != b && p > lower && p < nb) {
                        if (np == CL_PCAP) more = true;  // partners beyond this pass's list
                        if (np < CL_PCAP || p < pl[CL_PCAP - 1]) {
                            int k = np < CL_PCAP ? np++ : CL_PCAP - 1;  // the largest drops out of a full list
                            while (k > 0 && pl[k - 1] > p) {
                                pl[k] = pl[k - 1];
                                --k;
                            }
                            pl[k] = p;
                        }
                    }
                    node = __float_as_int(nh.w);
                } else {
                    node = __float_as_int(nl.w);
                }
            }
            for (int e = 0; e < np; ++e) {
                const int p = pl[e];
                if (LISTS == LIST_BUILD) {
                    if (listed < CL_LIST) list[(size_t)listed * nb + b] = p;
                    ++listed;
                    if (!cl_overlap(ql, qh, blo[p], bhi[p])) continue;
                }
                partner(p);
            }
            if (!more) break;
            lower = pl[CL_PCAP - 1];
        }
        if (LISTS == LIST_BUILD) {
            lcount[b] = (uint8_t)min(listed, CL_LIST);
            if (listed > CL_LIST) ctl->over = 1;
        }
    }
    float4 P = X, V = st.vel[b], q = st.quat[b], L = st.angm[b];
    integrate_body(P, V, q, L, i0[b], i1[b], Fx, Fy, Fz, Tx, Ty, Tz, c);
    ((float4*)out.pos)[b] = P;
    ((float4*)out.vel)[b] = V;
    ((float4*)out.quat)[b] = q;
    ((float4*)out.angm)[b] = L;
}

// Per-body sums of per-sphere forces over the body's sphere range, in sphere
// order: F = sum f, T = sum ((x_s - X) x f + tau_s).
__global__ void k_body_reduce(const float4* __restrict__ bpos, const int* __restrict__ first,
                              const int* __restrict__ count, int nb, const float4* __restrict__ spos,
                              const float4* __restrict__ sf, const float4* __restrict__ st,
                              float4* __restrict__ bf, float4* __restrict__ bt) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const float4 X = bpos[b];
    float Fx = 0.0f, Fy = 0.0f, Fz = 0.0f, Tx = 0.0f, Ty = 0.0f, Tz = 0.0f;
    const int f0 = first[b], fn = count[b];
    for (int i = f0; i < f0 + fn; ++i) {
        const float4 x = spos[i], f = sf[i], t = st[i];
        Fx = Fx + f.x;
        Fy = Fy + f.y;
        Fz = Fz + f.z;
        const float ax = x.x - X.x, ay = x.y - X.y, az = x.z - X.z;
        Tx = Tx + ((ay * f.z - az * f.y) + t.x);
        Ty = Ty + ((az * f.x - ax * f.z) + t.y);
        Tz = Tz + ((ax * f.y - ay * f.x) + t.z);
    }
    bf[b] = make_float4(Fx, Fy, Fz, 0.0f);
    bt[b] = make_float4(Tx, Ty, Tz, 0.0f);
}

// One semi-implicit step per body (integrate_body), in place.
__global__ void k_integrate_bodies(float4* __restrict__ pos, float4* __restrict__ vel, float4* __restrict__ quat,
                                   float4* __restrict__ angm, const float* __restrict__ inv6,
                                   const float4* __restrict__ force, const float4* __restrict__ torque, int nb,
                                   ContactDev c) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    float4 P = pos[b], V = vel[b], q = quat[b], L = angm[b];
    const float* I = inv6 + 6 * (size_t)b;
    const float4 i0 = make_float4(I[0], I[1], I[2], I[3]), i1 = make_float4(I[4], I[5], 0.0f, 0.0f);
    const float4 F = force[b], T = torque[b];
    integrate_body(P, V, q, L, i0, i1, F.x, F.y, F.z, T.x, T.y, T.z, c);
    pos[b] = P;
    vel[b] = V;
    quat[b] = q;
    angm[b] = L;
}

}  // namespace sd

using namespace sd;

extern "C" sd_status sd_body_reduce(const float* body_pos4, const int* first, const int* count, int nb,
                                    const float* sphere_pos4, const float* sphere_force4,
                                    const float* sphere_torque4, float* body_force4, float* body_torque4,
                                    void* stream) {
    SD_REQUIRE(nb >= 0, "sd_body_reduce: nb < 0");
    if (nb == 0) return SD_OK;
    SD_REQUIRE(body_pos4 && first && count && sphere_pos4 && sphere_force4 && sphere_torque4 && body_force4 &&
                   body_torque4,
               "sd_body_reduce: null pointer");
    hipLaunchKernelGGL(k_body_reduce, dim3(div_up(nb, 256)), dim3(256), 0, (hipStream_t)stream,
                       (const float4*)body_pos4, first, count, nb, (const float4*)sphere_pos4,
                       (const float4*)sphere_force4, (const float4*)sphere_torque4, (float4*)body_force4,
                       (float4*)body_torque4);
    SD_LAUNCH_CHECK();
    return SD_OK;
}

extern "C" sd_status sd_integrate_bodies(float* pos4, float* vel4, float* quat4, float* angmom4,
                                         const float* inv_inertia6, const float* force4, const float* torque4, int nb,
                                         const sd_contact_params* cp, void* stream) {
    SD_REQUIRE(nb >= 0 && cp, "sd_integrate_bodies: bad argument");
    if (nb == 0) return SD_OK;
    SD_REQUIRE(pos4 && vel4 && quat4 && angmom4 && inv_inertia6 && force4 && torque4,
               "sd_integrate_bodies: null pointer");
    sd_status st = check_contact(cp);
    if (st != SD_OK) return st;
    hipLaunchKernelGGL(k_integrate_bodies, dim3(div_up(nb, 256)), dim3(256), 0, (hipStream_t)stream, (float4*)pos4,
                       (float4*)vel4, (float4*)quat4, (float4*)angmom4, inv_inertia6, (const float4*)force4,
                       (const float4*)torque4, nb, to_dev(*cp));
    SD_LAUNCH_CHECK();
    return SD_OK;
}

// ------------------------------------------------------------------ clump scene context

struct sd_clump_ctx {
    sd_clump_params p{};
    hipStream_t stream = nullptr;
    int nb = 0, ns = 0;
    float4 *pos[2] = {}, *vel[2] = {}, *quat[2] = {}, *angm[2] = {};
    int cur = 0;
    float4 *i0 = nullptr, *i1 = nullptr, *omega = nullptr;
    int *bfirst = nullptr, *bcount = nullptr;
    float4 *slocal = nullptr, *sx = nullptr;
    float4 *blo = nullptr, *bhi = nullptr;
    float* domain = nullptr;
    float* dom_scratch = nullptr;
    uint64_t *mkeys = nullptr, *mkeys2 = nullptr;
    void* sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    int *left = nullptr, *right = nullptr, *parent = nullptr, *first = nullptr, *last = nullptr, *rope = nullptr;
    float4 *nlo = nullptr, *nhi = nullptr;
    float4* pnode = nullptr;  // 2 per node: the walk's packed tree
    int* counters = nullptr;
    void* q_scratch = nullptr;
    size_t q_scratch_bytes = 0;
    int* pairs = nullptr;
    int pair_cap = 0;
    int npairs = 0;
    const uint64_t* ksorted = nullptr;  // sorted Morton keys of the last step's tree
    bool have_tree = false;   // a step has run
    bool tree_last = false;   // the tree is that of the last step's boxes
    hipGraphExec_t graph[2][3] = {};  // two steps from buffer parity 0 / 1, by what they do with the lists
    hipGraph_t graph_obj[2][3] = {};
    // partner lists, and the inflated boxes of a step that builds them, all in
    // list_mem; NULL: none, every step walks a tree
    char* list_mem = nullptr;
    float4 *ilo = nullptr, *ihi = nullptr;
    int* list = nullptr;
    uint8_t* lcount = nullptr;
    ClumpCtl* ctl = nullptr;
    float size = 0.0f;        // mean extent of the bodies
    ListPlan plan;
    bool boxes = false;       // blo / bhi are those of the step before
    long long steps_done = 0;
    uint64_t static_hash = 0;  // of the fixed rows (inverse inertia, sphere ranges and offsets)
};

namespace {

template <typename T>
sd_status dalloc(T** p, size_t count) {
    SD_HIP(hipMalloc((void**)p, (count ? count : 1) * sizeof(T)));
    return SD_OK;
}

void drop_clump_graphs(sd_clump_ctx* c) {
    for (int k = 0; k < 2; ++k)
        for (int l = 0; l < 3; ++l) {
            if (c->graph[k][l]) (void)hipGraphExecDestroy(c->graph[k][l]);
            if (c->graph_obj[k][l]) (void)hipGraphDestroy(c->graph_obj[k][l]);
            c->graph[k][l] = nullptr;
            c->graph_obj[k][l] = nullptr;
        }
}

void cfree(sd_clump_ctx* c) {
    void* bufs[] = {c->pos[0],  c->pos[1],    c->vel[0],     c->vel[1],   c->quat[0], c->quat[1],  c->angm[0],
                    c->angm[1], c->i0,        c->i1,         c->omega,    c->bfirst,  c->bcount,
                    c->slocal,  c->sx,        c->blo,      c->bhi,     c->domain,   c->dom_scratch,
                    c->mkeys,   c->mkeys2,    c->sort_tmp,   c->left,     c->right,   c->parent,   c->first,
                    c->last,    c->rope,      c->nlo,        c->nhi,      c->counters, c->q_scratch,
                    c->pairs,   c->pnode,     c->ctl,        c->list_mem};
    drop_clump_graphs(c);
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    sd_clump_params keep = c->p;
    hipStream_t s = c->stream;
    *c = sd_clump_ctx();
    c->p = keep;
    c->stream = s;
}

sd_status grow_pairs(sd_clump_ctx* c, int need) {
    if (need <= c->pair_cap) return SD_OK;
    int cap = need + need / 2 + 1024;
    if (c->pairs) (void)hipFree(c->pairs);
    c->pairs = nullptr;
    sd_status st = dalloc(&c->pairs, 2 * (size_t)cap);
    if (st != SD_OK) return st;
    c->pair_cap = cap;
    return SD_OK;
}

int bits_for(uint64_t v) {
    int b = 1;
    while (b < 64 && (1ull << b) < v) ++b;
    return b;
}

ClumpState state_of(sd_clump_ctx* c, int k) { return ClumpState{c->pos[k], c->vel[k], c->quat[k], c->angm[k]}; }

// The tree of the boxes lo / hi over the domain of the exact ones.
sd_status clump_tree(sd_clump_ctx* c, const float4* lo, const float4* hi, hipEvent_t* ev) {
    hipStream_t s = c->stream;
    const int nb = c->nb;
    // Morton codes with their 6 lowest bits cleared (8 bits per axis), sorted
    // in 3 passes: partner sets are exact and contacts are gathered in
    // ascending partner id, so the results do not depend on the tree, and a
    // 256-cell axis is far finer than the bodies' spacing
    sd_status st = launch_morton((const float*)lo, (const float*)hi, nb, c->domain, c->mkeys, CL_MORTON_DROP, s);
    if (st != SD_OK) return st;
    uint64_t *K = c->mkeys, *Ka = c->mkeys2;
    st = radix_sort_keys_u64(&K, &Ka, nb, 32 + CL_MORTON_DROP, 62, c->sort_tmp, c->sort_tmp_bytes, s, 0);
    if (st != SD_OK) return st;
    if (ev) SD_HIP(hipEventRecord(ev[2], s));
    st = lbvh_build(K, nb, (const float*)lo, (const float*)hi, c->left, c->right, c->parent, c->first, c->last,
                    c->rope, (float*)c->nlo, (float*)c->nhi, c->counters, &c->ctl->error, c->pnode, s);
    c->ksorted = K;
    return st;
}

// One step. ev (optional, 7 events): poses and boxes | domain+morton+sort | lbvh build |
// (empty) | (empty) | partner search + contacts + integrate. lists: what the
// step does with the partner lists (LIST_*).
sd_status clump_step(sd_clump_ctx* c, hipEvent_t* ev, int lists) {
    hipStream_t s = c->stream;
    const int nb = c->nb, par = c->cur;
    const ClumpState cs = state_of(c, c->cur), nx = state_of(c, 1 - c->cur);
    const ContactDev cd = to_dev(c->p.contact);
    sd_status st;
#define MARK(i) \
    if (ev) SD_HIP(hipEventRecord(ev[i], s))
    MARK(0);
    hipLaunchKernelGGL(k_clump_pose, dim3(div_up(nb, 256 / POSE_LANES)), dim3(256), 0, s, cs, c->i0, c->i1, c->slocal,
                       c->bfirst, c->bcount, nb, c->omega, c->sx, c->blo, c->bhi, c->ctl, par, c->boxes ? 1 : 0);
    SD_LAUNCH_CHECK();
    c->boxes = true;
    MARK(1);
    if (lists != LIST_USE) {
        st = sd_global_domain((const float*)c->blo, (const float*)c->bhi, nb, c->domain, c->dom_scratch, s);
        if (st != SD_OK) return st;
        const float4 *lo = c->blo, *hi = c->bhi;
        if (lists == LIST_BUILD) {
            hipLaunchKernelGGL(k_clump_margin, dim3(1), dim3(64), 0, s, c->ctl, par, c->size,
                               (const float*)c->domain);
            SD_LAUNCH_CHECK();
            hipLaunchKernelGGL(k_clump_inflate, dim3(div_up(nb, 256)), dim3(256), 0, s, lo, hi, nb,
                               (const ClumpCtl*)c->ctl, c->ilo, c->ihi);
            SD_LAUNCH_CHECK();
            lo = c->ilo;
            hi = c->ihi;
        }
        st = clump_tree(c, lo, hi, ev);
        if (st != SD_OK) return st;
    } else {
        MARK(2);
    }
    c->tree_last = lists == LIST_NONE;
    MARK(3);
    MARK(4);  // (partner search is part of the contact kernel)
    MARK(5);
#define CONTACTS(L)                                                                                                   \
    hipLaunchKernelGGL(k_clump_contacts<L>, dim3(div_up(nb, CL_BLOCK)), dim3(CL_BLOCK), 0, s, cs, nx, c->omega, c->i0, \
                       c->i1, c->sx, c->slocal, c->bfirst, c->bcount, nb, c->blo, c->bhi, (const float4*)c->pnode, cd,     \
                       c->ctl, par, c->lcount, c->list)
    if (lists == LIST_USE) CONTACTS(LIST_USE);
    else if (lists == LIST_BUILD) CONTACTS(LIST_BUILD);
    else CONTACTS(LIST_NONE);
#undef CONTACTS
    SD_LAUNCH_CHECK();
    MARK(6);
#undef MARK
    c->cur = 1 - c->cur;
    return SD_OK;
}

// A changed state (upload, load): no lists, and the boxes say nothing about how far bodies move.
sd_status clump_forget_lists(sd_clump_ctx* c) {
    c->plan = ListPlan();
    c->boxes = false;
    return launch_fill_u32((uint32_t*)c->ctl, 0u, sizeof(ClumpCtl) / 4, c->stream);
}

}  // namespace

extern "C" sd_status sd_clump_create(const sd_clump_params* p, sd_clump_ctx** out) {
    SD_REQUIRE(p && out, "sd_clump_create: NULL argument");
    *out = nullptr;
    sd_status st = check_contact(&p->contact);
    if (st != SD_OK) return st;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return set_error(SD_ERR_NO_DEVICE, "sd_clump_create: no HIP device");
    sd_clump_ctx* c = new sd_clump_ctx();
    c->p = *p;
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete c;
        return hip_error(e, "hipStreamCreateWithFlags", __FILE__, __LINE__);
    }
    *out = c;
    return SD_OK;
}

// Replaces the contact law / dt / gravity of an existing context (takes effect
// from the next step; the state is kept).
extern "C" sd_status sd_clump_set_params(sd_clump_ctx* c, const sd_clump_params* p) {
    SD_REQUIRE(c && p, "sd_clump_set_params: NULL argument");
    sd_status st = check_contact(&p->contact);
    if (st != SD_OK) return st;
    (void)hipStreamSynchronize(c->stream);
    c->p = *p;
    drop_clump_graphs(c);  // the contact law is a launch argument of the captured steps
    return SD_OK;
}

extern "C" sd_status sd_clump_destroy(sd_clump_ctx* c) {
    if (!c) return SD_OK;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    cfree(c);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return SD_OK;
}

// Bodies: pos4 (x, y, z, mass), vel4 (v, 0), quat4 (w, x, y, z), angvel4 (w, 0) world,
// inertia6 (body frame xx, yy, zz, xy, xz, yz), first/count sphere ranges.
// Spheres: local4 (body-frame offset from the centre of mass, radius).
// Body rows from upload arguments: P = (x, y, z, 1/m), V = (v, 0) (zero for a
// static body), Q = q, L = R I R^T w (world angular momentum), I0/I1 = the
// body-frame inverse inertia; inverse and L in double precision on the host.
sd_status sd::prepare_rigid(const char* who, int nb, const float* pos4, const float* vel4, const float* quat4,
                        const float* angvel4, const float* inertia6, float4* P, float4* V, float4* Q, float4* L,
                        float4* I0, float4* I1) {
    for (int b = 0; b < nb; ++b) {
        const float* p = pos4 + 4 * (size_t)b;
        const float m = p[3];
        if (!(m >= 0.0f)) return set_error(SD_ERR_ARG, "%s: body %d has a negative mass", who, b);
        P[b] = make_float4(p[0], p[1], p[2], m > 0.0f ? 1.0f / m : 0.0f);
        const float* v = vel4 + 4 * (size_t)b;
        V[b] = m > 0.0f ? make_float4(v[0], v[1], v[2], 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float* q = quat4 + 4 * (size_t)b;
        Q[b] = make_float4(q[0], q[1], q[2], q[3]);
        // inverse of the symmetric body inertia (double precision on the host)
        const float* I = inertia6 + 6 * (size_t)b;
        const double a = I[0], e = I[1], f = I[2], xy = I[3], xz = I[4], yz = I[5];
        const double c00 = e * f - yz * yz, c01 = xz * yz - xy * f, c02 = xy * yz - xz * e;
        const double det = a * c00 + xy * c01 + xz * c02;
        if (m > 0.0f && !(det > 0.0))
            return set_error(SD_ERR_ARG, "%s: body %d has a singular inertia tensor", who, b);
        double inv[6] = {0, 0, 0, 0, 0, 0};
        if (m > 0.0f) {
            inv[0] = c00 / det;
            inv[1] = (a * f - xz * xz) / det;
            inv[2] = (a * e - xy * xy) / det;
            inv[3] = c01 / det;
            inv[4] = c02 / det;
            inv[5] = (xz * xy - a * yz) / det;
        }
        I0[b] = make_float4((float)inv[0], (float)inv[1], (float)inv[2], (float)inv[3]);
        I1[b] = make_float4((float)inv[4], (float)inv[5], 0.0f, 0.0f);
        // L = R I R^T w (world), in double
        const float* w = angvel4 + 4 * (size_t)b;
        const double qw = q[0], qx = q[1], qy = q[2], qz = q[3];
        const double R[9] = {1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
                             2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                             2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)};
        const double Ib[9] = {a, xy, xz, xy, e, yz, xz, yz, f};
        double u[3], t[3], Lw[3];
        for (int k = 0; k < 3; ++k) u[k] = R[0 + k] * w[0] + R[3 + k] * w[1] + R[6 + k] * w[2];
        for (int k = 0; k < 3; ++k) t[k] = Ib[3 * k] * u[0] + Ib[3 * k + 1] * u[1] + Ib[3 * k + 2] * u[2];
        for (int k = 0; k < 3; ++k) Lw[k] = R[3 * k] * t[0] + R[3 * k + 1] * t[1] + R[3 * k + 2] * t[2];
        L[b] = m > 0.0f ? make_float4((float)Lw[0], (float)Lw[1], (float)Lw[2], 0.0f)
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    return SD_OK;
}

namespace {

// Body rows as the context keeps them: P = (x, y, z, 1/m), V = (v, 0),
// Q = (w, x, y, z), L = world angular momentum, I0/I1 = the body-frame inverse
// inertia (xx, yy, zz, xy) / (xz, yz, 0, 0); first/count index the sphere
// rows local4 = (body-frame offset, r).
struct ClumpRows {
    int nb = 0, ns = 0;
    std::vector<float4> P, V, Q, L, I0, I1, loc;
    std::vector<int> first, count;
    void resize(int b, int sp) {
        nb = b;
        ns = sp;
        P.resize(b);
        V.resize(b);
        Q.resize(b);
        L.resize(b);
        I0.resize(b);
        I1.resize(b);
        first.resize(b);
        count.resize(b);
        loc.resize(sp);
    }
};

// Checks the body -> sphere ranges and fills sbody (every sphere in exactly one body).
sd_status body_ranges(const char* who, int nb, const int* first, const int* count, int ns, std::vector<int>& sbody) {
    sbody.assign(ns, -1);
    for (int b = 0; b < nb; ++b) {
        if (count[b] < 1 || first[b] < 0 || first[b] + count[b] > ns)
            return set_error(SD_ERR_ARG, "%s: body %d has a bad sphere range", who, b);
        for (int k = first[b]; k < first[b] + count[b]; ++k) {
            if (sbody[k] != -1) return set_error(SD_ERR_ARG, "%s: sphere %d belongs to two bodies", who, k);
            sbody[k] = b;
        }
    }
    for (int k = 0; k < ns; ++k)
        if (sbody[k] < 0) return set_error(SD_ERR_ARG, "%s: sphere %d belongs to no body", who, k);
    return SD_OK;
}

// The rows of nb bodies from the upload arguments, written at rows[at ..].
sd_status prepare_bodies(const char* who, int nb, const float* pos4, const float* vel4, const float* quat4,
                         const float* angvel4, const float* inertia6, ClumpRows& r, int at) {
    return prepare_rigid(who, nb, pos4, vel4, quat4, angvel4, inertia6, r.P.data() + at, r.V.data() + at,
                         r.Q.data() + at, r.L.data() + at, r.I0.data() + at, r.I1.data() + at);
}

// FNV-1a 64 over the rows that stay fixed while stepping (inverse inertia,
// sphere ranges and offsets): a checkpoint is loaded only into a context
// holding the same bodies.
uint64_t static_hash(const ClumpRows& r) {
    uint64_t h = 0xcbf29ce484222325ull;
    auto mix = [&](const void* p, size_t sz) {
        const unsigned char* b = (const unsigned char*)p;
        for (size_t i = 0; i < sz; ++i) h = (h ^ b[i]) * 0x100000001b3ull;
    };
    mix(r.I0.data(), r.I0.size() * sizeof(float4));
    mix(r.I1.data(), r.I1.size() * sizeof(float4));
    mix(r.first.data(), r.first.size() * sizeof(int));
    mix(r.count.data(), r.count.size() * sizeof(int));
    mix(r.loc.data(), r.loc.size() * sizeof(float4));
    return h;
}

// (Re)allocates the context for r.nb bodies and r.ns spheres and uploads the
// rows at buffer parity 0; drops the captured graphs.
sd_status write_clump_rows(sd_clump_ctx* c, const ClumpRows& r) {
    const int nb = r.nb, ns = r.ns;
    std::vector<int> sbody;
    sd_status st = body_ranges("sd_clump", nb, r.first.data(), r.count.data(), ns, sbody);
    if (st != SD_OK) return st;
    (void)hipStreamSynchronize(c->stream);
    drop_clump_graphs(c);
    cfree(c);
    c->nb = nb;
    c->ns = ns;
#define ALLOC(ptr, cnt)                  \
    if (st == SD_OK) st = dalloc(&(ptr), (size_t)(cnt))
    for (int k = 0; k < 2; ++k) {
        ALLOC(c->pos[k], nb);
        ALLOC(c->vel[k], nb);
        ALLOC(c->quat[k], nb);
        ALLOC(c->angm[k], nb);
    }
    ALLOC(c->i0, nb);
    ALLOC(c->i1, nb);
    ALLOC(c->omega, nb);
    ALLOC(c->bfirst, nb);
    ALLOC(c->bcount, nb);
    ALLOC(c->slocal, ns);
    ALLOC(c->sx, ns);
    ALLOC(c->blo, nb);
    ALLOC(c->bhi, nb);
    ALLOC(c->domain, 8);
    ALLOC(c->dom_scratch, 256 * 6);
    ALLOC(c->mkeys, nb);
    ALLOC(c->mkeys2, nb);
    c->sort_tmp_bytes = radix_temp_bytes(nb);
    ALLOC(*(char**)&c->sort_tmp, c->sort_tmp_bytes);
    ALLOC(c->left, nb);
    ALLOC(c->right, nb);
    ALLOC(c->parent, 2 * (size_t)nb);
    ALLOC(c->first, 2 * (size_t)nb);
    ALLOC(c->last, 2 * (size_t)nb);
    ALLOC(c->rope, 2 * (size_t)nb);
    ALLOC(c->nlo, 2 * (size_t)nb);
    ALLOC(c->nhi, 2 * (size_t)nb);
    ALLOC(c->pnode, 4 * (size_t)nb);
    ALLOC(c->counters, 3 * (size_t)nb + 8);
    sd_lbvh_query_scratch_bytes(nb, &c->q_scratch_bytes);
    ALLOC(*(char**)&c->q_scratch, c->q_scratch_bytes);
    ALLOC(c->ctl, 1);
#undef ALLOC
    if (st == SD_OK) st = grow_pairs(c, 8 * nb);
    if (st != SD_OK) {
        cfree(c);
        return st;
    }
    // (97 bytes a body; bodies that fit without lists step without)
    const size_t row = (size_t)nb * sizeof(float4), list = (size_t)nb * CL_LIST * sizeof(int);
    if (hipMalloc((void**)&c->list_mem, 2 * row + list + (size_t)nb) == hipSuccess) {
        c->ilo = (float4*)c->list_mem;
        c->ihi = (float4*)(c->list_mem + row);
        c->list = (int*)(c->list_mem + 2 * row);
        c->lcount = (uint8_t*)c->list_mem + 2 * row + list;
    } else {
        (void)hipGetLastError();
        c->list_mem = nullptr;
    }
    hipStream_t s = c->stream;
    SD_HIP(hipMemcpyAsync(c->pos[0], r.P.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->vel[0], r.V.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->quat[0], r.Q.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->angm[0], r.L.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->i0, r.I0.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->i1, r.I1.data(), nb * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->bfirst, r.first.data(), nb * sizeof(int), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->bcount, r.count.data(), nb * sizeof(int), hipMemcpyHostToDevice, s));
    SD_HIP(hipMemcpyAsync(c->slocal, r.loc.data(), ns * sizeof(float4), hipMemcpyHostToDevice, s));
    SD_HIP(hipStreamSynchronize(s));
    c->cur = 0;
    c->have_tree = false;
    c->npairs = -1;
    c->static_hash = static_hash(r);
    // mean extent of a body: twice the reach of its spheres from the centre
    double size = 0.0;
    for (int b = 0; b < nb; ++b) {
        float reach = 0.0f;
        for (int k = r.first[b]; k < r.first[b] + r.count[b]; ++k) {
            const float4 l = r.loc[k];
            reach = fmaxf(reach, sqrtf(l.x * l.x + l.y * l.y + l.z * l.z) + l.w);
        }
        size += 2.0 * (double)reach;
    }
    c->size = (float)(size / nb);
    st = clump_forget_lists(c);
    if (st != SD_OK) return st;
    SD_HIP(hipStreamSynchronize(s));
    return SD_OK;
}

// The context's rows (the current buffer parity) on the host.
sd_status read_clump_rows(sd_clump_ctx* c, ClumpRows& r) {
    r.resize(c->nb, c->ns);
    const size_t b4 = (size_t)c->nb * sizeof(float4);
    hipStream_t s = c->stream;
    const int k = c->cur;
    SD_HIP(hipMemcpyAsync(r.P.data(), c->pos[k], b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.V.data(), c->vel[k], b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.Q.data(), c->quat[k], b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.L.data(), c->angm[k], b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.I0.data(), c->i0, b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.I1.data(), c->i1, b4, hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.first.data(), c->bfirst, (size_t)c->nb * sizeof(int), hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.count.data(), c->bcount, (size_t)c->nb * sizeof(int), hipMemcpyDeviceToHost, s));
    SD_HIP(hipMemcpyAsync(r.loc.data(), c->slocal, (size_t)c->ns * sizeof(float4), hipMemcpyDeviceToHost, s));
    SD_HIP(hipStreamSynchronize(s));
    return SD_OK;
}

}  // namespace

extern "C" sd_status sd_clump_upload(sd_clump_ctx* c, int nb, const float* pos4, const float* vel4,
                                     const float* quat4, const float* angvel4, const float* inertia6,
                                     const int* first, const int* count, int ns, const float* local4) {
    SD_REQUIRE(c && nb >= 1 && ns >= 1, "sd_clump_upload: bad sizes");
    SD_REQUIRE(pos4 && vel4 && quat4 && angvel4 && inertia6 && first && count && local4, "sd_clump_upload: NULL array");
    SD_REQUIRE((uint64_t)nb * (uint64_t)nb < (1ull << 62), "sd_clump_upload: too many bodies");
    std::vector<int> sbody;
    sd_status st = body_ranges("sd_clump_upload", nb, first, count, ns, sbody);
    if (st != SD_OK) return st;
    ClumpRows r;
    r.resize(nb, ns);
    st = prepare_bodies("sd_clump_upload", nb, pos4, vel4, quat4, angvel4, inertia6, r, 0);
    if (st != SD_OK) return st;
    for (int b = 0; b < nb; ++b) {
        r.first[b] = first[b];
        r.count[b] = count[b];
    }
    for (int k = 0; k < ns; ++k)
        r.loc[k] = make_float4(local4[4 * (size_t)k], local4[4 * (size_t)k + 1], local4[4 * (size_t)k + 2],
                               local4[4 * (size_t)k + 3]);
    st = write_clump_rows(c, r);
    if (st != SD_OK) return st;
    c->steps_done = 0;
    return SD_OK;
}

// Two steps from the current buffer parity, captured once per parity and kind.
static sd_status clump_graph_pair(sd_clump_ctx* c, int lists) {
    const int k = c->cur;
    if (!c->graph[k][lists]) {
        SD_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        sd_status st = clump_step(c, nullptr, lists);
        if (st == SD_OK) st = clump_step(c, nullptr, lists);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(c->stream, &g);
        c->cur = k;  // capture advanced the parity twice: back where it was
        if (st != SD_OK) {
            if (g) (void)hipGraphDestroy(g);
            return st;
        }
        SD_HIP(e);
        hipGraphExec_t ge = nullptr;
        e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
        if (e != hipSuccess) {
            (void)hipGraphDestroy(g);
            SD_HIP(e);
        }
        c->graph[k][lists] = ge;
        c->graph_obj[k][lists] = g;
    }
    SD_HIP(hipGraphLaunch(c->graph[k][lists], c->stream));
    c->tree_last = lists == LIST_NONE;
    return SD_OK;
}

// The next launch sequence of at most `left` steps.
static ListRun clump_next(sd_clump_ctx* c, int left) {
    const float largest = clump_largest(c->size);
    return c->plan.next(left, c->list_mem && c->size > 0.0f && c->plan.pays(largest), false, largest,
                        CL_MARGIN_KEPT * clump_margin(c->plan.last, c->size));
}

// What a launch sequence left: the steps that ran set the buffer parity, the
// movement says how long lists will last.
static sd_status clump_read_ctl(sd_clump_ctx* c, int cur0, int limit, bool use, int* ran) {
    ClumpCtl ctl;
    SD_HIP(hipMemcpyAsync(&ctl, c->ctl, CLUMP_CTL_READ * sizeof(int), hipMemcpyDeviceToHost, c->stream));
    SD_HIP(hipStreamSynchronize(c->stream));
    if (ctl.ran < 0 || ctl.ran > limit || (ctl.ran == 0 && ctl.given_up == 0))
        return set_error(SD_ERR_STATE, "sd_clump_step: %d of %d steps ran", ctl.ran, limit);
    *ran = ctl.ran;
    c->cur = cur0 ^ (ctl.ran & 1);
    ListReport r;
    r.ran = ctl.ran;
    r.given_up = ctl.given_up != 0;
    r.crowded = ctl.over != 0;
    r.last = ctl.last;
    r.budget = ctl.limit;
    r.used = ctl.displaced[c->cur];
    r.lost = CL_MARGIN_KEPT * ctl.margin - ctl.limit;
    c->plan.read(r, use, clump_largest(c->size));
    if (ctl.error) return set_error(SD_ERR_STATE, "sd_clump_step: malformed tree (error bits %d)", ctl.error);
    return SD_OK;
}

extern "C" sd_status sd_clump_step(sd_clump_ctx* c, int nsteps) {
    SD_REQUIRE(c && nsteps >= 0, "sd_clump_step: bad argument");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_step: no bodies uploaded");
    if (nsteps == 0) return SD_OK;
    auto run = [&](int l, int lists) -> sd_status {
        sd_status e = SD_OK;
        for (; l >= 2 && e == SD_OK; l -= 2) e = clump_graph_pair(c, lists);
        if (l > 0 && e == SD_OK) e = clump_step(c, nullptr, lists);
        return e;
    };
    int left = nsteps;
    while (left > 0) {
        sd_status st = launch_fill_u32((uint32_t*)c->ctl, 0u, 3, c->stream);  // given_up, ran, error
        if (st != SD_OK) return st;
        const int cur0 = c->cur;
        const ListRun next = clump_next(c, left);
        const bool use = next.none == 0;
        if (!use) {
            // the first step's boxes are compared with none, so never one of a captured pair
            int l = next.none;
            if (!c->boxes) {
                st = clump_step(c, nullptr, LIST_NONE);
                --l;
            }
            if (st == SD_OK) st = run(l, LIST_NONE);
        } else {
            if (next.build) st = clump_step(c, nullptr, LIST_BUILD);
            if (st == SD_OK) st = run(next.use, LIST_USE);
        }
        if (st != SD_OK) return st;
        int ran = 0;
        st = clump_read_ctl(c, cur0, left, use, &ran);
        left -= ran;
        c->steps_done += ran;
        c->have_tree = true;
        c->npairs = -1;  // the pair list of the new last step is built when asked for
        if (st != SD_OK) return st;
    }
    return SD_OK;
}

extern "C" sd_status sd_clump_profile(sd_clump_ctx* c, int nsteps, float* stage_ms, int nstages) {
    SD_REQUIRE(c && stage_ms && nstages >= 1 && nsteps >= 1, "sd_clump_profile: bad argument");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_profile: no bodies uploaded");
    const int ns = nstages < 6 ? nstages : 6;
    for (int k = 0; k < nstages; ++k) stage_ms[k] = 0.0f;
    hipEvent_t ev[7];
    for (int k = 0; k < 7; ++k) SD_HIP(hipEventCreate(&ev[k]));
    sd_status st = SD_OK;
    for (int i = 0; i < nsteps && st == SD_OK; ++i) {
        // the lists as a run would use them, the step redone if they ran out
        const int cur0 = c->cur;
        const ListRun next = clump_next(c, 1);
        const bool use = next.none == 0;
        const int lists = !use ? LIST_NONE : (next.build ? LIST_BUILD : LIST_USE);
        st = launch_fill_u32((uint32_t*)c->ctl, 0u, 3, c->stream);
        if (st == SD_OK) st = clump_step(c, ev, lists);
        if (st != SD_OK) break;
        if (hipEventSynchronize(ev[6]) != hipSuccess) {
            st = set_error(SD_ERR_HIP, "sd_clump_profile: event wait failed");
            break;
        }
        int ran = 0;
        st = clump_read_ctl(c, cur0, 1, use, &ran);
        if (st != SD_OK) break;
        if (ran == 0) {
            --i;
            continue;
        }
        for (int k = 0; k < ns; ++k) {
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
            stage_ms[k] += ms;
        }
    }
    for (int k = 0; k < 7; ++k) (void)hipEventDestroy(ev[k]);
    if (st == SD_OK) {
        c->steps_done += nsteps;
        c->have_tree = true;
        c->npairs = -1;
    }
    return st;
}

// Body state in body order: pos4 (x, y, z, 0), vel4, quat4, angmom4 (world L); any may be NULL.
extern "C" sd_status sd_clump_download(sd_clump_ctx* c, float* pos4, float* vel4, float* quat4, float* angmom4) {
    SD_REQUIRE(c, "sd_clump_download: NULL");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_download: no bodies uploaded");
    const size_t bytes = (size_t)c->nb * sizeof(float4);
    hipStream_t s = c->stream;
    if (pos4) SD_HIP(hipMemcpyAsync(pos4, c->pos[c->cur], bytes, hipMemcpyDeviceToHost, s));
    if (vel4) SD_HIP(hipMemcpyAsync(vel4, c->vel[c->cur], bytes, hipMemcpyDeviceToHost, s));
    if (quat4) SD_HIP(hipMemcpyAsync(quat4, c->quat[c->cur], bytes, hipMemcpyDeviceToHost, s));
    if (angmom4) SD_HIP(hipMemcpyAsync(angmom4, c->angm[c->cur], bytes, hipMemcpyDeviceToHost, s));
    SD_HIP(hipStreamSynchronize(s));
    if (pos4)
        for (int b = 0; b < c->nb; ++b) pos4[4 * (size_t)b + 3] = 0.0f;
    return SD_OK;
}

// Unique candidate body pairs (a < b) of the last step's broadphase.
extern "C" sd_status sd_clump_pairs(sd_clump_ctx* c, int* pairs, int capacity, int* n_pairs) {
    SD_REQUIRE(c && n_pairs, "sd_clump_pairs: NULL");
    if (!c->have_tree) return set_error(SD_ERR_STATE, "sd_clump_pairs: no step has run");
    if (c->npairs < 0) {  // query the last step's tree
        int np = 0;
        sd_status st = SD_OK;
        if (!c->tree_last) {  // a step on lists has none, one that builds them a tree of inflated boxes
            st = sd_global_domain((const float*)c->blo, (const float*)c->bhi, c->nb, c->domain, c->dom_scratch,
                                  c->stream);
            if (st == SD_OK) st = clump_tree(c, c->blo, c->bhi, nullptr);
            if (st != SD_OK) return st;
            c->tree_last = true;
        }
        st = sd_lbvh_query(c->ksorted, c->nb, c->left, c->last, c->rope, (const float*)c->nlo,
                                     (const float*)c->nhi, c->pairs, c->pair_cap, &np, &c->ctl->error, c->q_scratch,
                                     c->q_scratch_bytes, c->stream);
        if (st == SD_ERR_CAPACITY) {
            st = grow_pairs(c, np);
            if (st != SD_OK) return st;
            st = sd_lbvh_query(c->ksorted, c->nb, c->left, c->last, c->rope, (const float*)c->nlo,
                               (const float*)c->nhi, c->pairs, c->pair_cap, &np, &c->ctl->error, c->q_scratch,
                               c->q_scratch_bytes, c->stream);
        }
        if (st != SD_OK) return st;
        c->npairs = np;
    }
    *n_pairs = c->npairs;
    if (pairs && capacity > 0) {
        const int k = c->npairs < capacity ? c->npairs : capacity;
        SD_HIP(hipMemcpyAsync(pairs, c->pairs, 2 * (size_t)k * sizeof(int), hipMemcpyDeviceToHost, c->stream));
        SD_HIP(hipStreamSynchronize(c->stream));
    }
    if (c->npairs > capacity) return set_error(SD_ERR_CAPACITY, "sd_clump_pairs: %d pairs", c->npairs);
    return SD_OK;
}

// Sphere world positions (x, y, z, r) of the last pose evaluation, in sphere order.
extern "C" sd_status sd_clump_spheres(sd_clump_ctx* c, float* pos4) {
    SD_REQUIRE(c && pos4, "sd_clump_spheres: NULL");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_spheres: no bodies uploaded");
    SD_HIP(hipMemcpyAsync(pos4, c->sx, (size_t)c->ns * sizeof(float4), hipMemcpyDeviceToHost, c->stream));
    SD_HIP(hipStreamSynchronize(c->stream));
    return SD_OK;
}

// ------------------------------------------------------------------ checkpoint, add / remove

namespace {
struct ClumpStateHeader {
    uint32_t magic;
    uint32_t version;
    int32_t nb;
    int32_t ns;
    int64_t steps_done;
    uint64_t static_hash;
};
constexpr uint32_t CLUMP_MAGIC = 0x5344434Bu;  // "SDCK"

size_t clump_state_bytes(const sd_clump_ctx* c) {
    return sizeof(ClumpStateHeader) + 4 * (size_t)c->nb * sizeof(float4);
}
}  // namespace

extern "C" sd_status sd_clump_state_bytes(sd_clump_ctx* c, size_t* bytes) {
    SD_REQUIRE(c && bytes, "sd_clump_state_bytes: NULL");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_state_bytes: no bodies uploaded");
    *bytes = clump_state_bytes(c);
    return SD_OK;
}

extern "C" sd_status sd_clump_save(sd_clump_ctx* c, void* buffer, size_t bytes) {
    SD_REQUIRE(c && buffer, "sd_clump_save: NULL");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_save: no bodies uploaded");
    SD_REQUIRE(bytes >= clump_state_bytes(c), "sd_clump_save: buffer too small (%zu < %zu)", bytes,
               clump_state_bytes(c));
    ClumpStateHeader h{CLUMP_MAGIC, 1u, c->nb, c->ns, c->steps_done, c->static_hash};
    char* b = (char*)buffer;
    memcpy(b, &h, sizeof h);
    b += sizeof h;
    const size_t b4 = (size_t)c->nb * sizeof(float4);
    float4* src[4] = {c->pos[c->cur], c->vel[c->cur], c->quat[c->cur], c->angm[c->cur]};
    for (int k = 0; k < 4; ++k) {
        SD_HIP(hipMemcpyAsync(b, src[k], b4, hipMemcpyDeviceToHost, c->stream));
        b += b4;
    }
    SD_HIP(hipStreamSynchronize(c->stream));
    return SD_OK;
}

extern "C" sd_status sd_clump_load(sd_clump_ctx* c, const void* buffer, size_t bytes) {
    SD_REQUIRE(c && buffer, "sd_clump_load: NULL");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_load: upload the same bodies first");
    SD_REQUIRE(bytes >= sizeof(ClumpStateHeader), "sd_clump_load: buffer too small");
    ClumpStateHeader h;
    memcpy(&h, buffer, sizeof h);
    SD_REQUIRE(h.magic == CLUMP_MAGIC && h.version == 1u, "sd_clump_load: not a clump state buffer");
    SD_REQUIRE(h.nb == c->nb && h.ns == c->ns, "sd_clump_load: state was saved from %d bodies / %d spheres, "
               "the context holds %d / %d", h.nb, h.ns, c->nb, c->ns);
    SD_REQUIRE(h.static_hash == c->static_hash,
               "sd_clump_load: state was saved from other bodies (inertia, sphere ranges or offsets differ)");
    SD_REQUIRE(bytes >= clump_state_bytes(c), "sd_clump_load: buffer too small");
    (void)hipStreamSynchronize(c->stream);
    const char* b = (const char*)buffer + sizeof h;
    const size_t b4 = (size_t)c->nb * sizeof(float4);
    c->cur = 0;
    float4* dst[4] = {c->pos[0], c->vel[0], c->quat[0], c->angm[0]};
    for (int k = 0; k < 4; ++k) {
        SD_HIP(hipMemcpyAsync(dst[k], b, b4, hipMemcpyHostToDevice, c->stream));
        b += b4;
    }
    const sd_status st = clump_forget_lists(c);
    if (st != SD_OK) return st;
    SD_HIP(hipStreamSynchronize(c->stream));
    c->steps_done = h.steps_done;
    c->have_tree = false;
    c->npairs = -1;
    return SD_OK;
}

extern "C" sd_status sd_clump_remove_bodies(sd_clump_ctx* c, const int* ids, int count) {
    SD_REQUIRE(c, "sd_clump_remove_bodies: NULL context");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_remove_bodies: no bodies uploaded");
    SD_REQUIRE(count >= 0 && (count == 0 || ids), "sd_clump_remove_bodies: bad id list");
    if (count == 0) return SD_OK;
    std::vector<char> gone(c->nb, 0);
    for (int k = 0; k < count; ++k) {
        SD_REQUIRE(ids[k] >= 0 && ids[k] < c->nb, "sd_clump_remove_bodies: id %d out of range [0, %d)", ids[k],
                   c->nb);
        SD_REQUIRE(!gone[ids[k]], "sd_clump_remove_bodies: id %d listed twice", ids[k]);
        gone[ids[k]] = 1;
    }
    SD_REQUIRE(count < c->nb, "sd_clump_remove_bodies: removing every body (destroy the context instead)");
    (void)hipStreamSynchronize(c->stream);
    ClumpRows r, o;
    sd_status st = read_clump_rows(c, r);
    if (st != SD_OK) return st;
    int ns = 0;
    for (int b = 0; b < r.nb; ++b)
        if (!gone[b]) ns += r.count[b];
    o.resize(r.nb - count, ns);
    int j = 0, sp = 0;
    for (int b = 0; b < r.nb; ++b) {
        if (gone[b]) continue;
        o.P[j] = r.P[b];
        o.V[j] = r.V[b];
        o.Q[j] = r.Q[b];
        o.L[j] = r.L[b];
        o.I0[j] = r.I0[b];
        o.I1[j] = r.I1[b];
        o.first[j] = sp;
        o.count[j] = r.count[b];
        for (int k = 0; k < r.count[b]; ++k) o.loc[sp + k] = r.loc[r.first[b] + k];
        sp += r.count[b];
        ++j;
    }
    const long long steps = c->steps_done;
    st = write_clump_rows(c, o);
    c->steps_done = steps;
    return st;
}

extern "C" sd_status sd_clump_add_bodies(sd_clump_ctx* c, int nb, const float* pos4, const float* vel4,
                                         const float* quat4, const float* angvel4, const float* inertia6,
                                         const int* first, const int* count, int ns, const float* local4) {
    SD_REQUIRE(c, "sd_clump_add_bodies: NULL context");
    if (c->nb == 0) return set_error(SD_ERR_STATE, "sd_clump_add_bodies: no bodies uploaded (use sd_clump_upload)");
    SD_REQUIRE(nb >= 0 && ns >= 0, "sd_clump_add_bodies: bad sizes");
    if (nb == 0) return SD_OK;
    SD_REQUIRE(pos4 && vel4 && quat4 && angvel4 && inertia6 && first && count && local4,
               "sd_clump_add_bodies: NULL array");
    SD_REQUIRE((uint64_t)(c->nb + nb) * (uint64_t)(c->nb + nb) < (1ull << 62), "sd_clump_add_bodies: too many bodies");
    std::vector<int> sbody;
    sd_status st = body_ranges("sd_clump_add_bodies", nb, first, count, ns, sbody);
    if (st != SD_OK) return st;
    (void)hipStreamSynchronize(c->stream);
    ClumpRows r;
    st = read_clump_rows(c, r);
    if (st != SD_OK) return st;
    const int nb0 = r.nb, ns0 = r.ns;
    ClumpRows o = r;
    o.resize(nb0 + nb, ns0 + ns);
    st = prepare_bodies("sd_clump_add_bodies", nb, pos4, vel4, quat4, angvel4, inertia6, o, nb0);
    if (st != SD_OK) return st;
    for (int b = 0; b < nb; ++b) {
        o.first[nb0 + b] = ns0 + first[b];
        o.count[nb0 + b] = count[b];
    }
    for (int k = 0; k < ns; ++k)
        o.loc[ns0 + k] = make_float4(local4[4 * (size_t)k], local4[4 * (size_t)k + 1], local4[4 * (size_t)k + 2],
                                     local4[4 * (size_t)k + 3]);
    const long long steps = c->steps_done;
    st = write_clump_rows(c, o);
    c->steps_done = steps;
    return st;
}
