// Internal C++ interfaces shared between the translation units of
// libstardust_hip.so (not part of the C ABI).
#pragma once

#include <math.h>

#include "sd_common.hpp"

namespace sd {

// ------------------------------------------------------------------ sort
// Bytes of scratch the radix sort needs for n elements (any tile size).
size_t radix_temp_bytes(int n);
// Items per thread the sort uses for n elements when the caller passes 0.
int radix_default_items(int n);

// Stable LSD sort over key bits [begin_bit, end_bit). On return *keys (and
// *vals) point at the buffer holding the sorted data; the other buffer of each
// pair is left in *alt. items = 4, 8 or 16 (0 = default for n).
sd_status radix_sort_pairs_u32(uint32_t** keys, uint32_t** vals, uint32_t** keys_alt, uint32_t** vals_alt,
                               int n, int begin_bit, int end_bit, void* temp, size_t temp_bytes,
                               hipStream_t s, int items);
sd_status radix_sort_keys_u64(uint64_t** keys, uint64_t** keys_alt, int n, int begin_bit, int end_bit,
                              void* temp, size_t temp_bytes, hipStream_t s, int items);
// As radix_sort_keys_u64, with an odd number of passes (the result of two keys
// or more always ends in *keys_alt's original buffer).
sd_status radix_sort_keys_u64_odd(uint64_t** keys, uint64_t** keys_alt, int n, int begin_bit, int end_bit, void* temp,
                                  size_t temp_bytes, hipStream_t s, int items);
// Number of LSD passes the sort makes over a bit range.
int radix_passes(int begin_bit, int end_bit);

// ------------------------------------------------------------------ scan
// Exclusive prefix sum of n int32 values (in may equal out). scratch must
// hold scan_temp_bytes(n) bytes. If total != nullptr the grand total is
// written there (device pointer).
size_t scan_temp_bytes(int n);
sd_status exclusive_scan_i32(const int* in, int* out, int n, int* total, void* scratch, hipStream_t s);

// ------------------------------------------------------------------ grid
struct GridDev {
    float lox, loy, loz, cell;
    int nx, ny, nz;
};
inline GridDev to_dev(const sd_grid& g) {
    return GridDev{g.lo[0], g.lo[1], g.lo[2], g.cell, g.n[0], g.n[1], g.n[2]};
}
int grid_bits(const sd_grid& g);  // bits needed for the largest cell id
sd_status check_grid(const sd_grid* g);

sd_status launch_fill_u32(uint32_t* dst, uint32_t value, size_t count, hipStream_t s);
sd_status launch_copy_u32(uint32_t* dst, const uint32_t* src, size_t count, hipStream_t s);
sd_status launch_hash_keys_u64(const float4* pos4, int n, const GridDev& g, uint64_t* keys, hipStream_t s);
struct SceneDev;
struct StepCtl;
// keys[i] = (scene cbase + cell of pos4[i] in the scene grid) << 32 | i
sd_status launch_hash_keys_batch(const float4* pos4, int n, const SceneDev* scenes, const int* scene_of,
                                 uint64_t* keys, hipStream_t s);
sd_status launch_cell_ranges_u32(const uint32_t* keys, int n, int n_cells, int* ranges, hipStream_t s);
sd_status launch_cell_ranges_u64(const uint64_t* keys, int n, int n_cells, int* ranges, hipStream_t s);
// Cell starts of sorted keys: start[c] = number of keys whose cell is below c,
// c = 0 .. n_cells (n_cells + 1 entries), every entry written. Also gathers pos
// into sorted order (pos_o) with permute, sets *next_count = 0, and begins the
// step's near lists; does nothing while *skip.
sd_status launch_step_starts_u64(const uint64_t* keys, int n, int n_cells, int* start, const int* skip, bool permute,
                                 const float4* pos, float4* pos_o, int* next_count, StepCtl* ctl, int lists,
                                 float list_cell, hipStream_t s);
// perm is either u32 values (perm32) or the low halves of u64 keys (perm64).
sd_status launch_permute(const uint32_t* perm32, const uint64_t* perm64, int n, const float4* pos, const float4* vel,
                         const float4* omg, const int* ids, float4* pos_o, float4* vel_o, float4* omg_o, int* ids_o,
                         hipStream_t s);

// ------------------------------------------------------------------ contacts
struct ContactDev {
    float kn, kt, c2z, mu, dt;
    float gx, gy, gz;
    int walls;
    float wlo[3], whi[3];
    int maxc;
};
ContactDev to_dev(const sd_contact_params& c);
sd_status check_contact(const sd_contact_params* c);

// Entries past n that the sorted-position buffer of a context carries, so the
// contact kernel's batched candidate loads need no clamping.
constexpr int CONTACT_POS_PAD = 4;

// Near lists of a stepping context. A step that builds them records, for every
// sphere, the spheres within reach of a contact plus a margin sigma; the steps
// after it test only those, until the spheres may have used the margin up. The
// bound is exact: displaced sums the largest displacement of any sphere per
// step since the build (and grows by each step's before the next one), and a
// pair outside the lists stays apart while 2 displaced < sigma. A step of a
// dilute scene then reads a list entry per sphere or so instead of testing 97
// candidates, one of a packing about 7.
//
// The host says what a step does: it builds lists, then runs as many steps on
// them as the last displacement lets expect, in one launch sequence. A step
// that was to use lists that have run out is given up on the device, as a
// re-sort of too many changes is, and redone.
constexpr int LIST_CAP = 24;  // entries per sphere; a scene with a fuller sphere searches in every step
constexpr int LIST_SLOTS = 64;  // displacement maxima, a 64-byte line each: the waves' atomics spread over them
enum { LIST_USE = 0, LIST_BUILD = 1, LIST_NONE = 2 };
enum { GIVEN_UP_SORT = 1, GIVEN_UP_LIST = 2 };
// State of a context's launch sequence that the host reads back (the first
// eight words) and its kernels share.
struct StepCtl {
    int given_up;     // != 0: a step was given up, every later kernel of the sequence returns at once
    int ran;          // steps that ran
    int overflow;     // most contacts of a sphere beyond the history's capacity
    int over;         // a sphere had more neighbours than its list holds when the lists were built
    float displaced;  // infinite: no lists
    float sigma;
    float last;       // largest displacement of the step before the current one
    int pad;
    int pad2[8];
    uint32_t dmax[LIST_SLOTS * 16];  // squared displacements of the current step (float bits), slot k at 16 k
};
constexpr int STEP_CTL_READ = 8;
// The margin lasts for LIST_LIFE / 2 steps of the last step's largest
// displacement, within [LIST_MIN, LIST_MAX] cells. 40 steps spread the cost of a
// build (about twice a step without lists at most) and keep the lists short.
constexpr float LIST_LIFE = 80.0f, LIST_MIN = 0.01f, LIST_MAX = 0.08f;
// The displacement that a margin allows, of the margin: half of it, each sphere
// of a pair moving, less what rounding can take.
constexpr float LIST_KEPT = 0.49f;
inline float list_sigma(float last, float cell) { return fminf(fmaxf(LIST_LIFE * last, LIST_MIN * cell), LIST_MAX * cell); }

// Fused step kernel modes. CONTACT_FUSED_BATCH: packed u64 keys, every sphere
// takes its grid, contact law and cell-id base from its scene's SceneDev.
enum { CONTACT_FORCES = 0, CONTACT_FUSED_U64 = 1, CONTACT_FUSED_BATCH = 2 };

// One scene of a batch: its grid, its contact law, the first global cell id of
// its cells and its slot range [first, first + n) (sorted positions of a batch
// keep scenes contiguous because cell ids are scene-major).
struct SceneDev {
    GridDev g;
    ContactDev c;
    uint32_t cbase;
    int first;
    int n;
    int pad;
};

struct ContactArgs {
    const float4* pos;  // sorted state; positions only where a sphere searches (fused modes)
    const float4* pos_rows;  // fused modes: positions in the previous order, as vel, omg and ids
    const float4* vel;
    const float4* omg;
    const int* ids;
    int n;
    GridDev g;
    const int* ranges;      // CONTACT_FORCES: (start, end) per cell, empty cells (0, 0)
    const int* cell_start;  // fused modes: first sorted position of every cell (n_cells + 1 entries)
    ContactDev c;
    // old order: either an int array or packed u64 keys
    const int* old_slot_i32;
    const uint64_t* old_slot_u64;
    const int* hcount_old;
    const float4* hist_old;
    int* hcount_new;
    float4* hist_new;
    int* overflow;       // receives max contacts seen when > capacity
    // CONTACT_FORCES outputs
    float4* force;
    float4* torque;
    // fused outputs: integrated state + next keys
    float4* pos_o;
    float4* vel_o;
    float4* omg_o;
    int* ids_o;
    uint64_t* keys_o64;
    // fused u64 modes: spheres whose cell changed this step, appended as
    // (new key, old key) while *mcount < mcap (nullable: not recorded)
    int* mcount;
    uint64_t* mnew;
    uint64_t* mold;
    int mcap;
    StepCtl* ctl;  // fused modes
    // CONTACT_FUSED_BATCH: scene table and scene of every slot
    const SceneDev* scenes;
    const int* scene_of;
    // CONTACT_FUSED_BATCH: the waves (64 consecutive slots from a multiple of
    // 64) whose slots span more than one scene, n_straddle of them. The main
    // launch leaves them out (its waves take their scene's parameters in scalar
    // registers); launch_contacts_straddle runs them with per-lane parameters.
    const int* straddle;
    int n_straddle;
    // fused modes: near lists (list_new NULL: the context has none; entry k of
    // slot s at k * n + s; the old ones in the previous step's order, with
    // newpos[old position] = position), what the step does with them (LIST_*),
    // and the largest radius (per scene in batch mode)
    int lists;
    const uint8_t* lcount_old;
    const int* list_old;
    uint8_t* lcount_new;
    int* list_new;
    const int* newpos;
    float rmax;
    const float* scene_rmax;
};
sd_status launch_contacts(int mode, const ContactArgs& a, hipStream_t s, int block);
// Persistent form of the fused u64 / batch step kernel (same results): a
// grid of resident blocks claiming runs of 64-slot tiles from one counter per
// XCD (counters: 512 ints, cleared here by a fill kernel) until every tile is
// done.
sd_status launch_contacts_persistent(int mode, const ContactArgs& a, hipStream_t s, int block, int* counters);
sd_status launch_contacts_straddle(const ContactArgs& a, hipStream_t s);

// Sorted order of the next step's u64 keys from the previous sorted order and
// the spheres that changed cell (see sd_resort.hip): writes the sorted keys to
// keys_out and the positions in that order to posB, turns cell_start (the
// previous order's cell starts, n_cells + 1 entries) into the new order's and
// sets *next_count = 0. With *mcount > cap (= resort_cap(n)) it gives the step up instead
// (ctl->given_up).
// Most changed cells a re-sort takes: 1,024, and one sphere in 256 of larger
// scenes up to 16,384. Ranking the movers grows with their square and the
// radix sort it saves with n: at 4,194,304 spheres a re-sort of 1,000 movers
// takes 38 us and the full sort with its cell starts 147; at 250,007 spheres 12
// and 41. A fixed 1,024 sent a 4,194,304-sphere column whose spheres move at 0.5 m/s
// to the full sort every few steps.
inline int resort_cap(int n) { return n / 256 < 1024 ? 1024 : (n / 256 > 16384 ? 16384 : n / 256); }
// sd_lbvh_build, and with pnode (2 per node) also the packed tree of a
// stackless walk: (box low corner, left child or leaf index), (box high corner, rope)
sd_status lbvh_build(const uint64_t* sorted_keys, int n, const float* lo4, const float* hi4, int* left, int* right,
                     int* parent, int* first, int* last, int* rope, float* node_lo4, float* node_hi4, int* counters,
                     int* error, float4* pnode, hipStream_t s);
// keys[i] = (morton30 of box i's centroid with its drop_bits lowest bits cleared) << 32 | i
sd_status launch_morton(const float* lo4, const float* hi4, int n, const float* domain6, uint64_t* keys,
                        int drop_bits, hipStream_t s);
sd_status launch_resort_u64(const int* mcount, int cap, const uint64_t* mnew, const uint64_t* mold, uint64_t* msorted_new,
                            uint64_t* msorted_old, const uint64_t* keys, int n, int* cell_start, int n_cells,
                            const float4* pos_state, float4* posB, uint64_t* keys_out, int* next_count,
                            StepCtl* ctl, int* newpos, int lists, float list_cell, hipStream_t s);
sd_status launch_integrate(float4* pos, float4* vel, float4* omg, const float4* f, const float4* t, int n,
                           const ContactDev& c, hipStream_t s);

// Rigid-body rows from upload arguments (pos4 = (x, y, z, mass), mass 0 =
// static; quat4 = (w, x, y, z); angvel4 world; inertia6 = (xx, yy, zz, xy, xz,
// yz) body frame): P = (x, y, z, 1/m), V, Q, L = world angular momentum,
// I0/I1 = body-frame inverse inertia (xx, yy, zz, xy) / (xz, yz, 0, 0).
sd_status prepare_rigid(const char* who, int nb, const float* pos4, const float* vel4, const float* quat4,
                        const float* angvel4, const float* inertia6, float4* P, float4* V, float4* Q, float4* L,
                        float4* I0, float4* I1);

// Rigid-body context (sd_hull_ctx, sd_hullbody.hip): one step enqueued on s
// with no host synchronisation; device errors of the steps since the last
// check; accessors used by a batch context that steps the bodies with its
// scenes. A step is two parts: the forces, which write nothing that outlives the
// step, and the move, which with *given_up (nullable) leaves the bodies as they
// are.
sd_status hull_enqueue_step(sd_hull_ctx* c, hipStream_t s);
sd_status hull_enqueue_forces(sd_hull_ctx* c, hipStream_t s);
sd_status hull_enqueue_move(sd_hull_ctx* c, hipStream_t s, const int* given_up);
sd_status hull_check_errors(sd_hull_ctx* c);
int hull_body_count(const sd_hull_ctx* c);
// Changes whenever the context's step changes (upload, parameters, warm start).
long long hull_generation(const sd_hull_ctx* c);
float hull_dt(const sd_hull_ctx* c);
void hull_count_steps(sd_hull_ctx* c, int nsteps);

// ------------------------------------------------------------------ hull narrowphase, enqueued only
// Hull boxes (pos4 = centre and sphere radius, quat4 = (w, x, y, z)).
sd_status launch_hull_aabbs(const float4* pos4, const float4* quat4, const int* vstart, const int* nv,
                            const float4* verts4, int n, float4* lo4, float4* hi4, hipStream_t s);
// sd_sap_pairs_batched without its host read-back: *total_out points at the
// device pair count (may exceed capacity; pairs past capacity are not
// written), *error_out at the device error bits of the scene ranges.
sd_status enqueue_sap_batched(const float4* lo4, const float4* hi4, int n, const int* scene_of,
                              const int* scene_first, int nscenes, int* pairs, int capacity, int** total_out,
                              int** error_out, void* scratch, size_t scratch_bytes, hipStream_t s);
// Cold GJK/EPA (as sd_gjk with no warm start) of the first min(*dcount,
// capacity) pairs; launches sized to capacity, scratch of
// gjk_cold_scratch_bytes(capacity) bytes.
size_t gjk_cold_scratch_bytes(int capacity);
sd_status enqueue_gjk_cold(const int* pairs, int capacity, const int* dcount, const float4* pos4,
                           const float4* quat4, const int* vstart, const int* nv, const float4* verts4, int n_hulls,
                           int n_verts, int max_iter, float near_margin, float* sep, float* normal3, int* flags,
                           int* iters, void* scratch, hipStream_t s);
// Warm-started GJK/EPA (as sd_gjk with warm_dir3) of the first min(*dcount,
// capacity) pairs, the rejected ones redone cold; same scratch.
sd_status enqueue_gjk_warm(const int* pairs, int capacity, const int* dcount, const float4* pos4,
                           const float4* quat4, const int* vstart, const int* nv, const float4* verts4, int n_hulls,
                           int n_verts, const float* warm_dir3, int warm_budget, int max_iter, float near_margin,
                           float* sep, float* normal3, int* flags, int* iters, void* scratch, hipStream_t s);

// ------------------------------------------------------------------ learned warm start, enqueued only
// sd_hull_descriptors on a stream (desc7: 7 floats per hull).
sd_status launch_hull_descriptors(const float4* pos4, const int* vstart, const int* nv, const float4* verts4, int n,
                                  float* desc7, hipStream_t s);
// Features (X: 22 floats per pair) and BF16 inference of the network packed
// by sd_mlp_pack_bf16 for the first min(*dcount, capacity) pairs: world
// directions (A -> B) in out_dir3.
sd_status enqueue_warm_dirs(const int* pairs, int capacity, const int* dcount, const float4* pos4,
                            const float4* quat4, const float* desc7, float* X, const void* packed, float* out_dir3,
                            hipStream_t s);

}  // namespace sd
