// Kernels and drivers of the state read-back (sd_readback.hpp). Replaces the
// position read-back of the reference's GL interop path
// (src/engine/engine.cpp:36-62) for host callers.
#include <string.h>

#include "sd_readback.hpp"

namespace sd {

void stage_release(HostStage& st) {
    if (st.p) (void)hipHostFree(st.p);
    st.p = nullptr;
    st.bytes = 0;
}

sd_status stage_reserve(HostStage& st, size_t bytes) {
    if (st.bytes >= bytes) return SD_OK;
    stage_release(st);
    SD_HIP(hipHostMalloc((void**)&st.p, bytes, hipHostMallocDefault));
    st.bytes = bytes;
    return SD_OK;
}

// inv[ids[s]] = s; *bad = 1 for an id outside [0, n).
__global__ __launch_bounds__(256) void k_inverse_ids(const int* __restrict__ ids, int n, int* __restrict__ inv,
                                                     int* __restrict__ bad) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int i = ids[s];
    if ((unsigned)i < (unsigned)n) inv[i] = s;
    else *bad = 1;
}

struct SoaOut {
    float* p[9];
};

// Ids i0 .. i0 + m - 1 from their slots' rows into arrays of their own (pinned
// host memory). Gathers 16-byte rows through inv and stores 256 bytes a wave
// and array; the host link bounds it.
__global__ __launch_bounds__(256) void k_gather_soa(const float4* __restrict__ pos, const float4* __restrict__ vel,
                                                    const float4* __restrict__ omg, const int* __restrict__ inv,
                                                    int n, int i0, int m, SoaOut o) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m) return;
    const int s = inv[i0 + k];
    if ((unsigned)s >= (unsigned)n) return;  // (an id that no slot has)
    if (o.p[0] || o.p[1] || o.p[2]) {
        const float4 r = pos[s];
        if (o.p[0]) o.p[0][k] = r.x;
        if (o.p[1]) o.p[1][k] = r.y;
        if (o.p[2]) o.p[2][k] = r.z;
    }
    if (o.p[3] || o.p[4] || o.p[5]) {
        const float4 r = vel[s];
        if (o.p[3]) o.p[3][k] = r.x;
        if (o.p[4]) o.p[4][k] = r.y;
        if (o.p[5]) o.p[5][k] = r.z;
    }
    if (o.p[6] || o.p[7] || o.p[8]) {
        const float4 r = omg[s];
        if (o.p[6]) o.p[6][k] = r.x;
        if (o.p[7]) o.p[7][k] = r.y;
        if (o.p[8]) o.p[8][k] = r.z;
    }
}

// Rows per chunk: about 1 MB of slot, so that the staging stays near 14 MB and
// a chunk's transfer (20 us) covers its launch. Whole sphere states into arrays
// in use (pages touched for the first time: 4,194,304 spheres 111 -> 12 ms):
// 4,194,304 spheres 96 -> 4.6 ms (33 GB/s; the link does 56), 250,007 4.6 -> 0.40 ms,
// 65,536 0.55 -> 0.11 ms, 1,000 0.09 -> 0.03 ms, against copies of the rows to
// pageable memory and a scatter by id on the host.
constexpr int SPHERE_CHUNK = 32768;

sd_status readback_spheres(HostStage& st, const float4* pos, const float4* vel, const float4* omg, const int* ids,
                           int n, int* inv, float* const out[9], hipStream_t s) {
    std::lock_guard<std::mutex> turn(st.lock);
    int want = 0;
    for (int j = 0; j < 9; ++j) want += out[j] != nullptr;
    const int per = std::min(n, SPHERE_CHUNK);
    const size_t lane = ((size_t)per * sizeof(float) + 255) & ~(size_t)255;
    const size_t slot = std::max<size_t>((size_t)want * lane, 256);
    // the flag lies behind the slots: reserve them together
    const int chunks = div_up(n, per);
    const int T = chunks == 1 ? 1 : std::min(READBACK_THREADS, (chunks + 1) / 2);
    const size_t flag_at = slot * (chunks == 1 ? 1 : 2 * (size_t)T);
    sd_status e = stage_reserve(st, flag_at + 256);
    if (e != SD_OK) return e;
    volatile int* const bad = (volatile int*)(st.p + flag_at);
    *bad = 0;
    hipLaunchKernelGGL(k_inverse_ids, dim3(div_up(n, 256)), dim3(256), 0, s, ids, n, inv, (int*)bad);
    SD_LAUNCH_CHECK();
    if (want) {
        auto fill = [=](int c, char* p, hipStream_t str) -> sd_status {
            const int i0 = c * per, m = std::min(per, n - i0);
            SoaOut o;
            char* q = p;
            for (int j = 0; j < 9; ++j) {
                o.p[j] = out[j] ? (float*)q : nullptr;
                if (out[j]) q += lane;
            }
            hipLaunchKernelGGL(k_gather_soa, dim3(div_up(m, 256)), dim3(256), 0, str, pos, vel, omg, (const int*)inv,
                               n, i0, m, o);
            SD_LAUNCH_CHECK();
            return SD_OK;
        };
        auto drain = [=](int c, const char* p) {
            const int i0 = c * per, m = std::min(per, n - i0);
            const char* q = p;
            for (int j = 0; j < 9; ++j) {
                if (!out[j]) continue;
                memcpy(out[j] + i0, q, (size_t)m * sizeof(float));
                q += lane;
            }
        };
        e = staged_chunks(st, chunks, slot, s, fill, drain);
        if (e != SD_OK) return e;
    } else {
        SD_HIP(hipStreamSynchronize(s));
    }
    if (*bad) return set_error(SD_ERR_STATE, "sd_ctx_download_spheres: corrupt id");
    return SD_OK;
}

}  // namespace sd
