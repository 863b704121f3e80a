// aos.hip -- conversion between the reference's 108-byte particle records (Particle.h:8-31) and
// the solver's structure-of-arrays state, on the device (for akua_solver_step_device).
#include "aos.h"

#include <cstddef>

namespace akua {

namespace {

// Records in buffer order become both the logical and the physical order (lid = phys = identity).
// blockMasses: per 256 records, whether a mass differs from 1.
__global__ void k_import_aos(const AosParticle* __restrict__ in, uint32_t n, float4* X, float4* V,
                             float4* VS, float4* DP, float* dens, float* lam, uint32_t* id,
                             uint32_t* lid, uint32_t* phys, float4* color, float* size, uint32_t* blockMasses) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const AosParticle& p = in[min(i, n - 1u)];
    const float mass = p.mass;
    if (i < n) {
        X[i] = make_float4(p.position[0], p.position[1], p.position[2], mass);
        V[i] = make_float4(p.velocity[0], p.velocity[1], p.velocity[2], 0.0f);
        VS[i] = make_float4(p.new_velocity[0], p.new_velocity[1], p.new_velocity[2], 0.0f);
        DP[i] = make_float4(p.position_delta[0], p.position_delta[1], p.position_delta[2], 0.0f);
        dens[i] = p.density;
        lam[i] = p.lambda;
        id[i] = i;
        lid[i] = i;
        phys[i] = i;
        color[i] = make_float4(p.color[0], p.color[1], p.color[2], p.color[3]);
        size[i] = p.size;
    }
    const int differ = __syncthreads_or(i < n && mass != 1.0f);  // NaN differs
    if (threadIdx.x == 0) blockMasses[blockIdx.x] = differ ? 1u : 0u;
}

// Physical slot i is written to its logical position, the order of the reference's buffer.
// new_velocity is the step's velocity before the wall damping, vorticity and XSPH
// (IntegrationCUDA.cu:45), position_delta the last iteration's delta (ConstraintSolverCUDA.cu:129).
// A wave's 64 records pass through LDS and leave word by word in record order: 64 consecutive words are
// two or three records, and the records of a cell follow one another, where one record per lane touched
// 64 records' lines with every store (1M records: 71 us before, 48 now).
constexpr uint32_t kRecordWords = sizeof(AosParticle) / 4u;
constexpr int kExportBlock = 256;

__global__ __launch_bounds__(kExportBlock) void k_export_aos(AosParticle* __restrict__ out, uint32_t n, const float4* X,
                             const float4* V, const float4* VS, const float4* DP,
                             const float* dens, const float* lam, const uint32_t* id,
                             const uint32_t* lid, const float4* W, const uint32_t* hash,
                             const float4* color, const float* size) {
    __shared__ uint32_t words[kExportBlock / 64][64 * kRecordWords];
    __shared__ uint32_t to[kExportBlock / 64][64];
    const uint32_t i = blockIdx.x * kExportBlock + threadIdx.x;
    const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
    uint32_t k = n;  // n: no record
    if (i < n) {
        k = lid[i];
        const uint32_t j = id[i];
        const float4 x = X[i], v = V[i], w = W[i], c = color[j], vs = VS[i], dp = DP[i];
        const float f[21] = {x.x, x.y, x.z, v.x, v.y, v.z, x.x, x.y, x.z, vs.x, vs.y, vs.z, dp.x, dp.y, dp.z,
                             w.x, w.y, w.z, x.w, dens[i], lam[i]};
        const float g[5] = {c.x, c.y, c.z, c.w, size[j]};
        uint32_t* const r = &words[wave][lane * kRecordWords];
#pragma unroll
        for (int q = 0; q < 21; ++q) r[q] = __float_as_uint(f[q]);
        r[21] = k < n ? hash[k] : 0u;
#pragma unroll
        for (int q = 0; q < 5; ++q) r[22 + q] = __float_as_uint(g[q]);
    }
    to[wave][lane] = k;
    __syncthreads();
    uint32_t* const dst = reinterpret_cast<uint32_t*>(out);
#pragma unroll
    for (uint32_t q = 0; q < kRecordWords; ++q) {
        const uint32_t e = q * 64u + lane, r = e / kRecordWords;
        const uint32_t at = to[wave][r];
        if (at < n) dst[(size_t)at * kRecordWords + (e - r * kRecordWords)] = words[wave][e];
    }
}
static_assert(sizeof(AosParticle) == 27 * 4 && offsetof(AosParticle, hash) == 21 * 4, "the record's words above");

// One thread per slot, written to its logical position: 40 B per particle instead of the 52 B of the
// slot arrays that the host would otherwise fetch and put in order itself.
__global__ __launch_bounds__(256) void k_export_state(StateArrays out, uint32_t n, uint32_t nslots,
                                                      const SceneDev* __restrict__ scenes,
                                                      const uint32_t* __restrict__ chunkScene,
                                                      const float4* __restrict__ X, const float4* __restrict__ V,
                                                      const float* __restrict__ dens, const float* __restrict__ lam,
                                                      const uint32_t* __restrict__ id,
                                                      const uint32_t* __restrict__ lid) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nslots) return;
    const SceneDev& sc = scenes[chunkScene[p >> 8]];
    if (p >= sc.end) return;
    const uint32_t k = sc.first + (lid[p] - sc.begin);
    if (k >= n) return;  // a consistent order never produces this
    const float4 x = X[p], v = V[p];
    float* const pos = out.pos + (size_t)3u * k;
    float* const vel = out.vel + (size_t)3u * k;
    pos[0] = x.x; pos[1] = x.y; pos[2] = x.z;
    vel[0] = v.x; vel[1] = v.y; vel[2] = v.z;
    out.mass[k] = x.w;
    out.dens[k] = dens[p];
    out.lam[k] = lam[p];
    out.id[k] = id[p];
}

}  // namespace

void launch_export_state(hipStream_t st, const StateArrays& out, uint32_t n, uint32_t nslots,
                         const SceneDev* scenes, const uint32_t* chunkScene, const float4* X, const float4* V,
                         const float* dens, const float* lam, const uint32_t* id, const uint32_t* lid) {
    if (nslots)
        k_export_state<<<(nslots + 255) / 256, 256, 0, st>>>(out, n, nslots, scenes, chunkScene, X, V, dens, lam, id,
                                                             lid);
}

void launch_import_aos(hipStream_t st, const AosParticle* in, uint32_t n, float4* X, float4* V,
                       float4* VS, float4* DP, float* dens, float* lam, uint32_t* id, uint32_t* lid,
                       uint32_t* phys, float4* color, float* size, uint32_t* blockMasses) {
    if (n)
        k_import_aos<<<(n + 255) / 256, 256, 0, st>>>(in, n, X, V, VS, DP, dens, lam, id, lid, phys,
                                                      color, size, blockMasses);
}

void launch_export_aos(hipStream_t st, AosParticle* out, uint32_t n, const float4* X,
                       const float4* V, const float4* VS, const float4* DP, const float* dens,
                       const float* lam, const uint32_t* id, const uint32_t* lid, const float4* W,
                       const uint32_t* hash, const float4* color, const float* size) {
    if (n)
        k_export_aos<<<(n + kExportBlock - 1) / kExportBlock, kExportBlock, 0, st>>>(out, n, X, V, VS, DP, dens, lam, id, lid, W,
                                                      hash, color, size);
}

}  // namespace akua
