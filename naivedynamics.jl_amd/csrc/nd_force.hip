// nd_force.hip -- forces over an explicit pair list: force_lennardjones!,
// force_coulomb!, sum_forces! (src/Forces.jl:15-74).
//
// The reference's arithmetic in Forces.jl is not physical (scalar distance
// broadcast to x/y/z, hard-coded eps=-1e10, sigma=1e-4, no Newton's third
// law); these kernels keep the entry points and compute the textbook forces
//   LJ:      F_i = 24 eps / r^2 [2 (s/r)^12 - (s/r)^6] r_ij,  F_j = -F_i
//   Coulomb: F_i = k q_i q_j r_ij / r^3,                       F_j = -F_i
// with r_ij = x_i - x_j for every listed pair inside the cutoff.  One lane per
// pair.  Both atoms' force components are summed as 64-bit integers in units
// of 2^-32 (integer addition is associative, so the result does not depend on
// the order in which lanes add, and the unit is finer than FP32's at every
// force above 2^-9); the pair energy is summed per workgroup in FP64 and the
// workgroup sums are added in index order by one workgroup.  Every pair index
// is checked against [0, n): a pair outside it is skipped and reported.
#include <algorithm>

#include "nd_internal.hpp"

namespace {

constexpr double kFixScale = 4294967296.0;          // 2^32 units per force unit
constexpr double kFixLimit = 1073741824.0;          // |per-pair component| < 2^30
enum : int32_t { kBadIndex = 1, kFixRange = 2 };

__device__ __forceinline__ double block_sum(double v, double *sh) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += sh[k];
    return s;
}

// A force component in fixed point; false (and a status bit) outside the range.
__device__ __forceinline__ bool to_units(double f, int32_t *status, unsigned long long &q) {
    if (!(fabs(f) < kFixLimit)) {  // also catches NaN
        atomicOr(status, kFixRange);
        return false;
    }
    q = (unsigned long long)__double2ll_rn(f * kFixScale);
    return true;
}

// Atoms a workgroup sums in LDS before it adds them to memory: a hash table of
// kSlots (atom, three 64-bit sums), 28 bytes a slot, 112 KB of a CU's 160 KB.
// Atomics on memory are what bounds this kernel (a 64-bit atomic from 256 CUs
// lands at ~19 per ns whatever its locality), and a pair list names the same
// atoms again and again: a list in the order of a search repeats each i over
// its neighbours and each j over the queries near it, so 18,800 consecutive
// pairs (1/256 of the list of 131,072 liquid atoms) name about 1,100 atoms.
// Six atomics per pair in memory took 1,098 us there, this takes 84.  An atom
// that finds no slot in kProbes places is added in memory, so a list in any
// order gives the same sums.
constexpr int kForceThreads = 1024;
constexpr int kSlotBits = 12, kSlots = 1 << kSlotBits, kProbes = 16;
constexpr size_t kForceLds = (size_t)kSlots * (3 * sizeof(unsigned long long) + sizeof(int32_t));

__global__ void __launch_bounds__(nd::kBlock)
k_force_clear(unsigned long long *__restrict__ acc, int64_t n3, int32_t *__restrict__ status) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k < n3) acc[k] = 0ull;
    if (k == 0) *status = 0;
}

template <int KIND>  // 0: Lennard-Jones, 1: Coulomb
__global__ void __launch_bounds__(kForceThreads)
k_pair_force(unsigned long long *__restrict__ acc, const nd_pair *__restrict__ pairs, int64_t npairs,
             int64_t per_block, const float *__restrict__ xyz, const float *__restrict__ charge, int32_t n,
             float eps, float sigma2, float rc2, float kc, float shift, double *__restrict__ partials,
             int32_t *__restrict__ status) {
    __shared__ double sh[kForceThreads / 64];
    extern __shared__ __align__(16) unsigned long long s_sum[];  // [3][kSlots], then the atoms
    int32_t *s_key = reinterpret_cast<int32_t *>(s_sum + 3 * kSlots);
    for (int t = threadIdx.x; t < 3 * kSlots; t += kForceThreads) s_sum[t] = 0ull;
    for (int t = threadIdx.x; t < kSlots; t += kForceThreads) s_key[t] = -1;
    __syncthreads();
    // slot of atom a (claimed if new), or -1
    auto slot_of = [&](int32_t a) -> int32_t {
        uint32_t h = ((uint32_t)a * 2654435761u) >> (32 - kSlotBits);
        for (int p = 0; p < kProbes; ++p) {
            int32_t k = __hip_atomic_load(&s_key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (k == -1) {
                k = atomicCAS(&s_key[h], -1, a);
                if (k == -1) return (int32_t)h;
            }
            if (k == a) return (int32_t)h;
            h = (h + 1) & (kSlots - 1);
        }
        return -1;
    };
    auto add = [&](int32_t slot, int32_t a, int c, unsigned long long q) {
        if (slot >= 0) atomicAdd(&s_sum[c * kSlots + slot], q);
        else atomicAdd(&acc[3 * (int64_t)a + c], q);
    };
    const int64_t k0 = blockIdx.x * per_block, k1 = min(k0 + per_block, npairs);
    double e = 0.0;
    for (int64_t k = k0 + threadIdx.x; k < k1; k += kForceThreads) {
        const int32_t i = pairs[k].i, j = pairs[k].j;
        if ((uint32_t)i >= (uint32_t)n || (uint32_t)j >= (uint32_t)n) {
            atomicOr(status, kBadIndex);
            continue;
        }
        const float dx = xyz[3 * (int64_t)i] - xyz[3 * (int64_t)j];
        const float dy = xyz[3 * (int64_t)i + 1] - xyz[3 * (int64_t)j + 1];
        const float dz = xyz[3 * (int64_t)i + 2] - xyz[3 * (int64_t)j + 2];
        const float r2 = dx * dx + dy * dy + dz * dz;
        if (!(r2 < rc2)) continue;
        float fs;
        const float ir2 = 1.0f / r2;
        if (KIND == 0) {
            const float sr2 = sigma2 * ir2;
            const float sr6 = sr2 * sr2 * sr2;
            fs = 24.0f * eps * ir2 * sr6 * (2.0f * sr6 - 1.0f);
            e += (double)(4.0f * eps * sr6 * (sr6 - 1.0f)) - (double)shift;
        } else {
            const float qq = kc * charge[i] * charge[j];
            const float ir = sqrtf(ir2);
            fs = qq * ir * ir2;
            e += (double)(qq * ir) - (double)(qq * shift);
        }
        const double f[3] = {(double)(fs * dx), (double)(fs * dy), (double)(fs * dz)};
        const int32_t si = slot_of(i), sj = slot_of(j);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            unsigned long long q;
            if (!to_units(f[c], status, q)) continue;
            add(si, i, c, q);
            add(sj, j, c, 0ull - q);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kSlots; t += kForceThreads) {
        const int32_t a = s_key[t];
        if (a < 0) continue;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const unsigned long long q = s_sum[c * kSlots + t];
            if (q != 0ull) atomicAdd(&acc[3 * (int64_t)a + c], q);
        }
    }
    const double s = block_sum(e, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// What the host waits for: the pair energy and the status word.
struct ForceResult {
    double energy;
    int32_t status;
};

// Fixed point to FP32; the first workgroup also adds the workgroup energies in
// a fixed order and hands the result to the host.
__global__ void __launch_bounds__(nd::kBlock)
k_force_finish(float *__restrict__ force, const unsigned long long *__restrict__ acc, int64_t n3,
               const double *__restrict__ partials, int64_t m, const int32_t *__restrict__ status,
               ForceResult *__restrict__ res) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k < n3) force[k] = (float)((double)(long long)acc[k] * (1.0 / kFixScale));
    if (blockIdx.x != 0) return;
    __shared__ double sh[nd::kBlock / 64];
    double v = 0.0;
    for (int64_t t = threadIdx.x; t < m; t += blockDim.x) v += partials[t];
    const double s = block_sum(v, sh);
    if (threadIdx.x == 0) {
        res->energy = s;
        res->status = *status;
    }
}

__global__ void __launch_bounds__(nd::kBlock)
k_sum3(float *__restrict__ out, const float *__restrict__ a, const float *__restrict__ b,
       int64_t n3) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k < n3) out[k] = a[k] + b[k];
}

template <int KIND>
void run_pair_force(nd_ctx *ctx, float *d_force, const nd_pair *d_pairs, int64_t npairs,
                    const float *d_xyz, const float *d_charge, int32_t n,
                    const nd_force_params *p, double *h_energy) {
    ND_HIP(hipSetDevice(ctx->device));
    const int64_t n3 = 3 * (int64_t)n;
    // one workgroup per CU (its table takes most of the CU's LDS), each with
    // one run of the list: the longer the run, the fewer sums leave LDS; a
    // short list keeps a pair per thread.  A call over the list of 131,072 /
    // 262,144 / 524,288 / 1,048,576 liquid atoms takes 100 / 166 / 416 / 2,964 us
    // (atomics on memory 1,151 / 2,088 / 4,517 / 9,034): up to 524,288 a run's
    // atoms (some 3,600) mostly fit the table, at 1,048,576 (6,000) those left over pay
    // for their probes and go to memory.  The pairs of 131,072 atoms in random
    // order, which do so almost always, take 873 (932).
    const int64_t per = std::max<int64_t>((npairs + 255) / 256, kForceThreads);
    const int64_t nblk = (npairs + per - 1) / per;
    ctx->force_acc.reserve(sizeof(unsigned long long) * (size_t)(n3 > 0 ? n3 : 1));
    ctx->force_part.reserve(sizeof(double) * 256);
    unsigned long long *acc = ctx->force_acc.as<unsigned long long>();
    double *part = ctx->force_part.as<double>();
    int32_t *status = ctx->status.as<int32_t>();
    ForceResult *res = nd::host_result<ForceResult>(ctx);
    ND_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_pair_force<KIND>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kForceLds));
    const unsigned gn = nd::grid_for(n3 > 0 ? n3 : 1);
    k_force_clear<<<gn, nd::kBlock, 0, ctx->stream>>>(acc, n3, status);
    const float rc = KIND == 0 ? p->rc : p->rc_coul;
    float shift = 0.0f;
    if (KIND == 0 && p->shift_lj) {
        const float c2 = p->sigma * p->sigma / (rc * rc), c6 = c2 * c2 * c2;
        shift = 4.0f * p->eps * c6 * (c6 - 1.0f);
    }
    if (KIND == 1 && p->shift_coul) shift = 1.0f / rc;
    if (npairs > 0)
        k_pair_force<KIND><<<(unsigned)nblk, kForceThreads, kForceLds, ctx->stream>>>(
            acc, d_pairs, npairs, per, d_xyz, d_charge, n, p->eps, p->sigma * p->sigma, rc * rc, p->k_coul,
            shift, part, status);
    k_force_finish<<<gn, nd::kBlock, 0, ctx->stream>>>(d_force, acc, n3, part, nblk, status, res);
    ND_HIP(hipGetLastError());
    ND_HIP(hipStreamSynchronize(ctx->stream));
    const double e = res->energy;
    const int32_t st = res->status;
    if (st) nd::clear_status(ctx);
    if (st & kBadIndex) throw nd::Error(ND_ERR_ARG, "pair index outside [0, n)");
    if (st & kFixRange) throw nd::Error(ND_ERR_DOMAIN, "pair force outside the summation range (|F| >= 2^30)");
    if (h_energy) *h_energy = e;
}

}  // namespace

extern "C" {

int nd_force_lennardjones(nd_ctx *ctx, float *d_force, const nd_pair *d_pairs, int64_t npairs,
                          const float *d_xyz, int32_t n, const nd_force_params *p,
                          double *h_energy) {
    ND_API_BEGIN
    ND_REQUIRE(ctx && d_force && d_xyz && p && n >= 0 && npairs >= 0 && (d_pairs || npairs == 0),
               "force_lennardjones!: bad argument");
    run_pair_force<0>(ctx, d_force, d_pairs, npairs, d_xyz, nullptr, n, p, h_energy);
    ND_API_END(ctx)
}

int nd_force_coulomb(nd_ctx *ctx, float *d_force, const nd_pair *d_pairs, int64_t npairs,
                     const float *d_xyz, const float *d_charge, int32_t n,
                     const nd_force_params *p, double *h_energy) {
    ND_API_BEGIN
    ND_REQUIRE(ctx && d_force && d_xyz && d_charge && p && n >= 0 && npairs >= 0 &&
                   (d_pairs || npairs == 0),
               "force_coulomb!: bad argument");
    run_pair_force<1>(ctx, d_force, d_pairs, npairs, d_xyz, d_charge, n, p, h_energy);
    ND_API_END(ctx)
}

int nd_sum_forces(nd_ctx *ctx, float *d_force, const float *d_f1, const float *d_f2, int32_t n) {
    ND_API_BEGIN
    ND_REQUIRE(ctx && d_force && d_f1 && d_f2 && n >= 0, "sum_forces!: bad argument");
    ND_HIP(hipSetDevice(ctx->device));
    const int64_t n3 = 3 * (int64_t)n;
    if (n3 > 0) {
        k_sum3<<<nd::grid_for(n3), nd::kBlock, 0, ctx->stream>>>(d_force, d_f1, d_f2, n3);
        ND_HIP(hipGetLastError());
    }
    ND_HIP(hipStreamSynchronize(ctx->stream));
    ND_API_END(ctx)
}

}  // extern "C"
