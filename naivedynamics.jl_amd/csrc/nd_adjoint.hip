// nd_adjoint.hip -- differentiable velocity Verlet with a hand-written adjoint.
//
// Forward model (one system, unit masses, no walls):
//   v_h = v_k + c F(x_k),  x_{k+1} = x_k + dt v_h,  v_{k+1} = v_h + c F(x_{k+1}),  c = dt / 2
// with shifted-force Lennard-Jones and shifted-force Coulomb pair forces
//   F_ij = s(r) r_ij,  s(r) = (F(r) - F(rc)) / r   (F(r) = -dU/dr)
// so every force goes to zero continuously at its cutoff.  The loss is
//   L = sum_b (g_b - t_b)^2,  g_b = norm_b sum_{i<j} K(r_ij - r_b),
//   K(d) = (1 - (d/h)^2)^3 for |d| < h (zero outside), r_b = (b + 1/2) dr,
// a smoothed radial distribution of the final frame against a target t.
//
// Reverse sweep.  With lambda_x, lambda_v the adjoints of x_{k+1}, v_{k+1}:
//   lambda_h = lambda_v + dt lambda_x;  lambda_v <- lambda_h
//   a = w_k lambda_h  (w_k = 2c for 0 < k, c for k = 0)
//   lambda_x <- lambda_x + J(x_k) a,   theta_bar += (dF(x_k)/dtheta)^T a
// J = dF/dx is symmetric, so the two Jacobian terms of a step that meet at
// x_k (from v_{k+1} = v_h + c F(x_{k+1}) of step k-1 and v_h = v_k + c F(x_k)
// of step k) merge into one Hessian-vector product per step.  Per pair,
//   M_ij = s I + (s'(r)/r) r_ij r_ij^T,  (J a)_i = sum_j M_ij (a_i - a_j).
// The forward pass keeps (x, v) every checkpoint_every steps, and of its last
// segment every position, list and order; the sweep walks that segment
// backwards at once and recomputes the earlier ones forward from their
// checkpoints first.  Pair lists (radius max(cutoffs, rdf range) + skin) are
// rebuilt at the same steps (multiples of rebuild_every) in the forward and
// the recompute.
//
// Atoms are kept in the order of the last list build, which is the order of
// the cells (side >= list radius) it searches: a neighbour gather then reads
// aligned records (position, and in FP64 the charge) that lie near each other,
// and the build needs no tree.  Systems whose clusters lie far apart take cells
// that do not depend on the extent (BinGrid's lines).  kRowLanes lanes share an atom's row of the list:
// at N = 32,768 one lane per atom leaves two waves per CU, and a row is a chain
// of dependent loads.  One launch makes a step: the pair sums of x_k, the half
// kick that ends step k - 1 and the half kick and drift of step k; in the
// reverse sweep the Hessian-vector product and the next step's lambda_h and a.
// Per step of the forward pass (FP64, 32,768 atoms) the launches of a force
// (21.8 us), kick (4.1) and kick-drift (3.0) kernel with four lanes per row
// became one (11.5), of a vector (4.9) and a Hessian-product (35.7) kernel one
// (16.7); per list build a key, sort, tree and walk of 21 launches (250 us) and
// a host synchronisation became seven launches (60 us) and none.  FP64 VALU
// issue bounds both step kernels.
//
// Forces are summed in 2^-40 fixed point: the sum does not depend on the
// order within a row or of the atoms, which the build leaves unspecified, so
// the recompute reproduces the forward trajectory bit for bit in both
// precisions.  The reverse sweep sums in FP64.
//
// No reference counterpart: NaiveDynamics.jl has no gradients.  This is the
// differentiation form of the simulate! hot path (Simulator.jl:154-256).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "nd_internal.hpp"

namespace {

constexpr double kFix = 1099511627776.0;  // 2^40
constexpr double kInvFix = 1.0 / 1099511627776.0;

struct AdjP {
    int32_t n, nbins;
    double eps, sigma, rc, rc2, kc, rcc, rcc2, dt, c;
    double sig2, inv_eps, inv_sigma, inv_rcc2;
    double flj_rc;   // F_LJ(rc)
    double glj_rc;   // dF_LJ/dsigma at rc
    double rmax, h, dr;
};

// F_LJ(r) = 24 eps (2 sigma^12 / r^13 - sigma^6 / r^7)
__host__ __device__ inline double lj_F(double r, double eps, double sigma) {
    const double sr = sigma / r, sr6 = sr * sr * sr * sr * sr * sr;
    return 24.0 * eps * (2.0 * sr6 * sr6 - sr6) / r;
}
// dF_LJ/dsigma = 24 eps (24 sigma^11 / r^13 - 6 sigma^5 / r^7)
__host__ __device__ inline double lj_G(double r, double eps, double sigma) {
    const double sr = sigma / r, sr6 = sr * sr * sr * sr * sr * sr;
    return 24.0 * eps * (24.0 * sr6 * sr6 - 6.0 * sr6) / (r * sigma);
}

// 1 / sqrt(x) in FP64 to its last place or so: the hardware's estimate (2^-23
// or better) and one cubically converging step (Halley's).  A division and a
// square root take some 25 instructions, this seven, and its square is 1 / x.
__device__ __forceinline__ double rsqrt64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// s(r) of the forward force in precision T (LJ + Coulomb, both shifted).  FP64
// takes one inverse square root per pair; FP32 keeps a division for each
// quotient, whose rounding its trajectories follow.
template <class T>
__device__ __forceinline__ T pair_s(T r2, T qq, const AdjP &P) {
    T s = (T)0;
    if constexpr (sizeof(T) == 8) {
        const T ir = rsqrt64(r2), ir2 = ir * ir;
        if (r2 < P.rc2) {
            const T sr2 = P.sig2 * ir2, sr6 = sr2 * sr2 * sr2;
            const T F = (24.0 * P.eps) * (sr6 * sr6 + sr6 * sr6 - sr6) * ir;
            s += (F - P.flj_rc) * ir;
        }
        if (r2 < P.rcc2) s += P.kc * qq * (ir2 - P.inv_rcc2) * ir;
    } else {
        const T r = sqrt(r2), ir = (T)1 / r;
        if (r2 < (T)P.rc2) {
            const T sr2 = (T)(P.sigma * P.sigma) / r2, sr6 = sr2 * sr2 * sr2;
            const T F = (T)(24.0 * P.eps) * (sr6 * sr6 + sr6 * sr6 - sr6) * ir;
            s += (F - (T)P.flj_rc) * ir;
        }
        if (r2 < (T)P.rcc2) {
            const T F = (T)P.kc * qq * ((T)1 / r2 - (T)(1.0 / P.rcc2));
            s += F * ir;
        }
    }
    return s;
}

// FP64 pair terms of the reverse sweep: s, ds = s'(r)/r, ds/deps, ds/dsigma
// and H with ds_coulomb/dq_i = kc q_j H.
struct PairD {
    double s, ds, s_eps, s_sig, H;
};
__device__ __forceinline__ PairD pair_d(double r2, double qi, double qj, const AdjP &P) {
    PairD o{0.0, 0.0, 0.0, 0.0, 0.0};
    const double ir = rsqrt64(r2), ir2 = ir * ir, r = r2 * ir, ir3 = ir * ir2;
    if (r2 < P.rc2) {
        const double sr2 = P.sig2 * ir2, sr6 = sr2 * sr2 * sr2, sr12 = sr6 * sr6;
        const double F = 24.0 * P.eps * (2.0 * sr12 - sr6) * ir;
        const double Fp = 24.0 * P.eps * (-26.0 * sr12 + 7.0 * sr6) * ir2;
        const double s = (F - P.flj_rc) * ir;
        o.s += s;
        o.ds += (Fp * r - (F - P.flj_rc)) * ir3;
        o.s_eps = s * P.inv_eps;
        const double G = 24.0 * P.eps * (24.0 * sr12 - 6.0 * sr6) * ir * P.inv_sigma;
        o.s_sig = (G - P.glj_rc) * ir;
    }
    if (r2 < P.rcc2) {
        const double qq = qi * qj;
        const double Hf = ir2 - P.inv_rcc2;  // F_c = kc qq Hf
        const double F = P.kc * qq * Hf;
        const double Fp = -2.0 * P.kc * qq * ir3;
        o.s += F * ir;
        o.ds += (Fp * r - F) * ir3;
        o.H = Hf * ir;
    }
    return o;
}

// Position records: (x, y, z) and, in FP64, the charge (FP32 keeps the charges
// apart in FP64, as their product is taken).
template <class T> struct V4;
template <> struct V4<float> { using R = float4; };
template <> struct V4<double> { using R = double4; };

// Rows of the pair list: atom s (in the order of its build) keeps cap entries
// from lists[s cap], cnt[s] of them used, all of the same order.
struct Rows {
    const int32_t *lists, *cnt;
    int32_t cap;
    __device__ __forceinline__ const int32_t *row(int32_t s) const { return lists + (int64_t)s * cap; }
    __device__ __forceinline__ int32_t count(int32_t s) const { return cnt[s] < cap ? cnt[s] : cap; }
};

// Lanes per row: lane t of an atom takes entries t, t + kRowLanes, ...  (32,768
// atoms, some 82 entries: 8 / 16 / 32 lanes take 16.7 / 18.2 / 21.9 us in the
// reverse step and 11.5 / 11.6 / 13.9 in the forward one.)
constexpr int kRowLanes = 8;

// x, v of the caller's order and precision as records, and the FP32 positions
// the list build bins.
template <class T>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_init(const double *__restrict__ x, const double *__restrict__ v, const double *__restrict__ q, int32_t n,
           typename V4<T>::R *__restrict__ xo, typename V4<T>::R *__restrict__ vo, float4 *__restrict__ x32,
           int32_t *__restrict__ orig) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    typename V4<T>::R a, b;
    a.x = (T)x[3 * (int64_t)i]; a.y = (T)x[3 * (int64_t)i + 1]; a.z = (T)x[3 * (int64_t)i + 2];
    a.w = sizeof(T) == 8 ? (T)q[i] : (T)0;
    b.x = (T)v[3 * (int64_t)i]; b.y = (T)v[3 * (int64_t)i + 1]; b.z = (T)v[3 * (int64_t)i + 2];
    b.w = 0;
    xo[i] = a;
    vo[i] = b;
    x32[i] = make_float4((float)a.x, (float)a.y, (float)a.z, 0.0f);
    orig[i] = i;
}

template <class R>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_to_f32(const R *__restrict__ x, int32_t n, float4 *__restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float4((float)x[i].x, (float)x[i].y, (float)x[i].z, 0.0f);
}

// What the list builds of a pass tell the host: the largest row, status bits,
// and the largest row of the first build that had no room for one (if another
// came after it).  A pass runs on with rows cut short and is repeated with longer
// ones, so the builds after that one list another trajectory.  lines: the last
// list is, or has to be, built over lines of cells (BinGrid).
struct ListFlags {
    int32_t most, status, first, lines;
};

// Tests an atom, above which a box's cells count as crowded and lines are taken.
// Forward passes of 20 steps (three lists) over two droplets at growing distance
// or with an atom far out, by tests: 32,768 atoms 832 / 892 / 1,094 / 1,875 /
// 4,312 / 16,384: 649 / 669 / 683 / 790 / 1,172 / 1,902 us with the box's cells,
// 687 / 668 / 692 / 690 / 688 / 700 with lines; 8,192 atoms 824 / 1,328: 519 / 602
// and 565 / 533.  262,144 atoms, 75,173 tests: 24.5 ms and 2.2.  (A liquid: 480-560.)
constexpr double kCrowded = 1200.0;

// Atom i goes to its place in the cells: the cell-sorted FP32 copy with its
// number in the state's order, and (xo != null) the state into that order.
template <class R>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_place(const float4 *__restrict__ x32, const int2 *__restrict__ cell_of, const int32_t *__restrict__ cells,
            int32_t n, float4 *__restrict__ cpos, int32_t *__restrict__ ckey, const R *__restrict__ x,
            const R *__restrict__ v, const int32_t *__restrict__ orig, const double *__restrict__ q,
            R *__restrict__ xo, R *__restrict__ vo, int32_t *__restrict__ origo, double *__restrict__ qs,
            int32_t cap, const nd::BinGrid *__restrict__ grid, ListFlags *__restrict__ flags) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0) {
        if (flags->most > cap && flags->first == 0) flags->first = flags->most;
        flags->lines = grid->lines > 0 || (double)grid->tests > kCrowded * n;
    }
    const int2 c = cell_of[i];
    const int32_t u = cells[c.x] + c.y;
    const float4 p = x32[i];
    cpos[u] = make_float4(p.x, p.y, p.z, __int_as_float(xo ? u : i));
    ckey[u] = c.x;
    if (!xo) return;
    xo[u] = x[i];
    vo[u] = v[i];
    const int32_t o = orig[i];
    origo[u] = o;
    qs[u] = q[o];
}

// Rows of the list: the pairs of cell-sorted atoms closer than the list radius,
// each in both rows.  A wave takes kListAtoms consecutive atoms in groups of
// one cell row (k cells of about two dozen atoms): a batch of 64 candidates
// from the nine rows of cells around the group is tested against its atoms one
// after another, and a ballot places the hits.  LINES: the cells are those of
// lines on a circle; a run of a line is two runs of the table where it passes
// the circle's end, and a candidate counts only in the run of its own line.
constexpr int kListAtoms = 8;
constexpr int kLineCells = 4;  // cells a group may lie in

template <bool LINES>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_rows(const float4 *__restrict__ cpos, const int32_t *__restrict__ ckey, const int32_t *__restrict__ cells,
           const nd::BinGrid *__restrict__ grid, int32_t n, float rl2, int32_t cap, int32_t *__restrict__ lists,
           int32_t *__restrict__ cnt, ListFlags *__restrict__ flags) {
    const int lane = threadIdx.x & 63;
    const int32_t t0 = __builtin_amdgcn_readfirstlane((int32_t)((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * kListAtoms);
    const int32_t lines = grid->lines;
    // (cells found crowded: no rows, the host asks for lines)
    if (t0 >= n || LINES != (flags->lines != 0)) return;
    constexpr int RUNS = LINES ? 18 : 9;
    const int32_t nt = min(kListAtoms, n - t0);
    const int32_t g0 = grid->cg.g[0], g1 = grid->cg.g[1], g2 = grid->cg.g[2];
    const int32_t k = LINES ? kLineCells : max(1, (int32_t)(24.0f * (float)grid->cg.ncell / (float)n));
    const double inv = grid->inv;
    float px = 0.0f, py = 0.0f, pz = 0.0f;
    int32_t pk = -1, pid = 0, found = 0;
    if (lane < nt) {
        const float4 p = cpos[t0 + lane];
        px = p.x;
        py = p.y;
        pz = p.z;
        pid = __float_as_int(p.w);
        pk = ckey[t0 + lane];
    }
    const int32_t prow = LINES ? 0 : pk / g0;
    const double py_ = LINES ? nd::line_coord(inv, py) : 0.0, pz_ = LINES ? nd::line_coord(inv, pz) : 0.0;
    auto lf = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    int32_t q0 = 0;
    while (q0 < nt) {
        const int32_t k0 = __builtin_amdgcn_readlane(pk, q0), row = __builtin_amdgcn_readlane(prow, q0);
        const double y0 = LINES ? __shfl(py_, q0, 64) : 0.0, z0 = LINES ? __shfl(pz_, q0, 64) : 0.0;
        // q0 and the atoms after it up to the first of another row or beyond k cells
        const bool same = LINES ? lane == q0 || (py_ == y0 && pz_ == z0) : prow == row;
        const uint64_t in = __builtin_amdgcn_ballot_w64(lane >= q0 && lane < nt && same && pk < k0 + k);
        const int32_t q1 = q0 + (LINES ? __builtin_ctzll(~(in >> q0)) : __builtin_popcountll(in));
        const int32_t k1 = __builtin_amdgcn_readlane(pk, q1 - 1);
        const int32_t c0 = k0 - row * g0, c1 = k1 - row * g0;
        const int32_t cy = row % g1, cz = row / g1;
        // lane j: the run of cell row j around the group (lines: 9 + j its rest
        // beyond the end of the table), and the row's cell
        int32_t from = 0, to = 0;
        double ry = 0.0, rz = 0.0;
        if (LINES && lane < RUNS) {
            const int32_t dy = lane % 9 % 3 - 1, dz = lane % 9 / 3 - 1, span = k1 - k0 + 3;
            ry = y0 + dy;
            rz = z0 + dz;
            // (cells so far out that one more is the same number have no others beside them)
            if ((dy == 0 || ry != y0) && (dz == 0 || rz != z0)) {
                int32_t at = (k0 - 1 + nd::line_start(ry, rz, lines) - nd::line_start(y0, z0, lines)) % lines;
                if (at < 0) at += lines;
                if (lane < 9) {
                    from = cells[at];
                    to = cells[min(at + span, lines)];
                } else if (at + span > lines) {
                    to = cells[at + span - lines];
                }
            }
        }
        if (!LINES && lane < RUNS) {
            const int32_t y = cy + lane % 3 - 1, z = cz + lane / 3 - 1;
            if (y >= 0 && y < g1 && z >= 0 && z < g2) {
                const int32_t b = (z * g1 + y) * g0;
                from = cells[b + max(c0 - 1, 0)];
                to = cells[b + min(c1 + 1, g0 - 1) + 1];
            }
        }
        // the runs as one sequence; lane j: candidates before run j, and its
        // start less those
        int32_t pre = to - from;
#pragma unroll
        for (int o = 1; o < RUNS; o <<= 1) {
            const int32_t v = __shfl_up(pre, o, 64);
            if (lane >= o) pre += v;
        }
        const int32_t total = __builtin_amdgcn_readlane(pre, RUNS - 1);
        pre -= to - from;
        const int32_t rise = from - pre;
        int32_t at_run = 0;
        // run: of each lane's candidate
        auto fetch = [&](int32_t s0, int32_t &u, int32_t &run) {
            const int32_t ci = s0 + lane;
            u = ci + __builtin_amdgcn_readlane(rise, at_run);
            run = at_run;
            while (at_run < RUNS - 1) {
                const int32_t p = __builtin_amdgcn_readlane(pre, at_run + 1);
                if (p > s0 + 63) break;
                ++at_run;
                u = ci >= p ? ci + __builtin_amdgcn_readlane(rise, at_run) : u;
                run = ci >= p ? at_run : run;
            }
            if (ci >= total) u = -1;
            return cpos[u < 0 ? t0 : u];
        };
        int32_t un, rn;
        float4 c = fetch(0, un, rn);
        for (int32_t s0 = 0; s0 < total; s0 += 64) {
            // the next batch is on its way while this one is tested
            int32_t u = un;
            const int32_t run = rn;
            const float4 d = c;
            if (s0 + 64 < total) c = fetch(s0 + 64, un, rn);
            if (LINES) {  // atoms of other lines in the same table cells
                const double wy = __shfl(ry, run, 64), wz = __shfl(rz, run, 64);
                if (nd::line_coord(inv, d.y) != wy || nd::line_coord(inv, d.z) != wz) u = -1;
            }
            for (int32_t q = q0; q < q1; ++q) {
                const float dx = d.x - lf(px, q), dy = d.y - lf(py, q), dz = d.z - lf(pz, q);
                const bool hit = (dx * dx + dy * dy + dz * dz < rl2) & (u >= 0) & (u != t0 + q);
                const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
                const int32_t have = __builtin_amdgcn_readlane(found, q);
                if (hit) {
                    const int32_t at = (int32_t)__builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)have));
                    if (at < cap) lists[(int64_t)__builtin_amdgcn_readlane(pid, q) * cap + at] = __float_as_int(d.w);
                }
                found = lane == q ? have + __builtin_popcountll(m) : found;
            }
        }
        q0 = q1;
    }
    if (lane < nt) cnt[pid] = found;
    int32_t mx = found;
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    if (lane == 0 && mx > __hip_atomic_load(&flags->most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&flags->most, mx);
}

__device__ __forceinline__ double fix_val(unsigned long long v) { return (double)(long long)v * kInvFix; }

// One launch of the forward model at x_k: F_i = sum_j s(r_ij) r_ij over row i,
// summed in 2^-40 fixed point (the same whatever the order of the row and
// however it is split); finish: the half kick that ends step k - 1; vck: the
// velocity at k kept; xo: the half kick and drift that begin step k.
// One instance serves every step (finish and a null xo are arguments): another
// could contract its products differently, and the recompute has to repeat the
// forward pass to the bit.
template <class T>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_step(Rows R, const typename V4<T>::R *__restrict__ x, const double *__restrict__ qs, AdjP P,
           typename V4<T>::R *__restrict__ v, int32_t finish, typename V4<T>::R *__restrict__ vck,
           typename V4<T>::R *__restrict__ xo, float4 *__restrict__ x32) {
    using V = typename V4<T>::R;
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int32_t s = (int32_t)(t / kRowLanes), sub = (int32_t)(t % kRowLanes);
    long long fx = 0, fy = 0, fz = 0;
    V xi{};
    if (s < P.n) {
        const int32_t *row = R.row(s);
        const int32_t c = R.count(s);
        xi = x[s];
        const double qi = sizeof(T) == 8 ? (double)xi.w : qs[s];
        int32_t j = sub < c ? row[sub] : 0;
        for (int32_t k = sub; k < c; k += kRowLanes) {
            const V xj = x[j];
            const double qj = sizeof(T) == 8 ? (double)xj.w : qs[j];
            j = k + kRowLanes < c ? row[k + kRowLanes] : 0;
            const T dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
            const T r2 = dx * dx + dy * dy + dz * dz;
            if (!(r2 < (T)P.rc2 || r2 < (T)P.rcc2)) continue;
            const T f = pair_s<T>(r2, (T)(qi * qj), P);
            fx += llrint((double)(f * dx) * kFix);
            fy += llrint((double)(f * dy) * kFix);
            fz += llrint((double)(f * dz) * kFix);
        }
    }
    // exact integer sums over the atom's lanes (all lanes take part)
#pragma unroll
    for (int off = 1; off < kRowLanes; off <<= 1) {
        fx += __shfl_xor(fx, off, 64);
        fy += __shfl_xor(fy, off, 64);
        fz += __shfl_xor(fz, off, 64);
    }
    if (s >= P.n || sub != 0) return;
    const T f[3] = {(T)fix_val((unsigned long long)fx), (T)fix_val((unsigned long long)fy),
                    (T)fix_val((unsigned long long)fz)};
    V w = v[s];
    if (finish) {
        w.x = w.x + (T)P.c * f[0];
        w.y = w.y + (T)P.c * f[1];
        w.z = w.z + (T)P.c * f[2];
    }
    if (vck) vck[s] = w;
    if (xo) {
        w.x = w.x + (T)P.c * f[0];
        w.y = w.y + (T)P.c * f[1];
        w.z = w.z + (T)P.c * f[2];
        xi.x = xi.x + (T)P.dt * w.x;
        xi.y = xi.y + (T)P.dt * w.y;
        xi.z = xi.z + (T)P.dt * w.z;
        xo[s] = xi;
        if (x32) x32[s] = make_float4((float)xi.x, (float)xi.y, (float)xi.z, 0.0f);
    }
    v[s] = w;
}

// RDF kernel weight of pair distance r for bin b
__device__ __forceinline__ double rdf_K(double d, double h) {
    const double u = d / h, t = 1.0 - u * u;
    return fabs(u) < 1.0 ? t * t * t : 0.0;
}
__device__ __forceinline__ double rdf_dK(double d, double h) {
    const double u = d / h, t = 1.0 - u * u;
    return fabs(u) < 1.0 ? -6.0 * u * t * t / h : 0.0;
}

// raw histogram sum_{i<j} K(r_ij - r_b) (normalisation on the host); bins are
// summed per workgroup in LDS, the workgroups' in index order by k_rdf_sum
constexpr int kMaxBins = 1024;
constexpr int kHistBlocks = 512;

template <class T>
__global__ void __launch_bounds__(nd::kBlock)
k_rdf_hist(Rows R, const typename V4<T>::R *__restrict__ x, AdjP P, double *__restrict__ part) {
    __shared__ double hb[kMaxBins];
    for (int b = threadIdx.x; b < P.nbins; b += blockDim.x) hb[b] = 0.0;
    __syncthreads();
    const int32_t sub = threadIdx.x % kRowLanes;
    for (int32_t s = (int32_t)((blockIdx.x * blockDim.x + threadIdx.x) / kRowLanes); s < P.n;
         s += (int32_t)(gridDim.x * blockDim.x / kRowLanes)) {
        const auto xi = x[s];
        const int32_t *row = R.row(s);
        const int32_t c = R.count(s);
        for (int32_t k = sub; k < c; k += kRowLanes) {
            const int32_t j = row[k];
            if (j < s) continue;  // each unordered pair once
            const auto xj = x[j];
            const double dx = (double)xi.x - (double)xj.x, dy = (double)xi.y - (double)xj.y,
                         dz = (double)xi.z - (double)xj.z;
            const double r = sqrt(dx * dx + dy * dy + dz * dz);
            if (!(r < P.rmax + P.h)) continue;
            const int32_t b0 = max(0, (int32_t)floor((r - P.h) / P.dr - 0.5));
            const int32_t b1 = min(P.nbins - 1, (int32_t)ceil((r + P.h) / P.dr - 0.5));
            for (int32_t b = b0; b <= b1; ++b) {
                const double w = rdf_K(r - (b + 0.5) * P.dr, P.h);
                if (w != 0.0) atomicAdd(&hb[b], w);
            }
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < P.nbins; b += blockDim.x) part[(int64_t)blockIdx.x * P.nbins + b] = hb[b];
}

// hist[b] = sum over the workgroups' parts, one workgroup per bin
__global__ void __launch_bounds__(nd::kBlock)
k_rdf_sum(const double *__restrict__ part, int32_t nparts, int32_t nbins, double *__restrict__ hist) {
    __shared__ double sh[nd::kBlock / 64];
    double v = 0.0;
    for (int32_t k = threadIdx.x; k < nparts; k += nd::kBlock) v += part[(int64_t)k * nbins + blockIdx.x];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < nd::kBlock / 64; ++k) v += sh[k];
        hist[blockIdx.x] = v;
    }
}

// Adjoint records of an atom, FP64.
struct Lam {
    double4 *x, *v, *a;  // lambda_x, lambda_v, a = w lambda_h
};

// lambda_h = lambda_v + dt lambda_x; lambda_v = lambda_h; a = w lambda_h
__device__ __forceinline__ void next_vec(const Lam &L, int32_t s, const double4 &lx, double dt, double w) {
    double4 h = L.v[s];
    h.x += dt * lx.x;
    h.y += dt * lx.y;
    h.z += dt * lx.z;
    L.v[s] = h;
    L.a[s] = make_double4(w * h.x, w * h.y, w * h.z, 0.0);
}

// Start of the reverse sweep: lambda_x = dL/dx_T with L = sum_b (g_b - t_b)^2,
// wb[b] = 2 (g_b - t_b) norm_b; lambda_v = 0; then the last step's vectors.
template <class T>
__global__ void __launch_bounds__(nd::kBlock)
k_rdf_grad(Rows R, const typename V4<T>::R *__restrict__ x, AdjP P, const double *__restrict__ wb, Lam L,
           double wvec) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int32_t s = (int32_t)(t / kRowLanes), sub = (int32_t)(t % kRowLanes);
    double gx = 0.0, gy = 0.0, gz = 0.0;
    if (s < P.n) {
        const int32_t *row = R.row(s);
        const int32_t c = R.count(s);
        const auto xi = x[s];
        for (int32_t k = sub; k < c; k += kRowLanes) {
            const auto xj = x[row[k]];
            const double dx = (double)xi.x - (double)xj.x, dy = (double)xi.y - (double)xj.y,
                         dz = (double)xi.z - (double)xj.z;
            const double r = sqrt(dx * dx + dy * dy + dz * dz);
            if (!(r < P.rmax + P.h)) continue;
            const int32_t b0 = max(0, (int32_t)floor((r - P.h) / P.dr - 0.5));
            const int32_t b1 = min(P.nbins - 1, (int32_t)ceil((r + P.h) / P.dr - 0.5));
            double g = 0.0;
            for (int32_t b = b0; b <= b1; ++b) g += wb[b] * rdf_dK(r - (b + 0.5) * P.dr, P.h);
            const double f = g / r;
            gx += f * dx;
            gy += f * dy;
            gz += f * dz;
        }
    }
#pragma unroll
    for (int off = 1; off < kRowLanes; off <<= 1) {
        gx += __shfl_xor(gx, off, 64);
        gy += __shfl_xor(gy, off, 64);
        gz += __shfl_xor(gz, off, 64);
    }
    if (s >= P.n || sub != 0) return;
    const double4 lx = make_double4(gx, gy, gz, 0.0);
    L.x[s] = lx;
    L.v[s] = make_double4(0.0, 0.0, 0.0, 0.0);
    next_vec(L, s, lx, P.dt, wvec);
}

// One launch of the reverse sweep at x_k: lambda_x += J(x_k) a; dq, (eps,
// sigma) += (dF/dtheta)^T a; and, for k > 0, the vectors of step k - 1 (the new
// a goes to anext, since others still read this one).  Row i gives atom i's own
// terms; each unordered pair sits in two rows, so its eps / sigma term is taken
// with weight 1/2 from each.
template <class T>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_hvp(Rows R, const typename V4<T>::R *__restrict__ x, const double *__restrict__ qs,
          const int32_t *__restrict__ orig, AdjP P, Lam L, double4 *__restrict__ anext, double wnext,
          double *__restrict__ dq, double *__restrict__ dpar) {
    __shared__ double sh[2][nd::kBlock / 64];
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int32_t s = (int32_t)(t / kRowLanes), sub = (int32_t)(t % kRowLanes);
    double ge = 0.0, gs = 0.0;
    double mx = 0.0, my = 0.0, mz = 0.0, gq = 0.0;
    if (s < P.n) {
        const auto xi = x[s];
        const double4 ai = L.a[s];
        const double qi = sizeof(T) == 8 ? (double)xi.w : qs[s];
        const int32_t *row = R.row(s);
        const int32_t c = R.count(s);
        int32_t j = sub < c ? row[sub] : 0;
        for (int32_t k = sub; k < c; k += kRowLanes) {
            const auto xj = x[j];
            const double4 aj = L.a[j];
            const double qj = sizeof(T) == 8 ? (double)xj.w : qs[j];
            j = k + kRowLanes < c ? row[k + kRowLanes] : 0;
            const double dx = (double)xi.x - (double)xj.x, dy = (double)xi.y - (double)xj.y,
                         dz = (double)xi.z - (double)xj.z;
            const double r2 = dx * dx + dy * dy + dz * dz;
            if (!(r2 < P.rc2 || r2 < P.rcc2)) continue;
            const PairD d = pair_d(r2, qi, qj, P);
            const double ax = ai.x - aj.x, ay = ai.y - aj.y, az = ai.z - aj.z;
            const double rda = dx * ax + dy * ay + dz * az;
            mx += d.s * ax + d.ds * rda * dx;
            my += d.s * ay + d.ds * rda * dy;
            mz += d.s * az + d.ds * rda * dz;
            gq += P.kc * qj * d.H * rda;
            ge += 0.5 * d.s_eps * rda;
            gs += 0.5 * d.s_sig * rda;
        }
    }
    // the atom's lanes combine their partial sums in a fixed order
#pragma unroll
    for (int off = 1; off < kRowLanes; off <<= 1) {
        mx += __shfl_xor(mx, off, 64);
        my += __shfl_xor(my, off, 64);
        mz += __shfl_xor(mz, off, 64);
        gq += __shfl_xor(gq, off, 64);
    }
    if (s < P.n && sub == 0) {
        double4 lx = L.x[s];
        lx.x += mx;
        lx.y += my;
        lx.z += mz;
        L.x[s] = lx;
        dq[orig[s]] += gq;
        if (anext) {
            Lam N = L;
            N.a = anext;
            next_vec(N, s, lx, P.dt, wnext);
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        ge += __shfl_down(ge, o, 64);
        gs += __shfl_down(gs, o, 64);
    }
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) { sh[0][w] = ge; sh[1][w] = gs; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double e = 0.0, g = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) { e += sh[0][k]; g += sh[1][k]; }
        // this workgroup's own words, summed over the sweep
        dpar[2 * (int64_t)blockIdx.x] += e;
        dpar[2 * (int64_t)blockIdx.x + 1] += g;
    }
}

// The adjoint records from one order to another, by way of the caller's.
__global__ void __launch_bounds__(nd::kBlock)
k_adj_to_caller(const int32_t *__restrict__ orig, int32_t n, Lam L, Lam O) {
    const int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int32_t o = orig[s];
    O.x[o] = L.x[s];
    O.v[o] = L.v[s];
    O.a[o] = L.a[s];
}
__global__ void __launch_bounds__(nd::kBlock)
k_adj_from_caller(const int32_t *__restrict__ orig, int32_t n, Lam O, Lam L, const double *__restrict__ q,
                  double *__restrict__ qs) {
    const int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int32_t o = orig[s];
    L.x[s] = O.x[o];
    L.v[s] = O.v[o];
    L.a[s] = O.a[o];
    qs[s] = q[o];
}

// (x, y, z) records in build order to n x 3 of the caller's order, in FP64.
template <class R>
__global__ void __launch_bounds__(nd::kBlock)
k_adj_export(const R *__restrict__ a, const int32_t *__restrict__ orig, int32_t n, double *__restrict__ out) {
    const int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t o = 3 * (int64_t)orig[s];
    out[o] = (double)a[s].x;
    out[o + 1] = (double)a[s].y;
    out[o + 2] = (double)a[s].z;
}

// The workgroups' eps / sigma sums in index order (one workgroup).
__global__ void __launch_bounds__(nd::kBlock)
k_adj_sum_par(const double *__restrict__ part, int32_t m, double *__restrict__ out) {
    __shared__ double sh[2][nd::kBlock / 64];
    double e = 0.0, g = 0.0;
    for (int32_t k = threadIdx.x; k < m; k += nd::kBlock) {
        e += part[2 * (int64_t)k];
        g += part[2 * (int64_t)k + 1];
    }
    for (int o = 32; o > 0; o >>= 1) {
        e += __shfl_down(e, o, 64);
        g += __shfl_down(g, o, 64);
    }
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = e; sh[1][threadIdx.x >> 6] = g; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < nd::kBlock / 64; ++k) { e += sh[0][k]; g += sh[1][k]; }
        out[0] = e;
        out[1] = g;
    }
}

__global__ void k_zero_f64(double *p, int64_t m) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k < m) p[k] = 0.0;
}

}  // namespace

struct nd_adj {
    nd_ctx *ctx = nullptr;
    nd_adj_params p{};
    AdjP P{};
    bool dbl = true;
    float rlist = 0.0f;
    // input of the call (FP64, caller's order) and charges
    nd::DevBuf x0, v0, q;
    // state: positions of the current segment (x_k for its every step) and of
    // x_T, the drifted positions before a build, velocities (two: a build
    // moves them), charges in build order (FP32)
    nd::DevBuf seg, xT, tmp, x32, vel[2], qs;
    int vcur = 0;
    nd::DevBuf ckx, ckv, ck_orig;  // checkpoints of all segments but the last
    // lists of the current segment's windows (slot w) and of x_T; a slot past
    // the memory kept for them is shared, tagged with the window it holds
    nd::DevBuf lists, lcnt, orig;
    int32_t nwin = 0;              // orders kept: windows of a segment, x_T, and one spare
    int32_t nslots = 0;            // rows kept
    std::vector<int32_t> holds;    // window of each slot's rows
    std::vector<int32_t> order;    // index of each window's order in orig
    int32_t spare = 0;             // index of the unused order
    nd::DevBuf bins, cell_of, cells, cpos, ckey;  // list build
    nd::BinMode bin_mode = nd::kBinBox;           // the cells of the pass, chosen at its first list
    nd::DevBuf lam, lam_caller, dq, dpar, out, hist, part, wb;
    int32_t cap = 0;  // row capacity
    bool have_forward = false;
    std::vector<double> target, rdf, norm, weights;
    double loss = 0.0;
};

namespace {

// Bytes of rows kept for the reverse sweep; windows past them are listed again.
constexpr size_t kListBytes = (size_t)4 << 30;

void reserve_rows(nd_adj *s) {
    const size_t one = sizeof(int32_t) * (size_t)s->cap * (size_t)s->p.n;
    s->nslots = (int32_t)std::max<size_t>(2, std::min<size_t>((size_t)s->nwin - 1, kListBytes / one));
    s->lists.reserve(one * (size_t)s->nslots);
    s->lcnt.reserve(sizeof(int32_t) * (size_t)s->p.n * (size_t)s->nslots);
    s->holds.assign(s->nslots, -1);
}

int32_t slot_of(const nd_adj *s, int32_t w) { return std::min(w, s->nslots - 1); }

Rows rows_of(nd_adj *s, int32_t w) {
    const int64_t o = (int64_t)slot_of(s, w) * s->p.n;
    return Rows{s->lists.as<int32_t>() + o * s->cap, s->lcnt.as<int32_t>() + o, s->cap};
}

int32_t *order_of(nd_adj *s, int32_t w) { return s->orig.as<int32_t>() + (size_t)s->order[w] * s->p.n; }

// the list builds' flags, then the histogram
ListFlags *flags_of(nd_adj *s) { return s->hist.as<ListFlags>(); }
double *hist_of(nd_adj *s) { return s->hist.as<double>() + 2; }

// Rows (and, move, the new order) of window w at the positions in s->x32.
template <class V>
void build_rows(nd_adj *s, int32_t w, nd::BinMode mode, const V *x, const V *v, const int32_t *orig, V *xo, V *vo,
                int32_t *origo) {
    hipStream_t st = s->ctx->stream;
    const int32_t n = s->p.n;
    const int32_t max_cells = std::max(27, n / 2);
    const float4 *x32 = s->x32.as<float4>();
    const nd::BinGrid *grid = nd::launch_cell_bins(st, s->bins.p, x32, n, s->rlist, max_cells, mode,
                                                   kCrowded, s->cell_of.as<int2>(), s->cells.as<int32_t>(),
                                                   &flags_of(s)->status);
    k_adj_place<V><<<nd::grid_for(n), nd::kBlock, 0, st>>>(
        x32, s->cell_of.as<int2>(), s->cells.as<int32_t>(), n, s->cpos.as<float4>(), s->ckey.as<int32_t>(), x, v, orig,
        s->q.as<double>(), xo, vo, origo, s->qs.as<double>(), s->cap, grid, flags_of(s));
    const Rows R = rows_of(s, w);
    const auto rows = mode == nd::kBinLines ? k_adj_rows<true> : k_adj_rows<false>;
    rows<<<nd::grid_for(((int64_t)n + kListAtoms - 1) / kListAtoms * 64), nd::kBlock, 0, st>>>(
        s->cpos.as<float4>(), s->ckey.as<int32_t>(), s->cells.as<int32_t>(), grid, n, s->rlist * s->rlist, s->cap,
        const_cast<int32_t *>(R.lists), const_cast<int32_t *>(R.cnt), flags_of(s));
    ND_HIP(hipGetLastError());
    s->holds[slot_of(s, w)] = w;
}

// The list of window w for the positions in s->tmp (order from): moves the
// state into its order, the positions to xo.
template <class T>
void build_list(nd_adj *s, int32_t w, int32_t from, typename V4<T>::R *xo, nd::BinMode mode) {
    using V = typename V4<T>::R;
    int32_t *orig = s->orig.as<int32_t>();
    const size_t n = (size_t)s->p.n;
    const int32_t src = from, dst = s->spare;
    build_rows<V>(s, w, mode, s->tmp.as<V>(), s->vel[s->vcur].as<V>(), orig + (size_t)src * n, xo,
                  s->vel[s->vcur ^ 1].as<V>(), orig + (size_t)dst * n);
    s->vcur ^= 1;
    // the order window w had before is free now
    s->spare = s->order[w];
    s->order[w] = dst;
}

template <class T>
typename V4<T>::R *seg_at(nd_adj *s, int32_t k) {
    return s->seg.as<typename V4<T>::R>() + (size_t)k * s->p.n;
}

// The launch at step k (positions x, rows of window w).
template <class T>
void launch_step(nd_adj *s, int32_t w, const typename V4<T>::R *x, bool finish, typename V4<T>::R *vck,
                 typename V4<T>::R *xo, bool to_bins) {
    using V = typename V4<T>::R;
    hipStream_t st = s->ctx->stream;
    const unsigned g = nd::grid_for((int64_t)s->p.n * kRowLanes);
    V *v = s->vel[s->vcur].as<V>();
    float4 *x32 = to_bins ? s->x32.as<float4>() : nullptr;
    const Rows R = rows_of(s, w);
    const double *qs = s->qs.as<double>();
    k_adj_step<T><<<g, nd::kBlock, 0, st>>>(R, x, qs, s->P, v, finish ? 1 : 0, vck, xo, x32);
    ND_HIP(hipGetLastError());
}

// Steps k0 .. of a segment, whose first list (window 0, x_k0 in seg[0]) is
// there.  forward: to k1, with the list at k1 (the next segment's first, or
// x_T's); else (recompute) to x_{k1-1}.
template <class T>
void advance(nd_adj *s, int32_t k0, int32_t k1, bool forward, bool finish_first, typename V4<T>::R *vck) {
    using V = typename V4<T>::R;
    const int32_t W = s->p.rebuild_every, T_ = s->p.nsteps;
    const int32_t last = forward ? k1 : k1 - 1;  // positions wanted up to here
    for (int32_t k = k0; k < last; ++k) {
        const int32_t w = (k - k0) / W;
        const bool end = k + 1 == k1, build = (k + 1) % W == 0 || k + 1 == T_;
        V *xo = build ? s->tmp.as<V>() : seg_at<T>(s, k + 1 - k0);
        launch_step<T>(s, w, seg_at<T>(s, k - k0), k > k0 || finish_first, k == k0 ? vck : nullptr, xo, build);
        if (!build) continue;
        if (k + 1 == T_) build_list<T>(s, s->nwin - 2, s->order[w], s->xT.as<V>(), s->bin_mode);
        else build_list<T>(s, end ? 0 : w + 1, s->order[w], seg_at<T>(s, end ? 0 : k + 1 - k0), s->bin_mode);
    }
}

// Longer rows are refused: at this length one list of a million atoms takes 262 GB.
constexpr int32_t kMaxRow = 65535;

// Whether the builds so far had room, which is made if not (the pass has to be
// repeated); throws what else they found.  The largest row of a pass that ran on
// without room says how much denser the system is about to get, but no more:
// without their repulsion atoms gather (32,768 atoms moving inwards, rows of at
// most 275: rows of 1,800 counted), so four times the last row known to be right
// is the most that is made for.
bool had_room(nd_adj *s, const ListFlags &f) {
    if (f.most <= s->cap) {
        if (f.status & nd::kStatusDomain) throw nd::Error(ND_ERR_DOMAIN, "adjoint: non-finite coordinate");
        return true;
    }
    const int32_t right = f.first > 0 ? f.first : f.most;
    if (right > kMaxRow) throw nd::Error(ND_ERR_CAPACITY, "adjoint: more than 65,535 neighbours per atom");
    s->cap = std::min(std::min(f.most + f.most / 4, 4 * right) + 8, s->p.n);
    reserve_rows(s);
    return false;
}

template <class T>
void forward_impl(nd_adj *s) {
    using V = typename V4<T>::R;
    hipStream_t st = s->ctx->stream;
    const int32_t K = s->p.checkpoint_every, T_ = s->p.nsteps, n = s->p.n, nb = s->p.nbins;
    const size_t vb = sizeof(V) * (size_t)n, ib = sizeof(int32_t) * (size_t)n;
    std::vector<double> h(2 + nb);
    static_assert(sizeof(ListFlags) == 2 * sizeof(double), "flags before the histogram");
    auto flags = [&] {
        ListFlags f;
        std::memcpy(&f, h.data(), sizeof f);
        return f;
    };
    // the first list says which cells the pass takes; every attempt after that has
    // longer rows and gets past the build that ended the one before
    s->bin_mode = nd::kBinCount;
    for (;;) {
        nd::launch_fill_i32(st, reinterpret_cast<int32_t *>(flags_of(s)), 4, 0);
        s->vcur = 0;
        k_adj_init<T><<<nd::grid_for(n), nd::kBlock, 0, st>>>(
            s->x0.as<double>(), s->v0.as<double>(), s->q.as<double>(), n, s->tmp.as<V>(), s->vel[0].as<V>(),
            s->x32.as<float4>(), order_of(s, s->nwin - 2));
        build_list<T>(s, 0, s->order[s->nwin - 2], seg_at<T>(s, 0), s->bin_mode);
        // room for the first list is made before the steps run on it
        ND_HIP(hipMemcpyAsync(h.data(), s->hist.p, sizeof(ListFlags), hipMemcpyDeviceToHost, st));
        ND_HIP(hipStreamSynchronize(st));
        if (s->bin_mode == nd::kBinCount) {
            s->bin_mode = flags().lines ? nd::kBinLines : nd::kBinBox;
            if (s->bin_mode == nd::kBinLines) continue;
        }
        if (!had_room(s, flags())) continue;
        for (int32_t c = 0; c * K < T_; ++c) {
            const int32_t k0 = c * K, k1 = std::min((c + 1) * K, T_);
            V *vck = nullptr;
            if (k1 < T_) {  // the last segment needs no checkpoint: its positions stay
                ND_HIP(hipMemcpyAsync(s->ckx.as<V>() + (size_t)c * n, seg_at<T>(s, 0), vb, hipMemcpyDeviceToDevice, st));
                ND_HIP(hipMemcpyAsync(s->ck_orig.as<int32_t>() + (size_t)c * n, order_of(s, 0), ib,
                                      hipMemcpyDeviceToDevice, st));
                vck = s->ckv.as<V>() + (size_t)c * n;
            }
            advance<T>(s, k0, k1, true, c > 0, vck);
        }
        // the last half kick, and the final frame's radial distribution
        launch_step<T>(s, s->nwin - 2, s->xT.as<V>(), true, nullptr, nullptr, false);
        const Rows R = rows_of(s, s->nwin - 2);
        const unsigned hb = std::min<unsigned>(nd::grid_for((int64_t)n * kRowLanes), kHistBlocks);
        k_rdf_hist<T><<<hb, nd::kBlock, 0, st>>>(R, s->xT.as<V>(), s->P, s->part.as<double>());
        k_rdf_sum<<<nb, nd::kBlock, 0, st>>>(s->part.as<double>(), (int32_t)hb, nb, hist_of(s));
        ND_HIP(hipGetLastError());
        ND_HIP(hipMemcpyAsync(h.data(), s->hist.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
        ND_HIP(hipStreamSynchronize(st));
        if (had_room(s, flags())) break;
    }
    s->rdf.resize(nb);
    s->loss = 0.0;
    for (int32_t b = 0; b < nb; ++b) {
        s->rdf[b] = s->norm[b] * h[2 + b];
        if (!s->target.empty()) s->loss += (s->rdf[b] - s->target[b]) * (s->rdf[b] - s->target[b]);
    }
    s->have_forward = true;
}

template <class T>
void backward_impl(nd_adj *s) {
    using V = typename V4<T>::R;
    hipStream_t st = s->ctx->stream;
    const int32_t K = s->p.checkpoint_every, T_ = s->p.nsteps, W = s->p.rebuild_every, n = s->p.n;
    const size_t vb = sizeof(V) * (size_t)n, ib = sizeof(int32_t) * (size_t)n;
    const unsigned g = nd::grid_for(n), gr = nd::grid_for((int64_t)n * kRowLanes);
    double4 *lam = s->lam.as<double4>(), *lc = s->lam_caller.as<double4>();
    Lam L{lam, lam + n, lam + 2 * (size_t)n}, C{lc, lc + n, lc + 2 * (size_t)n};
    double4 *a2 = lam + 3 * (size_t)n;
    k_zero_f64<<<g, nd::kBlock, 0, st>>>(s->dq.as<double>(), n);
    k_zero_f64<<<nd::grid_for(2 * (int64_t)gr), nd::kBlock, 0, st>>>(s->dpar.as<double>(), 2 * (int64_t)gr);
    std::vector<double> &wb = s->weights;  // outlives the copy
    wb.resize(s->p.nbins);
    for (int32_t b = 0; b < s->p.nbins; ++b) wb[b] = 2.0 * (s->rdf[b] - s->target[b]) * s->norm[b];
    ND_HIP(hipMemcpyAsync(s->wb.p, wb.data(), sizeof(double) * wb.size(), hipMemcpyHostToDevice, st));
    auto weight = [&](int32_t k) { return k == 0 ? s->P.c : 2.0 * s->P.c; };
    const int32_t fin = s->nwin - 2;
    if (s->holds[slot_of(s, fin)] != fin) throw nd::Error(ND_ERR_STATE, "adjoint: the final list is gone");
    k_rdf_grad<T><<<gr, nd::kBlock, 0, st>>>(rows_of(s, fin), s->xT.as<V>(), s->P, s->wb.as<double>(), L,
                                             weight(T_ - 1));
    const int32_t *at = order_of(s, fin);  // the adjoint records' order
    for (int32_t c = (T_ - 1) / K; c >= 0; --c) {
        const int32_t k0 = c * K, k1 = std::min((c + 1) * K, T_);
        if (k1 < T_) {
            // the records wait in the caller's order while the segment is
            // recomputed from its checkpoint
            k_adj_to_caller<<<g, nd::kBlock, 0, st>>>(at, n, L, C);
            at = nullptr;
            ND_HIP(hipMemcpyAsync(s->tmp.p, s->ckx.as<V>() + (size_t)c * n, vb, hipMemcpyDeviceToDevice, st));
            ND_HIP(hipMemcpyAsync(s->vel[s->vcur].p, s->ckv.as<V>() + (size_t)c * n, vb, hipMemcpyDeviceToDevice, st));
            ND_HIP(hipMemcpyAsync(order_of(s, fin), s->ck_orig.as<int32_t>() + (size_t)c * n, ib,
                                  hipMemcpyDeviceToDevice, st));
            k_adj_to_f32<V><<<g, nd::kBlock, 0, st>>>(s->tmp.as<V>(), n, s->x32.as<float4>());
            build_list<T>(s, 0, s->order[fin], seg_at<T>(s, 0), s->bin_mode);
            advance<T>(s, k0, k1, false, false, nullptr);
        }
        int32_t win = -1;
        for (int32_t k = k1 - 1; k >= k0; --k) {
            const int32_t w = (k - k0) / W;
            if (w != win) {
                if (at) k_adj_to_caller<<<g, nd::kBlock, 0, st>>>(at, n, L, C);
                at = order_of(s, w);
                k_adj_from_caller<<<g, nd::kBlock, 0, st>>>(at, n, C, L, s->q.as<double>(), s->qs.as<double>());
                if (s->holds[slot_of(s, w)] != w) {
                    // rows not kept: listed again for the window's first positions, in its order
                    k_adj_to_f32<V><<<g, nd::kBlock, 0, st>>>(seg_at<T>(s, w * W), n, s->x32.as<float4>());
                    build_rows<V>(s, w, s->bin_mode, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
                }
                win = w;
            }
            k_adj_hvp<T><<<gr, nd::kBlock, 0, st>>>(rows_of(s, w), seg_at<T>(s, k - k0), s->qs.as<double>(), at, s->P,
                                                    L, k > 0 ? a2 : nullptr, k > 0 ? weight(k - 1) : 0.0,
                                                    s->dq.as<double>(), s->dpar.as<double>());
            ND_HIP(hipGetLastError());
            std::swap(L.a, a2);
        }
    }
    double *out = s->out.as<double>();
    k_adj_export<double4><<<g, nd::kBlock, 0, st>>>(L.x, at, n, out);
    k_adj_export<double4><<<g, nd::kBlock, 0, st>>>(L.v, at, n, out + 3 * (size_t)n);
    k_adj_sum_par<<<1, nd::kBlock, 0, st>>>(s->dpar.as<double>(), (int32_t)gr, out + 6 * (size_t)n);
    ND_HIP(hipGetLastError());
}

}  // namespace

extern "C" {

int nd_adj_create(nd_ctx *ctx, const nd_adj_params *p, nd_adj **out) {
    ND_API_BEGIN
    ND_REQUIRE(ctx && p && out, "nd_adj_create: null argument");
    *out = nullptr;
    ND_REQUIRE(p->n >= 8 && p->n % 4 == 0 && p->nsteps >= 1 && p->checkpoint_every >= 1 &&
                   p->rebuild_every >= 1,
               "nd_adj_create: n >= 8 and a multiple of 4; nsteps, checkpoint_every, rebuild_every >= 1");
    ND_REQUIRE(p->checkpoint_every % p->rebuild_every == 0,
               "nd_adj_create: checkpoint_every must be a multiple of rebuild_every");
    ND_REQUIRE(p->precision == ND_PREC_FP32 || p->precision == ND_PREC_FP64,
               "nd_adj_create: precision must be FP32 or FP64");
    ND_REQUIRE(p->nbins >= 1 && p->nbins <= kMaxBins && p->rdf_rmax > 0.0 && p->rdf_h > 0.0 &&
                   p->volume > 0.0,
               "nd_adj_create: 1..1024 RDF bins; range, kernel width and volume must be positive");
    ND_REQUIRE(p->dt > 0.0 && p->eps > 0.0 && p->sigma > 0.0 && p->rc > 0.0 && p->skin >= 0.0,
               "nd_adj_create: dt, eps, sigma, rc > 0 and skin >= 0");
    ND_HIP(hipSetDevice(ctx->device));
    nd_adj *s = new nd_adj();
    try {
        s->ctx = ctx;
        s->p = *p;
        s->dbl = p->precision == ND_PREC_FP64;
        const double reach = std::max(std::max(p->rc, p->rc_coul), p->rdf_rmax + p->rdf_h);
        // FP32 copies of the coordinates feed the list: pad by their rounding
        s->rlist = (float)((reach + p->skin) * (1.0 + 2.0e-6) + 1e-6);
        const size_t n = (size_t)p->n, vb = (s->dbl ? sizeof(double4) : sizeof(float4)) * n;
        const int32_t K = std::min(p->checkpoint_every, p->nsteps);
        const size_t nck = (size_t)((p->nsteps - 1) / p->checkpoint_every);  // all segments but the last
        // windows of a segment, then x_T's, then the spare order
        s->nwin = (K + p->rebuild_every - 1) / p->rebuild_every + 2;
        s->order.resize(s->nwin - 1);
        for (int32_t w = 0; w < s->nwin - 1; ++w) s->order[w] = w;
        s->spare = s->nwin - 1;
        for (nd::DevBuf *b : {&s->x0, &s->v0}) b->reserve(24 * n);
        for (nd::DevBuf *b : {&s->q, &s->qs, &s->dq}) b->reserve(8 * n);
        for (nd::DevBuf *b : {&s->xT, &s->tmp, &s->vel[0], &s->vel[1]}) b->reserve(vb);
        s->seg.reserve(vb * (size_t)K);
        s->ckx.reserve(vb * nck);
        s->ckv.reserve(vb * nck);
        s->ck_orig.reserve(4 * n * nck);
        s->orig.reserve(4 * n * (size_t)s->nwin);
        s->x32.reserve(sizeof(float4) * n);
        s->cpos.reserve(sizeof(float4) * n);
        s->ckey.reserve(4 * n);
        s->cell_of.reserve(sizeof(int2) * n);
        s->cells.reserve(4 * (size_t)(std::max(27, p->n / 2) + 1));
        s->bins.reserve(nd::cell_bins_bytes());
        s->lam.reserve(4 * sizeof(double4) * n);
        s->lam_caller.reserve(3 * sizeof(double4) * n);
        s->dpar.reserve(16 * (size_t)nd::grid_for((int64_t)n * kRowLanes));
        s->out.reserve(8 * (6 * n + 2));
        s->hist.reserve(8 * (2 + (size_t)p->nbins));  // flags, then the bins
        s->part.reserve(8 * (size_t)kHistBlocks * (size_t)p->nbins);
        s->wb.reserve(8 * (size_t)p->nbins);
        s->cap = 96;
        reserve_rows(s);
        // RDF normalisation: ideal-gas pair count in each bin's shell
        const double dr = p->rdf_rmax / p->nbins, npair = 0.5 * (double)p->n * (p->n - 1);
        s->norm.resize(p->nbins);
        for (int32_t b = 0; b < p->nbins; ++b) {
            const double rb = (b + 0.5) * dr;
            s->norm[b] = p->volume / (npair * 4.0 * M_PI * rb * rb * dr);
        }
        nd_adj_set_potential(s, p->eps, p->sigma);
    } catch (...) {
        nd_adj_destroy(s);
        throw;
    }
    *out = s;
    ND_API_END(ctx)
}

int nd_adj_destroy(nd_adj *s) {
    if (!s) return ND_OK;
    if (s->ctx) {
        (void)hipSetDevice(s->ctx->device);
        (void)hipStreamSynchronize(s->ctx->stream);
    }
    nd::DevBuf *bufs[] = {&s->x0, &s->v0, &s->q, &s->seg, &s->xT, &s->tmp, &s->x32, &s->vel[0], &s->vel[1], &s->qs,
                          &s->ckx, &s->ckv, &s->ck_orig, &s->lists, &s->lcnt, &s->orig, &s->bins, &s->cell_of,
                          &s->cells, &s->cpos, &s->ckey, &s->lam, &s->lam_caller, &s->dq, &s->dpar, &s->out,
                          &s->hist, &s->part, &s->wb};
    for (auto *b : bufs) b->release();
    delete s;
    return ND_OK;
}

int nd_adj_set_potential(nd_adj *s, double eps, double sigma) {
    nd_ctx *ctx = s ? s->ctx : nullptr;
    ND_API_BEGIN
    ND_REQUIRE(s && eps > 0.0 && sigma > 0.0, "nd_adj_set_potential: eps, sigma > 0");
    const nd_adj_params &p = s->p;
    AdjP &P = s->P;
    P.n = p.n;
    P.nbins = p.nbins;
    P.eps = eps;
    P.sigma = sigma;
    P.rc = p.rc;
    P.rc2 = p.rc * p.rc;
    P.kc = p.k_coul;
    P.rcc = p.rc_coul;
    P.rcc2 = p.rc_coul > 0.0 ? p.rc_coul * p.rc_coul : 0.0;
    P.sig2 = sigma * sigma;
    P.inv_eps = 1.0 / eps;
    P.inv_sigma = 1.0 / sigma;
    P.inv_rcc2 = p.rc_coul > 0.0 ? 1.0 / P.rcc2 : 0.0;
    P.dt = p.dt;
    P.c = 0.5 * p.dt;
    P.flj_rc = lj_F(p.rc, eps, sigma);
    P.glj_rc = lj_G(p.rc, eps, sigma);
    P.rmax = p.rdf_rmax;
    P.h = p.rdf_h;
    P.dr = p.rdf_rmax / p.nbins;
    s->have_forward = false;
    ND_API_END(ctx)
}

int nd_adj_forward(nd_adj *s, const double *h_x0, const double *h_v0, const double *h_q,
                   const double *h_target, double *h_rdf, double *h_loss) {
    nd_ctx *ctx = s ? s->ctx : nullptr;
    ND_API_BEGIN
    ND_REQUIRE(s && h_x0 && h_v0, "nd_adj_forward: null argument");
    ND_HIP(hipSetDevice(ctx->device));
    const size_t n = (size_t)s->p.n, m = 3 * n;
    hipStream_t st = ctx->stream;
    std::vector<double> q(n, 0.0);
    if (h_q) q.assign(h_q, h_q + n);
    ND_HIP(hipMemcpyAsync(s->q.p, q.data(), 8 * n, hipMemcpyHostToDevice, st));
    ND_HIP(hipMemcpyAsync(s->x0.p, h_x0, 8 * m, hipMemcpyHostToDevice, st));
    ND_HIP(hipMemcpyAsync(s->v0.p, h_v0, 8 * m, hipMemcpyHostToDevice, st));
    s->have_forward = false;
    s->target.clear();
    if (h_target) s->target.assign(h_target, h_target + s->p.nbins);
    if (s->dbl) forward_impl<double>(s);
    else forward_impl<float>(s);
    if (h_rdf) std::copy(s->rdf.begin(), s->rdf.end(), h_rdf);
    if (h_loss) *h_loss = s->loss;
    ND_API_END(ctx)
}

int nd_adj_final_state(nd_adj *s, double *h_x, double *h_v) {
    nd_ctx *ctx = s ? s->ctx : nullptr;
    ND_API_BEGIN
    ND_REQUIRE(s && s->have_forward, "nd_adj_final_state: run nd_adj_forward first");
    ND_HIP(hipSetDevice(ctx->device));
    const size_t m = 3 * (size_t)s->p.n;
    hipStream_t st = ctx->stream;
    const unsigned g = nd::grid_for(s->p.n);
    const int32_t *at = order_of(s, s->nwin - 2);
    double *out = s->out.as<double>();
    if (s->dbl) {
        k_adj_export<double4><<<g, nd::kBlock, 0, st>>>(s->xT.as<double4>(), at, s->p.n, out);
        k_adj_export<double4><<<g, nd::kBlock, 0, st>>>(s->vel[s->vcur].as<double4>(), at, s->p.n, out + m);
    } else {
        k_adj_export<float4><<<g, nd::kBlock, 0, st>>>(s->xT.as<float4>(), at, s->p.n, out);
        k_adj_export<float4><<<g, nd::kBlock, 0, st>>>(s->vel[s->vcur].as<float4>(), at, s->p.n, out + m);
    }
    ND_HIP(hipGetLastError());
    if (h_x) ND_HIP(hipMemcpyAsync(h_x, out, 8 * m, hipMemcpyDeviceToHost, st));
    if (h_v) ND_HIP(hipMemcpyAsync(h_v, out + m, 8 * m, hipMemcpyDeviceToHost, st));
    ND_HIP(hipStreamSynchronize(st));
    ND_API_END(ctx)
}

int nd_adj_backward(nd_adj *s, double *h_dx0, double *h_dv0, double *h_dq, double *h_dparams) {
    nd_ctx *ctx = s ? s->ctx : nullptr;
    ND_API_BEGIN
    ND_REQUIRE(s && s->have_forward && !s->target.empty(),
               "nd_adj_backward: run nd_adj_forward with a target first");
    ND_HIP(hipSetDevice(ctx->device));
    if (s->dbl) backward_impl<double>(s);
    else backward_impl<float>(s);
    hipStream_t st = ctx->stream;
    const size_t n = (size_t)s->p.n;
    const double *out = s->out.as<double>();
    if (h_dx0) ND_HIP(hipMemcpyAsync(h_dx0, out, 24 * n, hipMemcpyDeviceToHost, st));
    if (h_dv0) ND_HIP(hipMemcpyAsync(h_dv0, out + 3 * n, 24 * n, hipMemcpyDeviceToHost, st));
    if (h_dq) ND_HIP(hipMemcpyAsync(h_dq, s->dq.p, 8 * n, hipMemcpyDeviceToHost, st));
    if (h_dparams) ND_HIP(hipMemcpyAsync(h_dparams, out + 6 * n, 16, hipMemcpyDeviceToHost, st));
    ND_HIP(hipStreamSynchronize(st));
    // the recompute overwrote the final state: the forward must be rerun before another backward
    s->have_forward = false;
    ND_API_END(ctx)
}

}  // extern "C"
