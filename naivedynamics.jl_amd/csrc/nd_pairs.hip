// nd_pairs.hip -- pair searches over uniform cells: the counting and emitting
// passes of the cell list and of the one-call LBVH lists.
//
// Every listed pair lies within the radius, so cells of side >= r (and the 27
// around an atom's own) hold all of an atom's partners whatever order the
// atoms are sorted in.  A tree walk from a leaf depends on that order: with
// the reference's masked key every walk covers most of the tree (3.5 ms per
// pass for 65,536 points in the unit cube), and even with the interleaved key
// a leaf of four atoms that straddles an octree jump overlaps thousands of
// leaves (1.7-1.9 ms per pass for 262,144 points at liquid density).
//
// One wave takes 16 or 32 consecutive cell-sorted atoms, in groups that lie in
// up to k cells of one row along x (k so that k cells hold about two dozen
// atoms).  A group's candidates are the rows of cells around it, each row one
// contiguous run of the cell-sorted atoms; they are loaded once into registers
// (kBatches x 64 lanes), then tested against the group's atoms one after
// another, the query in scalar registers and a candidate per lane: no
// divergence, and a ballot gives the hits' places.  Waves take atoms, not
// cells, so crowded cells spread over many waves.
//
// VALU issue bounds both passes, so a test is three FMAs and three compares:
// with positions taken from a point c inside the group (a for the query, b for
// the candidate), |p - q|^2 = |b|^2 - 2 b.a + |a|^2, the candidate keeps (-2b,
// |b|^2) and the query its limits for the rest.  That sum differs from the
// reference's s by less than E = 16 u ((2|a| + r)^2 + r^2), u = 2^-24, for a
// pair near the radius (rounding a and b: 2 u (|a|+|b|)^2; the squares: 3 u
// each; the FMAs: 3 u (|a|+|b|)^2; the limit and s itself: 5 u r^2; |b| <= |a| +
// r there), and farther pairs' distances grow faster than their error while
// |a| < 1e5 r.  A test inside +-E of a limit is redone by the exact one (some
// 1e-5 of the tests), so the lists are the exact test's.  Where |a| or r leave
// the range of this bound, E is not a number, neither limit decides and every
// test is the exact one (|b|^2 may overflow there for a pair within the radius).
//
// Order.  The lists have to come in the order of a single-threaded reference
// run, which is by place in the key order ("slot") of the later atom, not by
// cell.  The emitting pass therefore ranks each atom's hits by slot in LDS
// (an atom has some dozens).  For leaves of more than one atom the reference
// interleaves the atoms of a query leaf tile by tile: k_merge_leaf places
// each hit by binary searches in the sorted lists of its leaf's other atoms.
// The leaf's pairs lie in one run of the output both before and after, so it
// works in place and no buffer of the list's size is needed.
//
// Exactness.  The test is the reference's: s = ((dx^2 + dy^2) + dz^2) below a
// threshold, which for the sqrt(s) < r form is the smallest float whose
// correctly rounded root reaches r.  A tree walk also wants the leaves' boxes
// to overlap (or the query to lie inside the leaf's box).  Coordinates closer
// than r by more than the rounding of x +- r/2 imply that; a pair within that
// rounding of the radius (s >= certain) is tested against the boxes
// themselves.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "nd_internal.hpp"

namespace {

using nd::wave_lds_sync;

// Candidates in registers, in batches of 64: enough for a group at liquid
// density (475-520 atoms in 27 cells of the list radius, some 270 in a half
// shell's 14); more take another round.
__host__ __device__ constexpr int batches(int kind, bool many) { return !many ? 3 : (kind == nd::kPairsHalf ? 6 : 10); }
constexpr int kQueue = 512;  // hits a group may hold in LDS
constexpr int kWaves = nd::kBlock / 64;

struct PairArgs {
    const float4 *cpos;     // cell-sorted (x, y, z, slot); half shell: (x, y, z, input index)
    const float *xyz;       // positions by slot (lists over a tree)
    const int32_t *ckey;    // cell of each cell-sorted atom (ncell: none)
    const int32_t *cstart;  // ncell + 1
    nd::CellGrid cg;
    int32_t k, per_wave, many, n, apl;
    float thr, certain, r;
    const nd_node *nodes;   // leaf boxes (lists over a tree)
    const int32_t *idx;     // input index of each slot (lists over a tree)
    int64_t *counts;        // per slot (half shell: per cell-sorted place)
    const int64_t *offsets;
    int32_t *maxcnt;
    nd_pair *out;
    int32_t cap;            // hits a wave holds in LDS
};

__device__ __forceinline__ float lane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ int32_t lane_i(int32_t v, int l) { return __builtin_amdgcn_readlane(v, l); }

// The walk's own test for a pair at the edge of the radius: leaf boxes that
// overlap (strictly, all axes), or a query strictly inside the later leaf's box.
template <int KIND>
__device__ bool box_test(const PairArgs &A, int32_t sq, float qx, float qy, float qz, int32_t sc) {
    const int32_t tq = sq / A.apl, tc = sc / A.apl;
    const nd_node &c = A.nodes[tc];
    if (KIND == nd::kPairsLeaf) {
        if (tq == tc) return true;  // pairs inside a leaf see no box
        const nd_node &q = A.nodes[tq];
        return (q.min[0] < c.max[0]) & (q.max[0] > c.min[0]) & (q.min[1] < c.max[1]) & (q.max[1] > c.min[1]) &
               (q.min[2] < c.max[2]) & (q.max[2] > c.min[2]);
    }
    return (c.min[0] < qx) & (qx < c.max[0]) & (c.min[1] < qy) & (qy < c.max[1]) & (c.min[2] < qz) &
           (qz < c.max[2]);
}

template <int KIND, bool EMIT, bool MANY>
__global__ void __launch_bounds__(nd::kBlock)
k_cell_search(PairArgs A) {
    constexpr bool HALF = KIND == nd::kPairsHalf;
    constexpr int ROWS = HALF ? 5 : 9, kBatches = batches(KIND, MANY);
    // per wave: cap hits' places or slots, squared distances, queries
    extern __shared__ __align__(16) int32_t s_hits[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int32_t *hkey = s_hits + (size_t)w * 2 * A.cap;
    float *hs = reinterpret_cast<float *>(hkey + A.cap);
    uint8_t *hq = reinterpret_cast<uint8_t *>(s_hits + (size_t)kWaves * 2 * A.cap) + (size_t)w * A.cap;
    const int32_t t0 = __builtin_amdgcn_readfirstlane(((int32_t)blockIdx.x * kWaves + w) * A.per_wave);
    if (t0 >= A.n) return;
    const int32_t nt = min(A.per_wave, A.n - t0);
    const int32_t g0 = A.cg.g[0], g1 = A.cg.g[1], g2 = A.cg.g[2];
    // lane q holds atom t0 + q: cell, position, filter word, place of its count
    float px = 0.0f, py = 0.0f, pz = 0.0f;
    int32_t pk = A.cg.ncell, pf = 0, pslot = 0, pid = 0;
    int64_t off = 0;
    int32_t lim = 0;  // its hits (emitting)
    if (lane < nt) {
        const float4 p = A.cpos[t0 + lane];
        px = p.x;
        py = p.y;
        pz = p.z;
        pk = A.ckey[t0 + lane];
        pid = __float_as_int(p.w);
        pslot = HALF ? t0 + lane : pid;
        pf = KIND == nd::kPairsPointRoot ? A.idx[pslot] : pslot;
        if (EMIT) {
            off = A.offsets[pslot];
            lim = (int32_t)(A.offsets[pslot + 1] - off);
            if (!HALF) pid = (KIND == nd::kPairsLeaf && A.apl > 1) ? pslot : A.idx[pslot];
        }
    }
    int32_t found = 0;  // lane q: hits of query q so far
    // lane q: the LDS room of query q's hits (emitting): consecutive, in whole
    // fours where they are going to be ranked
    int32_t room = HALF ? lim : (lim + 3) & ~3, end = room;
    if (EMIT)
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t v = __shfl_up(end, o, 64);
            if (lane >= o) end += v;
        }
    const int32_t prow = pk / g0;
    // position of a candidate (place or slot)
    auto atom = [&](int32_t h) -> float3 {
        if constexpr (HALF) {
            const float4 c = A.cpos[h];
            return make_float3(c.x, c.y, c.z);
        } else {
            const float *c = A.xyz + 3 * (int64_t)h;
            return make_float3(c[0], c[1], c[2]);
        }
    };
    int32_t q0 = 0;
    while (q0 < nt) {
        // the group: atoms from q0 on in the next k cells of the same row,
        // and (emitting) as many as have room for their hits
        const int32_t k0 = lane_i(pk, q0), row = lane_i(prow, q0);
        if (k0 >= A.cg.ncell) break;  // atoms in no cell (a non-finite coordinate) pair with none
        const int32_t base = EMIT ? lane_i(end, q0) - lane_i(room, q0) : 0;  // LDS place 0 of the group
        const uint64_t in = __builtin_amdgcn_ballot_w64(lane >= q0 && lane < nt && prow == row && pk < k0 + A.k &&
                                                        (!EMIT || lane == q0 || end - base <= A.cap));
        const int32_t q1 = q0 + __builtin_popcountll(in);
        const int32_t held = EMIT ? lane_i(end, q1 - 1) - base : 0;  // LDS places of the group
        // more hits than LDS holds (half shell, one atom): straight to memory
        const bool direct = EMIT && held > A.cap;
        const int32_t c0 = k0 - row * g0, c1 = lane_i(pk, q1 - 1) - row * g0;
        const int32_t cy = row % g1, cz = row / g1;
        // candidate rows: lane j holds row j's run; the runs are read as one
        // sequence
        int32_t start = 0, len = 0;
        if (lane < ROWS) {
            int32_t dy, dz;
            if (HALF) {  // own row, the next row, the three rows of the next layer
                dy = lane == 0 ? 0 : (lane == 1 ? 1 : lane - 3);
                dz = lane < 2 ? 0 : 1;
            } else {
                dy = lane % 3 - 1;
                dz = lane / 3 - 1;
            }
            const int32_t y = cy + dy, z = cz + dz;
            if (y >= 0 && y < g1 && z >= 0 && z < g2) {
                const int32_t b = (z * g1 + y) * g0;
                start = HALF && lane == 0 ? t0 + q0 + 1 : A.cstart[b + max(c0 - 1, 0)];
                len = A.cstart[b + min(c1 + 1, g0 - 1) + 1] - start;
            }
        }
        // lane j: candidates before row j, and its start less those
        int32_t pre = len;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int32_t v = __shfl_up(pre, o, 64);
            if (lane >= o) pre += v;
        }
        const int32_t total = lane_i(pre, ROWS - 1);
        pre -= len;
        const int32_t rise = start - pre;
        const int mid = (q0 + q1) >> 1;
        const float ox = lane_f(px, mid), oy = lane_f(py, mid), oz = lane_f(pz, mid);
        // lane q's limits: below lo a candidate is a pair, from hi on it is none
        const float ax = px - ox, ay = py - oy, az = pz - oz;
        const float a2 = __builtin_fmaf(az, az, __builtin_fmaf(ay, ay, ax * ax));
        const float reach = 2.0f * sqrtf(a2) + A.r;
        const bool bound = A.r >= 1e-15f && A.r <= 1e12f && reach < 1e5f * A.r;
        const float E = bound ? 1.2e-6f * (reach * reach + A.r * A.r) : NAN;
        const float lo = (A.certain - a2) - E, hi = (A.thr - a2) + E;
        int32_t row_at = 0;  // row of the next batch's first candidate, or one before it
        for (int32_t s0 = 0; s0 < total; s0 += 64 * kBatches) {
            // candidates s0 + 64 b + lane (past the end: a copy that the
            // filter drops), the order word of the filter -- the place (every
            // row of the half shell but the own one lies after the group),
            // the slot or the input index -- and the place or slot
            float bx[kBatches], by[kBatches], bz[kBatches], bw[kBatches];
            int32_t bf[kBatches], bslot[kBatches];
#pragma unroll
            for (int b = 0; b < kBatches; ++b) {
                const int32_t ci = s0 + 64 * b + lane;
                const bool ok = ci < total;
                // the rows that begin before the batch's last candidate
                int32_t u = ci + lane_i(rise, row_at);
                while (row_at + 1 < ROWS) {
                    const int32_t p = lane_i(pre, row_at + 1);
                    if (p > s0 + 64 * b + 63) break;
                    ++row_at;
                    u = ci >= p ? ci + lane_i(rise, row_at) : u;
                }
                const float4 c = A.cpos[ok ? u : t0];
                const float x = c.x - ox, y = c.y - oy, z = c.z - oz;
                bx[b] = -2.0f * x;
                by[b] = -2.0f * y;
                bz[b] = -2.0f * z;
                bw[b] = __builtin_fmaf(z, z, __builtin_fmaf(y, y, x * x));
                bslot[b] = HALF ? u : __float_as_int(c.w);
                bf[b] = KIND == nd::kPairsPointRoot ? A.idx[bslot[b]] : bslot[b];
                if (!ok) bf[b] = INT32_MIN;
            }
            for (int32_t q = q0; q < q1; ++q) {
                const float sx = lane_f(ax, q), sy = lane_f(ay, q), sz = lane_f(az, q);
                const float slo = lane_f(lo, q), shi = lane_f(hi, q);
                const int32_t qf = lane_i(pf, q);
                // the next hit's LDS place (or, direct, its number)
                int32_t H = lane_i(found, q);
                const int32_t H0 = H, shift = EMIT && !direct ? lane_i(end, q) - lane_i(room, q) - base : 0;
#pragma unroll
                for (int b = 0; b < kBatches; ++b) {
                    if (s0 + 64 * b >= total) continue;
                    const float t = __builtin_fmaf(bx[b], sx, __builtin_fmaf(by[b], sy, __builtin_fmaf(bz[b], sz, bw[b])));
                    const uint64_t after = __builtin_amdgcn_ballot_w64(bf[b] > qf);
                    uint64_t m = __builtin_amdgcn_ballot_w64(t < slo) & after;
                    const uint64_t open = __builtin_amdgcn_ballot_w64(!(t >= shi)) & after & ~m;
                    if (open) {
                        const float qx = lane_f(px, q), qy = lane_f(py, q), qz = lane_f(pz, q);
                        const int32_t qslot = lane_i(pslot, q);
                        bool in = false;
                        if (__builtin_amdgcn_inverse_ballot_w64(open)) {
                            // opaque to the compiler, which would hoist this
                            // rare branch's addresses and divisions out of
                            // the loop and keep them in registers
                            int32_t sl = bslot[b];
                            asm volatile("" : "+v"(sl));
                            const float3 c = atom(sl);
                            const float s = nd::sqdist(qx, qy, qz, c.x, c.y, c.z);
                            in = s < A.thr;
                            if (!HALF) {
                                if (in && !(s < A.certain)) in = box_test<KIND>(A, qslot, qx, qy, qz, sl);
                            }
                        }
                        m |= __builtin_amdgcn_ballot_w64(in);
                    }
                    if (EMIT) {
                        if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                            const int32_t at = (int32_t)__builtin_amdgcn_mbcnt_hi(
                                (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)(shift + H)));
                            if (!HALF || !direct) {
                                if (at < A.cap) {
                                    hkey[at] = bslot[b];
                                    hq[at] = (uint8_t)q;
                                }
                            } else if (at < held) {
                                int32_t sl = bslot[b];
                                asm volatile("" : "+v"(sl));
                                const float4 c = A.cpos[sl];
                                const int32_t id = __float_as_int(c.w), qi = lane_i(pid, q0);
                                const int64_t o = ((int64_t)lane_i((int32_t)(off >> 32), q0) << 32) |
                                                  (uint32_t)lane_i((int32_t)off, q0);
                                nd_pair p;
                                p.i = min(qi, id);
                                p.j = max(qi, id);
                                p.d = sqrtf(nd::sqdist(lane_f(px, q0), lane_f(py, q0), lane_f(pz, q0), c.x, c.y, c.z));
                                A.out[o + at] = p;
                            }
                        }
                    }
                    H += __builtin_popcountll(m);
                }
                if (H != H0) found = lane == q ? H : found;
            }
        }
        if (EMIT && !direct && held > 0) {
            if (!HALF && lane >= q0 && lane < q1)
                for (int32_t e = lim; e < room; ++e) hq[end - room - base + e] = 0xFF;  // fill of the last four
            wave_lds_sync();
            const int64_t orun = ((int64_t)lane_i((int32_t)(off >> 32), q0) << 32) | (uint32_t)lane_i((int32_t)off, q0);
            constexpr int U = 4;  // gathers in flight per lane
            for (int32_t e0 = 0; e0 < held; e0 += 64 * U) {
                int32_t q[U], h[U];
                float3 c[U];
                int32_t other[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int32_t e = e0 + 64 * u + lane;
                    q[u] = e < held ? (int32_t)hq[e] : 0xFF;
                    h[u] = q[u] != 0xFF ? hkey[e] : 0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if constexpr (HALF) {
                        const float4 v = A.cpos[h[u]];
                        c[u] = make_float3(v.x, v.y, v.z);
                        other[u] = __float_as_int(v.w);
                    } else {
                        c[u] = atom(h[u]);
                        other[u] = h[u];
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    // all lanes take part in the shuffles
                    const int32_t e = e0 + 64 * u + lane, ql = q[u] & 63;
                    const float s = nd::sqdist(__shfl(px, ql, 64), __shfl(py, ql, 64), __shfl(pz, ql, 64), c[u].x,
                                               c[u].y, c[u].z);
                    if constexpr (HALF) {
                        // consecutive atoms' pairs are one run of the output
                        const int32_t qi = __shfl(pid, ql, 64);
                        if (q[u] != 0xFF) {
                            nd_pair p;
                            p.i = min(qi, other[u]);
                            p.j = max(qi, other[u]);
                            p.d = sqrtf(s);
                            A.out[orun + e] = p;
                        }
                    } else {
                        if (q[u] != 0xFF) hs[e] = s;
                        else if (e < held) hkey[e] = INT32_MAX;
                    }
                }
            }
            if constexpr (!HALF) {
                // each hit at the rank of its slot among its query's
                wave_lds_sync();
                const int32_t qbase = end - room - base;
                for (int32_t e0 = 0; e0 < held; e0 += 64) {
                    const int32_t e = e0 + lane;
                    const int32_t q = e < held ? (int32_t)hq[e] : 0xFF;
                    const int32_t b = __shfl(qbase, q & 63, 64), qi = __shfl(pid, q & 63, 64);
                    const int32_t m = __shfl(lim, q & 63, 64);
                    const int64_t o = ((int64_t)__shfl((int32_t)(off >> 32), q & 63, 64) << 32) |
                                      (uint32_t)__shfl((int32_t)off, q & 63, 64);
                    if (q == 0xFF) continue;
                    const int32_t key = hkey[e];
                    int32_t r = 0;
                    for (int32_t t = b; t < b + m; t += 4) {
                        const int4 v = *reinterpret_cast<const int4 *>(hkey + t);
                        r += (v.x < key) + (v.y < key) + (v.z < key) + (v.w < key);
                    }
                    nd_pair p;
                    p.i = qi;
                    // leaves of several atoms: slots, until k_merge_leaf
                    p.j = (KIND == nd::kPairsLeaf && A.apl > 1) ? key : A.idx[key];
                    p.d = sqrtf(hs[e]);
                    if (r < m) A.out[o + r] = p;
                }
            }
            wave_lds_sync();
        }
        q0 = q1;
    }
    if (!EMIT) {
        if (lane < nt) A.counts[pslot] = found;
        if (A.maxcnt) {
            int32_t mx = found;
            for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
            // the largest count only grows: most waves see it is not theirs
            if (lane == 0 && mx > __hip_atomic_load(A.maxcnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(A.maxcnt, mx);
        }
    }
}

// Pairs of query leaf q in out[offsets[q apl] .. offsets[(q + 1) apl]), atom by
// atom, each atom's by slot and as (slot, slot, d), into the reference's order:
// later leaf t first, then the query leaf's atom a, then t's atom.  Before the
// pair (a, t, b) come, of each other atom's list, the pairs with leaves before
// t, and with t itself for atoms before a.  NT threads per leaf: a wave, or a
// workgroup where a leaf's pairs are many.
template <int NT>
__global__ void __launch_bounds__(nd::kBlock)
k_merge_leaf(const int64_t *__restrict__ offsets, const int32_t *__restrict__ idx, int32_t nL, int32_t apl,
             int32_t cap, nd_pair *__restrict__ out) {
    extern __shared__ __align__(16) int32_t s_merge[];  // per leaf: apl + 1 offsets, cap x (slot, atom, d)
    const int32_t g = threadIdx.x / NT, t0 = threadIdx.x % NT;
    const int32_t q = (int32_t)blockIdx.x * (nd::kBlock / NT) + g;
    int32_t *loff = s_merge + (size_t)g * (apl + 1 + 3 * cap);
    int32_t *key = loff + apl + 1, *atom = key + cap;
    float *dist = reinterpret_cast<float *>(atom + cap);
    const int64_t seg = q < nL ? offsets[(int64_t)q * apl] : 0;
    const int32_t H = q < nL ? (int32_t)min((int64_t)cap, offsets[(int64_t)(q + 1) * apl] - seg) : 0;
    if (q < nL) {
        for (int32_t a = t0; a <= apl; a += NT) loff[a] = (int32_t)(offsets[(int64_t)q * apl + a] - seg);
        for (int32_t e = t0; e < H; e += NT) {
            const nd_pair p = out[seg + e];
            key[e] = p.j;
            atom[e] = p.i - q * apl;
            dist[e] = p.d;
        }
    }
    // everything is read before anything is written
    if constexpr (NT == 64) wave_lds_sync();
    else __syncthreads();
    for (int32_t e = t0; e < H; e += NT) {
        const int32_t sc = key[e], a = atom[e], first = sc / apl * apl;
        int32_t r = e - loff[a];
        for (int32_t b = 0; b < apl; ++b) {
            if (b == a) continue;
            const int32_t want = first + (b < a ? apl : 0);
            const int32_t lo = loff[b];
            int32_t x = lo, y = min(loff[b + 1], H);
            while (x < y) {
                const int32_t m = (x + y) >> 1;
                if (key[m] < want) x = m + 1;
                else y = m;
            }
            r += x - lo;
        }
        nd_pair p;
        p.i = idx[(int64_t)q * apl + a];
        p.j = idx[sc];
        p.d = dist[e];
        if (r < H) out[seg + r] = p;
    }
}

// ---- keys, cells and their counts for a list over a tree ----

// Keys' bits that vary, cells' crowding and the grid, for the host's one
// decision before the sort.
struct Prep {
    nd::BinGrid grid;
    int32_t stretched;  // cells larger than they need to be, or atoms outside the grid
    float certain;
    int32_t status;
    uint32_t key_or, key_and;
    uint64_t sum_sq;  // sum over cells of (atoms in it)^2
};

constexpr int kBoxBlocks = 256;
constexpr int kTileCells = 2048;  // cells per workgroup of the scan
constexpr int kMaxCells = 1 << 20;

__device__ __forceinline__ int32_t wave_min(int32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int32_t wave_max(int32_t v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int32_t f2ord(float f) {
    const int32_t i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7FFFFFFF;
}
__device__ __forceinline__ float ord2f(int32_t i) { return __int_as_float(i >= 0 ? i : i ^ 0x7FFFFFFF); }

// Positions as (x, y, z) triples or as float4.
struct Xyz3 {
    const float *p;
    __device__ __forceinline__ float3 operator()(int32_t i) const {
        return make_float3(p[3 * (int64_t)i], p[3 * (int64_t)i + 1], p[3 * (int64_t)i + 2]);
    }
};
struct Xyz4 {
    const float4 *p;
    __device__ __forceinline__ float3 operator()(int32_t i) const {
        const float4 v = p[i];
        return make_float3(v.x, v.y, v.z);
    }
};

// One workgroup's part of the bounding box (as ordered ints) and of the sums.
struct BoxPart {
    int32_t mn[3], mx[3];
    double sum[3], sq[3];
};

// Per-workgroup bounding boxes and sums of the finite coordinates (ATOMS: of
// the atoms whose three coordinates are finite).  No atomics: 64 workgroups' on
// six words took 21-29 us, these and the launch that joins them take 6 + 4.
// Also clears the cell counts and two words.
template <bool ATOMS, class SRC>
__global__ void __launch_bounds__(nd::kBlock)
k_prep_boxes(SRC xyz, int32_t n, BoxPart *__restrict__ part, int32_t *__restrict__ cells, int32_t ncells,
             int32_t *__restrict__ status, int32_t *__restrict__ maxcnt) {
    __shared__ BoxPart s[kWaves];
    const int32_t t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (int32_t c = t; c < ncells; c += stride) cells[c] = 0;
    if (t == 0) {
        *status = 0;
        *maxcnt = 0;
    }
    int32_t mn[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, mx[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
    double sum[3] = {0.0, 0.0, 0.0}, sq[3] = {0.0, 0.0, 0.0};
    for (int32_t i = t; i < n; i += stride) {
        const float3 p = xyz(i);
        const float v[3] = {p.x, p.y, p.z};
        const bool all = __builtin_isfinite(v[0]) & __builtin_isfinite(v[1]) & __builtin_isfinite(v[2]);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (!(ATOMS ? all : __builtin_isfinite(v[d]))) continue;
            mn[d] = min(mn[d], f2ord(v[d]));
            mx[d] = max(mx[d], f2ord(v[d]));
            sum[d] += (double)v[d];
            sq[d] += (double)v[d] * (double)v[d];
        }
    }
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        mn[d] = wave_min(mn[d]);
        mx[d] = wave_max(mx[d]);
        for (int o = 32; o > 0; o >>= 1) {
            sum[d] += __shfl_xor(sum[d], o, 64);
            sq[d] += __shfl_xor(sq[d], o, 64);
        }
        if ((threadIdx.x & 63) == 0) {
            s[w].mn[d] = mn[d];
            s[w].mx[d] = mx[d];
            s[w].sum[d] = sum[d];
            s[w].sq[d] = sq[d];
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int d = threadIdx.x;
        BoxPart &q = part[blockIdx.x];
        for (int k = 1; k < kWaves; ++k) {
            s[0].mn[d] = min(s[0].mn[d], s[k].mn[d]);
            s[0].mx[d] = max(s[0].mx[d], s[k].mx[d]);
            s[0].sum[d] += s[k].sum[d];
            s[0].sq[d] += s[k].sq[d];
        }
        q.mn[d] = s[0].mn[d];
        q.mx[d] = s[0].mx[d];
        q.sum[d] = s[0].sum[d];
        q.sq[d] = s[0].sq[d];
    }
}

// The joined box, for the host (thread d < 6: word d).
__global__ void __launch_bounds__(64)
k_box_result(const BoxPart *__restrict__ part, int32_t nparts, int32_t *__restrict__ host) {
    for (int d = 0; d < 3; ++d) {
        int32_t a = INT32_MAX, b = INT32_MIN;
        for (int32_t t = threadIdx.x; t < nparts; t += 64) {
            a = min(a, part[t].mn[d]);
            b = max(b, part[t].mx[d]);
        }
        a = wave_min(a);
        b = wave_max(b);
        if (threadIdx.x == 0) {
            host[d] = a;
            host[3 + d] = b;
        }
    }
}

// The box of the interleaved key (lo, 1024 / extent, as launch_bbox computes
// it), the cell grid, and the squared distance below which a pair passes the
// walk's box test whatever its leaves' boxes are: coordinates within r less
// two units in the last place of the largest coordinate +- r keep their order
// after rounding x +- r/2 (or x +- r).
//
// The grid spans four standard deviations around the mean where that is less
// than the bounding box: coordinates outside go to the edge cells, which keeps
// atoms within a cell's side in neighbouring cells, and a few outliers do not
// stretch the cells of all others (far clusters do: the lists over a tree walk it
// then, the adjoint's take lines).
__global__ void __launch_bounds__(nd::kBlock)
k_prep_grid(const BoxPart *__restrict__ part, int32_t nparts, int32_t n, float r, float thr, int32_t max_cells,
            float *__restrict__ box, Prep *__restrict__ prep) {
    __shared__ BoxPart s[kWaves];
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int32_t a = INT32_MAX, b = INT32_MIN;
        double u = 0.0, v = 0.0;
        for (int32_t t = threadIdx.x; t < nparts; t += nd::kBlock) {
            a = min(a, part[t].mn[d]);
            b = max(b, part[t].mx[d]);
            u += part[t].sum[d];
            v += part[t].sq[d];
        }
        a = wave_min(a);
        b = wave_max(b);
        for (int o = 32; o > 0; o >>= 1) {
            u += __shfl_xor(u, o, 64);
            v += __shfl_xor(v, o, 64);
        }
        if ((threadIdx.x & 63) == 0) {
            s[w].mn[d] = a;
            s[w].mx[d] = b;
            s[w].sum[d] = u;
            s[w].sq[d] = v;
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    nd::CellGrid cg;
    int64_t g[3];
    double lo[3], ext[3];
    float most = 0.0f;
    bool stretched = false;
    const double side = (double)r * (1.0 + 1e-4);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int32_t a = s[0].mn[d], b = s[0].mx[d];
        double u = s[0].sum[d], v = s[0].sq[d];
        for (int k = 1; k < kWaves; ++k) {
            a = min(a, s[k].mn[d]);
            b = max(b, s[k].mx[d]);
            u += s[k].sum[d];
            v += s[k].sq[d];
        }
        const float l = ord2f(a), h = ord2f(b), e = h - l;
        if (box) {
            box[d] = l;
            box[3 + d] = e > 0.0f ? 1024.0f / e : 0.0f;
        }
        const double mean = u / n, dev = 4.0 * sqrt(fmax(v / n - mean * mean, 0.0));
        lo[d] = fmax((double)l, mean - dev);
        ext[d] = a <= b ? fmin((double)h, mean + dev) - lo[d] : 0.0;
        const double q = ext[d] > 0.0 ? floor(ext[d] / side) : 1.0;
        g[d] = q >= 1.0 ? (q > 1024.0 ? 1024 : (int64_t)q) : 1;
        stretched |= q > 1024.0 || (a <= b && ((double)l < lo[d] || lo[d] + ext[d] < (double)h));
        if (a <= b) most = fmaxf(most, fmaxf(fabsf(l), fabsf(h)));
    }
    while (g[0] * g[1] * g[2] > max_cells) {
        stretched = true;
        const double f = cbrt((double)max_cells / (double)(g[0] * g[1] * g[2]));
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int64_t c = (int64_t)floor((double)g[d] * f);
            g[d] = c < 1 ? 1 : c;
        }
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        cg.lo[d] = lo[d];
        cg.g[d] = (int32_t)g[d];
        cg.inv[d] = ext[d] > 0.0 ? (double)g[d] / ext[d] : 0.0;
    }
    cg.ncell = (int32_t)(g[0] * g[1] * g[2]);
    prep->grid.cg = cg;
    prep->grid.lines = 0;
    prep->grid.tests = 0ull;
    prep->grid.inv = 1.0 / side;
    prep->stretched = stretched;
    const double in = (double)r * (1.0 - 0x1p-20) - 0x1p-22 * ((double)most + (double)r);
    prep->certain = in > 0.0 ? fminf((float)(in * in * (1.0 - 0x1p-20)), thr) : -1.0f;
}

// Counts an atom in cell c; returns its place among the cell's atoms.  A wave's
// atoms of one cell are counted together while the cells are crowded (131,072
// atoms of eight cells took 1 ms of atomics on their words); the first cell
// that few lanes share ends that.
__device__ __forceinline__ int32_t count_in_cell(int32_t *cells, int32_t c) {
    const int lane = threadIdx.x & 63;
    int32_t place = -1;
    while (place < 0) {
        const uint64_t same = __builtin_amdgcn_ballot_w64(c == __builtin_amdgcn_readfirstlane(c));
        if (__builtin_popcountll(same) < 4) break;
        if ((same >> lane) & 1ull) {
            const int first = __builtin_ctzll(same);
            int32_t b = 0;
            if (lane == first) b = atomicAdd(&cells[c], __builtin_popcountll(same));
            place = __builtin_amdgcn_readlane(b, first) + __builtin_popcountll(same & ((1ull << lane) - 1ull));
        }
    }
    return place < 0 ? atomicAdd(&cells[c], 1) : place;
}

__device__ __forceinline__ int32_t cell_index(const nd::CellGrid &cg, float x, float y, float z) {
    return (nd::cell_coord(cg, z, 2) * cg.g[1] + nd::cell_coord(cg, y, 1)) * cg.g[0] + nd::cell_coord(cg, x, 0);
}

// Lines without a look at the atoms' box.
__global__ void k_line_grid(float r, int32_t lines, Prep *__restrict__ prep) {
    prep->grid.lines = lines;
    prep->grid.tests = 0ull;
    prep->grid.inv = 1.0 / ((double)r * (1.0 + 1e-4));
}

// Cell and place of every atom.
__global__ void __launch_bounds__(nd::kBlock)
k_bin_atoms(const float4 *__restrict__ x, int32_t n, const Prep *__restrict__ prep, int32_t *__restrict__ cells,
            int2 *__restrict__ cell_of, int32_t *__restrict__ status) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x, lines = prep->grid.lines;
    if (i >= n) return;
    const float4 p = x[i];
    if (!(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z)))
        atomicOr(status, nd::kStatusDomain);
    int32_t c;
    if (lines) {
        const double inv = prep->grid.inv;
        c = nd::line_cell(nd::line_coord(inv, p.x), nd::line_coord(inv, p.y), nd::line_coord(inv, p.z), lines);
    } else {
        c = cell_index(prep->grid.cg, p.x, p.y, p.z);
    }
    cell_of[i] = make_int2(c, count_in_cell(cells, c));
}

// Key and cell of every atom, and the atom's place among its cell's (by an
// atomic count: in any order, the emitting pass sorts).  kb[2 b], kb[2 b + 1]:
// or and and of workgroup b's keys.
template <bool MASKED>
__global__ void __launch_bounds__(nd::kBlock)
k_prep_keys(const float *__restrict__ xyz, int32_t n, const float *__restrict__ box, const Prep *__restrict__ prep,
            int32_t *__restrict__ codes, int32_t *__restrict__ perm, int32_t *__restrict__ cells,
            int2 *__restrict__ cell_of, uint32_t *__restrict__ kb, int32_t *__restrict__ status) {
    __shared__ uint32_t so, sa;
    if (threadIdx.x == 0) {
        so = 0u;
        sa = 0xFFFFFFFFu;
    }
    __syncthreads();
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float x = xyz[3 * (int64_t)i], y = xyz[3 * (int64_t)i + 1], z = xyz[3 * (int64_t)i + 2];
        bool ok;
        const int32_t code = MASKED ? nd::masked_key(x, y, z, ok) : nd::interleaved_key(x, y, z, box, ok);
        codes[i] = code;
        perm[i] = i;
        if (!ok) atomicOr(status, nd::kStatusDomain);
        const int32_t c = cell_index(prep->grid.cg, x, y, z);
        const int32_t place = count_in_cell(cells, c);
        cell_of[i] = make_int2(c, place);
        const uint32_t k = (uint32_t)code ^ 0x80000000u;
        atomicOr(&so, k);
        atomicAnd(&sa, k);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        kb[2 * blockIdx.x] = so;
        kb[2 * blockIdx.x + 1] = sa;
    }
}

__device__ __forceinline__ int32_t table_cells(const nd::BinGrid &g) { return g.lines ? g.lines : g.cg.ncell; }

// Atoms in the cells around cell c of a box, itself included.
__device__ __forceinline__ int32_t atoms_around(const int32_t *__restrict__ cells, const nd::CellGrid &cg, int32_t c) {
    const int32_t g0 = cg.g[0], g1 = cg.g[1], g2 = cg.g[2];
    const int32_t x = c % g0, y = c / g0 % g1, z = c / g0 / g1;
    int32_t sum = 0;
#pragma unroll
    for (int k = 0; k < 27; ++k) {  // every load in flight
        const int32_t u = x + k % 3 - 1, v = y + k / 3 % 3 - 1, w = z + k / 9 - 1;
        const bool in = (uint32_t)u < (uint32_t)g0 && (uint32_t)v < (uint32_t)g1 && (uint32_t)w < (uint32_t)g2;
        const int32_t there = cells[in ? (w * g1 + v) * g0 + u : c];
        sum += in ? there : 0;
    }
    return sum;
}

// Sum and sum of squares of each tile of cell counts.  COUNT: where the cells are
// larger than they need to be, also the pairs of atoms in the same or
// neighbouring cells, all tiles' together.
template <bool COUNT>
__global__ void __launch_bounds__(nd::kBlock)
k_cell_tiles(const int32_t *__restrict__ cells, const Prep *__restrict__ prep, int32_t *__restrict__ tsum,
             uint64_t *__restrict__ tsq, double few, unsigned long long *__restrict__ tests) {
    __shared__ int32_t s1[kWaves];
    __shared__ uint64_t s2[kWaves];
    const int32_t ncell = table_cells(prep->grid), base = blockIdx.x * kTileCells;
    if (base >= ncell) return;
    int32_t a = 0;
    uint64_t b = 0;
    for (int32_t k = threadIdx.x; k < kTileCells && base + k < ncell; k += nd::kBlock) {
        const int32_t c = cells[base + k];
        a += c;
        b += (uint64_t)c * (uint64_t)c;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        s1[threadIdx.x >> 6] = a;
        s2[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kWaves; ++k) {
            a += s1[k];
            b += s2[k];
        }
        tsum[blockIdx.x] = a;
        tsq[blockIdx.x] = b;
    }
    if constexpr (COUNT) {
        // 27 sum c^2 bounds the pairs: tiles below `few` an atom are left out (the
        // look around costs 20 us, a gas has nothing to gain from it)
        __shared__ int32_t look;
        if (threadIdx.x == 0) look = prep->stretched && 27.0 * (double)b > few * (double)a;
        __syncthreads();
        if (look == 0) return;
        unsigned long long t = 0ull;
        for (int32_t k = threadIdx.x; k < kTileCells && base + k < ncell; k += nd::kBlock)
            if (const int32_t c = cells[base + k]; c > 0)
                t += (unsigned long long)c * (unsigned long long)atoms_around(cells, prep->grid.cg, base + k);
        for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if ((threadIdx.x & 63) == 0 && t > 0ull) atomicAdd(tests, t);
    }
}

// First place of each cell (in place over the counts: cells[ncell] = n); the
// first workgroup also joins the key bits and hands the host its Prep.
__global__ void __launch_bounds__(nd::kBlock)
k_cell_starts(int32_t *__restrict__ cells, int32_t n, const Prep *__restrict__ prep, const int32_t *__restrict__ tsum,
              const uint64_t *__restrict__ tsq, const uint32_t *__restrict__ kb, int32_t nkb,
              const int32_t *__restrict__ status, Prep *__restrict__ host) {
    __shared__ int32_t part[nd::kBlock];
    const int32_t ncell = table_cells(prep->grid), base = blockIdx.x * kTileCells, t = threadIdx.x;
    if (base >= ncell) return;
    // atoms before this tile
    int32_t before = 0;
    for (int32_t k = t; k < (int32_t)blockIdx.x; k += nd::kBlock) before += tsum[k];
    part[t] = before;
    __syncthreads();
    for (int o = nd::kBlock / 2; o > 0; o >>= 1) {
        if (t < o) part[t] += part[t + o];
        __syncthreads();
    }
    before = part[0];
    __syncthreads();
    constexpr int PER = kTileCells / nd::kBlock;
    int32_t c[PER], sum = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int32_t at = base + t * PER + k;
        c[k] = at < ncell ? cells[at] : 0;
        sum += c[k];
    }
    part[t] = sum;
    __syncthreads();
    for (int o = 1; o < nd::kBlock; o <<= 1) {
        const int32_t v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int32_t run = before + part[t] - sum;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int32_t at = base + t * PER + k;
        if (at < ncell) cells[at] = run;
        run += c[k];
    }
    if (blockIdx.x != 0) return;
    if (t == 0) cells[ncell] = n;
    if (host == nullptr) return;
    __shared__ uint32_t so, sa;
    __shared__ unsigned long long sq;
    if (t == 0) {
        so = 0u;
        sa = 0xFFFFFFFFu;
        sq = 0ull;
    }
    __syncthreads();
    uint32_t o = 0u, a = 0xFFFFFFFFu;
    for (int32_t k = t; k < nkb; k += nd::kBlock) {
        o |= kb[2 * k];
        a &= kb[2 * k + 1];
    }
    unsigned long long q = 0ull;
    for (int32_t k = t; k * kTileCells < ncell; k += nd::kBlock) q += tsq[k];
    atomicOr(&so, o);
    atomicAnd(&sa, a);
    atomicAdd(&sq, q);
    __syncthreads();
    if (t == 0) {
        Prep p = *prep;
        p.status = *status;
        p.key_or = so;
        p.key_and = sa;
        p.sum_sq = sq;
        *host = p;
    }
}

// Slot s of the key order: its position in that order and in its cell.
__global__ void __launch_bounds__(nd::kBlock)
k_slots_to_cells(const float *__restrict__ xyz, const int32_t *__restrict__ perm, const int2 *__restrict__ cell_of,
                 const int32_t *__restrict__ cstart, int32_t n, float *__restrict__ xyz_sorted,
                 float4 *__restrict__ cpos, int32_t *__restrict__ ckey) {
    const int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t o = perm[s];
    const float x = xyz[3 * o], y = xyz[3 * o + 1], z = xyz[3 * o + 2];
    xyz_sorted[3 * (int64_t)s] = x;
    xyz_sorted[3 * (int64_t)s + 1] = y;
    xyz_sorted[3 * (int64_t)s + 2] = z;
    const int2 c = cell_of[o];
    const int32_t u = cstart[c.x] + c.y;
    cpos[u] = make_float4(x, y, z, __int_as_float(s));
    ckey[u] = c.x;
}

// What the host needs after the counting pass.
struct CountResult {
    int64_t total;
    int32_t most, status;
};

__global__ void k_count_result(const int64_t *__restrict__ total, const int32_t *__restrict__ most,
                               const int32_t *__restrict__ status, CountResult *__restrict__ host) {
    if (threadIdx.x == 0) {
        host->total = *total;
        host->most = most ? *most : 0;
        host->status = *status;
    }
}

}  // namespace

namespace nd {

float root_threshold(float r) {
    if (!(r > 0.0f)) return 0.0f;  // no root is below r
    // sqrt is monotonic: sqrt(s) < r for exactly the floats below this one
    float t = r * r;
    while (t > 0.0f && std::sqrt(t) >= r) t = std::nextafter(t, 0.0f);
    while (std::sqrt(t) < r) t = std::nextafter(t, INFINITY);
    return t;
}

namespace {

// Cells per group: about two dozen atoms.  At liquid density a cell of the list
// radius holds 18, and groups of one cell test the fewest candidates; where
// cells hold one or two (65,536 points, 8 neighbours each), groups of one cell
// would spend their time on the row lookups.
PairArgs pair_args(const PairSearch &S) {
    PairArgs A{};
    A.cpos = S.cpos;
    A.ckey = S.ckey;
    A.cstart = S.cstart;
    A.cg = S.cg;
    const double mean = (double)S.n / S.cg.ncell;
    // longer runs share more of a group's set-up, shorter ones leave enough
    // waves.  Lists at radius 2.8 with 16 and 32: 32,768 atoms 279 and 325 us,
    // 131,072 408 and 415, 196,608 519 and 548, 262,144 620 and 627 (point
    // queries 510 and 513, cell lists 237 to 255 and 249), 524,288 1,007 and 997,
    // 1,048,576 1,865 and 1,824
    A.per_wave = S.n >= 262144 ? 32 : 16;
    // where squared distances underflow, atoms more than a cell apart could
    // pass the test: groups of one cell look at its 27 neighbours only
    A.k = S.thr < 1e-30f ? 1 : (int32_t)std::min(64.0, std::max(1.0, std::floor(24.0 / mean)));
    A.many = (S.kind == kPairsHalf ? 4.5 : 9.0) * (A.k + 2) * mean > 160.0;
    A.n = S.n;
    A.apl = S.apl;
    A.thr = S.thr;
    A.certain = S.kind == kPairsHalf ? S.thr : S.certain;
    A.r = S.r;
    A.xyz = S.xyz;
    A.nodes = S.nodes;
    A.idx = S.idx;
    return A;
}

unsigned search_grid(const PairArgs &A) {
    const int64_t per = (int64_t)A.per_wave * kWaves;
    return (unsigned)((A.n + per - 1) / per);
}

template <int KIND>
void count_kind(hipStream_t st, const PairArgs &A) {
    if (A.many) k_cell_search<KIND, false, true><<<search_grid(A), kBlock, 0, st>>>(A);
    else k_cell_search<KIND, false, false><<<search_grid(A), kBlock, 0, st>>>(A);
}

template <int KIND>
void emit_kind(hipStream_t st, const PairArgs &A) {
    const size_t lds = 9 * (size_t)A.cap * kWaves;
    if (A.many) k_cell_search<KIND, true, true><<<search_grid(A), kBlock, lds, st>>>(A);
    else k_cell_search<KIND, true, false><<<search_grid(A), kBlock, lds, st>>>(A);
}

}  // namespace

void launch_pair_count(hipStream_t st, const PairSearch &S, int64_t *counts, int32_t *maxcnt) {
    PairArgs A = pair_args(S);
    A.counts = counts;
    A.maxcnt = maxcnt;
    switch (S.kind) {
        case kPairsLeaf: count_kind<kPairsLeaf>(st, A); break;
        case kPairsPointOwn: count_kind<kPairsPointOwn>(st, A); break;
        case kPairsPointRoot: count_kind<kPairsPointRoot>(st, A); break;
        default: count_kind<kPairsHalf>(st, A); break;
    }
    ND_HIP(hipGetLastError());
}

namespace {
// a workgroup may use 64 KiB of LDS without asking for more
constexpr int64_t kLdsBytes = 65536;
int32_t hits_cap(int32_t maxcnt) { return std::max(kQueue, (maxcnt + 3) & ~3); }
int64_t merge_ints(int32_t apl, int64_t cap) { return apl + 1 + 3 * cap; }
}  // namespace

bool pair_emit_fits(int32_t kind, int32_t apl, int32_t maxcnt) {
    if ((int64_t)hits_cap(maxcnt) * 9 * kWaves > kLdsBytes) return false;
    return kind != kPairsLeaf || apl == 1 || merge_ints(apl, (int64_t)apl * maxcnt) * 4 <= kLdsBytes;
}

void launch_pair_emit(hipStream_t st, const PairSearch &S, const int64_t *offsets, int32_t maxcnt, nd_pair *out) {
    PairArgs A = pair_args(S);
    A.offsets = offsets;
    A.out = out;
    A.cap = S.kind == kPairsHalf ? kQueue : hits_cap(maxcnt);
    switch (S.kind) {
        case kPairsLeaf: emit_kind<kPairsLeaf>(st, A); break;
        case kPairsPointOwn: emit_kind<kPairsPointOwn>(st, A); break;
        case kPairsPointRoot: emit_kind<kPairsPointRoot>(st, A); break;
        default: emit_kind<kPairsHalf>(st, A); break;
    }
    if (S.kind == kPairsLeaf && S.apl > 1) {
        const int32_t nL = S.n / S.apl, cap = S.apl * maxcnt;
        // a wave per leaf where four leaves' pairs fit beside each other
        const size_t one = sizeof(int32_t) * (size_t)merge_ints(S.apl, cap);
        if (cap <= 1024 && 4 * one <= (size_t)kLdsBytes)
            k_merge_leaf<64><<<(unsigned)((nL + 3) / 4), kBlock, 4 * one, st>>>(offsets, S.idx, nL, S.apl, cap, out);
        else
            k_merge_leaf<kBlock><<<(unsigned)nL, kBlock, one, st>>>(offsets, S.idx, nL, S.apl, cap, out);
    }
    ND_HIP(hipGetLastError());
}

namespace {
// work words of launch_cell_bins
struct BinWork {
    BoxPart part[kBoxBlocks];
    Prep prep;
    uint64_t tsq[kMaxCells / kTileCells];
    int32_t tsum[kMaxCells / kTileCells];
    int32_t word;
};
}  // namespace

size_t cell_bins_bytes() { return sizeof(BinWork); }

const BinGrid *launch_cell_bins(hipStream_t st, void *work, const float4 *x, int32_t n, float r, int32_t max_cells,
                                BinMode mode, double few, int2 *cell_of, int32_t *cells, int32_t *status) {
    BinWork *w = static_cast<BinWork *>(work);
    if (max_cells > kMaxCells) max_cells = kMaxCells;
    const int32_t tiles = (max_cells + kTileCells - 1) / kTileCells;
    const unsigned g = grid_for(n), nb = std::min<unsigned>(g, kBoxBlocks);
    k_prep_boxes<true><<<nb, kBlock, 0, st>>>(Xyz4{x}, n, w->part, cells, max_cells + 1, &w->word, &w->word);
    if (mode == kBinLines) k_line_grid<<<1, 1, 0, st>>>(r, max_cells, &w->prep);
    else k_prep_grid<<<1, kBlock, 0, st>>>(w->part, (int32_t)nb, n, r, 0.0f, max_cells, nullptr, &w->prep);
    k_bin_atoms<<<g, kBlock, 0, st>>>(x, n, &w->prep, cells, cell_of, status);
    const auto count = mode == kBinCount ? k_cell_tiles<true> : k_cell_tiles<false>;
    count<<<tiles, kBlock, 0, st>>>(cells, &w->prep, w->tsum, w->tsq, few, &w->prep.grid.tests);
    k_cell_starts<<<tiles, kBlock, 0, st>>>(cells, n, &w->prep, w->tsum, w->tsq, nullptr, 0, nullptr, nullptr);
    ND_HIP(hipGetLastError());
    return &w->prep.grid;
}

bool atoms_box(nd_ctx *ctx, const float *d_xyz, int32_t n, double lo[3], double hi[3]) {
    hipStream_t st = ctx->stream;
    ctx->prep.reserve(sizeof(BoxPart) * kBoxBlocks);
    BoxPart *part = ctx->prep.as<BoxPart>();
    int32_t *status = ctx->status.as<int32_t>();
    struct Box { int32_t v[6]; };
    int32_t *hb = host_result<Box>(ctx)->v;
    const unsigned nb = std::min<unsigned>(grid_for(n), kBoxBlocks);
    k_prep_boxes<true><<<nb, kBlock, 0, st>>>(Xyz3{d_xyz}, n, part, nullptr, 0, status + 9, status + 10);
    k_box_result<<<1, 64, 0, st>>>(part, (int32_t)nb, hb);
    ND_HIP(hipGetLastError());
    ND_HIP(hipStreamSynchronize(st));
    for (int d = 0; d < 3; ++d) {
        if (hb[d] > hb[3 + d]) return false;
        for (int e = 0; e < 2; ++e) {
            const int32_t o = hb[3 * e + d], b = o >= 0 ? o : o ^ 0x7FFFFFFF;
            float f;
            std::memcpy(&f, &b, sizeof f);
            (e ? hi : lo)[d] = (double)f;
        }
    }
    return true;
}

int64_t pair_total(nd_ctx *ctx, int64_t n, const int32_t *maxcnt, int32_t *most, int32_t *status) {
    CountResult *hc = host_result<CountResult>(ctx);
    int32_t *word = ctx->status.as<int32_t>();
    launch_scan(ctx, n);
    k_count_result<<<1, 64, 0, ctx->stream>>>(ctx->offsets.as<int64_t>() + n, maxcnt, word, hc);
    ND_HIP(hipGetLastError());
    ND_HIP(hipStreamSynchronize(ctx->stream));
    if (most) *most = hc->most;
    if (status) *status = hc->status;
    return hc->total;
}

// The one-call lists over a tree: keys, sort, tree, pairs.  Counting and
// emitting go over cells; a case that cells serve badly takes the tree walk.
int64_t tree_list(nd_ctx *ctx, const float *d_xyz, int32_t kind, int32_t n, int32_t apl, float r, int32_t pred,
                  int32_t morton, nd_pair *d_out, int64_t cap) {
    hipStream_t st = ctx->stream;
    const int32_t nL = n / apl;
    const bool leaf = kind == kPairsLeaf;
    ctx->has_tree = false;
    // cells of at least two atoms on average
    const int32_t max_cells = (int32_t)std::min<int64_t>(kMaxCells, std::max<int64_t>(27, n / 2));
    const int32_t tiles = (max_cells + kTileCells - 1) / kTileCells;
    const unsigned g = grid_for(n);
    for (DevBuf *b : {&ctx->codes, &ctx->codes_sorted, &ctx->perm, &ctx->perm_alt, &ctx->cell_keys})
        b->reserve(sizeof(int32_t) * (size_t)n);
    ctx->xyz_sorted.reserve(sizeof(float) * 3 * (size_t)n);
    ctx->nodes.reserve(sizeof(nd_node) * (size_t)(2 * nL - 1));
    ctx->store.reserve(sizeof(int32_t) * lbvh_scratch_ints(nL));
    ctx->cell_pos.reserve(sizeof(float4) * (size_t)n);
    ctx->cell_start.reserve(sizeof(int32_t) * ((size_t)max_cells + 1));
    ctx->cell_vals.reserve(sizeof(int2) * (size_t)n);
    ctx->bbox.reserve(64);
    // work words: box parts, prep, tile sums, key bits
    const size_t off_prep = sizeof(BoxPart) * kBoxBlocks, off_sq = off_prep + 256,
                 off_sum = off_sq + sizeof(uint64_t) * (size_t)tiles, off_kb = off_sum + sizeof(int32_t) * (size_t)tiles;
    ctx->prep.reserve(off_kb + 8 * (size_t)g + 16);
    char *work = ctx->prep.as<char>();
    BoxPart *part = reinterpret_cast<BoxPart *>(work);
    Prep *prep = reinterpret_cast<Prep *>(work + off_prep);
    static_assert(sizeof(Prep) <= 256, "prep block");
    uint64_t *tsq = reinterpret_cast<uint64_t *>(work + off_sq);
    int32_t *tsum = reinterpret_cast<int32_t *>(work + off_sum);
    uint32_t *kb = reinterpret_cast<uint32_t *>(work + off_kb);
    int32_t *status = ctx->status.as<int32_t>(), *maxcnt = status + 8;
    int32_t *cells = ctx->cell_start.as<int32_t>();
    int2 *cell_of = ctx->cell_vals.as<int2>();
    float *box = ctx->bbox.as<float>();
    int32_t *codes = ctx->codes_sorted.as<int32_t>(), *perm = ctx->perm.as<int32_t>();
    float *xs = ctx->xyz_sorted.as<float>();
    nd_node *nodes = ctx->nodes.as<nd_node>();

    // mortoncodes!, and each atom's cell
    const float thr = pred == ND_PRED_SCALAR ? r * r : root_threshold(r);
    const unsigned nb = std::min<unsigned>(g, kBoxBlocks);
    Prep *hp = host_result<Prep>(ctx);
    k_prep_boxes<false><<<nb, kBlock, 0, st>>>(Xyz3{d_xyz}, n, part, cells, max_cells + 1, status, maxcnt);
    k_prep_grid<<<1, kBlock, 0, st>>>(part, (int32_t)nb, n, r, thr, max_cells, box, prep);
    if (morton == ND_MORTON_MASKED)
        k_prep_keys<true><<<g, kBlock, 0, st>>>(d_xyz, n, box, prep, codes, perm, cells, cell_of, kb, status);
    else
        k_prep_keys<false><<<g, kBlock, 0, st>>>(d_xyz, n, box, prep, codes, perm, cells, cell_of, kb, status);
    k_cell_tiles<false><<<tiles, kBlock, 0, st>>>(cells, prep, tsum, tsq, 0.0, nullptr);
    k_cell_starts<<<tiles, kBlock, 0, st>>>(cells, n, prep, tsum, tsq, kb, (int32_t)g, status, hp);
    ND_HIP(hipGetLastError());
    ND_HIP(hipStreamSynchronize(st));
    const Prep p = *hp;
    if (p.status) clear_status(ctx);
    if (p.status & kStatusDomain)
        throw Error(ND_ERR_DOMAIN,
                    "mortoncodes!: coordinate outside the Int32 quantisation domain "
                    "(reference throws InexactError)");
    // sortperm + permute!
    radix_sort_bits(st, ctx->sort, p.key_or ^ p.key_and, n, &codes, &perm, ctx->codes.as<int32_t>(),
                    ctx->perm_alt.as<int32_t>());
    k_slots_to_cells<<<g, kBlock, 0, st>>>(d_xyz, perm, cell_of, cells, n, xs, ctx->cell_pos.as<float4>(),
                                           ctx->cell_keys.as<int32_t>());
    // leafcluster_primitives (+- r/2 leaves) or cluster_primitives (+- r), and
    // bounding_volume_hierarchy!.  The point queries' tree: the build halves
    // its radius argument, 2r is exact below the callers' bound.  TreeData
    // overwrites the root box (BVHTraverse.jl:856-858), the root-started
    // form's build kernel keeps it (NaiveKA.jl:301-302).
    launch_lbvh(st, xs, 3, codes, nL, apl, leaf ? r : 2.0f * r, kind == kPairsPointRoot ? 0 : 1, nodes,
                ctx->store.as<int32_t>(), status);
    ctx->has_tree = true;
    ctx->tree_n = n;
    ctx->tree_apl = apl;
    ctx->tree_nodes = nodes;
    ctx->tree_perm = perm;
    ctx->tree_codes = codes;
    ctx->tree_store = ctx->store.as<int32_t>();

    auto walk = [&]() {
        return leaf ? leaf_traverse(ctx, nodes, xs, perm, n, apl, r, pred, d_out, cap, true)
                    : point_traverse(ctx, nodes, xs, perm, n, apl, r, kind == kPairsPointRoot ? ND_QUERY_ROOT : ND_QUERY_OWN_LEAF,
                                     d_out, cap);
    };
    // Cells serve radii whose squares are normal numbers, and atoms that are
    // not crowded into few of the cells (27 sum_sq bounds the candidates: one
    // far outlier stretches the grid until all others share a cell).  The line
    // lies where a walk draws level: 131,072 points at density 0.8, 4 per leaf,
    // radius 6 (4,800 candidates and 318 pairs an atom): 3.63 ms by cells, 3.99
    // walking, point queries 3.04 and 4.80; 65,536 points, radius 8 (14,200):
    // 4.14 and 3.78, point queries 10.3 and 7.3.  Leaves of 64 atoms (a hit is
    // placed in 63 other lists) draw level with a walk over a compact order:
    // 131,072 points 1.25 ms and 1.23; 32 atoms 0.70 and 1.12.
    const bool by_cells = r >= 1e-15f && r <= 1e18f && (double)p.sum_sq * 27.0 <= 5500.0 * n &&
                          apl <= (!leaf || morton == ND_MORTON_MASKED ? 64 : 32);
    if (!by_cells) return walk();
    PairSearch S{};
    S.kind = kind;
    S.n = n;
    S.apl = apl;
    S.cg = p.grid.cg;
    S.cpos = ctx->cell_pos.as<float4>();
    S.ckey = ctx->cell_keys.as<int32_t>();
    S.cstart = cells;
    S.xyz = xs;
    S.nodes = nodes;
    S.idx = perm;
    S.r = r;
    S.thr = thr;
    S.certain = p.certain;
    ctx->counts.reserve(sizeof(int64_t) * ((size_t)n + 1));
    ctx->offsets.reserve(sizeof(int64_t) * ((size_t)n + 1));
    const int64_t *off = ctx->offsets.as<int64_t>();
    launch_pair_count(st, S, ctx->counts.as<int64_t>(), maxcnt);
    CountResult c{};
    c.total = pair_total(ctx, n, maxcnt, &c.most, &c.status);
    if (c.status) clear_status(ctx);
    if (c.status & kStatusTree)
        throw Error(ND_ERR_STATE, "neighbour list: malformed tree (rope cycle or bad index)");
    if (c.total > cap || d_out == nullptr || c.total == 0) return c.total;
    if (!pair_emit_fits(kind, apl, c.most)) return walk();
    launch_pair_emit(st, S, off, c.most, d_out);
    ND_HIP(hipStreamSynchronize(st));
    return c.total;
}

}  // namespace nd
