// Walk of one i-cluster's list that hands the pairs inside the cutoff to the
// caller 64 at a time, and the FP64 pair terms its users share (energy
// steps, the lambda-window sums, the gradients).
//
// Why: these users spend 70 to 150 FP64 instructions on a pair, and in the
// cluster layout (16 lanes per listed cluster pair) a wave pays them whenever
// one of its 64 lanes is inside the cutoff; 18 to 36 % are. Here a scan finds
// the pairs inside the cutoff (about 70 instructions per 256 listed pairs)
// and queues them per i atom in LDS, and the terms run on full waves.
//
// Scan: 16 list entries a time, lane (e, jj) = (lane >> 2, lane & 3) holding
// one j atom against the cluster's four i atoms. r^2 = |a|^2 + |b|^2 - 2 a.b
// about the cluster's first atom, the product from three 16-block 4x4x1 FP32
// MFMAs (one per axis: 256 products each). The cutoff predicate stays the
// library's dr2_exact: a batch with a value closer to rc^2 than the
// expansion's rounding bound is tested again with dr2_exact itself.
#pragma once
#include "common.hpp"
#include "pair_math.hpp"

namespace snb {

constexpr int kDenseWaves = 8;     // i-clusters per block of the walk's kernels
constexpr int kDenseQueue = 112;   // queued pairs per i atom: at most 48 left by a drain, and 64 new ones
constexpr int kDenseEntries = 128; // list entries staged at a time

// The walk's kernels run as kDenseBlocks resident blocks whose waves stride
// over units of work, a unit being one of `parts` shares of a cluster's list:
// the erfc rows, the final sums and their atomics are then paid once per
// wave and not once per cluster.
constexpr int kDenseBlocks = 512;  // 2 of 8 waves on each of 256 CUs

// Shares of a cluster's list that give the waves the evenest rounds (a
// share's own fixed cost taken as 8 % of a whole list).
__device__ __forceinline__ int dense_parts(int clusters, int waves) {
    int best = 1;
    float least = 1e30f;
    for (int p = 1; p <= 8; p *= 2) {
        const float t = (float)((clusters * p + waves - 1) / waves) * (1.0f / p + 0.08f);
        if (t < least) {
            least = t;
            best = p;
        }
    }
    return best;
}

// Units of this wave: first, first + step, ... below end (each XCD a
// contiguous range of clusters). Blocks a multiple of kNumXcd.
struct DenseUnits {
    int parts, first, end, step;
};
__device__ __forceinline__ DenseUnits dense_units(int clusters) {
    DenseUnits u;
    u.parts = dense_parts(clusters, gridDim.x * kDenseWaves);
    const int total = clusters * u.parts, x = blockIdx.x % kNumXcd;
    u.step = gridDim.x / kNumXcd * kDenseWaves;
    // (uniform over the wave: the walk's loops and counts then stay scalar)
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    u.first = (int)((long)total * x / kNumXcd) + (int)(blockIdx.x / kNumXcd) * kDenseWaves + w;
    u.end = (int)((long)total * (x + 1) / kNumXcd);
    return u;
}

struct DenseLds {
    uint2 ent[kDenseEntries];
    int q[kClusterSize][kDenseQueue];
};

// ---- erfc from a table in LDS ---------------------------------------------
// Taylor pieces of degree 7 about the multiples of 1/64, |u| <= 1/128: the
// remainder is below 1e-17 (2e-15 of the value at x = 3.5), rounding that of
// a Horner chain. Every block computes its rows with the device library's
// erfc and exp, so no entry point holds a table. Coefficients are those of
// powers of 64 u (a power of two: exact). Rows are 80 bytes apart: 16-byte
// reads of random rows then spread over all LDS banks (64 bytes apart they
// would share a quarter of them).
constexpr int kErfcPieces = 64;        // per unit of x
constexpr int kErfcRow = 10;           // doubles from row to row, 8 used
constexpr int kErfcMaxRows = 514;      // x <= 8, past it 0: erfc(8) is 1.1e-29

// Rows for arguments up to beta * rc.
inline int erfc_rows(double beta, double rc) {
    const double x = beta * rc * 1.0001 * kErfcPieces;
    return x < kErfcMaxRows - 2 ? (int)x + 2 : kErfcMaxRows;
}
inline size_t erfc_lds(int rows) { return (size_t)rows * kErfcRow * sizeof(double); }

__device__ __forceinline__ void erfc_fill(double* tab, int rows) {
    for (int k = threadIdx.x; k < rows; k += blockDim.x) {
        const double x = k * (1.0 / kErfcPieces);
        double* c = tab + k * kErfcRow;
        // g = erfc', a_n = g^(n) / n!: a_{n+1} = (-2 x a_n - 2 a_{n-1}) / (n + 1)
        double a = -1.1283791670955125739 * exp(-x * x), before = 0.0, unit = 1.0 / kErfcPieces;
        c[0] = erfc(x);
        c[1] = a * unit;
#pragma unroll
        for (int n = 0; n < 6; n++) {
            const double next = (x * a + before) * (-2.0 / (n + 1));
            before = a;
            a = next;
            unit *= 1.0 / kErfcPieces;
            c[n + 2] = a * (1.0 / (n + 2)) * unit;
        }
    }
}

// erfc(x) for y = 64 x.
__device__ __forceinline__ double erfc_at(const double* tab, int rows, double y) {
    const double yk = __builtin_rint(y);
    const double u = y - yk;
    const int k = (int)yk;
    const double2* c = reinterpret_cast<const double2*>(tab + min(k, rows - 1) * kErfcRow);
    const double2 c0 = c[0], c2 = c[1], c4 = c[2], c6 = c[3];
    double v = fma(c6.y, u, c6.x);
    v = fma(v, u, c4.y);
    v = fma(v, u, c4.x);
    v = fma(v, u, c2.y);
    v = fma(v, u, c2.x);
    v = fma(v, u, c0.y);
    v = fma(v, u, c0.x);
    return k < kErfcMaxRows - 1 ? v : 0.0;
}

// 1 / sqrt(r2) and sqrt(r2) from v_rsq_f64 and one third-order step; r2 = 0
// gives inf and 0, as 1.0 / sqrt(0.0) does.
__device__ __forceinline__ void rsqrt_f64(double r2, double& rinv, double& r) {
    const double y = __builtin_amdgcn_rsq(r2);
    const double e = fma(-r2 * y, y, 1.0);
    rinv = fma(y * e, fma(e, 0.375, 0.5), y);
    r = r2 * rinv;
    if (__any(r2 == 0.0)) {
        if (r2 == 0.0) {
            rinv = __builtin_huge_val();
            r = 0.0;
        }
    }
}

// ---- the walk ---------------------------------------------------------------
// Calls use(active, jslot) with all 64 lanes, lane (i, k) = (lane >> 4,
// lane & 15) taking pairs of the cluster's slot i; every pair inside the
// cutoff is handed over once per side (HALF: once in all, from one of its
// clusters: the one the parity of the cluster numbers names, so that all
// clusters keep about half of their pairs). Every lane of the wave must call.
// `part` of `parts`: this wave's share of the cluster's list entries.
// Set bits of a wave mask below this lane.
__device__ __forceinline__ int below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

typedef float DenseF4 __attribute__((ext_vector_type(4)));

template <bool HALF, class Use>
__device__ __forceinline__ void dense_walk(int ic, const uint4* __restrict__ pk, const int* __restrict__ s2o,
                                           const int* __restrict__ list_n, const uint2* __restrict__ list,
                                           int list_cap, float cx, float cy, float cz, float rc2, int part,
                                           int parts, DenseLds& L, Use&& use) {
    const int lane = threadIdx.x & 63, jj = lane & 3;
    uint4 a[kClusterSize];
    float aa[kClusterSize], own[3] = {0.f, 0.f, 0.f};
    float ext = 0.f;
#pragma unroll
    for (int i = 0; i < kClusterSize; i++) {
        a[i] = pk[ic * kClusterSize + i];
        // padding (the last slots of a column) takes the first atom's place:
        // none of its pairs is listed
        const bool pad = s2o[ic * kClusterSize + i] < 0;
        const float x = pad ? 0.f : (float)(int)((a[i].x & ~3u) - (a[0].x & ~3u)) * cx;
        const float y = pad ? 0.f : (float)(int)((a[i].y & ~3u) - (a[0].y & ~3u)) * cy;
        const float z = pad ? 0.f : (float)(int)((a[i].z & ~3u) - (a[0].z & ~3u)) * cz;
        aa[i] = x * x + y * y + z * z;
        ext = fmaxf(ext, aa[i]);
        if (jj == i) {
            own[0] = -2.0f * x;
            own[1] = -2.0f * y;
            own[2] = -2.0f * z;
        }
    }
    ext = sqrtf(ext);
    const float rc = sqrtf(rc2), reach = rc + ext;
    // the displacement from the first atom names the nearest image of every
    // pair inside the cutoff only while cutoff + extent is below half a box
    // (2^31 units); else every batch takes the exact test
    const bool safe = reach * 1.0001f < 2147483648.0f * fminf(cx, fminf(cy, cz));
    // |a|, |b| <= reach near the cutoff: coordinates 8, |a|^2 and |b|^2 13,
    // the product's three steps 16, dr2_exact 7 units of 2^-24 reach^2
    const float eps = 4.0e-6f * reach * reach;
    const float lo = rc2 - eps, hi = rc2 + eps;
    int c[kClusterSize] = {0, 0, 0, 0};
    const int i4 = lane >> 4, k16 = lane & 15;

    // hands over up to 16 pairs of each i atom, the last queued ones first
    auto drain = [&]() {
        const int ci = i4 == 0 ? c[0] : i4 == 1 ? c[1] : i4 == 2 ? c[2] : c[3];
        const int at = max(ci - 16, 0) + k16;
        const bool active = at < ci;
        const int jslot = active ? L.q[i4][at] : ic * kClusterSize;
        __builtin_amdgcn_wave_barrier();
        use(active, jslot);
#pragma unroll
        for (int i = 0; i < kClusterSize; i++) c[i] = max(c[i] - 16, 0);
    };

    const int n_all = list_n[ic], first = n_all * part / parts, n = n_all * (part + 1) / parts - first;
    const uint2* __restrict__ lst = list + (size_t)ic * list_cap + first;
    const uint2 none = make_uint2((unsigned)ic, 0u);
    const int e0 = lane >> 2;
    int base = 0, it = 0, kept = 0;
    uint2 ent = none;
    uint4 b = a[0];
    for (;;) {
        while (it >= kept && base < n) {
            // stage the next entries this side takes
            kept = 0;
#pragma unroll
            for (int h = 0; h < kDenseEntries; h += 64) {
                const int e = base + h + lane;
                uint2 my = e < n ? lst[e] : none;
                if (HALF) {
                    const int jc = (int)my.x;
                    if (jc == ic) my.y &= 0x7310u;  // the cluster's own pairs with jj > ii
                    else if ((ic < jc) != (((ic ^ jc) & 1) != 0)) my.y = 0u;
                }
                const bool keep = my.y != 0u;
                const unsigned long long kb = __ballot(keep);
                if (keep) L.ent[kept + below(kb)] = my;
                kept += __popcll(kb);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            base += kDenseEntries;
            it = 0;
            ent = e0 < kept ? L.ent[e0] : none;
            b = pk[(int)ent.x * kClusterSize + jj];
        }
        const bool more = it < kept;
        if (more) {
            const int en = it + 16 + e0;
            const uint2 entn = en < kept ? L.ent[en] : none;
            const uint4 bn = pk[(int)entn.x * kClusterSize + jj];
            const int jslot = (int)ent.x * kClusterSize + jj;
            const unsigned m4 = (ent.y >> (jj * 4)) & 15u;
            const float x = (float)(int)((b.x & ~3u) - (a[0].x & ~3u)) * cx;
            const float y = (float)(int)((b.y & ~3u) - (a[0].y & ~3u)) * cy;
            const float z = (float)(int)((b.z & ~3u) - (a[0].z & ~3u)) * cz;
            const float bb = x * x + y * y + z * z;
            DenseF4 t = {bb + aa[0], bb + aa[1], bb + aa[2], bb + aa[3]};
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[0], x, t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[1], y, t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[2], z, t, 0, 0, 0);
            unsigned long long in[kClusterSize], near = 0ull;
#pragma unroll
            for (int i = 0; i < kClusterSize; i++) {
                const unsigned long long listed = __ballot((m4 >> i) & 1u);
                in[i] = listed & __ballot(t[i] < lo);
                near |= listed & ~in[i] & __ballot(t[i] < hi);
            }
            if (!safe || near) {
#pragma unroll
                for (int i = 0; i < kClusterSize; i++) {
                    const float dx = (float)(int)((b.x & ~3u) - (a[i].x & ~3u)) * cx;
                    const float dy = (float)(int)((b.y & ~3u) - (a[i].y & ~3u)) * cy;
                    const float dz = (float)(int)((b.z & ~3u) - (a[i].z & ~3u)) * cz;
                    in[i] = __ballot(((m4 >> i) & 1u) && dr2_exact(dx, dy, dz) < rc2);
                }
            }
#pragma unroll
            for (int i = 0; i < kClusterSize; i++) {
                if (__builtin_amdgcn_inverse_ballot_w64(in[i])) L.q[i][c[i] + below(in[i])] = jslot;
                c[i] += __popcll(in[i]);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            ent = entn;
            b = bn;
            it += 16;
        }
        // full rounds, more while a queue could not take the next 64, and
        // what is left at the end
        for (;;) {
            const int most = max(max(c[0], c[1]), max(c[2], c[3]));
            if (most <= (more ? 48 : 0) && min(min(c[0], c[1]), min(c[2], c[3])) < 16) break;
            drain();
        }
        if (!more) break;
    }
}

}  // namespace snb
