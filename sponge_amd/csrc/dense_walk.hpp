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
// over units of work, a unit being one of 1 to 8 shares of a cluster's list:
// the erfc rows, the final sums and their atomics are then paid once per
// wave and not once per cluster.
constexpr int kDenseBlocks = 512;  // 2 of 8 waves on each of 256 CUs

// Shares of a cluster's list (as a power of two) that give the waves the
// evenest rounds (a share's own fixed cost taken as 8 % of a whole list).
__device__ __forceinline__ int dense_split(int clusters, int waves) {
    int best = 0;
    float least = 1e30f;
    for (int k = 0; k <= 3; k++) {
        const float t = (float)(((clusters << k) + waves - 1) / waves) * (1.0f / (1 << k) + 0.08f);
        if (t < least) {
            least = t;
            best = k;
        }
    }
    return __builtin_amdgcn_readfirstlane(best);
}

// Units of a block: block-first `base` below `end`, `step` apart, wave w taking
// unit base + w, share u % 2^split of cluster u / 2^split; each XCD a
// contiguous range of clusters, and the shares of one cluster adjacent waves
// of one block. Blocks a multiple of kNumXcd.
struct DenseUnits {
    int split, base, end, step;
};
__device__ __forceinline__ DenseUnits dense_units(int clusters) {
    DenseUnits u;
    u.split = dense_split(clusters, gridDim.x * kDenseWaves);
    const int x = blockIdx.x % kNumXcd;
    u.step = gridDim.x / kNumXcd * kDenseWaves;
    u.base = ((int)((long)clusters * x / kNumXcd) << u.split) + (int)(blockIdx.x / kNumXcd) * kDenseWaves;
    u.end = (int)((long)clusters * (x + 1) / kNumXcd) << u.split;
    return u;
}
// Resident blocks for a list of at most `clusters` clusters.
inline int dense_blocks(int clusters) {
    const int most = xcd_grid(ceil_div(8l * clusters, kDenseWaves));
    return most < kDenseBlocks ? most : kDenseBlocks;
}
// The wave's number in its block, uniform over the wave (the walk's loops and
// counts then stay scalar).
__device__ __forceinline__ int wave_in_block() {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
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

// 1 / v from v_rcp_f64 and two Newton steps; v = 0 gives inf, as 1.0 / 0.0.
__device__ __forceinline__ double rcp_f64(double v) {
    double y = __builtin_amdgcn_rcp(v);
    y = fma(fma(-v, y, 1.0), y, y);
    y = fma(fma(-v, y, 1.0), y, y);
    if (__any(v == 0.0)) y = v == 0.0 ? __builtin_huge_val() : y;
    return y;
}

// Sums over the 16 lanes of a row (one i atom's in the walk), in all of them.
__device__ __forceinline__ float row_sum(float v) {
    v += dpp_row_ror<8>(v);
    v += dpp_row_ror<4>(v);
    v += dpp_row_ror<2>(v);
    return v + dpp_row_ror<1>(v);
}
template <int N>
__device__ __forceinline__ double dpp_row_ror(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + N, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + N, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_row_ror<8>(v);
    v += dpp_row_ror<4>(v);
    v += dpp_row_ror<2>(v);
    return v + dpp_row_ror<1>(v);
}

// ---- the walk ---------------------------------------------------------------
// Calls use(active, jslot) with all 64 lanes, lane (i, k) = (lane >> 4,
// lane & 15) taking pairs of the cluster's slot i; every pair inside the
// cutoff is handed over once per side (kEachSide), or once in all: from the
// side of its lower-index atom (kLowerAtom: per-atom sums credited to that
// atom), or from one of its clusters, the one that the parity of the cluster
// numbers names (kOneCluster: totals; half of the entries are scanned, about
// the same share of every cluster's). Every lane of the wave must call.
// `part` of 2^split: this wave's share of the cluster's list entries. ic and
// part uniform over the wave.
enum DenseSide { kEachSide, kLowerAtom, kOneCluster };
// Set bits of a wave mask below this lane.
__device__ __forceinline__ int below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// The first lane's value, in a scalar register.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// The value of lane K of this lane's quad.
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), K * 0x55, 0xF, 0xF, false));
}

typedef float DenseF4 __attribute__((ext_vector_type(4)));

template <DenseSide SIDE, class Use>
__device__ __forceinline__ void dense_walk(int ic, const uint4* __restrict__ pk, const int* __restrict__ s2o,
                                           const int* __restrict__ list_n, const uint2* __restrict__ list,
                                           int list_cap, float cx, float cy, float cz, float rc2, int part,
                                           int split, DenseLds& L, Use&& use) {
    const int lane = threadIdx.x & 63, jj = lane & 3;
    // the first atom's position (uniform), and this lane's i atom jj: -2 a for
    // the product, |a|^2 and the atom's index spread over the lane's quad
    const uint4 mine = pk[ic * kClusterSize + jj];
    const int mine_at = s2o[ic * kClusterSize + jj];
    const unsigned ox = uniform((int)(mine.x & ~3u)), oy = uniform((int)(mine.y & ~3u)),
                   oz = uniform((int)(mine.z & ~3u));
    // padding (the last slots of a column) takes the first atom's place: none
    // of its pairs is listed
    const bool pad = mine_at < 0;
    const float px = pad ? 0.f : (float)(int)((mine.x & ~3u) - ox) * cx;
    const float py = pad ? 0.f : (float)(int)((mine.y & ~3u) - oy) * cy;
    const float pz = pad ? 0.f : (float)(int)((mine.z & ~3u) - oz) * cz;
    const float own[3] = {-2.0f * px, -2.0f * py, -2.0f * pz};
    const float paa = px * px + py * py + pz * pz;
    const float aa[kClusterSize] = {quad_lane<0>(paa), quad_lane<1>(paa), quad_lane<2>(paa), quad_lane<3>(paa)};
    int at[kClusterSize] = {0, 0, 0, 0};
    if (SIDE == kLowerAtom) {
        const float t = __int_as_float(mine_at);
        at[0] = __float_as_int(quad_lane<0>(t));
        at[1] = __float_as_int(quad_lane<1>(t));
        at[2] = __float_as_int(quad_lane<2>(t));
        at[3] = __float_as_int(quad_lane<3>(t));
    }
    const float ext = __builtin_amdgcn_sqrtf(fmaxf(fmaxf(aa[0], aa[1]), fmaxf(aa[2], aa[3])));
    const float rc = sqrtf(rc2), reach = (rc + ext) * 1.0001f;
    // the displacement from the first atom names the nearest image of every
    // pair inside the cutoff only while cutoff + extent is below half a box
    // (2^31 units); else every batch takes the exact test
    const bool safe = reach < 2147483648.0f * fminf(cx, fminf(cy, cz));
    // |a|, |b| <= reach near the cutoff: coordinates 8, |a|^2 and |b|^2 13,
    // the product's three steps 16, dr2_exact 7 units of 2^-24 reach^2
    const float eps = 4.0e-6f * reach * reach;
    const float lo = rc2 - eps, hi = rc2 + eps;
    int c[kClusterSize] = {0, 0, 0, 0};
    const int i4 = lane >> 4, k16 = lane & 15;

    // hands over up to 16 pairs of each i atom, the last queued ones first
    auto drain = [&]() {
        const int ci = i4 == 0 ? c[0] : i4 == 1 ? c[1] : i4 == 2 ? c[2] : c[3];
        const int e = max(ci - 16, 0) + k16;
        const bool active = e < ci;
        const int jslot = active ? L.q[i4][e] : ic * kClusterSize;
        __builtin_amdgcn_wave_barrier();
        use(active, jslot);
#pragma unroll
        for (int i = 0; i < kClusterSize; i++) c[i] = max(c[i] - 16, 0);
    };

    const int n_all = uniform(list_n[ic]), first = (n_all * part) >> split,
              n = ((n_all * (part + 1)) >> split) - first;
    const uint2* __restrict__ lst = list + (size_t)ic * list_cap + first;
    const uint2 none = make_uint2((unsigned)ic, 0u);
    const int e0 = lane >> 2;
    int base = 0, it = 0, kept = 0;
    uint2 ent = none;
    uint4 b = mine;
    for (;;) {
        while (it >= kept && base < n) {
            // stage the next entries this side takes
            kept = 0;
#pragma unroll
            for (int h = 0; h < kDenseEntries; h += 64) {
                const int e = base + h + lane;
                uint2 my = e < n ? lst[e] : none;
                if (SIDE == kOneCluster) {
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
            const int aj = SIDE == kLowerAtom ? s2o[jslot] : 0;
            const float x = (float)(int)((b.x & ~3u) - ox) * cx;
            const float y = (float)(int)((b.y & ~3u) - oy) * cy;
            const float z = (float)(int)((b.z & ~3u) - oz) * cz;
            const float bb = x * x + y * y + z * z;
            DenseF4 t = {bb + aa[0], bb + aa[1], bb + aa[2], bb + aa[3]};
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[0], x, t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[1], y, t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_4x4x1f32(own[2], z, t, 0, 0, 0);
            unsigned long long in[kClusterSize], near = 0ull;
#pragma unroll
            for (int i = 0; i < kClusterSize; i++) {
                const unsigned long long listed = __ballot(((m4 >> i) & 1u) && (SIDE != kLowerAtom || at[i] < aj));
                in[i] = listed & __ballot(t[i] < lo);
                near |= listed & ~in[i] & __ballot(t[i] < hi);
            }
            if (!safe || near) {
#pragma unroll
                for (int i = 0; i < kClusterSize; i++) {
                    const uint4 a = pk[ic * kClusterSize + i];
                    const float dx = (float)(int)((b.x & ~3u) - (a.x & ~3u)) * cx;
                    const float dy = (float)(int)((b.y & ~3u) - (a.y & ~3u)) * cy;
                    const float dz = (float)(int)((b.z & ~3u) - (a.z & ~3u)) * cz;
                    in[i] = __ballot(((m4 >> i) & 1u) && (SIDE != kLowerAtom || at[i] < aj) &&
                                     dr2_exact(dx, dy, dz) < rc2);
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
