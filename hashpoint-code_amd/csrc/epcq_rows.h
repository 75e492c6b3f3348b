// Full-image sampler over row runs.
//
// A window row's buckets are neighbours in the row-major point list, so the
// candidates of a ray are k contiguous runs of list positions, one per window
// row (plus the repeats that clamping at the image's border makes).  A wave
// takes 64 consecutive rays of one image row: every lane visits the same
// window rows, and the only divergence left is the length of its run.
//
// A block of four waves (a 64 x 4 tile of rays) sweeps the window rows, in the
// canonical order (rows, then columns, then list position), once for each of
//   1. tmin, the smallest ray depth of a hit;
//   2. the depth slots hit once and at least twice: the first two slots with
//      two hits are the only ones a ray can visit (the host takes this path
//      only when epcq_max_live_samples is at most 2);
//   3. the distance sums of those two slots, and the neighbours of the two
//      sample points at them.
// The sweeps repeat the candidate test instead of storing the hits, so no
// list can overflow and every sum is taken in the canonical order.  What a
// sweep tests first is not the exact distance but a bound: each list position
// has (a, b, T, z) beside its point, its direction in the camera's frame, the
// squared reach of its radius there and a lower bound of the ray depth at
// which it matters (row_candidate); a lane rejects it with two subtractions,
// three multiplications and two comparisons, and collects the others as bits
// of a mask.  Only those run the exact operations of ray_t_e2 on the point
// itself.  z cuts what lies behind the part of the ray that is still of
// interest: behind the running tmin, behind the second slot.
//
// The block stages the candidates and points of as many window rows as the
// LDS holds, or a piece of a row that is too long for it.
//
// Rays that this does not cover go to a queue in the workspace and run one
// wave per ray (epcq_rows_wave.h) in a second launch: more than 48 candidates
// within the bound of a ray whose region has a bucket of more than 48 points
// (a bucket gives at most its first 48 hits), a table whose buckets are not in
// row-major list order, a row of several LDS loads, far more candidates than
// the wave's other rays, and a walk that two slots do not end.  The outputs are the same either way; a second launch spreads such
// rays, which come in clusters, over the whole GPU, and keeps their code out of
// this kernel's registers.
//
// What bounds it: the densest tiles, which end last, and waits.  Vector issue
// (about 10 instructions per candidate and sweep, about 60 per exact test, in
// which a third of the lanes take part) would take 36 % of the time for 1M points
// at 800 x 800 (0.44 ms), 27 % for 307k at 517 x 389 (0.35 ms, 882 tiles for 1024
// places) and 64 % for 20M at 1920 x 1080 (15.5 ms); the waves spend about half of
// their time waiting for LDS, memory or a barrier.
// Measured per call with the build, against the lane-set kernels and the build
// of three arrays: 1M points at 800 x 800, k = 5, dense layout 0.89 -> 0.53 ms;
// 307k points at 517 x 389, k = 5, with features 1.09 -> 0.42 ms; 20M points at
// 1920 x 1080, k = 15, with features 247 -> 21.7 ms.
#pragma once

#include "epcq_sampler.h"

namespace epcq {

// SampleOpts::rows: the lane-set kernels, row-run tiles, one wave per ray.
constexpr int kRowsNone = 0, kRowsTiles = 1, kRowsWave = 2;

constexpr int kRowTileW = kWave;   // rays of a wave: consecutive columns
constexpr int kRowTileH = 4;       // waves of a block: consecutive rows
constexpr int kRowThreads = kRowTileW * kRowTileH;
constexpr int kRowMaxK = 16;       // larger windows take the lane-set kernels
constexpr int kRowCap = 960;       // points staged at once: four blocks per CU, three with per-point radii
// A row of more points than this leaves its tile's rays to waves: a piece of it
// serves the k + 63 columns or fewer that it covers, and the others wait.
__device__ __forceinline__ int row_longest(int k) { return k <= 8 ? kRowCap : 4 * kRowCap; }
constexpr int kRowPad = 32;        // entries past its run that a lane may read (and ignore)
constexpr int kRowMaxRows = kRowTileH + kRowMaxK - 1;
constexpr int kRowCols = kRowTileW + kRowMaxK;  // columns of the region and the row's end
// A ray is left to a whole wave when its window holds more than
// SampleOpts::row_heavy * SampleOpts::heavy candidates and at most
// kHeavyMinority rays of its wave do (or 4 times as many).  The factor is what
// a SIMD's lanes have to do anyway, within these bounds: 4096 candidates take a
// lane about 0.2 ms, with its wave's other lanes, and a wave of its own 25 us.
// A least factor of 8 instead of 32: 1.39 -> 1.15 ms for 1M points on a sphere
// at 500 x 503, k = 7, and within 2 % where no ray is so heavy.
constexpr int kRowHeavyMost = 32;
constexpr int kRowHeavyLeast = 8;

template <bool PR>
struct RowSmem {
    float4 cand[kRowCap + kRowPad];  // (a, b, T, z) of the staged points
    float4 pts[kRowCap];             // (x, y, z, index bits)
    float lim[PR ? kRowCap : 1];     // squared radius thresholds
    int lo[kRowMaxRows][kRowCols];   // list position of the first point at or right of a column
    int base[kRowMaxRows + 1];       // points of the region's rows before this one
    int flags[kRowTileH];            // per wave: kRowIrregular | kRowBigBucket
};

constexpr int kRowIrregular = 1;  // buckets not contiguous in row-major order
constexpr int kRowBigBucket = 2;  // a bucket of more than kSampleLaneHits points

// Queue of deferred rays of one view: their count, then pixel ids (at most
// one entry per pixel), in the workspace's bucket-cone region, which this path
// leaves free.
struct RowQueue {
    int count;
    int pad[3];
    int ray[1];
};

// The view's frame: e1, e2, ec about orthonormal, ec the camera's forward axis.
struct RowFrame {
    float e1[3], e2[3], ec[3];
    float o[3];
    float om;  // origin part of the reach margin
};

// A value that every lane of the wave holds (read from LDS, where the compiler
// cannot know it), moved to a scalar register: the loops over rows and chunks
// then branch on scalars and their bounds take no vector registers.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uniform(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// From a camera-to-world matrix (row-major, 4 columns).  One whose forward
// column is zero or not finite gives a frame of NaNs, which rejects nothing.
__device__ __forceinline__ RowFrame row_frame(const float* __restrict__ m) {
    RowFrame f;
    const float c0 = m[2], c1 = m[6], c2 = m[10];
    const float ic = 1.0f / sqrtf(sqnorm3(c0, c1, c2));
    f.ec[0] = c0 * ic;
    f.ec[1] = c1 * ic;
    f.ec[2] = c2 * ic;
    const bool xaxis = fabsf(f.ec[0]) < 0.6f;
    const float a0 = xaxis ? 1.0f : 0.0f, a1 = xaxis ? 0.0f : 1.0f;
    const float c = a0 * f.ec[0] + a1 * f.ec[1];
    f.e1[0] = a0 - c * f.ec[0];
    f.e1[1] = a1 - c * f.ec[1];
    f.e1[2] = -c * f.ec[2];
    const float n = 1.0f / sqrtf(sqnorm3(f.e1[0], f.e1[1], f.e1[2]));
    f.e1[0] *= n;
    f.e1[1] *= n;
    f.e1[2] *= n;
    f.e2[0] = f.ec[1] * f.e1[2] - f.ec[2] * f.e1[1];
    f.e2[1] = f.ec[2] * f.e1[0] - f.ec[0] * f.e1[2];
    f.e2[2] = f.ec[0] * f.e1[1] - f.ec[1] * f.e1[0];
    f.o[0] = m[3];
    f.o[1] = m[7];
    f.o[2] = m[11];
    f.om = 4e-6f * (1.0f + fabsf(f.o[0]) + fabsf(f.o[1]) + fabsf(f.o[2]));
    return f;
}

// (a, b, T, z) of a point p of radius r (see row_run).  Let w = p - o have
// frame coordinates (x, y, z), a = x / z, b = y / z, and let a ray have
// (alpha, beta) the same way.  The line through the ray is at distance
//   |w| sin(angle) >= |z| sqrt(((a - alpha)^2 + (b - beta)^2) / (1 + alpha^2 + beta^2))
// from p (the cross product of (a, b, 1) and (alpha, beta, 1) is at least its
// first two components, and |w|^2 = z^2 (1 + a^2 + b^2)).  So a point within
// `reach` of the line has (a - alpha)^2 + (b - beta)^2 <= T g with
// T = reach^2 / z^2 and g = 1 + alpha^2 + beta^2.
// `reach` is r plus what the roundings of the exact tests (see cone_clears:
// below 1.1e-6 |w| and 3e-6 (1 + |o|_1), and below 1.1e-6 |w| for a sample
// point's own) and of a, b, alpha, beta here (below 2e-6 |w|; the frame is a
// linear map within 1e-6 of a rotation, which distorts angles by as much)
// can make of it, with room.  Such a point's ray depth t is at least
// |w| - reach^2 / |w| up to 4e-6 |w| when it lies ahead; z is that less
// `reach`, so that a sample point nearer than z cannot have it as neighbour
// either.  Points at more than 87 degrees from the axis get T = inf (always
// tested exactly), and points behind the origin z = -inf; comparisons are
// written so that a NaN is never rejected.
__device__ __forceinline__ float4 row_candidate(const RowFrame& f, const float4& p, float r) {
    const float w0 = p.x - f.o[0], w1 = p.y - f.o[1], w2 = p.z - f.o[2];
    const float x = dot3(w0, w1, w2, f.e1[0], f.e1[1], f.e1[2]);
    const float y = dot3(w0, w1, w2, f.e2[0], f.e2[1], f.e2[2]);
    const float z = dot3(w0, w1, w2, f.ec[0], f.ec[1], f.ec[2]);
    const float aw = __builtin_amdgcn_sqrtf(sqnorm3(w0, w1, w2));
    const float inf = __builtin_inff();
    const float reach = r * (1.0f + 4e-6f) + 8e-6f * aw + f.om;
    const float iz = __builtin_amdgcn_rcpf(z);
    const float q = reach * iz;
    const float T = fabsf(z) > 0.05f * aw ? q * q * (1.0f + 2e-5f) : inf;
    const float zl = z > 0.0f && reach < 0.25f * aw
                         ? aw * (1.0f - 1e-5f) - reach * reach * __builtin_amdgcn_rcpf(aw) * (1.0f + 1e-5f) - reach
                         : -inf;
    return make_float4(x * iz, y * iz, T, zl);
}

// The view's list: points in list order with their candidate form, and the
// squared radius thresholds (per-point radius only).  The candidates are
// followed by kRowPad readable entries.
template <bool PR>
struct RowPoints {
    const float4* pts;
    const float4* cand;
    const float* prad;
};

// Stages n points: of rows [r0, r1) of the region, from the `off`-th of row r0 on.
template <bool PR>
__device__ __forceinline__ void row_stage(const RowPoints<PR>& src, RowSmem<PR>& sm, int r0, int r1, int off, int n) {
    const int base0 = sm.base[r0] + off;
    for (int i = threadIdx.x; i < n; i += kRowThreads) {
        const int q = base0 + i;
        int lo = r0, hi = r1;  // last row whose first point is at or before q
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (sm.base[mid] <= q) lo = mid;
            else hi = mid;
        }
        const int j = sm.lo[lo][0] + (q - sm.base[lo]);
        sm.cand[i] = src.cand[j];
        sm.pts[i] = src.pts[j];
        if constexpr (PR) sm.lim[i] = src.prad[j];
    }
}

// A lane's ray in the view's frame: (alpha, beta), g, and the depth beyond
// which the current sweep has no interest (-inf: the lane rests).
struct RowRay {
    float a, b, g;
    float zb;
};

__device__ __forceinline__ RowRay row_ray(const float* __restrict__ c2w, const Ray& ray) {
    const RowFrame f = row_frame(c2w);
    const float c = dot3(ray.d[0], ray.d[1], ray.d[2], f.ec[0], f.ec[1], f.ec[2]);
    const float ic = c > 0.2f ? 1.0f / c : __builtin_nanf("");  // NaN: nothing is rejected
    RowRay rr;
    rr.a = dot3(ray.d[0], ray.d[1], ray.d[2], f.e1[0], f.e1[1], f.e1[2]) * ic;
    rr.b = dot3(ray.d[0], ray.d[1], ray.d[2], f.e2[0], f.e2[1], f.e2[2]) * ic;
    rr.g = (1.0f + rr.a * rr.a + rr.b * rr.b) * (1.0f + 1e-5f);
    rr.zb = __builtin_inff();
    return rr;
}

// Calls fn(p, lim, dup) for the `len` candidates of a lane's run that the
// bound does not reject, in order; `near` counts those that the radius alone
// does not reject, at any depth.  cand, pts and plim point at the run's first
// entry (LDS or global memory).  Up to 32 candidates at a time: the mask takes
// one bit per candidate from below (an add with carry), so the first
// candidate is its highest bit.  A point is read while the one before it is
// tested.
template <bool PR, class Fn>
__device__ __forceinline__ void row_run(const SampleOpts& o, RowRay& rr, const float4* cand, const float4* pts,
                                        const float* plim, int len, bool dup, int& near, Fn&& fn) {
    for (int c0 = 0; __any(c0 < len); c0 += 32) {
        const int n = len - c0;
        const int at = n > 0 ? c0 : 0;
        uint32_t m = 0, mr = 0;
        int it = 0;
#pragma unroll 1
        do {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 c = cand[at + it + q];
                const float da = c.x - rr.a, db = c.y - rr.b;
                const float s = __builtin_fmaf(db, db, da * da);
                const bool off = s > c.z * rr.g;
                mr = mr + mr + (off ? 0u : 1u);
                m = m + m + (off | (c.w > rr.zb) ? 0u : 1u);
            }
            it += 4;
        } while (it < 32 && __any(it < n));
        if (n < it) {
            m = n > 0 ? m >> (it - n) << (it - n) : 0u;
            mr = n > 0 ? mr >> (it - n) : 0u;
        }
        near += __popc(mr);
        if (m) {
            const int last = c0 + it - 1;
            int hb = 31 - __clz((int)m);
            float4 nxt = pts[last - hb];
            float nlim = PR ? plim[last - hb] : o.r2lim;
            while (true) {
                const int j = last - hb;
                const float4 p = nxt;
                const float lim = nlim;
                m &= ~(1u << hb);
                if (m) {
                    hb = 31 - __clz((int)m);
                    nxt = pts[last - hb];
                    if constexpr (PR) nlim = plim[last - hb];
                }
                fn(p, lim, dup);
                if (j == last - hb) break;
            }
        }
    }
}

// Fills, for each of the wave's nr rays (row stride `per` words from p), the
// words [skip, per) with value: the wave stores consecutive units of 16, 8 or
// 4 bytes, whichever the stride and the alignment allow.
template <class V>
__device__ __forceinline__ void row_fill_units(V* p, int nr, int per, int skip, V value) {
    const int n = per - skip;
    if (n <= 0) return;
    const int lane = __lane_id();
    if (skip == 0) {  // one span
        for (int i = lane; i < nr * per; i += kWave) p[i] = value;
        return;
    }
    // (ray, column) of unit lane, lane + 64, ...
    const int q = kWave / n, rem = kWave - q * n;
    int ray = lane / n, col = lane - ray * n;
    while (ray < nr) {
        p[(int64_t)ray * per + skip + col] = value;
        col += rem;
        ray += q;
        if (col >= n) col -= n, ++ray;
    }
}

__device__ __forceinline__ void row_fill(uint32_t* p, int nr, int per, int skip, uint32_t value) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(p);
    if (per % 4 == 0 && skip % 4 == 0 && (at & 15) == 0)
        row_fill_units(reinterpret_cast<uint4*>(p), nr, per / 4, skip / 4, make_uint4(value, value, value, value));
    else if (per % 2 == 0 && skip % 2 == 0 && (at & 7) == 0)
        row_fill_units(reinterpret_cast<uint2*>(p), nr, per / 2, skip / 2, make_uint2(value, value));
    else
        row_fill_units(p, nr, per, skip, value);
}

// Four consecutive words of an output row (as 16 bytes where `vec`).
__device__ __forceinline__ void row_store4(uint32_t* p, bool vec, int left, const uint32_t (&v)[4]) {
    if (vec) {
        *reinterpret_cast<uint4*>(p) = make_uint4(v[0], v[1], v[2], v[3]);
        return;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (c < left) p[c] = v[c];
}

// Neighbour outputs of sample `so` of ray `ri` (write_neighbours without the
// feature sums, which idw_rows_kernel takes from the weights written here).
template <int MODE, int KMAX, int LAY>
__device__ __forceinline__ void row_write_neighbours(const SampleOpts& o, const SampleOut& out, const Ray& ray,
                                                     const NbBuf<MODE, KMAX>& nb, int64_t ri, int so) {
    const int Kc = o.Kc;
    const int nkeep = nb.bsize < Kc ? nb.bsize : Kc;
    const int64_t row = LAY == kLayDense ? (ri * o.S + so) * (int64_t)Kc : (ri * out.s_max + so) * (int64_t)Kc;
    int* idx = (LAY == kLayDense ? out.pc_idx : out.nb_idx) + row;
    float den = 0.0f;
    if constexpr (LAY == kLayFeat) {
#pragma unroll
        for (int b = 0; b < KMAX; ++b)
            if (b < nkeep) den = den + 1.0f / (nb.bd[b] + 1e-6f);  // (1 / (d + 1e-6)) * mask, epcq.py:436
        den = den + 1e-6f;
    }
    constexpr bool td = MODE == EPCQ_MODE_KNN && LAY != kLayDense;
    const bool vec = Kc % 4 == 0;
    auto aligned = [&](const void* p) { return vec && (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vi = aligned(idx);
    float* nt = td && out.nb_t ? out.nb_t + row : nullptr;
    float* nd = td && out.nb_dist ? out.nb_dist + row : nullptr;
    float* nw = LAY == kLayFeat ? out.w + row : nullptr;
    const bool vt = aligned(nt), vd = aligned(nd), vw = aligned(nw);
    for (int b0 = KMAX; b0 < Kc; ++b0) {  // columns past the buffer
        idx[b0] = -1;
        if (nt) nt[b0] = 0.0f;
        if (nd) nd[b0] = 0.0f;
        if (nw) nw[b0] = 0.0f;
    }
#pragma unroll
    for (int b0 = 0; b0 < KMAX; b0 += 4) {
        if (b0 >= Kc) break;
        const int left = Kc - b0;
        uint32_t v[4];
        float px[4][3];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = b0 + c < nkeep ? (uint32_t)nb.bi[b0 + c] : 0xffffffffu;
        if constexpr (td) {
            if (nt || nd) {  // the four points' loads first, then their tests
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float* p = o.xyz + 3 * (int64_t)(b0 + c < nkeep ? nb.bi[b0 + c] : 0);
                    if (b0 + c < nkeep) {
                        px[c][0] = p[0];
                        px[c][1] = p[1];
                        px[c][2] = p[2];
                    }
                }
            }
        }
        row_store4(reinterpret_cast<uint32_t*>(idx + b0), vi, left, v);
        if constexpr (td) {
            if (nt || nd) {
                uint32_t tv[4], dv[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    tv[c] = dv[c] = 0u;
                    if (b0 + c < nkeep) {
                        float t, e2;
                        ray_t_e2(ray, make_float4(px[c][0], px[c][1], px[c][2], 0.0f), t, e2);
                        tv[c] = __float_as_uint(t);
                        dv[c] = __float_as_uint(sqrtf(e2));
                    }
                }
                if (nt) row_store4(reinterpret_cast<uint32_t*>(nt + b0), vt, left, tv);
                if (nd) row_store4(reinterpret_cast<uint32_t*>(nd + b0), vd, left, dv);
            }
        }
        if constexpr (LAY == kLayFeat) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                v[c] = b0 + c < nkeep ? __float_as_uint((1.0f / (nb.bd[b0 + c] + 1e-6f)) / den) : 0u;
            row_store4(reinterpret_cast<uint32_t*>(nw + b0), vw, left, v);
        }
    }
}

// Empty slots [ns, s_max) of a lane's ray in the compact layouts (write_tail
// without the feature sums).
template <int MODE, int LAY>
__device__ __forceinline__ void row_write_tail(const SampleOpts& o, const SampleOut& out, int64_t ri, int ns) {
    if (ns >= out.s_max) return;
    const int64_t a0 = ri * out.s_max + ns;
    const int n = out.s_max - ns;
    fill_words(reinterpret_cast<uint32_t*>(out.sample_t + a0), n, 0u);
    fill_words(reinterpret_cast<uint32_t*>(out.nb_idx + a0 * o.Kc), n * o.Kc, 0xffffffffu);
    if constexpr (MODE == EPCQ_MODE_KNN) {
        if (out.nb_t) fill_words(reinterpret_cast<uint32_t*>(out.nb_t + a0 * o.Kc), n * o.Kc, 0u);
        if (out.nb_dist) fill_words(reinterpret_cast<uint32_t*>(out.nb_dist + a0 * o.Kc), n * o.Kc, 0u);
    }
    if constexpr (LAY == kLayFeat) fill_words(reinterpret_cast<uint32_t*>(out.w + a0 * o.Kc), n * o.Kc, 0u);
}

// The same for a wave none of whose nr rays (ri0, ri0 + 1, ...) has a sample.
template <int MODE, int LAY>
__device__ __forceinline__ void row_fill_empty(const SampleOpts& o, const SampleOut& out, int64_t ri0, int nr) {
    const int s = out.s_max, sk = s * o.Kc;
    const int64_t a0 = ri0 * s;
    row_fill(reinterpret_cast<uint32_t*>(out.sample_t + a0), nr, s, 0, 0u);
    row_fill(reinterpret_cast<uint32_t*>(out.nb_idx + a0 * o.Kc), nr, sk, 0, 0xffffffffu);
    if constexpr (MODE == EPCQ_MODE_KNN) {
        if (out.nb_t) row_fill(reinterpret_cast<uint32_t*>(out.nb_t + a0 * o.Kc), nr, sk, 0, 0u);
        if (out.nb_dist) row_fill(reinterpret_cast<uint32_t*>(out.nb_dist + a0 * o.Kc), nr, sk, 0, 0u);
    }
    if constexpr (LAY == kLayFeat) row_fill(reinterpret_cast<uint32_t*>(out.w + a0 * o.Kc), nr, sk, 0, 0u);
}

// Slots [from, S) of the wave's nr rays in the dense layout.
__device__ __forceinline__ void row_fill_dense(const SampleOpts& o, const SampleOut& out, int64_t ri0, int nr,
                                               int from) {
    const int S = o.S;
    if (S <= from) return;
    const int64_t a0 = ri0 * S;
    row_fill(reinterpret_cast<uint32_t*>(out.sp_xyz + 3 * a0), nr, 3 * S, 3 * from, 0u);
    row_fill(reinterpret_cast<uint32_t*>(out.sp_t + a0), nr, S, from, 0u);
    row_fill(reinterpret_cast<uint32_t*>(out.pc_idx + a0 * o.Kc), nr, S * o.Kc, from * o.Kc, 0xffffffffu);
    uint8_t* m = out.mask + a0;
    const uintptr_t at = reinterpret_cast<uintptr_t>(m);
    if (S % 4 == 0 && from % 4 == 0 && at % 4 == 0)
        row_fill_units(reinterpret_cast<uint32_t*>(m), nr, S / 4, from / 4, 0u);
    else if (S % 2 == 0 && from % 2 == 0 && at % 2 == 0)
        row_fill_units(reinterpret_cast<uint16_t*>(m), nr, S / 2, from / 2, (uint16_t)0);
    else
        row_fill_units(m, nr, S, from, (uint8_t)0);
}

// One 64 x 4 tile of a view; the output row of ray (u, v) is v * W + u.
template <int MODE, int KMAX, int LAY, bool PR>
__device__ __forceinline__ void row_tile_body(const SampleOpts& o, const SampleOut& out, const ViewArgs& view,
                                              int tile, int tiles_x, RowQueue* queue, RowSmem<PR>& sm) {
    const int W = view.W, H = view.H, k = o.k, ko = o.ko;
    const int wave = uniform((int)threadIdx.x / kWave), lane = __lane_id();
    const int u0 = (tile % tiles_x) * kRowTileW, v0 = (tile / tiles_x) * kRowTileH;
    const int u = u0 + lane, v = v0 + wave;
    const bool inside = u < W && v < H;
    int ra, va, RW, RH;
    tile_region(W, H, k, ko, u0, v0, kRowTileW, kRowTileH, ra, va, RW, RH);
    const RowPoints<PR> src{view.pts, view.cand, view.prad};

    // ---- the region's rows: lo[r][x] is the start of the first bucket at or
    // right of column x, lo[r][RW] the row's end, so that columns [x0, x1] hold
    // the positions [lo[x0], lo[x1 + 1])
    // a tile of background is done here
    bool some = false;
    for (int r = wave; r < RH; r += kRowTileH)
        for (int x = lane; x < RW; x += kWave) some |= view.hash[(int64_t)(va + r) * W + ra + x].y > 0;
    if (!__syncthreads_or(some)) {
        const int nr = v < H ? min(kRowTileW, W - u0) : 0;
        const int64_t ri0 = (int64_t)v * W + u0;
        if (nr <= 0) return;
        if constexpr (LAY == kLayDense) {
            row_fill_dense(o, out, ri0, nr, 0);
        } else {
            if (inside) out.n_samples[ri0 + lane] = 0;
            row_fill_empty<MODE, LAY>(o, out, ri0, nr);
        }
        return;
    }
    int flags = 0;
    for (int r = wave; r < RH; r += kRowTileH) {
        const int2* h = view.hash + (int64_t)(va + r) * W + ra;
        int s[2], e[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int x = kWave * c + lane;
            const int2 q = x < RW ? h[x] : make_int2(-1, -1);
            s[c] = q.y > 0 ? q.x : INT_MAX;
            e[c] = q.y > 0 ? q.x + q.y : INT_MIN;
            if (q.y > kSampleLaneHits) flags |= kRowBigBucket;
        }
        int end = max(e[0], e[1]);
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) end = max(end, __shfl_xor(end, d));
        if (end == INT_MIN) end = 0;  // an empty row: every run is empty
        int f[2] = {s[0], s[1]};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int y = __shfl_down(f[c], d);
                if (lane + d < kWave) f[c] = min(f[c], y);
            }
        }
        f[0] = min(f[0], __shfl(f[1], 0));
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (f[c] == INT_MAX) f[c] = end;
            const int x = kWave * c + lane;
            if (x <= RW) sm.lo[r][x] = x < RW ? f[c] : end;
        }
        // every bucket ends where the next one of its row starts
        const int n0 = __shfl_down(f[0], 1), n1 = __shfl_down(f[1], 1), f10 = __shfl(f[1], 0);
        if (s[0] != INT_MAX && e[0] != (lane == kWave - 1 ? f10 : n0)) flags |= kRowIrregular;
        if (s[1] != INT_MAX && e[1] != (lane == kWave - 1 ? end : n1)) flags |= kRowIrregular;
    }
    flags = (__any(flags & kRowIrregular) ? kRowIrregular : 0) | (__any(flags & kRowBigBucket) ? kRowBigBucket : 0);
    if (lane == 0) sm.flags[wave] = flags;

    __syncthreads();
    if (wave == 0) {
        const int len = lane < RH ? sm.lo[lane][RW] - sm.lo[lane][0] : 0;
        int x = len;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {
            const int y = __shfl_up(x, d);
            if (lane >= d) x += y;
        }
        if (lane < RH) sm.base[lane] = x - len;
        if (lane == RH - 1) sm.base[RH] = x;
    }
    __syncthreads();
    flags = uniform(sm.flags[0] | sm.flags[1] | sm.flags[2] | sm.flags[3]);
    const bool staged_once = uniform(sm.base[RH]) <= kRowCap;
    Ray ray;
    view_ray(view, min(u, W - 1), min(v, H - 1), ray);
    RowRay rr = row_ray(view.c2w, ray);
#pragma unroll
    for (int i = 0; i < 3; ++i) ray.o[i] = uniform(ray.o[i]);

    // ---- the lane's window: columns [x0, x1] of the region, and the repeats
    // of the image's edge columns that clamping makes (cl before, cr after)
    const int x0 = min(max(u - (ko - 1), 0), W - 1) - ra, x1 = min(u + (k - ko), W - 1) - ra;
    const int rw0 = max(0, v + 1 - ko) - va, rw1 = v < H ? min(H - 1, v + k - ko) - va + 1 : 0;
    const int top = max(0, ko - 1 - v), bottom = max(0, v + (k - ko) - (H - 1));
    const int nleft = u0 < ko - 1 ? ko - 1 : 0, nright = u0 + kRowTileW + (k - ko) > W ? k - ko : 0;

    // an irregular table's rows overlap: nothing of them is staged
    const int RS = flags & kRowIrregular ? 0 : RH;
    bool defer = inside && (flags & kRowIrregular);
    bool live = inside && !defer;  // lanes the sweeps still work for
    if (!staged_once) {
        // a long row is staged in pieces, each of which serves only the few
        // rays whose windows it meets (and a clamped window would revisit the
        // row in an order that pieces cannot give)
        int longest = 0;
        for (int r = 0; r < RH; ++r) longest = max(longest, uniform(sm.base[r + 1] - sm.base[r]));
        const bool clamped = u < ko - 1 || u + (k - ko) > W - 1 || top > 0 || bottom > 0;
        if (live && (longest > row_longest(k) || (longest > kRowCap && clamped))) {
            defer = true;
            live = false;
        }
    }
    if (!staged_once && o.heavy > 0) {
        int64_t cand = 0;
        if (live)
            for (int r = rw0; r < rw1; ++r) cand += sm.lo[r][x1 + 1] - sm.lo[r][x0];
        const int64_t most = (int64_t)o.row_heavy * o.heavy;
        const int above = __popcll(__ballot(cand > most));
        if (cand > most && (above <= kHeavyMinority || cand > 4 * most)) {
            defer = true;
            live = false;
        }
    }

    // fn(p, lim, dup) for every candidate of every lane's window that passes
    // the bound, in the canonical order; after_row() after each of the wave's
    // rows.  Block-wide, except that a tile that is staged in one piece holds
    // no barrier after its first sweep.
    int near = 0;
    bool staged = false;
    auto sweep = [&](auto&& fn, auto&& after_row) {
        int r0 = 0, off = 0;
        while (r0 < RS) {
            // the next points to stage: whole rows [r0, r1), or a piece of row r0 from `off` on
            int r1 = r0 + 1;
            const int base0 = uniform(sm.base[r0]), len0 = uniform(sm.base[r0 + 1]) - base0;
            int n = len0 - off;
            if (n > kRowCap) {
                n = kRowCap;
            } else if (off == 0) {
                while (r1 < RH && uniform(sm.base[r1 + 1]) - base0 <= kRowCap) ++r1;
                n = uniform(sm.base[r1]) - base0;
            }
            if (!(staged && staged_once)) {
                if (staged) __syncthreads();  // the points staged before have been read
                row_stage<PR>(src, sm, r0, r1, off, n);
                __syncthreads();
                staged = true;
            }
            for (int r = max(r0, rw0); r < min(r1, rw1); ++r) {
                const int y = va + r;
                const int rep = 1 + (y == 0 ? top : 0) + (y == H - 1 ? bottom : 0);
                const int row0 = uniform(sm.lo[r][0]), at = uniform(sm.base[r]) - base0 - off - row0;
                const int from = row0 + (r == r0 ? off : 0);  // staged positions of this row
                const int to = r == r1 - 1 ? n - at : uniform(sm.lo[r][RW]);
                for (int rp = 0; rp < rep; ++rp) {
                    for (int part = -nleft; part <= nright; ++part) {
                        // repeats of the edge columns: ko - 1 - u before, u + k - ko - (W - 1) after
                        const bool use =
                            live && (part == 0 || (part < 0 ? -part <= ko - 1 - u : part <= u + (k - ko) - (W - 1)));
                        const int xa = part < 0 ? 0 : part > 0 ? RW - 1 : x0;
                        const int xb = part < 0 ? 0 : part > 0 ? RW - 1 : x1;
                        const int s = use ? max(sm.lo[r][xa], from) : 0;
                        const int len = use ? min(sm.lo[r][xb + 1], to) - s : 0;
                        const int l = len > 0 ? at + s : 0;
                        row_run<PR>(o, rr, sm.cand + l, sm.pts + l, sm.lim + (PR ? l : 0), len, rp > 0 || part != 0,
                                    near, fn);
                    }
                }
                after_row();
            }
            if (off + n < len0) {
                off += n;
            } else {
                r0 = r1;
                off = 0;
            }
        }
    };

    const float inf = __builtin_inff();
    const int64_t ri = (int64_t)v * W + u;
    float tmin = 1e3f;
    bool any = false;
    int s0 = kMaxSlots, s1 = kMaxSlots;
    float sum0 = 0.0f, cnt0 = 0.0f, sum1 = 0.0f, cnt1 = 0.0f;
    int ns = 0;
    bool touched = false;  // the lane has streamed indices to its output rows
    const bool bounded = o.t_intvl > 0.0f;
    auto slot_end = [&](int s) {  // a depth that no hit of slot s reaches
        return bounded ? tmin + (float)(s + 1) * o.t_intvl + (1e-3f * o.t_intvl + 1e-6f * fabsf(tmin)) : inf;
    };
    // ---- sweep 1: tmin.  Sweep 2: the first two slots with at least two hits.
    // One loop, so that both share their code.
    SlotMask seen1{0u, 0u, 0u, 0u}, seen2{0u, 0u, 0u, 0u};
    bool fresh = false;
#pragma unroll 1
    for (int step = 0; step < 2; ++step) {
        rr.zb = live ? (step == 0 ? inf : slot_end(kMaxSlots)) : -inf;
        sweep(
            [&](const float4& p, float lim, bool) {
                float t, e2;
                ray_t_e2(ray, p, t, e2);
                if (!within(e2, lim)) return;
                if (step == 0) {
                    any = true;
                    if (tmin > t) tmin = t;
                    rr.zb = tmin;
                    return;
                }
                const float qf = (t - tmin) / o.t_intvl;
                if (!(qf > -1.0f && qf < (float)kMaxSlots)) return;
                const SlotMask b = slot_bit((int)qf);
                seen2.w0 |= seen1.w0 & b.w0;
                seen2.w1 |= seen1.w1 & b.w1;
                seen2.w2 |= seen1.w2 & b.w2;
                seen2.w3 |= seen1.w3 & b.w3;
                seen1.w0 |= b.w0;
                seen1.w1 |= b.w1;
                seen1.w2 |= b.w2;
                seen1.w3 |= b.w3;
                fresh = true;
            },
            [&] {
                if (step == 0 || !__any(fresh)) return;
                fresh = false;
                s0 = next_slot(seen2, 0);
                s1 = s0 < kMaxSlots ? next_slot(seen2, s0 + 1) : kMaxSlots;
                if (s1 < kMaxSlots) rr.zb = slot_end(s1);
            });
        if (step == 0) {
            if ((flags & kRowBigBucket) && near > kSampleLaneHits && live) {
                // with 48 candidates or fewer in all, no bucket has more hits
                defer = true;
                live = false;
            }
            live = live && any;
            if (staged_once ? !__any(live) : !__syncthreads_or(live)) break;
        }
    }
    live = live && s0 < kMaxSlots;
    // ---- sweep 3: sums of the two slots and neighbours of their samples.
    // Buffers of more than 8 take a sweep per sample: two of them would halve
    // the waves that fit a SIMD.
    const bool two = s1 < kMaxSlots;
    const float ts0 = tmin + (float)s0 * o.t_intvl, ts1 = tmin + (float)s1 * o.t_intvl;
    const int room = LAY == kLayDense ? min(o.S, 2) : min(out.s_max, 2);  // samples with a place in the outputs
    constexpr bool stream = MODE == EPCQ_MODE_COMPAT && LAY != kLayFeat;
    using Buf = typename std::conditional<stream, CompatStream<KMAX>, NbBuf<MODE, KMAX>>::type;
    constexpr int NS = stream ? 2 : 1;
    touched = stream && live;
#pragma unroll 1
    for (int so0 = 0; so0 < 2; so0 += NS) {
        const bool work = live && (so0 == 0 || so0 < min(ns, room));
        if (staged_once ? !__any(work) : !__syncthreads_or(work)) break;
        float sp[NS][3];
        bool want[NS];
        Buf buf[NS];
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            const int so = so0 + q;
            const float ts = so == 0 ? ts0 : ts1;
            sp[q][0] = ray.o[0] + ts * ray.d[0];
            sp[q][1] = ray.o[1] + ts * ray.d[1];
            sp[q][2] = ray.o[2] + ts * ray.d[2];
            want[q] = so < room && (so == 0 || two);
            if constexpr (stream) {
                int* row = LAY == kLayDense ? out.pc_idx + (ri * o.S + so) * (int64_t)o.Kc
                                            : out.nb_idx + (ri * out.s_max + so) * (int64_t)o.Kc;
                buf[q].init(row, want[q] ? o.Kc : 0);
            } else {
                buf[q].init();
            }
        }
        rr.zb = work ? slot_end(two ? s1 : s0) : -inf;
        sweep(
            [&](const float4& p, float lim, bool dup) {
                if (so0 == 0) {
                    float t, e2;
                    ray_t_e2(ray, p, t, e2);
                    const float qf = (t - tmin) / o.t_intvl;
                    const int s = within(e2, lim) && qf > -1.0f && qf < (float)kMaxSlots ? (int)qf : -1;
                    if (s == s0 || s == s1) {
                        const float dist = sqrtf(e2);
                        sum0 = s == s0 ? sum0 + dist : sum0;
                        cnt0 = s == s0 ? cnt0 + 1.0f : cnt0;
                        sum1 = s == s1 ? sum1 + dist : sum1;
                        cnt1 = s == s1 ? cnt1 + 1.0f : cnt1;
                    }
                }
                if (MODE == EPCQ_MODE_KNN && dup) return;  // distinct window pixels only
                const int id = __float_as_int(p.w);
#pragma unroll
                for (int q = 0; q < NS; ++q) {
                    const float d2 = sqnorm3(sp[q][0] - p.x, sp[q][1] - p.y, sp[q][2] - p.z);
                    if (want[q] && within(d2, lim)) buf[q].add(sqrtf(d2), id);
                }
            },
            [] {});
        if (so0 == 0 && live) {
            // the front-to-back walk over the two slots (epcq_render_topk.cu:168-219)
            float T = 1.0f;
            bool em0 = false, em1 = false, open = false;
            if (!(T < 1e-3f || ns >= o.S)) {
                const float a0 = o.gamma * expf_cw(-(sum0 / (cnt0 + 1e-6f)) / o.alpha_p);
                em0 = a0 * T > 1e-3f;
                if (em0) ++ns;
                T -= a0;
                if (two && !(T < 1e-3f || ns >= o.S)) {
                    const float a1 = o.gamma * expf_cw(-(sum1 / (cnt1 + 1e-6f)) / o.alpha_p);
                    em1 = a1 * T > 1e-3f;
                    if (em1) ++ns;
                    T -= a1;
                    open = !(T < 1e-3f || ns >= o.S);  // a third slot could follow
                }
            }
            if (open || (em1 && !em0)) {
                defer = true;
                live = false;
                ns = 0;
            }
        }
        if (live) {
#pragma unroll
            for (int q = 0; q < NS; ++q) {
                const int so = so0 + q;
                if (so < ns && so < room) {
                    write_sample<LAY>(o, out, ray, ri, so, so == 0 ? ts0 : ts1);
                    if constexpr (stream) buf[q].finish();
                    else row_write_neighbours<MODE, KMAX, LAY>(o, out, ray, buf[q], ri, so);
                }
            }
        }
    }
    // ---- everything not written above: zeros / -1 / false
    const int nr = v < H ? min(kRowTileW, W - u0) : 0;
    const int64_t ri0 = (int64_t)v * W + u0;
    if constexpr (LAY == kLayDense) {
        if (nr > 0) row_fill_dense(o, out, ri0, nr, 2);  // no ray of this path has a third sample
        if (inside && ns < min(o.S, 2)) {
            const int64_t a0 = ri * o.S + ns;
            const int n = min(o.S, 2) - ns;
            fill_words(reinterpret_cast<uint32_t*>(out.sp_xyz + 3 * a0), 3 * n, 0u);
            fill_words(reinterpret_cast<uint32_t*>(out.sp_t + a0), n, 0u);
            fill_words(reinterpret_cast<uint32_t*>(out.pc_idx + a0 * o.Kc), n * o.Kc, 0xffffffffu);
            for (int q = 0; q < n; ++q) out.mask[a0 + q] = 0;
        }
    } else {
        if (inside) out.n_samples[ri] = ns;
        if (!__any(ns > 0 || touched)) {
            if (nr > 0) row_fill_empty<MODE, LAY>(o, out, ri0, nr);
        } else if (inside) {
            row_write_tail<MODE, LAY>(o, out, ri, ns);
        }
    }
    if (const uint64_t db = __ballot(defer)) {
        int at = 0;
        if (lane == 0) at = atomicAdd(&queue->count, __popcll(db));
        at = __shfl(at, 0);
        if (defer) queue->ray[at + __popcll(db & lanemask_lt())] = v * W + u;
    }
}

// Inverse-distance weighted feature sums of the compact rows (ray, sample
// slot) from the neighbour indices and weights that the sampler wrote: G
// lanes per row, four features each, so that a neighbour's features are read
// by adjacent lanes and several neighbours' loads are in flight (one lane per
// row waited for each neighbour's in turn).  Sums run over the neighbours in
// order, as write_neighbours takes them.
constexpr int kIdwUnroll = 4;

template <bool BF16, bool VEC>
__global__ __launch_bounds__(256) void idw_rows_kernel(const void* __restrict__ feat, int F, int G, int64_t rows,
                                                       int K, const int* __restrict__ nb_idx,
                                                       const float* __restrict__ w, float* __restrict__ agg) {
    const int per = 256 / G;  // rows of a block
    const int blk = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int g = (int)threadIdx.x % G, rl = (int)threadIdx.x / G;
    const int64_t row = (int64_t)blk * per + rl;
    if (rl >= per || row >= rows) return;
    const int* ids = nb_idx + row * K;
    const float* ws = w + row * K;
    for (int f0 = 4 * g; f0 < F; f0 += 4 * G) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int b0 = 0; b0 < K; b0 += kIdwUnroll) {
            int id[kIdwUnroll];
            float wb[kIdwUnroll], fv[kIdwUnroll][4];
#pragma unroll
            for (int c = 0; c < kIdwUnroll; ++c) {
                id[c] = b0 + c < K ? ids[b0 + c] : -1;
                wb[c] = b0 + c < K ? ws[b0 + c] : 0.0f;
            }
            if (id[0] < 0) break;  // valid neighbours come first
#pragma unroll
            for (int c = 0; c < kIdwUnroll; ++c) {
                if (id[c] < 0) continue;
                const int64_t at = (int64_t)id[c] * F + f0;
                if constexpr (VEC && BF16) {
                    const uint2 h = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(feat) + at);
                    fv[c][0] = __uint_as_float(h.x << 16);
                    fv[c][1] = __uint_as_float(h.x & 0xffff0000u);
                    fv[c][2] = __uint_as_float(h.y << 16);
                    fv[c][3] = __uint_as_float(h.y & 0xffff0000u);
                } else if constexpr (VEC) {
                    const float4 q = *reinterpret_cast<const float4*>(static_cast<const float*>(feat) + at);
                    fv[c][0] = q.x;
                    fv[c][1] = q.y;
                    fv[c][2] = q.z;
                    fv[c][3] = q.w;
                } else {
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        fv[c][x] = 0.0f;
                        if (f0 + x < F)
                            fv[c][x] = BF16 ? __uint_as_float((uint32_t)static_cast<const uint16_t*>(feat)[at + x] << 16)
                                            : static_cast<const float*>(feat)[at + x];
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < kIdwUnroll; ++c) {
                if (id[c] < 0) continue;
#pragma unroll
                for (int x = 0; x < 4; ++x) acc[x] = acc[x] + wb[c] * fv[c][x];
            }
        }
        float* ao = agg + row * F + f0;
        if (VEC && (reinterpret_cast<uintptr_t>(agg) & 15) == 0) {
            *reinterpret_cast<float4*>(ao) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (f0 + x < F) ao[x] = acc[x];
        }
    }
}

}  // namespace epcq
