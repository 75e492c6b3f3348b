// One ray by one wave, over row runs: the form of short ray lists and of the
// rays that the row-run tiles defer (epcq_rows.h).
//
// Each window row is a group of lanes that read the row's hash entries.  A row
// becomes one segment of consecutive list positions (plus one per column that
// clamping repeats), and the wave takes the concatenated candidates of all
// segments 64 at a time, whatever bucket they are in: the 75 candidates of an
// ordinary 5 x 5 window are two steps instead of 25, and the first kWaveCache
// chunks stay in registers for all walks, so a ray waits for memory twice
// (hash entries, points).  For a ray of more than kWaveCache chunks, a first
// pass tests only the candidate bounds (row_candidate; worked out on the way
// where the view has no copy of them) and leaves the positions that pass in
// LDS; the walks then take these.  Where they are too many, the pass is
// repeated without what lies more than kWaveDepth slots behind the first hit
// found so far (a walk that would have to go on there starts again with every
// candidate).  Where that leaves too many as well, what is listed is the chunks
// of 64 that hold a candidate within the bound, and the walks take all of
// these.  Where the table's buckets are not in row-major list order, every
// bucket is a segment of its own.
//
// The 48-hit cap counts hits per bucket: where a bucket holds more points than
// that, each candidate's bucket is found from its row's column starts, and the
// depth limit is off; a walk over the hits leaves a bucket after its 48th.
//
// The order-dependent steps are those of run_ray_wave: sums and neighbours
// take the candidates in the canonical order, lowest lane first.
//
// What bounds it: the latency of those two waits on a short list (4096 rays of
// 1M points at 800 x 800, k = 5: 57 -> 32 us against run_ray_wave), instruction
// issue on an image (600k points at 160 x 100, k = 9, build included: 1.82 ->
// 0.22 ms against the lane-set tiles), and the densest ray's wave where most of
// the points fall to few pixels.  The chunk list and the end at the 48th hit are
// for those, against walks over all candidates: 2726 rays of 1.4M points at 224
// x 170, k = 5, 1.41 -> 0.56 ms (lane sets 0.84); an image of 1.3M points at 240
// x 136, k = 15, 3.90 -> 1.07; over 150 images without features 2.6 % on
// average, over 500 lists 0.8 %, and neither way for most.
#pragma once

#include "epcq_rows.h"

namespace epcq {

constexpr int kWaveCache = 3;    // chunks of 64 candidates kept in registers
constexpr int kWaveList = 1024;  // positions that pass the bound, at most (else the walks take every candidate)
constexpr int kWaveDepth = 32;   // depth slots that the list covers

struct RowWaveSmem {
    int64_t pre[kRowMaxK * kRowMaxK];  // candidates before the segment
    int st[kRowMaxK * kRowMaxK];       // its first list position; sign bit: a repeat made by clamping
    uint8_t row[kRowMaxK * kRowMaxK];  // its window row, or kOneBucket
    int col[kRowMaxK][kRowMaxK];       // per window row and column: where the first bucket at or right of it starts
    int hist[kMaxSlots];               // hits per depth slot
    int pos[kWaveList];                // list positions that pass the bound, or first ones of chunks
    uint8_t seg[kWaveList];            // their segments
};

// What the walks of a ray go over: the segments' candidates, or the positions in
// pos; for a ray of more than these hold (its own instance of the walks, so that
// the others stay short), the chunks that start at the positions in pos, or all
// candidates where they are too many as well.
enum RowWaveOver { kOverAll, kOverList, kOverChunks };

// List point j and the squared threshold of its radius, from the pixel-ordered
// copies where there are any.
template <bool PR>
struct RowList {
    const float4* pts;      // or nullptr (gather by index)
    const float* prad;      // or nullptr
    const int* sorted_idx;
    const float* xyz;
    const float* radius;
    __device__ __forceinline__ float4 point(int j) const {
        if (pts) return pts[j];
        const int id = sorted_idx[j];
        const float* p = xyz + 3 * (int64_t)id;
        return make_float4(p[0], p[1], p[2], __int_as_float(id));
    }
    __device__ __forceinline__ float limit(const SampleOpts& o, int j, const float4& p) const {
        if constexpr (!PR) return o.r2lim;
        else return prad ? prad[j] : point_threshold(radius[__float_as_int(p.w)]);
    }
};

constexpr int kOneBucket = 255;

// Orders the wave's LDS accesses (its lanes exchange data through LDS without
// a block barrier).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Neighbour outputs of sample `so` with the wave's lanes sharing the columns
// (the buffer is the same in every lane), as write_neighbours computes them.
template <int MODE, int KMAX, int LAY>
__device__ __forceinline__ void row_wave_write(const SampleOpts& o, const SampleOut& out, const Ray& ray,
                                               const NbBuf<MODE, KMAX>& nb, int64_t ri, int so) {
    if constexpr (LAY == kLayFeat) {
        write_neighbours_wave<MODE, KMAX>(o, out, ray, nb, ri, so);
    } else {
        const int lane = __lane_id();
        const int nkeep = nb.bsize < o.Kc ? nb.bsize : o.Kc;
        const int64_t row = LAY == kLayDense ? (ri * o.S + so) * (int64_t)o.Kc : (ri * out.s_max + so) * (int64_t)o.Kc;
        int* idx = (LAY == kLayDense ? out.pc_idx : out.nb_idx) + row;
        for (int b = lane; b < o.Kc; b += kWave) {
            int id = -1;
#pragma unroll
            for (int c = 0; c < KMAX; ++c)
                if (c == b) id = nb.bi[c];
            const bool valid = b < KMAX && b < nkeep;
            idx[b] = valid ? id : -1;
            if constexpr (MODE == EPCQ_MODE_KNN && LAY == kLayCompact) {
                if (out.nb_t || out.nb_dist) {
                    float t = 0.0f, dist = 0.0f;
                    if (valid) {
                        const float* p = o.xyz + 3 * (int64_t)id;
                        float e2;
                        ray_t_e2(ray, make_float4(p[0], p[1], p[2], 0.0f), t, e2);
                        dist = sqrtf(e2);
                    }
                    if (out.nb_t) out.nb_t[row + b] = t;
                    if (out.nb_dist) out.nb_dist[row + b] = dist;
                }
            }
        }
    }
}

// The walks of one ray over its N candidates (all C of the segments, the listed
// positions, or 64 for each listed chunk) and its outputs.  Returns true when
// the list left out (`dropped`) what the walk needs; nothing written then stays.
template <int MODE, int KMAX, int LAY, bool PR, bool MANY>
__device__ __forceinline__ bool row_wave_walks(const SampleOpts& o, const SampleOut& out, const RowList<PR>& src,
                                               const Ray& ray, int64_t ri, RowWaveSmem& sm, int nseg, int64_t C,
                                               int64_t N, RowWaveOver over, bool dropped, bool capped) {
    const int lane = __lane_id();
    // ---- candidates, 64 at a time
    struct Cand {
        float4 p;
        float t, e2, lim;
        int seg;
        bool in, keep, dup;
    };
    struct Carry {
        int seg, kept;
    };
    auto segment_end = [&](int seg) {  // the list position after it
        const int64_t p1 = seg + 1 < nseg ? sm.pre[seg + 1] : C;
        return (sm.st[seg] & 0x7fffffff) + (int)(p1 - sm.pre[seg]);
    };
    auto load = [&](int64_t c0) {
        Cand x;
        const int64_t i = c0 + lane;
        x.in = i < N;
        x.seg = -1;
        x.dup = false;
        x.p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        x.lim = 0.0f;
        if (MANY && over == kOverChunks)
            x.in = x.in && sm.pos[c0 / kWave] + lane < segment_end(sm.seg[c0 / kWave]);
        if (x.in) {
            int j;
            if (!MANY && over == kOverList) {
                x.seg = sm.seg[i];
                j = sm.pos[i];
            } else if (MANY && over == kOverChunks) {
                x.seg = sm.seg[c0 / kWave];
                j = sm.pos[c0 / kWave] + lane;
            } else {
                int lo = 0, hi = nseg;  // last segment that starts at or before i
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (sm.pre[mid] <= i) lo = mid;
                    else hi = mid;
                }
                x.seg = lo;
                j = (sm.st[lo] & 0x7fffffff) + (int)(i - sm.pre[lo]);
            }
            x.dup = sm.st[x.seg] < 0;
            if (capped) {  // from here on the candidate's bucket visit
                const int r = sm.row[x.seg];
                int col = 0;
                if (r != kOneBucket)
                    for (int q = 1; q < o.k; ++q)
                        if (sm.col[r][q] <= j) col = q;
                x.seg = x.seg * kRowMaxK + col;
            }
            x.p = src.point(j);
            x.lim = src.limit(o, j, x.p);
        }
        return x;
    };
    // exact test, and the 48-hit cap per bucket visit; cy: hits so far of the
    // visit that the chunk before ended in
    auto test = [&](Cand& x, int64_t c0, Carry& cy) {
        ray_t_e2(ray, x.p, x.t, x.e2);
        const bool hit = x.in && within(x.e2, x.lim);
        x.keep = hit;
        if (capped) {
            const uint64_t hb = __ballot(hit);
            // hits of the lane's own visit: from its first lane in the chunk on
            const int before = __shfl_up(x.seg, 1);
            const uint64_t starts = __ballot(lane == 0 || before != x.seg);
            const int from = 63 - __clzll((long long)(starts & (lanemask_lt() | (1ull << lane))));
            const uint64_t next = from < 63 ? starts & (~0ull << (from + 1)) : 0ull;
            const uint64_t own = hb & (~0ull << from) & (next ? (1ull << (__ffsll((unsigned long long)next) - 1)) - 1ull
                                                              : ~0ull);
            x.keep = hit && __popcll(own & lanemask_lt()) + (x.seg == cy.seg ? cy.kept : 0) < kSampleLaneHits;
            const int last = MANY ? 63 - __clzll((long long)__ballot(x.in))  // the lanes of a chunk come first
                                  : (int)min<int64_t>(kWave, N - c0) - 1;
            const int total = __popcll(own) + (x.seg == cy.seg ? cy.kept : 0);
            cy.kept = lane_bcast(total, last);
            cy.seg = lane_bcast(x.seg, last);
        }
    };
    constexpr int kCache = MANY ? 0 : kWaveCache;  // chunks kept for all walks
    Cand cache[MANY ? 1 : kWaveCache];
#pragma unroll
    for (int q = 0; q < kCache; ++q) cache[q] = load((int64_t)q * kWave);
    Carry cy0{-1, 0};
#pragma unroll
    for (int q = 0; q < kCache; ++q)
        if ((int64_t)q * kWave < N) test(cache[q], (int64_t)q * kWave, cy0);
        else cache[q].keep = false;
    // The next chunk of a walk over the hits: where the bucket visit that the
    // last one ended in has given its 48, not before the visit's end (a bucket
    // may hold tens of thousands of points).
    auto past_full = [&](int64_t c0, const Carry& cy) -> int64_t {
        if (!MANY || !capped || cy.kept < kSampleLaneHits) return c0;
        const int seg = cy.seg / kRowMaxK, col = cy.seg % kRowMaxK, r = sm.row[seg];
        const int st = sm.st[seg] & 0x7fffffff;
        const int end = r != kOneBucket && col + 1 < o.k ? sm.col[r][col + 1] : segment_end(seg);
        if (over == kOverAll) return max<int64_t>(c0, sm.pre[seg] + (end - st));
        while (c0 < N && sm.seg[c0 / kWave] == seg && sm.pos[c0 / kWave] + kWave <= end) c0 += kWave;
        return c0;
    };
    auto walk = [&](bool hits, auto&& fn) {
#pragma unroll
        for (int q = 0; q < kCache; ++q)
            if ((int64_t)q * kWave < N) fn(cache[q]);
        Carry cy = cy0;
        int64_t c0 = (int64_t)kCache * kWave;
        while (c0 < N) {
            Cand x = load(c0);
            test(x, c0, cy);
            fn(x);
            c0 += kWave;
            if (hits) c0 = past_full(c0, cy);
        }
    };

    // ---- step 1: tmin / tmax
    int ns = 0;
    float ts_arr[2] = {0.0f, 0.0f};
    float tmin = 1e3f, tmax = -1e3f;
    walk(true, [&](const Cand& x) {
        if (x.keep) {
            tmin = tmin > x.t ? x.t : tmin;
            tmax = tmax < x.t ? x.t : tmax;
        }
    });
    tmin = wave_min(tmin);
    tmax = wave_max(tmax);
    if (!(tmin > tmax)) {
        // ---- step 2: hits per slot
        auto slot = [&](const Cand& x) {
            const float qf = (x.t - tmin) / o.t_intvl;
            return x.keep && qf > -1.0f && qf < (float)kMaxSlots ? (int)qf : -1;
        };
        walk(true, [&](const Cand& x) {
            const int s = slot(x);
            if (s >= 0) atomicAdd(&sm.hist[s], 1);
        });
        wave_lds_fence();
        const int n0 = sm.hist[lane], n1 = sm.hist[lane + kWave];
        uint64_t two[2] = {__ballot(n0 >= 2), __ballot(n1 >= 2)};
        if (dropped) {  // complete below kWaveDepth only
            two[0] &= (1ull << kWaveDepth) - 1ull;
            two[1] = 0;
        }
        // ---- step 3: front-to-back walk over the slots with >= 2 hits, each
        // slot's distances summed in walk order when it is reached
        float T = 1.0f;
        for (int half = 0; half < 2; ++half) {
            uint64_t b = two[half];
            bool stop = false;
            while (b) {
                if (T < 1e-3f || ns >= o.S) {
                    stop = true;
                    break;
                }
                const int x = __ffsll((unsigned long long)b) - 1;
                b &= b - 1ull;
                const int sl = half * kWave + x;
                float sum = 0.0f;
                walk(true, [&](const Cand& h) {
                    const bool in_slot = slot(h) == sl;
                    const float dist = in_slot ? sqrtf(h.e2) : 0.0f;
                    for (uint64_t m = __ballot(in_slot); m; m &= m - 1ull)
                        sum = sum + lane_bcast(dist, __ffsll((unsigned long long)m) - 1);
                });
                const float cnt = (float)lane_bcast(half == 0 ? n0 : n1, x);
                const float sdf = sum / (cnt + 1e-6f);
                const float alpha = o.gamma * expf_cw(-sdf / o.alpha_p);
                const float wgt = alpha * T;
                if (wgt > 1e-3f) {
                    const float ts = tmin + (float)sl * o.t_intvl;
                    if (lane == 0) write_sample<LAY>(o, out, ray, ri, ns, ts);
                    if (ns == 0) ts_arr[0] = ts;
                    if (ns == 1) ts_arr[1] = ts;
                    ++ns;
                }
                T -= alpha;
            }
            if (stop) break;
        }
        if (dropped && !(T < 1e-3f || ns >= o.S)) return true;
    } else if (dropped) {
        return true;
    }
    // ---- step 4: neighbours of the stored samples
    const int nstore = min(min(ns, 2), LAY == kLayDense ? o.S : out.s_max);
#pragma unroll 1
    for (int q = 0; q < nstore; ++q) {
        const float ts = q == 0 ? ts_arr[0] : ts_arr[1];
        const float s0 = ray.o[0] + ts * ray.d[0], s1 = ray.o[1] + ts * ray.d[1], s2 = ray.o[2] + ts * ray.d[2];
        NbBuf<MODE, KMAX> buf;
        buf.init();
        walk(false, [&](const Cand& x) {
            const float d2 = sqnorm3(s0 - x.p.x, s1 - x.p.y, s2 - x.p.z);
            const bool take = x.in && within(d2, x.lim) && !(MODE == EPCQ_MODE_KNN && x.dup);
            const float d = take ? sqrtf(d2) : 0.0f;
            const int id = __float_as_int(x.p.w);
            for (uint64_t m = __ballot(take); m; m &= m - 1ull) {
                const int y = __ffsll((unsigned long long)m) - 1;
                buf.add(lane_bcast(d, y), lane_bcast(id, y));
            }
        });
        row_wave_write<MODE, KMAX, LAY>(o, out, ray, buf, ri, q);
    }
    write_tail_wave<MODE, LAY>(o, out, ri, ns);
    return false;
}

// Samples and neighbours of the ray through pixel (u, v), whose output row is
// ri; every lane of the wave calls it with the same arguments.  For options
// under which at most two samples of a ray are stored.
template <int MODE, int KMAX, int LAY, bool PR>
__device__ __forceinline__ void run_ray_rows(const SampleOpts& o, const SampleOut& out, const ViewArgs& view,
                                             const RowList<PR>& src, const Ray& ray, int u, int v, int64_t ri,
                                             RowWaveSmem& sm) {
    const int W = view.W, H = view.H, k = o.k, ko = o.ko;
    const int lane = __lane_id();
    // ---- the window's segments.  Rows of 8 or 16 lanes, 8 or 4 at a time.
    const int sh = k <= 8 ? 3 : 4, per = kWave >> sh;
    const int c = lane & ((1 << sh) - 1);
    const int uu = u + c - (ko - 1);
    const bool inner = uu >= 0 && uu < W;
    const int first = max(0, (ko - 1) - u);  // column of the first pixel inside the image
    int nseg = 0;
    int64_t C = 0;
    bool split = false;   // every bucket is a segment
    bool capped = false;  // some bucket holds more than kSampleLaneHits points
    // two attempts at most: row segments, then (an irregular table) bucket segments
    for (int attempt = 0; attempt < 2; ++attempt) {
        nseg = 0;
        C = 0;
        bool again = false;
        for (int r0 = 0; r0 < k; r0 += per) {
            const int r = r0 + (lane >> sh);
            const bool active = r < k && c < k;
            const int vv = v + r + 1 - ko;
            const int vb = min(max(vv, 0), H - 1), ub = min(max(uu, 0), W - 1);
            int2 e = make_int2(-1, -1);
            if (active) e = view.hash[(int64_t)vb * W + ub];
            const bool full = e.y > 0;
            const bool mine = full && inner;
            // the row's run, and the start of the first bucket at or right of the column
            int lo = mine ? e.x : INT_MAX, hi = mine ? e.x + e.y : INT_MIN;
            int nxt = mine ? e.x : INT_MAX;
            for (int d = 1; d < (1 << sh); d <<= 1) {
                lo = min(lo, __shfl_xor(lo, d));
                hi = max(hi, __shfl_xor(hi, d));
                const int y = __shfl_down(nxt, d);
                if (c + d < (1 << sh)) nxt = min(nxt, y);
            }
            int right = __shfl_down(nxt, 1);
            if (c + 1 >= (1 << sh) || right == INT_MAX) right = hi;
            if (!split && __any(mine && e.x + e.y != right)) {
                again = true;
                break;
            }
            capped = capped || __any(full && e.y > kSampleLaneHits);
            if (active) sm.col[r][c] = nxt == INT_MAX ? hi : nxt;
            const bool main_run = !split && c == first && active && lo != INT_MAX;
            const bool head = split ? full : (main_run || (full && !inner));
            const int start = main_run ? lo : e.x;
            const int64_t len = !head ? 0 : main_run ? hi - lo : e.y;
            int64_t x = len;
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int64_t y = __shfl_up((long long)x, d);
                if (lane >= d) x += y;
            }
            const uint64_t hb = __ballot(head);
            if (head) {
                const int at = nseg + __popcll(hb & lanemask_lt());
                sm.pre[at] = C + x - len;
                sm.st[at] = (int)((uint32_t)start | (!inner || vv != vb ? 0x80000000u : 0u));
                sm.row[at] = (uint8_t)(main_run ? r : kOneBucket);
            }
            nseg += __popcll(hb);
            C += __shfl((long long)x, kWave - 1);
        }
        if (!again) break;
        split = true;
    }
    if (C == 0) {
        write_tail_wave<MODE, LAY>(o, out, ri, 0);
        return;
    }
    sm.hist[lane] = 0;
    sm.hist[lane + kWave] = 0;
    wave_lds_fence();

    // ---- the positions that pass the bound, four chunks in flight
    bool dropped = false;  // something beyond the list's depth was left out
    int64_t N = C;         // candidates of the walks
    RowWaveOver over = kOverAll;
    // the bounds of 4 chunks of segment positions [st + c0, st + len)
    auto bounds = [&](const RowFrame& f, const RowRay& rr, int st, int len, int c0, float4 (&cd)[4], bool (&pass)[4]) {
        const float r0 = __builtin_amdgcn_sqrtf(o.r2lim);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = c0 + q * kWave + lane;
            if (i >= len) continue;
            if (view.cand) {
                cd[q] = view.cand[st + i];
            } else {
                const float4 p = src.point(st + i);
                cd[q] = row_candidate(f, p, PR ? __builtin_amdgcn_sqrtf(src.limit(o, st + i, p)) : r0);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float da = cd[q].x - rr.a, db = cd[q].y - rr.b;
            pass[q] = c0 + q * kWave + lane < len && !(__builtin_fmaf(db, db, da * da) > cd[q].z * rr.g);
        }
    };
    auto segment_length = [&](int s) { return uniform((int)((s + 1 < nseg ? sm.pre[s + 1] : C) - sm.pre[s])); };
    bool many = false;  // too many for the list
    if (C > kWaveCache * kWave) {
        const RowFrame f = row_frame(view.c2w);
        const RowRay rr = row_ray(view.c2w, ray);
        const float depth = (float)(kWaveDepth + 1) * o.t_intvl;
        const float inf = __builtin_inff();
        float front = inf;  // ray depth of the first hit found so far
        int n = 0;
        bool cut = false;
        for (int s = 0; s < nseg; ++s) {
            const int st = uniform(sm.st[s]) & 0x7fffffff, len = segment_length(s);
            for (int c0 = 0; c0 < len; c0 += 4 * kWave) {
                float4 cd[4];
                bool pass[4];
                bounds(f, rr, st, len, c0, cd, pass);
                if (cut) {
                    // hits ahead of the front move it (first where none is known)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const bool ahead = pass[q] && !(cd[q].w > front);
                        if (!__any(ahead)) continue;
                        float t = inf;
                        if (ahead) {
                            const int j = st + c0 + q * kWave + lane;
                            const float4 p = src.point(j);
                            float e2;
                            ray_t_e2(ray, p, t, e2);
                            if (!within(e2, src.limit(o, j, p))) t = inf;
                        }
                        front = fminf(front, wave_min(t));
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool near = pass[q] && !(cut && cd[q].w > front + depth);
                    dropped = dropped || __any(pass[q] && !near);
                    const uint64_t pb = __ballot(near);
                    const int at = n + __popcll(pb & lanemask_lt());
                    if (near && at < kWaveList) {
                        sm.pos[at] = st + c0 + q * kWave + lane;
                        sm.seg[at] = (uint8_t)s;
                    }
                    n += __popcll(pb);
                }
                if (n > kWaveList) break;
            }
            if (n > kWaveList) {
                if (cut || capped || !(o.t_intvl > 0.0f)) break;
                cut = true;  // again from the first segment on
                n = 0;
                s = -1;
            }
        }
        many = n > kWaveList;
        if (!many) {
            over = kOverList;
            N = n;
        }
        wave_lds_fence();
    }
    // (in the feature layout a ray of too many walks all of its candidates: a
    // second instance of the sums cost all rays 2 % there, in scalar spills)
    constexpr bool kChunks = LAY != kLayFeat;
    if (!many || !kChunks) {
        dropped = dropped && !many;
        while (row_wave_walks<MODE, KMAX, LAY, PR, false>(o, out, src, ray, ri, sm, nseg, C, N, over, dropped, capped)) {
            // the walk has to go on beyond the list's depth
            many = true;
            dropped = false;
            over = kOverAll;
            N = C;
            sm.hist[lane] = 0;
            sm.hist[lane + kWave] = 0;
            wave_lds_fence();
            if (kChunks) break;
        }
        if (!many || !kChunks) return;
    }
    if constexpr (kChunks) {
        // ---- the chunks that hold a position within the bound, at any depth
        const RowFrame f = row_frame(view.c2w);
        const RowRay rr = row_ray(view.c2w, ray);
        int n = 0;
        for (int s = 0; s < nseg && n <= kWaveList; ++s) {
            const int st = uniform(sm.st[s]) & 0x7fffffff, len = segment_length(s);
            for (int c0 = 0; c0 < len && n <= kWaveList; c0 += 4 * kWave) {
                float4 cd[4];
                bool pass[4];
                bounds(f, rr, st, len, c0, cd, pass);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (!__any(pass[q])) continue;
                    if (n < kWaveList && lane == 0) {
                        sm.pos[n] = st + c0 + q * kWave;
                        sm.seg[n] = (uint8_t)s;
                    }
                    ++n;
                }
            }
        }
        const bool chunks = n <= kWaveList;
        wave_lds_fence();
        row_wave_walks<MODE, KMAX, LAY, PR, true>(o, out, src, ray, ri, sm, nseg, C, chunks ? (int64_t)n * kWave : C,
                                                  chunks ? kOverChunks : kOverAll, false, capped);
    }
}

}  // namespace epcq
