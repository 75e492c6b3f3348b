// Primary-surface search, K-nearest sampling and radius query for gfx950.
//
//   epcq_quick_sampling  dense drop-in layout of quick_sampling
//                        (epcq/csrc/epcq_render_topk.cu:10-220,341-417)
//   epcq_knn_sampling    compact layout, optional per-point radius, KNN
//                        neighbours with ray depth / distance, fused IDW
//   epcq_quick_query     radius query for a ray list (:222-339)
//   epcq_idw_features    IDW weights + weighted features (epcq/epcq.py:434-452)
//
// Sampling has three forms with the same outputs (takes_rows, takes_rows_list):
// tiles over the rows of the point list (epcq_rows.h), one wave per ray over
// these rows (epcq_rows_wave.h), and the lane sets.
//
// A lane-set image runs one 256-lane block per tile of rays.  The block first
// stages its tile's halo region -- the hash entries and bucket cones of the
// (tw + k - 1) x (th + k - 1) neighbour pixels and, row segment by row segment
// (contiguous in the row-major point lists), the coordinates and indices of
// their points as float4 -- into LDS with coalesced loads; every candidate walk
// of every ray then reads LDS.  A tile whose region holds more points than the
// LDS capacity, or a row that is no run of the list, reads global memory
// instead, in the same block.  Ray lists (no tile structure) read global
// memory, one wave or one lane per ray.  The per-ray logic of the lane sets is
// in epcq_sampler.h.
#include <cmath>
#include <mutex>

#include "epcq_common.h"
#include "epcq_rows.h"
#include "epcq_sampler.h"

namespace epcq {
// Defined in epcq_sample_kernels.h, instantiated in epcq_sample_inst_*.hip
// (NW = 1) and epcq_sample_wide_*.hip (NW = 4).
template <int MODE, int KMAX, int SMAX, int NW>
void launch_lay(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, const int* rays, int64_t R,
                const TilePlan& tp, hipStream_t st);
}  // namespace epcq

extern "C" int32_t epcq_max_live_samples(const epcq_options* opt, float r_max);

namespace epcq {

float squared_threshold(float r) {
    if (!(r > 0.0f)) return 0.0f;  // no distance is below r (NaN r included)
    if (std::isinf(r)) return INFINITY;
    float s = r * r;
    if (std::sqrt(s) >= r) {
        while (s > 0.0f && std::sqrt(std::nextafter(s, 0.0f)) >= r) s = std::nextafter(s, 0.0f);
    } else {
        while (!(std::sqrt(s) >= r)) s = std::nextafter(s, INFINITY);
    }
    return s;
}

TilePlan plan_tiles(int k, int tile_w, int tile_h, int cap, int flags, bool point_radius) {
    TilePlan p{};
    p.tw = tile_w;
    p.th = tile_h;
    p.xcd = (flags & EPCQ_TUNE_XCD_ORDER) != 0;
    p.rw_max = p.tw + k - 1;
    p.rh_max = p.th + k - 1;
    // per point: float4 + radius; per region pixel: cone_a, hash, cone_b; per row: lo, base
    const size_t fixed =
        align_up((size_t)p.rw_max * p.rh_max * (16 + 8 + 8) + (size_t)(2 * p.rh_max + 1) * 4, 16);
    // 64 KB: a larger stage leaves one block per CU, slower on every workload measured
    const size_t limit = 64 * 1024;
    size_t c = (size_t)std::max(cap, 0);
    const size_t per = point_radius ? 20 : 16;
    if (fixed + c * per > limit) c = fixed < limit ? (limit - fixed) / per : 0;
    p.cap = (int)c;
    p.lds_bytes = c * per + fixed;
    return p;
}

int check_tuning(const epcq_tuning& t, const char* who) {
    const std::string w(who);
    const int rays = t.tile_w * t.tile_h;
    if (t.tile_w < 1 || t.tile_w > 64 || (t.tile_w & (t.tile_w - 1)) || t.tile_h < 1 ||
        (rays != 64 && rays != 128 && rays != 256))
        return fail(EPCQ_ERR_INVALID, w + ": tile_w must be a power of two <= 64 and tile_w * tile_h 64, 128 or 256");
    if (t.tile_cap < 0) return fail(EPCQ_ERR_INVALID, w + ": negative tile_cap");
    if (t.heavy < 0) return fail(EPCQ_ERR_INVALID, w + ": negative heavy");
    if (t.list_wave < 0) return fail(EPCQ_ERR_INVALID, w + ": negative list_wave");
    if (t.flags & ~EPCQ_TUNE_XCD_ORDER) return fail(EPCQ_ERR_INVALID, w + ": unknown flags");
    return EPCQ_OK;
}

namespace {

constexpr int kBlock = 256;

std::mutex g_tuning_mu;
epcq_tuning g_tuning{32, 8, 1024, 0, kHeavyCandidates, kListWaveRays};

epcq_tuning current_tuning() {
    std::lock_guard<std::mutex> lk(g_tuning_mu);
    return g_tuning;
}

// Pixel-ordered copy of the points, one thread per list position: (x, y,
// z, index bits) and, with per-point radii, the radius's squared threshold.
// Positions holding no valid index (the -1 tail) are left alone; the hash
// entries never point there.  For the row-run sampler also cand, the points'
// candidate bounds (of the uniform radius r0 without prad), and queue, its
// deferred rays, emptied here.
__global__ __launch_bounds__(kBlock) void point_copy_kernel(const int* __restrict__ sorted_idx,
                                                            const float* __restrict__ xyz,
                                                            const float* __restrict__ radius, int64_t n,
                                                            float4* __restrict__ pts, float* __restrict__ prad,
                                                            float4* __restrict__ cand, float r0,
                                                            const float* __restrict__ c2w,
                                                            RowQueue* __restrict__ queue) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i == 0 && queue) queue->count = 0;
    if (i >= n) return;
    const int id = sorted_idx[i];
    if (id < 0 || id >= n) return;
    const float* q = xyz + 3 * (int64_t)id;
    const float4 p = make_float4(q[0], q[1], q[2], __int_as_float(id));
    pts[i] = p;
    float lim = 0.0f;
    if (prad) prad[i] = lim = point_threshold(radius[id]);
    if (cand) cand[i] = row_candidate(row_frame(c2w), p, prad ? __builtin_amdgcn_sqrtf(lim) : r0);
}

// Bucket cones, one thread per pixel: from the pixel-ordered copy pts_in
// when given, else gathering through sorted_idx / xyz (and then writing the
// copy into pts, when not null).
__global__ __launch_bounds__(kBlock) void bucket_cone_kernel(const int2* __restrict__ hash,
                                                             const int* __restrict__ sorted_idx,
                                                             const float* __restrict__ xyz,
                                                             const float4* __restrict__ pts_in,
                                                             const float* __restrict__ radius, float r0,
                                                             const float* __restrict__ c2w, int64_t P,
                                                             float4* __restrict__ cone_a, float2* __restrict__ cone_b,
                                                             float4* __restrict__ pts, float* __restrict__ prad) {
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p < P) bucket_cone_body(hash, sorted_idx, xyz, pts_in, radius, r0, c2w, p, cone_a, cone_b, pts, prad);
}

// Buckets of more points than this are taken one at a time, so that a group's
// candidates are always counted in 31 bits.
constexpr int kQueryBucket = 1 << 24;

// Rays from which on windows of at most 32 buckets take half a wave per ray:
// twice the rays per instruction, but with fewer rays whole waves fill the GPU
// better (2513 rays of 1.4M points, 23 us, take one wave each).
constexpr int64_t kQueryHalfWave = 16384;

// Fewer lanes per ray where a ray has few outputs, so that what is left is its
// buckets: with at most kQueryFew hits wanted, four lanes for windows of up to two
// columns and eight for three, and from kQueryMany rays on, which fill the GPU by
// themselves, four for up to three and eight for up to nine.  One lane per ray / 4 / 8 / 32, in ms with the
// call's 0.02: 571k rays, k = 1, 2 hits wanted 0.025 / 0.025 / 0.039 / 0.137; 334k, k
// = 3, 1 hit 0.024 / 0.026 / 0.031 / 0.081; 147k, k = 4, 4 hits 0.34 / 0.12 / 0.084 /
// 0.070; but 242k, k = 5, 256 hits 0.65 / 0.30 / 0.26 / 0.22.  Over 700 calls 1.06 of
// the best of these in the geometric mean, 1.15 without this rule.
constexpr int kQueryFew = 32;
constexpr int64_t kQueryMany = 131072;

// hashtable_query_for_nearby_point (:222-283): hits of each neighbour bucket
// (at most 32) appended in lane order.  G lanes take a ray, 32 or 64 of them or
// fewer (below): each reads the hash
// entry of one bucket, a prefix sum numbers the candidates of G buckets, and
// the lanes take G candidates at a time, whichever bucket they are in; a ballot
// gives each hit its place in the output, so that reads of the list and writes
// are consecutive.  With one lane per ray every candidate was a wait for
// memory.  What bounds it now: instruction issue (about 250 per ray of 25
// buckets) and the R * cap outputs.  Measured, one lane per ray against groups:
// all 120k rays of 200k points at 400 x 300, cap 256 0.253 -> 0.050 ms; 1024
// rays of 1M points at 200 x 160 1.97 -> 0.04; 480k rays of 2M points at 800 x
// 600 1.33 -> 0.82; 500k rays of a nearly empty image 0.206 -> 0.122.
template <int G>
__global__ __launch_bounds__(kBlock) void query_kernel(const float* __restrict__ xyz,
                                                       const int* __restrict__ sorted_idx,
                                                       const int2* __restrict__ hash,
                                                       const float* __restrict__ c2w, float fx, float fy,
                                                       float cx, float cy, int W, int H, int k, int ko,
                                                       float r0, const int* __restrict__ rays, int64_t R,
                                                       int cap, int* __restrict__ out) {
    const int64_t ri = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / G;
    if (ri >= R) return;  // whole groups
    const int lane = threadIdx.x % G;
    const int shift = threadIdx.x % kWave / G * G;  // the group's first lane in the wave
    const uint64_t group = ~0ull >> (kWave - G);
    const uint64_t below = (1ull << lane) - 1;  // of the group's ballots
    int* row = out + ri * cap;
    int total = 0;
    const int64_t q = rays[ri];
    if (q >= 0 && q < (int64_t)W * H) {
        const int u = (int)(q % W), v = (int)(q / W);
        float m[12];
#pragma unroll
        for (int i = 0; i < 12; ++i) m[i] = c2w[i];
        Ray ray;
        make_ray(m, fx, fy, cx, cy, u, v, ray);
        const int L = k * k;
        for (int l0 = 0; l0 < L && total < cap;) {
            int2 e = make_int2(0, 0);
            if (l0 + lane < L) e = hash[neighbor_pixel(k, ko, l0 + lane, u, v, W, H)];
            int n = max(e.y, 0);
            int step = G;
            if ((__ballot(n > kQueryBucket) >> shift & group) != 0) {
                step = 1;
                if (lane != 0) n = 0;
            }
            int end = n;  // candidates of the buckets up to the lane's
#pragma unroll
            for (int d = 1; d < G; d *= 2) {
                const int t = __shfl_up(end, d, G);
                if (lane >= d) end += t;
            }
            const int first = e.x - (end - n);  // list position of candidate c: first + c
            const int C = __shfl(end, G - 1, G);
            const bool capped = (__ballot(n > kQueryLaneHits) >> shift & group) != 0;
            int carry = 0;  // hits so far of a bucket that began before c0
            for (int c0 = 0; c0 < C && total < cap;) {
                const int c = c0 + lane;
                int b = 0;  // the candidate's bucket: the first that ends after it
#pragma unroll
                for (int d = G / 2; d > 0; d /= 2)
                    if (__shfl(end, b + d - 1, G) <= c) b += d;
                const int j = __shfl(first, b, G) + c;
                bool hit = false;
                int id = 0;
                if (c < C) {
                    id = sorted_idx[j];
                    const float* p = xyz + 3 * (int64_t)id;
                    float t, dist;
                    point_ray(ray, p[0], p[1], p[2], t, dist);
                    hit = dist < r0;
                }
                uint64_t mask = __ballot(hit) >> shift & group;
                int next = c0 + G;
                if (capped) {
                    const int start = __shfl(end - n, b, G);
                    const int s0 = max(start - c0, 0);  // the bucket's first lane
                    const int before = __popcll(mask & below & (~0ull << s0)) + (start < c0 ? carry : 0);
                    carry = __shfl(before + (hit ? 1 : 0), G - 1, G);
                    // the rest of a bucket that is full
                    const int stop = __shfl(end, __shfl(b, G - 1, G), G);
                    if (carry >= kQueryLaneHits) next = max(next, stop);
                    hit = hit && before < kQueryLaneHits;
                    mask = __ballot(hit) >> shift & group;
                }
                const int at = total + __popcll(mask & below);
                if (hit && at < cap) row[at] = id;
                total += __popcll(mask);
                c0 = next;
            }
            l0 += step;
        }
    }
    for (int j = total + lane; j < cap; j += G) row[j] = -1;
}

__global__ __launch_bounds__(kBlock) void idw_kernel(const float* __restrict__ xyz, const void* feat,
                                                     int feat_bf16, int F, const float* __restrict__ sp_xyz,
                                                     const int* __restrict__ nb_idx, int64_t M, int K,
                                                     float* __restrict__ w, float* __restrict__ agg) {
    const int64_t m = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (m >= M) return;
    const float s0 = sp_xyz[3 * m], s1 = sp_xyz[3 * m + 1], s2 = sp_xyz[3 * m + 2];
    const int* ids = nb_idx + m * K;
    float* wo = w + m * K;
    float den = 0.0f;
    for (int j = 0; j < K; ++j) {
        const int id = ids[j];
        float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f;
        if (id >= 0) {
            p0 = xyz[3 * (int64_t)id];
            p1 = xyz[3 * (int64_t)id + 1];
            p2 = xyz[3 * (int64_t)id + 2];
        }
        const float d = norm3(p0 - s0, p1 - s1, p2 - s2);
        const float inv = (1.0f / (d + 1e-6f)) * (id >= 0 ? 1.0f : 0.0f);
        wo[j] = inv;
        den = den + inv;
    }
    den = den + 1e-6f;
    for (int j = 0; j < K; ++j) wo[j] = wo[j] / den;
    float* ao = agg + m * (int64_t)F;
    for (int f = 0; f < F; ++f) {
        float acc = 0.0f;
        for (int j = 0; j < K; ++j) {
            const int id = ids[j];
            if (id < 0) continue;
            float fv;
            if (feat_bf16) {
                fv = __uint_as_float((uint32_t)static_cast<const uint16_t*>(feat)[(int64_t)id * F + f] << 16);
            } else {
                fv = static_cast<const float*>(feat)[(int64_t)id * F + f];
            }
            acc = acc + wo[j] * fv;
        }
        ao[f] = acc;
    }
}

int check_common(const epcq_camera* cam, const epcq_options* opt, const char* who) {
    if (!cam || !opt) return fail(EPCQ_ERR_INVALID, std::string(who) + ": null camera or options");
    if (cam->width <= 0 || cam->height <= 0)
        return fail(EPCQ_ERR_INVALID, std::string(who) + ": image size must be positive");
    if ((int64_t)cam->width * cam->height >= (int64_t(1) << 30))
        return fail(EPCQ_ERR_INVALID, std::string(who) + ": image too large");
    if (opt->kernel_size < 1) return fail(EPCQ_ERR_INVALID, std::string(who) + ": kernel_size must be >= 1");
    if (opt->kernel_size > 64) return fail(EPCQ_ERR_INVALID, std::string(who) + ": kernel_size must be <= 64");
    if (!cam->c2w) return fail(EPCQ_ERR_INVALID, std::string(who) + ": null c2w");
    return EPCQ_OK;
}

SampleOpts make_opts(const float* xyz, const epcq_options* opt, const float* radius) {
    SampleOpts o{};
    o.k = opt->kernel_size;
    o.ko = (opt->kernel_size + 1) / 2;
    o.kdiv = (65536 + opt->kernel_size - 1) / opt->kernel_size;
    o.L = opt->kernel_size * opt->kernel_size;
    o.r0 = opt->radius_threshold;
    o.r2lim = squared_threshold(opt->radius_threshold);
    o.radius = radius;
    o.t_intvl = opt->t_intvl;
    o.alpha_p = opt->sdf2weight_gaussian_alpha;
    o.gamma = opt->sdf2weight_gaussian_gamma;
    o.S = opt->num_sample_points_per_ray;
    o.Kc = opt->num_point_cloud_per_sp;
    o.xyz = xyz;
    const epcq_tuning tu = current_tuning();
    o.heavy = tu.heavy;
    o.list_wave = tu.list_wave;
    return o;
}

size_t sampling_bytes(int64_t n, int64_t P);

// Which form an image takes, by its pixels P, its points n and the points d that
// a ray's window holds on average.  The lines lie where the medians of 1,900
// images (cameras, scenes, radii and buffers varied; call with the build, which
// all forms share) cross: 0.68 of the lane sets' time in the geometric mean.  One
// image in 25 is more than 3 % slower than these, single ones up to 1.6 times,
// since how the points cluster is not known here.  Tile form / wave form /
// lane sets in ms:
// - P <= kWaveTiny: 64 rays per wave would leave SIMDs idle; waves.  260 x 147,
//   k = 5, d = 156: 0.46 / 0.17 / 0.66; 203 x 152, k = 11, d = 202: 0.36 / 0.19 /
//   0.29.
// - windows of up to eight columns, P <= kWaveImage: waves from kWaveFew points
//   on, below these the tiles, whose cost is the candidates rather than the rays:
//   400 x 300, d = 2: 0.09 / 0.18 / 0.09 in a box, 0.10 / 0.18 / 0.13 on a sphere,
//   d = 52: 0.51 / 0.27 / 0.67.  Rows of more than kWaveBuffer neighbours, whose
//   buffers take the wave form 213 registers, from kWaveMid on: 386 x 292, k = 7,
//   K = 32, d = 59: 0.34 / 0.92 / 0.47.
// - up to four times as many: each tile is a long serial walk, and the longest
//   ones end last.  Waves from kWaveDense points on (half the pixels: from
//   kWaveMid): a sphere at 500 x 503, k = 7: d = 195 1.15 / 0.71 / 1.03, d =
//   292 1.53 / 0.81 / 1.47; a box at 640 x 480, k = 7: d = 160 0.64 / 0.97 /
//   0.92, d = 319 1.15 / 1.26 / 1.62; d = 4400 10.6 / 6.2 / 8.0.  Not with more than
//   kWaveBuffer neighbours: 621 x 350, k = 7, K = 32, d = 138: waves 2.7, lane sets
//   1.7, and tiles 0.7 of these in the median.
// - wider windows, two blocks of whose tiles fit on a CU, cost more in both
//   forms.  Waves from kWaveFull points per pixel on, up to twice kWaveImage (345
//   x 261, k = 9, d = 3240: 3.8 / 1.0 / 4.6), and from kWaveFullest on up to four
//   times (685 x 683, k = 9, d = 279: 1.13 / 1.63 / 1.00); of twice these with more
//   than kWaveBuffer neighbours.  Below that the lane
//   sets, up to twice kWaveImage (400 x 340, k = 9, d = 35: 0.25 / 0.33 / 0.19;
//   500 x 503, k = 13, d = 90: 0.56 / 0.75 / 0.45), and from kWaveMid points on
//   up to four times (k = 11 at 640 x 480, d = 364 1.34 / 1.40 / 1.19), from 13
//   columns on eight times, there below kWaveWide (k = 15 at 800 x 800, d = 351
//   1.67 / - / 1.52).  The other images take the tiles: medians of 0.76 of the lane
//   sets' time at two to four times kWaveImage, 0.65 at four to eight, 0.4 above.
constexpr int64_t kWaveTiny = 40000;
constexpr int64_t kWaveImage = 131072;
constexpr int64_t kWaveFew = 25;
constexpr int64_t kWaveMid = 100;
constexpr int64_t kWaveDense = 256;
constexpr int64_t kWaveWide = 400;
constexpr int64_t kWaveFull = 3, kWaveFullest = 5;
constexpr int kWaveBuffer = 16;

// Where a window holds few points on average, a ray has next to nothing to test,
// and the rows' bounds and the fills are what is left: there the lane sets stay
// ahead.  Fewer than ten in the dense layout; measured, rows against lane sets, 800
// x 800 pixels, k = 5: 0.19 against 0.16 ms with 100k points, 0.24 against 0.21
// with 200k, 0.27 against 0.26 with 300k, 0.33 against 0.39 with 600k.  Fewer than
// five in the compact layout: 963 x 964, k = 5, d = 4: 0.38 against 0.32, 1635 x
// 1636, k = 3, d = 1: 0.48 against 0.36; the medians of 110 images are even below
// five and at 0.89 from there on.  Fewer than 15 with six to eight columns: 1423 x
// 1426, k = 7, d = 7: 1.06 against 0.66, 781 x 585, d = 11: 0.62 against 0.54; even in
// the median of 32 images, 0.8 from there on.
constexpr int64_t kRowsSparse = 10, kRowsSparseCompact = 5, kRowsSparseWide = 15;

// The tiles add the points of a region's rows in 31 bits, and a caller's table may
// let rows share their buckets, so that each holds up to n points.  Larger clouds
// (113 million points at k = 16, 268 million at k = 5) take the waves, which count
// in 63: a test in the tiles cost 20M points at 1920 x 1080 0.6 %.
int64_t rows_most(int k) { return INT32_MAX / (kRowTileH + k - 1); }

// Whether a full image takes the row-run sampler (epcq_rows.h): windows that
// its LDS rows hold, options under which a ray can visit two slots at most
// (with per-point radii the caller's s_max stands for that bound; a ray that
// visits more is run by a whole wave), and a workspace for the point copy and
// the queue of deferred rays.
int takes_rows(SampleOpts& o, int64_t P, int64_t n, int live_bound, bool compact, const void* workspace,
               size_t workspace_bytes) {
    if (o.k > kRowMaxK || live_bound > 2 || !workspace || workspace_bytes < sampling_bytes(n, P)) return kRowsNone;
    const int64_t d = (int64_t)o.L * n / std::max<int64_t>(P, 1);
    // candidates that the launch gives a lane of each SIMD: a ray with far more
    // would outlast the others
    o.row_heavy = (int)std::min<int64_t>(kRowHeavyMost, std::max<int64_t>(kRowHeavyLeast, (int64_t)o.L * n / (65536 * 128)));
    const bool wide = o.k > 8, large = o.Kc > kWaveBuffer;
    if (P <= kWaveTiny || n > rows_most(o.k)) return kRowsWave;
    if (wide) {
        const int64_t full = (P <= 2 * kWaveImage ? kWaveFull : kWaveFullest) * (large ? 2 : 1);
        if (P <= 4 * kWaveImage && n >= full * P) return kRowsWave;
        if (P <= 2 * kWaveImage) return kRowsNone;
    } else if (P <= kWaveImage && d >= (large ? kWaveMid : kWaveFew)) {
        return kRowsWave;
    }
    if (d < (compact ? kRowsSparseCompact : kRowsSparse) || (o.k > 5 && !wide && d < kRowsSparseWide)) return kRowsNone;
    if (wide) {
        if (P <= 4 * kWaveImage) return d >= kWaveMid ? kRowsNone : kRowsTiles;
        return o.k > 12 && P <= 8 * kWaveImage && d >= kWaveMid && d < kWaveWide ? kRowsNone : kRowsTiles;
    }
    if (!large && P > kWaveImage && P <= 4 * kWaveImage && d >= (P <= 2 * kWaveImage ? kWaveMid : kWaveDense))
        return kRowsWave;
    return kRowsTiles;
}

ViewArgs make_view(const epcq_camera* cam, const int* sorted_idx, const int* hash) {
    return ViewArgs{cam->c2w, cam->fx, cam->fy, cam->cx, cam->cy, cam->width, cam->height,
                    reinterpret_cast<const int2*>(hash), sorted_idx, nullptr, nullptr, nullptr, nullptr, nullptr,
                    nullptr};
}

// Workspace layout of the samplers: cone_a [P] float4 | cone_b [P] float2 |
// pixel-ordered points [n] float4 | pixel-ordered radii [n] float | candidate
// bounds [n + kRowPad] float4.
size_t cone_bytes(int64_t P) { return align_up((size_t)P * 16, 256) + align_up((size_t)P * 8, 256); }

size_t sampling_bytes(int64_t n, int64_t P) {
    return cone_bytes(P) + align_up((size_t)n * 16, 256) + align_up((size_t)n * 4, 256) + (size_t)(n + kRowPad) * 16;
}

// Bucket cones and the pixel-ordered point copy in the workspace (when it is
// large enough: then o.cull is set and view reads them).  They cost a pass
// over every pixel and point of the view, so a ray list (rays >= 0 rays)
// whose windows visit fewer than P / kConeVisitRatio buckets in all skips
// them.  Measured: a 4096-ray batch of a 1M-point 800x800 view with k = 5
// (visits 0.16 P) samples in 0.069 ms without them against 0.080 ms with,
// and both ways meet near 0.24 P; on a 20M-point 1080p view with k = 15 they
// meet near 0.2 P.  The outputs are the same either way.
constexpr int64_t kConeVisitRatio = 4;

// Whether a ray list takes the one-wave-per-ray form over row runs
// (epcq_rows_wave.h): under the same bounds as an image, lists of at most
// list_wave rays.  But one wave per ray over the lane sets (run_ray_wave) is ahead
// where the buckets that it skips outweigh the cones' pass: where the windows visit
// kListVisits buckets per pixel or more in all, and with more than 12 columns on
// views of up to twice kWaveImage.  Rows against lane sets, medians of 2,500 lists:
// 0.75 where the windows visit one to four buckets per pixel, 0.89 at eight to 16,
// 0.98 at 16 to 32, 1.3 to 1.9 beyond; with more than 12 columns 1.1 to 1.2 on the
// smaller views.  216 x 163, k = 11, 35,208 rays 0.27 / 0.14 ms; 202 x 204, k = 15,
// 4520 rays 0.12 / 0.06; 800 x 800, k = 5, 4096 rays 0.024 / 0.057.
constexpr int64_t kListVisits = 16;

int takes_rows_list(const SampleOpts& o, int64_t R, int64_t P, int live_bound, const void* workspace,
                    size_t workspace_bytes) {
    if (o.k > kRowMaxK || live_bound > 2 || R > o.list_wave) return kRowsNone;
    const bool cones = workspace && workspace_bytes >= cone_bytes(P) && R * o.L * kConeVisitRatio >= P;
    if (cones && (R * o.L >= kListVisits * P || (o.k > 12 && P <= 2 * kWaveImage))) return kRowsNone;
    return kRowsWave;
}

void prepare_bounds(SampleOpts& o, ViewArgs& view, int64_t n, const epcq_camera* cam, const int* sorted_idx,
                    const int* hash, void* workspace, size_t workspace_bytes, int64_t rays, hipStream_t st) {
    const int64_t P = (int64_t)cam->width * cam->height;
    o.cull = 0;
    if (!workspace || workspace_bytes < cone_bytes(P)) return;
    if (rays >= 0 && rays * o.L * kConeVisitRatio < P) return;
    if (o.rows) {
        // the row-run sampler: point copy and candidate bounds, and the queue
        // in the cones' place (only an image's tiles use it; a ray list whose
        // workspace has no room for the bounds works them out on the way)
        const size_t pts_off = cone_bytes(P), rad_off = pts_off + align_up((size_t)n * 16, 256);
        const size_t cand_off = rad_off + align_up((size_t)n * 4, 256);
        if (workspace_bytes < rad_off) return;
        char* w = static_cast<char*>(workspace);
        float4* pts = reinterpret_cast<float4*>(w + pts_off);
        float* prad = o.radius && workspace_bytes >= rad_off + (size_t)n * 4 ? reinterpret_cast<float*>(w + rad_off)
                                                                            : nullptr;
        float4* cand = workspace_bytes >= sampling_bytes(n, P) ? reinterpret_cast<float4*>(w + cand_off) : nullptr;
        RowQueue* queue = reinterpret_cast<RowQueue*>(w);
        point_copy_kernel<<<dim3((unsigned)ceil_div(std::max<int64_t>(n, 1), kBlock)), dim3(kBlock), 0, st>>>(
            sorted_idx, o.xyz, o.radius, n, pts, prad, cand, std::sqrt(o.r2lim), cam->c2w, queue);
        view.cone_a = reinterpret_cast<const float4*>(queue);
        view.pts = pts;
        view.prad = prad;
        view.cand = cand;
        return;
    }
    char* w = static_cast<char*>(workspace);
    float4* ca = reinterpret_cast<float4*>(w);
    float2* cb = reinterpret_cast<float2*>(w + align_up((size_t)P * 16, 256));
    const size_t pts_off = cone_bytes(P), rad_off = pts_off + align_up((size_t)n * 16, 256);
    float4* pts = workspace_bytes >= rad_off ? reinterpret_cast<float4*>(w + pts_off) : nullptr;
    float* prad = o.radius && workspace_bytes >= rad_off + (size_t)n * 4 ? reinterpret_cast<float*>(w + rad_off)
                                                                        : nullptr;
    if (pts) {
        // the copy first, in parallel over list positions, then the cones from it
        if (n > 0)
            point_copy_kernel<<<dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, st>>>(sorted_idx, o.xyz,
                                                                                          o.radius, n, pts, prad,
                                                                                          nullptr, 0.0f, nullptr, nullptr);
        bucket_cone_kernel<<<dim3((unsigned)ceil_div(P, kBlock)), dim3(kBlock), 0, st>>>(
            reinterpret_cast<const int2*>(hash), nullptr, nullptr, pts, o.radius, o.r0, cam->c2w, P, ca, cb, nullptr,
            nullptr);
    } else {
        bucket_cone_kernel<<<dim3((unsigned)ceil_div(P, kBlock)), dim3(kBlock), 0, st>>>(
            reinterpret_cast<const int2*>(hash), sorted_idx, o.xyz, nullptr, o.radius, o.r0, cam->c2w, P, ca, cb,
            nullptr, nullptr);
    }
    o.cull = 1;
    view.cone_a = ca;
    view.cone_b = cb;
    view.pts = pts;
    view.prad = prad;
}

// Windows of more than 64 lanes (k > 8) take the kernels with 4-word lane
// sets (exact culling up to k = 16; larger windows visit every lane).  The
// row-run sampler has one form for all of them.
template <int MODE, int KMAX>
void launch_smax(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, const int* rays, int64_t R,
                 const TilePlan& tp, int bound, hipStream_t st) {
    const bool wide = o.L > 64 && !o.rows;
    if (bound <= 2 || o.rows) {
        if (wide) launch_lay<MODE, KMAX, 2, 4>(o, out, view, rays, R, tp, st);
        else launch_lay<MODE, KMAX, 2, 1>(o, out, view, rays, R, tp, st);
    } else {
        if (wide) launch_lay<MODE, KMAX, kRegSamples, 4>(o, out, view, rays, R, tp, st);
        else launch_lay<MODE, KMAX, kRegSamples, 1>(o, out, view, rays, R, tp, st);
    }
}

// Feature sums of the compact rows after the row-run sampler.
void launch_idw_rows(const SampleOpts& o, const SampleOut& out, int64_t R, hipStream_t st) {
    const int64_t rows = R * out.s_max;
    int G = 1;  // lanes per row: a power of two, at most 32, about one per four features
    while (G < 32 && 4 * G < o.F) G *= 2;
    const dim3 grid((unsigned)ceil_div(rows, 256 / G)), block(256);
    if (o.feat_bf16 && o.feat_vec)
        idw_rows_kernel<true, true><<<grid, block, 0, st>>>(o.feat, o.F, G, rows, o.Kc, out.nb_idx, out.w, out.agg);
    else if (o.feat_bf16)
        idw_rows_kernel<true, false><<<grid, block, 0, st>>>(o.feat, o.F, G, rows, o.Kc, out.nb_idx, out.w, out.agg);
    else if (o.feat_vec)
        idw_rows_kernel<false, true><<<grid, block, 0, st>>>(o.feat, o.F, G, rows, o.Kc, out.nb_idx, out.w, out.agg);
    else
        idw_rows_kernel<false, false><<<grid, block, 0, st>>>(o.feat, o.F, G, rows, o.Kc, out.nb_idx, out.w, out.agg);
}

// `bound`: samples of one ray that are stored (kernels with a bound of 2 keep
// two sample depths in registers; the others keep kRegSamples and re-read
// later ones from the outputs).
int launch_sample(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, const int* rays, int64_t R,
                  int mode, int bound, hipStream_t st, const char* who) {
    if (R == 0) return EPCQ_OK;
    const epcq_tuning tu = current_tuning();
    const TilePlan tp = plan_tiles(o.k, tu.tile_w, tu.tile_h, tu.tile_cap, tu.flags, o.radius != nullptr);
    if (mode == EPCQ_MODE_COMPAT) {
        launch_smax<EPCQ_MODE_COMPAT, kCompatBuffer>(o, out, view, rays, R, tp, bound, st);
    } else if (o.Kc <= 8) {
        launch_smax<EPCQ_MODE_KNN, 8>(o, out, view, rays, R, tp, bound, st);
    } else if (o.Kc <= 16) {
        launch_smax<EPCQ_MODE_KNN, 16>(o, out, view, rays, R, tp, bound, st);
    } else {
        launch_smax<EPCQ_MODE_KNN, 32>(o, out, view, rays, R, tp, bound, st);
    }
    if (o.feat && o.rows == kRowsTiles) launch_idw_rows(o, out, R, st);  // the wave form sums the features itself
    return check_launch(who);
}

}  // namespace
}  // namespace epcq

using namespace epcq;

extern "C" int epcq_set_tuning(const epcq_tuning* t) {
    if (!t) return fail(EPCQ_ERR_INVALID, "set_tuning: null");
    if (int e = check_tuning(*t, "set_tuning")) return e;
    std::lock_guard<std::mutex> lk(g_tuning_mu);
    g_tuning = *t;
    return EPCQ_OK;
}

extern "C" int epcq_get_tuning(epcq_tuning* t) {
    if (!t) return fail(EPCQ_ERR_INVALID, "get_tuning: null");
    *t = current_tuning();
    return EPCQ_OK;
}

extern "C" float epcq_squared_threshold(float r) { return squared_threshold(r); }

extern "C" int32_t epcq_max_live_samples(const epcq_options* opt, float r_max) {
    // Every visited slot (count >= 2) lowers the transmittance by
    // alpha = gamma * exp(-mean / alpha_p) with mean < r_max, and a sample can
    // only be emitted while the transmittance is >= 1e-3.  Walk the worst case
    // (smallest alpha, shrunk by a margin that covers rounding) in double.
    if (!opt) return 0;
    const int S = opt->num_sample_points_per_ray;
    if (S <= 0) return 0;
    const double g = opt->sdf2weight_gaussian_gamma, ap = opt->sdf2weight_gaussian_alpha;
    if (!(g > 0.0) || !(ap > 0.0) || !(r_max >= 0.0f)) return S;
    const double amin = g * std::exp(-(double)r_max * (1.0 + 1e-3) / ap) * (1.0 - 1e-4);
    if (!(amin > 0.0)) return S;
    double T = 1.0;
    int visits = 0;
    while (T >= 1e-3 * (1.0 - 1e-4) && visits < S) {
        T -= amin;
        ++visits;
    }
    return visits;
}

extern "C" size_t epcq_sampling_workspace_size(int64_t n, int32_t height, int32_t width) {
    if (height <= 0 || width <= 0 || n < 0) return 0;
    return sampling_bytes(n, (int64_t)height * width);
}

extern "C" int32_t epcq_sampling_form(const epcq_options* opt, int64_t n, int32_t height, int32_t width, int32_t live,
                                      int32_t compact, int64_t rays, size_t workspace_bytes) {
    static_assert(kRowsNone == EPCQ_FORM_LANE_SETS && kRowsTiles == EPCQ_FORM_ROW_TILES && kRowsWave == EPCQ_FORM_ROW_WAVES,
                  "the forms' numbers");
    if (!opt || height <= 0 || width <= 0 || n < 0) return EPCQ_FORM_LANE_SETS;
    SampleOpts o = make_opts(nullptr, opt, nullptr);
    const int64_t P = (int64_t)height * width;
    if (rays >= 0) return takes_rows_list(o, rays, P, live, &o, workspace_bytes);
    return takes_rows(o, P, n, live, compact != 0, &o, workspace_bytes);
}

extern "C" int epcq_quick_sampling(const float* xyz, int64_t n, const epcq_camera* cam, const epcq_options* opt,
                                   const int32_t* sorted_idx, const int32_t* hash, int32_t mode, float* sp_xyz,
                                   int32_t* pc_idx, float* sp_t, uint8_t* mask, void* workspace,
                                   size_t workspace_bytes, void* stream) {
    if (int e = check_common(cam, opt, "quick_sampling")) return e;
    if (mode != EPCQ_MODE_COMPAT && mode != EPCQ_MODE_KNN)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: unknown mode");
    if (opt->num_sample_points_per_ray < 0 || opt->num_point_cloud_per_sp < 0)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: negative output size");
    if (mode == EPCQ_MODE_KNN && opt->num_point_cloud_per_sp > 32)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: num_point_cloud_per_sp > 32 in KNN mode");
    if (opt->num_sample_points_per_ray == 0) return EPCQ_OK;
    const int bound = epcq_max_live_samples(opt, opt->radius_threshold);
    SampleOpts o = make_opts(xyz, opt, nullptr);
    o.rows = takes_rows(o, (int64_t)cam->width * cam->height, n, bound, false, workspace, workspace_bytes);
    SampleOut out{};
    out.sp_xyz = sp_xyz;
    out.pc_idx = pc_idx;
    out.sp_t = sp_t;
    out.mask = mask;
    hipStream_t st = as_stream(stream);
    ViewArgs view = make_view(cam, sorted_idx, hash);
    prepare_bounds(o, view, n, cam, sorted_idx, hash, workspace, workspace_bytes, -1, st);
    return launch_sample(o, out, view, nullptr, (int64_t)cam->width * cam->height, mode, bound, st,
                         "quick_sampling");
}

extern "C" int epcq_quick_sampling_rays(const float* xyz, int64_t n, const epcq_camera* cam,
                                        const epcq_options* opt, const int32_t* sorted_idx, const int32_t* hash,
                                        int32_t mode, const int32_t* rays, int64_t R, float* sp_xyz, int32_t* pc_idx,
                                        float* sp_t, uint8_t* mask, void* workspace, size_t workspace_bytes,
                                        void* stream) {
    if (int e = check_common(cam, opt, "quick_sampling")) return e;
    if (mode != EPCQ_MODE_COMPAT && mode != EPCQ_MODE_KNN)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: unknown mode");
    if (opt->num_sample_points_per_ray < 0 || opt->num_point_cloud_per_sp < 0)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: negative output size");
    if (mode == EPCQ_MODE_KNN && opt->num_point_cloud_per_sp > 32)
        return fail(EPCQ_ERR_INVALID, "quick_sampling: num_point_cloud_per_sp > 32 in KNN mode");
    if (R < 0 || (R > 0 && !rays)) return fail(EPCQ_ERR_INVALID, "quick_sampling: bad ray list");
    if (opt->num_sample_points_per_ray == 0 || R == 0) return EPCQ_OK;
    const int bound = epcq_max_live_samples(opt, opt->radius_threshold);
    SampleOpts o = make_opts(xyz, opt, nullptr);
    o.rows = takes_rows_list(o, R, (int64_t)cam->width * cam->height, bound, workspace, workspace_bytes);
    SampleOut out{};
    out.sp_xyz = sp_xyz;
    out.pc_idx = pc_idx;
    out.sp_t = sp_t;
    out.mask = mask;
    hipStream_t st = as_stream(stream);
    ViewArgs view = make_view(cam, sorted_idx, hash);
    prepare_bounds(o, view, n, cam, sorted_idx, hash, workspace, workspace_bytes, R, st);
    return launch_sample(o, out, view, rays, R, mode, bound, st, "quick_sampling");
}

extern "C" int epcq_knn_sampling(const float* xyz, int64_t n, const epcq_camera* cam, const epcq_options* opt,
                                 const int32_t* sorted_idx, const int32_t* hash, const float* radius,
                                 const int32_t* rays, int64_t R, int32_t mode, int32_t s_max, int32_t* n_samples,
                                 float* sample_t, int32_t* nb_idx, float* nb_t, float* nb_dist, const void* feat,
                                 int32_t feat_bf16, int32_t F, float* w, float* agg, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    if (int e = check_common(cam, opt, "knn_sampling")) return e;
    if (mode != EPCQ_MODE_COMPAT && mode != EPCQ_MODE_KNN)
        return fail(EPCQ_ERR_INVALID, "knn_sampling: unknown mode");
    if (opt->num_point_cloud_per_sp < 1 || opt->num_point_cloud_per_sp > 32)
        return fail(EPCQ_ERR_INVALID, "knn_sampling: num_point_cloud_per_sp must be in [1, 32]");
    if (s_max < 1) return fail(EPCQ_ERR_INVALID, "knn_sampling: s_max must be >= 1");
    if (!n_samples || !sample_t || !nb_idx) return fail(EPCQ_ERR_INVALID, "knn_sampling: null output");
    if (feat && (F < 1 || !w || !agg)) return fail(EPCQ_ERR_INVALID, "knn_sampling: bad feature arguments");
    if (rays && R < 0) return fail(EPCQ_ERR_INVALID, "knn_sampling: negative ray count");
    // with per-point radii the caller's s_max stands for the bound
    const int bound = radius ? s_max : std::min<int>(epcq_max_live_samples(opt, opt->radius_threshold), s_max);
    SampleOpts o = make_opts(xyz, opt, radius);
    o.feat = feat;
    o.feat_bf16 = feat_bf16;
    o.F = feat ? F : 0;
    o.feat_vec = feat && F % 4 == 0 && reinterpret_cast<uintptr_t>(feat) % (feat_bf16 ? 8 : 16) == 0;
    SampleOut out{};
    out.s_max = s_max;
    out.n_samples = n_samples;
    out.sample_t = sample_t;
    out.nb_idx = nb_idx;
    out.nb_t = nb_t;
    out.nb_dist = nb_dist;
    out.w = w;
    out.agg = agg;
    const int64_t nr = rays ? R : (int64_t)cam->width * cam->height;
    const int live = radius ? s_max : epcq_max_live_samples(opt, opt->radius_threshold);
    o.rows = rays ? takes_rows_list(o, nr, (int64_t)cam->width * cam->height, live, workspace, workspace_bytes)
                  : takes_rows(o, nr, n, live, true, workspace, workspace_bytes);
    hipStream_t st = as_stream(stream);
    ViewArgs view = make_view(cam, sorted_idx, hash);
    prepare_bounds(o, view, n, cam, sorted_idx, hash, workspace, workspace_bytes, rays ? R : -1, st);
    return launch_sample(o, out, view, rays, nr, mode, bound, st, "knn_sampling");
}

extern "C" int epcq_quick_query(const float* xyz, int64_t n, const epcq_camera* cam, const epcq_options* opt,
                                const int32_t* sorted_idx, const int32_t* hash, const int32_t* rays, int64_t R,
                                int32_t* out, void* stream) {
    if (int e = check_common(cam, opt, "quick_query_for_nearby_point")) return e;
    // the reference's launch limit (epcq_render_topk.cu:317-323)
    const int k2 = opt->kernel_size * opt->kernel_size;
    const int need = (k2 + 31) / 32 * 32;
    int threads = 128;
    if (threads < need) threads = (need + 127) / 128 * 128;
    if (threads >= 1024)
        return fail(EPCQ_ERR_INVALID, "kernel size is too large, can not be handled by current CUDA kernel");
    if (opt->num_point_per_ray < 0) return fail(EPCQ_ERR_INVALID, "quick_query_for_nearby_point: negative num_point_per_ray");
    if (R < 0) return fail(EPCQ_ERR_INVALID, "quick_query_for_nearby_point: negative ray count");
    (void)n;
    if (R == 0 || opt->num_point_per_ray == 0) return EPCQ_OK;
    auto launch = [&](auto kernel, int lanes) {
        kernel<<<dim3((unsigned)ceil_div(R, kBlock / lanes)), dim3(kBlock), 0, as_stream(stream)>>>(
            xyz, sorted_idx, reinterpret_cast<const int2*>(hash), cam->c2w, cam->fx, cam->fy, cam->cx, cam->cy,
            cam->width, cam->height, opt->kernel_size, (opt->kernel_size + 1) / 2, opt->radius_threshold, rays, R,
            opt->num_point_per_ray, out);
    };
    const bool few = opt->num_point_per_ray <= kQueryFew && R >= kQueryHalfWave;
    const bool many = R >= kQueryMany;
    if (few && k2 <= (many ? 9 : 4)) launch(query_kernel<4>, 4);
    else if (few && k2 <= (many ? 81 : 9)) launch(query_kernel<8>, 8);
    else if (k2 <= 32 && R >= kQueryHalfWave) launch(query_kernel<32>, 32);
    else launch(query_kernel<64>, 64);
    return check_launch("quick_query_for_nearby_point");
}

extern "C" int epcq_idw_features(const float* xyz, const void* feat, int32_t feat_bf16, int32_t F,
                                 const float* sp_xyz, const int32_t* nb_idx, int64_t M, int32_t K, float* w,
                                 float* agg, void* stream) {
    if (M < 0 || K < 0 || F < 0) return fail(EPCQ_ERR_INVALID, "idw_features: negative size");
    if (M == 0) return EPCQ_OK;
    idw_kernel<<<dim3((unsigned)ceil_div(M, kBlock)), dim3(kBlock), 0, as_stream(stream)>>>(
        xyz, feat, feat_bf16, F, sp_xyz, nb_idx, M, K, w, agg);
    return check_launch("idw_features");
}
