// Kernels and launches of the row-run sampler (epcq_rows.h), one translation
// unit per neighbour mode and buffer size (epcq_rows_inst_*.hip) so that they
// compile in parallel; epcq_sample.hip dispatches to them.
#pragma once

#include "epcq_common.h"
#include "epcq_rows.h"
#include "epcq_rows_wave.h"

namespace epcq {

// LDS holds four blocks per CU (three with per-point radii, 41.5 KB); the registers of KMAX <= 8 do too
constexpr int kRowWavesPerSimd = 4;
constexpr int kRowWaveWaves = 4;       // waves of a block that takes one ray per wave
constexpr int kDeferredBlocks = 1024;  // blocks of the deferred rays' launch

namespace {

// The view's queue of deferred rays.
__device__ __forceinline__ RowQueue* row_queue(const ViewArgs& view) {
    return reinterpret_cast<RowQueue*>(const_cast<float4*>(view.cone_a));
}

// n deferred rays of a view, dealt to the launch's waves.
template <int MODE, int KMAX, int LAY, bool PR>
__device__ __forceinline__ void run_queue(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, int n,
                                          RowWaveSmem& sm) {
    const RowList<PR> src{view.pts, view.prad, view.sorted_idx, o.xyz, o.radius};
    const int* rays = row_queue(view)->ray;
    const int waves = (int)gridDim.x * kRowWaveWaves;
    for (int i = uniform((int)blockIdx.x * kRowWaveWaves + (int)threadIdx.x / kWave); i < n; i += waves) {
        const int q = uniform(rays[i]);
        const int u = q % view.W, v = q / view.W;
        Ray ray;
        view_ray(view, u, v, ray);
        run_ray_rows<MODE, KMAX, LAY, PR>(o, out, view, src, ray, u, v, q, sm);
        wave_lds_fence();  // the next ray reuses the wave's LDS
    }
}

// One block per tile; the blocks of an XCD take consecutive tiles, which share
// their window rows in its L2.
template <int MODE, int KMAX, int LAY, bool PR>
__global__ __launch_bounds__(kRowThreads, KMAX <= 8 ? kRowWavesPerSimd : 2) void sample_rows_kernel(
    SampleOpts o, SampleOut out, ViewArgs view, int tiles_x) {
    __shared__ RowSmem<PR> sm;
    row_tile_body<MODE, KMAX, LAY, PR>(o, out, view, xcd_tile((int)blockIdx.x, (int)gridDim.x), tiles_x,
                                       row_queue(view), sm);
}

// The rays that sample_rows_kernel put in its queue, one wave per ray.
template <int MODE, int KMAX, int LAY, bool PR>
__global__ __launch_bounds__(kRowWaveWaves* kWave) void sample_deferred_kernel(SampleOpts o, SampleOut out,
                                                                               ViewArgs view) {
    __shared__ RowWaveSmem sm[kRowWaveWaves];
    run_queue<MODE, KMAX, LAY, PR>(o, out, view, row_queue(view)->count, sm[threadIdx.x / kWave]);
}

// Waves per SIMD of the form of one wave per ray: LDS holds four blocks per CU,
// and the registers have to as well.  The feature layout takes what it needs (94
// to 104 registers with buffers of 8, up to 213 with 32).
template <int LAY>
constexpr int kListWavesPerSimd = LAY != kLayFeat ? 4 : 1;

// One wave per ray of a list, or of the whole image (rays null: R pixels).
template <int MODE, int KMAX, int LAY, bool PR>
__global__ __launch_bounds__(kRowWaveWaves* kWave, kListWavesPerSimd<LAY>) void sample_list_rows_kernel(SampleOpts o, SampleOut out,
                                                                                ViewArgs view,
                                                                                const int* __restrict__ rays,
                                                                                int64_t R) {
    __shared__ RowWaveSmem sm[kRowWaveWaves];
    const int64_t ri = (int64_t)blockIdx.x * kRowWaveWaves + uniform((int)threadIdx.x / kWave);
    if (ri >= R) return;  // the whole wave; the block has no barrier
    const int q = rays ? uniform(rays[ri]) : (int)ri;
    if (!(q >= 0 && q < (int64_t)view.W * view.H)) {
        write_tail_wave<MODE, LAY>(o, out, ri, 0);
        return;
    }
    const RowList<PR> src{view.pts, view.prad, view.sorted_idx, o.xyz, o.radius};
    const int u = q % view.W, v = q / view.W;
    Ray ray;
    view_ray(view, u, v, ray);
    run_ray_rows<MODE, KMAX, LAY, PR>(o, out, view, src, ray, u, v, ri, sm[threadIdx.x / kWave]);
}

}  // namespace

template <int MODE, int KMAX, int LAY, bool PR>
void launch_rows_lay(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, const int* rays, int64_t R,
                     hipStream_t st) {
    const dim3 wave_block(kRowWaveWaves * kWave);
    if (rays || o.rows == kRowsWave) {
        sample_list_rows_kernel<MODE, KMAX, LAY, PR>
            <<<dim3((unsigned)ceil_div(R, kRowWaveWaves)), wave_block, 0, st>>>(o, out, view, rays, R);
        return;
    }
    const int tiles_x = (int)ceil_div(view.W, kRowTileW);
    const unsigned tiles = (unsigned)(tiles_x * ceil_div(view.H, kRowTileH));
    sample_rows_kernel<MODE, KMAX, LAY, PR><<<dim3(tiles), dim3(kRowThreads), 0, st>>>(o, out, view, tiles_x);
    sample_deferred_kernel<MODE, KMAX, LAY, PR><<<dim3(kDeferredBlocks), wave_block, 0, st>>>(o, out, view);
}

template <int MODE, int KMAX>
void launch_rows(const SampleOpts& o, const SampleOut& out, const ViewArgs& view, const int* rays, int64_t R,
                 hipStream_t st) {
    if (out.sp_xyz) launch_rows_lay<MODE, KMAX, kLayDense, false>(o, out, view, rays, R, st);
    else if (o.feat && o.radius) launch_rows_lay<MODE, KMAX, kLayFeat, true>(o, out, view, rays, R, st);
    else if (o.feat) launch_rows_lay<MODE, KMAX, kLayFeat, false>(o, out, view, rays, R, st);
    else if (o.radius) launch_rows_lay<MODE, KMAX, kLayCompact, true>(o, out, view, rays, R, st);
    else launch_rows_lay<MODE, KMAX, kLayCompact, false>(o, out, view, rays, R, st);
}

}  // namespace epcq

#define EPCQ_INSTANTIATE_ROWS(MODE, KMAX)                                                                       \
    template void epcq::launch_rows<MODE, KMAX>(const epcq::SampleOpts&, const epcq::SampleOut&,                \
                                                const epcq::ViewArgs&, const int*, int64_t, hipStream_t);
