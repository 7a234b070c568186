// Groups of consecutive layers of a dense block on the matrix cores (fp32; 3D: the backward pass).
//
// The layers i, i + 1, ... of a group read the same channels [0, c) of the stack, c the number
// of channels in front of the first of them.  Taken together they are one matrix product over
// those channels: with one row per (output, tap) seven one-channel layers are a 63 x c weight
// matrix, which fills a slab of 64 rows to 98 %, and every channel is read once for seven layers
// (the backward pass: for up to fourteen, two slabs) instead of once (three rows at a time) per layer.
#pragma once
#include "msd_kernels.h"
#include "msd_rows.h"

namespace msd {
namespace group2d {

constexpr int kTaps = 9;
constexpr int kSlabOut = 7;                       // outputs of a slab: 7 * 9 = 63 of 64 matrix rows
constexpr int kSlabOut3d = 2;                     // 3D: 2 * 27 = 54
constexpr int kRows = 64;                         // matrix rows of a slab
constexpr int kMaxOut = 14;                       // outputs of a group: one or two slabs
constexpr int kMaxAbove = 7;                      // outputs that complete a channel of the group in one launch
constexpr int kMaxLower = 8;                      // channels of a group's lower half
constexpr int kTiles = kRows / 16;
constexpr int kChunk = 128;                       // channels whose weights are in LDS at a time

// The outputs of a group: dilation, and weights of the channels from 0 on, of each.
// Between LDS accesses of one wave: LDS executes them in order, only the compiler has to be kept from
// reordering them.
__device__ __forceinline__ void own_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Between the LDS accesses of a workgroup (of LDS only: the loads and stores of memory stay in flight).
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct Outputs {
    int n;
    int dil[kMaxOut];
    const float *k[kMaxOut];
};

// How the rows of an image are spread over waves: a team of `waves` waves owns one row (or one
// segment of a long row: 64 * waves voxels of which `inner` are its own, the rest overlap with its
// neighbours), `rpw` teams form a workgroup.
struct Teams {
    int waves, rpw, segs, inner;
};

// Chosen so that as few waves as possible work in all, counted with those that find no room: up
// to 16 waves share a compute unit, as one workgroup or as two of at most 8 (which also lets one
// work while the other finishes a row).
inline Teams make_teams(int W, int halo)
{
    Teams best{0, 0, 0, 0};
    double best_cost = 0;
    for (int w = 1; w <= 16; w++) {
        int inner = W, segs = 1;
        if (w * kWave < W) {
            inner = (w * kWave - 2 * halo) & ~3;
            if (inner < kWave) continue;
            segs = (W + inner - 1) / inner;
        }
        const int rpw = w <= 8 ? 8 / w : 1;
        const double cost = (double)segs * w * 16 / (w <= 8 ? 2 * rpw * w : w);
        if (best.waves == 0 || cost < best_cost) {
            best = Teams{w, rpw, segs, inner};
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace group2d

// Rows of W voxels that the launches of a forward group take where their alignment allows it.
bool group_rows_supported_2d(int64_t W);

// z[b][3 o + ky][y][x] = sum over the g.C channels and kx of k[o][c][ky][kx] * x[c][y][fold(x + dil_o (kx - 1))]:
// what row y of the channels contributes to the output rows that read it through tap row ky.
bool group_push_supported_2d(const Geom &g, const View<const float> &x, int dmax);
hipError_t group_push_2d(const Geom &g, const View<const float> &x, const group2d::Outputs &out, float *z, hipStream_t s);

// The same for up to kMaxOut outputs, more than kSlabOut.  table: group_table_floats_2d floats (their address a multiple of 16 bytes).
bool group_split_supported_2d(int64_t W, int dmax);
int64_t group_table_floats_2d(int64_t channels);
hipError_t group_push_split_2d(const Geom &g, const View<const float> &x, const group2d::Outputs &out, float *z, float *table,
                               hipStream_t s);

// One layer of the group from its planes and the g.C channels that the group has added (with ReLU).
bool group_finish_supported_2d(const Geom &g, const View<const float> &x, const View<float> &out);
hipError_t group_finish_2d(const Geom &g, const View<const float> &x, const float *k, const float *bias,
                           const View<float> &out, const ForwardSums &sums, hipStream_t s);

// Backward pass of a group over the channels [0, g.C) of the stack x: the first `update` channels of
// grads get grad_input (masked with their activations from `mask_from` on), gk[o] the weight gradients
// of output o's channels[o] input channels, gb the bias gradients.  The outputs' gradients are the
// channels from `first` on.  ws: group_pull_floats floats (rows: of an image, or of all slices of a volume).
int64_t group_pull_floats(int64_t batch, int64_t rows, int64_t W, int64_t channels);
bool group_pull_supported(const Geom &g, const View<const float> &x, const View<float> &gx);
hipError_t group_pull(const Geom &g, const View<const float> &x, const group2d::Outputs &out, int update, int mask_from,
                      const View<float> &grads, int first, const int *channels, float *const *gk, float *gb,
                      float *ws, bool reverse, hipStream_t s);

// All three gradients of a single layer (of dilation g.dil; g.Wd outputs of one slab) over an image, or a volume without gaps,
// written and not added to.  gy: the masked output gradient, rows as in x.  ws: group_pull_floats floats.
bool layer_pull_supported(const Geom &g, const View<const float> &x, const View<const float> &gy, const View<float> &gx);
hipError_t layer_pull(const Geom &g, const View<const float> &x, const View<const float> &gy, const float *k, const View<float> &gx,
                      float *gk, float *gb, float *ws, hipStream_t s);

// Completes the gradient of the `width` channels from `channel` on: adds what the outputs right
// above them (`above`, their weights of these channels) contribute, and applies the ReLU mask.
hipError_t group_finish_back(const Geom &g, const View<const float> &x, const View<float> &grads, int channel, int width,
                             const group2d::Outputs &above, hipStream_t s);

// Adds to the gradients of the `channels` channels from `channel` on what the outputs right above
// them (at most kSlabOut) contribute, and completes the last `width` of them.
hipError_t group_spread_back_2d(const Geom &g, const View<const float> &x, const View<float> &grads, int channel, int channels,
                                int width, const group2d::Outputs &above, hipStream_t s);

}  // namespace msd
