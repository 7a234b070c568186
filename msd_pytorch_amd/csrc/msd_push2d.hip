// Forward pass of a group of layers over the channels they share (msd_group.h).
//
// Per voxel v of an input row and matrix column m = (output o, tap t) the kernel forms
//     Y[v][m] = sum_c x[c][v] * k[o][c][t],
// a product with no shifts in it: the voxels are loaded as they lie in memory, the weights come
// from a table in LDS.  Then the shifts: along x they are taken through LDS while the row is
// complete in the workgroup,
//     Z[o][ky][x] = sum_kx Y[fold(x + dil_o (kx - 1))][o, ky, kx],
// and Z, three planes per output, is all that is written; the launch that finishes a layer adds
// the three rows y - dil, y, y + dil of its planes (ForwardSums).
//
// Bound by the matrix cores: 64 columns x 4 channels x 64 voxels are 16 instructions of 32 cycles
// per SIMD for 1 KB of input.  What stands beside them is the passage through LDS, whose price is
// the instructions of 16 waves on four SIMDs: the voxels are the rows of the product so that a
// lane's four results are consecutive voxels of one column (16-byte LDS writes as they come out
// of the matrix core), and the three columns of an (output, tap row) never straddle two tiles, so
// that a tile is finished with two barriers, no lane is masked and all its LDS reads are in flight
// together.  1024 x 1024, 7 layers: 35 us + 1.1 us per channel (0.95 us are the matrix instructions
// at the clock they run at), 139 us at 94 channels where seven launches of fwd_lattice took 520;
// output by output, with the voxels as columns, it was 45 us + 1.1 us.
// Counters over the 13 launches of a forward pass of depth 100 there: 4.1 GB in 1.14 ms, matrix cores busy 52 %.
#include "msd_group.h"

#include <algorithm>

namespace msd {
namespace group2d {
namespace {

constexpr int kMaxWaves = 16;
constexpr int kAhead = 2;                         // steps of four channels per register set
constexpr int kTriples = 5;                       // (output, tap row) triples of columns per tile

typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct PushArgs {
    int C, H, W, items, segs;                     // items: rows x segments x batch
    int64_t xsb, xsc, xsy;                        // strides of x
    int waves, rpw, inner, halo;
    Outputs out;
};

// Column 16 t + i of the product: the triple and the tap column kx it stands for.  Five triples fill
// 15 columns of a tile; the 21st lies in the last columns of the first three tiles.
__device__ __forceinline__ int triple_of(int t, int i) { return i < 15 ? kTriples * t + i / 3 : 20; }
__device__ __forceinline__ int kx_of(int t, int i) { return i < 15 ? i % 3 : t; }

// LDS rows of a team: 15 for the triples of the tile at hand, then the last columns of the four tiles.
constexpr int kStaged = 15 + kTiles;

__global__ __launch_bounds__(kMaxWaves *kWave) void push_rows(PushArgs a, const float *__restrict__ x,
                                                              float *__restrict__ z)
{
    extern __shared__ float lds[];
    const int S = a.waves * kWave, SP = S + 4;    // voxels of a team; rows 16 bytes apart in the banks
    f32x4_t *table = reinterpret_cast<f32x4_t *>(lds);              // [step][lane]: one value per tile
    const int table_steps = (min(a.C, kChunk) + 3) / 4;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int team = wave / a.waves, tw = wave % a.waves;
    const int n = lane % 16, q = lane / 16;
    const int tx = tw * kWave + lane;             // the voxel that the lane finishes
    float *const T = lds + (size_t)table_steps * kWave * kTiles + (size_t)team * kStaged * SP;
    float *const put = T + n * SP + tw * kWave + 4 * q;             // where the lane's results go
    const int last_column = n == 15 ? SP : 0;     // (the last columns of the tiles keep rows of their own)
    int loaded = -1;

    // where a team's item lies: row y of image b, the segment's voxels from `first` on
    struct Place {
        int y, b, own0, first;
        uint64_t base;
        uint32_t at[4];
    };
    auto locate = [&](int item0) {
        Place p;
        const int it = min(item0 + team, a.items - 1);
        const int seg = it % a.segs, row = it / a.segs;
        p.y = row % a.H;
        p.b = row / a.H;
        p.own0 = seg * a.inner;                   // the segment's own voxels start here
        p.first = a.segs == 1 ? 0 : max(0, min(p.own0 - a.halo, a.W - S));
        p.base = reinterpret_cast<uint64_t>(x + (int64_t)p.b * a.xsb + (int64_t)p.y * a.xsy);
#pragma unroll
        for (int j = 0; j < 4; j++)               // (lanes past the row end load its last voxel)
            p.at[j] = 4u * (uint32_t)min(p.first + tw * kWave + 16 * j + n, a.W - 1);
        return p;
    };
    // Step st of the chunk of cn channels from c0 on stands for the channels c0 + 4 st + q; past the
    // last channel the lanes repeat it, and its repetitions are cleared before they are used.
    auto request = [&](const Place &p, int c0, int cn, int st, float (&d)[4]) {
        const int s = min(st, (cn + 3) / 4 - 1);
        const uint64_t cb = p.base + (uint64_t)(c0 + 4 * s) * (uint64_t)a.xsc * 4u;
        const uint32_t cq = (uint32_t)min(q, cn - 1 - 4 * s) * (uint32_t)(a.xsc * 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float one[1];
            load_global_vec<1>(cb, cq + p.at[j], one);
            d[j] = one[0];
        }
    };

    int item0 = blockIdx.x * a.rpw;
    Place here = locate(item0);
    float set[2][kAhead][4];
#pragma unroll
    for (int u = 0; u < kAhead; u++) request(here, 0, min(kChunk, a.C), u, set[0][u]);
    for (; item0 < a.items; item0 += gridDim.x * a.rpw) {
        f32x4_t acc[4][kTiles];                   // [16 voxels][tile]
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int t = 0; t < kTiles; t++) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

        for (int c0 = 0; c0 < a.C; c0 += kChunk) {
            const int cn = min(kChunk, a.C - c0), steps = (cn + 3) / 4;
            if (loaded != c0) {                   // uniform
                __syncthreads();
                // a thread's entries are one column of the product, every blockDim / 64 channels;
                // eight loads at a time
                const int t = tid % kTiles, i = tid / kTiles % 16, tri = triple_of(t, i), o = min(tri / 3, kSlabOut - 1);
                const bool column = o < a.out.n && !(i == 15 && t == 3);
                const float *const k = a.out.k[column ? o : 0] + (int64_t)c0 * kTaps + (tri % 3) * 3 + kx_of(t, i);
                const int stride = blockDim.x / kWave, end = 4 * steps;
                for (int cb = tid / kWave; cb < end; cb += 8 * stride) {
                    float w[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) w[u] = k[min(cb + u * stride, cn - 1) * kTaps];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const int c = cb + u * stride;
                        if (c < end) lds[c * kWave + tid % kWave] = column && c < cn ? w[u] : 0.f;
                    }
                }
                __syncthreads();
                loaded = c0;
            }
            if (c0 > 0) {
#pragma unroll
                for (int u = 0; u < kAhead; u++) request(here, c0, cn, u, set[0][u]);
            }
            for (int st = 0; st < steps; st += 2 * kAhead) {
#pragma unroll
                for (int half = 0; half < 2; half++) {
                    const int s0 = st + half * kAhead;
#pragma unroll
                    for (int u = 0; u < kAhead; u++) request(here, c0, cn, s0 + kAhead + u, set[1 - half][u]);
#pragma unroll
                    for (int u = 0; u < kAhead; u++) {
                        if (s0 + u >= steps) break;                 // uniform
                        if (4 * (s0 + u) + 4 > cn) {                // uniform: an infinity times a weight of zero is NaN
                            const bool past = 4 * (s0 + u) + q >= cn;
#pragma unroll
                            for (int j = 0; j < 4; j++) set[half][u][j] = past ? 0.f : set[half][u][j];
                        }
                        const f32x4_t w = table[(s0 + u) * kWave + lane];
#pragma unroll
                        for (int j = 0; j < 4; j++)
#pragma unroll
                            for (int t = 0; t < kTiles; t++)
                                acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(set[half][u][j], w[t], acc[j][t], 0, 0, 0);
                    }
                }
            }
        }

        // The next row's first channels are asked for before this row's results are stored: loads
        // behind the stores would have to wait for them.
        const int xx = here.first + tx, first = here.first;
        const bool store = item0 + team < a.items && xx >= here.own0 && xx < min(a.W, here.own0 + a.inner);
        const uint64_t zb = reinterpret_cast<uint64_t>(z + ((int64_t)here.b * 3 * a.out.n * a.H + here.y) * a.W);
        here = locate(item0 + gridDim.x * a.rpw);
#pragma unroll
        for (int u = 0; u < kAhead; u++) request(here, 0, min(kChunk, a.C), u, set[0][u]);

        // acc[j][t][r] = Y[16 j + 4 q + r][16 t + n], tile by tile through LDS
        const uint32_t zat = 4u * (uint32_t)xx;
        const int xc = min(xx, a.W - 1);
#pragma unroll
        for (int t = 0; t < kTiles; t++) {
            if (kTriples * t >= 3 * a.out.n) break;                 // uniform
            __syncthreads();                      // (the tile before has been read)
#pragma unroll
            for (int j = 0; j < 4; j++) *reinterpret_cast<f32x4_t *>(put + t * last_column + 16 * j) = acc[j][t];
            __syncthreads();
            // all of the tile's reads before the first use, and no branch around them: one LDS round
            // trip per tile instead of one per triple (lanes that store nothing read what they hit)
            constexpr int kMost = kTriples + 1;
            const int triples = t == kTiles - 1 ? kMost : kTriples;
            float sum[kMost][3];
#pragma unroll
            for (int i = 0; i < kMost; i++) {
                if (i >= triples) break;
                const float *const r = T + 3 * i * SP;
                const int d = a.out.dil[(kTriples * t + i) / 3], lo = xc - d, hi = xc + d;
                sum[i][0] = r[max(lo, -1 - lo) - first];            // fold(xc - d), fold(xc + d): dil <= W
                sum[i][1] = r[SP + tx];
                sum[i][2] = r[2 * SP + min(hi, 2 * a.W - 1 - hi) - first];
            }
#pragma unroll
            for (int i = 0; i < kMost; i++) {
                const int tri = kTriples * t + i;
                if (i >= triples || tri >= 3 * a.out.n) break;      // uniform
                const float v[1] = {sum[i][0] + sum[i][1] + sum[i][2]};
                if (store) store_global_vec<1>(zb + (uint64_t)tri * (uint64_t)((int64_t)a.H * a.W * 4), zat, v);
            }
        }
    }
}

// Finishes one layer of a group: the planes that push_rows left, plus NC channels that the group
// itself has written since, bias and ReLU.
//
// A team of lanes owns a row, V voxels per lane; the 3 WOUT rows of planes and the 3 NC rows of
// channels are requested at once (they come from the caches), the x-taps of the channels meet
// through LDS behind one barrier as in fwd_lattice.  The launch is short: bound by its ramp and one
// chain of round trips.  Lattices of four or five rows per workgroup (fwd_lattice with the planes
// added) read the channels' rows half as often but take ten barriers one after the other:
// 9.7-12.5 us against 5.2-8.8 us at 1024 x 1024 for one to six channels.
template <int V, int NC, int WOUT>
__global__ __launch_bounds__(V == 1 ? 1024 : 512) void finish_rows(Geom g, RowTeams rt, View<const float> x,
                                                                  const float *__restrict__ k,
                                                                  const float *__restrict__ bias, View<float> out,
                                                                  ForwardSums sums)
{
    extern __shared__ float lds[];
    const int team = threadIdx.x / rt.lpr, lane = threadIdx.x % rt.lpr;
    const int lb = block_for_xcd(blockIdx.x, gridDim.x, true);
    if (lb * rt.rpw >= rt.nrows) return;          // padding block (whole workgroup)
    const int row = lb * rt.rpw + team, y = min(row, rt.nrows - 1), b = blockIdx.y;
    const bool act = row < rt.nrows && lane * V < g.W;
    const int x0 = min(lane * V, g.W - V);
    int rows[3];
#pragma unroll
    for (int ky = 0; ky < 3; ky++) rows[ky] = reflect_idx(y + (ky - 1) * g.dil, g.H);
    float zv[WOUT][3][V], xv[NC > 0 ? NC : 1][3][V];
#pragma unroll
    for (int co = 0; co < WOUT; co++)
#pragma unroll
        for (int ky = 0; ky < 3; ky++)
            load_vec<V>(sums.z + (int64_t)b * sums.zsb + ((int64_t)(3 * co + ky) * g.H + rows[ky]) * g.W + x0, zv[co][ky]);
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int ky = 0; ky < 3; ky++)
            load_vec<V>(x.p + (int64_t)b * x.sb + c * x.sc + rows[ky] * x.sy + x0, xv[c][ky]);

    float acc[WOUT][3][V];
#pragma unroll
    for (int co = 0; co < WOUT; co++) {
#pragma unroll
        for (int i = 0; i < V; i++) {
            acc[co][0][i] = acc[co][2][i] = 0.f;
            acc[co][1][i] = bias[co] + (zv[co][0][i] + zv[co][1][i] + zv[co][2][i]);
        }
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int ky = 0; ky < 3; ky++)
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    const float wv = k[co * sums.kco + c * kTaps + ky * 3 + r];
#pragma unroll
                    for (int i = 0; i < V; i++) acc[co][r][i] += xv[c][ky][i] * wv;
                }
    }
    const int rowlen = V * rt.lpr;
    float *const T = lds + (size_t)team * WOUT * 2 * rowlen;
    if constexpr (NC > 0) {
#pragma unroll
        for (int co = 0; co < WOUT; co++)
#pragma unroll
            for (int i = 0; i < V; i++) {
                T[(2 * co) * rowlen + i * rt.lpr + lane] = acc[co][0][i];
                T[(2 * co + 1) * rowlen + i * rt.lpr + lane] = acc[co][2][i];
            }
        __syncthreads();
    }
    if (!act) return;
#pragma unroll
    for (int co = 0; co < WOUT; co++) {
        float o[V];
#pragma unroll
        for (int i = 0; i < V; i++) {
            float s = acc[co][1][i];
            if constexpr (NC > 0)
                s += T[(2 * co) * rowlen + staged_index<V>(reflect_idx(x0 + i - g.dil, g.W), rt.lpr)] +
                     T[(2 * co + 1) * rowlen + staged_index<V>(reflect_idx(x0 + i + g.dil, g.W), rt.lpr)];
            o[i] = s > 0.f ? s : 0.f;
        }
        store_vec<V>(out.p + (int64_t)b * out.sb + (int64_t)co * out.sc + (int64_t)y * out.sy + x0, o);
    }
}

template <int V, int NC, int WOUT>
hipError_t finish_launch(const Geom &g, const View<const float> &x, const float *k, const float *bias,
                         const View<float> &out, const ForwardSums &sums, hipStream_t s)
{
    RowTeams rt;
    if (!make_row_teams(g, V, &rt) || (V > 1 && rt.lpr * rt.rpw > 512)) return hipErrorInvalidConfiguration;
    const size_t lds = NC > 0 ? (size_t)rt.rpw * WOUT * 2 * V * rt.lpr * sizeof(float) : 0;
    const int blocks = xcd_grid((rt.nrows + rt.rpw - 1) / rt.rpw);
    hipLaunchKernelGGL((finish_rows<V, NC, WOUT>), dim3(blocks, g.B, 1), dim3(rt.lpr * rt.rpw), lds, s, g, rt, x, k, bias,
                       out, sums);
    return hipGetLastError();
}

template <int V>
hipError_t finish_pick(const Geom &g, const View<const float> &x, const float *k, const float *bias,
                       const View<float> &out, const ForwardSums &sums, hipStream_t s)
{
    if (g.Wd == 1) {
        switch (g.C) {
        case 0: return finish_launch<V, 0, 1>(g, x, k, bias, out, sums, s);
        case 1: return finish_launch<V, 1, 1>(g, x, k, bias, out, sums, s);
        case 2: return finish_launch<V, 2, 1>(g, x, k, bias, out, sums, s);
        case 3: return finish_launch<V, 3, 1>(g, x, k, bias, out, sums, s);
        case 4: return finish_launch<V, 4, 1>(g, x, k, bias, out, sums, s);
        case 5: return finish_launch<V, 5, 1>(g, x, k, bias, out, sums, s);
        case 6: return finish_launch<V, 6, 1>(g, x, k, bias, out, sums, s);
        }
    } else if (g.Wd == 2) {
        switch (g.C) {
        case 0: return finish_launch<V, 0, 2>(g, x, k, bias, out, sums, s);
        case 2: return finish_launch<V, 2, 2>(g, x, k, bias, out, sums, s);
        case 4: return finish_launch<V, 4, 2>(g, x, k, bias, out, sums, s);
        }
    }
    return hipErrorInvalidConfiguration;
}

// Voxels per lane of the finishing launch: 4 where rows are whole aligned groups of four and fit a
// workgroup of 512 lanes, else 1 (rows of up to 1024 voxels); 0: none.
int finish_vec(const Geom &g, const View<const float> &x, const View<float> &out)
{
    if (rows_aligned(x, g.W, 4) && rows_aligned(out, g.W, 4) && g.W <= 2048) return 4;
    return g.W <= 1024 ? 1 : 0;
}

}  // namespace
}  // namespace group2d

bool group_rows_supported_2d(int64_t W)
{
    // (the longer rows: fwd_lattice with a workgroup of 1024 lanes, two or four voxels each)
    return W >= 32 && (W <= 1024 || (W % 2 == 0 && W <= 2048) || (W % 4 == 0 && W <= 4096));
}

bool group_push_supported_2d(const Geom &g, const View<const float> &x, int dmax)
{
    using namespace group2d;
    return g.ndim == 2 && x.sx == 1 && group_rows_supported_2d(g.W) && dmax <= 128 && g.C >= 1 && x.sc < ((int64_t)1 << 28) &&
           (int64_t)g.B * g.H * ((g.W + kWave - 1) / kWave) < ((int64_t)1 << 30);
}

hipError_t group_push_2d(const Geom &g, const View<const float> &x, const group2d::Outputs &out, float *z, hipStream_t s)
{
    using namespace group2d;
    int dmax = 0;
    for (int o = 0; o < out.n; o++) dmax = std::max(dmax, out.dil[o]);
    if (out.n < 1 || out.n > kSlabOut || !group_push_supported_2d(g, x, dmax)) return hipErrorInvalidValue;
    const int halo = (dmax + 3) & ~3;
    const Teams t = make_teams(g.W, halo);
    PushArgs a{g.C, g.H, g.W, g.B * g.H * t.segs, t.segs, x.sb, x.sc, x.sy, t.waves, t.rpw, t.inner, halo, out};
    const size_t lds = ((size_t)((std::min(g.C, kChunk) + 3) / 4) * kWave * kTiles + (size_t)t.rpw * kStaged * (t.waves * kWave + 4)) * 4;
    const int threads = t.waves * t.rpw * kWave;
    static LargeLds large;
    hipError_t e = large.allow(reinterpret_cast<const void *>(&push_rows), 160 * 1024);
    if (e != hipSuccess) return e;
    // as many workgroups as are resident: 16 waves of 128 registers per compute unit, 160 KB of LDS
    const int per_cu = std::max<int>(1, std::min<int>(kMaxWaves * kWave / threads, (int)(160 * 1024 / lds)));
    const int blocks = (a.items + t.rpw - 1) / t.rpw;
    hipLaunchKernelGGL(push_rows, dim3(std::min(blocks, 256 * per_cu)), dim3(threads), lds, s, a, x.p, z);
    return hipGetLastError();
}

bool group_finish_supported_2d(const Geom &g, const View<const float> &x, const View<float> &out)
{
    return g.ndim == 2 && x.sx == 1 && out.sx == 1 && group2d::finish_vec(g, x, out) != 0 &&
           ((g.Wd == 1 && g.C < group2d::kSlabOut) || (g.Wd == 2 && g.C < 6 && g.C % 2 == 0));
}

hipError_t group_finish_2d(const Geom &g, const View<const float> &x, const float *k, const float *bias,
                           const View<float> &out, const ForwardSums &sums, hipStream_t s)
{
    const int v = group2d::finish_vec(g, x, out);
    if (v == 4) return group2d::finish_pick<4>(g, x, k, bias, out, sums, s);
    if (v == 1) return group2d::finish_pick<1>(g, x, k, bias, out, sums, s);
    return hipErrorInvalidConfiguration;
}

}  // namespace msd
