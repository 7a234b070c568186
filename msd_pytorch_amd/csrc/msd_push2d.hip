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
#include "msd_split.h"

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

// ---- More than seven outputs: two slabs of columns, fp32 values in bf16 parts (msd_split.h).
//
// A wave walks a row, or a part of one, in segments of 64 voxels and forms the columns of one slab; no
// wave waits for another.  x arrives by channel in 256-byte pieces, four voxels of eight channels per lane: split, they are operands of the
// matrix cores as they stand (voxel 4 n + j is row n of product j).  The shifts along x are taken as in push_rows, tile by tile of the
// columns, through the wave's own part of LDS; what a segment's outputs need of the segment before stays in registers, so that nothing is formed
// twice.  Every channel leaves memory once for up to fourteen outputs: the workgroups of the two slabs are neighbours on one XCD and
// work on the same rows at the same time.
//
// A workgroup has one slab, so that the weights of 256 channels lie in LDS at a time: with both slabs in one it were 128, and to load them
// anew for every segment took 260 of the 1400 us over 131 channels.  Without them x is read through the L2 twice, which costs nothing
// measurable.  2048 x 2048, 14 outputs, us, both slabs in a workgroup / one: over 16 / 58 / 100 / 128 channels 559 / 553, 743 / 730, 918 / 890, 939 / 904, over
// 142 / 184 1390 / 1064, 1579 / 1247.  Above 256 the steps of one segment of a row go up and the next one's down, so that a part of the table is
// loaded once less per segment: over 268 / 324 / 380 2025 / 1914, 2250 / 2068, 2719 / 2449.  Every row (or part of one) begins upwards: the order in which a
// voxel's channels are added goes with its place in the row, as the sign does that its values are taken with, and not with the row or the image of a
// batch (rows of an odd number of segments load one part more; the times are the same).  (x by way of a transposition in LDS instead of in the operands' own layout: the same times.)
//
// Bound by latencies: eight waves per compute unit (their registers), each a chain of loads, split and matrix
// instructions; the matrix part is a quarter of the time.  With a workgroup per row, its waves
// side by side and barriers around each tile of the shifts: 2.3 ms at 2048 x 2048 over 120.
constexpr int kSlabs = 2;
constexpr int kPushWaves = 8;                     // of a workgroup; one workgroup per compute unit
constexpr int kHalo = 16;                         // dilations up to here
constexpr int kStepChannels = 32;
constexpr int kTileBytes = 3 * kWave * 16;        // weights of 16 columns, a step
constexpr int kTableSteps = 8;                    // steps whose weights (of a slab) are in LDS at a time
constexpr int kTableBytes = kTableSteps * kTiles * kTileBytes;
constexpr int kLine = 2 * kHalo + kWave + 4;      // floats of a staged row (16 bytes apart in the banks)
constexpr int kOwnBytes = kStaged * kLine * 4 + 16;                 // of a wave: staged rows
static_assert(kOwnBytes % 16 == 0, "16-byte accesses");
constexpr int kSplitLds = kTableBytes + kPushWaves * kOwnBytes;

struct SplitArgs {
    int C, H, W, items, parts, length;            // items: parts of all rows; outputs of a part
    int64_t xsb, xsc, xsy;                        // strides of x
    Outputs out;
};

// Channel (of the step's 32) that value e of the lanes q stands for.
__host__ __device__ __forceinline__ int channel_of(int q, int e) { return 4 * e + q; }

// [step][tile of columns][part][lane (column n, q)]: eight channels each; bad[step]: some of them have to be taken whole,
// and all of the step's lie so.
__global__ __launch_bounds__(kSlabs *kTiles *kWave) void push_table(const SplitArgs a, bf16x8_t *__restrict__ table, int *__restrict__ bad)
{
    const int step = blockIdx.x, t = threadIdx.x / kWave, lane = threadIdx.x % kWave, i = lane % 16, q = lane / 16;
    const int tri = triple_of(t % kTiles, i), o = t / kTiles * kSlabOut + tri / 3;
    const bool column = o < a.out.n && !(i == 15 && t % kTiles == 3);
    const float *const k = a.out.k[column ? o : 0] + (tri % 3) * 3 + kx_of(t % kTiles, i);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int c = step * kStepChannels + channel_of(q, e);
        const float w = k[min(c, a.C - 1) * kTaps];
        v[e] = column && c < a.C ? w : 0.f;
    }
    float scaled[8];
#pragma unroll
    for (int e = 0; e < 8; e++) scaled[e] = v[e] * kSplitScale;
    Split8 s;
    const int any = __syncthreads_or(taken_whole(split8(scaled, s)));
    if (any) put_whole(v, s);
    if (threadIdx.x == 0) bad[step] = any;
#pragma unroll
    for (int p = 0; p < 3; p++) table[((step * kSlabs * kTiles + t) * 3 + p) * kWave + lane] = s.p[p];
}

__global__ __launch_bounds__(kPushWaves *kWave, 2) void push_split(const SplitArgs a, const float *__restrict__ x,
                                                                  const bf16x8_t *__restrict__ table, const int *__restrict__ bad,
                                                                  float *__restrict__ z)
{
    constexpr int kStepEntries = kTiles * 3 * kWave;
    extern __shared__ __attribute__((aligned(16))) char split_lds[];
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), slab = blockIdx.x / kXcds % kSlabs;
    const int pair = blockIdx.x / (kSlabs * kXcds) * kXcds + blockIdx.x % kXcds, pairs = gridDim.x / kSlabs;      // of workgroups, on one XCD
    bf16x8_t *const weights = reinterpret_cast<bf16x8_t *>(split_lds);
    char *const own = split_lds + kTableBytes + wave * kOwnBytes;
    const int steps = (a.C + kStepChannels - 1) / kStepChannels;
    bool weights_split = true;
    for (int s = 0; s < steps; s++) weights_split = weights_split && bad[s] == 0;
    const uint32_t plane = (uint32_t)(a.xsc * 4);
    // (a lane's place, formed anew where it is used: nothing of the addresses is kept over a row)
    struct Lane {
        uint32_t id, n, q;
    };
    auto fresh = [&]() {
        uint32_t id = (uint32_t)lane;
        asm volatile("" : "+v"(id));
        return Lane{id, id % 16, id / 16 % 4};
    };

    // an item: outputs [from, to) of a row, formed from the voxels [start, end)
    struct Item {
        int b, y, from, to, start, end;
        bool valid;
    };
    auto locate = [&](int it0) {
        Item p;
        p.valid = it0 < a.items;
        const int it = min(it0, a.items - 1), row = it / a.parts, part = it - row * a.parts;
        p.b = row / a.H;
        p.y = row - p.b * a.H;
        p.from = min(part * a.length, a.W);
        p.to = min(p.from + a.length, a.W);
        p.start = max(p.from - kHalo, 0);
        p.end = min(p.to + kHalo, a.W);
        return p;
    };
    // Loads: lane (channel q of four, voxels 4 n ..) of 64 voxels, which is what the matrix cores take: voxel 4 n + j is row n of product j.
    // Past the row end its last four voxels, past the last channel that one again (its weights are zero).
    f32x4_t xv[8];
    auto image_of = [&](const Item &p) { return reinterpret_cast<uint64_t>(x) + (uint64_t)(((int64_t)p.b * a.xsb + (int64_t)p.y * a.xsy) * 4); };
    auto request = [&](uint64_t image, int first, int step) {
        const Lane l = fresh();
        const uint32_t at = 4u * (uint32_t)min(first + 4 * (int)l.n, a.W - 4), lane_plane = l.q * plane;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = min(step * kStepChannels + 4 * i, a.C - 1);              // uniform
            uint64_t base = image + (uint64_t)c * (uint64_t)(a.xsc * 4);
            asm volatile("" : "+s"(base));
            float v[4];
            load_global_vec_unaligned<4>(base, min(lane_plane, (uint32_t)min(a.C - 1 - c, 3) * plane) + at, v);
            xv[i] = f32x4_t{v[0], v[1], v[2], v[3]};
        }
    };
    const bool resident = steps <= kTableSteps;   // the weights are in LDS once and for all
    auto load_weights = [&](int step, int count) {
#pragma unroll 2
        for (int i = wave * kWave + (int)fresh().id; i < count * kStepEntries; i += kPushWaves * kWave)
            weights[i] = table[((step + i / kStepEntries) * kSlabs + slab) * kStepEntries + i % kStepEntries];
    };
    if (resident) {
        load_weights(0, steps);
        __syncthreads();
    }
    // (workgroups whose table does not hold all weights meet at each part of it: all their waves take as many segments, of a row without
    // parts no more than it has)
    const int most = ((a.parts > 1 ? a.length + 2 * kHalo : a.W) + kWave - 1) / kWave;
    bool up;                                      // the segment's steps go up: the part of the table that one ends with is the next one's first
    int loaded = -1;
    const int stride = pairs * kPushWaves;
    int it = pair * kPushWaves + wave;
    Item here = locate(it);
    request(image_of(here), here.start, 0);
    for (int it0 = pair * kPushWaves; it0 < a.items; it0 += stride, it += stride) {
        const Item next = locate(it + stride);
        f32x4_t before[2][kTiles];                // the last 32 voxels of the segment before: of lanes 32 + i, products 0 and 1 in lane i, 2 and 3 in theirs
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int t = 0; t < kTiles; t++) before[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        up = true;
        const int segs = resident ? (here.end - here.start + kWave - 1) / kWave : most;
        for (int seg = 0; seg < segs; seg++) {
            const int first = here.start + seg * kWave;
            const bool real = here.valid && first < here.end;                      // uniform
            f32x4_t acc[4][kTiles];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int t = 0; t < kTiles; t++) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            float rest = 0.f;
            for (int i = 0; i < steps; i++) {
                const int step = up ? i : steps - 1 - i;
                if (!resident && step / kTableSteps != loaded) {                   // uniform over the workgroup
                    loaded = step / kTableSteps;
                    lds_sync();
                    load_weights(loaded * kTableSteps, min(kTableSteps, steps - loaded * kTableSteps));
                    lds_sync();
                }
                const auto [id, n, q] = fresh();
                // the lane at the row end has loaded voxels further left
                const int over = first + 4 * (int)n - (a.W - 4);
                if (first + kWave > a.W && (a.W - first) % 4 != 0) {               // uniform
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const f32x4_t v = xv[i];
                        xv[i][0] = over == 1 ? v[1] : over == 2 ? v[2] : over == 3 ? v[3] : v[0];
                        xv[i][1] = over == 1 ? v[2] : over == 2 ? v[3] : v[1];
                        xv[i][2] = over == 1 ? v[3] : v[2];
                    }
                }
                bf16x8_t xa[4][3];                // [voxels 4 n + j][part]: channels channel_of(q, ..)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    // -x at every second voxel: the sums of the bf16 instruction are cut off towards minus infinity
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = xv[e][j] * (j % 2 ? -kSplitScale : kSplitScale);
                    Split8 s;
                    rest += split8(v, s);
#pragma unroll
                    for (int p = 0; p < 3; p++) xa[j][p] = s.p[p];
                }
                __builtin_amdgcn_sched_barrier(0);    // (the scheduler would move the loads to where they are used)
                const bool more = i + 1 < steps, row = more || seg + 1 < segs;
                request(image_of(row ? here : next), more ? first : row ? first + kWave : next.start, more ? (up ? step + 1 : step - 1) : resident || !row ? 0 : step);
                __builtin_amdgcn_sched_barrier(0);
                if (real) {
                    const bf16x8_t *const wt = weights + (resident ? step : step % kTableSteps) * kStepEntries + id;
                    bf16x8_t w[2][3];
#pragma unroll
                    for (int p = 0; p < 3; p++) w[0][p] = wt[p * kWave];
#pragma unroll
                    for (int t = 0; t < kTiles; t++) {
                        if (t + 1 < kTiles) {
#pragma unroll
                            for (int p = 0; p < 3; p++) w[(t + 1) % 2][p] = wt[((t + 1) * 3 + p) * kWave];
                        }
                        f32x4_t one[4];               // (summed from zero and then added: the instruction cuts its sums off)
#pragma unroll
                        for (int k = 0; k < 6; k++)
#pragma unroll
                            for (int j = 0; j < 4; j++)
                                one[j] = mfma_split(xa[j], w[t % 2], k == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : one[j], k);
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[j][t] += (j % 2 ? -kSplitUnit : kSplitUnit) * one[j];
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            up = resident || !up;
            if (!real) continue;
            if (!weights_split || __any(taken_whole(rest))) {                      // uniform
                // values to be taken whole: all of the segment's sums again, with the fp32 instruction
                const float *const image = x + (int64_t)here.b * a.xsb + (int64_t)here.y * a.xsy;
#pragma unroll
                for (int t = 0; t < kTiles; t++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[j][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                    for (int c0 = 0; c0 < a.C; c0 += 4) {
                        const auto [id, n, q] = fresh();
                        const int c = c0 + (int)q, cc = min(c, a.C - 1), s = c0 / kStepChannels;   // (channel_of: step s, lanes q, value e)
                        const __bf16 *const k = reinterpret_cast<const __bf16 *>(table + ((int64_t)(s * kSlabs + slab) * kTiles + t) * (3 * kWave) + id) +
                                                c0 % kStepChannels / 4;
                        const float w = bad[s] != 0 ? whole_value(k[0], k[8 * kWave])              // uniform
                                                    : ((float)k[0] + (float)k[8 * kWave] + (float)k[16 * kWave]) * (1.f / kSplitScale);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float v = image[(int64_t)cc * a.xsc + min(first + 4 * (int)n + j, a.W - 1)];
                            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(c < a.C ? v : 0.f, c < a.C ? w : 0.f, acc[j][t], 0, 0, 0);
                        }
                    }
                }
            }

            // The shifts along x: the staged rows hold the voxels first - 32 .., the outputs are first - 16 .. (at the row end
            // all that are left, which is a second round of a few lanes).
            const auto [id, n, q] = fresh();
            float *const T = reinterpret_cast<float *>(own);
            const int zero = first - 2 * kHalo;       // voxel of the staged rows' first value
            const int rounds = first + kWave >= a.W && here.to > first + kWave - kHalo ? 2 : 1;
            const bool folds = first - 2 * kHalo < 0 || first + kWave + kHalo > a.W;                  // uniform
            const uint64_t zb = reinterpret_cast<uint64_t>(z + ((int64_t)here.b * 3 * a.out.n * a.H + here.y) * a.W);
            const int triples_in = 3 * min(max(a.out.n - slab * kSlabOut, 0), kSlabOut);
#pragma unroll
            for (int t = 0; t < kTiles; t++) {
                if (kTriples * t >= triples_in) break;                             // uniform
                // acc[j][t][r] = Y[16 q + 4 r + j][16 t + n]
                float *const put = T + n * kLine + (n == 15 ? t * kLine : 0);                        // (the last columns keep rows of their own)
                own_sync();                           // (the tile before has been read)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    typedef float f32x2_t __attribute__((ext_vector_type(2)));
                    *reinterpret_cast<f32x2_t *>(put + 16 * (q % 2) + 4 * r + 2 * (q / 2)) = f32x2_t{before[0][t][r], before[1][t][r]};
                    *reinterpret_cast<f32x4_t *>(put + 2 * kHalo + 16 * q + 4 * r) = f32x4_t{acc[0][t][r], acc[1][t][r], acc[2][t][r], acc[3][t][r]};
                }
                own_sync();
                constexpr int kMost = kTriples + 1;
                const int triples = t == kTiles - 1 ? kMost : kTriples;
                for (int round = 0; round < rounds; round++) {
                    const int xx = first - kHalo + round * kWave + (int)id;
                    if (round > 0 && id >= kHalo) break;
                    const bool store = xx >= here.from && xx < here.to;
                    const int xc = min(max(xx, 0), a.W - 1) - zero;
                    float sum[kMost][3];
#pragma unroll
                    for (int i = 0; i < kMost; i++) {
                        if (i >= triples) break;
                        const float *const r = T + 3 * i * kLine;
                        const int d = a.out.dil[min(slab * kSlabOut + (kTriples * t + i) / 3, a.out.n - 1)];
                        int lo = xc - d, hi = xc + d;
                        if (folds) {                  // fold(x - d), fold(x + d)
                            lo = max(lo, -1 - 2 * zero - lo);
                            hi = min(hi, 2 * (a.W - zero) - 1 - hi);
                        }
                        sum[i][0] = r[lo];
                        sum[i][1] = r[kLine + xc];
                        sum[i][2] = r[2 * kLine + hi];
                    }
#pragma unroll
                    for (int i = 0; i < kMost; i++) {
                        const int tri = kTriples * t + i;
                        if (i >= triples || tri >= triples_in) break;              // uniform
                        const float v[1] = {sum[i][0] + sum[i][1] + sum[i][2]};
                        if (store)
                            store_global_vec<1>(zb + (uint64_t)(3 * slab * kSlabOut + tri) * (uint64_t)((int64_t)a.H * a.W * 4),
                                                4u * (uint32_t)xx, v);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int t = 0; t < kTiles; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        before[j][t][r] = __uint_as_float(
                            __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[j][t][r]), __float_as_uint(acc[j + 2][t][r]), false, false)[1]);
        }
        here = next;
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
    // (channels in batches of at most seven: registers)
    constexpr int kBatch = NC <= 7 ? (NC > 0 ? NC : 1) : (NC + 1) / 2;
    float zv[WOUT][3][V], xv[kBatch][3][V];
#pragma unroll
    for (int co = 0; co < WOUT; co++)
#pragma unroll
        for (int ky = 0; ky < 3; ky++)
            load_vec<V>(sums.z + (int64_t)b * sums.zsb + ((int64_t)(3 * co + ky) * g.H + rows[ky]) * g.W + x0, zv[co][ky]);
    auto load = [&](int c0) {
#pragma unroll
        for (int c = 0; c < kBatch; c++)
#pragma unroll
            for (int ky = 0; ky < 3; ky++)
                if (c0 + c < NC) load_vec<V>(x.p + (int64_t)b * x.sb + (c0 + c) * x.sc + rows[ky] * x.sy + x0, xv[c][ky]);
    };
    load(0);

    float acc[WOUT][3][V];
#pragma unroll
    for (int co = 0; co < WOUT; co++)
#pragma unroll
        for (int i = 0; i < V; i++) {
            acc[co][0][i] = acc[co][2][i] = 0.f;
            acc[co][1][i] = bias[co] + (zv[co][0][i] + zv[co][1][i] + zv[co][2][i]);
        }
#pragma unroll
    for (int c0 = 0; c0 < NC; c0 += kBatch) {
        if (c0 > 0) {
            __builtin_amdgcn_sched_barrier(0);
            load(c0);
        }
#pragma unroll
        for (int co = 0; co < WOUT; co++)
#pragma unroll
            for (int c = 0; c < kBatch; c++)
#pragma unroll
                for (int ky = 0; ky < 3; ky++)
#pragma unroll
                    for (int r = 0; r < 3; r++) {
                        if (c0 + c >= NC) continue;
                        const float wv = k[co * sums.kco + (c0 + c) * kTaps + ky * 3 + r];
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
        case 7: return finish_launch<V, 7, 1>(g, x, k, bias, out, sums, s);
        case 8: return finish_launch<V, 8, 1>(g, x, k, bias, out, sums, s);
        case 9: return finish_launch<V, 9, 1>(g, x, k, bias, out, sums, s);
        case 10: return finish_launch<V, 10, 1>(g, x, k, bias, out, sums, s);
        case 11: return finish_launch<V, 11, 1>(g, x, k, bias, out, sums, s);
        case 12: return finish_launch<V, 12, 1>(g, x, k, bias, out, sums, s);
        case 13: return finish_launch<V, 13, 1>(g, x, k, bias, out, sums, s);
        }
    } else if (g.Wd == 2) {
        switch (g.C) {
        case 0: return finish_launch<V, 0, 2>(g, x, k, bias, out, sums, s);
        case 2: return finish_launch<V, 2, 2>(g, x, k, bias, out, sums, s);
        case 4: return finish_launch<V, 4, 2>(g, x, k, bias, out, sums, s);
        case 6: return finish_launch<V, 6, 2>(g, x, k, bias, out, sums, s);
        case 8: return finish_launch<V, 8, 2>(g, x, k, bias, out, sums, s);
        case 10: return finish_launch<V, 10, 2>(g, x, k, bias, out, sums, s);
        case 12: return finish_launch<V, 12, 2>(g, x, k, bias, out, sums, s);
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

bool group_split_supported_2d(int64_t W, int dmax) { return W >= 32 && dmax <= group2d::kHalo; }

int64_t group_table_floats_2d(int64_t channels)
{
    using namespace group2d;
    const int64_t steps = (channels + kStepChannels - 1) / kStepChannels;
    return steps * (kSlabs * kTiles * kTileBytes / 4) + (steps + 3) / 4 * 4;
}

hipError_t group_push_split_2d(const Geom &g, const View<const float> &x, const group2d::Outputs &out, float *z, float *table,
                               hipStream_t s)
{
    using namespace group2d;
    int dmax = 0;
    for (int o = 0; o < out.n; o++) dmax = std::max(dmax, out.dil[o]);
    if (out.n <= kSlabOut || out.n > kMaxOut || !group_push_supported_2d(g, x, dmax) || !group_split_supported_2d(g.W, dmax))
        return hipErrorInvalidValue;
    const int steps = (g.C + kStepChannels - 1) / kStepChannels;
    SplitArgs a{g.C, g.H, g.W, 0, 1, 0, x.sb, x.sc, x.sy, out};
    // Parts of a row: the waves that are resident take as few segments one after the other as can be.
    const int64_t rows = (int64_t)g.B * g.H, slots = 256 / kSlabs * kPushWaves;
    int64_t best = INT64_MAX;
    for (int parts = 1; parts <= 32; parts++) {
        const int length = ((g.W + parts - 1) / parts + 3) & ~3;
        if (parts > 1 && length < kWave) break;
        const int64_t cost = (rows * parts + slots - 1) / slots * ((std::min(g.W, length + (parts > 1 ? 2 * kHalo : 0)) + kWave - 1) / kWave);
        if (cost < best) {
            best = cost;
            a.parts = parts;
            a.length = length;
        }
    }
    a.items = (int)(rows * a.parts);
    const int blocks = kSlabs * (int)std::min<int64_t>(256 / kSlabs, xcd_grid((a.items + kPushWaves - 1) / kPushWaves));
    bf16x8_t *const weights = reinterpret_cast<bf16x8_t *>(table);
    int *const bad = reinterpret_cast<int *>(table + (int64_t)steps * (kSlabs * kTiles * kTileBytes / 4));
    hipLaunchKernelGGL(push_table, dim3(steps), dim3(kSlabs * kTiles * kWave), 0, s, a, weights, bad);
    static LargeLds large;
    const hipError_t e = large.allow(reinterpret_cast<const void *>(&push_split), kSplitLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(push_split, dim3(blocks), dim3(kPushWaves * kWave), kSplitLds, s, a, x.p, weights, bad, z);
    return hipGetLastError();
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
           ((g.Wd == 1 && g.C < group2d::kMaxOut) || (g.Wd == 2 && g.C < group2d::kMaxOut - 1 && g.C % 2 == 0));
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
