// pull_rows_wide: pull_rows (msd_pull.hip) with eight waves that all gather and then all
// multiply: two slabs over five to eight blocks of 16 channels, of which every wave has one, and one slab over three and four, of which
// every wave has half of one, in large images.
//
// A workgroup owns a tile of four segments of 32 voxels and the 128 rows m of two slabs, or of eight segments and one slab.  Each wave gathers a segment's A of
// one slab, splits it and leaves it in LDS; behind a barrier each wave takes its own block through both products, 64 voxels at a time.  Over fewer
// blocks waves would be idle in the products, and pull_rows is faster; over five to eight of two slabs the three kinds of waves of pull_rows
// would need two blocks each, for which there are no registers (1024 x 1024, 14 outputs over 87 channels: 430 us; three kinds of waves with two blocks and
// registers spilt 528; these eight waves with the gather and the products of pull_rows 442).
#pragma once

#include "msd_pull_common.h"

namespace msd {
namespace group2d {
namespace {

constexpr int kWaves = 8;                         // of a workgroup; one workgroup per compute unit

// LDS of a wave for a unit of voxels: 16 channels of x in three parts (the sums for grad_input take less)
constexpr int unit_bytes(int voxels) { return 3 * 16 * (2 * voxels + 16); }

// What a workgroup of pull_rows_wide keeps in LDS besides A and the waves' own space.
struct Source {                                   // an output's place in bytes: its dilation in slices, rows and voxels, its plane
    uint32_t slices, rows, voxels, plane;
};
struct WideShared {
    Source sources[kMaxOut];
    int bad_again, bad_tile[kWaves];
    f32x4_t bias_sums[kWaves * kWave];                // of the lanes' outputs at their voxels (not in registers: there are none left)
};

// G slabs of rows; P waves share a block of 16 channels (the tile's voxels in as many parts).
template <int G, int P> struct WideShape {
    static_assert(G * P == 2, "a block per wave and two slabs, or half a block and one");
    static constexpr int kSegs = kWaves / G;             // segments of a tile
    static constexpr int kSteps = 2 * G;                 // of 32 rows m
    static constexpr int kTiles = 4 * G;                 // of 16 rows m
    static constexpr int kUnit = 64;                     // voxels that a wave takes through the products at a time
    static constexpr int kUnits = kSegs * kSegment / P / kUnit;
    static constexpr int kVec = kUnit / 16;              // 16-byte accesses per lane for a unit of 16 channels
    static constexpr int kLanes = kUnit / 4;             // lanes of a channel in one of them
    static constexpr int kOwnBytes = unit_bytes(kUnit);
    static constexpr int kLds = kSegs * G * kSlabBytes + kWaves * kOwnBytes;
};

// What the kernel keeps for its life: the weights of rows 32 step + 8 q .. of channel n in parts, the sums of
// grad_kernel.
template <int G> struct WideState {
    bf16x8_t w[2 * G][3];
    bool weights_split;
    f32x4_t sums[4 * G];
};

// The tiles of a workgroup.  True where units were left out that hold values which cannot be split: the second
// run (WHOLE) takes these, with the fp32 instruction.  Apart, so that it keeps no registers in the first.
template <int N, int G, int P, bool FRESH, bool WHOLE>
__device__ __forceinline__ bool wide_tiles(const PullArgs &a, const float *__restrict__ x, const float *gy, float *gx, char *lds,
                                           WideShared &shared, int tid, int wave, int blocks, int c0, int wgs, int wg, WideState<G> &state)
{
    using S = WideShape<G, P>;
    constexpr int kSegs = S::kSegs, kSteps = S::kSteps, kTiles = S::kTiles, kUnit = S::kUnit, kUnits = S::kUnits, kVec = S::kVec;
    constexpr int kLanes = S::kLanes, kOwnBytes = S::kOwnBytes;
    constexpr int kTaps = Gather<N>::kTaps, kLines = Gather<N>::kLines, kLaneOut = Gather<N>::kLaneOut, kSlabOut = Gather<N>::kOutputs;
    const int lane = tid % kWave;
    const int cb = wave / P, ch0 = c0 + cb * 16;  // the wave's block
    const bool active = cb < blocks, update = ch0 < a.update;       // uniform
    char *const A = lds;
    char *const own = lds + kSegs * G * kSlabBytes + wave * kOwnBytes;
    bf16x8_t(&w)[kSteps][3] = state.w;
    f32x4_t(&sums)[kTiles] = state.sums;

    auto tile_of = [&](int tile) { return tile_at<kSegs>(a, tile); };
    auto locate = [&](const Tile &t, int segment) { return place_at<N>(a, t, segment); };
    const uint32_t plane = (uint32_t)a.sc * 4u;
    auto row_at = [&](int z, int y) { return (Gather<N>::kIsVolume ? z * (int)a.sz : 0) + y * (int)a.sy; };

    // The tiles: kSegs consecutive segments of an image each; every workgroup of an XCD works on neighbouring ones.
    const int lb = block_for_xcd(wg, wgs, wgs % kXcds == 0);

    // ---- x and grad_input of a unit: lane (channel lane / kLanes of kVec x .., four voxels lane % kLanes)
    const int lv = lane % kLanes, lc = lane / kLanes;               // voxels 4 lv .., channels lc + kRows4 i
    constexpr int kChannels = kWave / kLanes;     // channels of one access
    const uint32_t lane_plane = (uint32_t)lc * plane;
    auto unit_of = [&](const Tile &t, int u) {
        const int first = ((wave % P) * kUnits + u) * (kUnit / kSegment);
        const Place p0 = locate(t, first), p1 = locate(t, first + kUnit / kSegment - 1);
        const int sel = lv / (kSegment / 4), v4 = lv % (kSegment / 4) * 4;
        const uint32_t at0 = 4u * (uint32_t)(row_at(p0.z, p0.y) + p0.x0), at1 = 4u * (uint32_t)(row_at(p1.z, p1.y) + p1.x0);
        Unit un;
        un.img = t.img;
        un.at = (sel ? at1 : at0) + 4u * (uint32_t)v4;
        un.skip = min(max((sel ? p1.skip : p0.skip) - v4, 0), 4);
        return un;
    };
    auto request = [&](const float *from, int limit, const Unit &un, f32x4_t (&d)[kVec]) { request_unit(from, ch0, limit, plane, lane_plane, un, d); };
    f32x4_t xs[kVec], gs[kVec];
    auto request_g = [&](const Unit &un) {
        if constexpr (FRESH) {
#pragma unroll
            for (int i = 0; i < kVec; i++) gs[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        } else {
            request(gx, max(a.update, 1), un, gs);
        }
    };

    // ---- the gather: lane (v, h) takes its outputs at voxel v of the wave's segment, 36 (27) values for 32 rows
    // m.  Its loads are issued in the tile before, in front of that tile's last stores and requests (all of
    // them retire in order: behind those it would wait for memory).
    const int segment = wave / G, slab = wave % G;
    const int v = lane % kSegment, h = lane / kSegment;
    const uint32_t bias = 4u * (uint32_t)row_at(a.dmax, a.dmax);
    auto output_of = [&](int j) { return Gather<N>::kIsVolume ? h : j < 3 ? 3 * h + j : 6; };
    auto source = [&](int j) {
        int o = output_of(j);
        asm volatile("" : "+v"(o));
        return shared.sources[slab * kSlabOut + o];
    };
    // the lane's voxel (kImage, kVolume: y and z are uniform)
    struct Voxel {
        int x, y, z;
    };
    auto voxel_of = [&](const Place &p) {
        Voxel vx{p.x0 + v, p.y, p.z};
        if constexpr (N == kFlat) {
            const int row = a.by_voxels.of(vx.x);
            vx.x -= row * a.W;
            vx.z = a.by_rows.of(row);
            vx.y = row - vx.z * a.H;
        }
        return vx;
    };
    auto away = [&](const Place &p) {             // uniform: from all edges
        return N != kFlat && p.x0 >= a.dmax && p.x0 + kSegment + a.dmax <= a.W && p.y >= a.dmax && p.y + a.dmax < a.H &&
               (N == kImage || (p.z >= a.dmax && p.z + a.dmax < a.D));
    };
    float val[kLaneOut][kLines][3];
    auto gather = [&](const Tile &t, const Place &p) {
        if (away(p)) {
            const uint32_t u = (uint32_t)(p.x0 + v);
            const uint64_t base = reinterpret_cast<uint64_t>(gy) + (uint64_t)(t.gimg + (int64_t)row_at(p.z, p.y) * 4) - bias;
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const Source o = source(j);
                const uint32_t c = o.plane + bias + 4u * u;
#pragma unroll
                for (int l = 0; l < kLines; l++) {
                    const uint32_t s = N == kImage || l / 3 == 1 ? c : l / 3 == 0 ? c + o.slices : c - o.slices;
                    const uint32_t r = l % 3 == 0 ? s + o.rows : l % 3 == 1 ? s : s - o.rows;
                    val[j][l][0] = load1(base, r + o.voxels);
                    val[j][l][1] = load1(base, r);
                    val[j][l][2] = load1(base, r - o.voxels);
                }
                __builtin_amdgcn_sched_barrier(0);    // (an output's addresses at a time: registers)
            }
        } else {
            const uint64_t base = reinterpret_cast<uint64_t>(gy) + (uint64_t)t.gimg;
            const Voxel vx = voxel_of(p);
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const Source o = source(j);
                const int d = (int)(o.voxels / 4u);
                const Sides sx = sides(vx.x, a.W, d), sy = sides(vx.y, a.H, d), sz = sides(vx.z, N == kImage ? 1 : a.D, N == kImage ? 0 : d);
#pragma unroll
                for (int l = 0; l < kLines; l++) {
                    const int y = l % 3 == 0 ? sy.up : l % 3 == 1 ? vx.y : sy.down;
                    const int z = N == kImage || l / 3 == 1 ? vx.z : l / 3 == 0 ? sz.up : sz.down;
                    const uint32_t r = o.plane + 4u * (uint32_t)row_at(z, y);
                    val[j][l][0] = load1(base, r + 4u * (uint32_t)sx.up);
                    val[j][l][1] = load1(base, r + 4u * (uint32_t)vx.x);
                    val[j][l][2] = load1(base, r + 4u * (uint32_t)sx.down);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // round: number of the tile among the workgroup's, below 0 where its biases have been counted
    auto gathered = [&](const Place &p, int round) {
        if (!away(p)) {
            const Voxel vx = voxel_of(p);
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const int d = (int)(source(j).voxels / 4u);
                const Sides sx = sides(vx.x, a.W, d), sy = sides(vx.y, a.H, d), sz = sides(vx.z, N == kImage ? 1 : a.D, N == kImage ? 0 : d);
#pragma unroll
                for (int l = 0; l < kLines; l++) fold(sx, val[j][l][0], val[j][l][2]);
#pragma unroll
                for (int l = 0; l < kLines; l += 3)
#pragma unroll
                    for (int r = 0; r < 3; r++) fold(sy, val[j][l][r], val[j][l + 2][r]);
                if constexpr (N != kImage) {
#pragma unroll
                    for (int l = 0; l < 3; l++)
#pragma unroll
                        for (int r = 0; r < 3; r++) fold(sz, val[j][l][r], val[j][l + 6][r]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (p.skip > 0 || a.out.n < G * kSlabOut) {                 // uniform
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const bool ok = v >= p.skip && slab * kSlabOut + output_of(j) < a.out.n;
#pragma unroll
                for (int t = 0; t < kTaps; t++) val[j][t / 3][t % 3] = ok ? val[j][t / 3][t % 3] : 0.f;
            }
        }
        if (round >= 0) {
            // (volumes: one value per lane, four chains of a quarter of the tiles)
            if constexpr (N != kImage) reinterpret_cast<float *>(&shared.bias_sums[tid])[round % 4] += val[0][4 * (kLines / 9)][1];
            else shared.bias_sums[tid] += f32x4_t{val[0][1][1], val[1][1][1], val[2][1][1], val[3][1][1]};
        }
        // -A at every second voxel: the sums of the bf16 instruction are cut off towards minus infinity, which adds up
        // over an image where the gradients themselves cancel (bias gradients: an error of 2e-6 instead of 1.2e-7).
        // For the same reason x changes its sign with the voxel and from tile to tile.
        const float factor = (v % 2 ? -1.f : 1.f) * (WHOLE ? 1.f : kSplitScale);
#pragma unroll
        for (int j = 0; j < kLaneOut; j++)
#pragma unroll
            for (int t = 0; t < kTaps; t++) val[j][t / 3][t % 3] *= factor;
        char *const at = A + (segment * G + slab) * kSlabBytes + v * kVoxelBytes;
        const uint32_t piece = 16 * (4 * (uint32_t)h ^ turn((uint32_t)v));
        float bad = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float e8[8];
            eight_rows<N>(val, h, i, e8);
            Split8 s;
            if constexpr (WHOLE) {
                float scaled[8];
#pragma unroll
                for (int e = 0; e < 8; e++) scaled[e] = e8[e] * kSplitScale;
                bad += split8(scaled, s);
                put_whole(e8, s);
            } else {
                bad += split8(e8, s);
            }
#pragma unroll
            for (int k = 0; k < 3; k++) *reinterpret_cast<bf16x8_t *>(at + k * kPartBytes + (piece ^ 16 * i)) = s.p[k];
        }
        const bool any = __any(taken_whole(bad));
        if (lane == 0) shared.bad_tile[wave] = any;
    };

    // ---- the products of a unit.  The wave's own space holds x as [part][channel][voxel], then what is added to
    // grad_input as [channel][voxel]: loads and stores go by channel in whole lines, the matrix cores take 16
    // channels at once (loaded in that form, 64 bytes of 16 channels at a time, memory gives 2.6 to 3.0 TB/s instead of 4).
    constexpr int kXRow = 2 * kUnit + 16, kDRow = 4 * kUnit + 16;   // bytes of a channel (16 apart in the banks)
    const int first_seg = (wave % P) * kUnits * (kUnit / kSegment); // of the wave's first unit
    // bit 4 i + e: the channel's gradient at voxel e is kept
    auto mask_of = [&]() {
        uint32_t bits = 0xffffu;
        if (ch0 + 16 > a.mask_from) {             // uniform
            bits = 0;
#pragma unroll
            for (int i = 0; i < kVec; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    bits |= ch0 + lc + kChannels * i < a.mask_from || 0.f < xs[i][e] ? 1u << (4 * i + e) : 0u;
        }
        return bits;
    };
    // x in parts to the wave's own space; not finite where a value cannot be split
    // (factors for the even and the odd voxels, in registers of their own: a sign in the instruction doubles its size)
    struct Factors {
        uint32_t even, odd;
        __device__ explicit Factors(float f, uint32_t sign = 0) : even(__float_as_uint(f) | sign), odd(even ^ 0x80000000u)
        {
            asm volatile("" : "+s"(even), "+s"(odd));
        }
        __device__ float of(int e) const { return __uint_as_float(e % 2 ? odd : even); }
    };
    auto put_x = [&](uint32_t sign_bit) {
        const Factors factor(kSplitScale, sign_bit);
        float rest = 0.f;
#pragma unroll
        for (int i = 0; i < kVec; i += 2) {
            float x8[8];
#pragma unroll
            for (int e = 0; e < 8; e++) x8[e] = xs[i + e / 4][e % 4] * factor.of(e);
            Split8 s;
            rest += split8(x8, s);
            typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
            for (int p = 0; p < 3; p++) {
                char *const at = own + (p * 16 + lc + kChannels * i) * kXRow + 8 * lv;
                *reinterpret_cast<bf16x4_t *>(at) = __builtin_shufflevector(s.p[p], s.p[p], 0, 1, 2, 3);
                *reinterpret_cast<bf16x4_t *>(at + kChannels * kXRow) = __builtin_shufflevector(s.p[p], s.p[p], 4, 5, 6, 7);
            }
        }
        return rest;
    };
    // what the wave's own space holds for grad_input, in units of `unit`, added to it and masked
    auto add_d = [&](uint32_t bits, const Factors unit) {
#pragma unroll
        for (int i = 0; i < kVec; i++) {
            const f32x4_t d = *reinterpret_cast<const f32x4_t *>(own + (lc + kChannels * i) * kDRow + 16 * lv);
#pragma unroll
            for (int e = 0; e < 4; e++) gs[i][e] = __builtin_fmaf(d[e], unit.of(e), gs[i][e]);
        }
        if (ch0 + 16 > a.mask_from) {             // uniform
#pragma unroll
            for (int i = 0; i < kVec; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) gs[i][e] = bits & 1u << (4 * i + e) ? gs[i][e] : 0.f;
        }
    };
    constexpr int kK = kUnit / 32;                // steps of 32 voxels: the segments of the unit
    // False where a value cannot be split (and nothing is computed).
    auto compute = [&](int u, bool split, uint32_t sign_bit, const Unit &un, const Unit &next) {
        uint32_t ll = (uint32_t)lane;
        if (G > 1) asm volatile("" : "+v"(ll));                     // (no LDS addresses are kept over the tiles: registers)
        const uint32_t nn = ll % 16, qq = ll / 16 % 4;
        const char *const Au = A + (first_seg + u * kK) * G * kSlabBytes;
        // rows 16 t + n, voxels 8 q .. of segment j (the lane's address is that of voxel 8 q + n / 4 (+ 4), rows
        // 4 (n % 4) .., which the read transposes)
        const uint32_t tr_voxel = 8 * qq + nn / 4;
        const char *const tr = Au + tr_voxel * kVoxelBytes + nn % 2 * 8;
        const uint32_t tr_piece = 16 * (nn % 4 / 2 ^ turn(tr_voxel)), tr_next = 16 * (nn % 4 / 2 ^ turn(tr_voxel + 4));
        auto read_rows = [&](int j, int t, bf16x8_t(&to)[3]) {
            typedef short s16x4_t __attribute__((ext_vector_type(4)));
            typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
            typedef __attribute__((address_space(3))) s16x4_t *lds_tr_t;
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const char *const at = tr + (j * G + t / 4) * kSlabBytes + p * kPartBytes;
                const bf16x4_t lo = __builtin_bit_cast(
                    bf16x4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + (tr_piece ^ (uint32_t)(t % 4 * 32)))));
                const bf16x4_t hi = __builtin_bit_cast(
                    bf16x4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + 4 * kVoxelBytes + (tr_next ^ (uint32_t)(t % 4 * 32)))));
                to[p] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        // voxels 16 s + n of the unit, rows 32 i + 8 q ..
        const char *const vox = Au + nn * kVoxelBytes;
        const uint32_t vox_piece = 16 * (qq ^ turn(nn));
        auto read_voxels = [&](int s, int i, bf16x8_t(&to)[3]) {
#pragma unroll
            for (int p = 0; p < 3; p++)
                to[p] = *reinterpret_cast<const bf16x8_t *>(vox + (s / 2 * G + i / 2) * kSlabBytes + p * kPartBytes +
                                                            s % 2 * 16 * kVoxelBytes + (vox_piece ^ (uint32_t)(i % 2 * 64)));
        };
        clear_skipped(un, xs);
        const uint32_t bits = mask_of();
        const float rest = put_x(sign_bit);
        const bool done = split && !__any(taken_whole(rest));       // uniform
        __builtin_amdgcn_sched_barrier(0);        // (the scheduler would move the loads to where they are used)
        request(x, a.C, next, xs);
        __builtin_amdgcn_sched_barrier(0);
        if (!done) return false;
        own_sync();
        // Both products in stages of two chains of six matrix instructions, whose operands are read from LDS a
        // stage ahead (where there are registers for it).
        constexpr bool kAhead = G == 1;
        bf16x8_t op[2][2][3], xp[kK][3];
        constexpr int kRowStages = kTiles * kK / 2, kVoxelStages = kSteps * kK;
        // stage r: tiles 2 (r / kK) and the next at segment r % kK
        auto stage_rows = [&](int r, bf16x8_t(&to)[2][3]) {
#pragma unroll
            for (int o = 0; o < 2; o++) read_rows(r % kK, r / kK * 2 + o, to[o]);
        };
        // stage r: step r % kSteps at the voxels of segment r / kSteps
        auto stage_voxels = [&](int r, bf16x8_t(&to)[2][3]) {
#pragma unroll
            for (int s = 0; s < 2; s++) read_voxels(r / kSteps * 2 + s, r % kSteps, to[s]);
        };
        f32x4_t acc[2];
        bf16x8_t high[2];
        stage_rows(0, op[0]);
#pragma unroll
        for (int j = 0; j < kK; j++)
#pragma unroll
            for (int p = 0; p < 3; p++)
                xp[j][p] = *reinterpret_cast<const bf16x8_t *>(own + (p * 16 + nn) * kXRow + (32 * j + 8 * qq) * 2);
#pragma unroll
        for (int r = 0; r < kRowStages; r++) {
            if (!kAhead && r > 0) stage_rows(r, op[r % 2]);
            if (kAhead && r + 1 < kRowStages) stage_rows(r + 1, op[(r + 1) % 2]);
            if (kAhead && r + 1 == kRowStages) stage_voxels(0, op[(r + 1) % 2]);
            __builtin_amdgcn_sched_barrier(0);
            // (the products of the high parts of both segments last: each instruction cuts its sum off at the size
            // that it has reached)
#pragma unroll
            for (int k = 0; k < 5; k++)
#pragma unroll
                for (int o = 0; o < 2; o++)
                    acc[o] = mfma_split(op[r % 2][o], xp[r % kK], k == 0 && r % kK == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : acc[o], k);
            if (r % kK == kK - 1) {
#pragma unroll
                for (int j = 0; j < kK; j++)
#pragma unroll
                    for (int o = 0; o < 2; o++)
                        acc[o] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(j == kK - 1 ? op[r % 2][o][0] : high[o], xp[j][0], acc[o], 0, 0, 0);
            } else {
#pragma unroll
                for (int o = 0; o < 2; o++) high[o] = op[r % 2][o][0];
            }
            if (r % kK == kK - 1) {
#pragma unroll
                for (int o = 0; o < 2; o++) {
                    sums[r / kK * 2 + o] += __uint_as_float(__float_as_uint(kSplitUnit) | sign_bit) * acc[o];
                    asm volatile("" : "+v"(sums[r / kK * 2 + o]));  // (here and not at the end of the tile: registers)
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (update) {                             // uniform
            // (x has been read: the wave's space is free for the sums)
            f32x4_t d[2], all[2];
#pragma unroll
            for (int r = 0; r < kVoxelStages; r++) {
                const int i = r % kSteps;
                if (!kAhead) stage_voxels(r, op[(kRowStages + r) % 2]);
                if (kAhead && r + 1 < kVoxelStages) stage_voxels(r + 1, op[(kRowStages + r + 1) % 2]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 5; k++)
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        d[s] = mfma_split(op[(kRowStages + r) % 2][s], w[i], k == 0 && i % 2 == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : d[s], k);
                if (i % 2 == 0) {
#pragma unroll
                    for (int s = 0; s < 2; s++) high[s] = op[(kRowStages + r) % 2][s][0];
                } else {
#pragma unroll
                    for (int j = 0; j < 2; j++)
#pragma unroll
                        for (int s = 0; s < 2; s++)
                            d[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(j ? op[(kRowStages + r) % 2][s][0] : high[s], w[i - 1 + j][0], d[s], 0, 0, 0);
                }
                // Summed slab by slab from zero and added to grad_input last: a chain of products that started from it
                // would round each of them to its size.
                if (i % 2 == 1) {
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        all[s] = i == 1 ? d[s] : all[s] + d[s];
                        if (i == kSteps - 1)
                            *reinterpret_cast<f32x4_t *>(own + nn * kDRow + (16 * (r / kSteps * 2 + s) + 4 * qq) * 4) = all[s];
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            own_sync();
            add_d(bits, Factors(kSplitUnit));
            own_sync();
        }
        return true;
    };
    // The same with the fp32 instruction, for values that cannot be split among x, A or the weights (A and the weights
    // lie whole in the place of their parts).
    auto compute_whole = [&](int u, uint32_t sign_bit, const Unit &un) {
        const float sign = __uint_as_float(sign_bit | 0x3f800000u);
        clear_skipped(un, xs);
        const uint32_t bits = mask_of();
        uint32_t ll = (uint32_t)lane;
        asm volatile("" : "+v"(ll));
        const uint32_t nn = ll % 16, qq = ll / 16 % 4;
        const char *const Au = A + (first_seg + u * kK) * G * kSlabBytes;
        auto value = [&](uint32_t voxel, uint32_t m) {
            const char *const at = Au + (voxel / kSegment * G + m / kRows) * kSlabBytes + voxel % kSegment * kVoxelBytes +
                                   16 * (m % kRows / 8 ^ turn(voxel)) + m % 8 * 2;
            return whole_value(*reinterpret_cast<const __bf16 *>(at), *reinterpret_cast<const __bf16 *>(at + kPartBytes));
        };
        own_sync();
#pragma unroll
        for (int i = 0; i < kVec; i++)
            *reinterpret_cast<f32x4_t *>(own + (lc + kChannels * i) * kDRow + 16 * lv) =
                xs[i] * f32x4_t{sign, -sign, sign, -sign};
        own_sync();
#pragma unroll
        for (int t = 0; t < kTiles; t++)
#pragma unroll
            for (int j = 0; j < kK; j++) {
                f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (int e = 0; e < 8; e++) {
                    const uint32_t voxel = 32 * j + 8 * qq + (uint32_t)e;
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(value(voxel, 16 * t + nn),
                                                               *reinterpret_cast<const float *>(own + nn * kDRow + 4 * voxel), acc, 0, 0, 0);
                }
                sums[t] += sign * acc;
            }
        if (update) {
            own_sync();
#pragma unroll 1
            for (int s = 0; s < kUnit / 16; s++) {
                f32x4_t all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < kSteps; i++) {
                    f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        d = __builtin_amdgcn_mfma_f32_16x16x4f32(value(16 * s + nn, 32 * i + 8 * qq + e),
                                                                 whole_value(w[i][0][e], w[i][1][e]), d, 0, 0, 0);
                    }
                    all += d;
                }
                *reinterpret_cast<f32x4_t *>(own + nn * kDRow + (16 * s + 4 * qq) * 4) = all;
            }
            own_sync();
            add_d(bits, Factors(1.f));
        }
        own_sync();
    };
    auto store = [&](const Unit &un, bool all) { store_unit(gx, ch0, a.update, plane, lane_plane, lc, un, gs, all); };
    // values of the tile at hand that can be split: A and the weights
    auto tile_split = [&]() {
        int bad = 0;
#pragma unroll
        for (int i = 0; i < kWaves; i++) bad |= shared.bad_tile[i];
        return state.weights_split && __builtin_amdgcn_readfirstlane(bad) == 0;
    };

    if constexpr (WHOLE) {
#pragma unroll 1
        for (int tile = lb; tile < a.tiles; tile += wgs) {
            const Tile t = tile_of(tile);
            const Place here = locate(t, segment);
            gather(t, here);
            gathered(here, -1);
            __syncthreads();
            if (active) {
                const bool split = tile_split();
#pragma unroll 1
                for (int u = 0; u < kUnits; u++) {
                    const Unit un = unit_of(t, u);
                    request(x, a.C, un, xs);
                    request_g(un);
                    clear_skipped(un, xs);
                    const float rest = put_x(t.sign);
                    if (split && !__any(taken_whole(rest))) continue;    // (the first run has done it)
                    compute_whole(u, t.sign, un);
                    store(un, true);
                }
            }
            __syncthreads();
        }
        return false;
    } else {
        Tile now = tile_of(lb);
        Unit un = unit_of(now, 0);
        request(x, a.C, un, xs);
        request_g(un);
        bool again = false;                       // units were left to the second run
        Place here = locate(now, segment);
        gather(now, here);
        int round = 0;
        for (int tile = lb; tile < a.tiles; tile += wgs) {          // uniform over the workgroup
            gathered(here, round++);
            lds_sync();
            const Tile then = tile_of(tile + wgs);
            here = locate(then, segment);
            if (active) {
                const bool split = tile_split();
#pragma unroll
                for (int u = 0; u < kUnits; u++) {
                    const Unit next = u + 1 < kUnits ? unit_of(now, u + 1) : unit_of(then, 0);
                    const bool done = compute(u, split, now.sign, un, next);
                    again = again || !done;
                    if (u + 1 == kUnits) gather(then, here);
                    store(un, done);
                    __builtin_amdgcn_sched_barrier(0);
                    request_g(next);
                    __builtin_amdgcn_sched_barrier(0);
                    un = next;
                }
            } else {
                gather(then, here);
            }
            now = then;
            lds_sync();
        }
        return again;
    }
}

// FRESH: grad_input is written, not added to.
template <int N, int G, int P, bool FRESH = false>
__global__ __launch_bounds__(kWaves *kWave, 2) void pull_rows_wide(const PullArgs a, const float *__restrict__ x, const float *gy,
                                                             float *gx, float *__restrict__ part, float *__restrict__ bias_part)
{
    constexpr int kSegs = WideShape<G, P>::kSegs, kTiles = WideShape<G, P>::kTiles;
    constexpr int kTaps = Gather<N>::kTaps, kLaneOut = Gather<N>::kLaneOut, kSlabOut = Gather<N>::kOutputs;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int n = lane % 16, q = lane / 16;
    const int bid = blockIdx.x, big = a.chunks.large * a.chunks.wgs;
    const int chunk = bid < big ? bid / a.chunks.wgs : a.chunks.large + (bid - big) / a.chunks.wgs_small;
    const int blocks = a.chunks.size(chunk), c0 = a.chunks.first_block(chunk) * 16;
    const int wgs = a.chunks.rows(chunk), wg = bid - a.chunks.first_wg(chunk);
    const int cb = wave / P, ch0 = c0 + cb * 16;  // the wave's block
    __shared__ WideShared shared;
    WideState<G> state;

    if (tid == 0) shared.bad_again = 0;
    if (tid < G * kSlabOut) {
        const int o = min(tid, a.out.n - 1), d = a.out.dil[o];
        shared.sources[tid] = Source{N == kVolume ? 4u * (uint32_t)(d * (int)a.sz) : 0u, 4u * (uint32_t)(d * (int)a.sy), 4u * (uint32_t)d, (uint32_t)o * ((uint32_t)a.gsc * 4u)};
    }
    auto load_weights = [&](bool whole) {
        int ch = ch0 + n, qq = q;
        if (whole) asm volatile("" : "+v"(ch), "+v"(qq));       // (nothing of the first call is kept for the second)
#pragma unroll
        for (int step = 0; step < 2 * G; step++) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const Slot m = slot_of<N>(32 * step + 8 * qq + i);
                const bool ok = m.tap >= 0 && m.output < a.out.n && ch < a.update;
                const float k = a.out.k[ok ? m.output : 0][ok ? (int64_t)ch * kTaps + m.tap : 0];
                v[i] = (ok ? k : 0.f) * (whole ? 1.f : kSplitScale);
            }
            Split8 s;
            if (whole) put_whole(v, s);
            else if (__any(taken_whole(split8(v, s)))) state.weights_split = false;
#pragma unroll
            for (int p = 0; p < 3; p++) state.w[step][p] = s.p[p];
        }
    };
    state.weights_split = true;
    load_weights(false);
    __syncthreads();

    float *const row = part + (int64_t)bid * (a.chunks.blocks * 1024 * G);
#pragma unroll
    for (int t = 0; t < kTiles; t++) state.sums[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    shared.bias_sums[tid] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const bool again = wide_tiles<N, G, P, FRESH, false>(a, x, gy, gx, lds, shared, tid, wave, blocks, c0, wgs, wg, state);
    if (lane == 0 && again) shared.bad_again = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(shared.bad_again) != 0) {    // uniform over the workgroup
        int tid2 = tid;
        asm volatile("" : "+v"(tid2));           // (nothing of the first run is kept for the second)
        load_weights(true);
        wide_tiles<N, G, P, FRESH, true>(a, x, gy, gx, lds, shared, tid2, wave, blocks, c0, wgs, wg, state);
    }

    // the sums, of the waves that share a block through LDS
    constexpr int kBlock = 1024 * G;              // sums of a block of channels
    if constexpr (P == 1) {
        if (cb < blocks) {
#pragma unroll
            for (int t = 0; t < kTiles; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) row[cb * kBlock + (t * 4 + r) * kWave + lane] = state.sums[t][r];
        }
    } else {
        float *const red = reinterpret_cast<float *>(lds);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kTiles; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[wave * kBlock + (t * 4 + r) * kWave + lane] = state.sums[t][r];
        __syncthreads();
        for (int i = tid; i < kWaves / P * kBlock; i += kWaves * kWave) {
            const int b = i / kBlock;
            const float *const r = red + b * P * kBlock + i % kBlock;
            if (b < blocks) row[i] = r[0] + r[kBlock];
        }
    }
    if (chunk != 0) return;
    const int v = lane % kSegment, h = lane / kSegment;
    // the bias gradients: the centre taps, over the lanes' voxels and the segments
    f32x4_t bias_sum = shared.bias_sums[tid];
    if constexpr (N != kImage) bias_sum[0] = (bias_sum[0] + bias_sum[1]) + (bias_sum[2] + bias_sum[3]);
#pragma unroll
    for (int j = 0; j < kLaneOut; j++)
#pragma unroll
        for (int off = kSegment / 2; off > 0; off >>= 1) bias_sum[j] += __shfl_down(bias_sum[j], off, kSegment);
    float *const red = reinterpret_cast<float *>(lds);
    __syncthreads();
    if (v == 0) {
#pragma unroll
        for (int j = 0; j < kLaneOut; j++)
            if (N != kImage || j < 3 || h == 0) red[wave * kBiasColumns + (N != kImage ? h : j < 3 ? 3 * h + j : 6)] = bias_sum[j];
    }
    __syncthreads();
    if (tid < G * kBiasColumns && tid % kBiasColumns < kSlabOut) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < kSegs; i++) s += red[i * G * kBiasColumns + tid];
        bias_part[wg * (G * kBiasColumns) + tid] = s;
    }
}

}  // namespace
}  // namespace group2d
}  // namespace msd
