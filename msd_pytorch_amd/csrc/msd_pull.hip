// Backward pass of a group of layers over the channels they share (msd_group.h).
//
// With A[m][v], m = (output o, tap t), the adjoint-form gather of the masked output gradients at
// voxel v, both gradients are matrix products with the same matrix:
//     grad_input[c][v]  += sum_m k[m][c] * A[m][v],
//     grad_kernel[c][m] += sum_v x[c][v] * A[m][v].
// fp32 values are taken in three bf16 parts and six products (msd_split.h).  A workgroup owns a tile of two segments of 32 voxels
// and the 128 rows m of two slabs (four segments where a group has at most seven outputs: one slab).  Four waves gather A
// (each half a slab at the voxels of two segments, so that the outputs are the wave's own and a tap away from the edges is a scalar
// address), split it and leave it in LDS as [part][voxel][m]: the grad_input product reads it as it lies (lane = voxel, eight
// rows m), the grad_kernel product through the transposing LDS read (ds_read_b64_tr_b16).  At the same time four waves take the
// tile before, which lies in a second buffer, through the one and four through the other product, a block of 16 channels at 32 voxels at a time; a
// barrier per tile, and the buffers change.  Weights and sums stay in registers over the tiles, the sums go to a second level in LDS
// every 16 additions, and leave as one row of partial sums per workgroup, which sum_group adds in double precision.  x and grad_input go through a transposition in the wave's own part of LDS:
// in the layout of the matrix cores a load touches 64 bytes of each of 16 channels, which memory
// serves at 2.6-3.0 TB/s whatever else happens, whole lines at 4.0 (probed with loads and
// stores alone, 64 channels of 1024 x 1024).  Five to eight blocks of two slabs, and three and four of one slab in large images: msd_pull_wide.h.
//
// Bound by waiting and issue together, not by one pipe.  Counters at 1024 x 1024, 14 outputs with 28 / 33 / 58 channels in the pass, and at 128^3, four with 17 / 33 / 49: the
// matrix cores are busy 21 / 24 / 31 and 23 / 27 / 36 % of the time, vector instructions take 44 / 37 / 41 and 49 / 43 / 48 % of the SIMDs' cycles (at four
// each), and waves spend 42 / 57 / 44 and 39 / 54 / 40 % of theirs waiting for loads, LDS and the barrier and 28 / 19 / 30 and 31 / 20 / 31 % for a turn to issue; eight waves that
// all gathered and then all multiplied: matrix cores 19 / 26 / 30 and 21 / 26 / 32 %.  (Loads requested two and four units ahead, and gathered two tiles
// ahead, change nothing.)  us, eight waves -> three kinds: 61 x 93 x 75, four outputs, 8 channels 62 -> 54; 128^3, four with 17 / 33 / 49 325 / 440 / 501 -> 299 / 426 /
// 455; 3 x 333 x 477, 14 with 32 92 -> 82; 1024 x 1024, 14 with 17 / 28 / 33 / 58 167 / 169 / 220 / 263 -> 157 / 159 / 228 / 258.
//
// Tried on the way: waves that walk the channels on their own tile (weights in LDS, loads in the matrix layout): 650 us
// over 95 channels, 320 over 45; two workgroups of four waves per compute unit: 604 and 293; for 5 to 8 blocks
// two chunks of at most 4: 588.  Any register spilt in the loop costs 10 % (its reload waits for all loads and stores).
// Of the kinds: four waves that gather and four that do both products (128^3 over 14: 310), two teams that gather in turn (354), priorities by
// kind (no gain), the next tile's loads spread among the split (271 for 250).
#include "msd_pull_common.h"
#include "msd_pull_wide.h"

#include <algorithm>

namespace msd {
namespace group2d {
namespace {

// Bytes of a channel of a segment in a worker's own part of LDS: of x in one of its parts, of what is added to grad_input (16 apart in
// the banks).
constexpr int kXRow = 2 * kSegment + 16, kDRow = 4 * kSegment + 16;
constexpr int kVec = 2, kLanes = kSegment / 4;    // 16-byte accesses per lane for a segment of 16 channels; lanes of a channel in one of them

// The same with masks of bits: `and` and `add` of registers issue in half the cycles of a select.
struct SideMasks {
    uint32_t up, down, no_up, no_down;            // all bits where the source lies inside; where it does not
    __device__ SideMasks(int u, int n, int d) : up(u + d < n ? ~0u : 0u), down(u >= d ? ~0u : 0u), no_up(~up), no_down(~down)
    {
        asm("" : "+v"(up), "+v"(down), "+v"(no_up), "+v"(no_down));                // (or they are selects again)
    }
};
__device__ __forceinline__ float masked(float v, uint32_t bits) { return __uint_as_float(__float_as_uint(v) & bits); }
__device__ __forceinline__ void fold(const SideMasks &s, float &tap0, float &tap2)
{
    const float up = tap0, down = tap2;
    tap0 = masked(up, s.up) + masked(down, s.no_down);
    tap2 = masked(down, s.down) + masked(up, s.no_up);
}

// What a workgroup of pull_rows keeps in LDS besides A and the waves' own space.
struct PullShared {
    int bad_again, bad_tile[2][4];                // (of a tile of A, by the waves that gather it)
};

// G slabs of rows.  A workgroup is three kinds of four waves, one of each kind per SIMD: gatherers, which form A of a tile,
// and those that take the tile before through the one and through the other product: kernel workers (grad_kernel) and input workers
// (grad_input).  A is there twice.  P workers of a kind share a block of 16 channels (the tile's voxels in as many parts).
enum Kind { kGatherer, kKernel, kInput };
constexpr int kOfKind = 4;                        // waves
constexpr int kPullThreads = 3 * kOfKind * kWave;
template <int G, int P> struct PullShape {
    static constexpr int kSegs = kOfKind / G;            // segments of a tile
    static constexpr int kSteps = 2 * G;                 // of 32 rows m
    static constexpr int kTiles = 4 * G;                 // of 16 rows m
    static constexpr int kUnits = kSegs / P;             // segments that a worker takes one after the other
    static constexpr int kTileBytes = kSegs * G * kSlabBytes;
    static constexpr int kXBytes = 16 * 3 * kXRow, kDBytes = 16 * kDRow;           // of a kernel, an input worker's own
    static constexpr int kSumBytes = kTiles * kWave * 16;           // of a kernel worker's sums
    static constexpr int kSumsAt = 2 * kTileBytes + kOfKind * (kXBytes + kDBytes);
    static constexpr int kLds = kSumsAt + kOfKind * kSumBytes;
};

// What a wave keeps for its life: an input worker the weights of rows 32 step + 8 q .. of channel n in parts, a kernel worker its sums
// of grad_kernel, a gatherer the sums of its outputs at its voxels (volumes: of one output, every fourth tile).  In the same registers:
// what is declared is kept by all three.
template <int G> struct PullState {
    f32x4_t kept[2 * G * 3];
    bool weights_split;
    __device__ f32x4_t &sums(int tile) { return kept[tile]; }
    __device__ f32x4_t &bias(int level) { return kept[level]; }
    __device__ bf16x8_t weights(int step, int part) const { return __builtin_bit_cast(bf16x8_t, kept[step * 3 + part]); }
    __device__ void set_weights(int step, int part, bf16x8_t w) { kept[step * 3 + part] = __builtin_bit_cast(f32x4_t, w); }
};

// The tiles of a workgroup.  True where units were left out that hold values which cannot be split: the second
// run (WHOLE) takes these, with the fp32 instruction.  Apart, so that it keeps no registers in the first.
template <int N, int G, int P, bool FRESH, bool WHOLE>
__device__ __forceinline__ bool pull_tiles(const PullArgs &a, const float *__restrict__ x, const float *gy, float *gx, char *lds,
                                           PullShared &shared, int kind, int number, int lane, int blocks, int c0, int wgs, int wg, PullState<G> &state)
{
    using S = PullShape<G, P>;
    constexpr int kSegs = S::kSegs, kSteps = S::kSteps, kTiles = S::kTiles, kUnits = S::kUnits;
    constexpr int kTaps = Gather<N>::kTaps, kLines = Gather<N>::kLines, kLaneOut = Gather<N>::kLaneOut, kSlabOut = Gather<N>::kOutputs;
    const int cb = number / P, ch0 = c0 + cb * 16;                  // a worker's block
    const int update_end = min(a.update, c0 + 16 * blocks);         // of the chunk
    int buffer = 0;                               // of A: what is gathered, or taken through a product, next
    char *A = lds;
    auto turn_over = [&]() {
        buffer = 1 - buffer;
        A = lds + buffer * S::kTileBytes;
    };
    char *const own_x = lds + 2 * S::kTileBytes + number * S::kXBytes;             // a kernel worker's own
    char *const own_d = lds + 2 * S::kTileBytes + kOfKind * S::kXBytes + number * S::kDBytes;      // an input worker's
    // Sums are added to a second level every so many tiles: a chain of n additions of terms of mixed sign rounds to about sqrt(n / 2)
    // 2^-24 of what it comes to.  Errors of the weight gradients against 64 bits (2-norm), a chain over all tiles / in two levels: 192^3,
    // four outputs over 30 / 46 channels 6.7 / 2.1, 6.8 / 2.0 e-7; 2048 x 2048, 14 outputs over 40 4.3 / 1.4; 1024 x 1024 2.2 / 1.1; 333 x 477
    // 0.96 / 0.71.  Times are the same
    // within 2 %.  (With a branch in the loop over the tiles instead of around it, or with the second level cleared before the loop and added behind the second run, 3 to 6 % more over
    // 33 to 64 channels: the compiler then orders the loops of all kinds of waves otherwise.)
    constexpr int kChain = 16;                    // additions
    const int chain = wgs * (kChain / kUnits), bias_chain = wgs * kChain * (N != kImage ? 4 : 1);      // tiles, of all workgroups
    bool two_levels = false;
    auto second_level = [&](bool back) {          // of a kernel worker; back: all of it is in the registers again
        char *const at = lds + S::kSumsAt + number * S::kSumBytes + lane * 16;
#pragma unroll
        for (int t = 0; t < kTiles; t++) {
            f32x4_t &sum = *reinterpret_cast<f32x4_t *>(at + t * kWave * 16);
            if (two_levels) state.sums(t) += sum;             // uniform
            if (!back) {
                sum = state.sums(t);
                state.sums(t) = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        two_levels = true;
    };

    auto tile_of = [&](int tile) { return tile_at<kSegs>(a, tile); };
    auto locate = [&](const Tile &t, int segment) { return place_at<N>(a, t, segment); };
    const uint32_t plane = (uint32_t)a.sc * 4u;
    auto row_at = [&](int z, int y) { return (Gather<N>::kIsVolume ? z * (int)a.sz : 0) + y * (int)a.sy; };

    // The tiles: kSegs consecutive segments of an image each; every workgroup of an XCD works on neighbouring ones.
    const int lb = block_for_xcd(wg, wgs, wgs % kXcds == 0);

    // ---- x and grad_input of a unit, one segment: lane (channel lane / kLanes of kChannels, four voxels lane % kLanes)
    const int lv = lane % kLanes, lc = lane / kLanes;               // voxels 4 lv .., channels lc + kChannels i
    constexpr int kChannels = kWave / kLanes;     // channels of one access
    const uint32_t lane_plane = (uint32_t)lc * plane;
    auto unit_of = [&](const Tile &t, int u) {
        const Place p = locate(t, number % P * kUnits + u);
        Unit un;
        un.img = t.img;
        un.at = 4u * (uint32_t)(row_at(p.z, p.y) + p.x0 + 4 * lv);
        un.skip = min(max(p.skip - 4 * lv, 0), 4);
        return un;
    };
    auto request = [&](const float *from, int limit, const Unit &un, f32x4_t (&d)[kVec]) { request_unit(from, ch0, limit, plane, lane_plane, un, d); };

    // ---- the gather: a wave takes the 32 rows m of half h of one slab, 36 (27) values, at the voxels of two segments, so
    // that the outputs and their dilations are the wave's own: away from the edges a tap is a scalar address.  The loads are
    // issued in the tile before, in front of that tile's last stores and requests (all of them retire in order: behind
    // those they would wait for memory).
    const int pair = number / (2 * G), slab = number % (2 * G) / 2, h = number % 2;                // uniform
    const int v = lane % kSegment, segment = 2 * pair + lane / kSegment;
    auto output_of = [&](int j) { return Gather<N>::kIsVolume ? h : j < 3 ? 3 * h + j : 6; };
    // (in registers: a scalar load in the loop is 400 cycles of waiting)
    int dilation[kLaneOut];
    uint32_t gplane[kLaneOut];                    // byte offset of the output's gradient
#pragma unroll
    for (int j = 0; j < kLaneOut; j++) {
        const int o = min(slab * kSlabOut + output_of(j), a.out.n - 1);
        dilation[j] = a.out.dil[o];
        gplane[j] = (uint32_t)o * (uint32_t)(a.gsc * 4);
        asm volatile("" : "+s"(dilation[j]), "+s"(gplane[j]));
    }
    // of the lane: its voxel, and how many voxels of its segment belong to the one before; of the wave: whether some have such, whether
    // all voxels are away from the edges along x; along y and z
    struct Voxel {
        int x, y, z, skip;
        int skips, away_x, away_yz;               // (integers: a branch on a bool that is kept is made as if lanes could differ)
    };
    auto locate_pair = [&](const Tile &t) {
        const Place p = locate(t, 2 * pair), p2 = locate(t, 2 * pair + 1);
        const bool second = lane >= kSegment;
        Voxel vx{(second ? p2.x0 : p.x0) + v, second ? p2.y : p.y, second ? p2.z : p.z, second ? p2.skip : p.skip, max(p.skip, p2.skip), 0, 0};
        if constexpr (N == kFlat) {
            const int row = a.by_voxels.of(vx.x);
            vx.x -= row * a.W;
            vx.z = a.by_rows.of(row);
            vx.y = row - vx.z * a.H;
            vx.away_x = __all(vx.x >= a.dmax && vx.x + a.dmax < a.W) != 0;
            vx.away_yz = __all(vx.y >= a.dmax && vx.y + a.dmax < a.H && vx.z >= a.dmax && vx.z + a.dmax < a.D) != 0;
        } else {
            vx.away_x = int(min(p.x0, p2.x0) >= a.dmax) & int(max(p.x0, p2.x0) + kSegment + a.dmax <= a.W);
            vx.away_yz = int(min(p.y, p2.y) >= a.dmax) & int(max(p.y, p2.y) + a.dmax < a.H);
            if (N != kImage) vx.away_yz &= int(min(p.z, p2.z) >= a.dmax) & int(max(p.z, p2.z) + a.dmax < a.D);
        }
        vx.away_x = __builtin_amdgcn_readfirstlane(vx.away_x);
        vx.away_yz = __builtin_amdgcn_readfirstlane(vx.away_yz);
        return vx;
    };
    float val[kLaneOut][kLines][3];
    auto gather = [&](const Tile &t, const Voxel &vx) {
        const uint64_t base = reinterpret_cast<uint64_t>(gy) + (uint64_t)t.gimg;
#pragma unroll
        for (int j = 0; j < kLaneOut; j++) {
            const int d = dilation[j];
            const uint64_t output = base + gplane[j];
            const int up = min(vx.x + d, 2 * a.W - 1 - d - vx.x), down = max(vx.x - d, d - 1 - vx.x);
            const int row = row_at(vx.z, vx.y);
            uint32_t au = 4u * (uint32_t)(row + up), ah = 4u * (uint32_t)(row + vx.x), ad = 4u * (uint32_t)(row + down);
            // (formed here: in the branch they may take registers that the other branch loads to, and wait for them)
            if (N != kFlat) asm volatile("" : "+v"(au), "+v"(ah), "+v"(ad));
            if (vx.away_yz != 0) {                    // uniform
#pragma unroll
                for (int l = 0; l < kLines; l++) {
                    const uint64_t line = output + (uint64_t)((int64_t)row_at(N == kImage ? 0 : (1 - l / 3) * d, (1 - l % 3) * d) * 4);
                    val[j][l][0] = load1(line, au);
                    val[j][l][1] = load1(line, ah);
                    val[j][l][2] = load1(line, ad);
                }
                asm volatile("; away" ::: "memory");  // (or the loads of both branches are one, at addresses that are kept for it)
            } else {
                const Sides sy = sides(vx.y, a.H, d), sz = sides(vx.z, N == kImage ? 1 : a.D, N == kImage ? 0 : d);
#pragma unroll
                for (int l = 0; l < kLines; l++) {
                    const int y = l % 3 == 0 ? sy.up : l % 3 == 1 ? vx.y : sy.down;
                    const int z = N == kImage || l / 3 == 1 ? vx.z : l / 3 == 0 ? sz.up : sz.down;
                    const int at = row_at(z, y);
                    val[j][l][0] = load1(output, 4u * (uint32_t)(at + up));
                    val[j][l][1] = load1(output, 4u * (uint32_t)(at + vx.x));
                    val[j][l][2] = load1(output, 4u * (uint32_t)(at + down));
                }
            }
            __builtin_amdgcn_sched_barrier(0);        // (an output's addresses at a time: registers)
        }
    };
    auto gathered = [&](const Voxel &vx) {
        if (vx.away_x == 0) {                         // uniform
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const SideMasks sx(vx.x, a.W, dilation[j]);
#pragma unroll
                for (int l = 0; l < kLines; l++) fold(sx, val[j][l][0], val[j][l][2]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (vx.away_yz == 0) {                        // uniform
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const int d = dilation[j];
                const SideMasks sy(vx.y, a.H, d), sz(vx.z, N == kImage ? 1 : a.D, N == kImage ? 0 : d);
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
        if (vx.skips > 0 || a.out.n < G * kSlabOut) { // uniform
#pragma unroll
            for (int j = 0; j < kLaneOut; j++) {
                const bool ok = v >= vx.skip && slab * kSlabOut + output_of(j) < a.out.n;
#pragma unroll
                for (int t = 0; t < kTaps; t++) val[j][t / 3][t % 3] = ok ? val[j][t / 3][t % 3] : 0.f;
            }
        }
        if constexpr (!WHOLE) {                       // (the second run's have been counted)
            // (volumes: one value per lane, four chains of a quarter of the tiles)
            f32x4_t &bias = state.bias(0);
            if constexpr (N != kImage) bias = f32x4_t{bias[1], bias[2], bias[3], bias[0] + val[0][4 * (kLines / 9)][1]};
            else bias += f32x4_t{val[0][1][1], val[1][1][1], val[2][1][1], val[3][1][1]};
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
        if (lane == 0) shared.bad_tile[buffer][number] = any;
    };

    // ---- the products of a unit.  A worker's own space holds x as [block][part][channel][voxel], or what is added to grad_input
    // as [block][channel][voxel]: loads and stores go by channel in whole lines, the matrix cores take 16
    // channels at once (loaded in that form, 64 bytes of 16 channels at a time, memory gives 2.6 to 3.0 TB/s instead of 4).
    const int first_seg = number % P * kUnits;    // of the wave's first unit
    // (factors for the even and the odd voxels, in registers of their own: a sign in the instruction doubles its size)
    struct Factors {
        uint32_t even, odd;
        __device__ explicit Factors(float f, uint32_t sign = 0) : even(__float_as_uint(f) | sign), odd(even ^ 0x80000000u)
        {
            asm volatile("" : "+v"(even), "+v"(odd));   // (a multiply-add with a scalar operand issues in twice the cycles)
        }
        __device__ float of(int e) const { return __uint_as_float(e % 2 ? odd : even); }
    };
    // Rows 16 t + n, voxels 8 q .. of segment j (the lane's address is that of voxel 8 q + n / 4 (+ 4), rows
    // 4 (n % 4) .., which the read transposes).
    auto read_rows = [&](uint32_t ll, int j, int t, bf16x8_t(&to)[3]) {
        typedef short s16x4_t __attribute__((ext_vector_type(4)));
        typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4_t *lds_tr_t;
        const uint32_t nn = ll % 16, voxel = 8 * (ll / 16) + nn / 4;
        const char *const tr = A + (j * G + t / 4) * kSlabBytes + voxel * kVoxelBytes + nn % 2 * 8;
        const uint32_t piece = 16 * (nn % 4 / 2 ^ turn(voxel)), next = 16 * (nn % 4 / 2 ^ turn(voxel + 4));
#pragma unroll
        for (int p = 0; p < 3; p++) {
            const bf16x4_t lo = __builtin_bit_cast(
                bf16x4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(tr + p * kPartBytes + (piece ^ (uint32_t)(t % 4 * 32)))));
            const bf16x4_t hi = __builtin_bit_cast(
                bf16x4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(tr + p * kPartBytes + 4 * kVoxelBytes + (next ^ (uint32_t)(t % 4 * 32)))));
            to[p] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    // Voxels 16 s + n of segment j, rows 32 i + 8 q ..
    auto read_voxels = [&](uint32_t ll, int j, int s, int i, bf16x8_t(&to)[3]) {
        const uint32_t nn = ll % 16, qq = ll / 16;
        const char *const vox = A + (j * G + i / 2) * kSlabBytes + nn * kVoxelBytes;
#pragma unroll
        for (int p = 0; p < 3; p++)
            to[p] = *reinterpret_cast<const bf16x8_t *>(vox + p * kPartBytes + s * 16 * kVoxelBytes + (16 * (qq ^ turn(nn)) ^ (uint32_t)(i % 2 * 64)));
    };
    // (no LDS addresses are kept over the tiles: registers)
    auto fresh_lane = [&]() {
        uint32_t ll = (uint32_t)lane;
        asm volatile("" : "+v"(ll));
        return ll & (kWave - 1);
    };
    // a value of A where it lies whole
    auto whole_A = [&](int j, uint32_t voxel, uint32_t m) {
        const char *const at = A + (j * G + m / kRows) * kSlabBytes + voxel * kVoxelBytes + 16 * (m % kRows / 8 ^ turn(voxel)) + m % 8 * 2;
        return whole_value(*reinterpret_cast<const __bf16 *>(at), *reinterpret_cast<const __bf16 *>(at + kPartBytes));
    };
    // values of the tile at hand that can be split
    auto tile_split = [&]() {
        int bad = 0;
#pragma unroll
        for (int i = 0; i < kOfKind; i++) bad |= shared.bad_tile[buffer][i];
        return __builtin_amdgcn_readfirstlane(bad) == 0;
    };

    // -- grad_kernel
    f32x4_t xs[kVec];
    auto request_x = [&](const Unit &un) {
        request(x, a.C, un, xs);
    };
    // x in parts to the wave's own space; not finite where a value cannot be split
    auto put_x = [&](uint32_t sign_bit) {
        const Factors factor(kSplitScale, sign_bit);
        float x8[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x8[e] = xs[e / 4][e % 4] * factor.of(e);
        Split8 s;
        const float rest = split8(x8, s);
        typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int p = 0; p < 3; p++) {
            char *const at = own_x + (p * 16 + lc) * kXRow + 8 * lv;
            *reinterpret_cast<bf16x4_t *>(at) = __builtin_shufflevector(s.p[p], s.p[p], 0, 1, 2, 3);
            *reinterpret_cast<bf16x4_t *>(at + kChannels * kXRow) = __builtin_shufflevector(s.p[p], s.p[p], 4, 5, 6, 7);
        }
        return rest;
    };
    // False where a value cannot be split (and nothing is computed).
    auto kernel_unit = [&](int u, bool split, uint32_t sign_bit, const Unit &un, const Unit &next) {
        clear_skipped(un, xs);
        own_sync();
        const float rest = put_x(sign_bit);
        const bool done = split && !__any(taken_whole(rest));       // uniform
        __builtin_amdgcn_sched_barrier(0);        // (the scheduler would move the loads to where they are used)
        request_x(next);
        __builtin_amdgcn_sched_barrier(0);
        if (!done) return false;
        own_sync();
        const uint32_t ll = fresh_lane();
        const Factors back(kSplitUnit, sign_bit);
        // Stages of two chains of six matrix instructions, whose operands are read from LDS a stage ahead.
        bf16x8_t op[2][2][3], xp[3];
        auto stage = [&](int r) {
#pragma unroll
            for (int o = 0; o < 2; o++) read_rows(ll, first_seg + u, 2 * r + o, op[r % 2][o]);
        };
        stage(0);
#pragma unroll
        for (int p = 0; p < 3; p++) xp[p] = *reinterpret_cast<const bf16x8_t *>(own_x + (p * 16 + ll % 16) * kXRow + ll / 16 * 16);
#pragma unroll
        for (int r = 0; r < kTiles / 2; r++) {
            if (r + 1 < kTiles / 2) stage(r + 1);
            __builtin_amdgcn_sched_barrier(0);
            f32x4_t acc[2];
#pragma unroll
            for (int k = 0; k < 6; k++)
#pragma unroll
                for (int o = 0; o < 2; o++) acc[o] = mfma_split(op[r % 2][o], xp, k == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : acc[o], k);
#pragma unroll
            for (int o = 0; o < 2; o++) {
                state.sums(2 * r + o) += back.of(0) * acc[o];
                asm volatile("" : "+v"(state.sums(2 * r + o)));                    // (here and not at the end of the tile: registers)
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return true;
    };
    // The same with the fp32 instruction, for values that cannot be split (A lies whole in the place of its parts).
    auto kernel_whole = [&](int u, uint32_t sign_bit) {
        const float sign = __uint_as_float(sign_bit | 0x3f800000u);
        const uint32_t ll = fresh_lane(), nn = ll % 16, qq = ll / 16;
        own_sync();
#pragma unroll
        for (int i = 0; i < kVec; i++)
            *reinterpret_cast<f32x4_t *>(own_x + (lc + kChannels * i) * kDRow + 16 * lv) = xs[i] * f32x4_t{sign, -sign, sign, -sign};
        own_sync();
#pragma unroll
        for (int t = 0; t < kTiles; t++) {
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int e = 0; e < 8; e++) {
                const uint32_t voxel = 8 * qq + (uint32_t)e;
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(whole_A(first_seg + u, voxel, 16 * t + nn),
                                                           *reinterpret_cast<const float *>(own_x + nn * kDRow + 4 * voxel), acc, 0, 0, 0);
            }
            state.sums(t) += sign * acc;
        }
        own_sync();
    };

    // -- grad_input
    f32x4_t gs[kVec];
    auto request_g = [&](const Unit &un) {
        if constexpr (FRESH) {
#pragma unroll
            for (int i = 0; i < kVec; i++) gs[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        } else {
            request(gx, max(update_end, 1), un, gs);
        }
    };
    // what the wave's own space holds for grad_input, in units of `unit`, added to it and masked with the activations m
    const bool masks = ch0 + 16 > a.mask_from && ch0 < update_end;                 // uniform
    auto add_d = [&](const f32x4_t (&m)[kVec], const Factors unit) {
#pragma unroll
        for (int i = 0; i < kVec; i++) {
            const f32x4_t d = *reinterpret_cast<const f32x4_t *>(own_d + (lc + kChannels * i) * kDRow + 16 * lv);
#pragma unroll
            for (int e = 0; e < 4; e++) gs[i][e] = __builtin_fmaf(d[e], unit.of(e), gs[i][e]);
        }
        if (masks) {
#pragma unroll
            for (int i = 0; i < kVec; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) gs[i][e] = ch0 + lc + kChannels * i < a.mask_from || 0.f < m[i][e] ? gs[i][e] : 0.f;
        }
    };
    auto store = [&](const Unit &un, bool all) { store_unit(gx, ch0, update_end, plane, lane_plane, lc, un, gs, all); };
    auto input_unit = [&](int u, const Unit &un) {
        f32x4_t m[kVec];
        if (masks) request(x, a.C, un, m);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t ll = fresh_lane(), nn = ll % 16, qq = ll / 16;
        own_sync();                               // (what was there has been read)
        // Stages of a step of rows at both halves of the voxels, read a stage ahead.
        bf16x8_t op[2][2][3], high[2];
        f32x4_t d[2], all[2];
        auto stage = [&](int r) {
#pragma unroll
            for (int s = 0; s < 2; s++) read_voxels(ll, first_seg + u, s, r, op[r % 2][s]);
        };
        stage(0);
#pragma unroll
        for (int i = 0; i < kSteps; i++) {
            if (i + 1 < kSteps) stage(i + 1);
            __builtin_amdgcn_sched_barrier(0);
            const bf16x8_t w[3] = {state.weights(i, 0), state.weights(i, 1), state.weights(i, 2)};
            // (the products of the high parts of a slab's two steps last: each instruction cuts its sum off at the size
            // that it has reached)
#pragma unroll
            for (int k = 0; k < 5; k++)
#pragma unroll
                for (int s = 0; s < 2; s++) d[s] = mfma_split(op[i % 2][s], w, k == 0 && i % 2 == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : d[s], k);
            if (i % 2 == 0) {
#pragma unroll
                for (int s = 0; s < 2; s++) high[s] = op[i % 2][s][0];
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        d[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(j ? op[i % 2][s][0] : high[s], state.weights(i - 1 + j, 0), d[s], 0, 0, 0);
                // Summed slab by slab from zero and added to grad_input last: a chain of products that started from it
                // would round each of them to its size.
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    all[s] = i == 1 ? d[s] : all[s] + d[s];
                    if (i == kSteps - 1) *reinterpret_cast<f32x4_t *>(own_d + nn * kDRow + (16 * s + 4 * qq) * 4) = all[s];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        own_sync();
        add_d(m, Factors(kSplitUnit));
    };
    // (the weights lie whole in the place of their parts)
    auto input_whole = [&](int u, const Unit &un) {
        const uint32_t ll = fresh_lane(), nn = ll % 16, qq = ll / 16;
        f32x4_t m[kVec];
        if (masks) request(x, a.C, un, m);
        own_sync();
#pragma unroll 1
        for (int s = 0; s < 2; s++) {
            f32x4_t all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < kSteps; i++) {
                f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 8; e++)
                    d = __builtin_amdgcn_mfma_f32_16x16x4f32(whole_A(first_seg + u, 16 * s + nn, 32 * i + 8 * qq + e),
                                                             whole_value(state.weights(i, 0)[e], state.weights(i, 1)[e]), d, 0, 0, 0);
                all += d;
            }
            *reinterpret_cast<f32x4_t *>(own_d + nn * kDRow + (16 * s + 4 * qq) * 4) = all;
        }
        own_sync();
        add_d(m, Factors(1.f));
    };

    const bool kernel = cb < blocks && kind == kKernel, input = cb < blocks && ch0 < update_end && kind == kInput;     // uniform
    if constexpr (WHOLE) {
#pragma unroll 1
        for (int tile = lb, count = 0; tile < a.tiles; tile += wgs, count += kUnits) {
            const Tile t = tile_of(tile);
            if (kernel && count > 0 && count % kChain == 0) second_level(false);   // uniform
            if (kind == kGatherer) {
                const Voxel here = locate_pair(t);
                gather(t, here);
                gathered(here);
            }
            __syncthreads();
            const bool split = tile_split();
#pragma unroll 1
            for (int u = 0; u < kUnits; u++) {    // (what the first run has done is left out)
                const Unit un = unit_of(t, u);
                if (kernel) {
                    request_x(un);
                    clear_skipped(un, xs);
                    own_sync();
                    if (!split || __any(taken_whole(put_x(t.sign)))) kernel_whole(u, t.sign);
                }
                if (input && !(split && state.weights_split)) {
                    request_g(un);
                    input_whole(u, un);
                    store(un, true);
                }
            }
            __syncthreads();
        }
        if (kernel && two_levels) second_level(true);
        return false;
    } else if (kind == kGatherer) {
        // A tile is formed in the one buffer while the workers have the other; a barrier, and they change.
        Voxel here = locate_pair(tile_of(lb));
        gather(tile_of(lb), here);
        for (int tile = lb; tile < a.tiles;) {    // uniform over the workgroup
            for (const int end = min(a.tiles, tile + bias_chain); tile < end; tile += wgs) {
                gathered(here);
                if (tile + wgs < a.tiles) {       // (the loads have the time of a tile to arrive)
                    const Tile then = tile_of(tile + wgs);
                    here = locate_pair(then);
                    gather(then, here);
                }
                turn_over();
                lds_sync();
            }
            state.bias(1) += state.bias(0);
            state.bias(0) = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        lds_sync();
        return false;
    } else if (kind == kKernel) {
        bool again = false;                       // units were left to the second run
        Tile now = tile_of(lb);
        Unit un = unit_of(now, 0);
        if (kernel) request_x(un);
        lds_sync();
        for (int tile = lb; tile < a.tiles;) {
            for (const int end = min(a.tiles, tile + chain); tile < end; tile += wgs) {
                if (kernel) {
                    const Tile then = tile_of(tile + wgs);
                    const bool split = tile_split();
#pragma unroll
                    for (int u = 0; u < kUnits; u++) {
                        const Unit next = u + 1 < kUnits ? unit_of(now, u + 1) : unit_of(then, 0);
                        again = !kernel_unit(u, split, now.sign, un, next) || again;
                        un = next;
                    }
                    now = then;
                }
                turn_over();
                lds_sync();
            }
            if (tile < a.tiles) second_level(false);
        }
        if (two_levels) second_level(true);
        return again;
    } else {
        bool again = false;
        Tile now = tile_of(lb);
        Unit un = unit_of(now, 0);
        if (input) request_g(un);
        lds_sync();
        for (int tile = lb; tile < a.tiles; tile += wgs) {
            if (input) {
                const Tile then = tile_of(tile + wgs);
                const bool split = tile_split() && state.weights_split;
#pragma unroll
                for (int u = 0; u < kUnits; u++) {
                    const Unit next = u + 1 < kUnits ? unit_of(now, u + 1) : unit_of(then, 0);
                    if (split) input_unit(u, un);
                    store(un, split);
                    __builtin_amdgcn_sched_barrier(0);
                    request_g(next);
                    __builtin_amdgcn_sched_barrier(0);
                    un = next;
                }
                again = again || !split;
                now = then;
            }
            turn_over();
            lds_sync();
        }
        return again;
    }
}

// FRESH: grad_input is written, not added to.
template <int N, int G, int P, bool FRESH = false>
__global__ __launch_bounds__(kPullThreads, 3) void pull_rows(const PullArgs a, const float *__restrict__ x, const float *gy,
                                                             float *gx, float *__restrict__ part, float *__restrict__ bias_part)
{
    using S = PullShape<G, P>;
    constexpr int kTiles = S::kTiles;
    constexpr int kTaps = Gather<N>::kTaps, kLaneOut = Gather<N>::kLaneOut, kSlabOut = Gather<N>::kOutputs;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int n = lane % 16, q = lane / 16;
    const int bid = blockIdx.x, big = a.chunks.large * a.chunks.wgs;
    const int chunk = bid < big ? bid / a.chunks.wgs : a.chunks.large + (bid - big) / a.chunks.wgs_small;
    const int blocks = a.chunks.size(chunk), c0 = a.chunks.first_block(chunk) * 16;
    const int wgs = a.chunks.rows(chunk), wg = bid - a.chunks.first_wg(chunk);
    // (the workers of the two products that have no block are on different SIMDs)
    const int kind = wave / kOfKind, number = (wave + (kind == kInput ? 2 : 0)) % kOfKind;
    const int cb = number / P, ch0 = c0 + cb * 16;                  // a worker's block
    __shared__ PullShared shared;
    PullState<G> state;

    if (tid == 0) shared.bad_again = 0;
    auto load_weights = [&](bool whole) {
        if (kind != kInput) return;               // uniform
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
            for (int p = 0; p < 3; p++) state.set_weights(step, p, s.p[p]);
        }
    };
    state.weights_split = true;
#pragma unroll
    for (f32x4_t &v : state.kept) v = f32x4_t{0.f, 0.f, 0.f, 0.f};
    load_weights(false);
    __syncthreads();

    float *const row = part + (int64_t)bid * (a.chunks.blocks * 1024 * G);
    const bool again = pull_tiles<N, G, P, FRESH, false>(a, x, gy, gx, lds, shared, kind, number, lane, blocks, c0, wgs, wg, state);
    if (lane == 0 && again) shared.bad_again = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(shared.bad_again) != 0) {    // uniform over the workgroup
        int lane2 = lane;
        asm volatile("" : "+v"(lane2));          // (nothing of the first run is kept for the second)
        load_weights(true);
        pull_tiles<N, G, P, FRESH, true>(a, x, gy, gx, lds, shared, kind, number, lane2, blocks, c0, wgs, wg, state);
    }

    // the sums, of the waves that share a block through LDS
    constexpr int kBlock = 1024 * G;              // sums of a block of channels
    if constexpr (P == 1) {
        if (kind == kKernel && cb < blocks) {
#pragma unroll
            for (int t = 0; t < kTiles; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) row[cb * kBlock + (t * 4 + r) * kWave + lane] = state.sums(t)[r];
        }
    } else {
        float *const red = reinterpret_cast<float *>(lds);
        __syncthreads();
        if (kind == kKernel) {
#pragma unroll
            for (int t = 0; t < kTiles; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) red[number * kBlock + (t * 4 + r) * kWave + lane] = state.sums(t)[r];
        }
        __syncthreads();
        for (int i = tid; i < kOfKind / P * kBlock; i += kPullThreads) {
            const int b = i / kBlock;
            const float *const r = red + b * P * kBlock + i % kBlock;
            if (b < blocks) row[i] = P == 2 ? r[0] + r[kBlock] : (r[0] + r[kBlock]) + (r[2 * kBlock] + r[3 * kBlock]);
        }
    }
    if (chunk != 0) return;
    // the bias gradients: the centre taps, over the lanes' voxels and the segments
    const int h = wave % 2;                       // (the waves' outputs: see the gather)
    f32x4_t bias_sum = state.bias(1);
    if constexpr (N != kImage) bias_sum[0] = (bias_sum[0] + bias_sum[1]) + (bias_sum[2] + bias_sum[3]);
#pragma unroll
    for (int j = 0; j < kLaneOut; j++)
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) bias_sum[j] += __shfl_down(bias_sum[j], off);
    float *const red = reinterpret_cast<float *>(lds);              // [waves of a slab][slab][column]
    __syncthreads();
    if (lane == 0 && kind == kGatherer) {
#pragma unroll
        for (int j = 0; j < kLaneOut; j++)
            if (N != kImage || j < 3 || h == 0) red[wave / 2 * kBiasColumns + (N != kImage ? h : j < 3 ? 3 * h + j : 6)] = bias_sum[j];
    }
    __syncthreads();
    if (tid < G * kBiasColumns && tid % kBiasColumns < kSlabOut) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < kOfKind / (2 * G); i++) s += red[i * G * kBiasColumns + tid];
        bias_part[wg * (G * kBiasColumns) + tid] = s;
    }
}

struct SumArgs {
    Chunks chunks;
    int columns;                                  // weight columns in all (a multiple of 1024 slabs)
    int slabs;
    int stride;                                   // of the rows of partial sums
    int n, fresh;                                 // outputs; gradients are written, not added to
    int channels[kMaxOut];                        // input channels of each output
    float *gk[kMaxOut];
    float *gb;
};

// Adds the rows of partial sums, 64 columns per workgroup: 16 waves take every 16th row, their
// sums are added in order.  The last workgroup takes the biases.
template <int N>
__global__ __launch_bounds__(1024) void sum_group(const SumArgs a, const float *__restrict__ part,
                                                  const float *__restrict__ bias_part)
{
    constexpr int kTaps = Gather<N>::kTaps, kSlabOut = Gather<N>::kOutputs;
    __shared__ double lds[16 * kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = blockIdx.x * kWave + lane, block = 1024 * a.slabs;
    const bool bias = (int)blockIdx.x * kWave >= a.columns;
    const int blk = col / block, big = a.chunks.large * a.chunks.blocks;
    const int chunk = blk < big ? blk / a.chunks.blocks
                                : (a.chunks.blocks > 1 ? a.chunks.large + (blk - big) / (a.chunks.blocks - 1) : 0);
    const int rows = a.chunks.rows(bias ? 0 : chunk);
    const float *p;
    int64_t stride;
    if (bias) {
        stride = a.slabs * kBiasColumns;
        p = bias_part + lane % (a.slabs * kBiasColumns);
    } else {
        p = part + (int64_t)a.chunks.first_wg(chunk) * a.stride + (blk - a.chunks.first_block(chunk)) * block + col % block;
        stride = a.stride;
    }
    double part_sum[4] = {0., 0., 0., 0.};        // (these are the largest sums)
    for (int r = wave; r < rows; r += 128) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = p[min(r + 16 * i, rows - 1) * stride];
#pragma unroll
        for (int i = 0; i < 8; i++) part_sum[i % 4] += r + 16 * i < rows ? (double)v[i] : 0.;
    }
    lds[wave * kWave + lane] = (part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]);
    __syncthreads();
    if (wave != 0) return;
    double tree[16];
#pragma unroll
    for (int w = 0; w < 16; w++) tree[w] = lds[w * kWave + lane];
#pragma unroll
    for (int w = 8; w > 0; w /= 2)
#pragma unroll
        for (int i = 0; i < w; i++) tree[i] += tree[i + w];
    const float s = (float)tree[0];
    if (bias) {
        const int o = lane / kBiasColumns * kSlabOut + lane % kBiasColumns;
        if (lane < a.slabs * kBiasColumns && lane % kBiasColumns < kSlabOut && o < a.n) a.gb[o] = a.fresh ? s : a.gb[o] + s;
        return;
    }
    // column (tile of 16 rows, r, lane (channel, q)) of a block: row 16 tile + 4 q + r
    const int i = col % block, l = i % kWave;
    const Slot m = slot_of<N>(i / 256 * 16 + l / 16 * 4 + i / kWave % 4);
    const int ch = blk * 16 + l % 16;
    if (m.tap >= 0 && m.output < a.n && ch < a.channels[m.output]) {
        float &k = a.gk[m.output][(int64_t)ch * kTaps + m.tap];
        k = a.fresh ? s : k + s;
    }
}

// grad_input of the channels that layers of a group wrote, from the outputs of the layers above them
// in the group.
//
// One voxel per lane; the nine (27) values of each output come straight from the caches (a group's planes
// were written or read by the launches before), not by way of LDS: the launches are bound by
// their ramp, the vector cache and, with scalar weights, the multiply-adds.
struct FinishArgs {
    int D, H, W, span, segs, items, dmax;         // (as in PullArgs, segments of 64)
    Divisor by_rows, by_voxels;
    int n, channels, masked;                      // spread_back: outputs above, channels, first one to mask
    int64_t sb, sc, sz, sy;
    int dil[kMaxAbove];
    const float *k[kMaxAbove];                    // of the first of the channels
};

// The lane's place, and the adjoint gather there.
struct FinishPlace {
    int z, y, u, own;                             // slice, row, voxel, whether the voxel is the lane's own
    bool away;                                    // uniform: from all edges
    int64_t img;
    uint32_t here;
};
template <int N> __device__ __forceinline__ FinishPlace finish_place(const FinishArgs &a, int it)
{
    FinishPlace p;
    const int row = it / a.segs, xw = (it - row * a.segs) * kWave;
    const int u0 = xw + threadIdx.x % kWave, at = min(u0, a.span - 1);
    p.own = u0 < a.span;
    if constexpr (N == kFlat) {                   // (a row is a volume)
        const int line = a.by_voxels.of(at);
        p.u = at - line * a.W;
        p.z = a.by_rows.of(line);
        p.y = line - p.z * a.H;
        p.away = false;
        p.img = (int64_t)row * a.sb * 4;
        p.here = 4u * (uint32_t)at;
    } else {
        const int slice = row / a.H, b = N == kVolume ? slice / a.D : slice;
        p.u = at;
        p.y = row - slice * a.H;
        p.z = slice - b * (N == kVolume ? a.D : 1);
        p.away = xw >= a.dmax && xw + kWave + a.dmax <= a.W && p.y >= a.dmax && p.y + a.dmax < a.H &&
                 (N == kImage || (p.z >= a.dmax && p.z + a.dmax < a.D));
        p.img = (int64_t)b * a.sb * 4;
        p.here = 4u * (uint32_t)((N == kVolume ? p.z * (int)a.sz : 0) + p.y * (int)a.sy + p.u);
    }
    return p;
}
template <int N>
__device__ __forceinline__ void finish_gather(const FinishArgs &a, const FinishPlace &p, uint64_t output, int d, float (&A)[Gather<N>::kLines][3])
{
    Sides sx = {p.u + d, p.u - d, true, true}, sy = {p.y + d, p.y - d, true, true};      // y, z: uniform
    Sides sz = {p.z + d, p.z - d, true, true};
    if (!p.away) {
        sx = sides(p.u, a.W, d);
        sy = sides(p.y, a.H, d);
        if (N != kImage) sz = sides(p.z, a.D, d);
    }
#pragma unroll
    for (int l = 0; l < Gather<N>::kLines; l++) {
        const int y = l % 3 == 0 ? sy.up : l % 3 == 1 ? p.y : sy.down;
        const int z = l / 3 == 0 ? sz.up : l / 3 == 1 ? p.z : sz.down;
        // (kFlat: an offset of the lane's, else a uniform base)
        const int64_t line = 4 * ((N != kImage ? (int64_t)z * a.sz : 0) + (int64_t)y * a.sy);
        if constexpr (N == kFlat) {
            const uint32_t at = (uint32_t)line;
            A[l][0] = load1(output, at + 4u * (uint32_t)sx.up);
            A[l][1] = load1(output, at + 4u * (uint32_t)p.u);
            A[l][2] = load1(output, at + 4u * (uint32_t)sx.down);
            continue;
        }
        const uint64_t base = output + (uint64_t)line;
        A[l][0] = load1(base, 4u * (uint32_t)sx.up);
        A[l][1] = load1(base, 4u * (uint32_t)p.u);
        A[l][2] = load1(base, 4u * (uint32_t)sx.down);
    }
}
template <int N>
__device__ __forceinline__ void finish_fold(const FinishArgs &a, const FinishPlace &p, int d, float (&A)[Gather<N>::kLines][3])
{
    const Sides sx = sides(p.u, a.W, d), sy = sides(p.y, a.H, d);
#pragma unroll
    for (int l = 0; l < Gather<N>::kLines; l++) fold(sx, A[l][0], A[l][2]);
#pragma unroll
    for (int l = 0; l < Gather<N>::kLines; l += 3)
#pragma unroll
        for (int r = 0; r < 3; r++) fold(sy, A[l][r], A[l + 2][r]);
    if constexpr (N != kImage) {
        const Sides sz = sides(p.z, a.D, d);
#pragma unroll
        for (int l = 0; l < 3; l++)
#pragma unroll
            for (int r = 0; r < 3; r++) fold(sz, A[l][r], A[l + 6][r]);
    }
}

// The NOUT channels of one layer from the NQ outputs right above, and the channels' ReLU mask: with it
// they are complete.
//
// Images with several outputs above take the weights through LDS into vector registers (see spread_back): 1000 x 1000, two channels
// from 2 / 4 / 6 outputs 9.8, 8.6 / 13.7, 11.3 / 18.7, 15.3 us; 1024 x 1024, one from 6: 12.6, 12.3; 3 x 333 x 477: 8.9, 8.1.  One output
// (4.8, 5.0) and volumes (128^3, one channel from 3: 37.3, 40.4) keep scalar ones.
template <int N, int NQ, int NOUT>
__global__ __launch_bounds__(256) void finish_back(const FinishArgs a, const float *__restrict__ act, float *g)
{
    constexpr int kTaps = Gather<N>::kTaps;
    const int lb = block_for_xcd(blockIdx.x, gridDim.x, true);
    const int it0 = lb * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), it = min(it0, a.items - 1);
    constexpr bool kStage = N == kImage && NQ > 1;
    if (!kStage && it0 >= a.items) return;        // uniform over the wave
    constexpr int kRow = (NOUT * kTaps + 3) / 4 * 4;                // an output's weights, in whole pieces of 16 bytes
    __shared__ __attribute__((aligned(16))) float weights[kStage ? NQ * kRow : 4];
    static_assert(!kStage || NQ * kRow <= 256, "a weight per thread");
    float w = 0.f;
    if constexpr (kStage) w = a.k[min((int)threadIdx.x / kRow, NQ - 1)][min((int)threadIdx.x % kRow, NOUT * kTaps - 1)];
    const FinishPlace p = finish_place<N>(a, it);
    const uint64_t img = reinterpret_cast<uint64_t>(g) + (uint64_t)p.img;
    const uint64_t ximg = reinterpret_cast<uint64_t>(act) + (uint64_t)p.img;
    const uint32_t plane = (uint32_t)a.sc * 4u;
    float sum[NOUT], m[NOUT];
#pragma unroll
    for (int c = 0; c < NOUT; c++) {
        sum[c] = load1(img, (uint32_t)c * plane + p.here);
        m[c] = load1(ximg, (uint32_t)c * plane + p.here);
    }
    float A[NQ][Gather<N>::kLines][3];
#pragma unroll
    for (int o = 0; o < NQ; o++) finish_gather<N>(a, p, img + (uint64_t)(NOUT + o) * plane, a.dil[o], A[o]);
    if constexpr (kStage) {
        if (threadIdx.x < NQ * kRow) weights[threadIdx.x] = w;
        __syncthreads();
        if (it0 >= a.items) return;               // uniform over the wave
    }
    if (!p.away) {
#pragma unroll
        for (int o = 0; o < NQ; o++) finish_fold<N>(a, p, a.dil[o], A[o]);
    }
#pragma unroll
    for (int c = 0; c < NOUT; c++) {
        float all = 0.f;                          // (output by output, and added to grad_input last: see pull_rows)
#pragma unroll
        for (int o = 0; o < NQ; o++) {
            float one = 0.f;
#pragma unroll
            for (int t = 0; t < kTaps; t++) one += (kStage ? weights[o * kRow + c * kTaps + t] : a.k[o][c * kTaps + t]) * A[o][t / 3][t % 3];
            all += one;
        }
        sum[c] += all;
        const float v[1] = {0.f < m[c] ? sum[c] : 0.f};
        if (p.own) store_global_vec<1>(img, (uint32_t)c * plane + p.here, v);
    }
}

// What the upper half of a group's outputs adds to all channels that its lower half wrote, before
// those are completed one layer after the other; the last of them, from `masked` on, are with it.
//
// The values of all outputs are requested at once, and the weights come through LDS into vector registers: a multiply-add of three of
// these issues in 2.4 cycles, one with a scalar operand in 4.3, and there is no round of scalar loads per output.  With scalar weights, output by
// output, the next one's values requested ahead: 1024 x 1024 48.2 -> 33.9 us, 2 x 512 x 512 26.0 -> 19.9, 3 x 333 x 477 25.1 ->
// 20.5, 256 x 256 11.1 -> 8.8.
__global__ __launch_bounds__(256) void spread_back(const FinishArgs a, const float *__restrict__ act, float *g)
{
    __shared__ __attribute__((aligned(16))) float weights[kMaxAbove * kMaxLower * 12];          // [output][channel][tap]
    const int lb = block_for_xcd(blockIdx.x, gridDim.x, true);
    const int it0 = lb * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), it = min(it0, a.items - 1);
    const FinishPlace p = finish_place<kImage>(a, it);
    const uint64_t img = reinterpret_cast<uint64_t>(g) + (uint64_t)p.img;
    const uint64_t ximg = reinterpret_cast<uint64_t>(act) + (uint64_t)p.img;
    const uint32_t plane = (uint32_t)a.sc * 4u;
    float w[2];
    const int count = a.n * a.channels * kTaps;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int at = min((int)threadIdx.x + 256 * i, count - 1), o = at / (a.channels * kTaps);
        w[i] = a.k[o][at - o * a.channels * kTaps];
    }
    float A[kMaxAbove][3][3], sum[kMaxLower], m[2];
#pragma unroll
    for (int o = 0; o < kMaxAbove; o++) {
        const int oo = min(o, a.n - 1);           // (what the rest holds is not used)
        finish_gather<kImage>(a, p, img + (uint64_t)(a.channels + oo) * plane, a.dil[oo], A[o]);
    }
#pragma unroll
    for (int c = 0; c < 2; c++) m[c] = load1(ximg, (uint32_t)min(a.masked + c, a.channels - 1) * plane + p.here);
#pragma unroll
    for (int c = 0; c < kMaxLower; c++) sum[c] = load1(img, (uint32_t)min(c, a.channels - 1) * plane + p.here);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int at = (int)threadIdx.x + 256 * i, o = at / (a.channels * kTaps), r = at - o * a.channels * kTaps;
        if (at < count) weights[(o * kMaxLower + r / kTaps) * 12 + r % kTaps] = w[i];
    }
    __syncthreads();
    if (it0 >= a.items) return;                   // uniform over the wave
    float all[kMaxLower] = {};
#pragma unroll
    for (int o = 0; o < kMaxAbove; o++) {
        if (o >= a.n) break;                      // uniform
        if (!p.away) finish_fold<kImage>(a, p, a.dil[o], A[o]);
#pragma unroll
        for (int c = 0; c < kMaxLower; c++) {
            const float *const k = weights + (o * kMaxLower + min(c, a.channels - 1)) * 12;
            float one = 0.f;
#pragma unroll
            for (int t = 0; t < kTaps; t++) one += k[t] * A[o][t / 3][t % 3];
            all[c] += one;
        }
    }
#pragma unroll
    for (int c = 0; c < kMaxLower; c++) {
        if (c >= a.channels) break;               // uniform
        const float act_c = c == a.masked ? m[0] : m[1];
        const float v[1] = {c < a.masked || 0.f < act_c ? sum[c] + all[c] : 0.f};
        if (p.own) store_global_vec<1>(img, (uint32_t)c * plane + p.here, v);
    }
}
// Wherever the voxels lie without gaps.  Backward pass of a block, us, as rows and as one row: 61 x 93 x 75, depth 20: 639, 499;
// 80 x 81 x 65, depth 30: 1051, 732; 127^3, depth 30: 2784, 2732; and with whole segments (no fold is ever skipped, but the
// lanes' rows cost no scalar work) 64^3, depth 30: 548, 529; 128^3: 2800, 2757.
Form form_of(const Geom &g, const View<const float> &x)
{
    if (g.ndim == 2) return kImage;
    return x.sy == g.W && x.sz == (int64_t)g.H * g.W ? kFlat : kVolume;
}

template <int N, int NQ, int NOUT>
hipError_t finish_back_launch(const FinishArgs &a, const float *act, float *g, hipStream_t s)
{
    hipLaunchKernelGGL((finish_back<N, NQ, NOUT>), dim3(xcd_grid((a.items + 3) / 4)), dim3(256), 0, s, a, act, g);
    return hipGetLastError();
}

FinishArgs finish_args(const Geom &g, const View<const float> &x, const group2d::Outputs &above)
{
    const int span = form_of(g, x) == kFlat ? g.nvox : g.W, segs = (span + kWave - 1) / kWave;
    FinishArgs a{g.D, g.H, g.W, span, segs, g.nvox / span * g.B * segs, 0, Divisor((uint32_t)g.H), Divisor((uint32_t)g.W),
                 above.n, 0, 0, x.sb, x.sc, x.sz, x.sy, {}, {}};
    for (int o = 0; o < above.n; o++) {
        a.dil[o] = above.dil[o];
        a.k[o] = above.k[o];
        a.dmax = std::max(a.dmax, above.dil[o]);
    }
    return a;
}

template <typename F>
hipError_t pull_launch(F *kernel, int threads, int lds, LargeLds &large, const PullArgs &a, int wgs, const float *x, const float *gy, float *gx, float *part,
                       float *bias_part, hipStream_t s)
{
    const hipError_t e = large.allow(reinterpret_cast<const void *>(kernel), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(wgs), dim3(threads), lds, s, a, x, gy, gx, part, bias_part);
    return hipGetLastError();
}

// Blocks of a chunk, at most (one slab, when all had eight waves: 411 us over 100 channels, 463 with 8).
int most_blocks(int slabs) { return slabs == 1 ? 4 : 8; }
// Blocks of a chunk of two slabs that pull_rows takes; pull_rows_wide the others, and three and four of one slab in large images.  There the eight waves of the
// latter are faster, which all gather a tile twice as large and then all multiply.  Volumes, and images whose gradients are written: from so many values of x and of the outputs'
// gradients on, which with grad_input fill 240 MB of the 256 MB cache, behind which the units of 32 voxels wait longer.  pull_rows to pull_rows_wide 1, a layer of one output: 80^3 over 60 / 64
// channels (31.2, 33.3 million values) 0.95 / 1.13; 80 x 81 x 83 over 56 / 60 / 64 (30.7, 32.8, 35.0) 0.92 / 1.00 / 1.03; 90^3 over 41 / 48 (30.6, 35.7) 0.94 / 1.06; 90 x 100 x 101 over 33 / 36 / 41 /
// 48 (30.9, 33.6, 38.2, 44.5) 0.95 / 1.02 / 1.07 / 1.15; 100^3 over 33 / 48 / 64 0.97 / 1.13 / 1.12; 108^3 1.01 / 1.18 / 1.15; two outputs 80^3 over 56 / 60 (29.7, 31.7) 0.96 / 1.08; three 512 x 513 over 64 (17.6) 0.86; 724 x
// 724 over 56 / 64 (30.9, 35.1) 0.95 / 1.02; 700 x 801 over 52 / 56 / 60 (30.8, 33.1, 35.3) 1.00 / 1.02 / 1.05; two outputs, added to, 90^3 over 36 / 44 / 60 0.92 / 0.97 / 0.98; 90 x 100 x 101
// 0.98 / 1.05 / 1.03; 113^3 1.00 / 1.03 / 1.01.
// Other images: from so many segments of 32 voxels on, for each 256 workgroups of the chunk.  Seven outputs, added to, over 36 / 44 / 52 / 60 channels: 512 x 513 0.94 / 0.93 / 0.90 /
// 0.89; 724 x 724 0.96 / 0.95 / 0.93 / 0.96; 700 x 801 0.99 / 0.98 / 0.95 / 0.97; over 40 / 48 / 60 below them 800 x 800 1.00 / 1.05 / 1.12, 1024 x 1000 1.04 / 1.01 / 1.00, 2048 x
// 2048 1.13 / 1.05 / 1.05.  Chunks side by side have fewer workgroups each (60 channels below seven outputs are five blocks, 3 + 2); over 64 / 70 / 100 / 130 512 x
// 512 1.02 / 0.97 / 0.99 / 1.06, 680 x 700 1.03 / 1.02 / 1.03 / 1.00; 61 x 93 x 75 1.02 / 0.93 / 1.02 / 1.02, 80^3 1.10 / 1.08 / 1.03 / 1.03, 90^3 1.14 / 1.08 /
// 1.00 / 1.00.
constexpr int kNarrowBlocks = 4, kNarrowOneSlab = 2;
constexpr int64_t kWideImage = 20000, kWideValues = 30 << 20;

// As many workgroups as are resident, shared out over the chunks by their size.
struct PullPlan {
    Chunks chunks;
    int segs, wgs, image_tiles, tiles;
    bool wide;                                    // pull_rows_wide
};

PullPlan pull_plan(int64_t batch, int64_t rows, int64_t span, int64_t channels, int slabs, bool volume = false, int outputs = 0)
{
    PullPlan p;
    const int nb = (int)((channels + 15) / 16);
    Chunks &c = p.chunks;
    const int most = most_blocks(slabs);
    c.n = (nb + most - 1) / most;
    c.blocks = (nb + c.n - 1) / c.n;
    c.large = nb - c.n * (c.blocks - 1);
    p.segs = (int)((span + kSegment - 1) / kSegment);
    const bool large = (outputs > 0 && batch * rows * span * (channels + outputs) >= kWideValues) || (!volume && batch * rows * p.segs * nb >= kWideImage * c.blocks);
    p.wide = slabs == 1 ? c.blocks > kNarrowOneSlab && large : c.blocks > kNarrowBlocks;
    const int per_tile = (p.wide ? kWaves : kOfKind) / slabs;
    p.image_tiles = (int)((rows * p.segs + per_tile - 1) / per_tile);
    p.tiles = (int)batch * p.image_tiles;
    auto share = [&](int blocks) {
        return (int)std::min<int64_t>(p.tiles, std::max(kXcds, 256 * blocks / nb / kXcds * kXcds));
    };
    c.wgs = share(c.blocks);
    c.wgs_small = share(std::max(1, c.blocks - 1));
    p.wgs = c.first_wg(c.n);
    return p;
}

int64_t pull_floats(const PullPlan &p, int slabs)
{
    return (int64_t)p.wgs * slabs * (p.chunks.blocks * 1024 + kBiasColumns);
}

// Channels of a launch: those of one full chunk (128; one slab: 64) where chunks in launches of their own, which use the whole chip one after the
// other, take less than chunks of about one size side by side, else all of them.
// Two slabs: a chunk of five to eight blocks takes 1.36, 1.54, 1.66 and 1.79 ms (2048 x 2048, 14 outputs), three 0.85 and one or two 0.56, so that full
// chunks and a small rest gain, a rest of six or more only in large images.  Time of a group of 14 (four in 3D) with all launches, side by side 1, over 9 / 10 / 13 / 14 / 16 / 17
// blocks: 512 x 513 0.95 / 0.97 / 1.05 / 1.12 / 1.11 / 0.94; 724 x 724 0.93 / 0.92 / 1.01 / 1.07 / 1.06 / 0.92; 960 x 960 0.90 / 0.89 / 0.99 / 1.03 / 1.02 / 0.87; 1500 x 1021
// 0.89 / 0.90 / 0.98 / 1.02 / 1.02 / 0.80; 64 x 66 x 65 over 9 / 10 / 11 / 13 0.91 / 0.91 / 0.86 / 1.02; 94^3 over 9 / 10 / 13 / 14 0.90 / 0.90 / 0.99 / 1.04; over 13 / 14 / 16 1448 x 1448
// 0.97 / 1.03 / 1.02, 2048 x 2048 0.94 / 1.00 / 1.00, 128^3 over 13 / 14 0.96 / 1.01.
// One slab: a chunk has at most four blocks, and its time goes with their number.  A launch per chunk gains where the chunks side by side would be of
// unequal size, five blocks most of all (4 + 1 for 3 + 2), the others only where gradients are written.  Side by side 1, a layer of three outputs (two
// in 3D) over 5 / 7 / 13 (unequal), 6 / 8 / 9 (equal) blocks: 512 x 513 0.93 / 1.07 / 1.23, 1.11 / 1.22 / 1.21; 724 x 724 0.98 / 1.13 / 1.17, 1.10 /
// 1.17 / 1.14; 900 x 900 0.89 / 1.01 / 1.04, 1.03 / 1.08 / 1.04; 1024 x 1024 0.80 / 0.92 / 0.93, 0.98 / 1.06 / 0.93; over 5 / 7, 6 / 9 80^3 0.92 / 1.09, 1.07 / 1.10, 128^3 0.78 / 0.91,
// 0.95 / 0.92; added to, a group of seven (two in 3D) over 5 / 7 / 11, 6 / 8 / 12: 724 x 724 0.99 / 1.02 / 1.04, 1.05 / 1.03 / 1.05; 1024 x 1024 0.91 / 0.99 / 0.98, 1.02 / 1.07 / 1.04;
// over 5 / 7 / 11 100^3 0.88 / 1.00 / 0.98, 128^3 0.86 / 0.96 / 0.94.
// Segments of a pass whose chunks have launches of their own (32 voxels each):
constexpr int64_t kAloneTenBlocks = 1 << 13, kAloneSmallRest = 14000, kAloneAnyRest = 1 << 16, kAloneOneSlab = 28000;
int64_t pull_channels(int64_t batch, int64_t rows, const PullPlan &p, int64_t channels, int slabs, bool fresh)
{
    const int64_t segments = batch * rows * p.segs, full = 16 * most_blocks(slabs);
    bool alone;
    if (slabs == 1) {
        const bool unequal = p.chunks.large < p.chunks.n, five = channels <= 5 * 16;
        alone = unequal && (fresh || five) && segments >= (fresh && five ? kAloneSmallRest : kAloneOneSlab);
    } else {
        alone = segments >= (channels <= 10 * 16 ? kAloneTenBlocks : channels % full <= 5 * 16 ? kAloneSmallRest : kAloneAnyRest);
    }
    return alone ? std::min(channels, full) : channels;
}
// Floats of the largest of the launches, whether the gradients are written or added to.
int64_t all_pull_floats(int64_t batch, int64_t rows, int64_t span, int64_t channels, int slabs)
{
    // (either kernel has as many workgroups where it is chosen by the voxels: fewer than tiles)
    const PullPlan p = pull_plan(batch, rows, span, channels, slabs);
    const int64_t step = pull_channels(batch, rows, p, channels, slabs, true), rest = channels % step;
    int64_t most = std::max(pull_floats(p, slabs), pull_floats(pull_plan(batch, rows, span, step, slabs), slabs));
    if (rest > 0) most = std::max(most, pull_floats(pull_plan(batch, rows, span, rest, slabs), slabs));
    return most;
}

}  // namespace
}  // namespace group2d

int64_t group_pull_floats(int64_t batch, int64_t rows, int64_t W, int64_t channels)
{
    using namespace group2d;
    // (volumes without gaps have fewer segments, and so no more workgroups)
    return std::max(all_pull_floats(batch, rows, W, channels, 1), all_pull_floats(batch, rows, W, channels, 2));
}

bool group_pull_supported(const Geom &g, const View<const float> &x, const View<float> &gx)
{
    using namespace group2d;
    const int64_t plane = (int64_t)(g.D - 1) * x.sz + (int64_t)(g.H - 1) * x.sy + g.W;
    const int span = form_of(g, x) == kFlat ? g.nvox : g.W;
    return x.sx == 1 && gx.sx == 1 && x.sb == gx.sb && x.sc == gx.sc && (g.ndim == 2 || x.sz == gx.sz) && x.sy == gx.sy &&
           span >= kSegment && x.sc < ((int64_t)1 << 26) && (g.ndim == 2 || x.sz < ((int64_t)1 << 26)) &&
           x.sy < ((int64_t)1 << 26) && plane < ((int64_t)1 << 26) &&
           (int64_t)g.B * g.D * g.H * ((g.W + kSegment - 1) / kSegment) < ((int64_t)1 << 30);
}

namespace {

// gy: the outputs' gradients, channels gsc apart, rows as in x.  fresh: the gradients are written, not added to (one slab;
// images, volumes without gaps).  gb: null where another launch forms the bias gradients.
hipError_t pull_part(const Geom &g, const View<const float> &x, const float *gy, int64_t gsb, int64_t gsc, const group2d::Outputs &out,
                     int update, int mask_from, const View<float> &grads, const int *channels, float *const *gk, float *gb, float *ws,
                     bool reverse, bool fresh, hipStream_t s)
{
    using namespace group2d;
    const int per_slab = g.ndim == 3 ? kSlabOut3d : kSlabOut;
    const Form form = form_of(g, x);
    const int slabs = out.n > per_slab ? 2 : 1;
    const int span = form == kFlat ? g.nvox : g.W, rows = g.nvox / span;
    const PullPlan p = pull_plan(g.B, rows, span, g.C, slabs, g.ndim == 3, g.ndim == 3 || fresh ? out.n : 0);
    PullArgs a{g.C, update, mask_from, g.D, g.H, g.W, span, p.segs, rows * p.segs, p.tiles, p.image_tiles, Divisor((uint32_t)p.segs),
               Divisor((uint32_t)p.image_tiles), Divisor((uint32_t)g.H), Divisor((uint32_t)g.W), reverse, 0, p.chunks,
               x.sb, x.sc, x.sz, x.sy, gsb, gsc, out};
    SumArgs sum;
    for (int o = 0; o < kMaxOut; o++) {
        if (o < out.n) a.dmax = std::max(a.dmax, out.dil[o]);
        sum.channels[o] = o < out.n ? channels[o] : 0;
        sum.gk[o] = o < out.n ? gk[o] : nullptr;
    }
    float *const bias_part = ws + (int64_t)p.wgs * slabs * p.chunks.blocks * 1024;
    hipError_t e = hipErrorInvalidConfiguration;
    const int blocks = p.chunks.blocks;
    auto launch = [&](auto f) {
        constexpr int N = decltype(f)::value;
        auto run = [&](auto g_, auto p_, auto fresh_) {
            constexpr int G = decltype(g_)::value, P = decltype(p_)::value;
            static LargeLds large;
            return pull_launch(&pull_rows<N, G, P, decltype(fresh_)::value>, kPullThreads, PullShape<G, P>::kLds, large, a, p.wgs, x.p, gy, grads.p, ws,
                               bias_part, s);
        };
        auto run_wide = [&](auto g_, auto p_, auto fresh_) {
            constexpr int G = decltype(g_)::value, P = decltype(p_)::value;
            static LargeLds large;
            return pull_launch(&pull_rows_wide<N, G, P, decltype(fresh_)::value>, kWaves * kWave, WideShape<G, P>::kLds, large, a, p.wgs, x.p, gy, grads.p,
                               ws, bias_part, s);
        };
        constexpr std::integral_constant<int, 1> one{};
        constexpr std::integral_constant<int, 2> two{};
        constexpr std::integral_constant<int, 4> four{};
        if constexpr (N != kVolume) {
            constexpr std::true_type yes{};
            if (fresh) return p.wide ? run_wide(one, two, yes) : blocks > 2 ? run(one, one, yes) : blocks > 1 ? run(one, two, yes) : run(one, four, yes);
        }
        constexpr std::false_type no{};
        if (slabs == 1) return p.wide ? run_wide(one, two, no) : blocks > 2 ? run(one, one, no) : blocks > 1 ? run(one, two, no) : run(one, four, no);
        if (p.wide) return run_wide(two, one, no);
        return blocks > 2 ? run(two, one, no) : run(two, two, no);
    };
    switch (form) {
    case kImage: e = launch(std::integral_constant<int, kImage>{}); break;
    case kVolume: e = launch(std::integral_constant<int, kVolume>{}); break;
    case kFlat: e = launch(std::integral_constant<int, kFlat>{}); break;
    }
    if (e != hipSuccess) return e;
    sum.chunks = p.chunks;
    sum.slabs = slabs;
    sum.columns = p.chunks.first_block(p.chunks.n) * 1024 * slabs;
    sum.stride = p.chunks.blocks * 1024 * slabs;
    sum.n = out.n;
    sum.fresh = fresh;
    sum.gb = gb;
    // (the last workgroup takes the biases)
    hipLaunchKernelGGL(g.ndim == 3 ? sum_group<kVolume> : sum_group<kImage>, dim3(sum.columns / kWave + (gb ? 1 : 0)), dim3(1024), 0, s, sum, ws, bias_part);
    return hipGetLastError();
}

hipError_t pull(const Geom &g, const View<const float> &x, const float *gy, int64_t gsb, int64_t gsc, const group2d::Outputs &out,
                int update, int mask_from, const View<float> &grads, const int *channels, float *const *gk, float *gb, float *ws,
                bool reverse, bool fresh, hipStream_t s)
{
    using namespace group2d;
    const int per_slab = g.ndim == 3 ? kSlabOut3d : kSlabOut;
    const Form form = form_of(g, x);
    if (out.n < 1 || out.n > 2 * per_slab || !group_pull_supported(g, x, grads) || (fresh && (form == kVolume || out.n > per_slab)))
        return hipErrorInvalidValue;
    const int slabs = out.n > per_slab ? 2 : 1, taps = g.ndim == 3 ? 27 : group2d::kTaps;
    const int span = form == kFlat ? g.nvox : g.W, rows = g.nvox / span;
    const int step = (int)pull_channels(g.B, rows, pull_plan(g.B, rows, span, g.C, slabs), g.C, slabs, fresh);
    for (int from = 0; from < g.C; from += step) {
        Geom part = g;
        View<const float> xp = x;
        View<float> gp = grads;
        Outputs op = out;
        int reads[kMaxOut];
        float *gkp[kMaxOut];
        part.C = std::min(step, g.C - from);
        xp.p += from * x.sc;
        gp.p += from * grads.sc;
        for (int o = 0; o < out.n; o++) {
            reads[o] = std::max(channels[o] - from, 0);
            if (from < update) op.k[o] += (int64_t)from * taps;      // (an output reads at least these; other weights are not needed)
            gkp[o] = reads[o] > 0 ? gk[o] + (int64_t)from * taps : gk[o];
        }
        const hipError_t e = pull_part(part, xp, gy, gsb, gsc, op, std::min(std::max(update - from, 0), part.C), mask_from - from, gp, reads,
                                       gkp, from == 0 ? gb : nullptr, ws, reverse, fresh, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

hipError_t group_pull(const Geom &g, const View<const float> &x, const group2d::Outputs &out, int update, int mask_from,
                      const View<float> &grads, int first, const int *channels, float *const *gk, float *gb,
                      float *ws, bool reverse, hipStream_t s)
{
    return pull(g, x, grads.p + (int64_t)first * grads.sc, grads.sb, grads.sc, out, update, mask_from, grads, channels, gk, gb, ws,
                reverse, false, s);
}

bool layer_pull_supported(const Geom &g, const View<const float> &x, const View<const float> &gy, const View<float> &gx)
{
    using namespace group2d;
    const bool rows = g.ndim == 3 ? form_of(g, x) == kFlat && form_of(g, gy) == kFlat : x.sy == gy.sy;
    return g.Wd <= (g.ndim == 3 ? kSlabOut3d : kSlabOut) && rows && gy.sx == 1 && gy.sc < ((int64_t)1 << 26) &&
           group_pull_supported(g, x, gx);
}

hipError_t layer_pull(const Geom &g, const View<const float> &x, const View<const float> &gy, const float *k, const View<float> &gx,
                      float *gk, float *gb, float *ws, hipStream_t s)
{
    group2d::Outputs out{};
    int channels[group2d::kSlabOut];
    float *gks[group2d::kSlabOut];
    const int64_t weights = (int64_t)g.C * (g.ndim == 3 ? 27 : group2d::kTaps);
    for (; out.n < g.Wd; out.n++) {
        out.dil[out.n] = g.dil;
        out.k[out.n] = k + out.n * weights;
        gks[out.n] = gk + out.n * weights;
        channels[out.n] = g.C;
    }
    return pull(g, x, gy.p, gy.sb, gy.sc, out, g.C, g.C, gx, channels, gks, gb, ws, false, true, s);
}

hipError_t group_finish_back(const Geom &g, const View<const float> &x, const View<float> &grads, int channel, int width,
                             const group2d::Outputs &above, hipStream_t s)
{
    using namespace group2d;
    const FinishArgs a = finish_args(g, x, above);
    const float *const act = x.p + (int64_t)channel * x.sc;
    float *const gp = grads.p + (int64_t)channel * grads.sc;
    if (g.ndim == 3) {
        auto launch = [&](auto form) {
            constexpr int N = decltype(form)::value;
            switch (width * 10 + above.n) {
            case 11: return finish_back_launch<N, 1, 1>(a, act, gp, s);
            case 12: return finish_back_launch<N, 2, 1>(a, act, gp, s);
            case 13: return finish_back_launch<N, 3, 1>(a, act, gp, s);
            case 21: return finish_back_launch<N, 1, 2>(a, act, gp, s);
            case 22: return finish_back_launch<N, 2, 2>(a, act, gp, s);
            }
            return hipErrorInvalidConfiguration;
        };
        return form_of(g, x) == kFlat ? launch(std::integral_constant<int, kFlat>{}) : launch(std::integral_constant<int, kVolume>{});
    } else if (width == 1) {
        switch (above.n) {
        case 1: return finish_back_launch<kImage, 1, 1>(a, act, gp, s);
        case 2: return finish_back_launch<kImage, 2, 1>(a, act, gp, s);
        case 3: return finish_back_launch<kImage, 3, 1>(a, act, gp, s);
        case 4: return finish_back_launch<kImage, 4, 1>(a, act, gp, s);
        case 5: return finish_back_launch<kImage, 5, 1>(a, act, gp, s);
        case 6: return finish_back_launch<kImage, 6, 1>(a, act, gp, s);
        case 7: return finish_back_launch<kImage, 7, 1>(a, act, gp, s);
        }
    } else if (width == 2) {
        switch (above.n) {
        case 1: return finish_back_launch<kImage, 1, 2>(a, act, gp, s);
        case 2: return finish_back_launch<kImage, 2, 2>(a, act, gp, s);
        case 3: return finish_back_launch<kImage, 3, 2>(a, act, gp, s);
        case 4: return finish_back_launch<kImage, 4, 2>(a, act, gp, s);
        case 5: return finish_back_launch<kImage, 5, 2>(a, act, gp, s);
        case 6: return finish_back_launch<kImage, 6, 2>(a, act, gp, s);
        }
    }
    return hipErrorInvalidConfiguration;
}

hipError_t group_spread_back_2d(const Geom &g, const View<const float> &x, const View<float> &grads, int channel, int channels,
                                int width, const group2d::Outputs &above, hipStream_t s)
{
    using namespace group2d;
    if (above.n < 1 || above.n > kSlabOut || channels > kMaxLower || width < 1 || width > 2 || channels < width) return hipErrorInvalidValue;
    FinishArgs a = finish_args(g, x, above);
    a.channels = channels;
    a.masked = channels - width;
    hipLaunchKernelGGL(spread_back, dim3(xcd_grid((a.items + 3) / 4)), dim3(256), 0, s, a, x.p + (int64_t)channel * x.sc,
                       grads.p + (int64_t)channel * grads.sc);
    return hipGetLastError();
}

}  // namespace msd
