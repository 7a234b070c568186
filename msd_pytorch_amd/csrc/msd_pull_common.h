// What pull_rows (msd_pull.hip) and pull_rows_wide (msd_pull_wide.h) share: the forms of a gather, the order of a slab's rows and their place in
// LDS, where a tile's segments lie, and how 16 channels of a unit of voxels cross memory.
#pragma once

#include "msd_group.h"
#include "msd_split.h"

namespace msd {
namespace group2d {
namespace {

constexpr int kSegment = 32;                      // voxels of a row that are gathered together
constexpr int kVoxelBytes = 2 * 64;               // of a voxel's rows of a slab in LDS
constexpr int kPartBytes = kSegment * kVoxelBytes;
constexpr int kSlabBytes = 3 * kPartBytes;
constexpr int kBiasColumns = 8;                   // per slab

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// What the kernels run over.  kFlat: a volume whose voxels lie without gaps, as one row: segments cross the
// ends of the rows, every lane has a row of its own.
enum Form { kImage = 2, kVolume = 3, kFlat = 4 };
template <int N> struct Gather {
    static constexpr bool kIsVolume = N != kImage;
    static constexpr int kTaps = kIsVolume ? 27 : group2d::kTaps;
    static constexpr int kLines = kTaps / 3;             // taps along x apart
    static constexpr int kOutputs = kIsVolume ? kSlabOut3d : kSlabOut;     // of a slab
    static constexpr int kLaneOut = kIsVolume ? 1 : 4;   // that a lane holds
};

// Row m of a slab's 64: the halves h = 0 and 1 of 32 are gathered apart.  A lane of a gatherer holds
// whole outputs (the folds at the image's edges move values between an output's rows).  2D: three of nine
// taps each, and of the seventh output, which both gather, five or four taps.  3D: one of 27.
struct Slot {
    int output, tap;                              // tap < 0: a row of zeros
};
template <int N> __host__ __device__ __forceinline__ Slot slot_of(int m)
{
    if (N != kImage) return Slot{m / 32, m % 32 < 27 ? m % 32 : -1};
    const int h = m / 32 % 2, s = m % 32, first = m / kRows * kSlabOut;
    if (s < 27) return Slot{first + 3 * h + s / kTaps, s % kTaps};
    const int tap = 5 * h + s - 27;
    return Slot{first + 6, tap < kTaps ? tap : -1};
}

// A voxel's rows lie in eight pieces of 16 bytes, piece i at i ^ turn(voxel): the 16 lanes that read one
// piece of 16 consecutive voxels, the 16 that write it and the 32 that read 16 rows of two times 4 voxels,
// 8 apart, transposed all meet the 64 banks once.
__device__ __forceinline__ uint32_t turn(uint32_t voxel) { return voxel / 2 % 2 * 2 + voxel / 8 % 2 * 4 + voxel / 4 % 2; }

// The channels' blocks of 16 are cut into n chunks: `large` chunks of `blocks` blocks, then chunks
// of one less.  A chunk has `wgs` workgroups (the smaller ones: `wgs_small`).
struct Chunks {
    int n, large, blocks, wgs, wgs_small;
    __host__ __device__ int size(int i) const { return i < large ? blocks : blocks - 1; }
    __host__ __device__ int rows(int i) const { return i < large ? wgs : wgs_small; }
    __host__ __device__ int first_block(int i) const { return i * blocks - (i > large ? i - large : 0); }
    __host__ __device__ int first_wg(int i) const { return i <= large ? i * wgs : large * wgs + (i - large) * wgs_small; }
};

// n / d for 0 <= n < 2^31 without a division.
struct Divisor {
    uint32_t magic;
    int shift;
    __host__ explicit Divisor(uint32_t d = 1) : shift(0)
    {
        while (((uint64_t)1 << shift) < d) shift++;
        magic = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << shift) - d)) / d + 1);
    }
    __device__ __forceinline__ int of(int n) const { return (int)((__umulhi((uint32_t)n, magic) + (uint32_t)n) >> shift); }
};

struct PullArgs {
    int C, update;                                // channels of x; the first `update` of them have grad_input
    int mask_from;                                // channels from here on are masked with their activation
    int D, H, W, span, segs, items;               // voxels of a row of segments (kFlat: of all); segments of one, of an image
    int tiles, image_tiles;                       // of all images, of one
    Divisor by_segs, by_tiles, by_rows, by_voxels;        // by_rows: rows of a slice; by_voxels: of a row
    int reverse;                                  // walk the tiles from the last to the first
    int dmax;
    Chunks chunks;
    int64_t sb, sc, sz, sy;                       // strides of x and of grad_input
    int64_t gsb, gsc;                             // of the outputs' gradients (their rows lie as those of x)
    Outputs out;
};

__device__ __forceinline__ float load1(uint64_t base, uint32_t off)
{
    float d[1];
    load_global_vec<1>(base, off, d);
    return d[0];
}

// The sources of one voxel (or row) u of an axis of n through the outer taps of dilation d
// (adjoint_sources): `up` is read by tap 0 where it lies inside and is otherwise the mirrored source of
// tap 2, `down` the other way round, so that two loads hold all of them.
struct Sides {
    int up, down;
    bool up_in, down_in;
};
__device__ __forceinline__ Sides sides(int u, int n, int d)
{
    Sides s;
    s.up_in = u + d < n;
    s.down_in = u >= d;
    s.up = s.up_in ? u + d : 2 * n - 1 - d - u;
    s.down = s.down_in ? u - d : d - 1 - u;
    return s;
}
__device__ __forceinline__ void fold(const Sides &s, float &tap0, float &tap2)
{
    const float up = tap0, down = tap2;
    tap0 = (s.up_in ? up : 0.f) + (s.down_in ? 0.f : down);
    tap2 = (s.down_in ? down : 0.f) + (s.up_in ? 0.f : up);
}

// ---- a workgroup's tiles: kSegs consecutive segments of an image each
struct Tile {
    int first;                                    // segment of its image
    int64_t img, gimg;                            // byte offsets of the image, of the outputs' gradients
    uint32_t sign;                                // of x in this tile
};
struct Place {
    int x0, skip, y, z;                           // first voxel, voxels that belong to the segment before, row, slice
    bool valid;
};
// (past the last tile that one again)
template <int kSegs> __device__ __forceinline__ Tile tile_at(const PullArgs &a, int tile)
{
    Tile t;
    const int it0 = min(tile, a.tiles - 1), it = a.reverse ? a.tiles - 1 - it0 : it0;
    const int b = a.by_tiles.of(it);
    t.first = (it - b * a.image_tiles) * kSegs;
    t.img = (int64_t)b * a.sb * 4;
    t.gimg = (int64_t)b * a.gsb * 4;
    t.sign = (uint32_t)it << 31;
    return t;
}
template <int N> __device__ __forceinline__ Place place_at(const PullArgs &a, const Tile &t, int segment)
{
    Place p;
    p.valid = t.first + segment < a.items;
    const int it = min(t.first + segment, a.items - 1);
    p.y = a.by_segs.of(it);
    const int own0 = (it - p.y * a.segs) * kSegment;
    p.z = N == kVolume ? a.by_rows.of(p.y) : 0;
    p.y -= N == kVolume ? p.z * a.H : 0;
    p.x0 = min(own0, a.span - kSegment);          // (the last segment of a row overlaps the one before)
    p.skip = p.valid ? own0 - p.x0 : kSegment;
    return p;
}

// Rows m of a lane or a wave (slot_of), eight at a time.
template <int N> __device__ __forceinline__ void eight_rows(const float (&val)[Gather<N>::kLaneOut][Gather<N>::kLines][3], int h, int i, float (&e8)[8])
{
    constexpr int kTaps = Gather<N>::kTaps;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int s = 8 * i + e;
        if (s < 27) {
            e8[e] = val[s / kTaps][s % kTaps / 3][s % 3];
        } else if constexpr (N != kImage) {
            e8[e] = 0.f;
        } else {
            const int t0 = s - 27, t1 = s - 22;
            e8[e] = h ? (t1 < kTaps ? val[3][t1 / 3 % 3][t1 % 3] : 0.f) : val[3][t0 / 3][t0 % 3];
        }
    }
}

// ---- 16 channels of a unit of 16 kVec voxels: lane (channel lane / (4 kVec) + 16 / kVec i, four voxels lane % (4 kVec))
struct Unit {
    int64_t img;                                  // byte offset of the image
    uint32_t at;                                  // the lane's of (row, voxel)
    int skip;                                     // first of its four voxels that is its segment's own (0: all, 4: none)
};
// channels from `limit` on: that channel before it again
template <int kVec>
__device__ __forceinline__ void request_unit(const float *from, int ch0, int limit, uint32_t plane, uint32_t lane_plane, const Unit &un, f32x4_t (&d)[kVec])
{
    uint64_t base = reinterpret_cast<uint64_t>(from) + (uint64_t)un.img + (uint64_t)min(ch0, limit - 1) * plane;
    asm volatile("" : "+s"(base));               // (scalar base, 32-bit lane offsets)
    const uint32_t last = (uint32_t)min(max(limit - 1 - ch0, 0), 15) * plane;
    uint32_t at = lane_plane;
    asm volatile("" : "+v"(at));                 // (nothing of this is kept over the tiles)
#pragma unroll
    for (int i = 0; i < kVec; i++) {
        float v4[4];
        load_global_vec_unaligned<4>(base, min(at + (uint32_t)(16 / kVec * i) * plane, last) + un.at, v4);
        d[i] = f32x4_t{v4[0], v4[1], v4[2], v4[3]};
    }
}
// An infinity in the voxels of another segment belongs to that one.
template <int kVec> __device__ __forceinline__ void clear_skipped(const Unit &un, f32x4_t (&xs)[kVec])
{
    if (__any(un.skip > 0)) {
#pragma unroll
        for (int i = 0; i < kVec; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) xs[i][e] = e >= un.skip ? xs[i][e] : 0.f;
    }
}
// Channels below `limit`; all: else none.
template <int kVec>
__device__ __forceinline__ void store_unit(float *gx, int ch0, int limit, uint32_t plane, uint32_t lane_plane, int lc, const Unit &un, const f32x4_t (&gs)[kVec],
                                           bool all)
{
    // Buffer stores, whose lanes past the end of the buffer store nothing: there is no branch around
    // them.  (Loads and stores retire through one in-order counter, and a store that may be skipped turns the
    // wait for the next unit's values, requested before it, into one for the store itself.)
    constexpr int kChannels = 16 / kVec;          // of one access
    const uint64_t base = reinterpret_cast<uint64_t>(gx) + (uint64_t)un.img + (uint64_t)ch0 * plane;
    uint32_t at = lane_plane;
    asm volatile("" : "+v"(at));
    const int end = un.skip == 0 && all ? limit - ch0 : 0;
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(base), 0, 0xfffffff0u, 0x00020000);
#pragma unroll
    for (int i = 0; i < kVec; i++) {
        typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
        const uint32_t plane_at = at + (uint32_t)(kChannels * i) * plane;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, gs[i]), to, lc + kChannels * i < end ? plane_at + un.at : 0xffffffffu, 0, 0);
    }
    if (__any(un.skip % 4 != 0)) {                // some lanes own the last of their four voxels only
#pragma unroll
        for (int i = 0; i < kVec; i++)
#pragma unroll
            for (int e = 1; e < 4; e++)
                if (all && lc + kChannels * i < limit - ch0 && un.skip > 0 && e >= un.skip)
                    reinterpret_cast<__attribute__((address_space(1))) float *>(base + (uint64_t)(lane_plane + (uint32_t)(kChannels * i) * plane) + un.at)[e] = gs[i][e];
    }
}

}  // namespace
}  // namespace group2d
}  // namespace msd
