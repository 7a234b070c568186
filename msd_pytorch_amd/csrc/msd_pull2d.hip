// Backward pass of a group of layers over the channels they share (msd_group.h).
//
// With A[m][v], m = (output o, tap t), the adjoint-form gather of the masked output gradients at
// voxel v (63 rows for seven outputs), both gradients are matrix products with the same matrix:
//     grad_input[c][v]  += sum_m k[m][c] * A[m][v],
//     grad_kernel[c][m] += sum_v x[c][v] * A[m][v].
// A wave owns 32 consecutive voxels of a row: it gathers their A into LDS once and then walks the
// channels in blocks of 16, lane (channel n, voxels 4 q .. 4 q + 3).  In that layout x is the
// second operand of the grad_kernel product as it is loaded, grad_input is the accumulator of the
// other product as it is loaded and as it is stored, and the activation that masks a finished
// channel is the x value in the same register.  The sums of grad_kernel stay in registers over all
// tiles of a workgroup; they leave as one row of partial sums per workgroup.
//
// Bound by the matrix cores and by memory about alike: per channel and voxel 128 multiply-adds
// (30 us per 16 channels at 1024 x 1024 and the clock they run at) and 12 bytes (40 us at the rate of
// a device copy), for seven layers at once, where passes of three layers move 28.  Seven layers at
// 1024 x 1024: 120 us over 20 channels, 186 over 48, 455 over 104 (2.9 TB/s; 118, 164 and 372 with the
// planes kept apart as the models do, csrc/host); three layers per pass of bwd_rows_fused took 112 (32
// channels), 157 (64) and 305 (over 96), two and a third of them for seven.
// Counters over the launches of a training step at 1024 x 1024, depth 100: 10.9 GB in 3.03 ms (3.6 TB/s), matrix
// cores busy 49 % of the time; at 2048 x 2048, two channels per layer: 4.2 TB/s.
// A step at 1024 x 1024, depth 100: 8.5 -> 6.7 ms (6.3 with the planes apart); 4 x 512 x 512: 8.0 -> 6.2;
// 2048 x 2048, two channels per layer, depth 200: 509 -> 319 (274).
//
// What it took to get there: a workgroup holds at most 64 channels (their sums, and a set of
// registers for x and grad_input of each block, asked for a whole tile ahead; 112 channels with two
// sets took 14 % longer); no test around loads or stores; the gather's loads in front of the last
// stores; the tiles at the row ends, whose gather takes twice the loads, shared out over the waves
// (200 -> 118 us over 20 channels: every 2048th tile of a row of 32 is the same end again).
#include "msd_group.h"

#include <algorithm>

namespace msd {
namespace group2d {
namespace {

constexpr int kPullWaves = 4;                     // per workgroup; two workgroups share a compute unit
constexpr int kTile = 32;                         // voxels of a wave
constexpr int kRowFloats = kTile + 4;             // of an LDS row of A (16 bytes apart in the banks)
constexpr int kMaxBlocks = 4;                     // blocks of 16 channels per workgroup: 16 sums per lane each
constexpr int kTriplesMax = 3 * kMaxOut;          // (output, tap row) pairs
constexpr int kBiasColumns = 8;

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));

// The channels' blocks of 16 are cut into n chunks: `large` chunks of `blocks` blocks, then chunks
// of one less.  A chunk has `wgs` workgroups (the smaller ones: `wgs_small`).
struct Chunks {
    int n, large, blocks, wgs, wgs_small;
    __host__ __device__ int size(int i) const { return i < large ? blocks : blocks - 1; }
    __host__ __device__ int rows(int i) const { return i < large ? wgs : wgs_small; }
    __host__ __device__ int first_block(int i) const { return i * blocks - (i > large ? i - large : 0); }
    __host__ __device__ int first_wg(int i) const { return i <= large ? i * wgs : large * wgs + (i - large) * wgs_small; }
};

struct PullArgs {
    int C, update;                                // channels of x; the first `update` of them have grad_input
    int mask_from;                                // channels from here on are masked with their activation
    int H, W, segs, items;                        // items: tiles (rows x segments x batch)
    int reverse;                                  // walk the tiles from the last to the first
    int dmax;
    Chunks chunks;
    int64_t sb, sc, sy;                           // strides of x and of the gradients
    Outputs out;
};

__device__ __forceinline__ float load1(uint64_t base, uint32_t off)
{
    float d[1];
    load_global_vec<1>(base, off, d);
    return d[0];
}

template <int NCB>
__global__ __launch_bounds__(kPullWaves *kWave, 2) void pull_rows(const PullArgs a, const float *__restrict__ x,
                                                                 const float *gy, float *gx,
                                                                 float *__restrict__ part,
                                                                 float *__restrict__ bias_part)
{
    extern __shared__ float lds[];
    f32x4_t *const table = reinterpret_cast<f32x4_t *>(lds);        // [block][4][lane]: weights of 4 rows m
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int n = lane % 16, q = lane / 16;
    float *const T = lds + NCB * 1024 + wave * (kRows * kRowFloats);
    const int bid = blockIdx.x, big = a.chunks.large * a.chunks.wgs;
    const int chunk = bid < big ? bid / a.chunks.wgs : a.chunks.large + (bid - big) / a.chunks.wgs_small;
    const int blocks = a.chunks.size(chunk), c0 = a.chunks.first_block(chunk) * 16;
    const int wgs = a.chunks.rows(chunk), wg = bid - a.chunks.first_wg(chunk);
    __shared__ int dils[kMaxOut + 1];
    if (tid < kMaxOut) dils[tid] = a.out.dil[tid];

    {   // the weights: row m of the product is a thread's own, every fourth channel
        const int m = tid % kRows, o = m / kTaps;
        const bool row = o < a.out.n;
        const float *const k = a.out.k[row ? o : 0] + m % kTaps;
        const int at = ((m / 16) * kWave + (m / 4 % 4) * 16) * 4 + m % 4;
#pragma unroll 4
        for (int c = tid / kRows; c < blocks * 16; c += kPullWaves) {
            const bool ok = row && c0 + c < a.update;
            const float w = k[(int64_t)(ok ? c0 + c : 0) * kTaps];
            lds[(c / 16) * 1024 + at + (c % 16) * 4] = ok ? w : 0.f;
        }
    }
    __syncthreads();

    struct Place {
        int x0, own0, y;                          // first voxel, first voxel that is its own, row
        uint64_t at;                              // byte offset of (image, row)
        int64_t img;                              // of the image
    };
    auto locate = [&](int t) {
        Place p;
        const int it0 = min(t, a.items - 1), it = a.reverse ? a.items - 1 - it0 : it0;
        const int row = it / a.segs;
        // (a wave comes back to the same segment where the row's segments divide its stride: turned by a
        // few with every round, so that the tiles at the ends of the rows are shared out)
        p.own0 = (it - row * a.segs + row * a.segs / (wgs * kPullWaves) * 5) % a.segs * kTile;
        p.x0 = min(p.own0, a.W - kTile);          // (the last tile of a row overlaps the one before)
        const int b = row / a.H;
        p.y = row - b * a.H;
        p.img = (int64_t)b * a.sb * 4;
        p.at = (uint64_t)(p.img + (int64_t)p.y * a.sy * 4);
        return p;
    };
    const uint32_t plane = (uint32_t)a.sc * 4u, nplane = (uint32_t)n * plane;
    // channels of block cb, voxels 16 s + 4 q ..  of the tile (past the last channel it is repeated)
    auto request = [&](const Place &p, int cb, f32x4_t (&xv)[2], f32x4_t (&gv)[2]) {
        const int ch = min(c0 + cb * 16, (a.C - 1) / 16 * 16);      // uniform
        const uint64_t base = p.at + (uint64_t)ch * (uint64_t)a.sc * 4u;
        uint64_t xb = reinterpret_cast<uint64_t>(x) + base, gb = reinterpret_cast<uint64_t>(gx) + base;
        int nn = n;
        asm volatile("" : "+v"(nn));             // (nothing of this is kept for every block over the tiles)
        uint32_t off = (uint32_t)min(nn, a.C - 1 - ch) * plane + 4u * (uint32_t)(p.x0 + 4 * q);
        // (scalar bases, and a lane offset that is formed here and not kept for every block)
        asm volatile("" : "+s"(xb), "+s"(gb), "+v"(off));
#pragma unroll
        for (int s = 0; s < 2; s++) {
            float v[4];
            load_global_vec4_unaligned(xb, off + 64u * s, v);
            xv[s] = f32x4_t{v[0], v[1], v[2], v[3]};
            load_global_vec4_unaligned(gb, off + 64u * s, v);
            gv[s] = f32x4_t{v[0], v[1], v[2], v[3]};
        }
    };

    float *const row = part + (int64_t)bid * (a.chunks.blocks * 1024);

    f32x4_t sums[NCB][kTiles];
#pragma unroll
    for (int cb = 0; cb < NCB; cb++)
#pragma unroll
        for (int t = 0; t < kTiles; t++) sums[cb][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;                             // lane (o, i): voxels 4 i .. 4 i + 3 of output o

    const int stride = wgs * kPullWaves;
    const int lb = block_for_xcd(wg, wgs, wgs % kXcds == 0);
    int tile = lb * kPullWaves + wave;
    Place here = locate(tile);
    f32x4_t xs[NCB][2], gs[NCB][2];               // a register set per block, asked for a whole tile ahead
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) request(here, cb, xs[cb], gs[cb]);
    // ---- the gather: lane (v, h) takes the triples (output, tap row) 2 i + h of voxel v.  Away from
    // the image's edges its loads are issued in the tile before, in front of that tile's last stores
    // and requests (all of them retire in order: behind those it would wait for memory).
    const int v = lane % kTile, h = lane / kTile;
    // triples (output, tap row) t0 (lanes h = 0) and t1 (h = 1) of a row away from the upper and
    // lower edges: plane and source row as a byte offset, dilation
    auto source = [&](int i, int y, uint32_t &at, int &d) {
        const int t0 = 2 * i, t1 = min(2 * i + 1, kTriplesMax - 1);
        const int o0 = min(t0 / 3, a.out.n - 1), o1 = min(t1 / 3, a.out.n - 1);
        const int e0 = a.out.dil[t0 / 3], e1 = a.out.dil[t1 / 3];
        const uint32_t r0 = (uint32_t)o0 * plane + 4u * (uint32_t)((y - (t0 % 3 - 1) * e0) * (int)a.sy);
        const uint32_t r1 = (uint32_t)o1 * plane + 4u * (uint32_t)((y - (t1 % 3 - 1) * e1) * (int)a.sy);
        at = h ? r1 : r0;
        d = h ? e1 : e0;
    };
    auto keep = [&](int i, bool own, const float (&val)[3]) {
        const int tri = 2 * i + h;        // (the 22nd stands for the row of zeros)
        const bool ok = own && tri < 3 * a.out.n;
#pragma unroll
        for (int r = 0; r < 3; r++)
            if (i < kTriplesMax / 2 || r == 0 || h == 0) T[(3 * tri + r) * kRowFloats + v] = ok ? val[r] : 0.f;
    };
    auto inside = [&](const Place &p) {           // uniform
        return p.x0 >= a.dmax && p.x0 + kTile + a.dmax <= a.W && p.y >= a.dmax && p.y + a.dmax < a.H;
    };
    float val[kTriplesMax / 2 + 1][3];
    auto gather = [&](const Place &p) {
        if (!inside(p)) return;
        const uint64_t base = reinterpret_cast<uint64_t>(gy) + (uint64_t)p.img;
        const uint32_t u = (uint32_t)(p.x0 + v);
#pragma unroll
        for (int i = 0; i <= kTriplesMax / 2; i++) {
            uint32_t at;
            int d;
            source(i, p.y, at, d);
            val[i][0] = load1(base, at + 4u * (u + d));
            val[i][1] = load1(base, at + 4u * u);
            val[i][2] = load1(base, at + 4u * (u - d));
        }
    };
    auto gathered = [&](const Place &p) {
        const int u = p.x0 + v, y = p.y;
        const bool own = u >= p.own0;
        const uint64_t base = reinterpret_cast<uint64_t>(gy) + (uint64_t)p.img;
        if (inside(p)) {
#pragma unroll
            for (int i = 0; i <= kTriplesMax / 2; i++) keep(i, own, val[i]);
        } else if (y >= a.dmax && y + a.dmax < a.H) {
#pragma unroll
            for (int i0 = 0; i0 <= kTriplesMax / 2; i0 += 4) {
                float val[4][5];
#pragma unroll
                for (int i = i0; i < i0 + 4 && i <= kTriplesMax / 2; i++) {
                    uint32_t at;
                    int d;
                    source(i, y, at, d);
                    // (adjoint_sources along x: one source inside the image, one mirrored at its edge)
                    val[i - i0][0] = load1(base, at + 4u * (uint32_t)(u + d < a.W ? u + d : u));
                    val[i - i0][1] = load1(base, at + 4u * (uint32_t)(u < d ? d - 1 - u : u));
                    val[i - i0][2] = load1(base, at + 4u * (uint32_t)u);
                    val[i - i0][3] = load1(base, at + 4u * (uint32_t)(u >= d ? u - d : u));
                    val[i - i0][4] = load1(base, at + 4u * (uint32_t)(u + d >= a.W ? 2 * a.W - 1 - d - u : u));
                }
#pragma unroll
                for (int i = i0; i < i0 + 4 && i <= kTriplesMax / 2; i++) {
                    const int d = h ? a.out.dil[min(2 * i + 1, kTriplesMax - 1) / 3] : a.out.dil[2 * i / 3];
                    const float(&w)[5] = val[i - i0];
                    const float s[3] = {(u + d < a.W ? w[0] : 0.f) + (u < d ? w[1] : 0.f), w[2],
                                        (u >= d ? w[3] : 0.f) + (u + d >= a.W ? w[4] : 0.f)};
                    keep(i, own, s);
                }
                __builtin_amdgcn_sched_barrier(0);    // (four triples at a time: registers)
            }
        } else {
#pragma unroll 2
            for (int i = 0; i <= kTriplesMax / 2; i++) {
                const int tri = 2 * i + h, o = min(tri / 3, a.out.n - 1), ky = tri % 3;
                const int d = dils[o];
                const uint32_t pl = (uint32_t)o * plane;
                // the sources of row y through tap ky and of voxel u through the outer tap columns
                // (adjoint_sources): one inside the image, one mirrored at its edge
                const int ra = y - (ky - 1) * d, rb = ky == 0 ? d - 1 - y : 2 * a.H - 1 - d - y;
                const bool oka = ra >= 0 && ra < a.H, okb = ky == 0 ? y < d : (ky == 2 && y + d >= a.H);
                const int xr = u + d, xrm = d - 1 - u, xl = u - d, xlm = 2 * a.W - 1 - d - u;
                const bool okr = xr < a.W, okrm = u < d, okl = u >= d, oklm = u + d >= a.W;
                float s[3] = {0.f, 0.f, 0.f};
#pragma unroll
                for (int z = 0; z < 2; z++) {
                    const bool ok = z ? okb : oka;
                    const uint32_t row = pl + 4u * (uint32_t)((ok ? (z ? rb : ra) : y) * (int)a.sy);
                    const float w0 = load1(base, row + 4u * (uint32_t)(okr ? xr : u));
                    const float w1 = load1(base, row + 4u * (uint32_t)(okrm ? xrm : u));
                    const float w2 = load1(base, row + 4u * (uint32_t)u);
                    const float w3 = load1(base, row + 4u * (uint32_t)(okl ? xl : u));
                    const float w4 = load1(base, row + 4u * (uint32_t)(oklm ? xlm : u));
                    s[0] += (ok && okr ? w0 : 0.f) + (ok && okrm ? w1 : 0.f);
                    s[1] += ok ? w2 : 0.f;
                    s[2] += (ok && okl ? w3 : 0.f) + (ok && oklm ? w4 : 0.f);
                }
                const bool ok = own && tri < 3 * a.out.n;
#pragma unroll
                for (int r = 0; r < 3; r++)
                    if (tri < kTriplesMax || r == 0) T[(3 * tri + r) * kRowFloats + v] = ok ? s[r] : 0.f;
            }
        }
    };
    gather(here);
    for (; tile < a.items; tile += stride) {
        gathered(here);
        // the tile is private to the wave and LDS executes a wave's accesses in order: only the
        // compiler has to be kept from reordering them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < 8 * kMaxOut) {                 // the bias gradient: the centre taps
            const f32x4_t c = *reinterpret_cast<const f32x4_t *>(T + (kTaps * (lane / 8) + 4) * kRowFloats + lane % 8 * 4);
            bsum += (c[0] + c[1]) + (c[2] + c[3]);
        }

        const Place next = locate(tile + stride);
        const int skip = here.own0 - here.x0;     // voxels of the tile that belong to the one before
        f32x4_t acc[kTiles];
        auto compute = [&](int cb, f32x4_t(&xv)[2], f32x4_t(&gv)[2]) {
            const int ch0 = c0 + cb * 16;
            if (skip > 0) {                       // uniform: an infinity there belongs to the other tile
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int e = 0; e < 4; e++) xv[s][e] = 16 * s + 4 * q + e >= skip ? xv[s][e] : 0.f;
            }
#pragma unroll
            for (int t = 0; t < kTiles; t++) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (cb < blocks) {                    // uniform
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    f32x4_t rv[kTiles];           // A[16 t + n][voxels 16 s + 4 q ..]
#pragma unroll
                    for (int t = 0; t < kTiles; t++)
                        rv[t] = *reinterpret_cast<const f32x4_t *>(T + (16 * t + n) * kRowFloats + 16 * s + 4 * q);
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int t = 0; t < kTiles; t++)
                            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[t][e], xv[s][e], acc[t], 0, 0, 0);
                }
                // Added to grad_input in two halves: a chain of 63 products that started from it would round
                // each of them to its size (2.7 times the error of passes of three layers, now 0.8 times).
                f32x4_t d[2];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const f32x4_t w = table[(cb * 4 + j) * kWave + lane];
                    float av[2][4];               // A[16 j + 4 q + e][voxel 16 s + n], whose weights are in w
#pragma unroll
                    for (int s = 0; s < 2; s++)
#pragma unroll
                        for (int e = 0; e < 4; e++) av[s][e] = T[(16 * j + 4 * q + e) * kRowFloats + 16 * s + n];
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        if (j % 2 == 0) d[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int s = 0; s < 2; s++)
                            d[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s][e], w[e], d[s], 0, 0, 0);
#pragma unroll
                    for (int s = 0; s < 2; s++)
                        if (j % 2 == 1) gv[s] += d[s];
                }
                if (ch0 + 16 > a.mask_from) {     // uniform
                    int nn = n;
                    asm volatile("" : "+v"(nn));
                    const bool open = ch0 + nn < a.mask_from;
#pragma unroll
                    for (int s = 0; s < 2; s++)
#pragma unroll
                        for (int e = 0; e < 4; e++) gv[s][e] = open || 0.f < xv[s][e] ? gv[s][e] : 0.f;
                }
            }
        };
        auto store = [&](int cb, const f32x4_t(&gv)[2]) {
            const int ch0 = c0 + cb * 16;
            // No test around the stores: loads and stores retire through one in-order counter, and
            // a store that may be skipped turns the wait for the next block's values, requested before
            // it, into one for the store itself.  Lanes with nothing to store write to the space of
            // their workgroup's partial sums, which are written last.
            const uint64_t base = reinterpret_cast<uint64_t>(gx) + here.at + (uint64_t)ch0 * (uint64_t)a.sc * 4u;
            uint32_t off = nplane + 4u * (uint32_t)(here.x0 + 4 * q);
            asm volatile("" : "+v"(off));
            int nn = n;
            asm volatile("" : "+v"(nn));
            uint32_t spare_off = 16u * threadIdx.x;
            asm volatile("" : "+v"(spare_off));
            const uint64_t spare = reinterpret_cast<uint64_t>(row) + spare_off;
            const bool channel = cb < blocks && nn < a.update - ch0;
            typedef __attribute__((address_space(1))) char *gbytes_t;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const uint64_t at = base + (off + 64u * s);
                const bool whole = channel && skip <= 16 * s + 4 * q;
                *reinterpret_cast<__attribute__((address_space(1))) f32x4u_t *>(whole ? at : spare) = gv[s];
            }
            if (skip % 4 != 0) {                  // uniform: some lanes own the last of their four voxels only
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    const int left = skip - (16 * s + 4 * q);
#pragma unroll
                    for (int e = 1; e < 4; e++)
                        if (channel && left > 0 && e >= left)
                            reinterpret_cast<__attribute__((address_space(1))) float *>(base + (off + 64u * s))[e] = gv[s][e];
                }
            }
        };
#pragma unroll
        for (int cb = 0; cb < NCB; cb++) {
            compute(cb, xs[cb], gs[cb]);
#pragma unroll
            for (int t = 0; t < kTiles; t++) {
                sums[cb][t] += acc[t];
                asm volatile("" : "+v"(sums[cb][t]));    // (added here and not at the end of the tile: registers)
            }
            if (cb + 1 == NCB) gather(next);
            store(cb, gs[cb]);
            __builtin_amdgcn_sched_barrier(0);    // (the scheduler would move the loads to where they are used)
            request(next, cb, xs[cb], gs[cb]);
            __builtin_amdgcn_sched_barrier(0);
        }
        here = next;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // the waves' sums, block by block, through the space of the A tiles
    float *const red = lds + NCB * 1024;
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) {
        if (cb < blocks) {                      // uniform
            __syncthreads();
#pragma unroll
            for (int t = 0; t < kTiles; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) red[wave * 1024 + (t * 4 + r) * kWave + lane] = sums[cb][t][r];
            __syncthreads();
            for (int i = tid; i < 1024; i += kPullWaves * kWave)
                row[cb * 1024 + i] = (red[i] + red[1024 + i]) + (red[2048 + i] + red[3072 + i]);
        }
    }
    if (chunk != 0) return;
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) bsum += __shfl_down(bsum, off, 8);
    __syncthreads();
    if (lane % 8 == 0) red[wave * 8 + lane / 8] = bsum;
    __syncthreads();
    if (tid < kBiasColumns)
        bias_part[wg * kBiasColumns + tid] = (red[tid] + red[8 + tid]) + (red[16 + tid] + red[24 + tid]);
}

struct SumArgs {
    Chunks chunks;
    int columns;                                  // weight columns in all (a multiple of 1024)
    int stride;                                   // of the rows of partial sums
    int n;
    int channels[kMaxOut];                        // input channels of each output
    float *gk[kMaxOut];
    float *gb;
};

// Adds the rows of partial sums, 64 columns per workgroup: 16 waves take every 16th row, their
// sums are added in order.  The last workgroup takes the biases.
__global__ __launch_bounds__(1024) void sum_group(const SumArgs a, const float *__restrict__ part,
                                                  const float *__restrict__ bias_part)
{
    __shared__ float lds[16 * kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = blockIdx.x * kWave + lane;
    const bool bias = (int)blockIdx.x * kWave >= a.columns;
    const int blk = col / 1024, big = a.chunks.large * a.chunks.blocks;
    const int chunk = blk < big ? blk / a.chunks.blocks
                                : (a.chunks.blocks > 1 ? a.chunks.large + (blk - big) / (a.chunks.blocks - 1) : 0);
    const int rows = a.chunks.rows(bias ? 0 : chunk);
    const float *p;
    int64_t stride;
    if (bias) {
        p = bias_part + lane % kBiasColumns;
        stride = kBiasColumns;
    } else {
        p = part + (int64_t)a.chunks.first_wg(chunk) * a.stride + (blk - a.chunks.first_block(chunk)) * 1024 + col % 1024;
        stride = a.stride;
    }
    float part_sum[4] = {0.f, 0.f, 0.f, 0.f};     // (short chains, then trees: these are the largest sums)
    for (int r = wave; r < rows; r += 128) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = p[min(r + 16 * i, rows - 1) * stride];
#pragma unroll
        for (int i = 0; i < 8; i++) part_sum[i % 4] += r + 16 * i < rows ? v[i] : 0.f;
    }
    lds[wave * kWave + lane] = (part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]);
    __syncthreads();
    if (wave != 0) return;
    float tree[16];
#pragma unroll
    for (int w = 0; w < 16; w++) tree[w] = lds[w * kWave + lane];
#pragma unroll
    for (int w = 8; w > 0; w /= 2)
#pragma unroll
        for (int i = 0; i < w; i++) tree[i] += tree[i + w];
    const float s = tree[0];
    if (bias) {
        if (lane < a.n) a.gb[lane] += s;
        return;
    }
    const int i = col % 1024, l = i % kWave;
    const int m = (i / 256) * 16 + (l / 16) * 4 + i / kWave % 4, o = m / kTaps;
    const int ch = col / 1024 * 16 + l % 16;
    if (o < a.n && ch < a.channels[o]) a.gk[o][(int64_t)ch * kTaps + m % kTaps] += s;
}

// grad_input of the NOUT channels that one layer of a group wrote, from the NQ outputs of the
// layers above it in the group, and the channels' ReLU mask: with it they are complete.
//
// One voxel per lane; the 9 NQ values come straight from the caches (a group's planes were written
// or read by the launches before), with no LDS and no barrier: the launch is bound by its ramp and
// by the vector cache.
struct FinishArgs {
    int H, W, segs, items, dmax;
    int64_t sb, sc, sy;
    int dil[kMaxOut];
    const float *k[kMaxOut];                      // of the first of the channels
};

template <int NQ, int NOUT>
__global__ __launch_bounds__(256) void finish_back(const FinishArgs a, const float *__restrict__ act, float *g)
{
    const int lb = block_for_xcd(blockIdx.x, gridDim.x, true);
    const int it = lb * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (it >= a.items) return;                    // uniform over the wave
    const int row = it / a.segs, xw = (it - row * a.segs) * kWave;
    const int b = row / a.H, y = row - b * a.H;
    const int u0 = xw + threadIdx.x % kWave, u = min(u0, a.W - 1);
    const uint64_t img = reinterpret_cast<uint64_t>(g) + (uint64_t)((int64_t)b * a.sb * 4);
    const uint64_t ximg = reinterpret_cast<uint64_t>(act) + (uint64_t)((int64_t)b * a.sb * 4);
    const uint32_t plane = (uint32_t)a.sc * 4u, here = 4u * (uint32_t)(y * (int)a.sy + u);
    float sum[NOUT], m[NOUT];
#pragma unroll
    for (int c = 0; c < NOUT; c++) {
        sum[c] = load1(img, (uint32_t)c * plane + here);
        m[c] = load1(ximg, (uint32_t)c * plane + here);
    }
    float A[NQ][9];
    if (xw >= a.dmax && xw + kWave + a.dmax <= a.W && y >= a.dmax && y + a.dmax < a.H) {      // uniform
#pragma unroll
        for (int o = 0; o < NQ; o++)
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                const int d = a.dil[o];
                const uint64_t base = img + (uint64_t)((NOUT + o) * plane) + (uint64_t)(4 * (int64_t)(y - (ky - 1) * d) * a.sy);
                A[o][3 * ky + 0] = load1(base, 4u * (uint32_t)(u + d));
                A[o][3 * ky + 1] = load1(base, 4u * (uint32_t)u);
                A[o][3 * ky + 2] = load1(base, 4u * (uint32_t)(u - d));
            }
    } else {
#pragma unroll
        for (int o = 0; o < NQ; o++) {
            const int d = a.dil[o];
            const AxisSources sx = adjoint_sources(u, a.W, d), sy = adjoint_sources(y, a.H, d);
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                float s[3] = {0.f, 0.f, 0.f};
#pragma unroll
                for (int z = 0; z < 2; z++) {
                    if (!sy.ok[ky][z]) continue;  // uniform
                    const uint64_t base = img + (uint64_t)((NOUT + o) * plane) + (uint64_t)(4 * (int64_t)sy.c[ky][z] * a.sy);
#pragma unroll
                    for (int r = 0; r < 3; r++)
#pragma unroll
                        for (int e = 0; e < 2; e++) {
                            if (r == 1 && e == 1) continue;
                            const float v = load1(base, 4u * (uint32_t)(sx.ok[r][e] ? sx.c[r][e] : u));
                            s[r] += sx.ok[r][e] ? v : 0.f;
                        }
                }
#pragma unroll
                for (int r = 0; r < 3; r++) A[o][3 * ky + r] = s[r];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NOUT; c++) {
        float all = 0.f;                          // (output by output, and added to grad_input last: see pull_rows)
#pragma unroll
        for (int o = 0; o < NQ; o++) {
            float one = 0.f;
#pragma unroll
            for (int t = 0; t < kTaps; t++) one += a.k[o][c * kTaps + t] * A[o][t];
            all += one;
        }
        sum[c] += all;
        const float v[1] = {0.f < m[c] ? sum[c] : 0.f};
        if (u0 < a.W) store_global_vec<1>(img, (uint32_t)c * plane + here, v);
    }
}

template <int NQ, int NOUT>
hipError_t finish_back_launch(const FinishArgs &a, const float *act, float *g, hipStream_t s)
{
    hipLaunchKernelGGL((finish_back<NQ, NOUT>), dim3(xcd_grid((a.items + 3) / 4)), dim3(256), 0, s, a, act, g);
    return hipGetLastError();
}

template <int NCB>
hipError_t pull_launch(const PullArgs &a, dim3 grid, size_t lds, const float *x, const float *gy, float *gx, float *part,
                       float *bias_part, hipStream_t s)
{
    static LargeLds large;
    const hipError_t e = large.allow(reinterpret_cast<const void *>(&pull_rows<NCB>), (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(pull_rows<NCB>, grid, dim3(kPullWaves * kWave), lds, s, a, x, gy, gx, part, bias_part);
    return hipGetLastError();
}

// Two workgroups per compute unit in all, shared out over the chunks by their size.
struct PullPlan {
    Chunks chunks;
    int segs, wgs;
    int64_t items;
};

PullPlan pull_plan(int64_t batch, int64_t H, int64_t W, int64_t channels)
{
    PullPlan p;
    const int nb = (int)((channels + 15) / 16);
    Chunks &c = p.chunks;
    c.n = (nb + kMaxBlocks - 1) / kMaxBlocks;
    c.blocks = (nb + c.n - 1) / c.n;
    c.large = nb - c.n * (c.blocks - 1);
    p.segs = (int)((W + kTile - 1) / kTile);
    p.items = batch * H * p.segs;
    const int64_t most = (p.items + kPullWaves - 1) / kPullWaves;
    auto share = [&](int blocks) { return (int)std::min<int64_t>(most, std::max(kXcds, 512 * blocks / nb / kXcds * kXcds)); };
    c.wgs = share(c.blocks);
    c.wgs_small = share(std::max(1, c.blocks - 1));
    p.wgs = c.first_wg(c.n);
    return p;
}

}  // namespace
}  // namespace group2d

int64_t group_pull_floats_2d(int64_t batch, int64_t H, int64_t W, int64_t channels)
{
    const group2d::PullPlan p = group2d::pull_plan(batch, H, W, channels);
    return (int64_t)p.wgs * (p.chunks.blocks * 1024 + group2d::kBiasColumns);
}

bool group_pull_supported_2d(const Geom &g, const View<const float> &x, const View<float> &gx)
{
    return g.ndim == 2 && x.sx == 1 && gx.sx == 1 && x.sb == gx.sb && x.sc == gx.sc && x.sy == gx.sy && g.W >= group2d::kTile &&
           x.sc < ((int64_t)1 << 26) && (int64_t)(g.H - 1) * x.sy + g.W < ((int64_t)1 << 26) &&
           (int64_t)g.B * g.H * ((g.W + group2d::kTile - 1) / group2d::kTile) < ((int64_t)1 << 30);
}

hipError_t group_pull_2d(const Geom &g, const View<const float> &x, const group2d::Outputs &out, int update, int mask_from,
                         const View<float> &grads, int first, const int *channels, float *const *gk, float *gb,
                         float *ws, bool reverse, hipStream_t s)
{
    using namespace group2d;
    if (out.n < 1 || out.n > kMaxOut || !group_pull_supported_2d(g, x, grads)) return hipErrorInvalidValue;
    const PullPlan p = pull_plan(g.B, g.H, g.W, g.C);
    PullArgs a{g.C, update, mask_from, g.H, g.W, p.segs, (int)p.items, reverse, 0, p.chunks, x.sb, x.sc, x.sy, out};
    SumArgs sum;
    for (int o = 0; o < kMaxOut; o++) {
        if (o < out.n) a.dmax = std::max(a.dmax, out.dil[o]);
        sum.channels[o] = o < out.n ? channels[o] : 0;
        sum.gk[o] = o < out.n ? gk[o] : nullptr;
    }
    float *const bias_part = ws + (int64_t)p.wgs * p.chunks.blocks * 1024;
    const float *const gy = grads.p + (int64_t)first * grads.sc;
    const dim3 grid(p.wgs);
    const size_t lds = ((size_t)p.chunks.blocks * 1024 + (size_t)kPullWaves * kRows * kRowFloats) * sizeof(float);
    hipError_t e = hipErrorInvalidConfiguration;
    switch (p.chunks.blocks) {
    case 1: e = pull_launch<1>(a, grid, lds, x.p, gy, grads.p, ws, bias_part, s); break;
    case 2: e = pull_launch<2>(a, grid, lds, x.p, gy, grads.p, ws, bias_part, s); break;
    case 3: e = pull_launch<3>(a, grid, lds, x.p, gy, grads.p, ws, bias_part, s); break;
    case 4: e = pull_launch<4>(a, grid, lds, x.p, gy, grads.p, ws, bias_part, s); break;
    }
    if (e != hipSuccess) return e;
    sum.chunks = p.chunks;
    sum.columns = p.chunks.first_block(p.chunks.n) * 1024;
    sum.stride = p.chunks.blocks * 1024;
    sum.n = out.n;
    sum.gb = gb;
    hipLaunchKernelGGL(sum_group, dim3(sum.columns / kWave + 1), dim3(1024), 0, s, sum, ws, bias_part);
    return hipGetLastError();
}

hipError_t group_finish_back_2d(const Geom &g, const View<const float> &x, const View<float> &grads, int channel, int width,
                                const group2d::Outputs &above, hipStream_t s)
{
    using namespace group2d;
    const int segs = (g.W + kWave - 1) / kWave;
    FinishArgs a{g.H, g.W, segs, g.B * g.H * segs, 0, x.sb, x.sc, x.sy, {}, {}};
    for (int o = 0; o < above.n; o++) {
        a.dil[o] = above.dil[o];
        a.k[o] = above.k[o];
        a.dmax = std::max(a.dmax, above.dil[o]);
    }
    const float *const act = x.p + (int64_t)channel * x.sc;
    float *const gp = grads.p + (int64_t)channel * grads.sc;
    if (width == 1) {
        switch (above.n) {
        case 1: return finish_back_launch<1, 1>(a, act, gp, s);
        case 2: return finish_back_launch<2, 1>(a, act, gp, s);
        case 3: return finish_back_launch<3, 1>(a, act, gp, s);
        case 4: return finish_back_launch<4, 1>(a, act, gp, s);
        case 5: return finish_back_launch<5, 1>(a, act, gp, s);
        case 6: return finish_back_launch<6, 1>(a, act, gp, s);
        }
    } else if (width == 2) {
        switch (above.n) {
        case 1: return finish_back_launch<1, 2>(a, act, gp, s);
        case 2: return finish_back_launch<2, 2>(a, act, gp, s);
        case 3: return finish_back_launch<3, 2>(a, act, gp, s);
        case 4: return finish_back_launch<4, 2>(a, act, gp, s);
        case 5: return finish_back_launch<5, 2>(a, act, gp, s);
        }
    }
    return hipErrorInvalidConfiguration;
}

}  // namespace msd
