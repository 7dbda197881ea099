// Binned 3D backprojection of the significant slices: the scatter of
// MyBackProjector::backproject (src/reconstruct.cpp:977-1164) reorganised so that the trilinear
// corner updates land in LDS instead of the HBM grids.
//
//   k_post  : per slice s = task * NOR + o, the weighted sum of the shifted unmasked images
//             V_s(p) = sum_t w_t/sumw * Minv CTF X_nomask(p) S_t(p) (float2 [S][Pf]) and
//             W_s = sum_t w_t/sumw (double [S]; 0: the slice has no significant sample).
//   count   : every (slice, pixel) with a positive weight, inside r_max -> trilinear base voxel ->
//             brick (16x8x4 base voxels of one class grid); counts per brick, first gathered per
//             block in an LDS hash table (one global atomic per distinct brick of the block).
//   scan    : exclusive prefix sums of the counts and of the chunks (kChunk records) per brick, the brick of
//             every chunk.
//   fill    : records (slice << 32 | pixel) grouped by brick; ranges reserved per distinct brick
//             of the block as in count.
//   brick   : one block per chunk of a brick's records (bricks near the origin, crossed by nearly
//             every slice, hold hundreds of thousands): the records' 8 corners accumulate in a
//             17x9x5 LDS box (base voxels plus the +1 corner halo), then each non-zero voxel goes to
//             the grids with one atomic per component.  Corner weights and values are computed
//             exactly as the direct scatter computes them; only the order of the FP32 additions
//             differs.
//
// 2D grids are small and every slice of a class covers the whole disc: k_bp_band accumulates a band of
// grid rows of one class in LDS and needs no records.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "device_util.h"
#include "kernels.h"

namespace rome {

namespace {

constexpr int kBoxX = kBrickX + 1, kBoxY = kBrickY + 1, kBoxZ = kBrickZ + 1, kBox3 = kBoxX * kBoxY * kBoxZ;
constexpr unsigned kChunk = 1024;  // records per brick block (or per round of one, where it takes a whole brick)
constexpr int kHash = 512;         // LDS hash slots for the <= 256 bricks of one count / fill block

// Slot of brick b in the block's hash table (keys b + 1, 0 = empty; linear probing).  At most 256
// keys go into 512 slots, so a free slot always exists.
DEV int hash_slot(unsigned* keys, unsigned b) {
    int h = (int)((b * 2654435761u) >> 23);  // 9 bits
    for (;;) {
        const unsigned k = keys[h];
        if (k == b + 1) return h;
        if (k == 0) {
            const unsigned old = atomicCAS(&keys[h], 0u, b + 1);
            if (old == 0 || old == b + 1) return h;
        }
        h = (h + 1) & (kHash - 1);
    }
}

struct Sample {
    Coords c;
    int k;
    float wgt;
};

// The pixel's contribution geometry, or false when the direct scatter would skip it.
DEV bool bp_sample(const BpArgs& a, long long s, int p, Sample& out) {
    const double wsl = a.slice_w[s];
    if (!(wsl > 0.)) return false;
    const unsigned q = (unsigned)s / (unsigned)a.NOR;  // slices are counted in 32 bits (records hold them so)
    const int o = (int)((unsigned)s - q * (unsigned)a.NOR);
    const int img = a.task_img[q], m = a.task_m[q];
    const int xy = a.f_xy[p];
    const int x = px_x(xy), y = px_y(xy);
    if (x * x + y * y > a.r_max * a.r_max) return false;
    const float wgt = (float)((double)a.MC2bp[(size_t)img * a.Pf + p] * wsl);
    if (!(wgt > 0.f)) return false;
    const int r = m % a.R;
    out.k = m / a.R;
    out.c = map_coords(a.Ai_fine + 6 * ((size_t)r * a.NOR + o), x, y, a.c, true);
    out.wgt = wgt;
    return true;
}

// brick of the base voxel: class-major, then z, y, x in bricks of 4, 8 and 16 (grid coordinates are >= 0)
DEV int brick_of(const BpArgs& a, const Sample& sm) {
    const int bx = sm.c.x0 / kBrickX, by = sm.c.y0 / kBrickY, bz = sm.c.z0 / kBrickZ;
    return sm.k * a.nb_class + (bz * a.nby + by) * a.nbx + bx;
}

// Slices of the pool: the host's count, or (device-driven pools) the device task total x NOR; 0 when
// the pool is aborted or its slices exceed the slice buffer (the direct scatter took it).
DEV long long bp_slices(const BpArgs& a, long long S_host) {
    if (!a.ntask_dev) return S_host;
    if (*a.abort) return 0;
    const long long S = *a.ntask_dev * a.NOR;
    return S > a.slice_cap ? 0 : S;
}

DEV void bp_count_one(const BpArgs& a, long long s, int pb, unsigned* keys, unsigned* cnt) {
    if (!(a.slice_w[s] > 0.)) return;  // a slice without weight has no record (whole block)
    for (int h = threadIdx.x; h < kHash; h += blockDim.x) {
        keys[h] = 0u;
        cnt[h] = 0u;
    }
    __syncthreads();
    const int p = pb * blockDim.x + threadIdx.x;
    Sample sm;
    if (p < a.Pf && bp_sample(a, s, p, sm)) atomicAdd(&cnt[hash_slot(keys, (unsigned)brick_of(a, sm))], 1u);
    __syncthreads();
    for (int h = threadIdx.x; h < kHash; h += blockDim.x)
        if (keys[h]) atomicAdd(&a.count[keys[h] - 1], cnt[h]);
}

// blockIdx.x = slice, blockIdx.y = pixel block; device-driven (Q): a fixed grid of the same shape whose
// blocks stride over the slices of the slice total on the device.  No work counter: a device-scope
// atomic on one address serialises about a million items a pool.
template <bool Q>
__global__ __launch_bounds__(256) void k_bp_count(BpArgs a, long long S_host) {
    __shared__ unsigned keys[kHash], cnt[kHash];
    if constexpr (!Q) {
        bp_count_one(a, blockIdx.x, blockIdx.y, keys, cnt);
        return;
    }
    const long long S = bp_slices(a, S_host);
    for (long long sl = blockIdx.x; sl < S; sl += gridDim.x) {  // slices strided over the grid
        bp_count_one(a, sl, (int)blockIdx.y, keys, cnt);
        __syncthreads();  // the hash table of the next slice
    }
}

// Exclusive scans of count[0..nb) into off[0..nb] and of the chunks per brick into coff[0..nb], the brick of every
// chunk into ck_brick, cursor cleared: k_bp_sums leaves the totals of blocks of 1024 bricks, each block of k_bp_scan adds
// up the totals before its own and scans its bricks.  (One block over all bricks, tile by tile: 78 us for 74 k bricks,
// 10 us now.)
constexpr int kScanBlock = 1024;  // bricks and threads per block
DEV unsigned bp_chunks(unsigned c, unsigned chunk) { return c / chunk + (c % chunk ? 1u : 0u); }
__global__ __launch_bounds__(kScanBlock) void k_bp_sums(const unsigned* __restrict__ count, int nb, unsigned chunk,
                                                        unsigned* __restrict__ sums) {
    __shared__ unsigned red[kScanBlock / 64];
    const int b = blockIdx.x * kScanBlock + threadIdx.x;
    const unsigned c = b < nb ? count[b] : 0u;
    const unsigned t = block_reduce(c, [](unsigned x, unsigned y) { return x + y; }, red);
    const unsigned ct = block_reduce(bp_chunks(c, chunk), [](unsigned x, unsigned y) { return x + y; }, red);
    if (threadIdx.x == 0) {
        sums[2 * blockIdx.x] = t;
        sums[2 * blockIdx.x + 1] = ct;
    }
}

__global__ __launch_bounds__(kScanBlock) void k_bp_scan(const unsigned* __restrict__ count, int nb, unsigned chunk,
                                                        const unsigned* __restrict__ sums, unsigned* __restrict__ off,
                                                        unsigned* __restrict__ coff, unsigned* __restrict__ cursor,
                                                        unsigned* __restrict__ ck_brick) {
    constexpr int NW = kScanBlock / 64;
    __shared__ unsigned wa[NW], wc[NW], red[NW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, b = blockIdx.x * kScanBlock + tid;
    unsigned pre = 0u, cpre = 0u;  // of the blocks before
    for (int q = tid; q < (int)blockIdx.x; q += kScanBlock) {
        pre += sums[2 * q];
        cpre += sums[2 * q + 1];
    }
    const unsigned c = b < nb ? count[b] : 0u, cc = bp_chunks(c, chunk);
    pre = block_reduce(pre, [](unsigned x, unsigned y) { return x + y; }, red);
    cpre = block_reduce(cpre, [](unsigned x, unsigned y) { return x + y; }, red);
    unsigned in = c, cin = cc;
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned v = __shfl_up(in, o, 64), cv = __shfl_up(cin, o, 64);
        if (lane >= o) {
            in += v;
            cin += cv;
        }
    }
    if (lane == 63) {
        wa[wid] = in;
        wc[wid] = cin;
    }
    __syncthreads();
    for (int w = 0; w < wid; ++w) {
        pre += wa[w];
        cpre += wc[w];
    }
    if (b >= nb) return;
    const unsigned o0 = pre + in - c, c0 = cpre + cin - cc;
    off[b] = o0;
    coff[b] = c0;
    cursor[b] = 0u;
    for (unsigned q = 0; q < cc; ++q) ck_brick[c0 + q] = (unsigned)b;
    if (b == nb - 1) {
        off[nb] = o0 + c;
        coff[nb] = c0 + cc;
    }
}

DEV void bp_fill_one(const BpArgs& a, long long s, int pb, unsigned* keys, unsigned* cnt, unsigned* base) {
    if (!(a.slice_w[s] > 0.)) return;  // a slice without weight has no record (whole block)
    for (int h = threadIdx.x; h < kHash; h += blockDim.x) {
        keys[h] = 0u;
        cnt[h] = 0u;
    }
    __syncthreads();
    const int p = pb * blockDim.x + threadIdx.x;
    Sample sm;
    int h = -1;
    unsigned rank = 0;
    if (p < a.Pf && bp_sample(a, s, p, sm)) {
        h = hash_slot(keys, (unsigned)brick_of(a, sm));
        rank = atomicAdd(&cnt[h], 1u);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < kHash; q += blockDim.x)
        if (keys[q]) base[q] = a.off[keys[q] - 1] + atomicAdd(&a.cursor[keys[q] - 1], cnt[q]);
    __syncthreads();
    if (h >= 0) a.rec[base[h] + rank] = ((unsigned long long)s << 32) | (unsigned)p;
}

template <bool Q>
__global__ __launch_bounds__(256) void k_bp_fill(BpArgs a, long long S_host) {
    __shared__ unsigned keys[kHash], cnt[kHash], base[kHash];
    if constexpr (!Q) {
        bp_fill_one(a, blockIdx.x, blockIdx.y, keys, cnt, base);
        return;
    }
    const long long S = bp_slices(a, S_host);
    for (long long sl = blockIdx.x; sl < S; sl += gridDim.x) {  // slices strided over the grid
        bp_fill_one(a, sl, (int)blockIdx.y, keys, cnt, base);
        __syncthreads();  // the hash table of the next slice
    }
}

// One chunk of a brick's records without floating-point atomics: the records are counting-sorted by
// base voxel in LDS, each thread sums the 8 corner contributions of the records of its base voxels in
// registers, then the corners are added to the box in 8 passes, one corner offset per pass, in which
// distinct base voxels reach distinct box voxels.
// WHOLE: all of a brick's records, 1024 a round, so that a voxel is one running FP32 sum whatever the number of images:
// around the origin hundreds of equal weights meet, whose rounding does not average out, and split sums were 1.8e-7
// away from the direct scatter's (400 images of 100^2: 88 -> 142 us).
template <bool WHOLE>
DEV void bp_brick_one(const BpArgs& a, unsigned ck) {
    constexpr int kVox = kBrickX * kBrickY * kBrickZ;  // base voxels of a brick
    static_assert(kVox == 512, "two base voxels a thread, eight a lane of the scan");
    // exactly 32 KB: five blocks per CU.  The records' fx, fy, fz, value re, value im (mirror applied) and weight; the
    // box once they are summed.
    __shared__ float rec_f[6][kChunk];
    __shared__ unsigned vcnt[kVox], voff[kVox];
    __shared__ unsigned short order[kChunk], vox[kChunk];
    typedef float Box[kBox3];
    Box* box = reinterpret_cast<Box*>(&rec_f[0][0]);
    static_assert(3 * kBox3 <= 6 * kChunk, "the box takes the records' place");
    const int tid = threadIdx.x;
    const int b = (int)a.ck_brick[ck];
    const unsigned r0 = a.off[b] + (ck - a.coff[b]) * kChunk;
    const unsigned r1 = WHOLE ? a.off[b + 1] : min(a.off[b + 1], r0 + kChunk);
    if (r0 >= r1) return;
    const int k = b / a.nb_class;
    const int rem = b - k * a.nb_class;
    const int bx = rem % a.nbx, by = (rem / a.nbx) % a.nby, bz = rem / (a.nbx * a.nby);
    float acc[2][8][3];  // per base voxel (this thread: tid and tid + 256): sums of the 8 corner contributions
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) acc[h][cc][0] = acc[h][cc][1] = acc[h][cc][2] = 0.f;
    unsigned q0 = r0;
    do {
        const int n = (int)min(r1 - q0, kChunk);
        for (int v = tid; v < kVox; v += blockDim.x) vcnt[v] = 0u;
        __syncthreads();
        // records -> LDS (geometry and values), base voxel histogram
        for (int i = tid; i < n; i += blockDim.x) {
            const unsigned long long rc = a.rec[q0 + i];
            const long long s = (long long)(rc >> 32);
            const int p = (int)(rc & 0xffffffffu);
            Sample sm;
            bp_sample(a, s, p, sm);  // true: the record was made from the same test
            const Coords& c = sm.c;
            const float2 v = a.slice_val[(size_t)s * a.Pf + p];
            const int lx = c.x0 - bx * kBrickX, ly = c.y0 - by * kBrickY, lz = c.z0 - bz * kBrickZ;
            const int lv = (lz * kBrickY + ly) * kBrickX + lx;
            vox[i] = (unsigned short)lv;
            rec_f[0][i] = c.fx;
            rec_f[1][i] = c.fy;
            rec_f[2][i] = c.fz;
            rec_f[3][i] = v.x;
            rec_f[4][i] = c.neg ? -v.y : v.y;
            rec_f[5][i] = sm.wgt;
            atomicAdd(&vcnt[lv], 1u);
        }
        __syncthreads();
        if (tid < 64) {  // exclusive scan of the 512 counts by one wave, 8 per lane
            unsigned loc[8], sum = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                loc[q] = vcnt[tid * 8 + q];
                sum += loc[q];
            }
            unsigned incl = sum;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const unsigned o = __shfl_up(incl, d, 64);
                if (tid >= d) incl += o;
            }
            unsigned run = incl - sum;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                voff[tid * 8 + q] = run;
                vcnt[tid * 8 + q] = run;  // becomes the scatter cursor
                run += loc[q];
            }
        }
        __syncthreads();
        for (int i = tid; i < n; i += blockDim.x) order[atomicAdd(&vcnt[vox[i]], 1u)] = (unsigned short)i;
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int lv = tid + 256 * h;
            const unsigned je = lv + 1 < kVox ? voff[lv + 1] : (unsigned)n;
            for (unsigned j = voff[lv]; j < je; ++j) {
                const int i = order[j];
                const float fx = rec_f[0][i], fy = rec_f[1][i], fz = rec_f[2][i];
                const float vr = rec_f[3][i], vi = rec_f[4][i], w = rec_f[5][i];
                const float mfx = 1.f - fx, mfy = 1.f - fy, mfz = 1.f - fz;
                const float dd[8] = {mfz * mfy * mfx, mfz * mfy * fx, mfz * fy * mfx, mfz * fy * fx,
                                     fz * mfy * mfx, fz * mfy * fx, fz * fy * mfx, fz * fy * fx};
#pragma unroll
                for (int cc = 0; cc < 8; ++cc) {
                    acc[h][cc][0] += dd[cc] * vr;
                    acc[h][cc][1] += dd[cc] * vi;
                    acc[h][cc][2] += dd[cc] * w;
                }
            }
        }
        __syncthreads();  // the records of the next round, or the box in their place
        q0 += kChunk;
    } while (WHOLE && q0 < r1);
    for (int v = tid; v < 3 * kBox3; v += blockDim.x) (&box[0][0])[v] = 0.f;
    __syncthreads();
#pragma unroll
    for (int cc = 0; cc < 8; ++cc) {
        const int dz = cc >> 2, dy = (cc >> 1) & 1, dx = cc & 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int lv = tid + 256 * h;
            const int lx = lv % kBrickX, ly = lv / kBrickX % kBrickY, lz = lv / (kBrickX * kBrickY);
            const int idx = ((lz + dz) * kBoxY + (ly + dy)) * kBoxX + (lx + dx);
            box[0][idx] += acc[h][cc][0];
            box[1][idx] += acc[h][cc][1];
            box[2][idx] += acc[h][cc][2];
        }
        __syncthreads();
    }
    float* gd = a.bp_data + a.grid_stride * 2 * k;
    float* gw = a.bp_weight + a.grid_stride * k;
    // to the grids: re and im in neighbouring lanes, as they lie there, so that one instruction's atomics fill their lines
    auto voxel = [&](int v, size_t& idx) {
        const int lx = v % kBoxX, ly = v / kBoxX % kBoxY, lz = v / (kBoxX * kBoxY);
        const int gx = bx * kBrickX + lx, gy = by * kBrickY + ly, gz = bz * kBrickZ + lz;
        idx = ((size_t)gz * a.pad + gy) * a.padF + gx;
        return gx < a.padF && gy < a.pad && gz < a.pad;  // else nothing lands there (zero)
    };
    size_t idx;
    for (int u = tid; u < 2 * kBox3; u += blockDim.x) {
        const float d = box[u & 1][u >> 1];
        if (d != 0.f && voxel(u >> 1, idx)) atomicAdd(&gd[2 * idx + (u & 1)], d);
    }
    for (int v = tid; v < kBox3; v += blockDim.x) {
        const float w = box[2][v];
        if (w != 0.f && voxel(v, idx)) atomicAdd(&gw[idx], w);
    }
}

// One block per chunk (the grid sized for the most chunks there can be), or (device-driven pools) a fixed grid whose
// blocks stride over the chunks, up to the total the scan left in coff[nb]; blocks reach the 8 XCDs round-robin, and
// each XCD strides over one contiguous eighth, so that neighbouring bricks share the lines of its L2 (259 x 259 x 130
// voxels a class, 4 classes, 250 images: 440 -> 396 us).
// What bounds it is the atomics' traffic past L2: bricks 16 voxels long (8 x 8 x 8: 703 us, 32 x 4 x 4: 669), re and
// im added by neighbouring lanes (954 us with an instruction each), chunks of 1024 records (512: + 10 %, 4096: tails);
// 2000 images of 128^2 in 4 classes: 995 -> 647 us.  Plain read-modify-writes of the voxels only one brick
// reaches were slower (1192 us).
template <bool Q, bool WHOLE>
__global__ __launch_bounds__(256, WHOLE ? 4 : 5) void k_bp_brick(BpArgs a, int nb) {
    if constexpr (!Q) {
        if (blockIdx.x < a.coff[nb]) bp_brick_one<WHOLE>(a, blockIdx.x);
        return;
    }
    if (*a.abort) return;
    const unsigned nck = a.coff[nb], per = (nck + 7) / 8, c0 = (blockIdx.x & 7) * per, c1 = min(c0 + per, nck);
    for (unsigned ck = c0 + (blockIdx.x >> 3); ck < c1; ck += gridDim.x >> 3) {
        bp_brick_one<WHOLE>(a, ck);
        __syncthreads();  // the box of the next chunk
    }
}

// 2D: block (band, slot) adds the bilinear corners that fall on its rows [y0, y0 + rows) of a class grid, over the
// slices of the slot's share of the class, in LDS; a class of one slot adds its band to the grids, the slots of
// several leave partial sums for k_bp_band_add.  Per tile of slices the block lists those of its class, then works through
// them one after the other, a corner of all pixels at a time: the pixels of a slice are two voxels apart, so no two of
// them have the same base voxel and the additions need no atomics (LDS float atomics take about a lane per two cycles: 298
// us).  A band is as many rows as fit in LDS (all 131 for 64^2 images at full resolution); with several, each works
// out every pixel's coordinates for the corners it keeps.  1000 images of 64^2 in ten classes: 54 us (direct
// scatter: 1.04 ms with the slices' own sums, 24 M float atomics to L2).
// The slots follow the classes' slices (slice_cnt, counted by k_post): the same number for every class left one
// that takes all of 200 images among 20 classes to two blocks of a slice a 1.15 us (6400 slices of 64^2: 7.3 ms, 0.53 now).
constexpr int kBandThreads = 1024;
constexpr int kBandParts = 32;  // most slots of a class: k_bp_band_add reads them all
struct BandSlots {
    int first, parts;  // of a class
};
// By the first wave: lane k has class k's share of the slots.  A slot each, the others by the number of slices, and
// at least four slices for each (a block clears and writes its whole band); classes without a slice have none.
DEV BandSlots band_slots(const unsigned* cnt, int K, int slots) {
    const int lane = threadIdx.x & 63;
    const unsigned c = lane < K ? cnt[lane] : 0u;
    unsigned long long all = c;
    for (int o = 32; o > 0; o >>= 1) all += __shfl_xor(all, o, 64);
    int p = 0;
    if (c) p = min(min(1 + (int)((unsigned long long)(slots - K) * c / all), kBandParts), (int)((c + 3u) / 4u));
    int in = p;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(in, o, 64);
        if (lane >= o) in += v;
    }
    return {in - p, p};
}

__global__ __launch_bounds__(kBandThreads) void k_bp_band(BpArgs a, long long S_host, int rows_max, float* work) {
    extern __shared__ float box[];  // [3][rows * padF]
    __shared__ int l_s[kBandThreads], l_img[kBandThreads], l_r[kBandThreads];  // the tile's slices of this class:
    __shared__ double l_w[kBandThreads];                                       // slice, image, rotation, weight
    __shared__ int cnt, s_slot[3];
    const long long ntask = bp_slices(a, S_host) / a.NOR;
    if (ntask == 0) return;
    const int tid = threadIdx.x, slot = blockIdx.y;
    if (tid == 0) s_slot[2] = 0;
    __syncthreads();
    if (tid < 64) {
        const BandSlots b = band_slots(a.slice_cnt, a.K, gridDim.y);
        if (slot >= b.first && slot < b.first + b.parts) {
            s_slot[0] = tid;
            s_slot[1] = slot - b.first;
            s_slot[2] = b.parts;
        }
    }
    __syncthreads();
    const int k = s_slot[0], part = s_slot[1], parts = s_slot[2];
    if (parts == 0) return;
    const int y0 = blockIdx.x * rows_max, rows = min(rows_max, a.pad - y0), nb = rows * a.padF;
    float *br = box, *bi = box + nb, *bw = box + 2 * nb;
    for (int i = tid; i < 3 * nb; i += kBandThreads) box[i] = 0.f;
    const long long s0 = ntask * part / parts * a.NOR, s1 = ntask * (part + 1) / parts * a.NOR;
    constexpr int PX = 2;  // pixels a thread at a time
    for (long long t0 = s0; t0 < s1; t0 += kBandThreads) {
        __syncthreads();  // the list before is done with
        if (tid == 0) cnt = 0;
        __syncthreads();
        const long long s = t0 + tid;
        if (s < s1) {
            const long long q = s / a.NOR;
            const int m = a.task_m[q], img = a.task_img[q];
            const double w = a.slice_w[s];
            if (m / a.R == k && w > 0.) {
                const int e = atomicAdd(&cnt, 1);
                l_s[e] = tid;
                l_img[e] = img;
                l_r[e] = (m - k * a.R) * a.NOR + (int)(s - q * a.NOR);
                l_w[e] = w;
            }
        }
        __syncthreads();
        for (int e = 0; e < cnt; ++e) {
            const double w = l_w[e];
            const float* mc = a.MC2bp + (size_t)l_img[e] * a.Pf;
            const float2* val = a.slice_val + (size_t)(t0 + l_s[e]) * a.Pf;
            const double* A = a.Ai_fine + 6 * (size_t)l_r[e];
            for (int p0 = 0; p0 < a.Pf; p0 += PX * kBandThreads) {
                int yb[PX], at[PX];  // row of the lower corner in the band (out of it: no contribution), its index
                float fx[PX], fy[PX], vr[PX], vi[PX], wgt[PX];
#pragma unroll
                for (int j = 0; j < PX; ++j) {
                    const int p = p0 + j * kBandThreads + tid, pc = min(p, a.Pf - 1);
                    const int xy = a.f_xy[pc];
                    const float m = mc[pc];
                    const float2 v = val[pc];
                    const int x = px_x(xy), y = px_y(xy);
                    const Coords c = map_coords(A, x, y, a.c, false);
                    wgt[j] = (float)((double)m * w);
                    const bool in = p < a.Pf && x * x + y * y <= a.r_max * a.r_max && wgt[j] > 0.f;
                    yb[j] = in ? c.y0 - y0 : -2;
                    at[j] = yb[j] * a.padF + c.x0;
                    fx[j] = c.fx;
                    fy[j] = c.fy;
                    vr[j] = v.x;
                    vi[j] = c.neg ? -v.y : v.y;
                }
#pragma unroll
                for (int cc = 0; cc < 4; ++cc) {
                    const int dy = cc >> 1, dx = cc & 1;
#pragma unroll
                    for (int j = 0; j < PX; ++j) {
                        if ((unsigned)(yb[j] + dy) >= (unsigned)rows) continue;
                        const int i = at[j] + dy * a.padF + dx;
                        const float dd = (dy ? fy[j] : 1.f - fy[j]) * (dx ? fx[j] : 1.f - fx[j]);
                        br[i] += dd * vr[j];
                        bi[i] += dd * vi[j];
                        bw[i] += dd * wgt[j];
                    }
                    __syncthreads();
                }
            }
        }
    }
    __syncthreads();
    const size_t gn = a.grid_stride, g0 = (size_t)y0 * a.padF;
    if (parts == 1) {
        float* gd = a.bp_data + 2 * (gn * k + g0);
        float* gw = a.bp_weight + gn * k + g0;
        for (int i = tid; i < nb; i += kBandThreads) {
            gd[2 * i] += br[i];
            gd[2 * i + 1] += bi[i];
            gw[i] += bw[i];
        }
    } else {
        float* o = work + 3 * gn * (size_t)slot + g0;
        for (int i = tid; i < nb; i += kBandThreads) {
            o[i] = br[i];
            o[gn + i] = bi[i];
            o[2 * gn + i] = bw[i];
        }
    }
}

// The slots' sums of a class of several (blockIdx.y) added to its grids.
__global__ __launch_bounds__(256) void k_bp_band_add(BpArgs a, long long S_host, int slots,
                                                     const float* __restrict__ work) {
    __shared__ BandSlots s_b;
    if (bp_slices(a, S_host) == 0) return;
    const size_t gn = a.grid_stride, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int k = blockIdx.y;
    if (threadIdx.x < 64) {
        const BandSlots b = band_slots(a.slice_cnt, a.K, slots);
        if ((int)threadIdx.x == k) s_b = b;
    }
    __syncthreads();
    if (i >= gn || s_b.parts < 2) return;
    const float* w = work + 3 * gn * (size_t)s_b.first + i;
    float s[3] = {0.f, 0.f, 0.f};
    for (int part = 0; part < s_b.parts; ++part)
#pragma unroll
        for (int q = 0; q < 3; ++q) s[q] += w[(3 * (size_t)part + q) * gn];
    a.bp_data[2 * (gn * k + i)] += s[0];
    a.bp_data[2 * (gn * k + i) + 1] += s[1];
    a.bp_weight[gn * k + i] += s[2];
}

void bp_scan(hipStream_t s, const BpArgs& a, int nb) {
    const unsigned blocks = (unsigned)((nb + kScanBlock - 1) / kScanBlock);
    const unsigned chunk = a.whole_bricks ? ~0u : kChunk;
    k_bp_sums<<<blocks, kScanBlock, 0, s>>>(a.count, nb, chunk, a.sums);
    k_bp_scan<<<blocks, kScanBlock, 0, s>>>(a.count, nb, chunk, a.sums, a.off, a.coff, a.cursor, a.ck_brick);
}

}  // namespace

BandPlan bp_band_plan(int K, int pad, int padF, int n_cu) {
    BandPlan b;
    const int fit = std::max(1, (138 << 10) / (12 * padF));  // rows in LDS beside the block's list
    b.bands = (pad + fit - 1) / fit;
    b.rows = (pad + b.bands - 1) / b.bands;
    b.slots = std::max(K, std::min(n_cu / b.bands, kBandParts * K));  // a block per CU
    b.work = b.slots > K ? (size_t)3 * b.slots * pad * padF : 0;
    return b;
}

hipError_t launch_backproject_bands(hipStream_t s, long long S, const BpArgs& a, const BandPlan& b, float* work) {
    if (!a.ntask_dev && S <= 0) return hipSuccess;
    const size_t lds = (size_t)12 * b.rows * a.padF;
    if (lds + 20 * kBandThreads + 16 > ((size_t)160 << 10) || b.bands < 1 || a.K > 64 || b.slots < a.K ||
        !a.slice_cnt || (b.slots > a.K && !work) || a.grid_stride != (size_t)a.pad * a.padF)
        return hipErrorInvalidValue;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_bp_band),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    k_bp_band<<<dim3((unsigned)b.bands, (unsigned)b.slots), kBandThreads, lds, s>>>(a, S, b.rows, work);
    if (b.slots > a.K)
        k_bp_band_add<<<dim3((unsigned)((a.grid_stride + 255) / 256), (unsigned)a.K), 256, 0, s>>>(a, S, b.slots, work);
    return hipGetLastError();
}

// at most one chunk per brick plus one per kChunk records
size_t bp_chunks_max(size_t nb, long long S, int Pf) { return nb + ((size_t)S * Pf + kChunk - 1) / kChunk; }

hipError_t launch_backproject_binned(hipStream_t s, long long S, const BpArgs& a, int persist_blocks) {
    const int nb = a.nb_class * a.K;
    hipError_t e;
    if (a.ntask_dev) {  // device-driven: fixed grids striding over the device counts
        if (a.whole_bricks || !a.abort || persist_blocks <= 0) return hipErrorInvalidValue;
        if ((unsigned long long)a.slice_cap * a.Pf >= (1ULL << 32)) return hipErrorInvalidValue;
        if ((e = launch_fill32(s, a.count, 0u, (size_t)nb)) != hipSuccess) return e;
        const int nPB = (a.Pf + 255) / 256;
        const dim3 g2((unsigned)std::max(1, persist_blocks / nPB), (unsigned)nPB);
        k_bp_count<true><<<g2, 256, 0, s>>>(a, 0);
        bp_scan(s, a, nb);
        k_bp_fill<true><<<g2, 256, 0, s>>>(a, 0);
        k_bp_brick<true, false><<<std::max(1, persist_blocks / 8) * 8, 256, 0, s>>>(a, nb);
        return hipGetLastError();
    }
    if (S <= 0) return hipSuccess;
    if (S > 0x7fffffffLL || (unsigned long long)S * a.Pf >= (1ULL << 32)) return hipErrorInvalidValue;
    if ((e = launch_fill32(s, a.count, 0u, (size_t)nb)) != hipSuccess) return e;
    const dim3 grid((unsigned)S, (a.Pf + 255) / 256);
    k_bp_count<false><<<grid, 256, 0, s>>>(a, S);
    bp_scan(s, a, nb);
    k_bp_fill<false><<<grid, 256, 0, s>>>(a, S);
    const unsigned long long chunks = bp_chunks_max(nb, S, a.Pf);
    if (a.whole_bricks) k_bp_brick<false, true><<<(unsigned)nb, 256, 0, s>>>(a, nb);
    else k_bp_brick<false, false><<<(unsigned)chunks, 256, 0, s>>>(a, nb);
    return hipGetLastError();
}

}  // namespace rome
