// Gridding-weight iterations of MyBackProjector::reconstruct (src/reconstruct.cpp:2196-2274) as dense
// transforms on the FP64 matrix units.
//
//   G = FFT( blob * FFT^-1( Fnewweight * Fweight ) ) / size,   Fnewweight /= max(1e-6, |G|)
//
// The grid has P = 4 r_max + 3 points per axis: always odd, often a prime or a product of two (259 = 7 x 37,
// 131), so a library FFT runs it as Bluestein convolutions of complex lines.  The data allow much less:
// F = Fnewweight * Fweight is real and F(-k) = F(k) (the x = 0 plane is folded first), hence with signed
// indices -h .. h, h = (P - 1) / 2, H = h + 1 and c = cos, s = sin of 2 pi k n / P
//   z : real lines      A(z')  = c e + i s o,  e = f(z) + f(-z), o = f(z) - f(-z), kept for z' >= 0 only
//   y : complex lines   B(+-y') = c E +- i s O
//   x : B(-x) = conj B(x), so M(+-x') = c b_re -+ s b_im (b = 2 B, B at x = 0): real, all x', z' >= 0
//   blob, then x, y, z back the same way; M(-n) = M(n), so z' < 0 is never stored.
// Every step is a product of a symmetric H x H cosine or sine matrix with many columns (v_mfma_f64_16x16x4:
// the accumulator rows 4 r + lane / 16 of one product are the operand rows of the next, so x, blob, x and
// z, update, z chain through LDS without a rearrangement): 6.9 H^3 P multiply-adds per iteration and four
// passes over H^2 P complex values, whatever P factors into.
//
// The reference's blob radius of index h is h + 1 (k < P / 2 ? k : k - P with an odd P), so blob(-n) differs
// from blob(n) on the planes |n| = h unless the table has ended there (it has when current_size = ori_size).
// SYM = false keeps every z' on the way back and the imaginary part of G: twice the y and z work back.
//
// Bound: FP64 MFMA (66 TFLOP/s in a large product on this card).  Only lines and rows inside the ball r^2 < max_r2 are computed before
// the first and after the last axis.  A block is one tile of 16 columns; its waves own up to 3 row tiles
// each, 12 independent accumulators, operands straight from L2 (a k step is 768 matrix cycles for 5 KB).
#include <hip/hip_runtime.h>

#include <utility>

#include "device_util.h"
#include "kernels.h"

namespace rome {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kU = 4;          // k steps whose operands are loaded together: 16 rows
constexpr int kMaxTiles = 15;  // row tiles: H <= 240; H = current_size + 2, of at most 202 (rome_configure)
// Row tiles of 16 per wave: 3 for the many columns of a 3D grid (the fewest operand loads that leave two
// waves per SIMD); 1 in 2D, where a whole pass is a handful of blocks and its time one wave's chain.
constexpr int max_threads(int TPW) { return TPW == 1 ? 64 * kMaxTiles : 64 * ((kMaxTiles + TPW - 1) / TPW); }

DEV d4 mfma64(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// The products' inner loops carry no branch and no mask, so that every load of 16 rows is in flight before the
// first matrix instruction (masked loads became a round trip each: y 90 us instead of 73, x 184 instead of 150).  The tables are zero past
// row and column H, a row index is clamped to one of the same column, and cos has 1/2 in column 0, where
// p(k) + p(-k) counts p(0) twice.
template <int NQ, int U = kU>
struct MatOps {
    double c[U][NQ], s[U][NQ];
    DEV void load(const GriddingArgs& a, int k0, int wave, int W, int lane) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const size_t o = ((size_t)(wave + q * W) * a.nk + k0 + u) * 64 + lane;
                c[u][q] = a.Cf[o];
                s[u][q] = a.Sf[o];
            }
    }
};

template <int N>
struct Num {
    static constexpr int value = N;
};
// body(Num<n>) for the wave's n of up to TPW row tiles below `tiles`
template <int TPW, typename F>
DEV void for_tiles(int wave, int W, int tiles, F&& body) {
    if (TPW > 2 && wave + 2 * W < tiles) body(Num<TPW>());
    else if (TPW > 1 && wave + W < tiles) body(Num<(TPW < 2 ? TPW : 2)>());
    else if (wave < tiles) body(Num<1>());
}

// body(Num<n>, k0) over k steps 0 .. n - 1 (a multiple of 4), n at a time: 4, or WIDE 8 and the rest
template <bool WIDE, typename F>
DEV void for_steps(int n, F&& body) {
    int k0 = 0;
    if constexpr (WIDE)
        for (; k0 + 2 * kU <= n; k0 += 2 * kU) body(Num<2 * kU>(), k0);
    for (; k0 < n; k0 += kU) body(Num<kU>(), k0);
}

// largest k with k^2 < m (m > 0), -1 otherwise
DEV int below_root(int m) {
    if (m <= 0) return -1;
    int r = (int)sqrt((double)(m - 1));
    while (r * r >= m) --r;
    while ((r + 1) * (r + 1) < m) ++r;
    return r;
}

// z lines of one (y, 16 x) tile.  BACK: G(+-z) from T, the weight update; FWD: the transform of
// Fnewweight * Fweight into out.  First iteration: FWD only; last: BACK only.  SPLIT: a block is one wave, blockIdx.z
// its row tile, and what the two halves hand over goes through a.mid instead of LDS, in a launch each.
template <int TPW, bool BACK, bool FWD, bool SYM, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 64 : max_threads(TPW)) void k_grid_z(GriddingArgs a, const double2* __restrict__ T,
                                                                          double2* __restrict__ out) {
    static_assert(!SPLIT || BACK != FWD, "one half a launch");
    extern __shared__ double lds[];  // [2][nt * 256]: e, o of the next transform
    const int lane = threadIdx.x & 63, wave = SPLIT ? blockIdx.z : threadIdx.x >> 6, W = SPLIT ? gridDim.z : blockDim.x >> 6;
    const int kr = lane >> 4, x = blockIdx.x * 16 + (lane & 15), iy = blockIdx.y;
    const int y = iy < a.H ? iy : iy - a.P;
    const int zlim = below_root(a.max_r2 - y * y - (int)(blockIdx.x * 16) * (int)(blockIdx.x * 16));
    if (zlim < 0) return;  // no point of the tile inside the ball: never read by the y pass
    const int ntz = (zlim >> 4) + 1;  // groups of 16 rows with a point inside the ball
    const bool xin = x < a.H;
    const int r2xy = y * y + x * x;
    const size_t zs = (size_t)a.Py * a.H;  // real arrays [z][y][H]
    const size_t xy = (size_t)iy * a.H + min(x, a.H - 1);
    const size_t ts = (size_t)a.Py * a.ldx, tx = (size_t)iy * a.ldx + x;  // T [z'][y][ldx]
    double* le = SPLIT ? a.mid + (size_t)blockIdx.x * a.nt * 512 : lds;
    double* lo = le + a.nt * 256;
    if constexpr (BACK) {
        d4 ce[TPW], so[TPW], ci[TPW], sr[TPW];
#pragma unroll
        for (int q = 0; q < TPW; ++q) ce[q] = so[q] = ci[q] = sr[q] = d4{0., 0., 0., 0.};
        for_tiles<TPW>(wave, W, ntz, [&](auto n) {
            constexpr int NQ = decltype(n)::value;
            for_steps<SPLIT>(a.nk, [&](auto steps, int k0) {
                constexpr int U = decltype(steps)::value;
                double2 p[U], m[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int z = min(4 * (k0 + u) + kr, a.H - 1);
                    p[u] = T[(size_t)z * ts + tx];
                    if constexpr (!SYM) m[u] = T[(size_t)(z ? a.P - z : 0) * ts + tx];
                }
                MatOps<NQ, U> A;
                A.load(a, k0, wave, W, lane);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    double er, oi, ei = 0., orr = 0.;
                    if constexpr (SYM) {
                        er = 2. * p[u].x;
                        oi = 2. * p[u].y;
                    } else {
                        er = p[u].x + m[u].x;
                        ei = p[u].y + m[u].y;
                        orr = p[u].x - m[u].x;
                        oi = p[u].y - m[u].y;
                    }
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        ce[q] = mfma64(A.c[u][q], er, ce[q]);
                        so[q] = mfma64(A.s[u][q], oi, so[q]);
                        if constexpr (!SYM) {
                            ci[q] = mfma64(A.c[u][q], ei, ci[q]);
                            sr[q] = mfma64(A.s[u][q], orr, sr[q]);
                        }
                    }
                }
            });
        });
#pragma unroll
        for (int q = 0; q < TPW; ++q) {
            const int t = wave + q * W;
            if (t >= a.nt) break;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int z = 16 * t + 4 * r + kr;
                double e = 0., o = 0.;
                if (xin && z < a.H && z * z + r2xy < a.max_r2) {
                    // G(+-z) = c E +- s O_im + i (c E_im -+ s O_re)
                    const size_t ip = (size_t)z * zs + xy, im = (size_t)(z ? a.P - z : 0) * zs + xy;
                    const double gp = (ce[q][r] + so[q][r]) / a.size, gm = (ce[q][r] - so[q][r]) / a.size;
                    double wp = fabs(gp), wm = fabs(gm);
                    if constexpr (!SYM) {
                        const double jp = (ci[q][r] - sr[q][r]) / a.size, jm = (ci[q][r] + sr[q][r]) / a.size;
                        wp = sqrt(gp * gp + jp * jp);
                        wm = sqrt(gm * gm + jm * jm);
                    }
                    const double np = a.Fnw[ip] / fmax(1e-6, wp), nm = a.Fnw[im] / fmax(1e-6, wm);
                    const double fp = np * a.Fw[ip], fm = nm * a.Fw[im];
                    a.Fnw[ip] = np;
                    if (z) a.Fnw[im] = nm;  // z = 0: the same element, np = nm
                    e = fp + fm;
                    o = fp - fm;
                }
                if constexpr (FWD || SPLIT) {
                    le[t * 256 + r * 64 + lane] = e;
                    lo[t * 256 + r * 64 + lane] = o;
                }
            }
        }
        if constexpr (FWD) __syncthreads();
    }
    if constexpr (FWD) {
        d4 ar[TPW], ai[TPW];
#pragma unroll
        for (int q = 0; q < TPW; ++q) ar[q] = ai[q] = d4{0., 0., 0., 0.};
        for_tiles<TPW>(wave, W, a.nt, [&](auto n) {
            constexpr int NQ = decltype(n)::value;
            for_steps<SPLIT>(4 * ntz, [&](auto steps, int k0) {
                constexpr int U = decltype(steps)::value;
                double e[U], o[U];
                if constexpr (BACK || SPLIT) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        e[u] = le[(k0 + u) * 64 + lane];
                        o[u] = lo[(k0 + u) * 64 + lane];
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int z = min(4 * (k0 + u) + kr, a.H - 1);
                        const size_t ip = (size_t)z * zs + xy, im = (size_t)(z ? a.P - z : 0) * zs + xy;
                        const double fp = a.Fnw[ip] * a.Fw[ip], fm = a.Fnw[im] * a.Fw[im];
                        const double in = xin ? 1. : 0.;
                        e[u] = in * (fp + fm);
                        o[u] = in * (fp - fm);
                    }
                }
                MatOps<NQ, U> A;
                A.load(a, k0, wave, W, lane);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        ar[q] = mfma64(A.c[u][q], e[u], ar[q]);
                        ai[q] = mfma64(A.s[u][q], o[u], ai[q]);
                    }
            });
        });
#pragma unroll
        for (int q = 0; q < TPW; ++q) {
            const int t = wave + q * W;
            if (t >= a.nt) break;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int z = 16 * t + 4 * r + kr;
                if (z < a.H) out[(size_t)z * ts + tx] = make_double2(ar[q][r], ai[q][r]);
            }
        }
    }
}

// y lines of (z', 16 x) tiles: BACK = false e^{+i}, input rows inside the ball; true e^{-i}, output rows
// inside the ball.  Each of the block's waves has its own tile, blockIdx.y the row tiles of all of them:
// the waves read the same matrix operands at about the same time (L1).
template <int TPW, bool BACK>
__global__ __launch_bounds__(256) void k_grid_y(GriddingArgs a, int nz, const double2* __restrict__ in,
                                                double2* __restrict__ out) {
    const int lane = threadIdx.x & 63, wave = blockIdx.y, W = gridDim.y;  // row tiles wave, wave + W, ..
    const int tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), xt = (a.xlim >> 4) + 1;
    const int kr = lane >> 4, iz = tile / xt, x0 = (tile - iz * xt) * 16;
    if (iz >= nz) return;
    const int ylim = __builtin_amdgcn_readfirstlane(below_root(a.max_r2 - x0 * x0));  // >= 0: x0 <= xlim
    const int nty = (ylim >> 4) + 1;
    const size_t base = (size_t)iz * a.Py * a.ldx + x0 + (lane & 15);
    d4 cr[TPW], ci[TPW], sr[TPW], si[TPW];
#pragma unroll
    for (int q = 0; q < TPW; ++q) cr[q] = ci[q] = sr[q] = si[q] = d4{0., 0., 0., 0.};
    const int kend = BACK ? a.nk : 4 * nty, ymax = BACK ? a.H - 1 : ylim;
    for_tiles<TPW>(wave, W, BACK ? nty : a.nt, [&](auto n) {
        constexpr int NQ = decltype(n)::value;
        for (int k0 = 0; k0 < kend; k0 += kU) {
            double2 p[kU], m[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int y = min(4 * (k0 + u) + kr, ymax);
                p[u] = in[base + (size_t)y * a.ldx];
                m[u] = in[base + (size_t)(y ? a.P - y : 0) * a.ldx];
            }
            MatOps<NQ> A;
            A.load(a, k0, wave, W, lane);
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                // forward: rows outside the ball are zero (never written: the clamped row counts as nothing)
                const double f = BACK || 4 * (k0 + u) + kr <= ylim ? 1. : 0.;
                const double er = f * (p[u].x + m[u].x), ei = f * (p[u].y + m[u].y);
                const double orr = f * (p[u].x - m[u].x), oi = f * (p[u].y - m[u].y);
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    cr[q] = mfma64(A.c[u][q], er, cr[q]);
                    ci[q] = mfma64(A.c[u][q], ei, ci[q]);
                    sr[q] = mfma64(A.s[u][q], orr, sr[q]);
                    si[q] = mfma64(A.s[u][q], oi, si[q]);
                }
            }
        }
    });
    const int nt = BACK ? nty : a.nt;
#pragma unroll
    for (int q = 0; q < TPW; ++q) {
        const int t = wave + q * W;
        if (t >= nt) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int y = 16 * t + 4 * r + kr;
            if (y >= a.H) continue;
            // e^{+i}: out(+-y') = c E +- i s O; e^{-i}: the signs swapped
            const double2 u = make_double2(cr[q][r] - si[q][r], ci[q][r] + sr[q][r]);
            const double2 v = make_double2(cr[q][r] + si[q][r], ci[q][r] - sr[q][r]);
            out[base + (size_t)y * a.ldx] = BACK ? v : u;
            if (y) out[base + (size_t)(a.P - y) * a.ldx] = BACK ? u : v;
        }
    }
}

// blob factor of signed index components given by their reference radii
DEV double blob_at(const GriddingArgs& a, int r2) {
    const double rval = sqrt((double)r2) / (double)a.npad;
    const int idx = (int)(fabs(rval) / a.sampling);
    return idx < a.ntab ? a.tab[idx] / a.tab0 : 0.;
}

// 16 x lines (y', z' >= 0; lines in memory order): forward to M, times the blob, back.  PART 1, 2: one of the halves, a
// block being one wave, blockIdx.y its row tile, and what they hand over in a.mid; 0: both, through LDS.
template <int TPW, bool SYM, int PART>
__global__ __launch_bounds__(PART ? 64 : max_threads(TPW)) void k_grid_x(GriddingArgs a, const double2* __restrict__ in,
                                                                         double2* __restrict__ out) {
    extern __shared__ double dyn[];  // SYM: [2][nt * 256]; else [4][nt * 256]
    double* lds = PART ? a.mid + (size_t)blockIdx.x * (SYM ? 2 : 4) * a.nt * 256 : dyn;
    const int lane = threadIdx.x & 63, wave = PART ? blockIdx.y : threadIdx.x >> 6, W = PART ? gridDim.y : blockDim.x >> 6;
    const int line = blockIdx.x * 16 + (lane & 15);
    const bool yin = line < a.H * a.Py;
    const int kr = lane >> 4, iz = (yin ? line : 0) / a.Py, iy = (yin ? line : 0) - iz * a.Py;
    const int y = iy < a.H ? iy : iy - a.P, h = a.H - 1;
    const size_t row = (size_t)(yin ? line : 0) * a.ldx;
    const int n1 = a.nt * 256;
    const int ntx = (a.xlim >> 4) + 1;  // 16-column groups with a point inside the ball
    if constexpr (PART != 2) {
        d4 tc[TPW], ts[TPW];
#pragma unroll
        for (int q = 0; q < TPW; ++q) tc[q] = ts[q] = d4{0., 0., 0., 0.};
        for_tiles<TPW>(wave, W, a.nt, [&](auto n) {
            constexpr int NQ = decltype(n)::value;
            for_steps<PART != 0>(4 * ntx, [&](auto steps, int k0) {
                constexpr int U = decltype(steps)::value;  // columns past the ball are zero
                double2 b[U];
#pragma unroll
                for (int u = 0; u < U; ++u) b[u] = in[row + 4 * (k0 + u) + kr];
                MatOps<NQ, U> A;
                A.load(a, k0, wave, W, lane);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        tc[q] = mfma64(A.c[u][q], 2. * b[u].x, tc[q]);
                        ts[q] = mfma64(A.s[u][q], 2. * b[u].y, ts[q]);
                    }
            });
        });
        // M(+-x') = tc -+ ts; reference radii of +n and -n differ at n = h only
        const int yp = abs(y) + (y == h), ym = abs(y) + (y == -h);
        const int zp = iz + (iz == h), zm = iz;
        const bool y1 = a.Py > 1;
        const int r2yz1 = (y1 ? yp * yp : 0) + zp * zp;  // line (y', z')
        const int r2yz2 = (y1 ? ym * ym : 0) + zm * zm;  // line (-y', -z')
#pragma unroll
        for (int q = 0; q < TPW; ++q) {
            const int t = wave + q * W;
            if (t >= a.nt) break;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int x = 16 * t + 4 * r + kr, o = t * 256 + r * 64 + lane;
                if constexpr (SYM) {
                    const double f = 2. * blob_at(a, r2yz2 + x * x);  // rows past H: tc = ts = 0
                    lds[o] = tc[q][r] * f;
                    lds[n1 + o] = ts[q][r] * f;
                } else {
                    const double mp = tc[q][r] - ts[q][r], mm = tc[q][r] + ts[q][r];
                    const int xp = x + (x == h), xm = x;
                    const double p1 = mp * blob_at(a, r2yz1 + xp * xp), q1 = mm * blob_at(a, r2yz1 + xm * xm);
                    const double p2 = mm * blob_at(a, r2yz2 + xp * xp), q2 = mp * blob_at(a, r2yz2 + xm * xm);
                    const double e1 = p1 + q1, o1 = p1 - q1, e2 = p2 + q2, o2 = p2 - q2;
                    lds[o] = e1;
                    lds[n1 + o] = o1;
                    lds[2 * n1 + o] = e2;
                    lds[3 * n1 + o] = o2;
                }
            }
        }
    }
    if constexpr (PART == 1) return;
    if constexpr (PART == 0) __syncthreads();
    d4 g[SYM ? 2 : 4][TPW];
#pragma unroll
    for (int p = 0; p < (SYM ? 2 : 4); ++p)
#pragma unroll
        for (int q = 0; q < TPW; ++q) g[p][q] = d4{0., 0., 0., 0.};
    for_tiles<TPW>(wave, W, ntx, [&](auto n) {
        constexpr int NQ = decltype(n)::value;
        for_steps<PART != 0>(a.nk, [&](auto steps, int k0) {
            constexpr int U = decltype(steps)::value;
            double b[U][SYM ? 2 : 4];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int p = 0; p < (SYM ? 2 : 4); ++p) b[u][p] = lds[p * n1 + (k0 + u) * 64 + lane];
            MatOps<NQ, U> A;
            A.load(a, k0, wave, W, lane);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int q = 0; q < NQ; ++q) {
                    g[0][q] = mfma64(A.c[u][q], b[u][0], g[0][q]);
                    g[1][q] = mfma64(A.s[u][q], b[u][1], g[1][q]);
                    if constexpr (!SYM) {
                        g[2][q] = mfma64(A.c[u][q], b[u][2], g[2][q]);
                        g[3][q] = mfma64(A.s[u][q], b[u][3], g[3][q]);
                    }
                }
        });
    });
    if (!yin) return;
    // the line (-y', -z'): another z' > 0 never writes it; at z' = 0 the y' tiles cover every line
    const size_t row2 = ((size_t)(a.P - iz) * a.Py + (iy ? a.Py - iy : 0)) * a.ldx;
#pragma unroll
    for (int q = 0; q < TPW; ++q) {
        const int t = wave + q * W;
        if (t >= ntx) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int x = 16 * t + 4 * r + kr;  // rows past H are zero (and inside the padded row)
            if constexpr (SYM) {
                out[row + x] = make_double2(g[0][q][r], g[1][q][r]);  // o = -2 blob ts: c e - i s o
            } else {
                out[row + x] = make_double2(g[0][q][r], -g[1][q][r]);
                if (iz) out[row2 + x] = make_double2(g[2][q][r], -g[3][q][r]);
            }
        }
    }
}

}  // namespace

template <int TPW>
static hipError_t iterate(hipStream_t s, const GriddingArgs& a, bool sym, int iters) {
    const int W = (a.nt + TPW - 1) / TPW, xt = (a.xlim >> 4) + 1, nth = 64 * W;
    const dim3 gz(xt, a.Py), gx((a.H * a.Py + 15) / 16);
    const size_t l1 = (size_t)a.nt * 256 * sizeof(double);
    // above 64 KB a launch needs the kernel's leave (without SYM from H = 129 on)
    if (!sym && 4 * l1 > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_grid_x<TPW, false, 0>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * l1));
        if (e != hipSuccess) return e;
    }
    k_grid_z<TPW, false, true, true, false><<<gz, nth, 0, s>>>(a, nullptr, a.T0);
    double2 *p = a.T0, *q = a.T1;
    for (int it = 0; it < iters; ++it) {
        const int nzb = sym ? a.H : a.P;
        if constexpr (TPW > 1) {  // (2D has no y)
            k_grid_y<TPW, false><<<dim3((xt * a.H + 3) / 4, W), 256, 0, s>>>(a, a.H, p, q);
            std::swap(p, q);
        }
        if (sym) k_grid_x<TPW, true, 0><<<gx, nth, 2 * l1, s>>>(a, p, q);
        else k_grid_x<TPW, false, 0><<<gx, nth, 4 * l1, s>>>(a, p, q);
        std::swap(p, q);
        if constexpr (TPW > 1) {
            k_grid_y<TPW, true><<<dim3((xt * nzb + 3) / 4, W), 256, 0, s>>>(a, nzb, p, q);
            std::swap(p, q);
        }
        const bool last = it + 1 == iters;
        if (sym && last) k_grid_z<TPW, true, false, true, false><<<gz, nth, 0, s>>>(a, p, q);
        else if (sym) k_grid_z<TPW, true, true, true, false><<<gz, nth, 2 * l1, s>>>(a, p, q);
        else if (last) k_grid_z<TPW, true, false, false, false><<<gz, nth, 0, s>>>(a, p, q);
        else k_grid_z<TPW, true, true, false, false><<<gz, nth, 2 * l1, s>>>(a, p, q);
        std::swap(p, q);
    }
    return hipGetLastError();
}

// 2D, large: every half transform a launch of one-wave blocks, a 16 x 16 tile each
template <bool SYM>
static hipError_t iterate_split(hipStream_t s, const GriddingArgs& a, int iters) {
    const int xt = (a.xlim >> 4) + 1;
    const unsigned nl = (unsigned)(a.H + 15) / 16;
    k_grid_z<1, false, true, true, false><<<dim3(xt, 1), 64 * a.nt, 0, s>>>(a, nullptr, a.T0);
    for (int it = 0; it < iters; ++it) {
        k_grid_x<1, SYM, 1><<<dim3(nl, a.nt), 64, 0, s>>>(a, a.T0, a.T1);
        k_grid_x<1, SYM, 2><<<dim3(nl, xt), 64, 0, s>>>(a, a.T0, a.T1);
        k_grid_z<1, true, false, SYM, true><<<dim3(xt, 1, a.nt), 64, 0, s>>>(a, a.T1, a.T0);
        if (it + 1 < iters) k_grid_z<1, false, true, SYM, true><<<dim3(xt, 1, a.nt), 64, 0, s>>>(a, a.T1, a.T0);
    }
    return hipGetLastError();
}

// 2D, from 7 row tiles on, or 5 without SYM: a block's matrix cores are the bound then, and a tile of 16 columns is one
// block.  Ten iterations of a class, whole against split: H = 88 0.385 and 0.396 ms, 98 0.394 and 0.359, 172 0.730
// and 0.489; without SYM H = 68 0.469 and 0.472, 74 0.465 and 0.444, 172 0.981 and 0.651.  One wave a SIMD hides no
// load by itself, so these blocks take 8 k steps at a time (4: 172 0.534, without SYM 0.682).
static bool gridding_split(int nt, bool is3d, bool sym) { return !is3d && nt >= (sym ? 7 : 5); }

size_t gridding_mid_len(int H, bool is3d, bool sym) {
    const int nt = (H + 15) / 16;
    return gridding_split(nt, is3d, sym) ? (size_t)nt * nt * 1024 : 0;
}

hipError_t gridding_iterations(hipStream_t s, const GriddingArgs& a, bool sym, int iters) {
    if (iters <= 0) return hipSuccess;
    if (a.nt < 1 || a.nt > kMaxTiles || a.nk != 4 * a.nt || a.ldx < 16 * a.nt || a.xlim < 0 || a.xlim >= a.H || a.P != 2 * a.H - 1 || (a.Py != 1 && a.Py != a.P))
        return hipErrorInvalidValue;
    if (a.Py > 1) return iterate<3>(s, a, sym, iters);
    if (!gridding_split(a.nt, false, sym)) return iterate<1>(s, a, sym, iters);
    if (!a.mid) return hipErrorInvalidValue;
    return sym ? iterate_split<true>(s, a, iters) : iterate_split<false>(s, a, iters);
}

}  // namespace rome
