// erp_narrow.hip — spectral chain of typed targets for a narrow band.
//
// A shot's refracted trace needs, of each (shot, target) pair's inward trace
// a (nr bins) and its compressed window z = crop(g * a), only the products
// X_k Z_k of their DFT_L values (L = 2 nr - 1) at the 2 K + 1 frequencies
// |k| <= K that cropSpectrum keeps (elementary_kernels.cu:258-278):
//     out[i] = 1/L sum_{|k| <= K} S_k exp(2 pi i k 2 i / L),
//     S_k = sum over the pairs of X_k Z_k.
// Both are linear in a, X_k = sum_m a[m] e_k[m] and Z_k = sum_m a[m] M_k[m]
// with e_k[m] = exp(-2 pi i k m / L) and
//     M_k[m] = sum_{0 <= j < nr} g[j - m] exp(-2 pi i k j / L).
// Where the band is a small part of the sample rate (1 MHz of 48 MHz keeps
// 4 % of the frequencies) transforming every pair at the full rate does
// mostly work that the crop throws away.  As functions of m, e_k and M_k are
// band-limited to |f| <= fp (the band, and half the chirp's bandwidth), so
// their values at every q-th bin and a low-pass filter h reproduce them:
//     sum_m a[m] phi[m] = sum_i a'[i] q phi[i q],  a'[i] = sum_m h[i q - m] a[m],
// with h flat to fp and stopping from 1/q - fp on (the carrier outside the band
// is far stronger than what is inside).  h is a Kaiser window designed for 180 dB;
// rounded to FP32 it reaches 156 to 163 dB and is flat to 2e-8 (q = 4 to 48),
// below the rounding of the FP32 sums it goes into: the chain's traces are as
// close to 64 bits as the transforms' (4.2e-7 against 7.0e-7 of 7e5 pairs).  The
// range kernel is the reference's 2nr-circular, kc-cropped one,
//     g[d] = s(d) for d >= -kc, s(d + 2 nr) below,  s(d) = sinc(d dr / res),
// so M_k has a kink at m = kc.  a is therefore filtered in two parts, m <=
// kc and m > kc, whose columns hold the two smooth continuations
//     left   sum over 0 <= j < nr of s(j - m) e_k[j]
//     right  e_k[m] (sum over -kc <= d < nr - m of s(d) e_k[d]
//                    - sum over -kc <= d < -m of s(d + 2 nr) e_k[d])
// (sums whose end lies below their start count negatively).
//
// Pairs come in slices of 32 of one shot; per launch of pairs
//   k_narrow_fir   a' of every pair: a product with the filter's Toeplitz
//                  matrix on the FP32 matrix cores
//   k_narrow_gemm  X and Z of a slice as a real matrix product, rows (Re e,
//                  Im e, Re M, Im M) per k, columns the pairs' Re a' and Im
//                  a'; e_-k and M_-k are the conjugates, so the products at k
//                  and -k follow in registers and are summed over the slice
//   k_narrow_sum   slices into the shot's sums, in order
// and k_narrow_out per batch.
//
// Bound by the matrix cores in principle (in k_narrow_fir a third and in
// k_narrow_gemm half of the time is products; the rest is the start of each
// short workgroup and the filter's scalar bookkeeping).  Per launch of 32768
// pairs of 4096 bins at 1 of 48 MHz: 202 + 158 + 12 us, against 1.1 ms for the
// transforms and 0.2 ms for their sums; a run of 100 shots and 7e5 pairs from
// 73.8 to 34.0 ms.
#include "erp_internal.h"

#include <cmath>

namespace {

constexpr int NNT = 256;
constexpr int GB = kNarrowSlice;  // pairs per slice
constexpr int GKT = 4;            // tiles of 4 frequencies per wave

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double range_sinc(double d, double kappa) {
    const double x = d * kappa;
    return fabs(x) < 1e-6 ? 1.0 : sinpi(x) / (M_PI * x);
}
// exp(-2 pi i n / L)
__device__ __forceinline__ void unit(long long n, long long L, double* re, double* im) {
    sincospi(-2.0 * (double)(n % L) / (double)L, im, re);
}

// Rows of one k (blockIdx.x) and part (blockIdx.y).  With N_i = M_k(q i)
// exp(2 pi i k q i / L), a window sum over d, N_{i+1} - N_i is the q terms
// that enter less the q that leave: the first by a direct sum, the others by
// a scan, so the table costs O(nr) terms per k.
__global__ void __launch_bounds__(NNT) k_narrow_table(float* __restrict__ tab, NarrowPlan p) {
    __shared__ double sx[NNT], sy[NNT];
    const int k = blockIdx.x, tid = threadIdx.x;
    const bool right = blockIdx.y;
    const long long L = 2LL * p.nr - 1, kc = p.nr / 2;
    const int n = right ? p.nR : p.nL, i0 = right ? p.iR0 : p.iL0;
    double rx, ry;
    unit(k, L, &rx, &ry);
    // sum over d in [a, b) of s(d + shift) e_k[d]
    auto part = [&](long long a, long long b, long long shift, double* x, double* y) {
        double cx, cy, ax = 0.0, ay = 0.0;
        unit((long long)k * a, L, &cx, &cy);
        for (long long d = a; d < b; ++d) {
            const double v = range_sinc((double)(d + shift), p.kappa);
            ax = fma(v, cx, ax);
            ay = fma(v, cy, ay);
            const double t = fma(cx, rx, -cy * ry);
            cy = fma(cx, ry, cy * rx);
            cx = t;
        }
        *x = ax;
        *y = ay;
    };
    // the same, cut over the workgroup; signed
    auto whole = [&](long long a, long long b, long long shift, double* x, double* y) {
        const double sg = b < a ? -1.0 : 1.0;
        if (b < a) {
            const long long t = a;
            a = b;
            b = t;
        }
        const long long w = (b - a + NNT - 1) / NNT, lo = a + tid * w;
        double ax = 0.0, ay = 0.0;
        if (lo < b) part(lo, lo + w < b ? lo + w : b, shift, &ax, &ay);
        __syncthreads();
        sx[tid] = ax;
        sy[tid] = ay;
        __syncthreads();
        for (int h = NNT / 2; h > 0; h >>= 1) {
            if (tid < h) {
                sx[tid] += sx[tid + h];
                sy[tid] += sy[tid + h];
            }
            __syncthreads();
        }
        *x += sg * sx[0];
        *y += sg * sy[0];
    };
    double bx = 0.0, by = 0.0;  // N at the column before the current 256
    const long long m0 = (long long)p.q * i0, nr2 = 2LL * p.nr;
    if (!right) {
        whole(-m0, p.nr - m0, 0, &bx, &by);
    } else {
        whole(-kc, p.nr - m0, 0, &bx, &by);
        double tx = 0.0, ty = 0.0;
        whole(-kc, -m0, nr2, &tx, &ty);
        bx -= tx;
        by -= ty;
    }
    for (int c0 = 0; c0 < n; c0 += NNT) {
        // step into column c (none into the first)
        const int c = c0 + tid;
        double dx = 0.0, dy = 0.0;
        if (c > 0 && c < n) {
            const long long m = (long long)p.q * (i0 + c);
            double ex, ey, lx, ly;
            part(-m, -m + p.q, right ? nr2 : 0, &ex, &ey);
            part(p.nr - m, p.nr - m + p.q, 0, &lx, &ly);
            dx = ex - lx;
            dy = ey - ly;
        }
        __syncthreads();
        sx[tid] = dx;
        sy[tid] = dy;
        __syncthreads();
        for (int h = 1; h < NNT; h <<= 1) {
            const double ux = tid >= h ? sx[tid - h] : 0.0, uy = tid >= h ? sy[tid - h] : 0.0;
            __syncthreads();
            sx[tid] += ux;
            sy[tid] += uy;
            __syncthreads();
        }
        if (c < n) {
            const double nx = bx + sx[tid], ny = by + sy[tid];
            double ex, ey;
            unit((long long)k * p.q * (i0 + c), L, &ex, &ey);
            float* o = tab + ((size_t)(k >> 2) * p.Nu + (right ? p.nL : 0) + c) * 16 + 4 * (k & 3);
            o[0] = (float)(p.q * ex);
            o[1] = (float)(p.q * ey);
            o[2] = (float)(p.q * (nx * ex - ny * ey));
            o[3] = (float)(p.q * (nx * ey + ny * ex));
        }
        bx += sx[NNT - 1];
        by += sy[NNT - 1];
    }
}

// Tables are read through global (not generic) pointers: a generic load also
// counts as an LDS access and would make every LDS read wait for it
typedef const __attribute__((address_space(1))) float* gfloat;
typedef const __attribute__((address_space(1))) v4f* gfloat4;

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ const float* uni(const float* x) {
    const unsigned long long u = (unsigned long long)x;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    return (const float*)((unsigned long long)hi << 32 | lo);
}

// The plan of the row a slice belongs to, in scalar registers
__device__ __forceinline__ NarrowPlan slice_plan(const NarrowPlan& pa, const NarrowMt& mt, int b) {
    if (!mt.trk) return pa;
    const NarrowPlan& s = mt.trk[mt.rk[mt.pshot[b]].trk].narrow;
    NarrowPlan p;
    p.nr = uni(s.nr);
    p.K = uni(s.K);
    p.q = uni(s.q);
    p.T = uni(s.T);
    p.iL0 = uni(s.iL0);
    p.nL = uni(s.nL);
    p.iR0 = uni(s.iR0);
    p.nR = uni(s.nR);
    p.Nu = uni(s.Nu);
    p.nfb = uni(s.nfb);
    p.tab = uni(s.tab);
    p.fir = uni(s.fir);
    return p;
}

// Bins [m0, m1) that some pair of a slice holds data in, and the columns they
// reach: [lo[h], hi[h]) of the left (h = 0) and right part, in multiples of
// 16.  pbase < 0: the whole row.
struct Live {
    int m0, m1, lo[2], hi[2];
};
__device__ __forceinline__ Live live_range(const NarrowPlan& p, const int* __restrict__ pbase,
                                           const int* __restrict__ pwin, int b, int e) {
    const int i = b + (threadIdx.x & 31);
    int m0 = p.nr, m1 = 0;
    if (i < e) {
        const int base = pbase[i], win = pwin[i];
        if (base < 0 || win > 0) {
            m0 = max(base, 0);
            m1 = base < 0 ? p.nr : min(base + win, p.nr);
        }
    }
#pragma unroll
    for (int d = 1; d < GB; d <<= 1) {
        m0 = min(m0, __shfl_xor(m0, d));
        m1 = max(m1, __shfl_xor(m1, d));
    }
    Live v;
    v.m0 = __builtin_amdgcn_readfirstlane(m0);
    v.m1 = __builtin_amdgcn_readfirstlane(m1);
    const int kc = p.nr / 2;
    v.lo[0] = v.hi[0] = v.lo[1] = v.hi[1] = 0;
    auto cols = [&](int a, int c, int i0, int n, int h) {  // bins [a, c]
        if (a > c) return;
        // i q within T of the bins (ceiling and floor of the quotients)
        const int f = a - p.T;
        const int ilo = f >= 0 ? (f + p.q - 1) / p.q : -(-f / p.q);
        const int l0 = max(ilo - i0, 0), h0 = min((c + p.T) / p.q - i0 + 1, n);
        if (l0 >= h0) return;
        v.lo[h] = l0 & ~15;
        v.hi[h] = (h0 + 15) & ~15;
    };
    cols(v.m0, min(v.m1 - 1, kc), p.iL0, p.nL, 0);
    cols(max(v.m0, kc + 1), v.m1 - 1, p.iR0, p.nR, 1);
    return v;
}

__device__ __forceinline__ int hi_tiles(const Live& v, int h) { return (v.hi[h] - v.lo[h]) >> 4; }

// a' of a slice in tiles of 16 columns, a workgroup per FT tiles, wave w for
// pairs 8 w .. 8 w + 7 (their re and im are the product's 16 columns).  The
// slice's bins pass through LDS 64 at a time (read once, masked there).  A
// tile's filter spans nfb blocks of 16 bins and the next tile's begins q
// blocks later, nfb < 4 q, so at most four tiles are open at a time: tile j
// sums in slot j mod 4, and every wave has the same work (a wave per tile
// instead leaves three of four SIMDs waiting wherever a slice has few tiles).
// The contraction over a block takes bin 4 g + t at step t in lane group g: a
// lane reads 4 consecutive bins.
constexpr int FT = 8;          // tiles per workgroup
constexpr int FB_ = 4;         // blocks staged at a time
constexpr int FLD = 64 + 4;    // floats per staged column (banks: 4 words on)
__global__ void __launch_bounds__(NNT) k_narrow_fir(float* __restrict__ Ad, int as,
                                                    const float2* __restrict__ A, int P,
                                                    const int* __restrict__ pbase,
                                                    const int* __restrict__ pwin,
                                                    const int* __restrict__ gb,
                                                    const int* __restrict__ ge, NarrowPlan pa,
                                                    NarrowMt mt) {
    __shared__ __align__(16) float sh[2][2 * GB * FLD];
    const int b = gb[blockIdx.x], e = ge[blockIdx.x];
    if (b >= e) return;  // padding slice of a replayed launch: never read
    const NarrowPlan p = slice_plan(pa, mt, b);
    const int lane = threadIdx.x & 63, g = lane >> 4, col = lane & 15;
    const int wv = uni((int)threadIdx.x >> 6);
    const Live lv = live_range(p, pbase, pwin, b, e);
    const int kc = p.nr / 2;
    const int n0 = (hi_tiles(lv, 0) + FT - 1) / FT, n1 = (hi_tiles(lv, 1) + FT - 1) / FT;
    // staging: this thread's two bins of rows tid / 32 + 8 i
    const int c2 = 2 * (threadIdx.x & 31), r0 = threadIdx.x >> 5;
    int base[4], end[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int j = b + r0 + 8 * i;
        const int bs = j < e ? pbase[j] : 0, w = j < e ? pwin[j] : 0;
        base[i] = max(bs, 0);
        end[i] = bs < 0 ? p.nr : min(bs + w, p.nr);
    }
    for (int grp = blockIdx.y; grp < n0 + n1; grp += gridDim.y) {
        const int h = grp >= n0 ? 1 : 0;
        const int u0 = (h ? lv.lo[1] + 16 * FT * (grp - n0) : lv.lo[0] + 16 * FT * grp);
        const int nt = min(FT, ((h ? lv.hi[1] : lv.hi[0]) - u0) >> 4);
        const int q0 = h ? max(lv.m0, kc + 1) : lv.m0, q1 = h ? lv.m1 : min(lv.m1, kc + 1);
        const int f = ((h ? p.iR0 : p.iL0) + u0) * p.q - p.T;
        const int ms = f & ~15;  // first bin of the first tile's blocks (f < 0: rounds down)
        const int b0 = max(0, (q0 - ms) >> 4);
        const int b1 = min(p.nfb + (nt - 1) * p.q, ((q1 - 1 - ms) >> 4) + 1);
        // loads of whole rows; what the pair's window and part do not hold is
        // masked on the way to LDS (masking here would wait for each load)
        v4f v[4];
        int vm = 0;
        auto fetch = [&](int blk) {
            vm = ms + 16 * blk + c2;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = *(gfloat4)(A + (size_t)min(b + r0 + 8 * i, e - 1) * P + min(vm, P - 2));
        };
        auto stage = [&](float* st) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int l = max(base[i], q0), u = min(end[i], q1);
                const bool k0 = vm >= l && vm < u, k1 = vm + 1 >= l && vm + 1 < u;
                float* d = st + 2 * (r0 + 8 * i) * FLD + c2;  // re, then im of a pair
                *reinterpret_cast<float2*>(d) =
                    make_float2(k0 ? v[i].x : 0.f, k1 ? v[i].z : 0.f);
                *reinterpret_cast<float2*>(d + FLD) =
                    make_float2(k0 ? v[i].y : 0.f, k1 ? v[i].w : 0.f);
            }
        };
        const gfloat4 fr = (gfloat4)p.fir + (size_t)(h * p.nfb) * 64 + lane;
        // slot s: tile jn - s, jn the newest begun; r blocks into it
        v4f acc[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[s] = v4f{0.f, 0.f, 0.f, 0.f};
        int jn = b0 / p.q, r = b0 - jn * p.q, open = 0;
        auto opened = [&]() {
            open = 0;
#pragma unroll
            for (int s = 0; s < 4; ++s) open |= jn >= s && jn - s < nt ? 1 << s : 0;
        };
        opened();
        // slice rows [column][re 0-31, im 0-31]; register c: column 4 g + c
        float* ob = Ad + ((size_t)blockIdx.x * as + (h ? p.nL : 0) + u0 + 4 * g) * (2 * GB) +
                    (col & 1) * GB + 8 * wv + (col >> 1);
        auto put = [&](int j, const v4f& a) {
            if (j < 0 || j >= nt) return;
#pragma unroll
            for (int c = 0; c < 4; ++c) ob[(16 * j + c) * 2 * GB] = a[c];
        };
        auto taps = [&](v4f(&t)[4], int rr) {
#pragma unroll
            for (int s = 0; s < 4; ++s) t[s] = fr[(size_t)min(rr + s * p.q, p.nfb - 1) * 64];
            __builtin_amdgcn_sched_barrier(0);
        };
        int ping = 0;
        const float* src = nullptr;
        // products of one block with its taps t; tn: those of the next
        auto block = [&](const v4f(&t)[4], v4f(&tn)[4], int blk) {
            const int k = (blk - b0) & (FB_ - 1);
            if (k == 0) {
                float* st = sh[ping];
                ping ^= 1;
                stage(st);
                __syncthreads();
                if (blk + FB_ < b1) fetch(blk + FB_);
                src = st + (16 * wv + col) * FLD + 4 * g;
            }
            const v4f x = *reinterpret_cast<const v4f*>(src + 16 * k);
            const int rn = r + 1 == p.q ? 0 : r + 1;
            taps(tn, rn);
            // a tile is done after nfb blocks: slot 3 within this run of q
            // blocks, slots 2 and 1 too where the band is below 1/144 (q stays
            // 48 there and the filter gets shorter than three runs)
            const int m = r + 3 * p.q < p.nfb   ? open
                          : r + 2 * p.q < p.nfb ? open & 7
                          : r + p.q < p.nfb     ? open & 3
                                                : open & 1;
            if (m == 15) {
                // four sums in turn: none waits for its own last product
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[s][d], x[d], acc[s], 0, 0,
                                                                      0);
            } else if (m == 7) {
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int s = 0; s < 3; ++s)
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[s][d], x[d], acc[s], 0, 0,
                                                                      0);
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (m >> s & 1) {
#pragma unroll
                        for (int d = 0; d < 4; ++d)
                            acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[s][d], x[d], acc[s], 0,
                                                                          0, 0);
                    }
            }
            if (rn == 0) {
                put(jn - 3, acc[3]);
                acc[3] = acc[2];
                acc[2] = acc[1];
                acc[1] = acc[0];
                acc[0] = v4f{0.f, 0.f, 0.f, 0.f};
                ++jn;
                opened();
            }
            r = rn;
            __builtin_amdgcn_sched_barrier(0);
        };
        __syncthreads();  // the last group's reads of sh
        v4f ta[4], tb[4];
        if (b0 < b1) {
            fetch(b0);
            taps(ta, r);
        }
        for (int blk = b0; blk < b1; blk += 2) {
            block(ta, tb, blk);
            if (blk + 1 < b1) block(tb, ta, blk + 1);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) put(jn - s, acc[s]);
        for (int j = jn + 1; j < nt; ++j) put(j, v4f{0.f, 0.f, 0.f, 0.f});
    }
}

// X and Z of a slice: 4 tiles of 4 frequencies per wave; the matrix
// instruction's 16 rows are 4 frequencies x (Re e, Im e, Re M, Im M), so a
// lane ends with all four of its frequency and pair.  The columns pass
// through LDS 64 at a time, shared by the four waves; each such part is summed
// by itself, which bounds the FP32 rounding.
constexpr int GU = 64;
constexpr int GLD = 80;  // floats per staged column (4 columns x 16 lanes on all banks)
__global__ void __launch_bounds__(NNT, 2) k_narrow_gemm(float4* __restrict__ part, int ps,
                                                     const float* __restrict__ Ad, int as,
                                                     const int* __restrict__ pbase,
                                                     const int* __restrict__ pwin,
                                                     const int* __restrict__ gb,
                                                     const int* __restrict__ ge, NarrowPlan pa,
                                                     NarrowMt mt) {
    __shared__ __align__(16) float sh[2][GU * GLD];
    const int b = gb[blockIdx.x], e = ge[blockIdx.x];
    if (b >= e) return;
    const NarrowPlan p = slice_plan(pa, mt, b);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int)blockIdx.y * (NNT / 64) * GKT * 4 > p.K) return;
    const int kt0 = (blockIdx.y * (NNT / 64) + wv) * GKT;
    const bool on = kt0 * 4 <= p.K;
    const Live lv = live_range(p, pbase, pwin, b, e);
    v4f sum[GKT][2][2];  // [tile][pairs 0-15 / 16-31][Re a', Im a']
#pragma unroll
    for (int t = 0; t < GKT; ++t)
#pragma unroll
        for (int g = 0; g < 2; ++g) sum[t][g][0] = sum[t][g][1] = v4f{0.f, 0.f, 0.f, 0.f};
    // both parts' live columns, one after the other, in chunks of at most GU
    const int nc0 = (lv.hi[0] - lv.lo[0] + GU - 1) / GU;
    const int nch = nc0 + (lv.hi[1] - lv.lo[1] + GU - 1) / GU;
    auto chunk = [&](int ch, int* n) -> int {  // first column and count
        const int h = ch >= nc0 ? 1 : 0, u = (h ? lv.lo[1] : lv.lo[0]) + GU * (h ? ch - nc0 : ch);
        *n = min(GU, (h ? lv.hi[1] : lv.hi[0]) - u);
        return (h ? p.nL : 0) + u;
    };
    v4f v[4];
    auto fetch = [&](int ch) {  // past n: the last value again, not used
        int n;
        const int u = chunk(ch, &n);
        const gfloat4 src = (gfloat4)(Ad + ((size_t)blockIdx.x * as + u) * (2 * GB));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = src[min((int)threadIdx.x + NNT * i, 16 * n - 1)];
    };
    if (nch > 0) fetch(0);
    for (int ch = 0; ch < nch; ++ch) {
        int n;
        const int u = chunk(ch, &n);
        float* st = sh[ch & 1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int x = threadIdx.x + NNT * i;
            *reinterpret_cast<v4f*>(st + (x >> 4) * GLD + 4 * (x & 15)) = v[i];
        }
        __syncthreads();
        if (ch + 1 < nch) fetch(ch + 1);
        if (!on) continue;
        v4f acc[GKT][2][2];
#pragma unroll
        for (int t = 0; t < GKT; ++t)
#pragma unroll
            for (int g = 0; g < 2; ++g) acc[t][g][0] = acc[t][g][1] = v4f{0.f, 0.f, 0.f, 0.f};
        // the table is padded to whole groups of GKT tiles
        const gfloat T = (gfloat)p.tab + ((size_t)kt0 * p.Nu + u) * 16 + lane;
        const float* B = st + (lane >> 4) * GLD + (lane & 15);
        // table values two steps (1024 cycles of products) ahead, in turn in
        // r0 and r1; the scheduler would move the loads down to their use
        float r0[2][GKT], r1[2][GKT];
        auto load = [&](float(&r)[2][GKT], int c) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int t = 0; t < GKT; ++t) r[s][t] = T[((size_t)t * p.Nu + c + 4 * s) * 16];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto step = [&](const float(&r)[2][GKT], int c) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const float xr = B[(c + 4 * s) * GLD + 16 * g];
                    const float xi = B[(c + 4 * s) * GLD + GB + 16 * g];
#pragma unroll
                    for (int t = 0; t < GKT; ++t) {
                        acc[t][g][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[s][t], xr,
                                                                            acc[t][g][0], 0, 0, 0);
                        acc[t][g][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(r[s][t], xi,
                                                                            acc[t][g][1], 0, 0, 0);
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        load(r0, 0);
        for (int c = 0; c < n; c += 16) {  // n is a multiple of 16
            load(r1, c + 8);
            step(r0, c);
            load(r0, c + 16 < n ? c + 16 : 0);
            step(r1, c + 8);
        }
#pragma unroll
        for (int t = 0; t < GKT; ++t)
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                sum[t][g][0] += acc[t][g][0];
                sum[t][g][1] += acc[t][g][1];
            }
    }
    if (!on) return;
    // with R the rows applied to Re a' and I to Im a': X_k = (R.x + i R.y) +
    // i (I.x + i I.y), X_-k = (R.x - i R.y) + i (I.x - i I.y); Z alike
#pragma unroll
    for (int t = 0; t < GKT; ++t) {
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const v4f R = sum[t][g][0], I = sum[t][g][1];
            const float xr = R.x - I.y, xi = R.y + I.x, zr = R.z - I.w, zi = R.w + I.z;
            const float yr = R.x + I.y, yi = I.x - R.y, wr = R.z + I.w, wi = I.z - R.w;
            o.x += xr * zr - xi * zi;
            o.y += xr * zi + xi * zr;
            o.z += yr * wr - yi * wi;
            o.w += yr * wi + yi * wr;
        }
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) {
            o.x += __shfl_xor(o.x, d);
            o.y += __shfl_xor(o.y, d);
            o.z += __shfl_xor(o.z, d);
            o.w += __shfl_xor(o.w, d);
        }
        const int k = (kt0 + t) * 4 + (lane >> 4);
        if ((lane & 15) == 0 && k <= p.K) part[(size_t)blockIdx.x * ps + k] = o;
    }
}

// S[shot] += scale x the slices of the shot; rows of ps float4: S_k, S_-k.
// A shot holds up to hundreds of slices: 64 frequencies x 4 waves per
// workgroup, the waves' slices interleaved, in a fixed order.
__global__ void __launch_bounds__(NNT) k_narrow_sum(float4* __restrict__ S,
                                                    const float4* __restrict__ part, int ps,
                                                    const int* __restrict__ seg_shot,
                                                    const int* __restrict__ seg_beg,
                                                    const int* __restrict__ seg_end,
                                                    const float* __restrict__ seg_scale,
                                                    float scale, int K, NarrowMt mt) {
    __shared__ float4 s[NNT];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane, sg = blockIdx.y;
    const int r0 = seg_beg[sg], r1 = seg_end[sg];
    if (r0 >= r1) return;
    const int shot = seg_shot[sg];
    if (mt.trk) K = mt.trk[mt.rk[shot].trk].narrow.K;
    if (seg_scale) scale = seg_scale[sg];
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k <= K) {
#pragma unroll 8
        for (int r = r0 + wv; r < r1; r += NNT / 64) {
            const float4 v = part[(size_t)r * ps + k];
            a.x += v.x;
            a.y += v.y;
            a.z += v.z;
            a.w += v.w;
        }
    }
    s[threadIdx.x] = a;
    __syncthreads();
    if (wv || k > K) return;
    float4* d = S + (size_t)shot * ps + k;
    const float4 b = s[64 + lane], c = s[128 + lane], e = s[192 + lane];
    float4 o = *d;
    o.x = fmaf(scale, (a.x + b.x) + (c.x + e.x), o.x);
    o.y = fmaf(scale, (a.y + b.y) + (c.y + e.y), o.y);
    o.z = fmaf(scale, (a.z + b.z) + (c.z + e.z), o.z);
    o.w = fmaf(scale, (a.w + b.w) + (c.w + e.w), o.w);
    *d = o;
}

// out[i] from S_k, S_-k (FP64 phases and sums: the phase of sample i turns by
// 4 pi i / L per k), plus the echo; one thread per sample
__global__ void __launch_bounds__(NNT) k_narrow_out(const float4* __restrict__ S, int ps, int nr,
                                                    int K, FinalOut fo) {
    const int r = blockIdx.y, i = blockIdx.x * NNT + threadIdx.x;
    float2* o;
    const float2* unused;
    if (!final_row(fo, r, nr, &o, &unused)) return;
    if (i >= nr) return;
    if (fo.trk) K = fo.trk[fo.rk[r].trk].narrow.K;
    const float4* x = S + (size_t)r * ps;
    const long long L = 2LL * nr - 1;
    double wx, wy;
    unit(-2LL * i, L, &wx, &wy);
    double ax = x[0].x, ay = x[0].y, cx = wx, cy = wy;
    for (int k = 1; k <= K; ++k) {
        const float4 v = x[k];
        // S_k c + S_-k conj(c)
        const double px = (double)v.x + v.z, py = (double)v.y + v.w;
        const double dx = (double)v.x - v.z, dy = (double)v.y - v.w;
        ax = fma(px, cx, fma(-dy, cy, ax));
        ay = fma(py, cx, fma(dx, cy, ay));
        const double t = fma(cx, wx, -cy * wy);
        cy = fma(cx, wy, cy * wx);
        cx = t;
    }
    const double inv = 1.0 / (double)L;
    o[i] = final_value(fo, (size_t)r * nr + i, fo.Vs[r] > 0,
                       make_float2((float)(ax * inv), (float)(ay * inv)));
}

double bessel_i0(double x) {
    double t = 1.0, s = 1.0;
    for (int k = 1; k < 500; ++k) {
        t *= (x / (2.0 * k)) * (x / (2.0 * k));
        s += t;
        if (t < 1e-18 * s) break;
    }
    return s;
}
constexpr double kAtt = 180.0;  // design stop band of the Kaiser window, dB
// The chain's work per pair grows with the band (columns x frequencies), the
// transforms' does not.  Calls of 8 shots x 1600 targets, transforms and this
// chain (us): 1024 bins 1030 and 527 at 1/48 of the sample rate, 1149 and 781
// at 1/12; 4096 bins 1760 and 661, 1754 and 1067; 16384 bins 5031 and 971 at
// 1/48.  1/12 is where the decimation ends at 4 (the filter's blocks then no
// longer fit four open tiles below it); past 64 MB the tables (46 MB at 16384
// bins and 1/25) are worth less than the memory they hold.
constexpr double kBandMax = 1.0 / 12.0;
constexpr size_t kTableMax = (size_t)64 << 20;
int round16(int n) { return (n + 15) & ~15; }
int ktiles(const NarrowPlan& p) {  // padded to whole groups of a wave
    return (p.K / 4 + GKT) / GKT * GKT;
}

}  // namespace

NarrowPlan narrow_plan(int nr, float dr, float res, float smpl, float B) {
    NarrowPlan p{};
    if (nr <= 512 || nr > 16384) return p;  // as the per-pair chain it stands for
    p.nr = nr;
    p.K = band_limit(nr, smpl, B);
    p.kappa = (double)dr / (double)res;
    if (p.K < 0 || !(p.kappa > 0.0)) return p;
    const double L = 2.0 * nr - 1.0, fp = std::max(p.K / L, 0.5 * p.kappa);
    if (!(fp < kBandMax)) return p;
    p.q = (int)std::min(48.0, std::floor(1.0 / (3.0 * fp)));
    // Kaiser window over the transition from fp to 1/q - fp
    const double df = 1.0 / p.q - 2.0 * fp;
    p.Tq = (int)std::ceil(0.5 * (kAtt - 8.0) / (2.285 * 2.0 * M_PI * df) / p.q);
    p.T = p.Tq * p.q;
    const int kc = nr / 2, f = kc + 1 - p.T;
    p.iL0 = -p.Tq;
    p.nL = round16(kc / p.q + 2 * p.Tq + 1);
    p.iR0 = f >= 0 ? (f + p.q - 1) / p.q : -(-f / p.q);
    p.nR = round16((nr - 1) / p.q + p.Tq - p.iR0 + 1);
    p.Nu = p.nL + p.nR;
    p.nfb = (15 + 15 * p.q + 2 * p.T) / 16 + 1;
    p.ok = sizeof(float) * narrow_table_floats(p) <= kTableMax;
    return p;
}

size_t narrow_table_floats(const NarrowPlan& p) {
    return (size_t)ktiles(p) * p.Nu * 16 + (size_t)2 * p.nfb * 256;
}

void narrow_build(NarrowPlan& p, float* tab, hipStream_t st) {
    const size_t n = (size_t)ktiles(p) * p.Nu * 16, nf = (size_t)2 * p.nfb * 256;
    p.tab = tab;
    p.fir = tab + n;
    // filter taps h(x), |x| <= T, in the order k_narrow_fir's lanes take them
    std::vector<float> h((size_t)2 * p.T + 1), fr(nf);
    const double beta = 0.1102 * (kAtt - 8.7), i0 = bessel_i0(beta), fc = 0.5 / p.q;
    for (int t = 0; t <= 2 * p.T; ++t) {
        const double x = t - p.T, a = 2.0 * fc * x, r = x / p.T;
        const double sinc = t == p.T ? 1.0 : std::sin(M_PI * a) / (M_PI * a);
        h[t] = (float)(2.0 * fc * sinc * bessel_i0(beta * std::sqrt(std::max(0.0, 1.0 - r * r))) /
                       i0);
    }
    for (int part = 0; part < 2; ++part) {
        const int f = (part ? p.iR0 : p.iL0) * p.q - p.T, d = f - (f & ~15);
        for (int blk = 0; blk < p.nfb; ++blk)
            for (int lane = 0; lane < 64; ++lane)
                for (int t = 0; t < 4; ++t) {
                    const int x = d + (lane & 15) * p.q - 16 * blk - 4 * (lane >> 4) - t;
                    fr[(((size_t)part * p.nfb + blk) * 64 + lane) * 4 + t] =
                        x >= -2 * p.T && x <= 0 ? h[x + 2 * p.T] : 0.f;
                }
    }
    ERP_HIP_TRY(hipMemcpyAsync(const_cast<float*>(p.fir), fr.data(), sizeof(float) * nf,
                               hipMemcpyHostToDevice, st));
    zero_words(reinterpret_cast<float2*>(tab), n / 2, st);  // rows past the band: zero
    hipLaunchKernelGGL(k_narrow_table, dim3(p.K + 1, 2), dim3(NNT), 0, st, tab, p);
    ERP_CHECK_LAUNCH("k_narrow_table");
    ERP_HIP_TRY(hipStreamSynchronize(st));  // fr is a host temporary
}

void narrow_pairs(const NarrowPlan& p, const NarrowMt& mt, const float2* A, int P,
                  const int* pbase, const int* pwin, const int* gb, const int* ge, int nslices,
                  float* Ad, float4* part, hipStream_t st) {
    if (nslices <= 0) return;
    const int tiles = p.Nu / 16, w = NNT / 64;
    hipLaunchKernelGGL(k_narrow_fir, dim3(nslices, (tiles + FT - 1) / FT), dim3(NNT), 0, st, Ad,
                       p.Nu, A, P, pbase, pwin, gb, ge, p, mt);
    ERP_CHECK_LAUNCH("k_narrow_fir");
    hipLaunchKernelGGL(k_narrow_gemm, dim3(nslices, (ktiles(p) + GKT * w - 1) / (GKT * w)),
                       dim3(NNT), 0, st, part, p.K + 1, Ad, p.Nu, pbase, pwin, gb, ge, p, mt);
    ERP_CHECK_LAUNCH("k_narrow_gemm");
}

void narrow_sum(const NarrowPlan& p, const NarrowMt& mt, const float4* part, const int* seg_shot,
                const int* seg_beg, const int* seg_end, int nseg, const float* seg_scale,
                float scale, float4* S, hipStream_t st) {
    if (nseg <= 0) return;
    hipLaunchKernelGGL(k_narrow_sum, dim3(p.K / 64 + 1, nseg), dim3(NNT), 0, st, S, part,
                       p.K + 1, seg_shot, seg_beg, seg_end, seg_scale, scale, p.K, mt);
    ERP_CHECK_LAUNCH("k_narrow_sum");
}

void narrow_final_rows(const NarrowPlan& p, const float4* S, int rows, const FinalOut& fo,
                       hipStream_t st) {
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_narrow_out, dim3((p.nr + NNT - 1) / NNT, rows), dim3(NNT), 0, st, S,
                       p.K + 1, p.nr, p.K, fo);
    ERP_CHECK_LAUNCH("k_narrow_out");
}
