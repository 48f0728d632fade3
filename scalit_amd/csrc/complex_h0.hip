// Complex level matrices (the reference's sCX = T): MYHX_CX on split complex
// vectors, and the C-ABI that loads H0CX / DEPCX / OUTHCX and switches them
// on.  (The sCX set-up of the OSB preconditioner is block_diag's complex
// branch in kernels_diag.hip; P*X keeps the real MYPX_DX.)
//
// MYHX_CX (src/iterate/module/osb.hxcx.h:191-245):
//   Y = (RES - E0 +- i A) X + sum_l level_l(X), with
//   level_l(X)(d, i, b) = [DEPCX(d)] sum_j H0CX(i, j) X(d, j, b)
//     (H1X_XYZ_CX / H1X_DEP_CX, src/iterate/libiterate/hpx/hpx_cx.f90:6-39,
//      over H1X_CX / H2X_CX, src/libutil/serial/base/matrix_cx.f90:97-160)
//   and, for the sNDVR layer, Y(p, i) = sum_j OUTHCX(p, i, j) X(p, j)
//     (H3X_CX, matrix_cx.f90:194-208).
// TMAPR takes -APR, as the parallel MYHX_CX (mosb3.hxcx.h:92-94) does; the
// serial one (osb.hxcx.h:234-235) takes -APP there.
//
// Vectors are split (N real parts, then N imaginary parts, per vector); the
// level matrices keep the reference's (re, im) pairs.  The products run on FP64
// MFMA: the diagonal and levels 1 and 2 in one pass, each further level in one
// that adds to Y.  MYHX_CX of one vector at 64 x 96 x 80, passes back to back: 29 us (each
// by itself under the profiler: levels 1 and 2 19.0 with the matrix pipe 31% busy, level 3 12.8
// with 20%), against 121 us with one thread per output point (k_cxh_level_lds: 40 us
// per level, bound by a load of H0CX per multiply-add), which stays for a level of one
// column per block (one-level operators, and level 1 under a dense sNDVR layer) and for
// levels of a few points in many planes.
#include "device_common.hpp"
#include "solver_state.hpp"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace scalit {

static unsigned cxh_grid(long n) { return (unsigned)std::max<long>(1, std::min<long>((n + 255) / 256, 4096)); }

// y = (RES - sh) x + i sign a x (a null: no imaginary diagonal)
__global__ void __launch_bounds__(256) k_cxh_diag(long N, const double *__restrict__ res, double sh,
                                                  const double *__restrict__ a, double sign,
                                                  const double *__restrict__ x, double *__restrict__ y)
{
    const int v = blockIdx.y;
    const double *xr = x + 2L * v * N, *xi = xr + N;
    double *yr = y + 2L * v * N, *yi = yr + N;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
        const double d = res[e] - sh, t = a ? sign * a[e] : 0.0;
        const double r = xr[e], i = xi[e];
        yr[e] = d * r - t * i;
        yi[e] = d * i + t * r;
    }
}

// y(d, i, b) += [DEP(d)] sum_j H(i, j) x(d, j, b) on every vector
__global__ void __launch_bounds__(256) k_cxh_level(int nin, int n, int blk, const dcx *__restrict__ h,
                                                   const dcx *__restrict__ dep, long N,
                                                   const double *__restrict__ x, double *__restrict__ y)
{
    const int v = blockIdx.y;
    const double *xr = x + 2L * v * N, *xi = xr + N;
    double *yr = y + 2L * v * N, *yi = yr + N;
    const long total = (long)nin * n * blk;
    for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
        const int d = (int)(idx % nin);
        const long t = idx / nin;
        const int i = (int)(t % n);
        const long base = (t / n) * (long)nin * n + d;
        double ar = 0.0, ai = 0.0;
        for (int j = 0; j < n; j++) {
            const dcx hv = h[i + (long)n * j];
            const double pr = xr[base + (long)nin * j], pi = xi[base + (long)nin * j];
            ar += hv.re * pr - hv.im * pi;
            ai += hv.re * pi + hv.im * pr;
        }
        if (dep) {
            const dcx dv = dep[d];
            const double r = dv.re * ar - dv.im * ai;
            ai = dv.re * ai + dv.im * ar;
            ar = r;
        }
        yr[idx] += ar;
        yi[idx] += ai;
    }
}

// The same with the X columns staged in LDS.  Column c = (d, b) of a level
// is the n-vector x(d, ., b) (stride nin); a workgroup stages XC columns
// (XC consecutive d of one b, or XC consecutive b when nin = 1) once, and its
// threads, XC apart in the column and 256 / XC apart in the row, form every
// output of those columns from LDS: each X value is read from HBM once per
// level instead of once per output row.
constexpr int XC = 16;
__global__ void __launch_bounds__(256) k_cxh_level_lds(int nin, int n, int blk, const dcx *__restrict__ h,
                                                       const dcx *__restrict__ dep, long N,
                                                       const double *__restrict__ x, double *__restrict__ y)
{
    extern __shared__ char smem_raw[];
    dcx *xt = (dcx *)smem_raw;   // xt[j XC + cc]
    const int v = blockIdx.y;
    const double *xr = x + 2L * v * N, *xi = xr + N;
    double *yr = y + 2L * v * N, *yi = yr + N;
    const long ncol = (long)nin * blk, c0 = (long)blockIdx.x * XC;
    for (int e = threadIdx.x; e < n * XC; e += 256) {
        // nin = 1: a column is contiguous, so walk it first
        const int cc = nin == 1 ? e / n : e % XC, j = nin == 1 ? e % n : e / XC;
        const long c = c0 + cc;
        dcx val{0.0, 0.0};
        if (c < ncol) {
            const long off = (c % nin) + (long)nin * (j + (long)n * (c / nin));
            val = {xr[off], xi[off]};
        }
        xt[j * XC + cc] = val;
    }
    __syncthreads();
    constexpr int NG = 256 / XC;
    const int cc = threadIdx.x % XC, ig = threadIdx.x / XC;
    const long c = c0 + cc;
    if (c >= ncol) return;   // no barrier follows
    const long d = c % nin, b = c / nin;
    for (int i = ig; i < n; i += NG) {
        double ar = 0.0, ai = 0.0;
        for (int j = 0; j < n; j++) {
            const dcx hv = h[i + (long)n * j], xv = xt[j * XC + cc];
            ar += hv.re * xv.re - hv.im * xv.im;
            ai += hv.re * xv.im + hv.im * xv.re;
        }
        if (dep) {
            const dcx dv = dep[d];
            const double r = dv.re * ar - dv.im * ai;
            ai = dv.re * ai + dv.im * ar;
            ar = r;
        }
        const long off = d + (long)nin * (i + (long)n * b);
        yr[off] += ar;
        yi[off] += ai;
    }
}

// ---------------------------------------------------------------- MFMA
// The level products as four real products on FP64 MFMA, each complex 16 x 16
// output tile one wave's: re += xr hr - xi hi, im += xr hi + xi hr.
__device__ __forceinline__ dcx buf_ld_cx(__amdgpu_buffer_rsrc_t r, int voff)
{
    return __builtin_bit_cast(dcx, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}
struct cacc {
    d4_t re, im;
};
// c += a b for an MFMA step: H the A operand (HA) or the B operand
template <bool HA>
__device__ __forceinline__ void cx_mma(cacc &c, dcx h, double xr, double xi)
{
    using M = Mfma<double>;
    if constexpr (HA) {
        c.re = M::run(h.re, xr, c.re);
        c.im = M::run(h.im, xr, c.im);
        c.re = M::run(-h.im, xi, c.re);
        c.im = M::run(h.re, xi, c.im);
    } else {
        c.re = M::run(xr, h.re, c.re);
        c.im = M::run(xr, h.im, c.im);
        c.re = M::run(xi, -h.im, c.re);
        c.im = M::run(xi, h.re, c.im);
    }
}

// The diagonal and levels 1 and 2 of every (n1 x n2) plane in one pass:
//   Y(i,c) = (RES - sh + i sign A)(i,c) X(i,c) + sum_j H1(i,j) X(j,c) + DEP(i) sum_j H2(c,j) X(i,j)
// as k_hx_levels12 (kernels_hx.hip) does it for real matrices: tiles computed
// transposed, KSPL waves of a workgroup per tile, the first sum's X through LDS
// in chunks of CX_KC rows, the operands of the next groups of 16 k in flight by
// buffer loads that return zero past the end.  Grid: (i tiles, c tiles,
// plane and vector).
constexpr int CX_KC = 64;
template <int KSPL>
__global__ void __launch_bounds__(256) k_cxh_levels12(int n1, int n2, int nvec, const dcx *__restrict__ h1,
                                                      const dcx *__restrict__ h2, const dcx *__restrict__ dep2, long N,
                                                      const double *__restrict__ res, double sh,
                                                      const double *__restrict__ a, double sign,
                                                      const double *__restrict__ x, double *__restrict__ y)
{
    using M = Mfma<double>;
    constexpr int TI = 4 / KSPL;                 // i tiles of a workgroup
    constexpr int GC = CX_KC / 16 / KSPL;        // groups of 16 k per wave and chunk
    constexpr int PF = 2;                        // groups in flight of each sum
    constexpr int LDX = CX_KC + 1, NST = 16 * CX_KC / 256;
    __shared__ double sx[2][2][16 * LDX];        // [buffer][plane]: X(k0 + k, c) at k + LDX c
    const int v = (int)(blockIdx.z % (unsigned)nvec);
    const long b = blockIdx.z / (unsigned)nvec;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    const int ks = wave % KSPL, ti = (int)blockIdx.x * TI + wave / KSPL, tc = (int)blockIdx.y;
    const int P = n1 * n2;
    const double *xp = x + 2L * v * N + (long)P * b;
    const int i = min(ti * 16 + lr, n1 - 1), ca = min(tc * 16 + lr, n2 - 1);
    const auto rxr = buf_rsrc(xp, 8L * P), rxi = buf_rsrc(xp + N, 8L * P), rh1 = buf_rsrc(h1, 16L * n1 * n1),
               rh2 = buf_rsrc(h2, 16L * n2 * n2), rr = buf_rsrc(res + (long)P * b, 8L * P);
    // without an imaginary diagonal: one zero, read by every lane
    const auto ra = a ? buf_rsrc(a + (long)P * b, 8L * P) : buf_rsrc(&k_zero_d, 8);

    // first sum, A(c,k) = X(k,c), B(k,i) = H1(i,k)
    const int xk = tid & (CX_KC - 1), xc = tid / CX_KC;
    const int xv = (xk + n1 * (tc * 16 + xc)) * 8, xstep = n1 * (256 / CX_KC) * 8;
    struct Chunk {
        double re[NST], im[NST];
    };
    auto load_x = [&](int k0, Chunk &r) {
#pragma unroll
        for (int u = 0; u < NST; u++) {
            r.re[u] = buf_ld<double, double>(rxr, xv + k0 * 8 + u * xstep, 0);
            r.im[u] = buf_ld<double, double>(rxi, xv + k0 * 8 + u * xstep, 0);
        }
    };
    auto stage_x = [&](int k0, const Chunk &r, double (&d)[2][16 * LDX]) {   // a k past the end has read the next column
#pragma unroll
        for (int u = 0; u < NST; u++) {
            const int o = xk + LDX * (xc + 256 / CX_KC * u);
            d[0][o] = k0 + xk < n1 ? r.re[u] : 0.0;
            d[1][o] = k0 + xk < n1 ? r.im[u] : 0.0;
        }
    };
    const int hv = (i + n1 * lk) * 16;
    auto load_h = [&](int g, dcx(&r)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) r[u] = buf_ld_cx(rh1, hv + n1 * (16 * g + 4 * u) * 16);
    };
    // second sum, A(c,j) = H2(c,j), B(j,i) = X(i,j)
    const int gv = (ca + n2 * lk) * 16, yv = (i + n1 * lk) * 8;
    const int G2 = (n2 + 15) / 16;
    auto load2 = [&](int g, dcx(&h)[4], double (&p)[4], double (&q)[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            h[u] = buf_ld_cx(rh2, gv + n2 * (16 * g + 4 * u) * 16);
            p[u] = buf_ld<double, double>(rxr, yv + n1 * (16 * g + 4 * u) * 8, 0);
            q[u] = buf_ld<double, double>(rxi, yv + n1 * (16 * g + 4 * u) * 8, 0);
        }
    };
    Chunk st[2];
    dcx hb[PF][4], qh[PF][4];
    double qr[PF][4], qi[PF][4];
    load_x(0, st[0]);
    load_x(CX_KC, st[1]);
#pragma unroll
    for (int u = 0; u < PF; u++) load_h(ks + KSPL * u, hb[u]);
    const int ov = i + n1 * (tc * 16 + lk);
    const dcx d2 = dep2 ? dep2[i] : dcx{1.0, 0.0};
#pragma unroll
    for (int u = 0; u < PF; u++) load2(ks + KSPL * u, qh[u], qr[u], qi[u]);
    cacc acc{}, acc2{};
    const int nch = (n1 + CX_KC - 1) / CX_KC;
    stage_x(0, st[0], sx[0]);
    // chunk ch, while chunk ch + 2 loads and chunk ch + 1 goes to the other buffer
    auto chunk = [&](int ch, Chunk &mine, const Chunk &next, double (&cur)[2][16 * LDX], double (&other)[2][16 * LDX],
                     auto hslot) {
        constexpr int H0 = decltype(hslot)::value;
        __syncthreads();   // chunk ch is staged, and the other buffer read by all
        load_x(CX_KC * (ch + 2), mine);
        const int o = LDX * lr + 16 * ks + lk, g0 = ch * (CX_KC / 16) + ks;
#pragma unroll
        for (int u = 0; u < GC; u++) {
#pragma unroll
            for (int w = 0; w < 4; w++)
                cx_mma<false>(acc, hb[(H0 + u) % PF][w], cur[0][o + 16 * KSPL * u + 4 * w],
                              cur[1][o + 16 * KSPL * u + 4 * w]);
            load_h(g0 + KSPL * (u + PF), hb[(H0 + u) % PF]);
        }
        stage_x(CX_KC * (ch + 1), next, other);
    };
    int ch = 0;
    for (; ch + 2 <= nch; ch += 2) {
        chunk(ch, st[0], st[1], sx[0], sx[1], std::integral_constant<int, 0>());
        chunk(ch + 1, st[1], st[0], sx[1], sx[0], std::integral_constant<int, GC % PF>());
    }
    if (ch < nch) chunk(ch, st[0], st[1], sx[0], sx[1], std::integral_constant<int, 0>());
    const int G = (G2 - ks + KSPL - 1) / KSPL;   // groups of this share
    int g = 0;
    for (; g + PF <= G; g += PF) {
#pragma unroll
        for (int u = 0; u < PF; u++) {
#pragma unroll
            for (int w = 0; w < 4; w++) cx_mma<true>(acc2, qh[u][w], qr[u][w], qi[u][w]);
            load2(ks + KSPL * (g + u + PF), qh[u], qr[u], qi[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < PF - 1; u++)
        if (g + u < G)
#pragma unroll
            for (int w = 0; w < 4; w++) cx_mma<true>(acc2, qh[u][w], qr[u][w], qi[u][w]);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        acc.re[q] += d2.re * acc2.re[q] - d2.im * acc2.im[q];
        acc.im[q] += d2.re * acc2.im[q] + d2.im * acc2.re[q];
    }
    if constexpr (KSPL > 1) {
        double *red = &sx[0][0][0];   // 4 waves x 2 x 256 <= 2 planes x 16 x 65 x 2
        __syncthreads();              // the last chunk is read
#pragma unroll
        for (int q = 0; q < 4; q++) {
            red[512 * wave + 64 * q + lane] = acc.re[q];
            red[512 * wave + 256 + 64 * q + lane] = acc.im[q];
        }
        __syncthreads();
        if (ks != 0) return;   // no barrier follows
#pragma unroll
        for (int q = 0; q < 4; q++)
            for (int k = 1; k < KSPL; k++) {
                acc.re[q] += red[512 * (wave + k) + 64 * q + lane];
                acc.im[q] += red[512 * (wave + k) + 256 + 64 * q + lane];
            }
    }
    double *yp = y + 2L * v * N + (long)P * b;
    const auto ryr = buf_rsrc(yp, 8L * P), ryi = buf_rsrc(yp + N, 8L * P);
    double dv[4], av[4], pr[4], pi[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int o = (ov + n1 * M::row(0, q)) * 8;
        dv[q] = buf_ld<double, double>(rr, o, 0);
        av[q] = buf_ld<double, double>(ra, a ? o : 0, 0);
        pr[q] = buf_ld<double, double>(rxr, o, 0);
        pi[q] = buf_ld<double, double>(rxi, o, 0);
    }
    // rows past the last c lie past the plane and are dropped
    if (ti * 16 + lr < n1)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int o = (ov + n1 * M::row(0, q)) * 8;
            const double d = dv[q] - sh, t = sign * av[q];
            buf_st<double, double>(ryr, o, 0, acc.re[q] + (d * pr[q] - t * pi[q]));
            buf_st<double, double>(ryi, o, 0, acc.im[q] + (d * pi[q] + t * pr[q]));
        }
}

// A further level, added to Y: y(d, i, b) += [DEP(d)] sum_j H(i, j) x(d, j, b).
// A wave takes 16 points d and 16 rows i, a workgroup four such tiles of d;
// grid: (groups of d tiles, i tiles, block and vector).
__global__ void __launch_bounds__(256) k_cxh_outer(int nin, int n, int nvec, const dcx *__restrict__ h,
                                                   const dcx *__restrict__ dep, long N, const double *__restrict__ x,
                                                   double *__restrict__ y)
{
    using M = Mfma<double>;
    constexpr int PF = 4;
    const int v = (int)(blockIdx.z % (unsigned)nvec);
    const long b = blockIdx.z / (unsigned)nvec;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    const int d0 = ((int)blockIdx.x * 4 + wave) * 16, i0 = (int)blockIdx.y * 16;
    if (d0 >= nin) return;
    const long P = (long)nin * n;
    const double *xp = x + 2L * v * N + P * b;
    double *yp = y + 2L * v * N + P * b;
    const auto rxr = buf_rsrc(xp, 8 * P), rxi = buf_rsrc(xp + N, 8 * P), ryr = buf_rsrc(yp, 8 * P),
               ryi = buf_rsrc(yp + N, 8 * P), rh = buf_rsrc(h, 16L * n * n);
    const int d = min(d0 + lr, nin - 1);
    const int hv = (min(i0 + lr, n - 1) + n * lk) * 16, xv = (d + nin * lk) * 8;
    dcx hb[PF][4];
    double qr[PF][4], qi[PF][4];
    auto load = [&](int g, int s) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = 16 * g + 4 * u;
            hb[s][u] = buf_ld_cx(rh, hv + n * k * 16);
            qr[s][u] = buf_ld<double, double>(rxr, xv + nin * k * 8, 0);
            qi[s][u] = buf_ld<double, double>(rxi, xv + nin * k * 8, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < PF; u++) load(u, u);
    double yr[4], yi[4];
    const int ov = (d + nin * (i0 + lk)) * 8;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        yr[q] = buf_ld<double, double>(ryr, ov + nin * M::row(0, q) * 8, 0);
        yi[q] = buf_ld<double, double>(ryi, ov + nin * M::row(0, q) * 8, 0);
    }
    const dcx dv = dep ? dep[d] : dcx{1.0, 0.0};
    cacc acc{};
    const int G = (n + 15) / 16;
    int g = 0;
    for (; g + PF <= G; g += PF) {
#pragma unroll
        for (int u = 0; u < PF; u++) {
#pragma unroll
            for (int w = 0; w < 4; w++) cx_mma<true>(acc, hb[u][w], qr[u][w], qi[u][w]);
            load(g + u + PF, u);
        }
    }
#pragma unroll
    for (int u = 0; u < PF - 1; u++)
        if (g + u < G)
#pragma unroll
            for (int w = 0; w < 4; w++) cx_mma<true>(acc, hb[u][w], qr[u][w], qi[u][w]);
    // rows past the last i lie past the block and are dropped
    if (d0 + lr < nin)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int o = ov + nin * M::row(0, q) * 8;
            buf_st<double, double>(ryr, o, 0, yr[q] + (dv.re * acc.re[q] - dv.im * acc.im[q]));
            buf_st<double, double>(ryi, o, 0, yi[q] + (dv.re * acc.im[q] + dv.im * acc.re[q]));
        }
}

// 32-bit byte offsets of the loads in flight (less than 1,024 indices past the
// end) and the grid's y and z ranges
static bool cx_tiles_fit(long nin, long n, long nz)
{
    return (nin + 1024) * (n + 1024) * 8 < 0x7fffffffL && (n + 1024) * (n + 1024) * 16 < 0x7fffffffL && nz <= 65535;
}

// Where the tiles pay, as in the real generic path: about 6 ns per workgroup and
// chunk of 64 summed indices of the first pass, 2.5 ns per wave of a further level, against
// 1 ps per multiply-add of k_cxh_level_lds and the launches that the first pass saves.
// us of MYHX_CX with the first pass by tiles / by outputs: (4,4,12,12,12) with 16 vectors
// 394 / 48, (1,50,20,20) with 16 547 / 66, (2,100,12,12,12) with 4 1,273 / 185, (32,32,10,10) with
// 4 35 / 50; a further level of 2 points on 144 inner
// ones 162 / 118, of 96 points 100 / 150.
static bool cx_levels12_pays(long n1, long n2, long nz)
{
    const long ti = (n1 + 15) / 16, tc = (n2 + 15) / 16, tiles = ti * tc * nz, simds = 4L * g_num_cu;
    const long k = 4 * tiles <= simds ? 4 : (2 * tiles <= simds ? 2 : 1);
    const long wg = (ti * k + 3) / 4 * tc * nz, chunks = (n1 + 63) / 64 + (n2 + 63) / 64;
    return wg * chunks * 6000 <= 8000000L + n1 * n2 * nz * (n1 + n2);
}
static bool cx_outer_pays(long P, long n, long nz)
{
    const long waves = ((P + 15) / 16) * ((n + 15) / 16) * nz;
    return waves <= 4L * g_num_cu || waves * 2500 <= P * n * nz * n;
}

// waves per tile: as many as leave about one wave per SIMD
static void launch_cxh_levels12(int n1, int n2, int nplane, int nvec, const dcx *h1, const dcx *h2, const dcx *dep2,
                                long N, const double *res, double sh, const double *a, double sign, const double *x,
                                double *y, hipStream_t s)
{
    const int nti = (n1 + 15) / 16, ntc = (n2 + 15) / 16;
    const long simds = 4L * g_num_cu, tiles = (long)nti * ntc * nplane * nvec;
#define CL(K)                                                                                              \
    hipLaunchKernelGGL((k_cxh_levels12<K>), dim3((nti * K + 3) / 4, ntc, nplane *nvec), dim3(256), 0, s, n1, n2, \
                       nvec, h1, h2, dep2, N, res, sh, a, sign, x, y)
    if (4 * tiles <= simds) CL(4);
    else if (2 * tiles <= simds) CL(2);
    else CL(1);
#undef CL
}

// the sNDVR layer: y(p, i) += sum_j A(p, i, j) x(p, j), A(p, i, j) at
// p + nin (i + n j)
__global__ void __launch_bounds__(256) k_cxh_outh(int nin, int n, const dcx *__restrict__ a, long N,
                                                  const double *__restrict__ x, double *__restrict__ y)
{
    const int v = blockIdx.y;
    const double *xr = x + 2L * v * N, *xi = xr + N;
    double *yr = y + 2L * v * N, *yi = yr + N;
    const long total = (long)nin * n;
    for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
        const int p = (int)(idx % nin), i = (int)(idx / nin);
        double ar = 0.0, ai = 0.0;
        for (int j = 0; j < n; j++) {
            const dcx av = a[p + (long)nin * (i + (long)n * j)];
            const double pr = xr[p + (long)nin * j], pi = xi[p + (long)nin * j];
            ar += av.re * pr - av.im * pi;
            ai += av.re * pi + av.im * pr;
        }
        yr[idx] += ar;
        yi[idx] += ai;
    }
}

static bool scx_complete(const scalit_ctx *c)
{
    for (int l = 0; l < c->sF; l++) {
        const Level &L = c->lv[l];
        if (c->ndvr && l == c->sF - 1) {
            if (!c->has_outhcx) return false;
        } else if (!L.has_h0cx || (L.dep && !L.has_depcx)) {
            return false;
        }
    }
    return true;
}

// the real level matrices that MYHX_DX applies are all there
bool real_levels_ready(const scalit_ctx *c)
{
    for (int l = 0; l < c->sF; l++) {
        const Level &L = c->lv[l];
        if (c->ndvr && l == c->sF - 1) continue;   // the OUTH layer
        if (!L.has_h0 || (L.dep && !L.has_dep)) return false;
    }
    return true;
}

int hx_apply_cxh(scalit_ctx *c, int ntype, int nvec, const double *x, double *y, hipStream_t s)
{
    int rc = SCALIT_OK;
    double sign = 0.0;
    const double *a = cx_imag_diag(c, ntype, &sign, &rc);
    SC_TRY(rc);
    if (!c->has_res || !scx_complete(c)) return SCALIT_ESTATE;
    const long N = c->N;
    const double sh = (ntype == SCALIT_TA0 || ntype == SCALIT_TAAP0 || ntype == SCALIT_TMAP0) ? 0.0 : c->e0;
    const Level *L = c->lv;
    auto hcx = [&](int l) { return (const dcx *)L[l].h0cx.p; };
    auto dcxp = [&](int l) { return L[l].dep ? (const dcx *)L[l].depcx.p : (const dcx *)nullptr; };
    // the diagonal and levels 1 and 2 in one pass where both are level matrices
    int l = 0;
    if (c->sF >= 2 + (c->ndvr ? 1 : 0) && cx_tiles_fit(L[0].n, L[0].n, 1) &&
        cx_tiles_fit(L[0].n, L[1].n, (long)L[1].blk * nvec) &&
        cx_levels12_pays(L[0].n, L[1].n, (long)L[1].blk * nvec)) {
        launch_cxh_levels12(L[0].n, L[1].n, L[1].blk, nvec, hcx(0), hcx(1), dcxp(1), N, c->res.p, sh, a, sign, x, y, s);
        l = 2;
    } else {
        hipLaunchKernelGGL(k_cxh_diag, dim3(cxh_grid(N), nvec), dim3(256), 0, s, N, c->res.p, sh, a, sign, x, y);
    }
    for (; l < c->sF; l++) {
        const int n = L[l].n, nin = L[l].dim, blk = L[l].blk;
        if (c->ndvr && l == c->sF - 1)
            hipLaunchKernelGGL(k_cxh_outh, dim3(cxh_grid((long)nin * n), nvec), dim3(256), 0, s, nin, n,
                               (const dcx *)c->outhcx.p, N, x, y);
        else if (nin > 1 && cx_tiles_fit(nin, n, (long)blk * nvec) && cx_outer_pays(nin, n, (long)blk * nvec))
            hipLaunchKernelGGL(k_cxh_outer,
                               dim3((unsigned)((nin + 63) / 64), (unsigned)((n + 15) / 16), (unsigned)(blk * nvec)),
                               dim3(256), 0, s, nin, n, nvec, hcx(l), dcxp(l), N, x, y);
        else if (n <= 256)
            hipLaunchKernelGGL(k_cxh_level_lds, dim3((unsigned)(((long)nin * blk + XC - 1) / XC), nvec), dim3(256),
                               sizeof(dcx) * (size_t)XC * n, s, nin, n, blk, hcx(l), dcxp(l), N, x, y);
        else
            hipLaunchKernelGGL(k_cxh_level, dim3(cxh_grid(N), nvec), dim3(256), 0, s, nin, n, blk, hcx(l), dcxp(l), N,
                               x, y);
    }
    HIP_TRY(hipGetLastError());
    return SCALIT_OK;
}

// upload n complex values given as separate real and imaginary parts into
// buf as (re, im) pairs; a new allocation bumps the operator generation
static int upload_cx(scalit_ctx *c, DBuf<double> &buf, long n, const double *re, const double *im)
{
    std::vector<double> t(2 * (size_t)n);
    for (long k = 0; k < n; k++) {
        t[2 * k] = re[k];
        t[2 * k + 1] = im[k];
    }
    const double *old = buf.p;
    SC_TRY(buf.alloc(2 * (size_t)n));
    if (buf.p != old) c->gen++;
    HIP_TRY(hipMemcpy(buf.p, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice));
    return SCALIT_OK;
}

}  // namespace scalit

using namespace scalit;

extern "C" {

int scalit_set_h0_cx(scalit_ctx *c, int level, const double *h0_re, const double *h0_im)
{
    if (!c || level < 1 || level > c->sF || !h0_re || !h0_im) return SCALIT_EINVAL;
    HIP_TRY(hipSetDevice(c->device));
    Level &L = c->lv[level - 1];
    SC_TRY(upload_cx(c, L.h0cx, (long)L.n * L.n, h0_re, h0_im));
    L.has_h0cx = true;
    return SCALIT_OK;
}

int scalit_set_dep_cx(scalit_ctx *c, int level, const double *dep_re, const double *dep_im)
{
    if (!c || level < 1 || level > c->sF || !dep_re || !dep_im) return SCALIT_EINVAL;
    HIP_TRY(hipSetDevice(c->device));
    Level &L = c->lv[level - 1];
    if (!L.dep) return SCALIT_EINVAL;
    SC_TRY(upload_cx(c, L.depcx, L.dim, dep_re, dep_im));
    L.has_depcx = true;
    return SCALIT_OK;
}

int scalit_set_outh_cx(scalit_ctx *c, const double *outh_re, const double *outh_im)
{
    if (!c || !outh_re || !outh_im) return SCALIT_EINVAL;
    if (c->sF < 2) return SCALIT_EINVAL;
    HIP_TRY(hipSetDevice(c->device));
    SC_TRY(upload_cx(c, c->outhcx, c->N * (long)c->lv[c->sF - 1].n, outh_re, outh_im));
    c->has_outhcx = true;
    // sNDVR, as scalit_set_outh sets it: the outermost level is the layer
    // and has no DEP (osb.print.h:204)
    c->ndvr = true;
    c->lv[c->sF - 1].dep = false;
    c->fast3 = fast3_ok(c);
    return SCALIT_OK;
}

int scalit_set_scx(scalit_ctx *c, int on)
{
    if (!c) return SCALIT_EINVAL;
    if (on && !scx_complete(c)) return SCALIT_ESTATE;
    if (c->scx != (on != 0)) {
        c->scx = on != 0;
        c->gen++;
    }
    return SCALIT_OK;
}

}  // extern "C"
