// The OSB set-up of a real separable level: the joint Jacobi of MJACOBI
// (src/iterate/libiterate/diag/jacobi.f90:2-83) on the blocks
//   HOSB(d) = DEP(d) H0 + diag(EIG0(d, .)),  d = 1..NDK
// (hinitxyz.f90:7-29, hinitdep.f90:10-34) without HOSB in memory and without
// one launch, or one workgroup pass, per rotation.
//
//  * Order.  Rotations of disjoint pairs touch disjoint entries of what the
//    angles are computed from, so they commute; only pairs that share an
//    index keep the reference's order (i = 1..MAK-1, j = 1..MAK-i, pair
//    (j, j+i)).  Scheduling every pair right after the last earlier pair with
//    one of its indices leaves 190 steps of up to 35 rotations for the 3,160
//    pairs of MAK = 80 (230 of up to 45 for the 4,560 of MAK = 96): the same
//    sweep with a 17 to 20 times shorter serial chain.
//  * No HOSB.  With V the accumulated rotation and U = H0 V, the entries a
//    rotation of (p, q) needs are
//      H_d(p,q) = sum_k E(d,k) V(k,p) V(k,q) + DEP(d) (V(:,p) . U(:,q))
//    for all d at once, a product of the NDK x MAK matrix E = EIG0 with the
//    columns V(:,p) o V(:,q) of a step's pairs (FP64 MFMA), and the diagonals
//    H_d(p,p), which are kept and updated.  A rotation then updates two
//    columns of V and of U instead of two rows and two columns of NDK
//    matrices.
//  * NDK > MAK + 1.  The angles depend on the NDK matrices through sums over
//    d of products of their entries, which an orthogonal mixing of d leaves
//    unchanged, and the matrices span at most MAK + 1 dimensions (H0 and the
//    MAK diagonal positions): the R factor of a Householder QR of the
//    NDK x (MAK + 1) matrix (DEP | EIG0) replaces it (tsqr below).
//  * The stopping measure changes only by the pairs that rotate (the other
//    entries of a rotated row pair keep their sum of squares), so its change
//    over a sweep is the sum over rotations of A' - A, A' the pair's sum of
//    squares after the rotation, from the A, B, C of the angle.
//
// What bounds it: the serial chain of steps (a few hundred per sweep, each a
// handful of dependent LDS, MFMA and square-root latencies; the matrix pipe is 6% busy in
// level 2 at 64 x 96 x 80).  The set-up there: level 1 11.7 ms, level 2 6.4, level 3 4.2 and
// 1.1 for its R factor; 25 to 29 ms with the first P*X, against 679 with HOSB in memory
// and one launch (level 3, 24.6 us each), one workgroup pass (level 2) or one wave's
// pass (level 1) per rotation.  Those kernels (kernels_diag.hip) stay for what this
// form does not hold: complex level matrices, the dense sNDVR layer,
// levels above 128 points (8-bit pair indices, 9 tiles of d for 16 waves), and an
// H0 that is not symmetric (V(:,p) . U(:,q) would mix H0(p,q) and H0(q,p), of
// which the reference reads one).
#include "device_common.hpp"

#include <algorithm>
#include <vector>

namespace scalit {

// The rotation of a pair from A = sum H(p,q)^2, B = 2 sum H(p,q) DDG and
// C = sum DDG^2, and the change of A it makes.  The reference's angle is
// X = atan(B / (A - C)) / 4, less or plus pi/4 where A > C (jacobi.f90): a
// quarter of the angle T of the point (C - A, -B).  Its sine and cosine come
// from two half-angle steps, each by the root that does not cancel (atan, sin
// and cos would take the registers of this kernel's fragments).
struct Rot {
    double cs, sn, c2, s2, sc, dA;
};
// r = 1 / sqrt(x) and s = sqrt(x) to about an ulp for x in [1/4, 2]: the hardware estimate, a
// third-order and a second-order step, and s corrected by its own residual (a few
// dependent operations each where the library's square root and division take
// several times as many; the rotations of a step wait for them: level 1 at
// 64 x 96 x 80 13.7 -> 11.7 ms)
__device__ __forceinline__ void rsqrt_unit(double x, double &r, double &s)
{
    double y = __builtin_amdgcn_rsq(x);
    double e = fma(-(x * y), y, 1.0);
    y = fma(y * e, fma(0.375, e, 0.5), y);
    e = fma(-(x * y), y, 1.0);
    r = fma(0.5 * y, e, y);
    s = x * r;
    s = fma(fma(-s, s, x), 0.5 * r, s);
}
__device__ __forceinline__ Rot jacobi_rot(double A, double B, double C)
{
    double x = C - A, y = -B;
    const double m = fmax(fabs(x), fabs(y));
    Rot r{1.0, 0.0, 1.0, 0.0, 0.0, 0.0};
    if (m == 0.0) return r;
    int e;
    (void)frexp(m, &e);   // x, y scaled to at most 1, exactly
    x = ldexp(x, -e);
    y = ldexp(y, -e);
    double ih, t;
    rsqrt_unit(x * x + y * y, ih, t);   // in [1/4, 2)
    const double ct = x * ih, st = y * ih;
    // T / 2 in [-pi/2, pi/2] (T = -pi where B = 0 and A > C)
    double rg, g;
    rsqrt_unit(0.5 + 0.5 * fabs(ct), rg, g);
    const double h = fabs(st) * (0.5 * rg);
    const double cu = ct >= 0.0 ? g : h;
    const double su = copysign(ct >= 0.0 ? h : g, st > 0.0 ? 1.0 : -1.0);
    double rc;
    rsqrt_unit(0.5 + 0.5 * cu, rc, r.cs);
    r.sn = su * (0.5 * rc);
    // scaled back onto the circle: the half-angle steps leave cos^2 + sin^2 - 1 with a mean of
    // -3e-17 for angles of some 1e-5, which the thousands of rotations of a
    // column add up (V^T V - 1 at 24 x 32 x 24 1.5e-15 rms; with cos and sin, and with this
    // step, 5e-16)
    const double d = 0.5 * fma(-r.sn, r.sn, fma(-r.cs, r.cs, 1.0));
    r.cs = fma(r.cs, d, r.cs);
    r.sn = fma(r.sn, d, r.sn);
    r.c2 = r.cs * r.cs;
    r.s2 = r.sn * r.sn;
    r.sc = r.sn * r.cs;
    const double cc = r.c2 - r.s2, ss = 2 * r.sc;
    r.dA = cc * cc * A + cc * ss * B + ss * ss * C - A;
    return r;
}

// The sum over the 16 lanes of a row, the same value on each of them.
template <int N>
__device__ __forceinline__ double row_ror(double v)
{
    const long b = __builtin_bit_cast(long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + N, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + N, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double row_sum16(double v)
{
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    return v;
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Sum over the workgroup, the same value on every thread (red: one double
// per wave).
template <int NW>
__device__ __forceinline__ double wg_sum(double v, double *red)
{
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < NW; k++) s += red[k];
    return s;
}

// The reference's test between sweeps (hosbdiag.f90:23-43): the change of the
// measure as the difference of two rounded values, so that a change below
// its last place counts as none.
struct Conv {
    double ye, init, dye;
    int k;
    __device__ __forceinline__ Conv(double off) : ye(off), init(off), dye(off), k(1) {}
    __device__ __forceinline__ bool go(int bjmax, double bjtol) const { return fabs(dye) > init * bjtol && k <= bjmax; }
    __device__ __forceinline__ void sweep(double change)
    {
        const double s = ye + change;
        dye = s - ye;
        ye = s;
        k++;
    }
};

// ---------------------------------------------------------------- NDK = 1
// One workgroup per block, a row of 16 lanes per rotation of a step, KL
// elements of each column per lane: the lanes read the two columns of V and U
// once, form H(p,q) = V(:,p) . U(:,q) (U = (H0 + diag(EIG0)) V), rotate them in registers
// and write them back; one barrier per step.  U (and V, VL) in LDS.
// sched: nstep x mw pairs (p | q << 8), 0xffff where a step has fewer.
template <int KL, bool VL>
__global__ void __launch_bounds__(1024) k_jacobi_vec(int n, int nstep, int mw, const unsigned short *__restrict__ sched,
                                                     const double *__restrict__ h0, double *__restrict__ eig0,
                                                     double *__restrict__ vosb, int bjmax, double bjtol)
{
    extern __shared__ char smem_raw[];
    const int ld = n | 1;   // odd: the columns of a step start in different banks
    double *sU = (double *)smem_raw;
    double *sD = sU + (long)ld * n;   // the diagonal
    double *sR = sD + n;              // one value per wave
    const int tid = threadIdx.x, nt = blockDim.x, nw = nt >> 6;
    const long nn = (long)n * n;
    double *vb = vosb + nn * blockIdx.x;
    double *V = VL ? sR + 16 : vb;
    const int ldv = VL ? ld : n;
    double *eb = eig0 + (long)blockIdx.x * n;
    double off = 0.0;
    for (int e = tid; e < (int)nn; e += nt) {
        const int c = e / n, r = e - c * n;
        const double h = h0[e];
        sU[r + ld * c] = r == c ? h + eb[r] : h;
        V[r + ldv * c] = r == c ? 1.0 : 0.0;
        if (r == c) sD[r] = h + eb[r];
        if (r > c) off += h * h;
    }
    auto total = [&](double v) {
        v = wave_sum(v);
        __syncthreads();
        if ((tid & 63) == 0) sR[tid >> 6] = v;
        __syncthreads();
        double s = 0.0;
        for (int k = 0; k < nw; k++) s += sR[k];
        return s;
    };
    Conv cv(2.0 * total(off));
    const int grp = tid >> 4, lr = tid & 15;
    while (cv.go(bjmax, bjtol)) {
        double change = 0.0;
        unsigned pq = grp < mw ? sched[grp] : 0xffffu;
        for (int t = 0; t < nstep; t++) {
            const unsigned cur = pq;
            pq = (grp < mw && t + 1 < nstep) ? sched[(long)(t + 1) * mw + grp] : 0xffffu;
            if (cur != 0xffffu) {   // the same on the 16 lanes of a row
                const int p = cur & 255, q = cur >> 8;
                double *vp = V + (long)ldv * p, *vq = V + (long)ldv * q, *up = sU + ld * p, *uq = sU + ld * q;
                double a[KL], b[KL], c[KL], d[KL], h = 0.0;
                const double hpp = sD[p], hqq = sD[q];
#pragma unroll
                for (int k = 0; k < KL; k++) {
                    const int r = lr + 16 * k, rc = min(r, n - 1);
                    a[k] = vp[rc];
                    b[k] = vq[rc];
                    c[k] = up[rc];
                    d[k] = uq[rc];
                }
#pragma unroll
                for (int k = 0; k < KL; k++) h += lr + 16 * k < n ? a[k] * d[k] : 0.0;
                h = row_sum16(h);
                const double ddg = 0.5 * hpp - 0.5 * hqq;
                const Rot R = jacobi_rot(h * h, 2.0 * (h * ddg), ddg * ddg);
#pragma unroll
                for (int k = 0; k < KL; k++) {
                    const int r = lr + 16 * k;
                    if (r < n) {
                        vp[r] = R.cs * a[k] - R.sn * b[k];
                        vq[r] = R.cs * b[k] + R.sn * a[k];
                        up[r] = R.cs * c[k] - R.sn * d[k];
                        uq[r] = R.cs * d[k] + R.sn * c[k];
                    }
                }
                if (lr == 0) {
                    sD[p] = R.c2 * hpp + R.s2 * hqq - 2 * R.sc * h;
                    sD[q] = R.c2 * hqq + R.s2 * hpp + 2 * R.sc * h;
                    change += R.dA;
                }
            }
            __syncthreads();
        }
        cv.sweep(2.0 * total(change));
    }
    __syncthreads();
    if constexpr (VL)
        for (int e = tid; e < (int)nn; e += nt) {
            const int c = e / n, r = e - c * n;
            vb[e] = V[r + ld * c];
        }
    for (int r = tid; r < n; r += nt) eb[r] = sD[r];
}

// ---------------------------------------------------------------- NDK > 1
// One workgroup of 16 waves per block.  E is nd x n (value (d, k) at
// E + d + lde k + bse b), dep its nd factors of H0 (stride bsd per block; null:
// 1).  Wave w holds the MFMA A fragments of the 16 rows d of tile w % ndt for
// the whole kernel; per step it forms H_d(p,q) of its 16-pair tiles (B
// fragments V(k,p) V(k,q) from LDS), the pair's A/B/C over its d, and, once
// the workgroup's sums give the angle, rotates its part of the diagonals dg
// (nd rounded up to tiles x n per block, global); then all waves rotate the columns of V and U.
// Writes V to vosb and the rotated H0's diagonal V(:,i) . U(:,i) to wii.
constexpr int JB_WAVES = 16;
template <int NR, bool UL>
__global__ void __launch_bounds__(64 * JB_WAVES) k_jacobi_block(
    int n, int nd, int nstep, int mw, const int *__restrict__ cnt, const unsigned short *__restrict__ sched,
    const double *__restrict__ h0, const double *__restrict__ E, long lde, long bse, const double *__restrict__ dep,
    long bsd, double *dg, double *ug, double *__restrict__ vosb, double *__restrict__ wii, int bjmax, double bjtol)
{
    using M = Mfma<double>;
    constexpr int KS = 4 * NR, NT = 64 * JB_WAVES, PT = (NR + 1) / 2;   // pair tiles: at most n / 2 <= 8 NR pairs
    extern __shared__ char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    const int b = blockIdx.x;
    const long nn = (long)n * n;
    // columns padded with zeros to the MFMA tiles' rows (no bounds in the
    // products), and by one more in LDS to start in different banks
    constexpr int ld = 16 * NR + 1, ldu = UL ? ld : 16 * NR;
    const int ndt = (nd + 15) / 16, mp = 16 * PT;
    double *sV = (double *)smem_raw;
    double *sR = sV + (long)ld * n;                    // A/B/C of (d tile, pair): 3 ndt mp
    double *sC = sR + 3 * max(ndt, 6) * mp;            // cos, sin of a pair
    double *sU = UL ? sC + 2 * mp : ug + (long)ldu * n * b;
    E += bse * b;
    if (dep) dep += bsd * b;
    const int ndp = 16 * ndt;
    dg += (long)ndp * n * b;
    // the waves of one d tile: wpt of them, taking the pair tiles in turn
    const int wpt = JB_WAVES / ndt;
    const int dt = wave % ndt, wg = wave / ndt;
    const bool work = wg < wpt;
    // Row i of the A tile is d = 16 dt + 4 (i % 4) + i / 4, so that accumulator q of a
    // lane (row lk + 4 q) is d0 + q: its four diagonals are adjacent.
    const int d0 = 16 * dt + 4 * lk;
    double ef[KS], df[4];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const int d = 16 * dt + 4 * (lr & 3) + (lr >> 2), k = 4 * s + lk;
        ef[s] = (d < nd && k < n) ? E[d + lde * k] : 0.0;
    }
    double dsq = 0.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int d = d0 + q;
        df[q] = d < nd ? (dep ? dep[d] : 1.0) : 0.0;
        if (wg == 0 && lr == 0) dsq += df[q] * df[q];
    }
    double off = 0.0;
    for (int e = tid; e < 16 * NR * n; e += NT) {
        const int c = e / (16 * NR), r = e - c * (16 * NR);
        const double h = r < n ? h0[r + (long)n * c] : 0.0;
        sU[r + ldu * c] = h;
        sV[r + ld * c] = r == c ? 1.0 : 0.0;
        if (r > c) off += h * h;
    }
    for (int e = tid; e < ndp * n; e += NT) {
        const int i = e / ndp, d = e - i * ndp;
        dg[e] = d < nd ? (dep ? dep[d] : 1.0) * h0[i + (long)n * i] + E[d + lde * i] : 0.0;
    }
    const double sumd = wg_sum<JB_WAVES>(dsq, sC);
    off = wg_sum<JB_WAVES>(off, sC + JB_WAVES);
    Conv cv(2.0 * (sumd * off));
    __syncthreads();
    while (cv.go(bjmax, bjtol)) {
        double change = 0.0;
        for (int t = 0; t < nstep; t++) {
            const int m = cnt[t];
            const unsigned short *sp = sched + (long)t * mw;
            d4_t acc[PT];
            // H_d(p,q) and the sums over this wave's d
            if (work) {
#pragma unroll
                for (int u = 0; u < PT; u++) {
                    const int pr = 16 * (wg + wpt * u) + lr;
                    if (16 * (wg + wpt * u) >= m) break;
                    const unsigned pq = pr < m ? sp[pr] : 0u;
                    const int p = pq & 255, q = pq >> 8;
                    const d4_t gp = *(const d4_t *)(dg + d0 + ndp * p), gq = *(const d4_t *)(dg + d0 + ndp * q);
                    const double *vp = sV + ld * p + lk, *vq = sV + ld * q + lk, *uq = sU + ldu * q + lk;
                    d4_t ac = d4_t{0, 0, 0, 0};
                    double w = 0.0;
                    // groups of 4 k steps; the scheduling barrier bounds the values in flight
#pragma unroll
                    for (int s0 = 0; s0 < KS; s0 += 4) {
#pragma unroll
                        for (int s = s0; s < s0 + 4; s++) {
                            const double a = vp[4 * s];
                            ac = M::run(ef[s], a * vq[4 * s], ac);
                            w += a * uq[4 * s];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    w += __shfl_xor(w, 16);
                    w += __shfl_xor(w, 32);
                    double A = 0.0, B = 0.0, C = 0.0;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        ac[r] += df[r] * w;
                        const double ddg = 0.5 * gp[r] - 0.5 * gq[r];   // 0 past nd
                        A += ac[r] * ac[r];
                        B += ac[r] * ddg;
                        C += ddg * ddg;
                    }
                    acc[u] = ac;
                    A += __shfl_xor(A, 16);
                    B += __shfl_xor(B, 16);
                    C += __shfl_xor(C, 16);
                    A += __shfl_xor(A, 32);
                    B += __shfl_xor(B, 32);
                    C += __shfl_xor(C, 32);
                    if (lk == 0) {
                        double *o = sR + 3 * (dt * mp + pr);
                        o[0] = A;
                        o[1] = B;
                        o[2] = C;
                    }
                }
            }
            __syncthreads();
            // the angle (every wave of a pair the same), the diagonals
            if (work) {
#pragma unroll
                for (int u = 0; u < PT; u++) {
                    const int pr = 16 * (wg + wpt * u) + lr;
                    if (16 * (wg + wpt * u) >= m) break;
                    const unsigned pq = pr < m ? sp[pr] : 0u;
                    const int p = pq & 255, q = pq >> 8;
                    double A = 0.0, B = 0.0, C = 0.0;
                    for (int k = 0; k < ndt; k++) {
                        const double *o = sR + 3 * (k * mp + pr);
                        A += o[0];
                        B += o[1];
                        C += o[2];
                    }
                    const Rot R = jacobi_rot(A, 2.0 * B, C);
                    if (pr < m) {
                        d4_t *gp = (d4_t *)(dg + d0 + ndp * p), *gq = (d4_t *)(dg + d0 + ndp * q);
                        const d4_t hp = *gp, hq = *gq;
                        d4_t np, nq;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            np[r] = R.c2 * hp[r] + R.s2 * hq[r] - 2 * R.sc * acc[u][r];
                            nq[r] = R.c2 * hq[r] + R.s2 * hp[r] + 2 * R.sc * acc[u][r];
                        }
                        *gp = np;
                        *gq = nq;
                        if (dt == 0 && lk == 0) {
                            sC[2 * pr] = R.cs;
                            sC[2 * pr + 1] = R.sn;
                            change += R.dA;
                        }
                    }
                }
            }
            __syncthreads();
            // columns p and q of V and U
            for (int pr = wave; pr < m; pr += JB_WAVES) {
                const unsigned pq = sp[pr];
                const int p = pq & 255, q = pq >> 8;
                const double cs = sC[2 * pr], sn = sC[2 * pr + 1];
                for (int r = lane; r < n; r += 64) {
                    const double a = sV[r + ld * p], c = sV[r + ld * q];
                    const double e = sU[r + ldu * p], f = sU[r + ldu * q];
                    sV[r + ld * p] = cs * a - sn * c;
                    sV[r + ld * q] = cs * c + sn * a;
                    sU[r + ldu * p] = cs * e - sn * f;
                    sU[r + ldu * q] = cs * f + sn * e;
                }
            }
            __syncthreads();
        }
        cv.sweep(2.0 * wg_sum<JB_WAVES>(change, sC));
        __syncthreads();
    }
    for (int e = tid; e < (int)nn; e += NT) {
        const int c = e / n, r = e - c * n;
        vosb[nn * b + e] = sV[r + ld * c];
    }
    for (int i = wave; i < n; i += JB_WAVES) {
        double s = 0.0;
        for (int r = lane; r < n; r += 64) s += sV[r + ld * i] * sU[r + ldu * i];
        s = wave_sum(s);
        if (lane == 0) wii[(long)n * b + i] = s;
    }
}

// EIG0(d,i) = DEP(d) (V^T H0 V)(i,i) + sum_k E(d,k) V(k,i)^2, in place (E the
// old EIG0): a workgroup per 64 points d of a block, its E staged in LDS.
__global__ void __launch_bounds__(256) k_jacobi_eig(int n, int ndk, const double *__restrict__ dep,
                                                    const double *__restrict__ vosb, const double *__restrict__ wii,
                                                    double *__restrict__ eig0)
{
    extern __shared__ char smem_raw[];
    double *sE = (double *)smem_raw;   // E(d0 + dl, k) at dl + 64 k
    const int b = blockIdx.y, tid = threadIdx.x, dl = tid & 63, w = tid >> 6;
    const long d = (long)blockIdx.x * 64 + dl;
    double *eb = eig0 + (long)ndk * n * b;
    const double *vb = vosb + (long)n * n * b;
    const double dd = d < ndk ? (dep ? dep[d] : 1.0) : 0.0;
    for (int k = w; k < n; k += 4) sE[dl + 64 * k] = d < ndk ? eb[d + (long)ndk * k] : 0.0;
    __syncthreads();
    for (int i = w; i < n; i += 4) {
        const double *v = vb + (long)n * i;
        double s = dd * wii[(long)n * b + i];
        for (int k = 0; k < n; k++) s += sE[dl + 64 * k] * (v[k] * v[k]);
        if (d < ndk) eb[d + (long)ndk * i] = s;
    }
}

// ---------------------------------------------------------------- R factor
// Householder QR of chunks of mc rows of a rows x nc matrix (mc >= 2 nc), one
// workgroup per chunk: R (nc x nc, upper triangle, zeros below) of chunk g to
// rows g nc.. of the next round's matrix.  Applied until one chunk is left
// (R of stacked R factors is R of the whole).  The first round's matrix is
// (DEP | EIG0): column 0 dep (or 1), column 1 + k EIG0(., k).  The chunk is held
// in LDS (column r + mc c), or where that does not hold 2 nc rows in `buf`.
// In round j every wave forms the reflector of column j by itself (the same
// values) and applies it to columns j + 1 + wave, ...: one barrier a column.
constexpr int TS_NT = 1024, TS_RL = 8;   // rows per lane: mc <= 64 TS_RL
template <bool FIRST, bool LDS>
__global__ void __launch_bounds__(TS_NT) k_tsqr(long rows, int nc, int mc, const double *__restrict__ dep,
                                               const double *__restrict__ src, long sstride, double *buf,
                                               double *__restrict__ out, long ldo, long ostride)
{
    extern __shared__ char smem_raw[];
    const int b = blockIdx.y, g = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double *A = LDS ? (double *)smem_raw : buf + ((long)b * gridDim.x + g) * (long)mc * nc;
    src += sstride * b;
    out += ostride * b + (long)g * nc;
    const long r0 = (long)g * mc;
    for (int e = tid; e < mc * nc; e += TS_NT) {
        const int c = e / mc;
        const long r = r0 + (e - c * mc);
        double v = 0.0;
        if (r < rows) {
            if constexpr (FIRST) v = c == 0 ? (dep ? dep[r] : 1.0) : src[r + rows * (c - 1)];
            else v = src[r + rows * c];
        }
        A[e] = v;
    }
    __syncthreads();
    const int nrl = (mc + 63) / 64;
    for (int j = 0; j < nc; j++) {
        const double *aj = A + (long)mc * j;
        double v[TS_RL], s = 0.0;
#pragma unroll
        for (int u = 0; u < TS_RL; u++) {
            const int r = lane + 64 * u;
            v[u] = (u < nrl && r >= j && r < mc) ? aj[r] : 0.0;
            s += v[u] * v[u];
        }
        s = wave_sum(s);
        const double ajj = aj[j];
        const double alpha = ajj > 0.0 ? -sqrt(s) : sqrt(s);
        const double den = s - alpha * ajj;   // v . v / 2
        if (den > 0.0) {
            const double beta = 1.0 / den;
#pragma unroll
            for (int u = 0; u < TS_RL; u++)
                if (lane + 64 * u == j) v[u] = ajj - alpha;
            for (int c = j + 1 + wave; c < nc; c += TS_NT / 64) {
                double *ac = A + (long)mc * c;
                double x[TS_RL], t = 0.0;
#pragma unroll
                for (int u = 0; u < TS_RL; u++) {
                    const int r = lane + 64 * u;
                    x[u] = (u < nrl && r >= j && r < mc) ? ac[r] : 0.0;
                    t += v[u] * x[u];
                }
                t = beta * wave_sum(t);
#pragma unroll
                for (int u = 0; u < TS_RL; u++) {
                    const int r = lane + 64 * u;
                    if (u < nrl && r >= j && r < mc) ac[r] = x[u] - t * v[u];
                }
            }
        }
        // R(j,j); the entries below it are never read again
        if (wave == 0 && lane == 0) out[j + ldo * j] = den > 0.0 ? alpha : ajj;
        __syncthreads();
    }
    for (int e = tid; e < nc * nc; e += TS_NT) {
        const int c = e / nc, r = e - c * nc;
        if (r < c) out[r + ldo * c] = A[r + (long)mc * c];
        else if (r > c) out[r + ldo * c] = 0.0;
    }
}

// ---------------------------------------------------------------- host
// the steps of one sweep: nstep rows of mw pairs (p | q << 8, 0xffff past a
// step's count)
struct Schedule {
    int nstep = 0, mw = 0;
    std::vector<int> cnt;
    std::vector<unsigned short> pairs;
    explicit Schedule(int n)
    {
        std::vector<int> last(n, 0);
        std::vector<std::vector<unsigned short>> st;
        for (int i = 1; i < n; i++)
            for (int p = 0; p + i < n; p++) {
                const int q = p + i, s = std::max(last[p], last[q]);
                last[p] = last[q] = s + 1;
                if ((int)st.size() <= s) st.resize(s + 1);
                st[s].push_back((unsigned short)(p | (q << 8)));
            }
        nstep = (int)st.size();
        for (auto &v : st) {
            cnt.push_back((int)v.size());
            mw = std::max(mw, (int)v.size());
        }
        pairs.assign((size_t)nstep * mw, 0xffffu);
        for (int t = 0; t < nstep; t++) std::copy(st[t].begin(), st[t].end(), pairs.begin() + (size_t)t * mw);
    }
};

// one sweep's schedule on the device (host copies end with this call)
static int upload_schedule(const Schedule &sc, DBuf<int> &cnt, DBuf<unsigned short> &pairs, hipStream_t s)
{
    SC_TRY(cnt.alloc(std::max<size_t>(sc.cnt.size(), 1)));
    SC_TRY(pairs.alloc(std::max<size_t>(sc.pairs.size(), 1)));
    if (sc.nstep > 0) {
        HIP_TRY(hipMemcpyAsync(cnt.p, sc.cnt.data(), sizeof(int) * sc.cnt.size(), hipMemcpyHostToDevice, s));
        HIP_TRY(hipMemcpyAsync(pairs.p, sc.pairs.data(), sizeof(unsigned short) * sc.pairs.size(),
                               hipMemcpyHostToDevice, s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    return SCALIT_OK;
}

constexpr size_t JC_LDS = 160 * 1024;

// LDS of k_jacobi_vec: U, the diagonal, one value per wave (and V)
static size_t vec_lds(int n, bool vl) { return sizeof(double) * ((size_t)(n | 1) * n * (vl ? 2 : 1) + n + 16); }

template <int KL>
static void launch_vec(int n, int nblk, const Schedule &sc, const unsigned short *pairs, const double *h0,
                       double *eig0, double *vosb, int bjmax, double bjtol, hipStream_t s)
{
    const int nt = std::max(64, (16 * sc.mw + 63) / 64 * 64);   // a row of 16 lanes for every pair of a step
    if (vec_lds(n, true) <= JC_LDS) {
        allow_full_lds((const void *)k_jacobi_vec<KL, true>);
        hipLaunchKernelGGL((k_jacobi_vec<KL, true>), dim3(nblk), dim3(nt), vec_lds(n, true), s, n, sc.nstep, sc.mw,
                           pairs, h0, eig0, vosb, bjmax, bjtol);
    } else {
        allow_full_lds((const void *)k_jacobi_vec<KL, false>);
        hipLaunchKernelGGL((k_jacobi_vec<KL, false>), dim3(nblk), dim3(nt), vec_lds(n, false), s, n, sc.nstep, sc.mw,
                           pairs, h0, eig0, vosb, bjmax, bjtol);
    }
}

bool jacobi_vec_fits(int n) { return n <= 128 && vec_lds(n, false) <= JC_LDS; }

int jacobi_level_vec(scalit_ctx *c, int l, int bjmax, double bjtol, hipStream_t s)
{
    Level &L = c->lv[l];
    const Schedule sc(L.n);
    DBuf<int> cnt;
    DBuf<unsigned short> pairs;
    SC_TRY(upload_schedule(sc, cnt, pairs, s));
    // values per lane: the next built count (3 and 7 are not built: 33 to 48 points run
    // as 64, 97 to 112 as 128)
#define JV(KL) launch_vec<KL>(L.n, L.blk, sc, pairs.p, L.h0.p, c->eig0.p, L.vosb.p, bjmax, bjtol, s)
    const int kl = (L.n + 15) / 16;
    if (kl <= 2) JV(2);
    else if (kl <= 4) JV(4);
    else if (kl == 5) JV(5);
    else if (kl == 6) JV(6);
    else JV(8);
#undef JV
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));
    return SCALIT_OK;
}

static size_t block_lds(int n, int nd, int nr, bool ul)
{
    const size_t mp = 16 * (size_t)((nr + 1) / 2), ndt = std::max((nd + 15) / 16, 6);
    return sizeof(double) * ((size_t)(16 * nr + 1) * n * (ul ? 2 : 1) + 3 * ndt * mp + 2 * mp);
}

template <int NR>
static int launch_block(int n, int nd, int nblk, const Schedule &sc, const int *cnt, const unsigned short *pairs,
                        const double *h0, const double *E, long lde, long bse, const double *dep, long bsd,
                        double *dg, DBuf<double> &ug, double *vosb, double *wii, int bjmax, double bjtol,
                        hipStream_t s)
{
    const bool ul = block_lds(n, nd, NR, true) <= JC_LDS;
    const size_t lds = block_lds(n, nd, NR, ul);
    if (ul) {
        allow_full_lds((const void *)k_jacobi_block<NR, true>);
        hipLaunchKernelGGL((k_jacobi_block<NR, true>), dim3(nblk), dim3(64 * JB_WAVES), lds, s, n, nd, sc.nstep,
                           sc.mw, cnt, pairs, h0, E, lde, bse, dep, bsd, dg, (double *)nullptr, vosb, wii, bjmax,
                           bjtol);
    } else {
        SC_TRY(ug.alloc((size_t)(16 * NR) * n * nblk));
        allow_full_lds((const void *)k_jacobi_block<NR, false>);
        hipLaunchKernelGGL((k_jacobi_block<NR, false>), dim3(nblk), dim3(64 * JB_WAVES), lds, s, n, nd, sc.nstep,
                           sc.mw, cnt, pairs, h0, E, lde, bse, dep, bsd, dg, ug.p, vosb, wii, bjmax, bjtol);
    }
    HIP_TRY(hipGetLastError());
    return SCALIT_OK;
}

// n <= 128: 8-bit indices, 9 tiles of d at most (one wave each)
bool jacobi_block_fits(int n) { return n <= 128; }

int jacobi_level_block(scalit_ctx *c, int l, int bjmax, double bjtol, hipStream_t s)
{
    Level &L = c->lv[l];
    const int n = L.n, ndk = L.dim, nblk = L.blk, nc = n + 1;
    const double *dep = L.dep ? L.depv.p : nullptr;
    const Schedule sc(n);
    DBuf<int> cnt;
    DBuf<unsigned short> pairs;
    DBuf<double> dg, ug, wii, r0, r1, chunk;
    SC_TRY(upload_schedule(sc, cnt, pairs, s));
    SC_TRY(wii.alloc((size_t)n * nblk));
    // (DEP | EIG0), or its R factor when that is smaller
    const double *E = c->eig0.p, *dd = dep;
    long lde = ndk, bse = (long)ndk * n, bsd = 0;
    int nd = ndk;
    if (ndk > nc) {
        int mc = (int)std::min<size_t>(64 * TS_RL, JC_LDS / sizeof(double) / nc);
        const bool in_lds = mc >= 2 * nc;
        if (!in_lds) mc = 64 * TS_RL;
        const size_t lds = in_lds ? sizeof(double) * (size_t)mc * nc : 0;
        long rows = ndk;
        bool first = true;
        DBuf<double> *in = &r0, *out = &r1;
        while (first || rows > nc) {
            const long g = (rows + mc - 1) / mc;
            SC_TRY(out->alloc((size_t)g * nc * nc * nblk));
            if (!in_lds) SC_TRY(chunk.alloc((size_t)g * mc * nc * nblk));
            const double *src = first ? c->eig0.p : in->p;
            const long ss = first ? bse : rows * nc;
            const dim3 grid((unsigned)g, (unsigned)nblk);
#define TS(F, LD)                                                                                            \
    do {                                                                                                     \
        allow_full_lds((const void *)k_tsqr<F, LD>);                                                         \
        hipLaunchKernelGGL((k_tsqr<F, LD>), grid, dim3(TS_NT), lds, s, rows, nc, mc, dep, src, ss, chunk.p,  \
                           out->p, g * nc, g * nc * nc);                                                     \
    } while (0)
            if (first && in_lds) TS(true, true);
            else if (first) TS(true, false);
            else if (in_lds) TS(false, true);
            else TS(false, false);
#undef TS
            HIP_TRY(hipGetLastError());
            rows = g * nc;
            first = false;
            std::swap(in, out);
        }
        // column 0 the factors of H0, column 1 + k the diagonal's
        nd = nc;
        dd = in->p;
        E = in->p + nc;
        lde = nc;
        bse = bsd = (long)nc * nc;
    }
    SC_TRY(dg.alloc((size_t)((nd + 15) / 16 * 16) * n * nblk));
    // tiles along n: the next built count (3 and 7 are not built here either)
#define JB(NR)                                                                                                      \
    launch_block<NR>(n, nd, nblk, sc, cnt.p, pairs.p, L.h0.p, E, lde, bse, dd, bsd, dg.p, ug, L.vosb.p, wii.p, bjmax, \
                     bjtol, s)
    const int nr = (n + 15) / 16;
    if (nr <= 2) SC_TRY(JB(2));
    else if (nr <= 4) SC_TRY(JB(4));
    else if (nr == 5) SC_TRY(JB(5));
    else if (nr == 6) SC_TRY(JB(6));
    else SC_TRY(JB(8));
#undef JB
    hipLaunchKernelGGL(k_jacobi_eig, dim3((unsigned)((ndk + 63) / 64), (unsigned)nblk), dim3(256),
                       sizeof(double) * 64 * (size_t)n, s, n, ndk, dep, L.vosb.p, wii.p, c->eig0.p);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(s));   // the scoped buffers end here
    return SCALIT_OK;
}

}  // namespace scalit
