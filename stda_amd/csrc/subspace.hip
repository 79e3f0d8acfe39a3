// Rayleigh-Ritz step of the block Davidson solver on the device: the kk lowest
// eigenpairs of the live part of the subspace matrix H, in one work-group.
//
// The host's LAPACK took 0.14 / 0.33 / 0.57 ms for 60 / 90 / 120 vectors plus two
// transfers and a wait of the idle device per iteration, half of a solve's time
// for molecules up to ~100 atoms; this kernel takes 0.11 / 0.17 / 0.24 ms (20
// pairs).  Everything below is latency: one work-group of four (or eight) waves
// keeps the matrix in registers, as an RT x 16 grid of threads (element (r, c) of
// the matrix at thread (r mod RT, c mod 16)): a row of the grid is one 16-lane
// DPP row, so the sums of a matrix-vector product need no LDS.  A column of the
// tridiagonalisation takes about 1 us (two barriers, two LDS round trips, three
// row sums and a square root in sequence), more than half of the kernel.
//
//  1. tridiagonalisation by Householder reflectors (Golub & Van Loan, Matrix
//     Computations, Alg. 8.3.1), two barriers per column; the reflectors go to
//     global scratch and come back in chunks of 32 for the back transformation;
//  2. the lowest kk eigenvalues by multisection of the Sturm count (Wilkinson),
//     eight lanes per eigenvalue: an interval shrinks ninefold per round.  The
//     count uses the polynomial recurrence, one dependent FMA per row, with the
//     rows read and the values rescaled in groups of eight;
//  3. eigenvectors of the tridiagonal from the twisted factorisation (Dhillon &
//     Parlett): forward and backward pivots on two waves, the twist where
//     |gamma| is least, two outward sweeps;
//  4. Z <- Z (3 I - Z^T Z) / 2 until Z is orthonormal to rounding; vectors of
//     eigenvalues too close for this (|Z^T Z - I| > 0.1) clear the ok flag and
//     the host solves the problem as before;
//  5. the reflectors applied to Z, two columns per 16-lane row.
//
// The matrix H itself stays on the device: the kernel adds the new columns'
// Gram block (mirrored) and keeps the result for the next iteration.
//
// Squares of the elements are summed unscaled: the largest element is to lie well
// within 1e-150 .. 1e150 (the solvers' are energies; stda_hip_sym_lowest scales).

#include "common.h"

#include <type_traits>

namespace stda {

namespace {

constexpr int RR_K = 32;          // vectors at most
constexpr int RR_LD = RR_K + 1;   // leading dimension of the LDS vector arrays
constexpr double RR_TINY = 1.0e-30;   // smallest |off-diagonal| of the scaled tridiagonal
constexpr double RR_PIV = 1.0e-100;   // smallest |pivot| of its factorisations

template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// sum over the 16 lanes of a DPP row, the same bits in every lane (rotations by
// 8, 4, 2, 1: each step adds the same two partial sums in both of their lanes)
__device__ __forceinline__ double row_sum(double x) {
    x += dpp_d<0x128>(x);
    x += dpp_d<0x124>(x);
    x += dpp_d<0x122>(x);
    x += dpp_d<0x121>(x);
    return x;
}
// 1/x to about an ulp (hardware reciprocal and one Newton step)
__device__ __forceinline__ double fast_rcp(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    return fma(r, fma(-x, r, 1.0), r);
}

// f(integral_constant<0>), ..., f(integral_constant<N - 1>)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

template <int MX>
struct RRSmem {
    double col[2][MX];    // the column being eliminated and the next one
    double pv[MX];        // A v
    double2 de[MX];       // d_i, e_{i-1}^2
    double d[MX], e[MX], e2[MX], tau[MX];
    double f[MX * RR_LD];   // forward pivots, then the vectors Z
    double g[MX * RR_LD];   // backward pivots, then reflector chunks
    double2 gram[RR_K * RR_K / 2];
    double lam[RR_K], lo[RR_K], hi[RR_K];
    double gam[RR_K];
    double red[16];
    int tw[RR_K];
    int idx[MX];
    int na, nnew, bad;
};

template <int MX, int RT>
__global__ void __launch_bounds__(16 * RT, 1) rr_lowest_kernel(RRArgs p) {
    constexpr int T = 16 * RT, NR = MX / RT, NC = MX / 16;
    constexpr int SUB = T / RR_K;            // lanes per eigenvalue
    constexpr int YC = (RR_K + RT - 1) / RT; // columns of Y per row of the grid
    static_assert(MX % RT == 0 && MX % 16 == 0 && RR_LD * MX >= 32 * MX, "sizes");
    __shared__ RRSmem<MX> sm;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tr = tid >> 4, tc = tid & 15;
    const int m0 = p.m0, m = p.m0 + p.mnew;

    // live columns, in order (wave 0)
    if (wave == 0) {
        int base = 0, nn = 0;
        for (int c = 0; c < m; c += 64) {
            const int i = c + lane;
            bool a = false;
            if (i < m0) a = p.restart || p.alive[i] != 0;
            else if (i < m) a = p.flags == nullptr || p.flags[i - m0] != 0.0;
            const unsigned long long mask = __ballot(a), old = __ballot(a && i < m0);
            if (a) sm.idx[base + __popcll(mask & ((1ull << lane) - 1))] = i;
            base += __popcll(mask);
            nn += __popcll(mask) - __popcll(old);
            if (i < m) p.alive[i] = a ? 1 : 0;
        }
        if (lane == 0) {
            sm.na = base;
            sm.nnew = nn;
            sm.bad = 0;
        }
    }
    __syncthreads();
    const int na = sm.na, kk = min(p.k, na);
    if (na == 0) {   // no live column (a start block of non-finite vectors): no pairs, ok = 0
        const int kc = min(p.k, m);
        for (int e = tid; e < m * kc; e += T) p.Y[e] = 0.0;
        if (tid < kc) p.theta[tid] = 0.0;
        if (tid < 4) p.info[tid] = 0.0;
        return;
    }

    // the symmetric matrix, kept in H for the next call.  Every element is read
    // by unconditional loads from a chosen address, so that they all overlap.
    // Lanes of a grid row read neighbouring rows of a column of H or gram.
    double A[NR][NC];
    {
        int ir[NR], ic[NC];
#pragma unroll
        for (int a = 0; a < NR; ++a) ir[a] = sm.idx[min(tr + RT * a, na - 1)];
#pragma unroll
        for (int b = 0; b < NC; ++b) ic[b] = sm.idx[min(tc + 16 * b, na - 1)];
#pragma unroll
        for (int a = 0; a < NR; ++a) {
            double u[NC], v[NC];
#pragma unroll
            for (int b = 0; b < NC; ++b) {
                const double *old = p.restart ? p.theta + min(ir[a], m0 - 1)
                                              : p.H + ic[b] + (int64_t)p.ldh * ir[a];
                const double *byc = ic[b] >= m0 ? p.gram + ir[a] + (int64_t)m * (ic[b] - m0) : old;
                const double *x = ir[a] >= m0 ? p.gram + ic[b] + (int64_t)m * (ir[a] - m0) : byc;
                u[b] = *x;
                v[b] = *(ic[b] >= m0 ? byc : x);
            }
#pragma unroll
            for (int b = 0; b < NC; ++b) {
                const bool in = tr + RT * a < na && tc + 16 * b < na;
                const bool zero = p.restart && ir[a] != ic[b] && max(ir[a], ic[b]) < m0;
                A[a][b] = in && !zero ? 0.5 * (u[b] + v[b]) : 0.0;
            }
        }
        __syncthreads();   // every element of H (and theta) read before any is written
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int b = 0; b < NC; ++b)
                if (tr + RT * a < na && tc + 16 * b < na)
                    p.H[ic[b] + (int64_t)p.ldh * ir[a]] = A[a][b];
    }

    // 1. tridiagonalisation; the owners of column j write it, diagonal included.
    // Columns 16 ph .. 16 ph + 15 touch the blocks a, b >= ph only: a loop body of
    // its own for each ph, without branches (conditions per block made every LDS
    // read of a column wait alone: 2.8 us a column at 120 rows).
    if (tc == 0) {
#pragma unroll
        for (int a = 0; a < NR; ++a) sm.col[0][tr + RT * a] = A[a][0];
    }
    __syncthreads();
    static_for<NC>([&](auto phase) {
        constexpr int ph = decltype(phase)::value, pr = 16 * ph / RT;   // first active blocks
        const int jend = min(16 * ph + 16, na);
        for (int j = 16 * ph; j < jend; ++j) {
            const double *x = sm.col[j & 1];
            // this thread's rows and columns of the column, and the sum of squares
            double vr[NR], vc[NC], s = 0.0;
#pragma unroll
            for (int a = pr; a < NR; ++a) vr[a] = x[tr + RT * a];
#pragma unroll
            for (int a = ph; a < NC; ++a) vc[a] = x[tc + 16 * a];
            const double alpha = x[min(j + 1, MX - 1)], dj = x[j];
#pragma unroll
            for (int a = ph; a < NC; ++a) {   // entries up to j + 1 left out
                const double y = (a > ph + 1 || tc + 16 * a > j + 1) ? vc[a] : 0.0;
                s = fma(y, y, s);
            }
            const double sigma = row_sum(s);
            double tau = 0.0, beta = alpha, inv = 0.0;
            if (sigma > 0.0) {
                const double t = fma(alpha, alpha, sigma);
                double r = __builtin_amdgcn_rsq(t);   // and two Newton steps
                r = fma(0.5 * r, fma(-t * r, r, 1.0), r);
                r = fma(0.5 * r, fma(-t * r, r, 1.0), r);
                const double mu = t * r;
                beta = alpha >= 0.0 ? -mu : mu;
                tau = (beta - alpha) * (alpha >= 0.0 ? -r : r);
                inv = fast_rcp(alpha - beta);
            }
            if (tid == 0) {
                sm.d[j] = dj;
                sm.e[j] = beta;
                sm.tau[j] = tau;
            }
            if (tau != 0.0) {
#pragma unroll
                for (int a = pr; a < NR; ++a) {   // the reflector: 0, 1 at j + 1, x inv beyond
                    vr[a] *= inv;
                    const int ri = tr + RT * a;
                    if (a <= pr + 1) vr[a] = ri > j + 1 ? vr[a] : (ri == j + 1 ? 1.0 : 0.0);
                }
#pragma unroll
                for (int a = ph; a < NC; ++a) {
                    vc[a] *= inv;
                    const int ci = tc + 16 * a;
                    if (a <= ph + 1) vc[a] = ci > j + 1 ? vc[a] : (ci == j + 1 ? 1.0 : 0.0);
                }
                if (tr == 0) {
#pragma unroll
                    for (int a = ph; a < NC; ++a) p.refl[(int64_t)MX * j + tc + 16 * a] = vc[a];
                }
                double t[NR];
#pragma unroll
                for (int a = pr; a < NR; ++a) {
                    t[a] = 0.0;
#pragma unroll
                    for (int b = ph; b < NC; ++b) t[a] = fma(A[a][b], vc[b], t[a]);
                }
#pragma unroll
                for (int a = pr; a < NR; ++a) t[a] = row_sum(t[a]);
                if (tc == 0) {
#pragma unroll
                    for (int a = pr; a < NR; ++a) sm.pv[tr + RT * a] = tau * t[a];
                }
                __syncthreads();
                double wr[NR], wc[NC], vp = 0.0;
#pragma unroll
                for (int a = pr; a < NR; ++a) wr[a] = sm.pv[tr + RT * a];
#pragma unroll
                for (int a = ph; a < NC; ++a) wc[a] = sm.pv[tc + 16 * a];
#pragma unroll
                for (int a = ph; a < NC; ++a) vp = fma(vc[a], wc[a], vp);
                const double K = -0.5 * tau * row_sum(vp);
#pragma unroll
                for (int a = pr; a < NR; ++a) wr[a] = fma(K, vr[a], wr[a]);
#pragma unroll
                for (int a = ph; a < NC; ++a) wc[a] = fma(K, vc[a], wc[a]);
#pragma unroll
                for (int a = pr; a < NR; ++a)
#pragma unroll
                    for (int b = ph; b < NC; ++b)
                        A[a][b] = fma(-vr[a], wc[b], fma(-wr[a], vc[b], A[a][b]));
            }
            double *y = sm.col[(j + 1) & 1];   // column j + 1, of block column ph or ph + 1
            const bool next = j + 1 == 16 * ph + 16;
            if (tc == ((j + 1) & 15)) {
#pragma unroll
                for (int a = pr; a < NR; ++a)
                    y[tr + RT * a] = next ? A[a][ph + 1 < NC ? ph + 1 : ph] : A[a][ph];
            }
            __syncthreads();
        }
    });

    // scaled to norm one; Gershgorin interval
    {
        double mn = 1.0e300, mx = -1.0e300, big = 0.0;
        if (tid < na) {
            const double r = (tid > 0 ? fabs(sm.e[tid - 1]) : 0.0) +
                             (tid + 1 < na ? fabs(sm.e[tid]) : 0.0);
            mn = sm.d[tid] - r;
            mx = sm.d[tid] + r;
            big = fmax(fabs(mn), fabs(mx));
            if (!(big < 1.0e300)) sm.bad = 1;   // infinities and NaN
        }
        for (int o = 32; o > 0; o >>= 1) {
            mn = fmin(mn, __shfl_xor(mn, o, 64));
            mx = fmax(mx, __shfl_xor(mx, o, 64));
        }
        if (lane == 0) {
            sm.red[wave] = mn;
            sm.red[8 + wave] = mx;
        }
    }
    __syncthreads();
    double glo = sm.red[0], ghi = sm.red[8];
#pragma unroll
    for (int q = 1; q < T / 64; ++q) {
        glo = fmin(glo, sm.red[q]);
        ghi = fmax(ghi, sm.red[8 + q]);
    }
    const double tn = fmax(fmax(fabs(glo), fabs(ghi)), 1.0e-290), sc = 1.0 / tn;
    if (tid < na) {
        sm.d[tid] *= sc;
        double e = tid + 1 < na ? sm.e[tid] * sc : 0.0;
        if (fabs(e) < RR_TINY) e = RR_TINY;
        sm.e[tid] = e;
        sm.e2[tid] = e * e;
        sm.de[tid].x = sm.d[tid];
        if (tid + 1 < na) sm.de[tid + 1].y = e * e;
        if (tid == 0) sm.de[0].y = 0.0;
    } else if (tid < (na + 7) / 8 * 8) {
        // rows that fill the last group: p_i = 2 p_{i-1} or more, no change of sign
        sm.de[tid] = make_double2(4.0, 0.0);
    }
    __syncthreads();

    // 2. multisection: the SUB lanes of group t narrow [lo, hi] around eigenvalue t
    const int t = tid / SUB, sub = tid % SUB;
    {
        double lo = glo * sc - 4.0e-15, hi = ghi * sc + 4.0e-15;
        for (int round = 0; round < (SUB == 16 ? 14 : 18); ++round) {   // (SUB + 1)^rounds > 1e17
            const double h = (hi - lo) * (1.0 / (SUB + 1));
            const double x = fma(h, (double)(sub + 1), lo);
            double pp = 0.0, pc = 1.0;
            unsigned sg = 0;      // sign bits of the last rows, newest first
            int cnt = 0;
            for (int i0 = 0; i0 < na; i0 += 8) {   // rows beyond na repeat the sign
                double2 de[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) de[q] = sm.de[i0 + q];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const double nx = fma(de[q].x - x, pc, -(de[q].y * pp));
                    pp = pc;
                    pc = nx;
                    sg = __builtin_amdgcn_alignbit(sg, (unsigned)__double2hiint(pc), 31);
                }
                cnt += __popc((sg ^ (sg >> 1)) & 0xffu);
                const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(pc), fabs(pp)));
                pc = __builtin_amdgcn_ldexp(pc, -ex);
                pp = __builtin_amdgcn_ldexp(pp, -ex);
            }
            const unsigned long long le = __ballot(cnt <= t);   // points below eigenvalue t
            const int q = __popc((unsigned)(le >> (lane / SUB * SUB)) & ((1u << SUB) - 1));
            hi = q < SUB ? fma(h, (double)(q + 1), lo) : hi;
            lo = q > 0 ? fma(h, (double)q, lo) : lo;
        }
        if (sub == 0) sm.lam[t] = 0.5 * (lo + hi);
    }
    __syncthreads();

    // 3. twisted factorisation: forward pivots (wave 0), backward pivots (wave 1)
    if (wave < 2 && lane < kk) {
        const double l = sm.lam[lane];
        if (wave == 0) {
            double D = sm.d[0] - l;
            if (fabs(D) < RR_PIV) D = -RR_PIV;
            sm.f[lane] = D;
            for (int i = 1; i < na; ++i) {
                D = fma(-sm.e2[i - 1], fast_rcp(D), sm.d[i] - l);
                if (fabs(D) < RR_PIV) D = -RR_PIV;
                sm.f[i * RR_LD + lane] = D;
            }
        } else {
            double D = sm.d[na - 1] - l;
            if (fabs(D) < RR_PIV) D = -RR_PIV;
            sm.g[(na - 1) * RR_LD + lane] = D;
            for (int i = na - 2; i >= 0; --i) {
                D = fma(-sm.e2[i], fast_rcp(D), sm.d[i] - l);
                if (fabs(D) < RR_PIV) D = -RR_PIV;
                sm.g[i * RR_LD + lane] = D;
            }
        }
    }
    __syncthreads();
    {   // the twist: least |gamma_i| = |D+_i + D-_i - (d_i - lambda)|
        double best = 1.0e301, bg = 0.0;
        int bi = 0;
        if (t < kk)
            for (int i = sub; i < na; i += SUB) {
                const double g = sm.f[i * RR_LD + t] + sm.g[i * RR_LD + t] - (sm.d[i] - sm.lam[t]);
                if (fabs(g) < best) { best = fabs(g); bg = g; bi = i; }
            }
        for (int o = SUB / 2; o > 0; o >>= 1) {
            const double ob = __shfl_xor(best, o, 64), og = __shfl_xor(bg, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ob < best || (ob == best && oi < bi)) { best = ob; bg = og; bi = oi; }
        }
        if (sub == 0) {
            sm.tw[t] = bi;
            sm.gam[t] = bg;
        }
    }
    __syncthreads();
    // outward sweeps into f: z_r = 1, z_i = -(e_i / D+_i) z_{i+1}, z_i = -(e_{i-1} / D-_i) z_{i-1}
    if (wave < 2 && lane < kk) {
        const int r = sm.tw[lane];
        double z = 1.0;
        if (wave == 0) {
            for (int i = na - 2; i >= 0; --i)
                if (i < r) {
                    z = -(sm.e[i] * fast_rcp(sm.f[i * RR_LD + lane])) * z;
                    sm.f[i * RR_LD + lane] = z;
                }
            sm.f[r * RR_LD + lane] = 1.0;
        } else {
            for (int i = 1; i < na; ++i)
                if (i > r) {
                    z = -(sm.e[i - 1] * fast_rcp(sm.g[i * RR_LD + lane])) * z;
                    sm.f[i * RR_LD + lane] = z;
                }
        }
    }
    __syncthreads();
    {   // unit vectors; eigenvalue corrected by gamma_r / |z|^2
        double s = 0.0;
        if (t < kk)
            for (int i = sub; i < na; i += SUB) s = fma(sm.f[i * RR_LD + t], sm.f[i * RR_LD + t], s);
        for (int o = SUB / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (t < kk) {
            if (!(s > 0.0 && s < 1.0e300)) sm.bad = 1;
            const double f = 1.0 / sqrt(s);
            for (int i = sub; i < na; i += SUB) sm.f[i * RR_LD + t] *= f;
            if (sub == 0) sm.lam[t] = fma(sm.gam[t], f * f, sm.lam[t]);
        }
    }
    __syncthreads();

    // 4. orthonormal to rounding; the step squares the deviation, so that one
    // from below 1e-8 needs no further look
    for (int pass = 0; pass < 8; ++pass) {
        constexpr int Q = RR_K / SUB;
        double acc[Q] = {};
        if (t < kk) {
#pragma unroll 4
            for (int i = 0; i < na; ++i) {   // columns from kk on hold stale pivots: not used
                const double zt = sm.f[i * RR_LD + t];
#pragma unroll
                for (int q = 0; q < Q; ++q) acc[q] = fma(zt, sm.f[i * RR_LD + sub + SUB * q], acc[q]);
            }
        }
        double dev = 0.0;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int u = sub + SUB * q;
            const bool in = t < kk && u < kk;
            const double one = t == u ? 1.0 : 0.0;
            const double x = in ? fabs(acc[q] - one) : 0.0;
            dev = x > dev || !(x == x) ? x : dev;
            reinterpret_cast<double *>(sm.gram)[t * RR_K + u] = in ? 1.5 * one - 0.5 * acc[q] : 0.0;
        }
        for (int o = 32; o > 0; o >>= 1) {
            const double x = __shfl_xor(dev, o, 64);
            dev = x > dev || !(x == x) ? x : dev;
        }
        if (lane == 0) sm.red[wave] = dev;
        __syncthreads();
        double dmax = 0.0;
#pragma unroll
        for (int q = 0; q < T / 64; ++q) dmax = sm.red[q] > dmax || !(sm.red[q] == sm.red[q]) ? sm.red[q] : dmax;
        if (!(dmax <= 0.1)) {   // or NaN
            if (tid == 0) sm.bad = 1;
            break;
        }
        // T / 256 threads a row, all of which read it before any writes
        const int row = tid % 256, part = tid / 256;
        double z[RR_K];
        if (row < na) {
#pragma unroll
            for (int q = 0; q < RR_K; ++q) z[q] = q < kk ? sm.f[row * RR_LD + q] : 0.0;
        }
        __syncthreads();
        if (row < na) {
            for (int u = 4 * part; u < kk; u += 4 * (T / 256)) {   // gram is zero beyond kk
                double y[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < RR_K; ++q) {
                    const double2 w0 = sm.gram[(q * RR_K + u) / 2], w1 = sm.gram[(q * RR_K + u) / 2 + 1];
                    y[0] = fma(z[q], w0.x, y[0]);
                    y[1] = fma(z[q], w0.y, y[1]);
                    y[2] = fma(z[q], w1.x, y[2]);
                    y[3] = fma(z[q], w1.y, y[3]);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) sm.f[row * RR_LD + u + r] = y[r];
            }
        }
        __syncthreads();
        if (dmax < 1.0e-8) break;
    }
    __syncthreads();

    // 5. Y = H_0 H_1 ... Z: columns tr + RT y, rows tc + 16 a
    double y[YC][NC];
#pragma unroll
    for (int a = 0; a < NC; ++a)
#pragma unroll
        for (int q = 0; q < YC; ++q) {
            const int i = tc + 16 * a, c = tr + RT * q;
            y[q][a] = (i < na && c < kk) ? sm.f[i * RR_LD + c] : 0.0;
        }
    for (int jc = (na - 1) / 32 * 32; jc >= 0; jc -= 32) {
        __syncthreads();   // the previous chunk consumed
        const int je = min(jc + 32, na);
        for (int e = tid; e < (je - jc) * MX; e += T) {
            const int j = jc + e / MX, i = e % MX;
            sm.g[e] = (i > j && i < na && sm.tau[j] != 0.0) ? p.refl[(int64_t)MX * jc + e] : 0.0;
        }
        __syncthreads();
        double va[NC];
#pragma unroll
        for (int a = 0; a < NC; ++a) va[a] = sm.g[(je - 1 - jc) * MX + tc + 16 * a];
        for (int j = je - 1; j >= jc; --j) {
            const double tau = sm.tau[j];
            double vn[NC], s[YC];   // the next reflector under way
            const double *v = sm.g + max(j - 1 - jc, 0) * MX;
#pragma unroll
            for (int a = 0; a < NC; ++a) vn[a] = v[tc + 16 * a];
#pragma unroll
            for (int q = 0; q < YC; ++q) {
                double s0 = 0.0, s1 = 0.0;
#pragma unroll
                for (int a = 0; a < NC; a += 2) {
                    s0 = fma(va[a], y[q][a], s0);
                    if (a + 1 < NC) s1 = fma(va[a + 1], y[q][a + 1], s1);
                }
                s[q] = -tau * row_sum(s0 + s1);
            }
#pragma unroll
            for (int a = 0; a < NC; ++a) {
#pragma unroll
                for (int q = 0; q < YC; ++q) y[q][a] = fma(s[q], va[a], y[q][a]);
                va[a] = vn[a];
            }
        }
    }
    // dead rows are zero, and so are the columns beyond the live ones
    const int kc = min(p.k, m);
    for (int e = tid; e < m * kc; e += T) p.Y[e] = 0.0;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NC; ++a)
#pragma unroll
        for (int q = 0; q < YC; ++q) {
            const int i = tc + 16 * a, c = tr + RT * q;
            if (i < na && c < kk) p.Y[sm.idx[i] + (int64_t)m * c] = y[q][a];
        }
    if (tid < kc) p.theta[tid] = tid < kk ? sm.lam[tid] * tn : 0.0;
    if (tid == 0) {
        p.info[0] = sm.bad ? 0.0 : 1.0;
        p.info[1] = (double)na;
        p.info[2] = (double)sm.nnew;
        p.info[3] = 0.0;
    }
}

}  // namespace

void launch_rr_lowest(hipStream_t s, const RRArgs &a) {
    const int m = a.m0 + a.mnew;
    if (m < 1 || m > RR_MMAX || a.k < 1 || a.k > RR_KMAX)
        throw Error(3, "rr_lowest: subspace outside the kernel's range");
    // The smallest tile that holds the matrix: the work per column grows with its
    // square.  With four waves a thread of the 128 tile holds 64 elements (all of
    // the kernel's sizes up to 128 measure within 5 % with four or eight waves);
    // beyond that eight waves share the matrix.
#define STDA_RR(MX, RT) \
    hipLaunchKernelGGL((rr_lowest_kernel<MX, RT>), dim3(1), dim3(16 * RT), 0, s, a)
    if (m <= 64) STDA_RR(64, 16);
    else if (m <= 96) STDA_RR(96, 16);
    else if (m <= 128) STDA_RR(128, 16);
    else if (m <= 160) STDA_RR(160, 32);
    else STDA_RR(192, 32);
#undef STDA_RR
    STDA_HIP_CHECK(hipGetLastError());
}

}  // namespace stda
