// linalg.hip -- fp64 reductions, the dense Hermitian Gram S = O^H diag(w) O, and
// the fp64 Cholesky / triangular solves of the shifted SR system (S + lambda I) x = F.
//
// The reference builds S with one complex atomic per (sample, k, k') and leaves
// the solve to the caller (source/network_functions/TDVP.cu.template:181-302);
// here S is a tiled GEMM with fp64 accumulation and the solve stays on the GPU.
#include "kernels.hpp"

#include <algorithm>

namespace ann {

namespace {

constexpr int kRed = 1024;
constexpr int kCus = 256;   // compute units of an MI355X

__global__ __launch_bounds__(kRed) void weighted_sums_kernel(const cplx<double>* e, const double* w,
                                                             int64_t n, double* out) {
    __shared__ double s0[kRed], s1[kRed], s2[kRed], s3[kRed];
    double a = 0, b = 0, c = 0, d = 0;
    for (int64_t i = threadIdx.x; i < n; i += kRed) {
        const double wi = w[i];
        const cplx<double> ei = e[i];
        a += wi * ei.re;
        b += wi * ei.im;
        c += wi * (ei.re * ei.re + ei.im * ei.im);
        d += wi;
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = b;
    s2[threadIdx.x] = c;
    s3[threadIdx.x] = d;
    __syncthreads();
    for (int o = kRed / 2; o > 0; o >>= 1) {
        if (int(threadIdx.x) < o) {
            s0[threadIdx.x] += s0[threadIdx.x + o];
            s1[threadIdx.x] += s1[threadIdx.x + o];
            s2[threadIdx.x] += s2[threadIdx.x + o];
            s3[threadIdx.x] += s3[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s0[0];
        out[1] = s1[0];
        out[2] = s2[0];
        out[3] = s3[0];
    }
}

// ---------------------------------------- complex fp64 tiles on matrix cores
// A 64 x 64 complex output tile per workgroup of 4 waves; wave (wr, wc) owns the
// 32 x 32 quarter at rows 32 wr, columns 32 wc as 2 x 2 tiles of
// v_mfma_f64_16x16x4f64 with real and imaginary accumulators apart.  Operands come
// from LDS stages of 16 k values, each four [16][64] fp64 arrays: the real and
// imaginary parts of A[i][k] (stored [k][i]) and of B[k][j] (stored [k][j]), so that
// the tile accumulates the plain complex product D += A B (a loader stores conjugates
// and weights as its product needs them).  f64 16x16x4 operand layout: lane l gives
// A[row l%16][k l/16] and B[k l/16][column l%16]; result item r of lane l is row
// l/16 + 4 r, column l%16.
typedef double double4_t __attribute__((ext_vector_type(4)));
constexpr int kCT = 64;        // output tile
constexpr int kCS = 16;        // k values per LDS stage
constexpr int kCStage = 4 * kCS * kCT;   // doubles per stage (Ar, Ai, Br, Bi)

struct CTileAcc {
    double4_t re[2][2], im[2][2];
};

__device__ inline void ctile_zero(CTileAcc& c) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int u = 0; u < 2; u++) c.re[t][u] = c.im[t][u] = {0.0, 0.0, 0.0, 0.0};
}

// the 16 k values of one stage into the wave's quarter
__device__ inline void ctile_stage(const double* st, int lane, int wr, int wc, CTileAcc& c) {
    const double* Ar = st;
    const double* Ai = st + kCS * kCT;
    const double* Br = st + 2 * kCS * kCT;
    const double* Bi = st + 3 * kCS * kCT;
#pragma unroll
    for (int q = 0; q < kCS / 4; q++) {
        const int kk = 4 * q + (lane >> 4);
        double ar[2], ai[2], br[2], bi[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int i = wr * 32 + 16 * t + (lane & 15);
            ar[t] = Ar[kk * kCT + i];
            ai[t] = Ai[kk * kCT + i];
            const int j = wc * 32 + 16 * t + (lane & 15);
            br[t] = Br[kk * kCT + j];
            bi[t] = Bi[kk * kCT + j];
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                c.re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[t], br[u], c.re[t][u], 0, 0, 0);
                c.re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai[t], bi[u], c.re[t][u], 0, 0, 0);
                c.im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[t], bi[u], c.im[t][u], 0, 0, 0);
                c.im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[t], br[u], c.im[t][u], 0, 0, 0);
            }
    }
}

// tile-local (row, column) of result item r of sub-tile (t, u) of the wave's quarter
__device__ inline int ctile_row(int lane, int wr, int t, int r) { return wr * 32 + 16 * t + (lane >> 4) + 4 * r; }
__device__ inline int ctile_col(int lane, int wc, int u) { return wc * 32 + 16 * u + (lane & 15); }

// (ti, tj), ti <= tj, of upper-triangular tile pair t (tj(tj+1)/2 <= t < (tj+1)(tj+2)/2)
__device__ inline void upper_pair(int64_t t, int& ti, int& tj) {
    int j = int((sqrt(8.0 * double(t) + 1.0) - 1.0) * 0.5);
    while (int64_t(j) * (j + 1) / 2 > t) j--;
    while (int64_t(j + 1) * (j + 2) / 2 <= t) j++;
    tj = j;
    ti = int(t - int64_t(j) * (j + 1) / 2);
}

// XCD-aware order: consecutive workgroups go to the 8 XCDs in turn, so logical tile t
// is given to workgroups of one XCD in runs (tiles that share operands share an L2)
__device__ inline int64_t xcd_tile(int64_t b, int64_t n) {
    const int64_t per = (n + 7) / 8;
    return (b % 8) * per + b / 8;
}

// ------------------------------------------------------------------ Gram
// S[k][k'] = sum_s w_s conj(O_sk) O_sk' for the upper-triangular tile pairs, mirrored
// into the lower triangle; samples are the k of the product, 16 per stage, staged in
// LDS double-buffered with the next stage's global loads in flight during the MFMAs.  SPLIT:
// workgroup (tile, z) takes the samples of chunk z and leaves its tile in out
// ([chunk][tile][64][64]) for gram_finish_kernel; else out is S.  (With the choice at run time the
// stores of one chunk cost 4-24 % at 256 to 32 samples.)
template <typename T, bool SPLIT>
__global__ __launch_bounds__(256) void gram_mfma_kernel(const cplx<T>* O, const double* w, int64_t total, int P,
                                                        int64_t pairs, int64_t chunk, cplx<double>* out) {
    extern __shared__ double lds[];   // [2][kCStage]
    const int64_t t = xcd_tile(blockIdx.x, pairs);
    if (t >= pairs) return;
    const int64_t first = SPLIT ? int64_t(blockIdx.y) * chunk : 0;
    const int64_t count = SPLIT && first + chunk < total ? first + chunk : total;
    int ti, tj;
    upper_pair(t, ti, tj);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int row0 = ti * kCT, col0 = tj * kCT;
    // loader: thread -> sample (tid / 16) of the stage, 4 consecutive parameters (tid % 16) * 4
    const int ls = threadIdx.x >> 4, lc = (threadIdx.x & 15) * 4;
    cplx<T> ra[4], ca[4];
    double ws = 0.0;
    auto fetch = [&](int64_t s0) {
        const int64_t s = s0 + ls;
        const bool ok = s < count;
        ws = ok ? w[s] : 0.0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            ra[e] = ok && row0 + lc + e < P ? O[s * P + row0 + lc + e] : cplx<T>{T(0), T(0)};
            ca[e] = ok && col0 + lc + e < P ? O[s * P + col0 + lc + e] : cplx<T>{T(0), T(0)};
        }
    };
    auto stash = [&](double* st) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int o = ls * kCT + lc + e;
            st[o] = ws * double(ra[e].re);                      // A = w conj(O) of the rows
            st[kCS * kCT + o] = -ws * double(ra[e].im);
            st[2 * kCS * kCT + o] = double(ca[e].re);           // B = O of the columns
            st[3 * kCS * kCT + o] = double(ca[e].im);
        }
    };
    CTileAcc acc;
    ctile_zero(acc);
    const int64_t stages = (count - first + kCS - 1) / kCS;
    fetch(first);
    stash(lds);
    __syncthreads();
    for (int64_t g = 0; g < stages; g++) {
        if (g + 1 < stages) fetch(first + (g + 1) * kCS);
        ctile_stage(lds + (g & 1) * kCStage, lane, wr, wc, acc);
        if (g + 1 < stages) stash(lds + ((g + 1) & 1) * kCStage);
        __syncthreads();
    }
#pragma unroll
    for (int tt = 0; tt < 2; tt++)
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int lr = ctile_row(lane, wr, tt, r), lc2 = ctile_col(lane, wc, u);
                const int gr = row0 + lr, gc = col0 + lc2;
                if constexpr (SPLIT) {
                    out[((int64_t(blockIdx.y) * pairs + t) * kCT + lr) * kCT + lc2] = {acc.re[tt][u][r],
                                                                                       acc.im[tt][u][r]};
                } else if (gr < P && gc < P) {
                    out[int64_t(gr) * P + gc] = {acc.re[tt][u][r], acc.im[tt][u][r]};
                    if (ti != tj) out[int64_t(gc) * P + gr] = {acc.re[tt][u][r], -acc.im[tt][u][r]};
                }
            }
}

// the chunks' tiles added in chunk order, and the mirrored triangle
__global__ __launch_bounds__(256) void gram_finish_kernel(const cplx<double>* part, int chunks, int P, int64_t pairs,
                                                          cplx<double>* S) {
    const int64_t t = blockIdx.x / (kCT * kCT / 256);
    const int e = int(blockIdx.x % (kCT * kCT / 256)) * 256 + threadIdx.x;
    int ti, tj;
    upper_pair(t, ti, tj);
    const int gr = ti * kCT + e / kCT, gc = tj * kCT + e % kCT;
    if (gr >= P || gc >= P) return;
    cplx<double> x = {0.0, 0.0};
    for (int z = 0; z < chunks; z++) x = cadd(x, part[(int64_t(z) * pairs + t) * kCT * kCT + e]);
    S[int64_t(gr) * P + gc] = x;
    if (ti != tj) S[int64_t(gc) * P + gr] = cconj(x);
}

__global__ __launch_bounds__(256) void dense_matvec_kernel(const cplx<double>* S, const cplx<double>* x,
                                                           int P, double shift, cplx<double>* y) {
    const int r = blockIdx.x;
    __shared__ double sr[256], si[256];
    double re = 0, im = 0;
    for (int k = threadIdx.x; k < P; k += 256) {
        const cplx<double> a = S[int64_t(r) * P + k], b = x[k];
        re += a.re * b.re - a.im * b.im;
        im += a.re * b.im + a.im * b.re;
    }
    sr[threadIdx.x] = re;
    si[threadIdx.x] = im;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (int(threadIdx.x) < o) {
            sr[threadIdx.x] += sr[threadIdx.x + o];
            si[threadIdx.x] += si[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) y[r] = {sr[0] + shift * x[r].re, si[0] + shift * x[r].im};
}

// -------------------------------------------------------------- Cholesky
// Solve of (S + shift) x = F by a blocked Cholesky of the diagonally scaled matrix, in a
// buffer of P + 1 rows: row P holds F^H scaled and takes part in the panel and trailing
// updates like any other row, so that it ends as (L^-1 F)^H and the forward
// substitution costs no launch of its own.  64-column blocks: potrf_inv_kernel forms the inverse of
// the diagonal block's factor in registers; the rows below become A L^-H on matrix
// cores (ctile_update_kernel<true, ..>); the trailing lower tiles take A -= L L^H
// (ctile_update_kernel<false, ..>), inside an outer panel of kOuter columns per block (K = 64,
// the panel's columns only), to the right of it once per outer panel (K = kOuter).
constexpr int kNB = 64;           // factor block
// The trailing matrix is read and written once per outer panel: with K = 64 its HBM traffic
// (16 B in and out per 8 * 64 flop) and not the matrix cores set the time of a large solve.
// A small one is bound by its chain of launches and skips the second level: P = 1,536 1,577 us
// without and 1,679 with it, 2,048 2,310 and 2,340, 2,560 3,203 and 3,117, 4,096 7,033 and 6,116.
constexpr int kOuter = 256;
constexpr int kOuterFrom = 2048;

// Scaled copy of the lower triangle: A[i][j] = (S + shift)[i][j] dinv_i dinv_j, j <= i,
// dinv_i = (S_ii + shift)^-1/2 (1 where that is not positive), and row P = (dinv F)^H.
// The scaled matrix has the same solution and a far smaller condition number when the
// parameters' scales differ.
__global__ __launch_bounds__(256) void chol_scale_kernel(const cplx<double>* S, const cplx<double>* F, int P,
                                                         double shift, double* dinv, cplx<double>* A) {
    const int cols = (P + 255) / 256;   // column blocks of a row
    const int i = int(blockIdx.x / cols), j0 = int(blockIdx.x % cols) * 256;
    const int j = j0 + threadIdx.x;
    if (j0 > i || j >= P) return;
    auto scale = [&](int r) {
        const double d = S[int64_t(r) * P + r].re + shift;
        return d > 0.0 ? 1.0 / sqrt(d) : 1.0;
    };
    const double fj = scale(j);
    if (i == P) {
        dinv[j] = fj;
        A[int64_t(P) * P + j] = {F[j].re * fj, -F[j].im * fj};
        return;
    }
    if (j > i) return;
    const cplx<double> a = S[int64_t(i) * P + j];
    const double f = fj * scale(i);
    A[int64_t(i) * P + j] = {(i == j ? a.re + shift : a.re) * f, a.im * f};
}

// The inverse Linv [kNB][kNB] of the factor of the diagonal block A[k:k+nb, k:k+nb] (lower);
// the factor itself is read by nothing and not stored.  One workgroup, bound by its chain of
// dependent steps, so the block stays in registers as matrix-core accumulators (both
// triangles; wave w holds rows 16 w .. 16 w + 15) and four pivots are taken per step: the four
// rows of a step are one accumulator item of their wave, they go through LDS (one barrier),
// every wave that still has rows factors the 4 x 4 block and substitutes the rows by itself,
// one column a lane (right of the block conj(L), left of it the rows of the inverse so far,
// in it the inverse of the 4 x 4 factor), and the rows below take the rank-4 update as one
// K = 4 matrix product.  The block's columns start from zero there and become columns of the
// inverse, in place, as in a Gauss-Jordan inversion.
// A 64 x 64 block: 128 us with the block in LDS, an element-wise update and three barriers a
// pivot; 48 us in registers with one pivot a barrier; 34 us here.
__global__ __launch_bounds__(256) void potrf_inv_kernel(const cplx<double>* A, int P, int k, int nb, int* info,
                                                        cplx<double>* Linv) {
    __shared__ double2 row[2][4][kNB];   // the step's rows
    __shared__ double2 ysh[4][4][kNB];   // each wave's substituted rows
    const int lane = threadIdx.x & 63, w = uniform_int(threadIdx.x >> 6);
    const int lc = lane & 15, lk = lane >> 4;
    double4_t re[4], im[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 16 * w + lk + 4 * i, c = 16 * u + lc, hi = r > c ? r : c, lo = r > c ? c : r;
            cplx<double> x = {0.0, 0.0};
            if (hi < nb) x = A[int64_t(k + hi) * P + k + lo];
            re[u][i] = x.re;
            im[u][i] = c > r ? -x.im : x.im;
        }
#pragma unroll 1   // (sixteen copies of the step would run from cold instruction lines)
    for (int t = 0; 4 * t < nb; t++) {
        const int j0 = 4 * t, owner = t >> 2, rr = t & 3, b = t & 1;
        if (w == owner) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i == rr) {
#pragma unroll
                    for (int u = 0; u < 4; u++) row[b][lk][16 * u + lc] = double2{re[u][i], im[u][i]};
                }
        }
        __syncthreads();   // double-buffered: the next write of buffer b follows the next barrier
        if (w < owner) continue;   // (wave-uniform) all rows finished
        double2 y[4], u_[4][4];    // u_[q][s], s >= q: entry (j0 + q, j0 + s)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            y[q] = row[b][q][lane];
#pragma unroll
            for (int s = q; s < 4; s++) u_[q][s] = row[b][q][j0 + s];
        }
        const int in = lane - j0;
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (in >= 0 && in < 4) y[q] = double2{in == q && j0 + q < nb ? 1.0 : 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            double d = u_[q][q].x;
            if (!(d > 0.0)) {
                if (j0 + q < nb && threadIdx.x == 64 * owner) atomicCAS(info, 0, k + j0 + q + 1);
                d = 1.0;
            }
            const double inv = rsqrt(d);
            y[q].x *= inv;
            y[q].y *= inv;
#pragma unroll
            for (int s = q + 1; s < 4; s++) {
                u_[q][s].x *= inv;   // conj(L_sq)
                u_[q][s].y *= inv;
            }
            // rows s > q lose L_sq = conj(u_qs) times row q
#pragma unroll
            for (int s = q + 1; s < 4; s++) {
                const double lr = u_[q][s].x, li = -u_[q][s].y;
#pragma unroll
                for (int v = s; v < 4; v++) {
                    u_[s][v].x = fma(-lr, u_[q][v].x, fma(li, u_[q][v].y, u_[s][v].x));
                    u_[s][v].y = fma(-lr, u_[q][v].y, fma(-li, u_[q][v].x, u_[s][v].y));
                }
                y[s].x = fma(-lr, y[q].x, fma(li, y[q].y, y[s].x));
                y[s].y = fma(-lr, y[q].y, fma(-li, y[q].x, y[s].y));
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) ysh[w][q][lane] = y[q];
        wave_sync();
        // operands of A_rc -= sum_q L_r,j0+q y_qc (L_r,j0+q = conj(y_qr), rows below the block)
        const double2 yr = ysh[w][lk][16 * w + lc];
        const bool below = 16 * w + lc > j0 + 3;
        const double ar = below ? -yr.x : 0.0, ai = below ? yr.y : 0.0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const double2 yc = ysh[w][lk][16 * u + lc];
            if (u == owner && (lc >> 2) == rr) {
                re[u] = {0.0, 0.0, 0.0, 0.0};
                im[u] = {0.0, 0.0, 0.0, 0.0};
            }
            re[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, yc.x, re[u], 0, 0, 0);
            im[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, yc.y, im[u], 0, 0, 0);
            re[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, yc.y, re[u], 0, 0, 0);
            im[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, yc.x, im[u], 0, 0, 0);
            if (w == owner) {   // the block's own rows
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (i == rr) {
                        re[u][i] = yc.x;
                        im[u][i] = yc.y;
                    }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 16 * w + lk + 4 * i, c = 16 * u + lc;
            Linv[r * kNB + c] = r < nb && c <= r ? cplx<double>{re[u][i], im[u][i]} : cplx<double>{0.0, 0.0};
        }
}

// Complex tiles of A (rows below, ld = P, `rows` rows), K values of k in stages of KS:
//   SOLVE:  A[i][k0+j] <- sum_m A[i][k0+m] conj(Linv[j][m]) for the rows from s0 (in place: a
//           tile spans the block's columns and its rows are read whole before they are written)
//   else:   A[i][j] -= sum_m A[i][k0+m] conj(A[j][k0+m]), j <= i, for the row tiles from s0 and
//           the column tiles from s0 below cend (every pair of the triangle when ctiles == 0)
// Four waves as WR x (4 / WR), T x T matrix-core tiles of 16 x 16 each.  Both operands are rows
// read along m; they are staged as complex [row][KS] with a row of KS + 1 (a 16-row fragment
// then takes 16 different 16-byte bank groups; the operands transposed into [m][row] put a
// wave's 64 writes into one bank).  KS = 64 holds all of a K = 64 product, whose loads are then
// one memory round trip; KS = 16 is double-buffered, the next stage's global loads in flight
// during the matrix instructions.  A 64 x 64 tile of K = 64 keeps one CU's matrix cores busy
// for 7 us, so where the tiles do not fill the chip smaller ones shorten the chain of launches.
template <int KS, int WR, int T>
struct UpdateTile {
    static constexpr int kRows = 16 * T * WR, kCols = 16 * T * (4 / WR);
    static constexpr int kRow = KS + 1;   // padded complex row
    static constexpr int kBuf = (kRows + kCols) * kRow;
    static constexpr size_t kLds = sizeof(double2) * (KS == kNB ? 1 : 2) * kBuf;
};
template <bool SOLVE, int KS, int WR, int T>
__global__ __launch_bounds__(256) void ctile_update_kernel(cplx<double>* A, int P, int rows, int k0, int K, int s0,
                                                           int ctiles, int cend, int64_t tiles,
                                                           const cplx<double>* Linv) {
    using U = UpdateTile<KS, WR, T>;
    static_assert(SOLVE ? U::kCols == kNB : U::kRows == U::kCols, "tile shape");
    constexpr int WC = 4 / WR;
    extern __shared__ double2 ust[];   // [buffers][kRows of A, kCols of the second operand][kRow]
    int bi, bj = 0;
    if constexpr (SOLVE) {
        bi = blockIdx.x;
    } else if (ctiles > 0) {
        bj = int(blockIdx.x) % ctiles;
        bi = int(blockIdx.x) / ctiles;
        if (bi < bj) return;
    } else {
        const int64_t t = xcd_tile(blockIdx.x, tiles);
        if (t >= tiles) return;
        upper_pair(t, bj, bi);   // bj <= bi
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave / WC, wc = wave % WC;
    const int r0 = s0 + bi * U::kRows, c0 = SOLVE ? 0 : s0 + bj * U::kCols;
    constexpr int kStep = 256 / KS;                              // rows per load round
    constexpr int kA = U::kRows / kStep, kB = U::kCols / kStep;  // loads per thread
    const int lm = threadIdx.x & (KS - 1), lr = threadIdx.x / KS;
    double2 fa[kA], fb[kB];
    auto load_row = [&](int r, int m) {
        return m < K && r < rows ? *reinterpret_cast<const double2*>(A + int64_t(r) * P + k0 + m) : double2{0.0, 0.0};
    };
    auto fetch = [&](int g) {
        const int m = g * KS + lm;
#pragma unroll
        for (int e = 0; e < kA; e++) fa[e] = load_row(r0 + lr + kStep * e, m);
#pragma unroll
        for (int e = 0; e < kB; e++) {
            const int r = c0 + lr + kStep * e;
            if constexpr (SOLVE)
                fb[e] = *reinterpret_cast<const double2*>(Linv + r * kNB + m);
            else
                fb[e] = load_row(r, m);
        }
    };
    auto stash = [&](int buf) {
        double2* st = ust + buf * U::kBuf;
#pragma unroll
        for (int e = 0; e < kA; e++) st[(lr + kStep * e) * U::kRow + lm] = fa[e];
#pragma unroll
        for (int e = 0; e < kB; e++) st[(U::kRows + lr + kStep * e) * U::kRow + lm] = fb[e];
    };
    // f64 16x16x4 result layout: item r of lane l is row l/16 + 4 r, column l%16
    auto row_of = [&](int t, int r) { return r0 + (wr * T + t) * 16 + (lane >> 4) + 4 * r; };
    auto col_of = [&](int u) { return c0 + (wc * T + u) * 16 + (lane & 15); };
    const int stages = (K + KS - 1) / KS;
    fetch(0);
    double4_t re[T][T], im[T][T];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int u = 0; u < T; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                cplx<double> x = {0.0, 0.0};
                const int gi = row_of(t, r), gj = col_of(u);
                if (!SOLVE && gi < rows && gj <= gi && gj < cend) x = A[int64_t(gi) * P + gj];
                re[t][u][r] = -x.re;
                im[t][u][r] = -x.im;
            }
    stash(0);
    __syncthreads();
    for (int g = 0; g < stages; g++) {
        if (g + 1 < stages) fetch(g + 1);
        const double2* As = ust + (KS == kNB ? 0 : g & 1) * U::kBuf;
        const double2* Bs = As + U::kRows * U::kRow;
#pragma unroll
        for (int q = 0; q < KS / 4; q++) {
            const int kk = 4 * q + (lane >> 4);
            double2 a[T], b[T];
#pragma unroll
            for (int t = 0; t < T; t++) {
                a[t] = As[((wr * T + t) * 16 + (lane & 15)) * U::kRow + kk];
                b[t] = Bs[((wc * T + t) * 16 + (lane & 15)) * U::kRow + kk];
            }
            // A times the conjugate of the second operand's rows
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int u = 0; u < T; u++) {
                    re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].x, b[u].x, re[t][u], 0, 0, 0);
                    im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].y, b[u].x, im[t][u], 0, 0, 0);
                    re[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].y, b[u].y, re[t][u], 0, 0, 0);
                    im[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[t].x, b[u].y, im[t][u], 0, 0, 0);
                }
        }
        if (g + 1 < stages) stash((g + 1) & 1);
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int u = 0; u < T; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gi = row_of(t, r), gj = col_of(u);
                if constexpr (SOLVE) {
                    if (gi < rows && gj < K) A[int64_t(gi) * P + k0 + gj] = {re[t][u][r], im[t][u][r]};
                } else {
                    if (gi < rows && gj <= gi && gj < cend)
                        A[int64_t(gi) * P + gj] = {-re[t][u][r], -im[t][u][r]};
                }
            }
}

// One block of the backward substitution L^H x = y, in conjugated form on row P of A (y^H on
// entry): x'_j = sum_m Linv[m][j] y'_m for the block's columns, then y'_i -= sum_m L[k+m][i] x'_m
// for the 64 columns i < k of this workgroup, and x = conj(x') dinv.  Every workgroup forms the
// block's x' itself (64 KB of Linv from L2), so a block is one launch; its rows of L are in
// flight meanwhile.  (A single-thread triangular solve of 32 columns took 28-51 us a block.)
__global__ __launch_bounds__(256) void chol_back_kernel(cplx<double>* A, int P, int k, int nb,
                                                        const cplx<double>* Linv, const double* dinv,
                                                        cplx<double>* x) {
    __shared__ cplx<double> sy[kNB], sx[kNB], part[4][kNB];
    const int c = threadIdx.x & 63, q = threadIdx.x >> 6;
    cplx<double>* row = A + int64_t(P) * P;
    const int i = blockIdx.x * 64 + c;
    cplx<double> l[16];
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int m = q * 16 + e;
        l[e] = i < k && m < nb ? A[int64_t(k + m) * P + i] : cplx<double>{0.0, 0.0};
    }
    if (q == 0) sy[c] = c < nb ? row[k + c] : cplx<double>{0.0, 0.0};
    __syncthreads();
    cplx<double> s = {0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int m = q * 16 + e;
        s = cadd(s, cmul(Linv[m * kNB + c], sy[m]));
    }
    part[q][c] = s;
    __syncthreads();
    if (q == 0) {
        s = cadd(cadd(part[0][c], part[1][c]), cadd(part[2][c], part[3][c]));
        sx[c] = s;
        if (blockIdx.x == 0 && c < nb) x[k + c] = {s.re * dinv[k + c], -s.im * dinv[k + c]};
    }
    __syncthreads();
    s = {0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 16; e++) s = cadd(s, cmul(l[e], sx[q * 16 + e]));
    part[q][c] = s;   // (the first use of part is over: sx was formed from it)
    __syncthreads();
    if (q == 0 && i < k) {
        s = cadd(cadd(part[0][c], part[1][c]), cadd(part[2][c], part[3][c]));
        row[i] = csub(row[i], s);
    }
}

}  // namespace

void launch_weighted_sums(const cplx<double>* e_loc, const double* w, int64_t count, double* out4,
                          hipStream_t stream) {
    weighted_sums_kernel<<<1, kRed, 0, stream>>>(e_loc, w, count, out4);
    ANN_LAUNCH_CHECK();
}

// Sample chunks of the Gram: one where the tile pairs fill the chip, else chunks of whole
// stages up to about two workgroups per CU, of at least 128 samples (below that the chunks'
// tiles cost more traffic than the samples).  P = 648, 4,096 samples: 66 tiles on 256 CUs
// 724 us, in 7 chunks 207 us with the reduction.
static int gram_chunks(int P, int64_t count, int64_t* chunk) {
    const int64_t nt = (P + kCT - 1) / kCT, pairs = nt * (nt + 1) / 2;
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>(2 * kCus / pairs, count / 128));
    *chunk = std::max<int64_t>(kCS, ((count + want - 1) / want + kCS - 1) / kCS * kCS);
    return int(std::max<int64_t>(1, (count + *chunk - 1) / *chunk));
}

size_t gram_work_elems(int P, int64_t count) {
    int64_t chunk = 0;
    const int z = gram_chunks(P, count, &chunk);
    const int64_t nt = (P + kCT - 1) / kCT;
    return z > 1 ? size_t(z) * (nt * (nt + 1) / 2) * kCT * kCT : 0;
}

template <typename T>
void launch_gram(const cplx<T>* O, const double* w, int64_t count, int P, cplx<double>* work, cplx<double>* S,
                 hipStream_t stream) {
    const int64_t nt = (P + kCT - 1) / kCT;
    const int64_t pairs = nt * (nt + 1) / 2;
    const size_t lds_bytes = sizeof(double) * 2 * kCStage;   // 64 KiB
    const int64_t grid = (pairs + 7) / 8 * 8;
    int64_t chunk = 0;
    const int chunks = gram_chunks(P, count, &chunk);
    auto run = [&](auto kernel, cplx<double>* out) {
        ANN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds_bytes)));
        kernel<<<dim3(unsigned(grid), unsigned(chunks)), 256, lds_bytes, stream>>>(O, w, count, P, pairs, chunk, out);
        ANN_LAUNCH_CHECK();
    };
    if (chunks > 1) {
        run(gram_mfma_kernel<T, true>, work);
        gram_finish_kernel<<<unsigned(pairs * (kCT * kCT / 256)), 256, 0, stream>>>(work, chunks, P, pairs, S);
        ANN_LAUNCH_CHECK();
    } else {
        run(gram_mfma_kernel<T, false>, S);
    }
}
template void launch_gram<float>(const cplx<float>*, const double*, int64_t, int, cplx<double>*, cplx<double>*,
                                 hipStream_t);
template void launch_gram<double>(const cplx<double>*, const double*, int64_t, int, cplx<double>*, cplx<double>*,
                                  hipStream_t);

void launch_dense_matvec(const cplx<double>* S, const cplx<double>* x, int P, double shift, cplx<double>* y,
                         hipStream_t stream) {
    dense_matvec_kernel<<<unsigned(P), 256, 0, stream>>>(S, x, P, shift, y);
    ANN_LAUNCH_CHECK();
}

size_t cholesky_matrix_elems(int P) { return size_t(P + 1) * P; }
size_t cholesky_work_elems(int P) { return size_t((P + kNB - 1) / kNB) * kNB * kNB; }

void cholesky_solve(const cplx<double>* S, const cplx<double>* F, int P, double shift, cplx<double>* A,
                    cplx<double>* work, double* dinv, int* d_info, cplx<double>* x, hipStream_t stream) {
    if (P <= 0) return;
    chol_scale_kernel<<<unsigned((P + 255) / 256) * unsigned(P + 1), 256, 0, stream>>>(S, F, P, shift, dinv, A);
    ANN_LAUNCH_CHECK();
    const int rows = P + 1;
    const int outer = P >= kOuterFrom ? kOuter : kNB;
    auto launch = [&](auto kernel, size_t lds, int64_t grid, auto... args) {
        ANN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        kernel<<<unsigned(grid), 256, lds, stream>>>(A, P, rows, args...);
        ANN_LAUNCH_CHECK();
    };
    auto tiles = [](int n, int t) { return int64_t((n + t - 1) / t); };
    // the columns [s0, cend) of the rows from s0 take the product of the columns [k, k + K)
    auto update = [&](int k, int K, int s0, int cend) {
        const bool tri = cend == P;   // the whole trailing triangle
        auto run = [&](auto kernel, size_t lds, int tile) {
            const int64_t nt = tiles(rows - s0, tile), ct = tiles(cend - s0, tile), pairs = nt * (nt + 1) / 2;
            launch(kernel, lds, tri ? (pairs + 7) / 8 * 8 : nt * ct, k, K, s0, tri ? 0 : int(ct), cend, pairs,
                   static_cast<const cplx<double>*>(nullptr));
        };
        const int64_t nt64 = tiles(rows - s0, 64), n64 = tri ? nt64 * (nt64 + 1) / 2 : nt64 * tiles(cend - s0, 64);
        if (K > kNB)
            run(ctile_update_kernel<false, 16, 2, 2>, UpdateTile<16, 2, 2>::kLds, 64);
        else if (n64 < kCus)
            run(ctile_update_kernel<false, kNB, 2, 1>, UpdateTile<kNB, 2, 1>::kLds, 32);
        else
            run(ctile_update_kernel<false, kNB, 2, 2>, UpdateTile<kNB, 2, 2>::kLds, 64);
    };
    for (int p = 0; p < P; p += outer) {
        const int pend = P - p < outer ? P : p + outer;
        for (int k = p; k < pend; k += kNB) {
            const int nb = pend - k < kNB ? pend - k : kNB;
            const int s0 = k + nb;
            cplx<double>* Linv = work + int64_t(k / kNB) * kNB * kNB;
            potrf_inv_kernel<<<1, 256, 0, stream>>>(A, P, k, nb, d_info, Linv);
            ANN_LAUNCH_CHECK();
            launch(ctile_update_kernel<true, kNB, 1, 1>, UpdateTile<kNB, 1, 1>::kLds, tiles(rows - s0, 16), k, nb, s0,
                   0, 0, int64_t(0), static_cast<const cplx<double>*>(Linv));
            if (s0 < pend) update(k, nb, s0, pend);
        }
        if (pend < P) update(p, pend - p, pend, P);
    }
    for (int k = (P - 1) / kNB * kNB; k >= 0; k -= kNB) {
        const int nb = P - k < kNB ? P - k : kNB;
        chol_back_kernel<<<unsigned(k > 0 ? tiles(k, 64) : 1), 256, 0, stream>>>(
            A, P, k, nb, work + int64_t(k / kNB) * kNB * kNB, dinv, x);
        ANN_LAUNCH_CHECK();
    }
}

}  // namespace ann
