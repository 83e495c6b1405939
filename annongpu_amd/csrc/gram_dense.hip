// gram_dense.hip -- the dense S = <O^* O> - <O^*><O> of a one-layer net from its structure.
//
// With O_k(s) = s_i g_j(s), k = (site i, unit j), extended by a constant site (s = 1: the
// biases, O = g_j) and a constant unit (g = 1: the visible parameters, O = s_i),
//   sum_s w O_k^* O_k' = sum_s (s_i s_i') (w conj(g_j) g_j'),
// which depends on the unordered pairs {i, i'} (real, +-1) and {j, j'} (complex, Hermitian).
// So S needs one real x complex product per pair of pairs, P^2 flop per sample, where
// a complex Gram of the materialised O needs 4 P^2, and neither O nor its traffic.  The sums are
// of uncentred O: the caller takes this form only while no parameter's mean dominates its spread.
//   pairs_gemm   T[site pair][unit pair] on v_mfma_f64_16x16x4_f64, signs from the
//                transposed spin bits, the unit products formed into LDS once per 256 site pairs
//   assemble     S[k][k'] = T - conj(m_k) m_k', m = <O>, read from the constant's row of T
// Site pairs: index 0 is i = i' (s_i^2 = 1 for every i), 1 + i'(i' - 1) / 2 + i is i < i'.
// Unit pairs: j'(j' + 1) / 2 + j, j <= j'.  The constants are site N and unit M.
// 64-site ring, M = 256 (P = 16,704), 8,192 samples: 163.4 ms as a Gram of the materialised O
// (56 TFLOP/s of 4 P^2 flop per sample), 45.8 ms here (product 40.1 ms, 58 TFLOP/s; assembly 5.7 ms).
#include "kernels.hpp"
#include "wave_net.hpp"

#include <algorithm>

namespace ann {

namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr int kGRows = 256;    // site pairs per workgroup: 64 per wave
constexpr int kGPairs = 32;    // unit pairs per workgroup (64 real columns)
constexpr int kGStage = 16;    // samples per LDS stage
constexpr int kGRow = 80;      // padded row of a stage: two rows of 16 columns share no bank

// pair t of an upper triangle, t = b (b + 1) / 2 + a, a <= b
__device__ inline void tri_pair(int64_t t, int& a, int& b) {
    int j = int((sqrt(8.0 * double(t) + 1.0) - 1.0) * 0.5);
    while (int64_t(j) * (j + 1) / 2 > t) j--;
    while (int64_t(j + 1) * (j + 2) / 2 <= t) j++;
    b = j;
    a = int(t - int64_t(j) * (j + 1) / 2);
}
__device__ inline int64_t site_row(int i, int ip) {
    const int64_t lo = i < ip ? i : ip, hi = i < ip ? ip : i;
    return lo == hi ? 0 : 1 + hi * (hi - 1) / 2 + lo;
}

// T[row][2 pair + re/im] (+= nothing: chunk z writes its own slice) for the samples of chunk z.
// Wave w: rows 64 w .. of the workgroup's 256 as 4 tiles, times 4 column tiles.  A fragment:
// lane l holds row l%16 of sample 4 q + l/16, +-1 from one bit of the row's 64-sample word; B
// fragment: column l%16 of the same sample, from LDS.  The next stage's g are in flight during
// the matrix instructions.
template <typename T>
__global__ __launch_bounds__(256) void pairs_gemm_kernel(const uint64_t* bits, int vpad, const cplx<T>* g, int Mpad,
                                                         int N, int M, const double* w, int64_t count, int64_t chunk,
                                                         int64_t rows, int64_t pairs, int row_blocks, int64_t ncol,
                                                         int64_t slice, double* out) {
    __shared__ double hs[2][kGStage][kGRow];
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6);
    const int lc = lane & 15, lk = lane >> 4;
    // row blocks of one column block run together (they share its g columns in L2)
    const int64_t cb = blockIdx.x / row_blocks;
    const int rb = int(blockIdx.x % row_blocks);
    const int64_t s0 = int64_t(blockIdx.y) * chunk, s1 = s0 + chunk < count ? s0 + chunk : count;
    // loader: sample tid / 16 of a stage, unit pairs tid % 16 and + 16
    const int ls = threadIdx.x >> 4;
    int ja[2], jb[2];
    bool ok[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int64_t p = cb * kGPairs + (threadIdx.x & 15) + 16 * e;
        ok[e] = p < pairs;
        ja[e] = jb[e] = 0;
        if (ok[e]) tri_pair(p, ja[e], jb[e]);
    }
    double fw = 0.0;
    cplx<T> fa[2], fb[2];
    auto fetch = [&](int64_t s) {
        const bool in = s + ls < s1;
        const int64_t sc = in ? s + ls : s1 - 1;
        fw = in ? w[sc] : 0.0;
        const cplx<T>* gs = g + sc * Mpad;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            fa[e] = gs[ja[e] < M ? ja[e] : 0];
            fb[e] = gs[jb[e] < M ? jb[e] : 0];
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const double ar = ja[e] < M ? double(fa[e].re) : 1.0, ai = ja[e] < M ? double(fa[e].im) : 0.0;
            const double br = jb[e] < M ? double(fb[e].re) : 1.0, bi = jb[e] < M ? double(fb[e].im) : 0.0;
            const double wr = ok[e] ? fw * ar : 0.0, wi = ok[e] ? fw * ai : 0.0;
            *reinterpret_cast<double2*>(&hs[buf][ls][2 * ((threadIdx.x & 15) + 16 * e)]) =
                double2{wr * br + wi * bi, wr * bi - wi * br};
        }
    };
    // the two sites of this lane's row in each of the wave's row tiles; both the constant for
    // the diagonal pair and for rows beyond the last (never stored)
    int va[4], vb[4];
    const int64_t row0 = int64_t(rb) * kGRows + 64 * wave;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int64_t r = row0 + 16 * t + lc;
        va[t] = vb[t] = N;
        if (r >= 1 && r < rows) {
            tri_pair(r - 1, va[t], vb[t]);
            vb[t]++;
        }
    }
    const bool active = row0 < rows;   // (wave-uniform; every wave joins the barriers)
    double4_t acc[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[t][u] = {0.0, 0.0, 0.0, 0.0};
    if (s0 < s1) {
        fetch(s0);
        stash(0);
    }
    __syncthreads();
    int buf = 0;
    uint64_t x[4] = {0, 0, 0, 0};
    for (int64_t s = s0; s < s1; s += kGStage, buf ^= 1) {   // s0 is a multiple of 64
        const int off = int(s & 63);
        if (off == 0) {
            const uint64_t* bw = bits + (s >> 6) * vpad;
#pragma unroll
            for (int t = 0; t < 4; t++) x[t] = (bw[va[t]] ^ bw[vb[t]]) >> lk;
        }
        const bool more = s + kGStage < s1;
        if (more) fetch(s + kGStage);
        if (active) {
#pragma unroll
            for (int q = 0; q < kGStage / 4; q++) {
                double a[4], b[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const uint32_t bit = uint32_t(x[t] >> (4 * q)) & 1u;   // the two spins differ
                    a[t] = __hiloint2double(int(0x3FF00000u | (bit << 31)), 0);
                }
#pragma unroll
                for (int u = 0; u < 4; u++) b[u] = hs[buf][4 * q + lk][16 * u + lc];
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[u], acc[t][u], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; t++) x[t] >>= kGStage;
        if (more) stash(buf ^ 1);
        __syncthreads();
    }
    if (!active) return;
    double* o = out + int64_t(blockIdx.y) * slice;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t row = row0 + 16 * t + lk + 4 * r;   // f64 result layout: row l/16 + 4 r, column l%16
            if (row >= rows) continue;
#pragma unroll
            for (int u = 0; u < 4; u++) o[row * ncol + cb * (2 * kGPairs) + 16 * u + lc] = acc[t][u][r];
        }
}

__global__ __launch_bounds__(256) void sum_slices_kernel(double* out, int slices, int64_t slice) {
    const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= slice) return;
    double s = 0.0;
    for (int z = 0; z < slices; z++) s += out[z * slice + e];
    out[e] = s;
}

// (site, unit) of parameter k, the constants being site N and unit M
struct ParamPair {
    int layout, N, M;
    const uint32_t* conn;
    __device__ void get(int k, int& i, int& j) const {
        if (layout == LAYOUT_RBM) {
            i = k / M;
            j = k % M;
        } else if (k < N) {
            i = k;
            j = M;
        } else if (k < N + M) {
            i = N;
            j = k - N;
        } else {
            const int q = k - N - M;
            i = int(conn[q]);
            j = q % M;
        }
    }
};

// <O_k> = conj(T[{i, N}][{j, M}])
__global__ __launch_bounds__(256) void pairs_mean_kernel(ParamPair pm, const double* T, int64_t ncol, int P,
                                                         cplx<double>* m) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= P) return;
    int i, j;
    pm.get(k, i, j);
    const double* t = T + site_row(i, pm.N) * ncol + 2 * (int64_t(pm.M) * (pm.M + 1) / 2 + j);
    m[k] = {t[0], -t[1]};
}

// one row of S per blockIdx.x (rows ordered as the parameters: the rows of a connection share
// their unit pairs' columns of T in the caches), 16 bytes a thread
__global__ __launch_bounds__(256) void pairs_assemble_kernel(ParamPair pm, const double* T, int64_t ncol,
                                                             const cplx<double>* m, int P, cplx<double>* S) {
    const int k = blockIdx.x;
    int i, j;
    pm.get(k, i, j);
    const cplx<double> mk = m[k];
    for (int kp = threadIdx.x; kp < P; kp += 256) {
        int ip, jp;
        pm.get(kp, ip, jp);
        const int64_t a = j < jp ? j : jp, b = j < jp ? jp : j;
        const double2 t = *reinterpret_cast<const double2*>(T + site_row(i, ip) * ncol + 2 * (b * (b + 1) / 2 + a));
        const cplx<double> mp = m[kp];
        // minus conj(m_k) m_k'
        S[int64_t(k) * P + kp] = {t.x - (mk.re * mp.re + mk.im * mp.im),
                                  (j <= jp ? t.y : -t.y) - (mk.re * mp.im - mk.im * mp.re)};
    }
}

struct PairsPlan {
    int64_t rows, pairs, ncol, slice, chunk;
    int row_blocks, chunks;
    int64_t col_blocks;
};

PairsPlan pairs_plan(int N, int M, int64_t count) {
    PairsPlan p;
    p.rows = 1 + int64_t(N + 1) * N / 2;
    p.pairs = int64_t(M + 1) * (M + 2) / 2;
    p.col_blocks = (p.pairs + kGPairs - 1) / kGPairs;
    p.ncol = p.col_blocks * 2 * kGPairs;
    p.row_blocks = int((p.rows + kGRows - 1) / kGRows);
    // samples split over chunks of whole 64-sample words where the tiles alone leave the
    // chip idle (about two workgroups per CU); the chunks' slices are summed in order
    const int64_t tiles = p.col_blocks * p.row_blocks;
    int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(512 / tiles, (count + 63) / 64));
    p.chunk = std::max<int64_t>(64, ((count + chunks - 1) / chunks + 63) / 64 * 64);
    p.chunks = int(std::max<int64_t>(1, (count + p.chunk - 1) / p.chunk));
    p.slice = p.rows * p.ncol;
    return p;
}

}  // namespace

size_t dense_gram_work_elems(int N, int M, int64_t count) {
    const PairsPlan p = pairs_plan(N, M, count);
    return size_t(p.slice) * p.chunks;
}

template <typename T>
void launch_dense_gram(int layout, int N, int M, int Mpad, const uint32_t* conn, const uint64_t* bits, int vpad,
                       const cplx<T>* g, const double* w, int64_t count, int P, double* work, cplx<double>* mean,
                       cplx<double>* S, hipStream_t stream) {
    if (count <= 0 || P <= 0) return;
    if (N + 1 > vpad) throw std::invalid_argument("dense Gram: the spin bits need a row of ones");
    const PairsPlan p = pairs_plan(N, M, count);
    const dim3 grid(unsigned(p.col_blocks * p.row_blocks), unsigned(p.chunks));
    pairs_gemm_kernel<T><<<grid, 256, 0, stream>>>(bits, vpad, g, Mpad, N, M, w, count, p.chunk, p.rows, p.pairs,
                                                   p.row_blocks, p.ncol, p.slice, work);
    ANN_LAUNCH_CHECK();
    if (p.chunks > 1) {
        sum_slices_kernel<<<unsigned((p.slice + 255) / 256), 256, 0, stream>>>(work, p.chunks, p.slice);
        ANN_LAUNCH_CHECK();
    }
    const ParamPair pm{layout, N, M, conn};
    pairs_mean_kernel<<<unsigned((P + 255) / 256), 256, 0, stream>>>(pm, work, p.ncol, P, mean);
    ANN_LAUNCH_CHECK();
    pairs_assemble_kernel<<<unsigned(P), 256, 0, stream>>>(pm, work, p.ncol, mean, P, S);
    ANN_LAUNCH_CHECK();
}
template void launch_dense_gram<float>(int, int, int, int, const uint32_t*, const uint64_t*, int, const cplx<float>*,
                                       const double*, int64_t, int, double*, cplx<double>*, cplx<double>*, hipStream_t);
template void launch_dense_gram<double>(int, int, int, int, const uint32_t*, const uint64_t*, int,
                                        const cplx<double>*, const double*, int64_t, int, double*, cplx<double>*,
                                        cplx<double>*, hipStream_t);

}  // namespace ann
