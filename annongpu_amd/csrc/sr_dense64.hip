// sr_dense64.hip -- the fp64 products of a dense net on matrix cores: theta = S Wd + b,
// the spin-weighted sums behind <O>, F and the gradient, and the structured S.v of the
// stochastic reconfiguration (sr_mfma.hip is its fp32 counterpart).
//
// v_mfma_f64_16x16x4_f64 adds its four products one after the other, each with one
// rounding (k = 0..3), so a chain of these instructions gives the sums of a scalar loop
// over k bit for bit.  theta, S V and the spin sums within a chunk of samples keep the order of such
// a loop; the chunks are added in order, and <O>.v and O.v over threads, lanes and units in one fixed
// order of their own.  Every one of these orders is part of the results: a conjugate-gradient solve
// of 40 iterations amplifies a difference in the last bit of one product by five orders of
// magnitude.  Lanes: A lane l = row l%16, k = l/16; B lane l = k = l/16, column
// l%16; D item r of lane l = row l/16 + 4r, column l%16.
#include "ops.hpp"
#include "wave_net.hpp"

#include <algorithm>

namespace ann {

namespace {

using namespace wave;

typedef double double4_t __attribute__((ext_vector_type(4)));

__device__ inline double4_t mfma64(double a, double b, double4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ inline double spin_of(uint64_t word, int bit) { return ((word >> bit) & 1) ? 1.0 : -1.0; }

// the words of sample s, shifted so that bit 4t of word kb is the spin of site
// 64 kb + 4t + kk (the A operand of step t for the lanes with k = kk)
struct SpinRow {
    uint64_t w[kMaxWords];
    __device__ SpinRow(const uint64_t* confs, int64_t s, int words, int kk) {
#pragma unroll
        for (int i = 0; i < kMaxWords; i++) w[i] = i < words ? confs[s * words + i] >> kk : 0;
    }
    __device__ uint64_t word(int kb) const { return kb == 0 ? w[0] : kb == 1 ? w[1] : kb == 2 ? w[2] : w[3]; }
};

// 16 steps (64 sites) of a column of B [N][ld]; rows past N are zero
__device__ inline void load_b(double (&b)[16], const double* B, int64_t ld, int N, int kb, int kk) {
#pragma unroll
    for (int t = 0; t < 16; t++) {
        const int v = kb * 64 + 4 * t + kk;
        const double x = B[int64_t(min(v, N - 1)) * ld];
        b[t] = v < N ? x : 0.0;
    }
}

__device__ inline double4_t chain(const double (&b)[16], uint64_t word, int steps, double4_t acc) {
#pragma unroll
    for (int t = 0; t < 16; t++)
        if (t < steps) acc = mfma64(spin_of(word, 4 * t), b[t], acc);
    return acc;
}

// theta of 16 samples x 16 columns (re / im interleaved) per wavefront.  Bound by the
// matrix cores (64 cycles per 16x16x4 step); a block of 4 waves covers 64 columns, so that
// 1,000 samples of 72 units still give 252 blocks.  One thread per unit, every element of
// Wd read from L2 by every sample, took 34 us for 4,096 samples, 64 sites and 128 units;
// this takes 8.
__global__ __launch_bounds__(256) void theta64_kernel(DenseView<double> net, const uint64_t* confs, int words,
                                                      int64_t count, double* theta) {
    const int lane = threadIdx.x & 63, kk = lane >> 4;
    const int64_t s0 = int64_t(blockIdx.x) * 16;
    const int col = blockIdx.y * 64 + (threadIdx.x >> 6) * 16 + (lane & 15);
    const int64_t ld = 2 * net.Mpad;
    const double* B = reinterpret_cast<const double*>(net.Wd) + col;
    const SpinRow row(confs, min(s0 + (lane & 15), count - 1), words, kk);
    const double bias = reinterpret_cast<const double*>(net.b)[col];
    double4_t acc = {bias, bias, bias, bias};
    for (int kb = 0; kb * 64 < net.N; kb++) {
        double b[16];
        load_b(b, B, ld, net.N, kb, kk);
        acc = chain(b, row.word(kb), (net.N - kb * 64 + 3) / 4, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int64_t s = s0 + kk + 4 * r;
        if (s < count) theta[s * ld + col] = acc[r];
    }
}

// ------------------------------------------------------------------ S.v, first half

constexpr int kDot = 64;   // blocks of <O>.v

// beta = r^H z (this iteration) / r^H z (previous) as cg.hip's direction kernel forms it
__device__ inline double cg_beta(const CgDir& dir) {
    __shared__ double sh[4][4];
    double x[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const double* part = i < 2 ? dir.newpart : dir.oldpart;
        x[i] = int(threadIdx.x) < dir.parts ? part[int64_t(threadIdx.x) * 4 + (i & 1)] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const double s = wave_sum(x[i]);
        if ((threadIdx.x & 63) == 0) sh[i][threadIdx.x >> 6] = s;
    }
    __syncthreads();
    double t[4];
#pragma unroll
    for (int i = 0; i < 4; i++) t[i] = sh[i][0] + sh[i][1] + sh[i][2] + sh[i][3];
    const double rn = t[0] + t[1], ro = t[2] + t[3];
    return ro != 0.0 ? rn / ro : 0.0;
}

// One launch before the products: blocks [0, kDot) form the partials of <O>.v and, with
// dir.z set, write the direction v = z + beta p_old to dir.p_new (p_old once dir.done[0]
// is set); the other blocks write v re-indexed onto the visible units (V[conn(i,j)][j] +=
// v_W(i,j)), va and vb, forming v by themselves.
__global__ __launch_bounds__(256) void sr_prepare64_kernel(DenseView<double> net, const int* inv,
                                                           const cplx<double>* v, CgDir dir,
                                                           const cplx<double>* obar, double* dpart,
                                                           cplx<double>* va, cplx<double>* vb, cplx<double>* V) {
    const bool cg = dir.z != nullptr;
    const bool frozen = cg && dir.done[0];
    const double beta = cg && !frozen ? cg_beta(dir) : 0.0;
    auto value = [&](int64_t k) -> cplx<double> {
        if (!cg) return v[k];
        const cplx<double> p = dir.p_old[k];
        if (frozen) return p;
        const cplx<double> z = dir.z[k];
        return {z.re + beta * p.re, z.im + beta * p.im};
    };
    if (blockIdx.x < kDot) {
        __shared__ double sh[2][256];
        double acc[2] = {0, 0};
        for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < net.num_params; i += kDot * 256) {
            const cplx<double> p = value(i);
            if (cg) dir.p_new[i] = p;
            const cplx<double> o = obar[i];
            acc[0] += fma(o.re, p.re, -(o.im * p.im));
            acc[1] += fma(o.im, p.re, o.re * p.im);
        }
        for (int k = 0; k < 2; k++) sh[k][threadIdx.x] = acc[k];
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (int(threadIdx.x) < o)
                for (int k = 0; k < 2; k++) sh[k][threadIdx.x] += sh[k][threadIdx.x + o];
            __syncthreads();
        }
        if (threadIdx.x < 2) dpart[blockIdx.x * 2 + threadIdx.x] = sh[threadIdx.x][0];
        return;
    }
    const int64_t e = int64_t(blockIdx.x - kDot) * 256 + threadIdx.x;
    const int64_t nV = int64_t(net.N) * net.Mpad;
    const bool deep = net.layout == LAYOUT_DEEP1;
    if (e < nV) {
        const int vis = int(e / net.Mpad), j = int(e % net.Mpad);
        cplx<double> x = {0.0, 0.0};
        if (j < net.M) {
            if (!deep) {
                x = value(int64_t(vis) * net.M + j);
            } else {
                // inv[vis][j]: the unique i with conn(i, j) = vis, -1 if none, -2 if several
                const int i0 = inv[e];
                if (i0 >= 0) {
                    x = value(net.N + net.M + int64_t(i0) * net.M + j);
                } else if (i0 == -2) {
                    for (int i = 0; i < net.C; i++) {
                        if (int(net.conn[int64_t(i) * net.M + j]) == vis) {
                            const cplx<double> y = value(net.N + net.M + int64_t(i) * net.M + j);
                            x.re += y.re;
                            x.im += y.im;
                        }
                    }
                }
            }
        }
        V[e] = x;
    } else if (deep && e < nV + net.M) {
        vb[e - nV] = value(net.N + (e - nV));
    } else if (deep && e >= nV + net.Mpad && e < nV + net.Mpad + net.N) {
        va[e - nV - net.Mpad] = value(e - nV - net.Mpad);
    }
}

// u_s = w_s (O_s.v - <O>.v), O_s.v = sum_j g_sj (vb_j + sum_v s_v V[v][j]) + sum_i s_i va_i.
// Block of 8 waves: 16 samples.  Per group of 64 units each wave multiplies 16 of the 128
// columns of V on matrix cores and leaves them in LDS; then wave w, lane = unit, adds its
// two samples' terms over the groups.  The product was written to memory and read back
// (8 MB for 4,096 samples and 128 units), which with a product of one thread per unit and
// separate kernels for O.v, <O>.v and the centring took 53 us; this one takes 10.
constexpr int kOvWaves = 8, kOvStride = 144;   // doubles per row in LDS (rows 32 banks apart)
__global__ __launch_bounds__(64 * kOvWaves) void sr_ov64_kernel(DenseView<double> net, const uint64_t* confs,
                                                                int words, const cplx<double>* g,
                                                                const cplx<double>* V, const cplx<double>* vb,
                                                                const cplx<double>* va, const double* w,
                                                                const double* dpart, int64_t count,
                                                                cplx<double>* u_out) {
    __shared__ double sv[2][16][kOvStride];
    __shared__ double sd[2 * kDot], sc[2];
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6), kk = lane >> 4;
    const int64_t s0 = int64_t(blockIdx.x) * 16;
    const SpinRow row(confs, min(s0 + (lane & 15), count - 1), words, kk);
    if (threadIdx.x < 2 * kDot) sd[threadIdx.x] = dpart[threadIdx.x];
    const int col = wave * 16 + (lane & 15);
    const int64_t ld = 2 * net.Mpad;
    const double* B = reinterpret_cast<const double*>(V) + col;
    const int U = net.Mpad / 64;
    int64_t s[2];
#pragma unroll
    for (int i = 0; i < 2; i++) s[i] = min(s0 + 2 * wave + i, count - 1);
    double re[2] = {0, 0}, im[2] = {0, 0};
    double b[16];
    load_b(b, B, ld, net.N, 0, kk);
    for (int u = 0; u < U; u++) {
        const int j = lane + 64 * u;
        cplx<double> gv[2];
#pragma unroll
        for (int i = 0; i < 2; i++) gv[i] = g[s[i] * net.Mpad + j];
        const cplx<double> bj = vb && j < net.M ? vb[j] : cplx<double>{0.0, 0.0};
        double4_t acc = {0.0, 0.0, 0.0, 0.0};
        for (int kb = 0; kb * 64 < net.N; kb++) {
            double c[16];
#pragma unroll
            for (int t = 0; t < 16; t++) c[t] = b[t];
            // the next 64 sites, or the first ones of the next group, while these are multiplied
            if ((kb + 1) * 64 < net.N)
                load_b(b, B + 128 * u, ld, net.N, kb + 1, kk);
            else if (u + 1 < U)
                load_b(b, B + 128 * (u + 1), ld, net.N, 0, kk);
            acc = chain(c, row.word(kb), (net.N - kb * 64 + 3) / 4, acc);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) sv[u & 1][kk + 4 * r][col] = acc[r];
        __syncthreads();
        if (u == 0 && threadIdx.x < 2) {
            double a = 0.0;
#pragma unroll
            for (int k = 0; k < kDot; k++) a += sd[2 * k + threadIdx.x];
            sc[threadIdx.x] = a;
        }
        if (j < net.M) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                double xr = sv[u & 1][2 * wave + i][2 * lane], xi = sv[u & 1][2 * wave + i][2 * lane + 1];
                if (vb) {
                    xr += bj.re;
                    xi += bj.im;
                }
                re[i] += fma(gv[i].re, xr, -(gv[i].im * xi));
                im[i] += fma(gv[i].im, xr, gv[i].re * xi);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
        if (va) {
            const Conf c = load_conf(confs, s[i], words);
            for (int k = lane; k < net.N; k += 64) {
                const double sk = spin_bit(c, k) ? 1.0 : -1.0;
                re[i] += sk * va[k].re;
                im[i] += sk * va[k].im;
            }
        }
        const double tr = wave_sum(re[i]), ti = wave_sum(im[i]);
        if (lane == 0 && s0 + 2 * wave + i < count) {
            const double ws = w[s[i]];
            u_out[s[i]] = {ws * (tr - sc[0]), ws * (ti - sc[1])};
        }
    }
}

// ------------------------------------------------------------------ spin-weighted sums

// Chunks of samples of the spin GEMM: their number follows from the sizes alone, and the
// partials are added in chunk order, so the sums are the same however the rows and columns
// of a chunk are spread over blocks.  Columns of a partial: per 16 units their real, then
// their imaginary parts; a last group of which only the first unit is used is the
// coefficient itself (visible parameters).
struct SpinPlan64 {
    int vpad, ncols;
    int64_t chunk, chunks, n;
};

SpinPlan64 spin_plan64(int N, int Mpad, int64_t count) {
    SpinPlan64 p;
    p.vpad = (N + 1 + 15) / 16 * 16;
    p.ncols = 2 * Mpad + 32;
    const int ctiles = (2 * Mpad + 16) / 16, groups = (p.vpad / 16 + 7) / 8;
    int64_t chunks = std::max<int64_t>(1, 4096 / (int64_t(ctiles) * groups));
    chunks = std::min<int64_t>(chunks, (count + 63) / 64);
    p.chunk = ((count + chunks - 1) / chunks + 3) / 4 * 4;
    p.chunks = (count + p.chunk - 1) / p.chunk;
    p.n = int64_t(p.vpad) * p.ncols;
    return p;
}

__host__ __device__ inline int unit_col(int j) { return (j / 16) * 32 + j % 16; }

// partial[chunk][v][c] = sum_s spin_sv X_sc: rows v < N are spins (+-1, exact), row N is all
// ones (bias parameters); X = coef_s g_sj (conj_g = 0), coef_s conj g_sj (1) or coef_s
// |g_sj|^2 (2).  Block: 16 units x all rows of a chunk, 64 samples at a time: the products X
// are formed once, by all threads, into LDS (conflict-free: a row of 16 doubles is half the
// banks); then wave w multiplies the real (w even) or imaginary columns by row tiles
// first_tile + w / 2 + 2i.  A block waits for memory once per 64 samples, and g is read once.
// 64 sites, 128 units, 4,096 samples: one wave per 16 columns, which read g and coef for
// itself 16 samples at a time, took 21 us; this kernel takes 16 (2.5 us of matrix-core time,
// 12 MB of partials).  Adding the chunks inside a block instead (16 rows x 8 units, a chunk
// per wave) leaves two thirds of the chip idle at these sizes: 35 us.
constexpr int kSub = 64;
template <int J>
__global__ __launch_bounds__(256) void spin_gemm64_kernel(DenseView<double> net, const uint64_t* confs, int words,
                                                          const cplx<double>* g, int conj_g,
                                                          const cplx<double>* coef, int64_t count, SpinPlan64 p,
                                                          int first_tile, double* partial) {
    __shared__ double sx[2][kSub][16];
    __shared__ uint64_t sw[kMaxWords][kSub];
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6), kk = lane >> 4;
    const int unit = threadIdx.x & 15, row = threadIdx.x >> 4;   // samples row + 16 i of the 64
    const int j = blockIdx.x * 16 + unit;
    const bool is_g = j < net.Mpad;
    const int64_t s0 = int64_t(blockIdx.y) * p.chunk, s1 = min(s0 + p.chunk, count);
    const int part = wave & 1, tile0 = first_tile + (wave >> 1);
    const bool last = tile0 + 2 * (J - 1) < p.vpad / 16;
    double4_t acc[J];
#pragma unroll
    for (int i = 0; i < J; i++) acc[i] = {0.0, 0.0, 0.0, 0.0};
    cplx<double> cf[4], gv[4];
    uint64_t cw = 0;
    auto load = [&](int64_t sq) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t s = min(sq + row + 16 * i, s1 - 1);
            cf[i] = coef[s];
            gv[i] = g[s * net.Mpad + min(j, net.Mpad - 1)];
        }
        cw = wave < words ? confs[min(sq + lane, s1 - 1) * words + wave] : 0;
    };
    load(s0);
    for (int64_t sq = s0; sq < s1; sq += kSub) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const cplx<double> c = cf[i];
            const double gr = gv[i].re, gi = conj_g ? -gv[i].im : gv[i].im;
            double xr = fma(c.re, gr, -(c.im * gi)), xi = fma(c.im, gr, c.re * gi);
            if (conj_g == 2) {   // diagonal of S
                xr = c.re * fma(gr, gr, gi * gi);
                xi = 0.0;
            }
            if (!is_g) {
                xr = unit == 0 ? c.re : 0.0;
                xi = unit == 0 ? c.im : 0.0;
            }
            const bool in = sq + row + 16 * i < s1;
            sx[0][row + 16 * i][unit] = in ? xr : 0.0;
            sx[1][row + 16 * i][unit] = in ? xi : 0.0;
        }
        sw[wave][lane] = cw;
        __syncthreads();
        if (sq + kSub < s1) load(sq + kSub);
        // (the products past the last sample are zero)
        const int rows = int(min(int64_t(kSub), s1 - sq));
        for (int r = 0; r < rows; r += 16) {
            double b[4];
            uint64_t word[J][4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                b[t] = sx[part][r + 4 * t + kk][lane & 15];
#pragma unroll
                for (int i = 0; i < J; i++) word[i][t] = sw[min((tile0 + 2 * i) >> 2, kMaxWords - 1)][r + 4 * t + kk];
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
#pragma unroll
                for (int i = 0; i < J; i++) {
                    const int v = (tile0 + 2 * i) * 16 + (lane & 15);
                    const double a = v < net.N ? spin_of(word[i][t], v & 63) : v == net.N ? 1.0 : 0.0;
                    if (i < J - 1 || last) acc[i] = mfma64(a, b[t], acc[i]);
                }
            }
        }
    }
    const int col = blockIdx.x * 32 + part * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < J; i++) {
        if (i < J - 1 || last) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int v = (tile0 + 2 * i) * 16 + kk + 4 * r;
                partial[(int64_t(blockIdx.y) * p.vpad + v) * p.ncols + col] = acc[i][r];
            }
        }
    }
}

// Y[v][c], v <= N: the partials added in chunk order, 64 loads in flight (with one at a
// time, 17 us for 64 chunks of 65 x 288; now 5).  A kernel of its own, one wave per 64
// columns: a connection's row differs from unit to unit, so that adding the partials in
// parameter order reads a memory line per number (14 us)
__global__ __launch_bounds__(64) void spin_chunks64_kernel(const double* partial, int chunks, int64_t stride,
                                                           int64_t first, int64_t n, double* Y) {
    constexpr int kFly = 64;
    const int64_t e = int64_t(blockIdx.x) * 64 + threadIdx.x;
    if (e >= n) return;
    const double* q = partial + first + e;
    double acc = 0.0;
    for (int c0 = 0; c0 < chunks; c0 += kFly, q += kFly * stride) {
        const int left = chunks - c0;
        double y[kFly];
#pragma unroll
        for (int i = 0; i < kFly; i++) y[i] = i < left ? q[i * stride] : 0.0;
#pragma unroll
        for (int i = 0; i < kFly; i++)
            if (i < left) acc += y[i];
    }
    Y[first + e] = acc;
}

// y[k] = Y of parameter k's row and column (+ shift v_k), a wave for the real and one for
// the imaginary parts of 64 parameters; ypart[k / 64] = Re(v^H y) of the 64
__global__ __launch_bounds__(128) void spin_pack64_kernel(DenseView<double> net, SpinPlan64 p, const double* Y,
                                                          double shift, const cplx<double>* v, double* y,
                                                          double* ypart) {
    __shared__ double sh[64];
    const int lane = threadIdx.x & 63, part = uniform_int(threadIdx.x >> 6);
    const int k = blockIdx.x * 64 + lane;
    double r = 0.0, x = 0.0;
    if (k < net.num_params) {
        int row, col;
        if (net.layout == LAYOUT_RBM) {
            row = k / net.M;
            col = unit_col(k % net.M);
        } else if (k < net.N) {
            row = k;
            col = 2 * net.Mpad;
        } else if (k < net.N + net.M) {
            row = net.N;
            col = unit_col(k - net.N);
        } else {
            const int q = k - net.N - net.M;
            row = int(net.conn[q]);
            col = unit_col(q % net.M);
        }
        if (v) x = reinterpret_cast<const double*>(v)[2 * k + part];
        r = Y[int64_t(row) * p.ncols + col + 16 * part];
        if (v) r = fma(shift, x, r);
        y[2 * k + part] = r;
    }
    if (ypart) {
        if (part == 1) sh[lane] = x * r;
        __syncthreads();
        if (part == 0) {
            const double d = wave_sum(fma(x, r, sh[lane]));
            if (lane == 0) ypart[blockIdx.x] = d;
            // the last block fills up its group of four
            if (lane == 0 && blockIdx.x == gridDim.x - 1)
                for (unsigned i = blockIdx.x + 1; i & 3; i++) ypart[i] = 0.0;
        }
    }
}

__global__ __launch_bounds__(64) void spin_bias64_kernel(DenseView<double> net, const double* Yrow,
                                                         cplx<double>* Yb) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    if (j < net.Mpad) Yb[j] = {Yrow[unit_col(j)], Yrow[unit_col(j) + 16]};
}

template <int J>
void spin_gemm64_rows(int jobs, const DenseView<double>& net, const uint64_t* confs, int words,
                      const cplx<double>* g, int conj_g, const cplx<double>* coef, int64_t count,
                      const SpinPlan64& p, int first_tile, double* partial, hipStream_t stream) {
    if constexpr (J > 1) {
        if (jobs < J)
            return spin_gemm64_rows<J - 1>(jobs, net, confs, words, g, conj_g, coef, count, p, first_tile, partial,
                                           stream);
    }
    const dim3 grid{unsigned(p.ncols / 32), unsigned(p.chunks)};
    spin_gemm64_kernel<J><<<grid, 256, 0, stream>>>(net, confs, words, g, conj_g, coef, count, p, first_tile,
                                                    partial);
    ANN_LAUNCH_CHECK();
}

// Y of rows [first_row, N] from the row tiles that hold them, behind the partials in work
double* spin_gemm64(const DenseView<double>& net, const uint64_t* confs, int words, const cplx<double>* g, int conj_g,
                    const cplx<double>* coef, int64_t count, const SpinPlan64& p, int first_row, double* work,
                    hipStream_t stream) {
    // (N + 1 <= 257 rows are at most 17 tiles, two of which are worked on at a time)
    const int first_tile = first_row / 16;
    spin_gemm64_rows<9>((p.vpad / 16 - first_tile + 1) / 2, net, confs, words, g, conj_g, coef, count, p, first_tile,
                        work, stream);
    double* Y = work + p.n * p.chunks;
    const int64_t first = int64_t(first_row) * p.ncols, n = int64_t(net.N + 1) * p.ncols - first;
    spin_chunks64_kernel<<<unsigned((n + 63) / 64), 64, 0, stream>>>(work, int(p.chunks), p.n, first, n, Y);
    ANN_LAUNCH_CHECK();
    return Y;
}

}  // namespace

void launch_theta64(const DenseView<double>& net, const uint64_t* confs, int words, int64_t count,
                    cplx<double>* theta, hipStream_t stream) {
    if (count <= 0) return;
    const dim3 grid{unsigned((count + 15) / 16), unsigned(net.Mpad / 32)};
    theta64_kernel<<<grid, 256, 0, stream>>>(net, confs, words, count, reinterpret_cast<double*>(theta));
    ANN_LAUNCH_CHECK();
}

int sr_dot_parts64() { return kDot; }

void launch_sr_prepare64(const DenseView<double>& net, const int* inv, const cplx<double>* v, const CgDir& dir,
                         const cplx<double>* obar, double* dpart, cplx<double>* va, cplx<double>* vb,
                         cplx<double>* V, hipStream_t stream) {
    if (dir.parts > 256) throw std::invalid_argument("too many partial sums");
    const int64_t n = int64_t(net.N) * net.Mpad + net.Mpad + net.N;
    sr_prepare64_kernel<<<unsigned(kDot + (n + 255) / 256), 256, 0, stream>>>(net, inv, v, dir, obar, dpart, va, vb,
                                                                              V);
    ANN_LAUNCH_CHECK();
}

void launch_sr_ov64(const DenseView<double>& net, const uint64_t* confs, int words, const cplx<double>* g,
                    const cplx<double>* V, const cplx<double>* vb, const cplx<double>* va, const double* w,
                    const double* dpart, int64_t count, cplx<double>* u, hipStream_t stream) {
    if (count <= 0) return;
    sr_ov64_kernel<<<unsigned((count + 15) / 16), 64 * kOvWaves, 0, stream>>>(net, confs, words, g, V, vb, va, w,
                                                                              dpart, count, u);
    ANN_LAUNCH_CHECK();
}

size_t spin_sums64_work(int N, int Mpad, int64_t count) {
    if (count <= 0) return 0;
    const SpinPlan64 p = spin_plan64(N, Mpad, count);
    return size_t(p.n) * (p.chunks + 1);
}

int spin_sums64_parts(int64_t num_params) { return int((num_params + 63) / 64); }

void launch_spin_sums64(const DenseView<double>& net, const uint64_t* confs, int words, const cplx<double>* g,
                        int conj_g, const cplx<double>* coef, int64_t count, double* work, double shift,
                        const cplx<double>* v, cplx<double>* y, double* ypart, hipStream_t stream) {
    if (count <= 0) return;
    const SpinPlan64 p = spin_plan64(net.N, net.Mpad, count);
    const double* Y = spin_gemm64(net, confs, words, g, conj_g, coef, count, p, 0, work, stream);
    spin_pack64_kernel<<<unsigned(spin_sums64_parts(net.num_params)), 128, 0, stream>>>(
        net, p, Y, shift, v, reinterpret_cast<double*>(y), ypart);
    ANN_LAUNCH_CHECK();
}

void launch_spin_bias64(const DenseView<double>& net, const uint64_t* confs, int words, const cplx<double>* g,
                        int mode, const cplx<double>* coef, int64_t count, double* work, cplx<double>* Yb,
                        hipStream_t stream) {
    if (count <= 0) return;
    const SpinPlan64 p = spin_plan64(net.N, net.Mpad, count);
    const double* Y = spin_gemm64(net, confs, words, g, mode, coef, count, p, net.N, work, stream);
    spin_bias64_kernel<<<unsigned(net.Mpad / 64), 64, 0, stream>>>(net, Y + int64_t(net.N) * p.ncols, Yb);
    ANN_LAUNCH_CHECK();
}

}  // namespace ann
