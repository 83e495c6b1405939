// cnn_pair.hip -- PsiCNN of two layers and one symmetry class with a first kernel of at most
// nine sites: log psi, Metropolis chains, local energies and O_k.
//
// The first layer's activation at a site depends on the spins of that site's kernel alone, so a
// table of 2^v0 spin patterns per channel, built in LDS once per workgroup, replaces the layer:
// a configuration is held as one pattern per site (a flip toggles one bit in the patterns of the
// sites that read it), and nothing of the first layer is stored or recomputed per chain.  What
// is left of a proposal are the second layer's pre-activations at the sites the flip reaches: a
// lane takes a site with all channels (blocks of CB) in registers, so that an activation read
// from LDS serves CB products and the weights, uniform over the wave, come through scalar loads.
// A flip of a 3 x 3 net reaches 25 sites: a half wave takes a chain, 2 chains a wave.
// (The kernels of cnn.hip, which stay for other nets, hold 40 KB of activations per chain, one
// chain per SIMD, and read a weight and an activation from LDS for every product.)
// 12 x 12, 2 x 8 channels, fp32, against them: a sweep of 16,384 chains 64.0 -> 5.9 ms, and of 4,096
// samples the transverse field's local energies 16.0 -> 1.85 ms, O_k 6.9 -> 0.37 ms, log psi
// 0.72 -> 0.09 ms.  The sweep is bound by the vector units: 3,893 of their instructions a pair of
// proposals, 3,456 of them the products, one in 3.1 cycles on every SIMD (a loop of plain multiply-adds
// reaches one in 4.1 to 4.3); LDS bank conflicts take 11 % of the cycles.
//
// Every sum that a Metropolis decision depends on is taken in the order of cnn.hip's kernels:
// input channels, then kernel sites, then output channels, then sites in increasing order over
// the lanes of one reduction tree.
#include "cnn.hpp"
#include "wave_net.hpp"

#include <algorithm>
#include <type_traits>

namespace ann {

namespace {

using namespace wave;

constexpr int kPThreads = 512;
constexpr int kPWaves = kPThreads / kWave;
constexpr int kPList = 4096;     // most off-diagonal terms of an operator (listed per wave)
constexpr int kPLds = 150 * 1024;

// pre-activation table of the first layer: lut[ci << v0 | pattern], bit k of a pattern = spin of
// kernel site k up
template <typename T, bool ACT>
__device__ void build_lut(const CnnPair<T>& f, const cplx<T>* params, cplx<T>* lut) {
    for (int e = threadIdx.x; e < f.C0 << f.v0; e += blockDim.x) {
        const int ci = e >> f.v0, p = e & ((1 << f.v0) - 1);
        cplx<T> z = {0, 0};
        for (int k = 0; k < f.v0; k++) {
            const cplx<T> q = params[ci * f.v0 + k];
            const T s = (p >> k) & 1 ? T(1) : T(-1);
            z.re += q.re * s;
            z.im += q.im * s;
        }
        lut[e] = ACT ? act(z, 0) : z;
    }
}

__device__ __forceinline__ uint16_t pattern_of(const int* nbr0, int v0, const uint64_t (&w)[kMaxWords], int x) {
    int p = 0;
    for (int k = 0; k < v0; k++) {
        const int y = nbr0[x * v0 + k];
        p |= int((word_at(w, y >> 6) >> (y & 63)) & 1u) << k;
    }
    return uint16_t(p);
}

// second-layer pre-activations z[c] of the channels cb CB .. at a site whose kernel sites have
// the patterns p: input channels outer, kernel sites inner
template <typename T, int CB, int VM>
__device__ __forceinline__ void site_z(const CnnPair<T>& f, const cplx<T>* lut, const int (&p)[VM], int cb,
                                       cplx<T> (&z)[CB]) {
#pragma unroll
    for (int c = 0; c < CB; c++) z[c] = {0, 0};
    const cplx<T>* w = f.wf + size_t(cb) * f.C0 * f.v1 * CB;
    for (int ci = 0; ci < f.C0; ci++) {
        const cplx<T>* l = lut + (ci << f.v0);
        cplx<T> a[VM];
#pragma unroll
        for (int k = 0; k < VM; k++)
            if (VM == 9 || k < f.v1) a[k] = l[p[k]];
#pragma unroll
        for (int k = 0; k < VM; k++) {
            if (k < f.v1) {
#pragma unroll
                for (int c = 0; c < CB; c++) {
                    const cplx<T> q = {ld_uniform(&w[k * CB + c].re), ld_uniform(&w[k * CB + c].im)};
                    z[c].re += q.re * a[k].re - q.im * a[k].im;
                    z[c].im += q.re * a[k].im + q.im * a[k].re;
                }
            }
        }
        w += f.v1 * CB;
    }
}

// sum over the output channels of the activations at a site (channel order)
template <typename T, int CB, int VM>
__device__ __forceinline__ cplx<T> site_out(const CnnPair<T>& f, const cplx<T>* lut, const int (&p)[VM]) {
    cplx<T> s = {0, 0};
    for (int cb = 0; cb < f.blocks; cb++) {
        cplx<T> z[CB];
        site_z<T, CB, VM>(f, lut, p, cb, z);
#pragma unroll
        for (int c = 0; c < CB; c++)
            if (cb * CB + c < f.C1) s = cadd(s, act(z[c], 1));
    }
    return s;
}

// patterns of the second-layer kernel sites of x
template <int VM>
__device__ __forceinline__ void site_patterns(const uint8_t* nbr1, int v1, const uint16_t* pat, int x, int (&p)[VM]) {
#pragma unroll
    for (int k = 0; k < VM; k++) p[k] = k < v1 ? int(pat[nbr1[x * v1 + k]]) : 0;
}

// tables of a workgroup in LDS
template <typename T>
struct PairTables {
    cplx<T>* lut;
    uint32_t* aff0;   // [N][n0] site | toggled pattern bits << 8
    uint8_t* nbr1;    // [N][v1]
    uint8_t* aff1;    // [N][n1] sites in increasing order
    __device__ PairTables(const CnnPair<T>& f, unsigned char* smem) {
        lut = reinterpret_cast<cplx<T>*>(smem);
        aff0 = reinterpret_cast<uint32_t*>(lut + (size_t(f.C0) << f.v0));
        nbr1 = reinterpret_cast<uint8_t*>(aff0 + f.N * f.n0);
        aff1 = nbr1 + f.N * f.v1;
    }
    __device__ void fill(const CnnPair<T>& f, const cplx<T>* params) {
        build_lut<T, true>(f, params, lut);
        for (int e = threadIdx.x; e < f.N * f.n0; e += blockDim.x) aff0[e] = f.aff0[e];
        for (int e = threadIdx.x; e < f.N * f.v1; e += blockDim.x) nbr1[e] = uint8_t(f.nbr1[e]);
        for (int e = threadIdx.x; e < f.N * f.n1; e += blockDim.x) aff1[e] = f.aff1[e];
    }
};
template <typename T>
__host__ __device__ inline size_t pair_table_bytes(const CnnPair<T>& f) {
    return ((size_t(f.C0) << f.v0) * sizeof(cplx<T>) + sizeof(uint32_t) * f.N * f.n0 + size_t(f.N) * (f.v1 + f.n1) + 15) /
           16 * 16;
}

// sum over the LPC lanes of a chain in the order of wave_sum (whose upper rows hold zeros when a
// half wave's 32 lanes carry the sites)
template <int LPC, typename T>
__device__ __forceinline__ T lanes_sum(T v) {
    if constexpr (LPC == 64) {
        return wave_sum(v);
    } else if constexpr (sizeof(T) == 4) {
        v += dpp_f32<0xB1>(v);
        v += dpp_f32<0x4E>(v);
        v += dpp_f32<0x141>(v);
        v += dpp_f32<0x140>(v);
        return v + __shfl_xor(v, 16);
    } else {
        v += dpp_f64<0xB1>(v);
        v += dpp_f64<0x4E>(v);
        v += dpp_f64<0x141>(v);
        v += dpp_f64<0x140>(v);
        return v + __shfl_xor(v, 16);
    }
}

// toggles site i in the patterns (tl: lane of the chain; its own inverse)
template <typename T>
__device__ __forceinline__ void toggle(const CnnPair<T>& f, const PairTables<T>& t, uint16_t* pat, int i, int tl) {
    if (tl < f.n0) {
        const uint32_t e = t.aff0[i * f.n0 + tl];
        pat[e & 255u] ^= uint16_t(e >> 8);
    }
    wave_sync();
}

// the site of lane tl among those that a flip of i (and k, when k >= 0) reaches, -1 beyond them
template <typename T>
__device__ __forceinline__ int reached(const CnnPair<T>& f, const PairTables<T>& t, int i, int k, int tl) {
    if (k < 0) return tl < f.n1 ? int(t.aff1[i * f.n1 + tl]) : -1;
    // the union of the two masks in increasing order (one chain per wave: i, k uniform)
    int at = -1, n = 0;
#pragma unroll
    for (int u = 0; u < kMaxWords; u++) {
        const uint64_t m = f.mask1[i * kMaxWords + u] | f.mask1[k * kMaxWords + u];
        const int c = __popcll(m);
        if (at < 0 && tl < n + c) at = 64 * u + select64(m, uint32_t(tl - n));
        n += c;
    }
    return at;
}

template <typename T, int CB, int VM>
__global__ __launch_bounds__(kPThreads) void cnn_pair_log_psi_kernel(CnnPair<T> f, const cplx<T>* params, T final_factor,
                                                                     const int* nbr0, const uint64_t* confs, int words,
                                                                     int64_t count, cplx<double> lp,
                                                                     cplx<double>* log_psi, double* weight) {
    extern __shared__ __align__(16) unsigned char smem[];
    PairTables<T> t(f, smem);
    t.fill(f, params);
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6);
    uint16_t* pat = reinterpret_cast<uint16_t*>(smem + pair_table_bytes(f)) + wave * 256;
    __syncthreads();
    for (int64_t s = int64_t(blockIdx.x) * kPWaves + wave; s < count; s += int64_t(gridDim.x) * kPWaves) {
        uint64_t w[kMaxWords];
#pragma unroll
        for (int k = 0; k < kMaxWords; k++) w[k] = k < words ? uniform_u64(confs[s * words + k]) : 0;
        for (int x = lane; x < f.N; x += 64) pat[x] = pattern_of(nbr0, f.v0, w, x);
        wave_sync();
        cplx<T> part = {0, 0};
        for (int x = lane; x < f.N; x += 64) {
            int p[VM];
            site_patterns<VM>(t.nbr1, f.v1, pat, x, p);
            part = cadd(part, site_out<T, CB, VM>(f, t.lut, p));
        }
        const cplx<T> L = {final_factor * wave_sum(part.re), final_factor * wave_sum(part.im)};
        if (lane == 0) {
            const cplx<double> r = {lp.re + double(L.re), lp.im + double(L.im)};
            log_psi[s] = r;
            if (weight) weight[s] = exp(2.0 * r.re);
        }
        wave_sync();
    }
}

// Metropolis chains, LPC lanes each (32: single flips that reach at most 32 sites; else 64).
// Proposals as in cnn.hip: the same Philox stream, the same decisions.
template <typename T, int CB, int VM, int LPC>
__global__ __launch_bounds__(kPThreads) void cnn_pair_mc_kernel(CnnPair<T> f, const cplx<T>* params, T final_factor,
                                                                const int* nbr0, uint64_t* chain_confs, int words,
                                                                int num_chains, int move, int64_t num_proposals,
                                                                uint64_t counter, uint32_t key0, uint32_t key1,
                                                                uint32_t* accepted) {
    constexpr int CPW = 64 / LPC;   // chains per wave
    extern __shared__ __align__(16) unsigned char smem[];
    PairTables<T> t(f, smem);
    t.fill(f, params);
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6);
    const int h = lane / LPC, tl = lane % LPC, N = f.N;
    const int slot = wave * CPW + h;
    T* out = reinterpret_cast<T*>(smem + pair_table_bytes(f)) + slot * N;
    uint16_t* pat = reinterpret_cast<uint16_t*>(reinterpret_cast<T*>(smem + pair_table_bytes(f)) + kPWaves * CPW * N) +
                    slot * N;
    const int c0 = (int(blockIdx.x) * kPWaves + wave) * CPW + h;
    const bool live = c0 < num_chains;
    const int c = live ? c0 : num_chains - 1;   // a half without a chain repeats the last one and stores nothing
    __syncthreads();
    uint64_t w[kMaxWords], msk[kMaxWords];
#pragma unroll
    for (int k = 0; k < kMaxWords; k++) {
        w[k] = k < words ? chain_confs[int64_t(c) * words + k] : 0;
        if constexpr (LPC == 64) w[k] = uniform_u64(w[k]);
        const int bits = N - 64 * k;
        msk[k] = k >= words ? 0 : bits >= 64 ? ~uint64_t(0) : bits > 0 ? (uint64_t(1) << bits) - 1 : 0;
    }
    for (int x = tl; x < N; x += LPC) pat[x] = pattern_of(nbr0, f.v0, w, x);
    wave_sync();
    for (int x = tl; x < N; x += LPC) {
        int p[VM];
        site_patterns<VM>(t.nbr1, f.v1, pat, x, p);
        out[x] = site_out<T, CB, VM>(f, t.lut, p).re;
    }
    wave_sync();
    uint32_t acc = 0;
    // random words of LPC proposals at a time, one per lane of the chain
    uint32_t rx = 0, ry = 0, rz = 0;
    for (int64_t q = 0; q < num_proposals; q++) {
        const int ql = int(q & (LPC - 1));
        if (ql == 0) {
            const uint64_t tt = counter + uint64_t(q) + uint64_t(tl);
            const u32x4 r = philox(uint32_t(c), uint32_t(tt), uint32_t(tt >> 32), 0u, key0, key1);
            rx = r.x;
            ry = r.y;
            rz = r.z;
        }
        uint32_t r_x, r_z;
        if constexpr (LPC == 64) {
            r_x = readlane_u32(rx, ql);
            r_z = readlane_u32(rz, ql);
        } else {
            r_x = uint32_t(__shfl(int(rx), h * LPC + ql));
            r_z = uint32_t(__shfl(int(rz), h * LPC + ql));
        }
        const int i = int(range32(r_x, uint32_t(N)));
        int kp = -1;
        if constexpr (LPC == 64) {
            if (move == MOVE_EXCHANGE) {
                const uint32_t r_y = readlane_u32(ry, ql);
                const int si_bit = int((word_at(w, i >> 6) >> (i & 63)) & 1u);
                uint64_t o[kMaxWords];
                uint32_t n_opp = 0;
#pragma unroll
                for (int k = 0; k < kMaxWords; k++) {
                    o[k] = (si_bit ? ~w[k] : w[k]) & msk[k];
                    n_opp += uint32_t(__popcll(o[k]));
                }
                if (n_opp == 0) continue;
                kp = select_bit(o, words, range32(r_y, n_opp));
            }
        }
        toggle(f, t, pat, i, tl);
        if constexpr (LPC == 64)
            if (kp >= 0) toggle(f, t, pat, kp, tl);
        const int x = reached(f, t, i, LPC == 64 ? kp : -1, tl);
        int p[VM];
        site_patterns<VM>(t.nbr1, f.v1, pat, x >= 0 ? x : 0, p);
        const T sx = site_out<T, CB, VM>(f, t.lut, p).re;
        const T d = lanes_sum<LPC>(x >= 0 ? sx - out[x] : T(0));
        const T d2 = T(2) * final_factor * d;
        const T uu = (T(r_z) + T(0.5)) * T(2.3283064365386963e-10);
        const bool accept = d2 > T(0) || uu <= dexp(d2);
        if (accept) {
            if (x >= 0) out[x] = sx;
            if constexpr (LPC == 64) {
                flip_bit(w, i);
                if (kp >= 0) flip_bit(w, kp);
            }
            acc++;
            wave_sync();
        } else {
            toggle(f, t, pat, i, tl);
            if constexpr (LPC == 64)
                if (kp >= 0) toggle(f, t, pat, kp, tl);
        }
    }
    if (!live) return;
    // the spins are the patterns' bits of the kernel site that is the site itself
    for (int k = tl; k < words; k += LPC) {
        uint64_t x = 0;
        for (int b = 0; b < 64 && 64 * k + b < N; b++) x |= uint64_t((pat[64 * k + b] >> f.self0) & 1u) << b;
        chain_confs[int64_t(c) * words + k] = x;
    }
    if (tl == 0) accepted[c] += acc;
}

// Local energies, a wave per sample, 64 / LPC terms at a time (every term of one flip that
// reaches at most 32 sites: LPC = 32)
template <typename T, int CB, int VM, int LPC>
__global__ __launch_bounds__(kPThreads) void cnn_pair_local_energy_kernel(CnnPair<T> f, const cplx<T>* params,
                                                                          T final_factor, const int* nbr0, OpView op,
                                                                          const uint64_t* confs, int64_t count,
                                                                          cplx<double>* e_loc) {
    constexpr int TPW = 64 / LPC;
    extern __shared__ __align__(16) unsigned char smem[];
    PairTables<T> t(f, smem);
    t.fill(f, params);
    const int lane = threadIdx.x & 63, wave = uniform_int(threadIdx.x >> 6);
    const int h = lane / LPC, tl = lane % LPC, N = f.N, words = op.words, G = op.num_groups;
    cplx<T>* out = reinterpret_cast<cplx<T>*>(smem + pair_table_bytes(f)) + wave * N;
    uint16_t* list = reinterpret_cast<uint16_t*>(reinterpret_cast<cplx<T>*>(smem + pair_table_bytes(f)) + kPWaves * N) +
                     wave * G;
    uint16_t* pat = reinterpret_cast<uint16_t*>(reinterpret_cast<cplx<T>*>(smem + pair_table_bytes(f)) + kPWaves * N) +
                    kPWaves * G + (wave * TPW + h) * N;
    // the flipped sites of the terms: first | second << 8 (the first again where there is one)
    uint16_t* sites = reinterpret_cast<uint16_t*>(reinterpret_cast<cplx<T>*>(smem + pair_table_bytes(f)) + kPWaves * N) +
                      kPWaves * (G + TPW * N);
    for (int g = threadIdx.x; g < G; g += kPThreads) {
        const int a = op.group_sites[2 * g], b = op.group_sites[2 * g + 1];
        sites[g] = uint16_t(a < 0 ? 0 : a | (b < 0 ? a : b) << 8);
    }
    __syncthreads();
    for (int64_t s = int64_t(blockIdx.x) * kPWaves + wave; s < count; s += int64_t(gridDim.x) * kPWaves) {
        uint64_t w[kMaxWords];
#pragma unroll
        for (int k = 0; k < kMaxWords; k++) w[k] = k < words ? uniform_u64(confs[s * words + k]) : 0;
        auto strings = [&](int b0, int b1, int step, double& re, double& im) {
            re = im = 0.0;
            for (int n = b0; n < b1; n += step) {
                int par = 0;
#pragma unroll
                for (int k = 0; k < kMaxWords; k++)
                    if (k < words) par += __popcll(~w[k] & op.string_zy[int64_t(n) * words + k]);
                const double sg = (par & 1) ? -1.0 : 1.0;
                re += sg * op.string_coef[2 * n];
                im += sg * op.string_coef[2 * n + 1];
            }
        };
        double e_re = 0.0, e_im = 0.0;
        if (op.diag_group >= 0)
            strings(op.group_begin[op.diag_group] + lane, op.group_begin[op.diag_group + 1], 64, e_re, e_im);
        int terms = 0;
        for (int g0 = 0; g0 < G; g0 += 64) {
            const int g = g0 + lane;
            bool on = false;
            if (g < G && g != op.diag_group) {
                double re, im;
                strings(op.group_begin[g], op.group_begin[g + 1], 1, re, im);
                on = re != 0.0 || im != 0.0;
            }
            const uint64_t b = __ballot(on);
            if (on)
                list[terms + int(__builtin_amdgcn_mbcnt_hi(uint32_t(b >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(b), 0u)))] =
                    uint16_t(g);
            terms += __popcll(b);
        }
        for (int x = tl; x < N; x += LPC) pat[x] = pattern_of(nbr0, f.v0, w, x);
        wave_sync();
        for (int x = lane; x < N; x += 64) {
            int p[VM];
            site_patterns<VM>(t.nbr1, f.v1, pat, x, p);
            out[x] = site_out<T, CB, VM>(f, t.lut, p);
        }
        wave_sync();
        // the terms' log-ratios wait in the lanes of their half until there are LPC of them
        T q_re = 0, q_im = 0;
        int q_g = -1;
        for (int m = 0; m < terms; m += TPW) {
            const int g = m + h < terms ? int(list[m + h]) : -1;
            const int st = g >= 0 ? int(sites[g]) : 0, i = st & 255, k = LPC == 64 && (st >> 8) != i ? st >> 8 : -1;
            toggle(f, t, pat, i, tl);
            if constexpr (LPC == 64)
                if (k >= 0) toggle(f, t, pat, k, tl);
            const int x = reached(f, t, i, k, tl);
            int p[VM];
            site_patterns<VM>(t.nbr1, f.v1, pat, x >= 0 ? x : 0, p);
            cplx<T> sx = site_out<T, CB, VM>(f, t.lut, p);
            toggle(f, t, pat, i, tl);
            if constexpr (LPC == 64)
                if (k >= 0) toggle(f, t, pat, k, tl);
            if (x >= 0)
                sx = csub(sx, out[x]);
            else
                sx = {0, 0};
            const T dr = lanes_sum<LPC>(sx.re), di = lanes_sum<LPC>(sx.im);
            const int at = (m / TPW) % LPC;
            if (tl == at) {
                q_re = dr;
                q_im = di;
                q_g = g;
            }
            if (at == LPC - 1 || m + TPW >= terms) {
                if (q_g >= 0) {
                    double c_re, c_im;
                    strings(op.group_begin[q_g], op.group_begin[q_g + 1], 1, c_re, c_im);
                    const double r = exp(double(final_factor) * double(q_re));
                    double sn, cs;
                    sincos(double(final_factor) * double(q_im), &sn, &cs);
                    e_re += c_re * r * cs - c_im * r * sn;
                    e_im += c_re * r * sn + c_im * r * cs;
                }
                q_g = -1;
            }
        }
        e_re = wave_sum(e_re);
        e_im = wave_sum(e_im);
        if (lane == 0) e_loc[s] = {e_re, e_im};
        wave_sync();
    }
}

// O_k by back-propagation, a workgroup of 4 waves per sample: D1 = d log psi / d z1 (a site per
// thread), the second layer's gradient sum_x D1[cj][x] a0[ci][nbr(x, k)] as a matrix product on
// matrix cores ((ci, k) x (cj re, im), the sites as its K dimension, real and imaginary parts of
// a0 in turn), D0 from the transposed weights, and the first layer's gradient, whose inputs are
// pattern bits.
constexpr int kOThreads = 256;
template <typename T>
struct Acc4;
template <>
struct Acc4<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static __device__ type mma(float a, float b, type c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
template <>
struct Acc4<double> {
    typedef double type __attribute__((ext_vector_type(4)));
    static __device__ type mma(double a, double b, type c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};

template <typename T, int CB, int VM>
__global__ __launch_bounds__(kOThreads) void cnn_pair_ok_kernel(CnnPair<T> f, const cplx<T>* params, T final_factor,
                                                                const int* nbr0, const uint64_t* confs, int words,
                                                                int64_t count, int num_params, cplx<T>* O) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = f.N, tid = threadIdx.x, lane = tid & 63, wave = uniform_int(tid >> 6);
    cplx<T>* lut = reinterpret_cast<cplx<T>*>(smem);              // z0
    cplx<T>* A0 = lut + (size_t(f.C0) << f.v0);                   // [C0][N]
    cplx<T>* D1 = A0 + f.C0 * N;                                  // [C1][N]
    cplx<T>* D0 = D1 + f.C1 * N;                                  // [C0][N]
    cplx<double>* red = reinterpret_cast<cplx<double>*>(D0 + f.C0 * N);   // [kOThreads]
    uint16_t* pat = reinterpret_cast<uint16_t*>(red + kOThreads); // [N]
    uint8_t* nbr1 = reinterpret_cast<uint8_t*>(pat + N);          // [N][v1]
    uint8_t* inv1 = nbr1 + N * f.v1;                              // [N][v1]
    build_lut<T, false>(f, params, lut);
    for (int e = tid; e < N * f.v1; e += kOThreads) {
        nbr1[e] = uint8_t(f.nbr1[e]);
        inv1[e] = f.inv1[e];
    }
    const int link1 = f.C0 * f.v0;   // first parameter of the second layer
    for (int64_t s = blockIdx.x; s < count; s += gridDim.x) {
        cplx<T>* row = O + s * num_params;
        __syncthreads();   // the tables are there; the previous sample is done
        uint64_t w[kMaxWords];
#pragma unroll
        for (int k = 0; k < kMaxWords; k++) w[k] = k < words ? uniform_u64(confs[s * words + k]) : 0;
        if (tid < N) pat[tid] = pattern_of(nbr0, f.v0, w, tid);
        __syncthreads();
        for (int e = tid; e < f.C0 * N; e += kOThreads) A0[e] = act(lut[((e / N) << f.v0) + pat[e % N]], 0);
        __syncthreads();
        if (tid < N) {
            int y[VM];
#pragma unroll
            for (int k = 0; k < VM; k++) y[k] = k < f.v1 ? int(nbr1[tid * f.v1 + k]) : 0;
            for (int cb = 0; cb < f.blocks; cb++) {
                cplx<T> z[CB];
#pragma unroll
                for (int c = 0; c < CB; c++) z[c] = {0, 0};
                const cplx<T>* wq = f.wf + size_t(cb) * f.C0 * f.v1 * CB;
                for (int ci = 0; ci < f.C0; ci++)
#pragma unroll
                    for (int k = 0; k < VM; k++)
                        if (k < f.v1) {
                            const cplx<T> a = A0[ci * N + y[k]];
#pragma unroll
                            for (int c = 0; c < CB; c++) {
                                const cplx<T>* q = wq + (ci * f.v1 + k) * CB + c;
                                const T qr = ld_uniform(&q->re), qi = ld_uniform(&q->im);
                                z[c].re = fma(qr, a.re, fma(-qi, a.im, z[c].re));
                                z[c].im = fma(qr, a.im, fma(qi, a.re, z[c].im));
                            }
                        }
#pragma unroll
                for (int c = 0; c < CB; c++)
                    if (cb * CB + c < f.C1) D1[(cb * CB + c) * N + tid] = cscale(dact(z[c], 1), final_factor);
            }
        }
        __syncthreads();
        // second layer's gradient: tiles of 16 (ci, k) rows over the waves, 8 output channels
        // (re, im columns) at a time; 16 sites are summed in T, their sums in fp64 (one chain
        // over the sites in fp32 doubled the error of the SR solution)
        using M = Acc4<T>;
        const int lc = lane & 15, lk = lane >> 4, rows = f.C0 * f.v1;
        for (int tile = wave; tile * 16 < rows; tile += kOThreads / kWave) {
            const int r = min(tile * 16 + lc, rows - 1), ci = r / f.v1, k = r % f.v1;
            for (int c0 = 0; c0 < f.C1; c0 += 8) {
                const int cj = min(c0 + (lc & 7), f.C1 - 1);
                double sum[4] = {0.0, 0.0, 0.0, 0.0};
                for (int x0 = 0; x0 < N; x0 += 16) {
                    typename M::type acc[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int x = x0 + 4 * u + lk;
                        cplx<T> a = {0, 0}, d = {0, 0};
                        if (x < N) {
                            a = A0[ci * N + nbr1[x * f.v1 + k]];
                            d = D1[cj * N + x];
                        }
                        acc[u] = M::mma(a.re, lc < 8 ? d.re : d.im, typename M::type{0, 0, 0, 0});
                        acc[u] = M::mma(a.im, lc < 8 ? -d.im : d.re, acc[u]);
                    }
                    const typename M::type part = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
                    for (int e = 0; e < 4; e++) sum[e] += double(part[e]);
                }
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int ro = tile * 16 + M::row(lane, e), co = c0 + (lc & 7);
                    if (ro < rows && co < f.C1) {
                        T* o = reinterpret_cast<T*>(row + link1 + ((ro / f.v1) * f.C1 + co) * f.v1 + ro % f.v1);
                        o[lc >> 3] = T(sum[e]);
                    }
                }
            }
        }
        // D0 = (sum over the sites x that read y and the output channels of w D1) tanh(z0)
        if (tid < N) {
            int x[VM];
#pragma unroll
            for (int k = 0; k < VM; k++) x[k] = k < f.v1 ? int(inv1[tid * f.v1 + k]) : 0;
            for (int cb = 0; cb < f.blocks0; cb++) {
                cplx<T> g[CB];
#pragma unroll
                for (int c = 0; c < CB; c++) g[c] = {0, 0};
                const cplx<T>* wq = f.wb + size_t(cb) * f.C1 * f.v1 * CB;
                for (int cj = 0; cj < f.C1; cj++)
#pragma unroll
                    for (int k = 0; k < VM; k++)
                        if (k < f.v1) {
                            const cplx<T> d = D1[cj * N + x[k]];
#pragma unroll
                            for (int c = 0; c < CB; c++) {
                                const cplx<T>* q = wq + (cj * f.v1 + k) * CB + c;
                                const T qr = ld_uniform(&q->re), qi = ld_uniform(&q->im);
                                g[c].re = fma(qr, d.re, fma(-qi, d.im, g[c].re));
                                g[c].im = fma(qr, d.im, fma(qi, d.re, g[c].im));
                            }
                        }
#pragma unroll
                for (int c = 0; c < CB; c++)
                    if (cb * CB + c < f.C0)
                        D0[(cb * CB + c) * N + tid] = cmul(g[c], dact(lut[((cb * CB + c) << f.v0) + pat[tid]], 0));
            }
        }
        __syncthreads();
        // first layer's gradient: (channel, kernel site) pairs times parts of the sites
        const int outs = f.C0 * f.v0, parts = kOThreads / outs;
        const int part = tid / outs, o = tid % outs;
        cplx<double> sum = {0.0, 0.0};
        if (part < parts) {
            const int c = o / f.v0, k = o % f.v0;
            for (int y = part; y < N; y += parts) {
                const cplx<T> d = D0[c * N + y];
                const bool up = (pat[y] >> k) & 1;
                sum.re += double(up ? d.re : -d.re);
                sum.im += double(up ? d.im : -d.im);
            }
        }
        red[tid] = sum;
        __syncthreads();
        if (tid < outs) {
            sum = red[tid];
            for (int q = 1; q < parts; q++) sum = cadd(sum, red[q * outs + tid]);
            row[tid] = {T(sum.re), T(sum.im)};
        }
    }
}

template <int V>
struct PTag {
    static constexpr int value = V;
};

// f(CB, VM): channels per block and kernel sites in registers
template <typename T, typename F>
void dispatch_pair(const CnnPair<T>& f, F&& fn) {
    auto vm = [&](auto cb) {
        if (f.v1 <= 4)
            fn(cb, PTag<4>{});
        else
            fn(cb, PTag<9>{});
    };
    switch (f.cb) {
        case 2: vm(PTag<2>{}); break;
        case 4: vm(PTag<4>{}); break;
        case 8: vm(PTag<8>{}); break;
        default: throw std::logic_error("PsiCNN channel block");
    }
}

template <typename K>
void pair_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        ANN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
}

// persistent workgroups (they build their table once), no more than have work
unsigned pair_grid(int64_t items, int64_t per_block, int per_cu) {
    return unsigned(std::max<int64_t>(1, std::min<int64_t>((items + per_block - 1) / per_block, 256 * int64_t(per_cu))));
}

template <typename T>
size_t pair_ok_lds(const CnnPair<T>& f) {
    return sizeof(cplx<T>) * ((size_t(f.C0) << f.v0) + size_t(2 * f.C0 + f.C1) * f.N) + sizeof(cplx<double>) * kOThreads +
           sizeof(uint16_t) * f.N + 2 * size_t(f.N) * f.v1;
}
template <typename T>
size_t pair_mc_lds(const CnnPair<T>& f, int cpw) {
    return pair_table_bytes(f) + size_t(kPWaves) * cpw * f.N * (sizeof(T) + sizeof(uint16_t));
}
template <typename T>
size_t pair_energy_lds(const CnnPair<T>& f, int tpw, int G) {
    return pair_table_bytes(f) + size_t(kPWaves) * (f.N * sizeof(cplx<T>) + sizeof(uint16_t) * (G + tpw * f.N)) +
           sizeof(uint16_t) * G;
}

// Rounds of 64 lanes in which the general kernels take the outputs that `reached` changed sites
// have: their lanes hold (site, channel) pairs, the lanes here sites with the channels one after
// another.  So for many channels at few sites and no more chains (samples) than the general kernels
// hold at once, `resident`, those are the faster ones (beyond, the more chains in flight here win: 32
// sites, kernels of 3, 4,096 chains, 24 channels 2.2 times, 12 channels 1.5 times).
template <typename T>
int general_rounds(const CnnPair<T>& f, int reached) {
    return (reached * f.C1 + 63) / 64;
}
int64_t resident(size_t general_lds) { return 256 * std::max<int64_t>(1, 160 * 1024 / int64_t(general_lds)); }

}  // namespace

template <typename T>
bool cnn_pair_log_psi(const CnnView<T>& v, const uint64_t* confs, int words, int64_t count, cplx<double> lp,
                      cplx<double>* log_psi, double* weight, hipStream_t stream) {
    const CnnPair<T>& f = v.pair;
    if (!f.wf) return false;
    const size_t lds = pair_table_bytes(f) + sizeof(uint16_t) * 256 * kPWaves;
    if (lds > kPLds) return false;
    dispatch_pair(f, [&](auto cb, auto vm) {
        auto kernel = cnn_pair_log_psi_kernel<T, decltype(cb)::value, decltype(vm)::value>;
        pair_lds(kernel, lds);
        kernel<<<pair_grid(count, kPWaves, 3), kPThreads, lds, stream>>>(f, v.params, v.final_factor, v.nbr, confs, words,
                                                                         count, lp, log_psi, weight);
    });
    ANN_LAUNCH_CHECK();
    count_route("cnn_pair_log_psi");
    return true;
}

template <typename T>
bool cnn_pair_mc(const CnnView<T>& v, uint64_t* chain_confs, int words, int num_chains, int move, int64_t num_proposals,
                 uint64_t counter, uint64_t seed, uint32_t* accepted, size_t general_lds, hipStream_t stream) {
    const CnnPair<T>& f = v.pair;
    if (!f.wf || (move != MOVE_FLIP && move != MOVE_EXCHANGE)) return false;
    // Two rounds for a block of 8 channels is where both take as long: 100 chains in fp32, flips of 32
    // sites, here against there, kernels of 3 (5 sites reached), 8 channels 176 and 247 us, 12 channels
    // 475 and 308, 32 channels 2,817 and 1,634; kernels of 3 x 3 (25 reached), 12 channels 2,580 and 2,580,
    // 16 channels 3,403 and 6,091.
    const int reached = (move == MOVE_EXCHANGE ? 2 : 1) * f.n1;
    if (f.C1 > 8 && num_chains <= resident(general_lds) && general_rounds(f, reached) < 2 * f.blocks) return false;
    const bool half = move == MOVE_FLIP && f.n1 <= 32;
    // a lane per reached site of one or two flips
    if ((move == MOVE_EXCHANGE ? 2 : 1) * f.n1 > 64 || f.n0 > (half ? 32 : 64)) return false;
    const int cpw = half ? 2 : 1;
    const size_t lds = pair_mc_lds(f, cpw);
    if (lds > kPLds) return false;
    const unsigned grid = unsigned((num_chains + kPWaves * cpw - 1) / (kPWaves * cpw));
    dispatch_pair(f, [&](auto cb, auto vm) {
        auto run = [&](auto kernel) {
            pair_lds(kernel, lds);
            kernel<<<grid, kPThreads, lds, stream>>>(f, v.params, v.final_factor, v.nbr, chain_confs, words, num_chains,
                                                     move, num_proposals, counter, uint32_t(seed), uint32_t(seed >> 32),
                                                     accepted);
        };
        if (half)
            run(cnn_pair_mc_kernel<T, decltype(cb)::value, decltype(vm)::value, 32>);
        else
            run(cnn_pair_mc_kernel<T, decltype(cb)::value, decltype(vm)::value, 64>);
    });
    ANN_LAUNCH_CHECK();
    count_route("cnn_pair_mc");
    return true;
}

template <typename T>
bool cnn_pair_local_energy(const CnnView<T>& v, const OpView& op, const uint64_t* confs, int64_t count,
                           cplx<double>* e_loc, size_t general_lds, hipStream_t stream) {
    const CnnPair<T>& f = v.pair;
    if (!f.wf || op.max_flips > 2 || op.num_groups > kPList) return false;
    // as for the chains; two flips at a time are on a par at three rounds a block of channels (512
    // samples, 31 bonds, kernels of 5: 12 channels 443 and 350 us, of 3 x 3: 1.35 times), pairs of single
    // flips at half a round (32 channels, kernels of 2 in fp64: 1,190 and 1,024 us)
    const int rounds = general_rounds(f, std::max(op.max_flips, 1) * f.n1);
    if (f.C1 > 8 && count <= resident(general_lds) &&
        (op.max_flips == 2 ? rounds < 3 * f.blocks : f.blocks >= 4 && 2 * rounds <= f.blocks))
        return false;
    const bool half = op.max_flips <= 1 && f.n1 <= 32;
    if ((op.max_flips == 2 ? 2 : 1) * f.n1 > 64 || f.n0 > (half ? 32 : 64)) return false;
    const size_t lds = pair_energy_lds(f, half ? 2 : 1, op.num_groups);
    if (lds > kPLds) return false;
    dispatch_pair(f, [&](auto cb, auto vm) {
        auto run = [&](auto kernel) {
            pair_lds(kernel, lds);
            kernel<<<pair_grid(count, kPWaves, 2), kPThreads, lds, stream>>>(f, v.params, v.final_factor, v.nbr, op, confs,
                                                                             count, e_loc);
        };
        if (half)
            run(cnn_pair_local_energy_kernel<T, decltype(cb)::value, decltype(vm)::value, 32>);
        else
            run(cnn_pair_local_energy_kernel<T, decltype(cb)::value, decltype(vm)::value, 64>);
    });
    ANN_LAUNCH_CHECK();
    count_route("cnn_pair_local_energy");
    return true;
}

template <typename T>
bool cnn_pair_ok(const CnnView<T>& v, const uint64_t* confs, int words, int64_t count, cplx<T>* O, hipStream_t stream) {
    const CnnPair<T>& f = v.pair;
    if (!f.wf || f.C0 * f.v0 > kOThreads) return false;
    // A workgroup per sample waits 5 us at its barriers whatever the net; a net of few products is the
    // faster on the general kernel's single waves where there are many samples: 40 sites, 5,000 samples, one
    // channel, kernels of 2, here against there 69 and 14 us, 3 channels, kernels of 5, 86 and 84, 4
    // channels 103 and 134; 600 samples, one channel 18 and 10, 4 channels 24 and 88.
    if (125 * int64_t(f.C0) * f.C1 * f.v1 * std::max(f.N, 64) < 64 * std::min<int64_t>(5000, count)) return false;
    const size_t lds = pair_ok_lds(f);
    if (lds > kPLds) return false;
    dispatch_pair(f, [&](auto cb, auto vm) {
        auto kernel = cnn_pair_ok_kernel<T, decltype(cb)::value, decltype(vm)::value>;
        pair_lds(kernel, lds);
        kernel<<<pair_grid(count, 1, 2), kOThreads, lds, stream>>>(f, v.params, v.final_factor, v.nbr, confs, words, count,
                                                                   v.num_params, O);
    });
    ANN_LAUNCH_CHECK();
    count_route("cnn_pair_ok");
    return true;
}

#define ANN_CNN_PAIR_INSTANTIATE(T)                                                                                     \
    template bool cnn_pair_log_psi<T>(const CnnView<T>&, const uint64_t*, int, int64_t, cplx<double>, cplx<double>*,  \
                                      double*, hipStream_t);                                                           \
    template bool cnn_pair_mc<T>(const CnnView<T>&, uint64_t*, int, int, int, int64_t, uint64_t, uint64_t, uint32_t*, \
                                 size_t, hipStream_t);                                                                 \
    template bool cnn_pair_local_energy<T>(const CnnView<T>&, const OpView&, const uint64_t*, int64_t, cplx<double>*, \
                                           size_t, hipStream_t);                                                       \
    template bool cnn_pair_ok<T>(const CnnView<T>&, const uint64_t*, int, int64_t, cplx<T>*, hipStream_t);
ANN_CNN_PAIR_INSTANTIATE(float)
ANN_CNN_PAIR_INSTANTIATE(double)

}  // namespace ann
