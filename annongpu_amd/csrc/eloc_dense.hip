// eloc_dense.hip -- local energies of a dense net for operators whose strings flip at most two
// sites (bonds, transverse fields): a lane per off-diagonal term.
//
// fp32 only: an fp64 evaluation keeps the general kernel and with it its last bits, which a CG
// solve of an ill-conditioned S carries into the 9th digit of its solution after 40 iterations.
//
//   E_loc(s) = sum_g c_g(s) exp(sum_j f_j (lc(theta_j + c_a W_aj + c_b W_bj) - lc(theta_j)))
//
// With the hidden units across the lanes (dense_net.hip's kernel, which stays for operators
// with longer strings) every term pays two wave reductions, the units are padded to whole
// waves and the coefficient is recomputed by all lanes: 300 vector instructions per term and
// wave at 400 units.  Here a lane owns two terms of a sample and walks the units: no
// reduction, no padding, and terms with a zero coefficient (parallel spins of a Heisenberg
// bond) are dropped before they take a lane.  With u = theta_j^2, d = c_a W_aj + c_b W_bj and
// v = d (2 theta_j + d), the change of u, the polynomial lc(u) = u/2 - u^2/12 + u^3/45 changes by
//   v (C1 + v (C2 + v / 45)),  C1 = 1/2 - u/6 + u^2/15,  C2 = -1/12 + u/15,
// 16 instructions per term and unit with f_j in C1, C2 (which depend on the sample alone and are
// staged with 2 theta); it is also 2.5 times closer to the exact value in fp32 than the difference
// of two log-cosh values, which cancels.  A workgroup stages in LDS, per tile of units, its
// samples' 2 theta, C1, C2 and for every term D = 2 (W_b - W_a), [unit][term] (of two equal spins
// -2 (W_b + W_a), where an operator needs them); d is +-D.  Per unit a lane reads the sample's 24
// bytes once and 8 bytes for each of its two terms.  The unit sums are taken per tile in fp32 and
// over the tiles in fp64.
// Bound by the vector units: 0.83 of their issue slots, LDS bank conflicts in 16 % of the cycles.
// 10x10 Heisenberg, 400 units, 16,384 samples, fp32: 1,205 -> 565 us.  With few terms for the units
// the general kernel is the faster one: local_energy_terms_serves.
#include "kernels.hpp"
#include "wave_net.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace ann {

namespace {

using namespace wave;

constexpr int kEThreads = 512;
constexpr int kERounds = 2;     // term pairs per lane and pass over the units
constexpr int kEList = 16384;   // most terms listed per workgroup (2 bytes each)

constexpr int kETile = 52 * 1024;   // most bytes of D in a tile of units

// an LDS entry that is loaded in one piece (cplx<float> is aligned to 4 bytes only)
struct alignas(8) Pair {
    float re, im;
};

struct alignas(8) Angle {
    float re, im, c1re, c1im, c2re, c2im;   // 2 theta_j, f_j C1, f_j C2
};

// LDS of the tile (units x entries of D, the samples' angles, f), which the terms' values
// share afterwards
__host__ __device__ inline size_t eloc_tile_bytes(int threads, int per_block, int units, int entries) {
    const size_t tile = sizeof(Angle) * per_block * units + sizeof(Pair) * units * (entries + 1);
    const size_t values = sizeof(double2) * 2 * kERounds * threads;
    return ((tile > values ? tile : values) + 15) / 16 * 16;
}

template <bool REALF, int WORDS>
__global__ __launch_bounds__(kEThreads, 4) void local_energy_terms_kernel(
    DenseView<float> net, OpView op, const uint64_t* confs, const cplx<float>* theta, int64_t count, int per_block,
    int tu_log2, cplx<double>* e_loc) {
    constexpr int R = kERounds, kEWaves = kEThreads / kWave;
    const int TU = 1 << tu_log2;
    extern __shared__ __align__(16) unsigned char smem[];
    const int G = op.num_groups;
    const int E = op.equal_spins ? 2 * G : G;   // D of every group, then that of two equal spins
    // the tile, and after the units the log-ratios and values of the terms (2 r + k of a thread)
    double2* value = reinterpret_cast<double2*>(smem);                  // [2 R][kEThreads]
    Angle* ang = reinterpret_cast<Angle*>(smem);                        // [per_block][TU]
    Pair* Dt = reinterpret_cast<Pair*>(ang + per_block * TU);           // [TU][E]
    // [2][TU] f / 45, re and im (a scalar load would be waited for together with the LDS reads)
    float* c3 = reinterpret_cast<float*>(Dt + TU * E);
    double2* diag = reinterpret_cast<double2*>(smem + eloc_tile_bytes(kEThreads, per_block, TU, E));   // [per_block]
    uint64_t* cw = reinterpret_cast<uint64_t*>(diag + per_block);       // [per_block][kMaxWords]
    int* first = reinterpret_cast<int*>(cw + per_block * kMaxWords);    // [per_block + 1] first term pair
    int* num = first + per_block + 1;                                   // [per_block] terms
    uint16_t* list = reinterpret_cast<uint16_t*>(num + per_block);      // [per_block][G]
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform_int(tid >> 6);
    constexpr int words = WORDS;
    const int64_t s0 = int64_t(blockIdx.x) * per_block;
    const int samples = int(count - s0 < per_block ? count - s0 : per_block);

    // sum over the strings [b0, b1) of their signed coefficients, `step` strings apart
    auto string_sum = [&](const uint64_t* c, int b0, int b1, int step) {
        double2 r = {0.0, 0.0};
        for (int n = b0; n < b1; n += step) {
            int par = 0;
            for (int k = 0; k < words; k++) par += __popcll(~c[k] & op.string_zy[int64_t(n) * words + k]);
            const double sg = (par & 1) ? -1.0 : 1.0;
            r.x += sg * op.string_coef[2 * n];
            r.y += sg * op.string_coef[2 * n + 1];
        }
        return r;
    };
    auto group_coef = [&](const uint64_t* c, int g) {
        return string_sum(c, op.group_begin[g], op.group_begin[g + 1], 1);
    };
    // the terms of every sample: diagonal energy (strings over the lanes) and the list of
    // off-diagonal groups with a coefficient, in group order
    for (int sl = wave; sl < samples; sl += kEWaves) {
        if (lane < kMaxWords) cw[sl * kMaxWords + lane] = lane < words ? confs[(s0 + sl) * words + lane] : 0;
        wave_sync();
        const uint64_t* c = cw + sl * kMaxWords;
        double2 d = {0.0, 0.0};
        if (op.diag_group >= 0)
            d = string_sum(c, op.group_begin[op.diag_group] + lane, op.group_begin[op.diag_group + 1], 64);
        d = {wave_sum(d.x), wave_sum(d.y)};
        int n = 0;
        for (int g0 = 0; g0 < G; g0 += 64) {
            const int g = g0 + lane;
            bool on = false;
            if (g < G && g != op.diag_group) {
                const double2 x = group_coef(c, g);
                on = x.x != 0.0 || x.y != 0.0;
            }
            const uint64_t b = __ballot(on);
            if (on)
                list[sl * G + n + int(__builtin_amdgcn_mbcnt_hi(uint32_t(b >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(b), 0u)))] =
                    uint16_t(g);
            n += __popcll(b);
        }
        if (lane == 0) {
            diag[sl] = d;
            num[sl] = n;
        }
    }
    __syncthreads();
    if (tid == 0) {
        int p = 0;
        for (int sl = 0; sl < samples; sl++) {
            first[sl] = p;
            p += (num[sl] + 1) >> 1;
        }
        for (int sl = samples; sl <= per_block; sl++) first[sl] = p;
    }
    __syncthreads();
    const int total = first[per_block];
    // 32 threads add up a sample, taking its term pairs in turn
    const int my = tid >> 5;
    // the waves take the places of a round in turn over the workgroups: the last round is
    // rarely full, and its waves would always be those of the same SIMDs
    const int turn = (wave + int(blockIdx.x)) % kEWaves, slot = turn * kWave + lane;
    double er = 0.0, ei = 0.0;
    const int units = net.M;
    for (int base = 0; base < total; base += R * kEThreads) {
        // term pair t: its sample, and its terms e and e + half of the sample's list (neighbouring
        // lanes then read neighbouring sites, few of them in one LDS bank)
        auto find = [&](int t, int& smp, int& g0, int& g1) {
            int lo = 0, hi = per_block;   // first[lo] <= t < first[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (first[mid] <= t) lo = mid; else hi = mid;
            }
            const bool in = t < total;
            const int e = in ? t - first[lo] : 0, n = in ? num[lo] : 0, half = (n + 1) >> 1;
            smp = in ? lo : 0;
            g0 = in ? int(list[lo * G + e]) : -1;
            g1 = e + half < n ? int(list[lo * G + e + half]) : -1;
        };
        int sl[R], o[R][2];
        float sg[R][2];
        double D[R][4];
#pragma unroll
        for (int r = 0; r < R; r++) {
            int g[2];
            find(base + r * kEThreads + slot, sl[r], g[0], g[1]);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int gk = g[k] >= 0 ? g[k] : 0;
                const int v0 = max(op.group_sites[2 * gk], 0), v1 = op.group_sites[2 * gk + 1];
                const uint64_t* c = cw + sl[r] * kMaxWords;
                const bool up = (c[v0 >> 6] >> (v0 & 63)) & 1;
                const bool equal = v1 >= 0 && ((c[v1 >> 6] >> (v1 & 63)) & 1) == uint64_t(up);
                o[r][k] = equal && op.equal_spins ? G + gk : gk;
                sg[r][k] = up ? 1.0f : -1.0f;
                D[r][2 * k] = D[r][2 * k + 1] = 0.0;
            }
        }
        for (int u0 = 0; u0 < units; u0 += TU) {
            __syncthreads();   // the previous tile is consumed
            // D = 2 (W_b - W_a), of two equal spins -2 (W_b + W_a); W_b = 0 for a single site
            const int su = tid & (TU - 1);
            const bool in = u0 + su < net.Mpad;
            const cplx<float>* Wu = net.Wd + (in ? u0 + su : 0);
#pragma unroll 4
            for (int q = tid >> tu_log2; q < E; q += kEThreads >> tu_log2) {
                const int2 v = reinterpret_cast<const int2*>(op.group_sites)[q < G ? q : q - G];
                const cplx<float> a = Wu[int64_t(v.x < 0 ? 0 : v.x) * net.Mpad], b = Wu[int64_t(v.y < 0 ? 0 : v.y) * net.Mpad];
                const float sa = in && v.x >= 0 ? -2.0f : 0.0f, sb = !in || v.y < 0 ? 0.0f : q < G ? 2.0f : -2.0f;
                Dt[su * E + q] = {sb * b.re + sa * a.re, sb * b.im + sa * a.im};
            }
            if (tid < TU) {
                const cplx<float> f = u0 + tid < net.Mpad ? net.f[u0 + tid] : cplx<float>{0.0f, 0.0f};
                c3[tid] = f.re * float(1.0 / 45.0);
                c3[TU + tid] = f.im * float(1.0 / 45.0);
            }
#pragma unroll 1
            for (int e = tid; e < samples * TU; e += kEThreads) {
                const int q = e >> tu_log2, u = e & (TU - 1);
                cplx<float> z = {0.0f, 0.0f};
                if (u0 + u < net.Mpad) z = theta[(s0 + q) * net.Mpad + u0 + u];
                const cplx<float> f = u0 + u < net.Mpad ? net.f[u0 + u] : cplx<float>{0.0f, 0.0f};
                const cplx<float> x = cmul(z, z), x2 = cmul(x, x);
                cplx<float> c1 = {0.5f - x.re * float(1.0 / 6.0) + x2.re * float(1.0 / 15.0),
                              x2.im * float(1.0 / 15.0) - x.im * float(1.0 / 6.0)};
                cplx<float> c2 = {x.re * float(1.0 / 15.0) - float(1.0 / 12.0), x.im * float(1.0 / 15.0)};
                c1 = REALF ? cscale(c1, f.re) : cmul(c1, f);
                c2 = REALF ? cscale(c2, f.re) : cmul(c2, f);
                ang[e] = {2.0f * z.re, 2.0f * z.im, c1.re, c1.im, c2.re, c2.im};
            }
            __syncthreads();
            const int nu = units - u0 < TU ? (units - u0 + 3) / 4 * 4 : TU;   // (f is zero beyond the units)
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (base + r * kEThreads + turn * kWave >= total) break;   // wave-uniform
                float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                const Angle* as = ang + sl[r] * TU;
                const Pair* w[2] = {Dt + o[r][0], Dt + o[r][1]};
                for (int u = 0; u < nu; u += 4) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const Angle z = as[u + q];
                        const float fr = c3[u + q], fi = REALF ? 0.0f : c3[TU + u + q];
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            const Pair d = *w[k];
                            w[k] += E;
                            const float sr = fma(sg[r][k], z.re, d.re), si = fma(sg[r][k], z.im, d.im);
                            const float vr = d.re * sr - d.im * si, vi = d.re * si + d.im * sr;
                            float hr = z.c2re + vr * fr, hi = z.c2im + vi * fr;
                            if constexpr (!REALF) {
                                hr -= vi * fi;
                                hi += vr * fi;
                            }
                            const float gr = fma(-vi, hi, fma(vr, hr, z.c1re)), gi = fma(vi, hr, fma(vr, hi, z.c1im));
                            p[2 * k] = fma(-vi, gi, fma(vr, gr, p[2 * k]));
                            p[2 * k + 1] = fma(vi, gr, fma(vr, gi, p[2 * k + 1]));
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; k++) D[r][k] += double(p[k]);
            }
        }
        // The terms' values, through LDS so that one copy of the exponential serves all of a
        // thread's terms (a copy per term took the registers of the loop above), then added per
        // sample in a fixed order.
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; r++) {
            value[2 * r * kEThreads + slot] = double2{D[r][0], D[r][1]};
            value[(2 * r + 1) * kEThreads + slot] = double2{D[r][2], D[r][3]};
        }
#pragma unroll 1
        for (int i = 0; i < 2 * R; i++) {
            int smp, g[2];
            find(base + (i >> 1) * kEThreads + slot, smp, g[0], g[1]);
            const int gi = i & 1 ? g[1] : g[0];
            double2 x = {0.0, 0.0};
            if (gi >= 0) {
                const double2 d = value[i * kEThreads + slot];
                const double2 q = group_coef(cw + smp * kMaxWords, gi);
                const double m = exp(d.x);
                double sn, cs;
                sincos(d.y, &sn, &cs);
                x = {q.x * (m * cs) - q.y * (m * sn), q.x * (m * sn) + q.y * (m * cs)};
            }
            value[i * kEThreads + slot] = x;
        }
        __syncthreads();
        if (my < samples) {
            const int lo = max(first[my], base), hi = min(first[my + 1], base + R * kEThreads);
            for (int t = lo + (tid & 31); t < hi; t += 32) {
                const double2* v = value + 2 * ((t - base) / kEThreads) * kEThreads + (t - base) % kEThreads;
                er += v[0].x + v[kEThreads].x;
                ei += v[0].y + v[kEThreads].y;
            }
        }
    }
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        er += __shfl_xor(er, d);
        ei += __shfl_xor(ei, d);
    }
    if (my < samples && (tid & 31) == 0) e_loc[s0 + my] = {diag[my].x + er, diag[my].y + ei};
}

}  // namespace

namespace {

struct TermsPlan {
    int units = 0;       // log2 of the units per tile, 32 at most and 4 at least, whose D fit the tile
    int per_block = 0;   // samples per workgroup
    size_t lds = 0;
};

// false: too many terms
bool terms_plan(const OpView& op, int64_t count, TermsPlan* p) {
    const int G = std::max(op.num_groups, 1);
    const int entries = op.equal_spins ? 2 * G : G;
    if (op.max_flips > 2 || G > kEList) return false;
    p->units = 5;
    while (p->units >= 2 && (int64_t(entries) << p->units) * int64_t(sizeof(Pair)) > kETile) p->units--;
    if (p->units < 2) return false;
    // as many samples per workgroup as pay for its tile, fewer where that would leave CUs
    // without their two workgroups, and no more than the term list holds
    const int64_t want = std::min<int64_t>(kEThreads / 32, (count + 511) / 512);
    p->per_block = int(std::min<int64_t>(want, std::max(1, kEList / G)));
    p->lds = eloc_tile_bytes(kEThreads, p->per_block, 1 << p->units, entries) + sizeof(double2) * p->per_block +
             sizeof(uint64_t) * p->per_block * kMaxWords + sizeof(int) * (2 * p->per_block + 1) +
             sizeof(uint16_t) * size_t(p->per_block) * G;
    return true;
}

}  // namespace

// The kernel's time is that of its rounds of workgroups, each a walk over the units per 2,048 terms:
// 0.05 us a unit, 4 us a tile, and the terms' own operations; an operator with few terms leaves
// most of its lanes idle.  The general kernel's is that of its chain of groups (0.8 us a group of up
// to 64 units, more for more units; beyond 512 its registers spill), or of its waves in turn where
// the samples fill the chip.  So: whichever is the shorter by this estimate, fitted to 1,327
// measurements of both (3 to 1,596 groups, 2 to 1,000 units, 1 to 65,536 samples); the one it takes
// is the faster within 5 % for all but 31 of them, within 10 % for all but 15.
// 448 units, 4,000 samples, us here and there: 4 fields 92 and 15, 36 fields 106 and 72, 100 fields
// 170 and 203, 100 bonds 136 and 186; 16,384 samples, 780 pairs of 40 sites, 128 units 1,166 and 2,583,
// 448 units 3,540 and 3,432; 1,596 pairs, 448 units 13,732 and 6,753.
bool local_energy_terms_serves(int M, const OpView& op, int64_t count) {
    TermsPlan p;
    if (!terms_plan(op, count, &p)) return false;
    const int64_t blocks = (count + p.per_block - 1) / p.per_block;
    const int64_t resident = 256 * (p.lds > 80 * 1024 ? 1 : 2);
    const double rounds = double((blocks + resident - 1) / resident);
    const double terms = double(op.terms) * p.per_block;
    const double passes = std::ceil(terms / (2 * kERounds * kEThreads));
    const double here = rounds * (12.5 + M * (passes * (0.048 + 4.0 / (1 << p.units)) + 0.00015 * terms));
    int lane_units = 1;   // units per lane of the general kernel
    for (int u : {1, 2, 4, 7, 8, 16})
        if ((M + 63) / 64 <= (lane_units = u)) break;
    const double wide = lane_units <= 8 ? 1.0 + 0.064 * (lane_units - 1) : 5.3;
    const double general = 4.8 + op.num_groups * wide * std::max(0.78, 0.256e-3 * double(count));
    return here < general;
}

void launch_local_energy_terms(const DenseView<float>& net, const OpView& op, const uint64_t* confs,
                               const cplx<float>* theta, int64_t count, cplx<double>* e_loc, hipStream_t stream) {
    if (count <= 0) return;
    TermsPlan plan;
    if (!terms_plan(op, count, &plan)) throw std::invalid_argument("local energies: too many terms");
    const int per_block = plan.per_block, units = plan.units;
    const size_t lds = plan.lds;
    auto pick = [&](auto realf, auto words) {
        auto kernel = local_energy_terms_kernel<decltype(realf)::value, decltype(words)::value>;
        if (lds > 64 * 1024)
            ANN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        kernel<<<unsigned((count + per_block - 1) / per_block), kEThreads, lds, stream>>>(net, op, confs, theta, count,
                                                                                          per_block, units, e_loc);
    };
    auto pick_words = [&](auto realf) {
        switch (op.words) {
            case 1: pick(realf, std::integral_constant<int, 1>{}); break;
            case 2: pick(realf, std::integral_constant<int, 2>{}); break;
            case 3: pick(realf, std::integral_constant<int, 3>{}); break;
            case 4: pick(realf, std::integral_constant<int, 4>{}); break;
            default: throw HipError("configurations of 1..4 words are supported");
        }
    };
    if (net.real_f)
        pick_words(std::true_type{});
    else
        pick_words(std::false_type{});
    ANN_LAUNCH_CHECK();
    count_route("local_energy_terms");
}

}  // namespace ann
