// k_reduce.hip - on-device FP64 observables, replacing the reference's D2H copy of the
// spins every spins::update steps and the host loop of util::calc_mag method 0
// (src/cuda.cu:234-256, src/util_mag.cpp:44-63).
//
// Determinism: each block reduces its grid-stride share with 64-wide wavefront
// shuffles and a fixed-order combine of its 4 waves; a single block then sums the
// per-block partials in a fixed order.  No floating-point atomics, so the result is
// bitwise reproducible for a given n and launch shape.
#include <algorithm>
#include <map>
#include <mutex>

#include "field.hpp"
#include "kernels.hpp"
#include "philox.hpp"

namespace sllg {

constexpr int kRedBlocks = 512;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block sum of v in fixed order; result valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double* lds) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) lds[w] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int k = 0; k < kTPB / 64; ++k) r += lds[k];
    return r;
}

template <class SpinT>
__device__ __forceinline__ void mag_partial(uint32_t n, uint32_t nsub, uint32_t nblocks, const SpinT* __restrict__ S,
                                            const uint8_t* __restrict__ sub, double* __restrict__ part, double* lds) {
    const uint32_t stride = nblocks * kTPB;
    for (uint32_t s = 0; s < nsub; ++s) {
        double a[3] = {0.0, 0.0, 0.0};
        for (uint32_t i = blockIdx.x * kTPB + threadIdx.x; i < n; i += stride) {
            if (sub && sub[i] != s) continue;
            a[0] += (double)S[i];
            a[1] += (double)S[(size_t)n + i];
            a[2] += (double)S[2 * (size_t)n + i];
        }
        for (int c = 0; c < 3; ++c) {
            const double r = block_sum(a[c], lds);
            if (threadIdx.x == 0) part[(size_t)blockIdx.x * nsub * 3 + s * 3 + c] = r;
        }
    }
}

template <class SpinT>
__global__ __launch_bounds__(kTPB) void k_mag_partial(uint32_t n, uint32_t nsub, const SpinT* __restrict__ S,
                                                      const uint8_t* __restrict__ sub, double* __restrict__ part) {
    __shared__ double lds[kTPB / 64];
    mag_partial<SpinT>(n, nsub, gridDim.x, S, sub, part, lds);
}

// Factors of a sum's values by sublattice (1 / its spins for <M>), passed with the launch.
struct SubScale {
    double v[kMaxSub];
};

// out[v] = scale[v / 3] * sum_b part[b][v]
__device__ __forceinline__ void sum_partials(uint32_t nblocks, uint32_t nval, const double* __restrict__ part,
                                             const double* scale, double* __restrict__ out, double* lds) {
    for (uint32_t v = 0; v < nval; ++v) {
        double a = 0.0;
        for (uint32_t b = threadIdx.x; b < nblocks; b += kTPB) a += part[(size_t)b * nval + v];
        const double r = block_sum(a, lds);
        if (threadIdx.x == 0) out[v] = r * scale[v / 3];
    }
}

__global__ __launch_bounds__(kTPB) void k_sum_partials(uint32_t nblocks, uint32_t nval, const double* __restrict__ part,
                                                       SubScale scale, double* __restrict__ out) {
    __shared__ double lds[kTPB / 64];
    sum_partials(nblocks, nval, part, scale.v, out, lds);
}

// <M> of many FP32 systems in one pair of launches.  A system alone keeps the chip busy for
// some 3 us but costs two launches of 3.6 us each: the members' blocks share a grid, block
// row blockIdx.y being member blockIdx.y, with the blocks, strides and order of sums of the
// single-system kernels (the same bits).
struct MagMember {
    const float* S;
    const uint8_t* sub;  // sublattice per spin, null for one
    double* part;
    double* out;
    uint32_t n, nsub, nblocks, pad_;
    SubScale scale;
};

__global__ __launch_bounds__(kTPB) void k_mag_batch_partial(const MagMember* __restrict__ mem) {
    const MagMember& m = mem[blockIdx.y];
    if (blockIdx.x >= m.nblocks) return;
    __shared__ double lds[kTPB / 64];
    mag_partial<float>(m.n, m.nsub, m.nblocks, m.S, m.sub, m.part, lds);
}

__global__ __launch_bounds__(kTPB) void k_mag_batch_sum(const MagMember* __restrict__ mem) {
    __shared__ double lds[kTPB / 64];
    const MagMember& m = mem[blockIdx.x];
    sum_partials(m.nblocks, m.nsub * 3, m.part, m.scale.v, m.out, lds);
}

// Per-spin energy (J) in FP64:
//   mu mu_B [ -1/2 S.(H_ex + H_dip + H_quad) - 1/4 S.(H_cubic + H_4spin) - S.(B + H_stag) ]
// where H_quad collects the terms linear in S (uniaxial, K2, K4).
struct EnergyArgs {
    uint32_t n;
    int multi;
    double B[3];
    const void* dem;  // float (FP32 path) or double (plain), current dipolar field or null
    const void* stg;
    int f64;
    const uint8_t* spec;
    const Species<double>* sp;
    const double* mu;  // per species, mu_B units
    AnisG<double> an;
    Exch<double> ex;
};

template <int FMT, int NC, class SpinT>
__device__ __forceinline__ void exch_dispatch(const Exch<double>& e, uint32_t i, const SpinT* S, double dot[3]);

template <int FMT, int NC, class SpinT>
__global__ __launch_bounds__(kTPB) void k_energy_partial(EnergyArgs a, const SpinT* __restrict__ S,
                                                         double* __restrict__ part);

}  // namespace sllg

// The sliced-ELL row reader lives in k_fused.hip; the energy kernel needs the same
// traversal in FP64, so it is restated here for the reduction's own translation unit.
namespace sllg {

template <int NC, class SpinT>
__device__ __forceinline__ void exch_row_sell64(const Exch<double>& e, uint32_t i, const SpinT* __restrict__ S,
                                                double dot[3]) {
    const uint32_t n = e.n;
    dot[0] = dot[1] = dot[2] = 0.0;
    const uint32_t sl = i >> 6, lane = i & 63u;
    const uint2 sd = e.slice[sl];
    const uint32_t q0 = sd.x, len = sd.y;
    double v[NC];
    for (uint32_t q = 0; q < len; ++q) {
        uint32_t w, j;
        if (e.fmt == FMT_SELL_PACK)
            w = e.ent[(size_t)q0 * kSlice + pack_pos(q, lane, len)];
        else
            w = e.ent[((size_t)q0 + q) * kSlice + lane];
        if (e.fmt == FMT_SELL_PACK) {
            j = pack_nb(w, i, e.dbits);
            const double* dv = e.dict + (size_t)pack_dict(w, e.dbits) * NC;
            for (int k = 0; k < NC; ++k) v[k] = dv[k];
        } else {
            j = w;
            for (int k = 0; k < NC; ++k) v[k] = e.dict[(size_t)k * e.nent + ((size_t)q0 + q) * kSlice + lane];
        }
        const double s[3] = {(double)S[j], (double)S[n + j], (double)S[2 * (size_t)n + j]};
        accum<NC, double>(v, s, dot);
    }
}

template <int FMT, int NC, class SpinT>
__device__ __forceinline__ void exch_dispatch(const Exch<double>& e, uint32_t i, const SpinT* S, double dot[3]) {
    if constexpr (FMT == FMT_SELL_PACK || FMT == FMT_SELL_RAW)
        exch_row_sell64<NC, SpinT>(e, i, S, dot);
    else if constexpr (FMT == FMT_UNI) {
        if constexpr (sizeof(SpinT) == sizeof(double)) exch_row_uni<NC>(e, i, S, dot);  // FP64 handles only
    } else if constexpr (FMT == FMT_NONE)
        dot[0] = dot[1] = dot[2] = 0.0;
    else
        exch_row_ref<NC, double, double, SpinT>(e, i, S, dot);
}

template <int FMT, int NC, class SpinT>
__global__ __launch_bounds__(kTPB) void k_energy_partial(EnergyArgs a, const SpinT* __restrict__ S,
                                                         double* __restrict__ part) {
    __shared__ double lds[kTPB / 64];
    const uint32_t n = a.n;
    const uint32_t stride = gridDim.x * kTPB;
    double acc = 0.0;
    for (uint32_t i = blockIdx.x * kTPB + threadIdx.x; i < n; i += stride) {
        double dot[3];
        exch_dispatch<FMT, NC, SpinT>(a.ex, i, S, dot);
        const double s[3] = {(double)S[i], (double)S[(size_t)n + i], (double)S[2 * (size_t)n + i]};
        const uint32_t spx = a.multi ? a.spec[i] : 0;
        const Species<double> sp = a.sp[spx];
        double hp[3] = {dot[0], dot[1], dot[2]};
        if (a.dem) {
            for (int c = 0; c < 3; ++c)
                hp[c] += a.f64 ? ((const double*)a.dem)[(size_t)c * n + i] : (double)((const float*)a.dem)[(size_t)c * n + i];
        }
        double hq[3] = {0.0, 0.0, 0.0};
        local_terms<double>(sp.k1u, sp.k1dir, 0.0, a.an, s, hq);
        double hz[3];
        for (int c = 0; c < 3; ++c) {
            hz[c] = a.B[c];
            if (a.stg)
                hz[c] += a.f64 ? ((const double*)a.stg)[(size_t)c * n + i] : (double)((const float*)a.stg)[(size_t)c * n + i];
        }
        const double ep = s[0] * hp[0] + s[1] * hp[1] + s[2] * hp[2];
        const double eq = s[0] * hq[0] + s[1] * hq[1] + s[2] * hq[2];
        const double ec = sp.kc * (s[0] * s[0] * s[0] * s[0] + s[1] * s[1] * s[1] * s[1] + s[2] * s[2] * s[2] * s[2]);
        const double ez = s[0] * hz[0] + s[1] * hz[1] + s[2] * hz[2];
        double e4 = 0.0;  // four-spin: quartic in the spins, -1/4 S.H4
        if (a.ex.fs_xadj) {
            double h4[3];
            fourspin_row<double, double, SpinT>(a.ex, i, S, h4);
            e4 = s[0] * h4[0] + s[1] * h4[1] + s[2] * h4[2];
        }
        acc += a.mu[spx] * LLG_MU_B * (-0.5 * ep - 0.5 * eq - 0.25 * ec - 0.25 * e4 - ez);
    }
    const double r = block_sum(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = r;
}

__global__ __launch_bounds__(kTPB) void k_noise_f64(uint32_t n, Perm perm, uint64_t seed, uint64_t stream, uint64_t t,
                                                    double* out) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    if (i >= n) return;
    double z[3];
    normals3_f64(seed, stream, perm.to_ref(i), t, z);
    for (int c = 0; c < 3; ++c) out[(size_t)c * n + i] = z[c];
}

__global__ __launch_bounds__(kTPB) void k_noise_f32(uint32_t n, Perm perm, uint64_t seed, uint64_t stream, uint64_t t,
                                                    double* out) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    if (i >= n) return;
    float z[3];
    normals3_f32(seed, stream, perm.to_ref(i), t, z);
    for (int c = 0; c < 3; ++c) out[(size_t)c * n + i] = (double)z[c];
}

template <class SpinT>
__global__ __launch_bounds__(kTPB) void k_check_finite(uint32_t n3, const SpinT* __restrict__ S, int* flag) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    if (i >= n3) return;
    const double v = (double)S[i];
    if (!(v == v) || v > 1e300 || v < -1e300) atomicOr(flag, 1);
}

// Binned FP64 sums out[b] = sum over the spins of bin b of w_i S_i.  The spins of a bin are
// listed in ascending device order and cut into chunks of at most kBinChunk; one block
// reduces one chunk (fixed-order block sum), then one thread per bin adds its chunks in
// order.  Deterministic, no atomics.
constexpr uint32_t kBinChunk = 4096;

template <class SpinT>
__global__ __launch_bounds__(kTPB) void k_bin_partial(uint32_t n, const uint32_t* __restrict__ cs,
                                                      const uint32_t* __restrict__ idx, const double* __restrict__ w,
                                                      const SpinT* __restrict__ S, double* __restrict__ part) {
    __shared__ double lds[kTPB / 64];
    const uint32_t b = cs[blockIdx.x], e = cs[blockIdx.x + 1];
    double a[3] = {0.0, 0.0, 0.0};
    for (uint32_t q = b + threadIdx.x; q < e; q += kTPB) {
        const uint32_t i = idx[q];
        const double wq = w ? w[q] : 1.0;
        a[0] += wq * (double)S[i];
        a[1] += wq * (double)S[(size_t)n + i];
        a[2] += wq * (double)S[2 * (size_t)n + i];
    }
    for (int c = 0; c < 3; ++c) {
        const double r = block_sum(a[c], lds);
        if (threadIdx.x == 0) part[(size_t)blockIdx.x * 3 + c] = r;
    }
}

__global__ __launch_bounds__(kTPB) void k_bin_finish(uint32_t nbins, const uint32_t* __restrict__ cb,
                                                     const double* __restrict__ part, double* __restrict__ out) {
    const uint32_t b = blockIdx.x * kTPB + threadIdx.x;
    if (b >= nbins) return;
    double a[3] = {0.0, 0.0, 0.0};
    for (uint32_t k = cb[b]; k < cb[b + 1]; ++k)
        for (int c = 0; c < 3; ++c) a[c] += part[(size_t)k * 3 + c];
    for (int c = 0; c < 3; ++c) out[(size_t)b * 3 + c] = a[c];
}

// Transverse structure factor at a list of mesh wave-vectors k:
//   out[g][k] = sum_{i in g} (S_a(i) ua_i + i S_b(i) ub_i) exp(-2 pi i sum_d k_d x_d(i) / N_d).
// The phase splits over the axes, so the sum is taken in two passes: along one axis d (chosen
// by set_sq) the spins of each mesh plane x_d = const are summed first, once per distinct pair
// of the other two wave-vector components (a "projection" p), then out[g][k] is the sum of the
// planes' values at p(k) times exp(-2 pi i k_d x_d / N_d).  A line of wave-vectors (q, 0, 0),
// which spin-wave runs sample, has one projection with no phase: n complex additions instead
// of n nk phase evaluations.  The planes are cut into chunks of at most kSqChunk spins, one
// block each (4 spins a thread, kept in registers over the projections); partial sums are
// combined in a fixed order.  Phases: (k x mod N) / N exactly in FP64 (products below 2^53),
// then sincospi.
// Wave-vector lists with many projections, or spins in many groups (few to a plane), are summed
// directly instead (k_sq_direct) where that is estimated faster (set_sq).
// Bound by latency (262,144 spins read 1 MB of rows and 2 MB of spins).  64^3 spins, 33
// wave-vectors (q, 0, 0), trace durations: 90 + 125 us for the two passes with one sincospi per
// (spin, k) and one thread per k in the second; 5.1 + 3.8 us here.
constexpr uint32_t kSqChunk = 1024;
constexpr uint32_t kSqTile = 32;  // projections a block takes per pass over its registers

struct SqArgs {
    uint32_t n, nk, np, axis;
    double nu, nv, nd;         // mesh extents along the two projected axes and the plane axis
    const uint32_t* row;       // device row per listed spin
    const uint2* uv;           // mesh coordinates along the two projected axes
    const double2* w;          // (ua, ub) or null
    const uint32_t* cs;        // chunk starts [nch + 1]
    const uint32_t* cx;        // plane coordinate of each chunk
    const uint32_t* cg;        // first chunk of each group [ngroups + 1]
    const uint2* proj;         // [np] wave-vector components along the projected axes
    const uint2* kp;           // [nk] {projection, component along the plane axis}
};

// k x / N modulo 1, k and x below N
__device__ __forceinline__ double sq_turns(double k, double x, double N) {
    const double t = k * x;
    double r = t - floor(t / N) * N;
    if (r < 0.0) r += N;
    if (r >= N) r -= N;
    return r / N;
}

template <class SpinT>
__global__ __launch_bounds__(kTPB) void k_sq_partial(SqArgs a, const SpinT* __restrict__ S, double* __restrict__ part) {
    constexpr uint32_t SPT = kSqChunk / kTPB, NW = kTPB / 64;
    __shared__ double2 lds[kSqTile][NW];
    const uint32_t ch = blockIdx.x, b = a.cs[ch], e = a.cs[ch + 1];
    const uint32_t ca = a.axis == 0 ? 1u : 0u, cb = a.axis == 2 ? 1u : 2u;
    double re[SPT], im[SPT];
    uint2 x[SPT];
#pragma unroll
    for (uint32_t j = 0; j < SPT; ++j) {
        const uint32_t q = b + j * kTPB + threadIdx.x;
        re[j] = im[j] = 0.0;
        x[j] = make_uint2(0u, 0u);
        if (q < e) {
            const uint32_t i = a.row[q];
            const double2 w = a.w ? a.w[q] : make_double2(1.0, 1.0);
            re[j] = (double)S[(size_t)ca * a.n + i] * w.x;
            im[j] = (double)S[(size_t)cb * a.n + i] * w.y;
            x[j] = a.uv[q];
        }
    }
    for (uint32_t p0 = blockIdx.y * kSqTile; p0 < a.np; p0 += gridDim.y * kSqTile) {
        const uint32_t p1 = p0 + kSqTile < a.np ? p0 + kSqTile : a.np;
        for (uint32_t p = p0; p < p1; ++p) {
            const uint2 k = a.proj[p];
            double sr = 0.0, si = 0.0;
            if ((k.x | k.y) == 0u) {
#pragma unroll
                for (uint32_t j = 0; j < SPT; ++j) {
                    sr += re[j];
                    si += im[j];
                }
            } else {
#pragma unroll
                for (uint32_t j = 0; j < SPT; ++j) {
                    const double t = sq_turns(k.x, x[j].x, a.nu) + sq_turns(k.y, x[j].y, a.nv);
                    double sn, cn;
                    sincospi(2.0 * (t - floor(t)), &sn, &cn);
                    // (c_re + i c_im)(cos - i sin)
                    sr += re[j] * cn + im[j] * sn;
                    si += im[j] * cn - re[j] * sn;
                }
            }
            sr = wave_sum(sr);
            si = wave_sum(si);
            if ((threadIdx.x & 63u) == 0) lds[p - p0][threadIdx.x >> 6] = make_double2(sr, si);
        }
        __syncthreads();
        if (threadIdx.x < p1 - p0) {
            double2 v = lds[threadIdx.x][0];
            for (uint32_t w = 1; w < NW; ++w) {
                v.x += lds[threadIdx.x][w].x;
                v.y += lds[threadIdx.x][w].y;
            }
            reinterpret_cast<double2*>(part)[(size_t)ch * a.np + p0 + threadIdx.x] = v;
        }
        __syncthreads();
    }
}

// The direct sum: the spins of each group in chunks of kSqDirect, staged in LDS; each thread takes
// one wave-vector over a chunk.  Phases as above, the residue of k x by a reciprocal: k x and q N are
// exact, and a quotient off by one only moves the phase by a whole turn.
constexpr uint32_t kSqDirect = 512;

struct SqDirect {
    uint32_t n, nk, axis;
    double N[3], inv[3];   // mesh extents, 1 / N
    const uint4* spin;     // {device row, x, y, z} per listed spin
    const double2* w;      // (ua, ub) or null
    const uint32_t* cs;    // chunk starts [nch + 1]
    const uint32_t* cg;    // first chunk of each group [ngroups + 1]
    const uint32_t* kp;    // [nk][3]
};

// k x modulo N, in [-N, 2 N)
__device__ __forceinline__ double sq_residue(double k, double x, double N, double inv) {
    const double t = k * x;
    return fma(-floor(t * inv), N, t);
}

template <class SpinT>
__global__ __launch_bounds__(kTPB) void k_sq_direct(SqDirect a, const SpinT* __restrict__ S, double2* __restrict__ part) {
    __shared__ double sre[kSqDirect], sim[kSqDirect], px[kSqDirect], py[kSqDirect], pz[kSqDirect];
    const uint32_t ch = blockIdx.x, b = a.cs[ch], e = a.cs[ch + 1];
    const uint32_t ca = a.axis == 0 ? 1u : 0u, cb = a.axis == 2 ? 1u : 2u;
    for (uint32_t q = b + threadIdx.x; q < e; q += kTPB) {
        const uint4 sp = a.spin[q];
        const double2 w = a.w ? a.w[q] : make_double2(1.0, 1.0);
        const uint32_t l = q - b;
        sre[l] = (double)S[(size_t)ca * a.n + sp.x] * w.x;
        sim[l] = (double)S[(size_t)cb * a.n + sp.x] * w.y;
        px[l] = (double)sp.y;
        py[l] = (double)sp.z;
        pz[l] = (double)sp.w;
    }
    __syncthreads();
    for (uint32_t k = blockIdx.y * kTPB + threadIdx.x; k < a.nk; k += gridDim.y * kTPB) {
        const double kx = a.kp[3 * (size_t)k], ky = a.kp[3 * (size_t)k + 1], kz = a.kp[3 * (size_t)k + 2];
        double re = 0.0, im = 0.0;
#pragma unroll 2
        for (uint32_t l = 0; l < e - b; ++l) {
            double t = sq_residue(kx, px[l], a.N[0], a.inv[0]) * a.inv[0];
            t = fma(sq_residue(ky, py[l], a.N[1], a.inv[1]), a.inv[1], t);
            t = fma(sq_residue(kz, pz[l], a.N[2], a.inv[2]), a.inv[2], t);
            double sn, cn;
            sincospi(2.0 * (t - floor(t)), &sn, &cn);
            re = fma(sre[l], cn, fma(sim[l], sn, re));
            im = fma(sim[l], cn, fma(-sre[l], sn, im));
        }
        part[(size_t)ch * a.nk + k] = make_double2(re, im);
    }
}

__global__ __launch_bounds__(kTPB) void k_sq_direct_finish(SqDirect a, uint32_t ngroups, const double2* __restrict__ part,
                                                           double* __restrict__ out) {
    const uint32_t v = blockIdx.x * kTPB + threadIdx.x;
    if (v >= ngroups * a.nk) return;
    const uint32_t g = v / a.nk, k = v % a.nk;
    double2 s = make_double2(0.0, 0.0);
    for (uint32_t ch = a.cg[g]; ch < a.cg[g + 1]; ++ch) {
        const double2 c = part[(size_t)ch * a.nk + k];
        s.x += c.x;
        s.y += c.y;
    }
    out[(size_t)v * 2] = s.x;
    out[(size_t)v * 2 + 1] = s.y;
}

// One wave per (group, wave-vector): its lanes take the group's chunks in a stride.
__global__ __launch_bounds__(kTPB) void k_sq_finish(SqArgs a, uint32_t ngroups, const double* __restrict__ part,
                                                     double* __restrict__ out) {
    const uint32_t v = blockIdx.x * (kTPB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (v >= ngroups * a.nk) return;
    const uint32_t g = v / a.nk;
    const uint2 k = a.kp[v % a.nk];
    double re = 0.0, im = 0.0;
    for (uint32_t ch = a.cg[g] + lane; ch < a.cg[g + 1]; ch += 64u) {
        const double2 c = reinterpret_cast<const double2*>(part)[(size_t)ch * a.np + k.x];
        double sn, cn;
        sincospi(2.0 * sq_turns(k.y, a.cx[ch], a.nd), &sn, &cn);
        re += c.x * cn + c.y * sn;
        im += c.y * cn - c.x * sn;
    }
    re = wave_sum(re);
    im = wave_sum(im);
    if (lane == 0) {
        out[(size_t)v * 2] = re;
        out[(size_t)v * 2 + 1] = im;
    }
}

// ---------------------------------------------------------------- host launchers

// A handle's red_out, in doubles: <M> per sublattice [0, 48), the energy, the flag of
// check_finite [63], the species' moments from kRedMu.
constexpr size_t kRedEnergy = kMaxSub * 3, kRedMu = 64;
static_assert(kRedEnergy < 63, "red_out layout");
constexpr size_t kGridRows = 65535;

static int ensure_red(llg_ctx* c) {
    const size_t need = (size_t)kRedBlocks * (size_t)std::max<uint32_t>(c->nsub * 3, 1) * sizeof(double);
    if (c->red_part.bytes < need) SLLG_TRY(c->red_part.alloc(need));
    if (!c->red_out.p) {
        SLLG_TRY(c->red_out.alloc((kRedMu + std::max<size_t>(64, c->mu_sp.size())) * sizeof(double)));
        SLLG_HIP(hipMemcpyAsync(c->red_out.as<double>() + kRedMu, c->mu_sp.data(), c->mu_sp.size() * sizeof(double),
                                hipMemcpyHostToDevice, c->stream));
    }
    return 0;
}

static SubScale inverse_counts(const llg_ctx* c) {
    SubScale s{};
    for (uint32_t k = 0; k < c->nsub; ++k) s.v[k] = c->sub_count[k] ? 1. / (double)c->sub_count[k] : 0.0;
    return s;
}

static unsigned red_blocks(uint32_t n) { return std::min<unsigned>(kRedBlocks, std::max<unsigned>(1, blocks_for(n, kTPB))); }

int reduce_mag(llg_ctx* c, double* dev_out) {
    SLLG_TRY(sync_spins(c));
    SLLG_TRY(ensure_red(c));
    const unsigned nb = red_blocks(c->n);
    const uint8_t* sub = (c->nsub > 1) ? c->sub.as<uint8_t>() : nullptr;
    if (c->prec == LLG_FP64_PLAIN)
        k_mag_partial<double><<<nb, kTPB, 0, c->stream>>>(c->n, c->nsub, c->S.as<double>(), sub, c->red_part.as<double>());
    else
        k_mag_partial<float><<<nb, kTPB, 0, c->stream>>>(c->n, c->nsub, c->S.as<float>(), sub, c->red_part.as<double>());
    SLLG_HIP(hipGetLastError());
    k_sum_partials<<<1, kTPB, 0, c->stream>>>(nb, c->nsub * 3, c->red_part.as<double>(), inverse_counts(c),
                                              dev_out);
    SLLG_HIP(hipGetLastError());
    return 0;
}

int reduce_result(llg_ctx* c, double** m, double** energy) {
    SLLG_TRY(ensure_red(c));
    *m = c->red_out.as<double>();
    *energy = *m + kRedEnergy;
    return 0;
}

// One table upload and two launches for all the members (each on stream s).  48 requests of
// 10^3..48^3 spins with 650 member samples: 174 ms, and 188 ms with two launches and an upload
// of the counts a member.
int batch_reduce_mag(hipStream_t s, const std::vector<llg_ctx*>& members, double* dev_out, uint32_t stride,
                     DevBuf& work) {
    if (members.empty()) return 0;
    std::vector<MagMember> tab(members.size());
    size_t parts = 0;
    uint32_t most = 1;
    for (size_t k = 0; k < members.size(); ++k) {
        llg_ctx* c = members[k];
        SLLG_TRY(sync_spins(c));
        MagMember& m = tab[k];
        m = MagMember{};
        m.n = c->n;
        m.nsub = c->nsub;
        m.nblocks = red_blocks(c->n);
        m.S = c->S.as<float>();
        m.sub = c->nsub > 1 ? c->sub.as<uint8_t>() : nullptr;
        m.out = dev_out + k * (size_t)stride;
        m.scale = inverse_counts(c);
        parts += (size_t)m.nblocks * m.nsub * 3;
        most = std::max(most, m.nblocks);
    }
    const size_t tb = tab.size() * sizeof(MagMember), need = tb + parts * sizeof(double);
    if (work.bytes < need) SLLG_TRY(work.alloc(need + need / 2));
    double* part = reinterpret_cast<double*>(work.as<char>() + tb);
    for (auto& m : tab) {
        m.part = part;
        part += (size_t)m.nblocks * m.nsub * 3;
    }
    SLLG_HIP(hipMemcpyAsync(work.p, tab.data(), tb, hipMemcpyHostToDevice, s));
    for (size_t k0 = 0; k0 < tab.size(); k0 += kGridRows) {  // grid.y holds at most 65535 members
        const unsigned cnt = (unsigned)std::min<size_t>(kGridRows, tab.size() - k0);
        k_mag_batch_partial<<<dim3(most, cnt), kTPB, 0, s>>>(work.as<MagMember>() + k0);
        SLLG_HIP(hipGetLastError());
        k_mag_batch_sum<<<cnt, kTPB, 0, s>>>(work.as<MagMember>() + k0);
        SLLG_HIP(hipGetLastError());
    }
    return 0;
}

// ---------------------------------------------------------------- allocation-free <M>

// Device scratch of llg_reduce_mag_noalloc: one file-scope array per GPU (each GPU that runs
// the library holds its own copy until the process ends).  Layout of one call:
//   [0, nb nsub 3)          per-block partial sums (every slot written by its block)
//   [kPartDoubles, +48)     the results, nsub x 3
// Every call on one GPU uses the same array: calls that overlap on one GPU (two host
// threads, or two streams without ordering between them) race.
constexpr size_t kPartDoubles = (size_t)kRedBlocks * kMaxSub * 3;
constexpr size_t kScratchDoubles = kPartDoubles + kMaxSub * 3;  // 196,992 bytes
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_dev[kMaxDevices] = {};  // device address of each GPU's copy of `scratch`
}  // namespace

// Address of `scratch` on device dev (current), looked up once per device.
static int scratch_of(int dev, double** out) {
    if (dev < 0 || dev >= kMaxDevices) SLLG_FAIL(LLG_E_INVALID, "device %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            SLLG_FAIL(LLG_E_DEVICE, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_dev[dev] = static_cast<double*>(p);
    }
    *out = g_scratch_dev[dev];
    return 0;
}

int reduce_mag_noalloc(llg_ctx* c, double* m) {
    const uint32_t nsub = c->nsub;
    const unsigned nb = red_blocks(c->n);
    if (nsub == 0 || nsub > kMaxSub || (size_t)nb * nsub * 3 > kPartDoubles)
        SLLG_FAIL(LLG_E_UNSUPPORTED, "allocation-free reduction: %u sublattices x %u blocks exceed its %zu-double "
                  "device scratch", nsub, nb, kScratchDoubles);
    double* base = nullptr;
    SLLG_TRY(scratch_of(c->device, &base));
    double* part = base;
    double* out = base + kPartDoubles;
    SLLG_TRY(sync_spins(c));  // rebuilds S in place when only its AoS3 copy is current
    const uint8_t* sub = (nsub > 1) ? c->sub.as<uint8_t>() : nullptr;
    if (c->prec == LLG_FP64_PLAIN)
        k_mag_partial<double><<<nb, kTPB, 0, c->stream>>>(c->n, nsub, c->S.as<double>(), sub, part);
    else
        k_mag_partial<float><<<nb, kTPB, 0, c->stream>>>(c->n, nsub, c->S.as<float>(), sub, part);
    SLLG_HIP(hipGetLastError());
    k_sum_partials<<<1, kTPB, 0, c->stream>>>(nb, nsub * 3, part, inverse_counts(c), out);
    SLLG_HIP(hipGetLastError());
    SLLG_HIP(hipMemcpyAsync(m, out, nsub * 3 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    SLLG_HIP(hipStreamSynchronize(c->stream));
    return 0;
}

int reduce_energy(llg_ctx* c, const void* dem_now, double* dev_out) {
    SLLG_TRY(sync_spins(c));
    SLLG_TRY(ensure_red(c));
    const unsigned nb = red_blocks(c->n);
    EnergyArgs a{};
    a.n = c->n;
    a.multi = c->multi_species ? 1 : 0;
    for (int k = 0; k < 3; ++k) a.B[k] = c->B[k];
    a.f64 = c->prec == LLG_FP64_PLAIN;
    a.dem = dem_now;
    a.stg = c->stag_set ? c->STG.p : nullptr;
    a.spec = c->spec.as<uint8_t>();
    a.sp = c->sp64d.as<Species<double>>();
    a.mu = c->red_out.as<double>() + kRedMu;
    a.an = c->an64;
    a.ex = c->ex64;
    double* part = c->red_part.as<double>();
    const int fmt = c->ex64.fmt;  // the FP32 path's FP64 view is the packed or raw encoding
    const int nc = c->ex64.ncomp;
#define SLLG_E(F, N)                                                                                 \
    do {                                                                                             \
        if (a.f64)                                                                                   \
            k_energy_partial<F, N, double><<<nb, kTPB, 0, c->stream>>>(a, c->S.as<double>(), part);  \
        else                                                                                         \
            k_energy_partial<F, N, float><<<nb, kTPB, 0, c->stream>>>(a, c->S.as<float>(), part);    \
    } while (0)
#define SLLG_E_NC(F)                         \
    do {                                     \
        if (nc == 1) SLLG_E(F, 1);           \
        else if (nc == 3) SLLG_E(F, 3);      \
        else SLLG_E(F, 9);                   \
    } while (0)
    switch (fmt) {
        case FMT_NONE: SLLG_E(FMT_NONE, 1); break;
        case FMT_CSR: SLLG_E_NC(FMT_CSR); break;
        case FMT_UNI: SLLG_E_NC(FMT_UNI); break;
        case FMT_DIA: SLLG_E_NC(FMT_DIA); break;
        case FMT_STENCIL: SLLG_E_NC(FMT_STENCIL); break;
        case FMT_SELL_PACK: SLLG_E_NC(FMT_SELL_PACK); break;
        default: SLLG_E_NC(FMT_SELL_RAW); break;
    }
#undef SLLG_E_NC
#undef SLLG_E
    SLLG_HIP(hipGetLastError());
    SubScale one{};
    one.v[0] = 1.0;
    k_sum_partials<<<1, kTPB, 0, c->stream>>>(nb, 1, part, one, dev_out);
    SLLG_HIP(hipGetLastError());
    return 0;
}

int noise_sample(llg_ctx* c, uint64_t t, double* dev_out) {
    if (c->prec == LLG_FP64_PLAIN)
        k_noise_f64<<<blocks_for(c->n, kTPB), kTPB, 0, c->stream>>>(c->n, c->perm, c->seed, c->stream_id, t, dev_out);
    else
        k_noise_f32<<<blocks_for(c->n, kTPB), kTPB, 0, c->stream>>>(c->n, c->perm, c->seed, c->stream_id, t, dev_out);
    SLLG_HIP(hipGetLastError());
    return 0;
}

int check_finite(llg_ctx* c, int* bad) {
    SLLG_TRY(sync_spins(c));
    SLLG_TRY(ensure_red(c));
    int* flag = reinterpret_cast<int*>(c->red_out.as<double>() + 63);
    SLLG_HIP(hipMemsetAsync(flag, 0, sizeof(int), c->stream));
    const uint32_t n3 = 3 * c->n;
    if (c->prec == LLG_FP64_PLAIN)
        k_check_finite<double><<<blocks_for(n3, kTPB), kTPB, 0, c->stream>>>(n3, c->S.as<double>(), flag);
    else
        k_check_finite<float><<<blocks_for(n3, kTPB), kTPB, 0, c->stream>>>(n3, c->S.as<float>(), flag);
    SLLG_HIP(hipGetLastError());
    SLLG_HIP(hipMemcpyAsync(bad, flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    SLLG_HIP(hipStreamSynchronize(c->stream));
    return 0;
}

int set_bins(llg_ctx* c, uint32_t nbins, const uint32_t* bin, const double* weight) {
    const uint32_t n = c->n;
    // spins of each bin in ascending device order (bin and weight are given in reference order)
    std::vector<uint32_t> cnt(nbins + 1, 0);
    for (uint32_t i = 0; i < n; ++i)
        if (bin[i] < nbins) ++cnt[bin[i] + 1];
    for (uint32_t b = 0; b < nbins; ++b) cnt[b + 1] += cnt[b];
    std::vector<uint32_t> idx(std::max<uint32_t>(1, cnt[nbins])), fill(cnt.begin(), cnt.end() - 1);
    std::vector<double> w(weight ? idx.size() : 0);
    for (uint32_t d = 0; d < n; ++d) {
        const uint32_t i = c->perm.to_ref(d);
        const uint32_t b = bin[i];
        if (b >= nbins) continue;
        if (weight) w[fill[b]] = weight[i];
        idx[fill[b]++] = d;
    }
    std::vector<uint32_t> cs(1, 0), cb(nbins + 1, 0);
    for (uint32_t b = 0; b < nbins; ++b) {
        cb[b] = (uint32_t)cs.size() - 1;
        for (uint32_t q = cnt[b]; q < cnt[b + 1]; q += kBinChunk) cs.push_back(std::min(cnt[b + 1], q + kBinChunk));
    }
    cb[nbins] = (uint32_t)cs.size() - 1;
    const uint32_t nch = (uint32_t)cs.size() - 1;
    auto up = [&](DevBuf& d, const void* h, size_t bytes) -> int {
        SLLG_TRY(d.alloc(std::max<size_t>(bytes, 8)));
        if (bytes) SLLG_HIP(hipMemcpyAsync(d.p, h, bytes, hipMemcpyHostToDevice, c->stream));
        return 0;
    };
    SLLG_TRY(up(c->bin_idx, idx.data(), idx.size() * 4));
    if (weight)
        SLLG_TRY(up(c->bin_w, w.data(), w.size() * 8));
    else
        c->bin_w.release();
    SLLG_TRY(up(c->bin_cs, cs.data(), cs.size() * 4));
    SLLG_TRY(up(c->bin_cb, cb.data(), cb.size() * 4));
    SLLG_TRY(c->bin_part.alloc(std::max<size_t>(1, nch) * 3 * sizeof(double)));
    SLLG_HIP(hipStreamSynchronize(c->stream));
    c->nbins = nbins;
    c->nbin_chunks = nch;
    return 0;
}

int reduce_bins(llg_ctx* c, double* dev_out) {
    SLLG_TRY(sync_spins(c));
    if (c->nbins == 0) return 0;
    const double* w = c->bin_w.p ? c->bin_w.as<double>() : nullptr;
    if (c->nbin_chunks) {
        if (c->prec == LLG_FP64_PLAIN)
            k_bin_partial<double><<<c->nbin_chunks, kTPB, 0, c->stream>>>(
                c->n, c->bin_cs.as<uint32_t>(), c->bin_idx.as<uint32_t>(), w, c->S.as<double>(), c->bin_part.as<double>());
        else
            k_bin_partial<float><<<c->nbin_chunks, kTPB, 0, c->stream>>>(
                c->n, c->bin_cs.as<uint32_t>(), c->bin_idx.as<uint32_t>(), w, c->S.as<float>(), c->bin_part.as<double>());
        SLLG_HIP(hipGetLastError());
    }
    k_bin_finish<<<blocks_for(c->nbins, kTPB), kTPB, 0, c->stream>>>(c->nbins, c->bin_cb.as<uint32_t>(),
                                                                     c->bin_part.as<double>(), dev_out);
    SLLG_HIP(hipGetLastError());
    return 0;
}

int set_sq(llg_ctx* c, const uint32_t grid[3], const uint32_t* mesh, uint32_t nk, const uint32_t* kpts, int axis,
           const double* ua, const double* ub, uint32_t ngroups, const uint32_t* group) {
    const uint32_t n = c->n;
    // The plane axis: the one with the least work, (spins x projections) in the first pass and
    // (planes x wave-vectors) in the second.  Projections: the distinct pairs of the other two
    // wave-vector components.
    const int ax[3][3] = {{0, 1, 2}, {1, 0, 2}, {2, 0, 1}};  // plane axis, projected axes
    int d = 0;
    std::vector<uint2> kp(nk), proj;
    double best = 0.0;
    for (int t = 0; t < 3; ++t) {
        std::map<std::pair<uint32_t, uint32_t>, uint32_t> seen;
        std::vector<uint2> kq(nk), pr;
        for (uint32_t k = 0; k < nk; ++k) {
            const uint32_t* q = kpts + 3 * (size_t)k;
            const auto it = seen.emplace(std::make_pair(q[ax[t][1]], q[ax[t][2]]), (uint32_t)pr.size());
            if (it.second) pr.push_back(make_uint2(q[ax[t][1]], q[ax[t][2]]));
            kq[k] = make_uint2(it.first->second, q[ax[t][0]]);
        }
        const double planes = (double)std::min<uint64_t>(n, (uint64_t)ngroups * grid[ax[t][0]]) + (double)n / kSqChunk;
        const double cost = (double)n * pr.size() + planes * ((double)nk + (double)kTPB * pr.size());
        if (t == 0 || cost < best) {
            best = cost;
            d = t;
            kp.swap(kq);
            proj.swap(pr);
        }
    }
    // Spins of each group, and of each of its planes: counted where there are not many more
    // (group, plane) pairs than spins, else from a sorted list.
    const uint64_t D = grid[ax[d][0]], pairs = (uint64_t)ngroups * D;
    const bool counted = pairs <= 4ull * n + 1024;
    std::vector<std::pair<uint64_t, uint32_t>> list;  // (group, plane), device row
    std::vector<uint32_t> at(counted ? pairs + 1 : 0, 0), first(ngroups + 1, 0);
    auto each = [&](auto&& take) {
        for (uint32_t r = 0; r < n; ++r) {
            const uint32_t i = c->perm.to_ref(r), g = group ? group[i] : 0u;
            if (g < ngroups) take(g, mesh[3 * (size_t)i + ax[d][0]], r, i);
        }
    };
    uint64_t planes = 0;  // chunks of planes
    if (counted) {
        each([&](uint32_t g, uint32_t x, uint32_t, uint32_t) { ++at[g * D + x + 1]; });
        for (uint64_t k = 0; k < pairs; ++k) {
            planes += (at[k + 1] + kSqChunk - 1) / kSqChunk;
            first[k / D + 1] += at[k + 1];
            at[k + 1] += at[k];
        }
    } else {
        list.reserve(n);
        each([&](uint32_t g, uint32_t x, uint32_t r, uint32_t) { list.emplace_back(((uint64_t)g << 32) | x, r); });
        std::sort(list.begin(), list.end());
        for (size_t q = 0, from = 0; q < list.size(); ++q) {
            ++first[(list[q].first >> 32) + 1];
            if (q + 1 < list.size() && list[q + 1].first == list[q].first) continue;
            planes += (q + 1 - from + kSqChunk - 1) / kSqChunk;
            from = q + 1;
        }
    }
    uint32_t longest = 0;  // spins of the longest direct chunk
    for (uint32_t g = 0; g < ngroups; ++g) {
        longest = std::max(longest, std::min(kSqDirect, first[g + 1]));
        first[g + 1] += first[g];
    }
    const uint32_t listed = first[ngroups];
    const bool weighted = ua || ub;
    auto up = [&](DevBuf& b, const void* h, size_t bytes) -> int {
        SLLG_TRY(b.alloc(std::max<size_t>(bytes, 8)));
        if (bytes) SLLG_HIP(hipMemcpyAsync(b.p, h, bytes, hipMemcpyHostToDevice, c->stream));
        return 0;
    };
    // Two passes or the direct sum, by an estimate of their times in us: a chunk of a plane and a
    // projection take 4.0 ns with the chip full (0.5 without a phase), whatever the spins in the
    // chunk, and a block 1.5 us for each of its projections; a spin and 256 wave-vectors take 0.65 ns
    // with the chip full, and a direct chunk of 512 spins 100 us.  us a sample, two passes and direct:
    // 64^3 spins, 1,000 wave-vectors 974 and 691; 500 in 16 groups 1,990 and 429; 48^3, 300 in 300
    // groups 15,575 and 386; 14 x 5 x 4, 1,202 in 2 groups 75 and 58; 32^3, 50 wave-vectors 72 and 126; a
    // line of 33 of 64^3 29 and 215.
    double phases = 0.0;
    for (const uint2& p : proj) phases += (p.x | p.y) ? 4.0e-3 : 0.5e-3;
    const double tile = 1.5 / 4.0e-3 * std::min(phases, kSqTile * 4.0e-3);
    const double two_pass = std::max((double)planes * phases, tile);
    const double direct = std::max(100.0 / kSqDirect * (double)longest, 0.65e-3 * (double)listed * ((nk + 255) / 256));
    if (direct < two_pass) {
        std::vector<uint4> sp(std::max<uint32_t>(1, listed));
        std::vector<double2> w(weighted ? sp.size() : 0);
        std::vector<uint32_t> fill(first.begin(), first.end() - 1), cs(1, 0), cg(ngroups + 1, 0);
        each([&](uint32_t g, uint32_t, uint32_t r, uint32_t i) {
            const uint32_t q = fill[g]++;
            sp[q] = make_uint4(r, mesh[3 * (size_t)i], mesh[3 * (size_t)i + 1], mesh[3 * (size_t)i + 2]);
            if (weighted) w[q] = make_double2(ua ? ua[i] : 1.0, ub ? ub[i] : 1.0);
        });
        for (uint32_t g = 0; g < ngroups; ++g) {
            cg[g] = (uint32_t)cs.size() - 1;
            for (uint32_t q = first[g]; q < first[g + 1]; q += std::min(kSqDirect, first[g + 1] - q))
                cs.push_back(q + std::min(kSqDirect, first[g + 1] - q));
        }
        const uint32_t dchunks = cg[ngroups] = (uint32_t)cs.size() - 1;
        SLLG_TRY(up(c->sq_row, sp.data(), sp.size() * sizeof(uint4)));
        c->sq_uv.release();
        c->sq_cx.release();
        c->sq_proj.release();
        if (weighted)
            SLLG_TRY(up(c->sq_w, w.data(), w.size() * sizeof(double2)));
        else
            c->sq_w.release();
        SLLG_TRY(up(c->sq_cs, cs.data(), cs.size() * 4));
        SLLG_TRY(up(c->sq_cg, cg.data(), cg.size() * 4));
        SLLG_TRY(up(c->sq_k, kpts, (size_t)nk * 3 * 4));
        SLLG_TRY(c->sq_part.alloc(std::max<size_t>(1, (size_t)dchunks * nk) * 2 * sizeof(double)));
        SLLG_TRY(c->sq_out.alloc(std::max<size_t>(1, (size_t)ngroups * nk) * 2 * sizeof(double)));
        SLLG_HIP(hipStreamSynchronize(c->stream));
        c->sq_nk = nk;
        c->sq_np = 0;
        c->sq_ngroups = ngroups;
        c->sq_nch = dchunks;
        c->sq_axis = axis;
        for (int a = 0; a < 3; ++a) c->sq_grid[a] = grid[a];
        return 0;
    }
    // listed spins by (group, plane), ascending device row within a plane
    if (counted) {
        list.resize(listed);
        each([&](uint32_t g, uint32_t x, uint32_t r, uint32_t) { list[at[g * D + x]++] = {((uint64_t)g << 32) | x, r}; });
    }
    std::vector<uint32_t> row(std::max<size_t>(1, list.size()));
    std::vector<uint2> uv(row.size());
    std::vector<double2> w(weighted ? row.size() : 0);
    std::vector<uint32_t> cs(1, 0), cx, cg(ngroups + 1, 0);
    for (size_t q = 0; q < list.size(); ++q) {
        const uint32_t r = list[q].second, i = c->perm.to_ref(r);
        row[q] = r;
        uv[q] = make_uint2(mesh[3 * (size_t)i + ax[d][1]], mesh[3 * (size_t)i + ax[d][2]]);
        if (weighted) w[q] = make_double2(ua ? ua[i] : 1.0, ub ? ub[i] : 1.0);
        if (q + 1 == list.size() || list[q + 1].first != list[q].first || q + 1 - cs.back() == kSqChunk) {
            cs.push_back((uint32_t)q + 1);
            cx.push_back((uint32_t)list[q].first);
            cg[(list[q].first >> 32) + 1] = (uint32_t)cx.size();  // end of the group's chunks so far
        }
    }
    for (uint32_t g = 0; g < ngroups; ++g) cg[g + 1] = std::max(cg[g + 1], cg[g]);  // groups without spins
    const uint32_t nch = (uint32_t)cx.size();
    SLLG_TRY(up(c->sq_row, row.data(), row.size() * 4));
    SLLG_TRY(up(c->sq_uv, uv.data(), uv.size() * sizeof(uint2)));
    if (weighted)
        SLLG_TRY(up(c->sq_w, w.data(), w.size() * sizeof(double2)));
    else
        c->sq_w.release();
    SLLG_TRY(up(c->sq_cs, cs.data(), cs.size() * 4));
    SLLG_TRY(up(c->sq_cx, cx.data(), cx.size() * 4));
    SLLG_TRY(up(c->sq_cg, cg.data(), cg.size() * 4));
    SLLG_TRY(up(c->sq_proj, proj.data(), proj.size() * sizeof(uint2)));
    SLLG_TRY(up(c->sq_k, kp.data(), kp.size() * sizeof(uint2)));
    SLLG_TRY(c->sq_part.alloc(std::max<size_t>(1, (size_t)nch * proj.size()) * 2 * sizeof(double)));
    SLLG_TRY(c->sq_out.alloc(std::max<size_t>(1, (size_t)ngroups * nk) * 2 * sizeof(double)));
    SLLG_HIP(hipStreamSynchronize(c->stream));
    c->sq_nk = nk;
    c->sq_np = (uint32_t)proj.size();
    c->sq_ngroups = ngroups;
    c->sq_nch = nch;
    c->sq_axis = axis;
    for (int a = 0; a < 3; ++a) c->sq_grid[a] = grid[ax[d][a]];
    return 0;
}

int sample_sq(llg_ctx* c, double* dev_out) {
    SLLG_TRY(sync_spins(c));
    if (c->sq_nk == 0 || c->sq_ngroups == 0) return 0;
    if (c->sq_np == 0) {  // the direct sum
        SqDirect a{};
        a.n = c->n;
        a.nk = c->sq_nk;
        a.axis = (uint32_t)c->sq_axis;
        for (int k = 0; k < 3; ++k) {
            a.N[k] = (double)c->sq_grid[k];
            a.inv[k] = 1.0 / a.N[k];
        }
        a.spin = c->sq_row.as<uint4>();
        a.w = c->sq_w.as<double2>();
        a.cs = c->sq_cs.as<uint32_t>();
        a.cg = c->sq_cg.as<uint32_t>();
        a.kp = c->sq_k.as<uint32_t>();
        double2* const part = c->sq_part.as<double2>();
        if (c->sq_nch) {
            const dim3 grid(c->sq_nch, std::min(blocks_for(a.nk, kTPB), 65535u));
            if (c->prec == LLG_FP64_PLAIN)
                k_sq_direct<double><<<grid, kTPB, 0, c->stream>>>(a, c->S.as<double>(), part);
            else
                k_sq_direct<float><<<grid, kTPB, 0, c->stream>>>(a, c->S.as<float>(), part);
            SLLG_HIP(hipGetLastError());
        }
        k_sq_direct_finish<<<blocks_for((size_t)c->sq_ngroups * c->sq_nk, kTPB), kTPB, 0, c->stream>>>(
            a, c->sq_ngroups, part, dev_out);
        SLLG_HIP(hipGetLastError());
        return 0;
    }
    SqArgs a{};
    a.n = c->n;
    a.nk = c->sq_nk;
    a.np = c->sq_np;
    a.axis = (uint32_t)c->sq_axis;
    a.nd = (double)c->sq_grid[0];
    a.nu = (double)c->sq_grid[1];
    a.nv = (double)c->sq_grid[2];
    a.row = c->sq_row.as<uint32_t>();
    a.uv = c->sq_uv.as<uint2>();
    a.w = c->sq_w.as<double2>();
    a.cs = c->sq_cs.as<uint32_t>();
    a.cx = c->sq_cx.as<uint32_t>();
    a.cg = c->sq_cg.as<uint32_t>();
    a.proj = c->sq_proj.as<uint2>();
    a.kp = c->sq_k.as<uint2>();
    if (c->sq_nch) {
        const dim3 grid(c->sq_nch, std::min(blocks_for(a.np, kSqTile), 65535u));
        if (c->prec == LLG_FP64_PLAIN)
            k_sq_partial<double><<<grid, kTPB, 0, c->stream>>>(a, c->S.as<double>(), c->sq_part.as<double>());
        else
            k_sq_partial<float><<<grid, kTPB, 0, c->stream>>>(a, c->S.as<float>(), c->sq_part.as<double>());
        SLLG_HIP(hipGetLastError());
    }
    k_sq_finish<<<blocks_for((size_t)c->sq_ngroups * c->sq_nk, kTPB / 64), kTPB, 0, c->stream>>>(
        a, c->sq_ngroups, c->sq_part.as<double>(), dev_out);
    SLLG_HIP(hipGetLastError());
    return 0;
}

}  // namespace sllg
