// k_conv.hip - FP32 convolution of a spin mesh with a mirror-symmetric real-space kernel:
// the dipolar field (src/intmat.cpp:263-331, src/cuda.cu:61-90) and FFT exchange of one species
// whose tensors are symmetric and mirror-symmetric (src/exch_intmat.cpp:28-160), zero-padded, on
// meshes of up to 128 x 128 x 32 points.
//
//   N_ab(r) = N_ba(r),  N_ab(.., -r_d, ..) = s N_ab(.., r_d, ..),  s = -1 if exactly one of a, b is d.
//
// Its transform is then real with the same mirror symmetry in k, so one octant (kx <= Gx/2, ky <=
// Gy/2, kz <= Gz/2) holds all of it.  It is stored as [kx][kz][ky][3][3], both triangles, so that
// the wave of one component reads its row as three neighbouring floats: 10.2 MB for the 128 x
// 128 x 16 film (six components would be 6.8) instead of 26.7 MB (six real components over the whole
// kx range) or 80 MB (nine complex ones).  Gx and Gy are the powers
// of two of at least twice the extents: a linear convolution may be padded further, so extents
// that are no powers of two take this path too.  Gz is twice the extent: z is transformed
// directly.
//
// The transforms along z at kz = 0 and kz = Gz/2 are real, so the two travel as one sequence
// F = X_0 + i X_{Gz/2} through the y and x transforms (rows s = 0 .. lz - 1 instead of lz + 1):
// with F' = conj F(-kx, -ky), X_0 = (F + F') / 2 and i X_{Gz/2} = (F - F') / 2, so the product
// is P F + Q F' with P, Q = (N(0) +- N(Gz/2)) / 2.  Row 0 is stored in an order that puts the
// columns ky and -ky side by side (pair_pos).
//
// Three kernels a convolution, spectra [component][x][s][ky] in HBM between them:
//   k_conv_fwd  one (component, x) plane a block: direct DFT along z, FFT along y
//   k_conv_x    FFT along x, product with N(k), inverse FFT along x, columns in registers
//   k_conv_inv  one plane a block: inverse FFT along y, inverse DFT along z
// The FFTs hold R points of a sequence in each of T = G / R threads and go through LDS once:
// a radix-R butterfly in registers, twiddles, an exchange inside the wave, a radix-T butterfly.
// The radix-2 form they replaced made four LDS passes and a block barrier a pass per transform
// and was bound by them (about 20 LDS accesses a point and x transform against 4 here).
// 128 x 128 x 16 film (trace durations): forward planes 16.1 -> 9.3 us, x 25.4 -> 15.8 us (26.3
// with the complex FFT-exchange kernel), inverse planes 13.4 -> 9.6 us.  The three move 67 MB,
// the kernel's 10 included (13 us at copy rate).  A film's 1,024 to 1,536 waves of work are 1.5 a
// SIMD in the plane kernels and 2.6 in the x kernel, and busy CUs issue VALU work 44, 58 and 44 %
// of their time (forward, x, inverse): waves wait for data (about 40 % of their lives), and in the
// x kernel a third of the CUs' time goes to LDS bank conflicts of the exchange.  100 x 84 x 12 (padded to 256 x 256 x 24, 200 x
// 168 x 24 with hipFFT and the scatter, product and gather kernels): 102 -> 35 us a
// refresh.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

#include "conv.hpp"

namespace sllg {

namespace {

// Points per thread (R) and threads per sequence (T) of a G-point transform.
constexpr int fft_r(int g) { return g >= 128 ? 16 : (g >= 32 ? 8 : 4); }
constexpr int fft_t(int g) { return g / fft_r(g); }
constexpr int fft_cols(int g) { return 64 / fft_t(g); }                  // sequences a wave holds
constexpr int fft_lds(int g) { return fft_r(g) * (fft_t(g) + 1); }       // exchange slots a sequence

typedef float2 c2;
__device__ __forceinline__ c2 add(c2 a, c2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ c2 sub(c2 a, c2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ c2 mul(c2 w, c2 v) { return make_float2(w.x * v.x - w.y * v.y, w.x * v.y + w.y * v.x); }
// v times w (forward) or conj(w) (inverse)
template <bool FWD>
__device__ __forceinline__ c2 mulw(c2 w, c2 v) {
    return FWD ? mul(w, v) : make_float2(w.x * v.x + w.y * v.y, w.x * v.y - w.y * v.x);
}
// v times -i (forward) or i (inverse)
template <bool FWD>
__device__ __forceinline__ c2 roti(c2 v) {
    return FWD ? make_float2(v.y, -v.x) : make_float2(-v.y, v.x);
}

// 4-point butterfly in natural order; HALF: a2 = a3 = 0.
template <bool FWD, bool HALF>
__device__ __forceinline__ void dft4(c2& a0, c2& a1, c2& a2, c2& a3) {
    if constexpr (HALF) {
        const c2 t = roti<FWD>(a1), x0 = a0, x1 = a1;
        a0 = add(x0, x1);
        a1 = add(x0, t);
        a2 = sub(x0, x1);
        a3 = sub(x0, t);
    } else {
        const c2 t0 = add(a0, a2), t1 = sub(a0, a2), t2 = add(a1, a3), t3 = roti<FWD>(sub(a1, a3));
        a0 = add(t0, t2);
        a1 = add(t1, t3);
        a2 = sub(t0, t2);
        a3 = sub(t1, t3);
    }
}

// exp(-2 pi i m / 16), m = 0 .. 9
__device__ __forceinline__ c2 w16(int m) {
    constexpr float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f, h = 0.70710678118654752440f;
    switch (m) {
        case 1: return make_float2(c1, -s1);
        case 2: return make_float2(h, -h);
        case 3: return make_float2(s1, -c1);
        case 4: return make_float2(0.f, -1.f);
        case 6: return make_float2(-h, -h);
        case 9: return make_float2(-c1, s1);
        default: return make_float2(1.f, 0.f);
    }
}
// v times w16^m (conjugated for the inverse); m is a constant after unrolling
template <bool FWD>
__device__ __forceinline__ c2 tw16(int m, c2 v) {
    if (m == 0) return v;
    if (m == 4) return roti<FWD>(v);
    if (m == 2) {
        constexpr float h = 0.70710678118654752440f;
        return FWD ? make_float2(h * (v.x + v.y), h * (v.y - v.x)) : make_float2(h * (v.x - v.y), h * (v.y + v.x));
    }
    if (m == 6) {
        constexpr float h = 0.70710678118654752440f;
        return FWD ? make_float2(h * (v.y - v.x), -h * (v.x + v.y)) : make_float2(-h * (v.x + v.y), h * (v.x - v.y));
    }
    return mulw<FWD>(w16(m), v);
}

// L-point transform of v[0, L) in registers, natural order in and out (L = 4, 8, 16);
// HALF: the upper half of the input is zero and not read.
template <int L, bool FWD, bool HALF>
__device__ __forceinline__ void dft(c2* v) {
    if constexpr (L == 4) {
        dft4<FWD, HALF>(v[0], v[1], v[2], v[3]);
    } else {
        constexpr int B = L / 4;  // x[B a + b] -> over a, twiddle w_L^(b c), over b -> X[c + 4 d]
        c2 y[L];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            c2 a0 = v[b], a1 = v[B + b], a2 = HALF ? make_float2(0.f, 0.f) : v[2 * B + b],
               a3 = HALF ? make_float2(0.f, 0.f) : v[3 * B + b];
            dft4<FWD, HALF>(a0, a1, a2, a3);
            y[b] = a0;
            y[B + b] = tw16<FWD>(16 / L * b, a1);
            y[2 * B + b] = tw16<FWD>(16 / L * 2 * b, a2);
            y[3 * B + b] = tw16<FWD>(16 / L * 3 * b, a3);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            c2* q = y + c * B;
            if constexpr (B == 4) {
                dft4<FWD, false>(q[0], q[1], q[2], q[3]);
            } else {
                const c2 s = add(q[0], q[1]), t = sub(q[0], q[1]);
                q[0] = s;
                q[1] = t;
            }
#pragma unroll
            for (int d = 0; d < B; ++d) v[c + 4 * d] = q[d];
        }
    }
}

// The wave's LDS operations are issued and executed in order; this keeps the compiler from
// moving them across the point.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Forward transform of one sequence: thread t of T holds x[t + T j] in v[j] (j < R/2; the
// upper half is zero) and ends with X[t + T m + R k2] in v[m T + k2].  w[k] = exp(-2 pi i t k / G).
template <int G>
__device__ __forceinline__ void fft_fwd(c2* v, const c2* w, c2* ex, uint32_t t) {
    constexpr int R = fft_r(G), T = fft_t(G);
    dft<R, true, true>(v);
#pragma unroll
    for (int k = 0; k < R; ++k) ex[k * (T + 1) + t] = k ? mul(w[k], v[k]) : v[0];
    wave_sync();
#pragma unroll
    for (int m = 0; m < R / T; ++m) {
#pragma unroll
        for (int q = 0; q < T; ++q) v[m * T + q] = ex[(t + T * m) * (T + 1) + q];
        dft<T, true, false>(v + m * T);
    }
    wave_sync();
}

// Inverse (unnormalised): X[t + T m + R k2] in v[m T + k2] to x[t + T j] in v[j], j < R/2 of use.
template <int G>
__device__ __forceinline__ void fft_inv(c2* v, const c2* w, c2* ex, uint32_t t) {
    constexpr int R = fft_r(G), T = fft_t(G);
#pragma unroll
    for (int m = 0; m < R / T; ++m) {
        dft<T, false, false>(v + m * T);
#pragma unroll
        for (int q = 0; q < T; ++q) ex[(t + T * m) * (T + 1) + q] = v[m * T + q];
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const c2 x = ex[k * (T + 1) + t];
        v[k] = k ? mulw<false>(w[k], x) : x;
    }
    wave_sync();
    dft<R, false, false>(v);
}

template <int G>
__device__ __forceinline__ void load_tw(c2* w, const c2* __restrict__ tab, uint32_t t) {
#pragma unroll
    for (int k = 0; k < fft_r(G); ++k) w[k] = tab[t * k];  // t k <= (T - 1)(R - 1) < G
}

struct ConvArgs {
    uint32_t n, lx, ly, lz;
    uint32_t dense;       // the map is the identity (every point, mesh order)
    uint32_t si, sc;      // component c of spin i at [si i + sc c] of the spins
    const uint32_t* map;  // [x][y][z]: device spin or ~0
    const float* mu;      // moments (dipolar) or null (FFT exchange)
    const c2* twx;        // exp(-2 pi i m / Gx), m < Gx
    const c2* twy;
    const c2* zt;         // [lz][lz]: row 0 (1, (-1)^z), row s exp(-2 pi i s z / Gz)
    const float* N;       // [kx <= Gx/2][kz][ky <= Gy/2][3][3]
    c2* spec;             // [component][x][s < lz][ky], row 0 by pair_pos
};

// Column position of ky in row 0: 0, G/2, then the pairs (1, G - 1), (2, G - 2), ..
__device__ __forceinline__ uint32_t pair_pos(uint32_t k, uint32_t G) {
    return k == 0u ? 0u : (k == G / 2u ? 1u : (k < G / 2u ? 2u * k : 2u * (G - k) + 1u));
}
__device__ __forceinline__ uint32_t pair_ky(uint32_t p, uint32_t G) {
    return p == 0u ? 0u : (p == 1u ? G / 2u : ((p & 1u) ? G - p / 2u : p / 2u));
}

// Waves of a plane block: each takes fft_cols sequences at a time.
constexpr uint32_t kConvWaves = 4;

// Forward plane.
template <int GY>
__global__ __launch_bounds__(64 * kConvWaves) void k_conv_fwd(ConvArgs a, const float* __restrict__ S) {
    constexpr int R = fft_r(GY), T = fft_t(GY), C = fft_cols(GY);
    extern __shared__ c2 conv_lds[];
    const uint32_t nt = blockDim.x, nw = nt / 64u, lz = a.lz, ls = lz + 1u;
    c2* const exch = conv_lds;                                     // nw C sequences
    c2* const zt = exch + nw * C * fft_lds(GY);                    // lz lz
    float* const P = reinterpret_cast<float*>(zt + lz * lz);       // GY/2 rows of lz + 1
    const uint32_t c = blockIdx.x / a.lx, x = blockIdx.x % a.lx, pts = a.ly * lz;
    const uint32_t i0 = x * pts;
    const uint32_t lane = threadIdx.x & 63u, t = lane % T, col = lane / T, wave = threadIdx.x / 64u;
    c2 w[R];
    load_tw<GY>(w, a.twy, t);
    // the plane in batches of loads that are all in flight before the first is used (one load
    // at a time, each waited for: 11.2 us on the 128 x 128 x 16 film against 9.3)
    constexpr uint32_t U = 8;
    for (uint32_t e0 = threadIdx.x; e0 < (GY / 2) * lz; e0 += U * nt) {
        float r[U];
        uint32_t i[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t e = e0 + u * nt;
            i[u] = e >= pts ? 0xFFFFFFFFu : (a.dense ? i0 + e : a.map[i0 + e]);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t q = i[u] == 0xFFFFFFFFu ? 0u : i[u];
            r[u] = (a.mu ? a.mu[q] : 1.f) * S[(size_t)q * a.si + (size_t)c * a.sc];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t e = e0 + u * nt;
            if (e < (GY / 2) * lz) P[e + e / lz] = i[u] == 0xFFFFFFFFu ? 0.f : r[u];
        }
    }
    for (uint32_t e = threadIdx.x; e < lz * lz; e += nt) zt[e] = a.zt[e];
    c2* const ex = exch + (wave * C + col) * fft_lds(GY);
    c2* const out = a.spec + ((size_t)c * a.lx + x) * lz * GY;
    __syncthreads();
    for (uint32_t s0 = wave * C; s0 < lz; s0 += nw * C) {
        const bool on = s0 + col < lz;
        const uint32_t s = on ? s0 + col : lz - 1u;
        c2 v[R];
#pragma unroll
        for (int j = 0; j < R / 2; ++j) v[j] = make_float2(0.f, 0.f);
#pragma unroll 4
        for (uint32_t z = 0; z < lz; ++z) {
            const c2 q = zt[s * lz + z];
#pragma unroll
            for (int j = 0; j < R / 2; ++j) {
                const float r = P[(t + T * j) * ls + z];
                v[j].x += r * q.x;
                v[j].y += r * q.y;
            }
        }
        fft_fwd<GY>(v, w, ex, t);
        if (on) {
            c2* const row = out + (size_t)s * GY;
#pragma unroll
            for (int m = 0; m < R / T; ++m)
#pragma unroll
                for (int q = 0; q < T; ++q) {
                    const uint32_t k = t + T * m + R * q;
                    row[s == 0u ? pair_pos(k, GY) : k] = v[m * T + q];
                }
        }
    }
}

// Real inverse DFT along z of LY rows, h(z) = dot(X_0, zt_0(z)) + 2 sum_s dot(X_s, zt_s(z)), Z
// values of z a thread.
template <int LY, uint32_t Z>
__device__ __forceinline__ void conv_z(const c2* X, const c2* zt, float* P, uint32_t lz, float scale) {
    const uint32_t ls = lz + 1u, nz = (lz + Z - 1u) / Z;
    for (uint32_t e = threadIdx.x; e < LY * nz; e += blockDim.x) {
        const uint32_t y = e % LY, z0 = e / LY * Z;
        float h0[Z], h[Z];
        const c2 x0 = X[y];
#pragma unroll
        for (uint32_t q = 0; q < Z; ++q) {
            h0[q] = x0.x + (((z0 + q) & 1u) ? -x0.y : x0.y);
            h[q] = 0.f;
        }
        for (uint32_t s = 1; s < lz; ++s) {
            const c2 v = X[s * LY + y];
#pragma unroll
            for (uint32_t q = 0; q < Z; ++q) {
                const c2 u = zt[s * lz + (z0 + q < lz ? z0 + q : lz - 1u)];
                h[q] += v.x * u.x + v.y * u.y;
            }
        }
#pragma unroll
        for (uint32_t q = 0; q < Z; ++q)
            if (z0 + q < lz) P[y * ls + z0 + q] = (h0[q] + 2.f * h[q]) * scale;
    }
}

// Inverse plane: the y transforms of the lz sequences (row 0: H_0 + i H_{Gz/2}, whose results
// are real) into LDS by the block's first nw waves, then the z transforms by all of them: eight z
// a thread, fewer where that would leave threads without any.  With only the nw waves and always
// eight z a thread, 64 of the 128 threads of a 16 x 16 x 32 mesh carried the serial z sums (13.0
// us a kernel).  A step with the dipolar field of a 16 x 16 x 32 mesh takes 27.7 us (31.7 before),
// 64 x 8 x 24 27.3 (31.7), 128 x 128 x 32 78.3 (88.8); with FFT exchange 40.2 (53.1), 40.5 (53.8)
// and 136 (159); flat meshes stay as they were.
template <int GY>
__global__ __launch_bounds__(64 * kConvWaves) void k_conv_inv(ConvArgs a, uint32_t nw, float scale, float* __restrict__ H) {
    constexpr int R = fft_r(GY), T = fft_t(GY), C = fft_cols(GY), LY = GY / 2;
    extern __shared__ c2 conv_lds[];
    const uint32_t nt = blockDim.x, lz = a.lz;
    c2* const zt = conv_lds;                          // lz lz
    c2* const X = zt + lz * lz;                       // lz sequences of LY
    c2* const exch = X + lz * LY;                     // nw C sequences, then the plane's field
    float* const P = reinterpret_cast<float*>(exch);  // LY rows of lz + 1
    const uint32_t c = blockIdx.x / a.lx, x = blockIdx.x % a.lx, pts = a.ly * lz;
    const uint32_t lane = threadIdx.x & 63u, t = lane % T, col = lane / T, wave = threadIdx.x / 64u;
    for (uint32_t e = threadIdx.x; e < lz * lz; e += nt) zt[e] = a.zt[e];
    c2 w[R];
    load_tw<GY>(w, a.twy, t);
    c2* const ex = exch + (wave * C + col) * fft_lds(GY);
    const c2* const in = a.spec + ((size_t)c * a.lx + x) * lz * GY;
    for (uint32_t s0 = wave < nw ? wave * C : lz; s0 < lz; s0 += nw * C) {
        const bool on = s0 + col < lz;
        const uint32_t s = on ? s0 + col : lz - 1u;
        const c2* const row = in + (size_t)s * GY;
        c2 v[R];
#pragma unroll
        for (int m = 0; m < R / T; ++m)
#pragma unroll
            for (int q = 0; q < T; ++q) {
                const uint32_t k = t + T * m + R * q;
                v[m * T + q] = row[s == 0u ? pair_pos(k, GY) : k];
            }
        fft_inv<GY>(v, w, ex, t);
        if (on) {
#pragma unroll
            for (int j = 0; j < R / 2; ++j) X[s * LY + t + T * j] = v[j];
        }
    }
    __syncthreads();
    if (LY * ((lz + 7u) / 8u) >= nt)
        conv_z<LY, 8>(X, zt, P, lz, scale);
    else if (LY * ((lz + 3u) / 4u) >= nt)
        conv_z<LY, 4>(X, zt, P, lz, scale);
    else if (LY * ((lz + 1u) / 2u) >= nt)
        conv_z<LY, 2>(X, zt, P, lz, scale);
    else
        conv_z<LY, 1>(X, zt, P, lz, scale);
    __syncthreads();
    const uint32_t i0 = x * pts;
    for (uint32_t e = threadIdx.x; e < pts; e += nt) {
        const uint32_t i = a.dense ? i0 + e : a.map[i0 + e];
        if (i != 0xFFFFFFFFu) H[(size_t)c * a.n + i] = P[e + e / lz];
    }
}

// Columns (s, ky): a block of three waves, one per component, takes fft_cols(GX) neighbouring
// columns, whole in registers.  The spectra pass between the waves through LDS once for the
// product (every wave holds the same (column, kx) per lane; row 0 also reads F at (-kx, -ky),
// in the neighbouring column), and each wave reads the three kernel values of its row, once per
// (column, |kx|, |ky|).  One wave holding all three components needs no barrier, but a thousand
// such waves leave each SIMD with one or two and nothing to overlap their loads with (29.2 us
// on the 128 x 128 x 16 film).
// Blocks are dealt so that each XCD takes a contiguous range of columns (neighbouring columns
// share cache lines).
template <int GX>
__global__ __launch_bounds__(192, 4) void k_conv_x(ConvArgs a, uint32_t gy) {
    constexpr int R = fft_r(GX), T = fft_t(GX), C = fft_cols(GX);
    __shared__ c2 exch[3][C * fft_lds(GX)];  // at least R 64 slots a wave
    const uint32_t nb = gridDim.x, per = nb >> 3, rem = nb & 7u, xb = blockIdx.x & 7u;
    const uint32_t blk = xb * per + (xb < rem ? xb : rem) + (blockIdx.x >> 3);
    const uint32_t lane = threadIdx.x & 63u, t = lane / C, col = lane % C;
    const uint32_t c = __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
    const uint32_t M = a.lz * gy, j = blk * C + col;  // gy is a multiple of C: a block is in one row
    c2* const ex = exch[c] + col * fft_lds(GX);
    c2* const sp = a.spec + (size_t)c * a.lx * M + j;
    c2 w[R], v[R];
#pragma unroll
    for (int q = 0; q < R / 2; ++q) {
        const uint32_t x = t + T * q;
        v[q] = x < a.lx ? sp[(size_t)x * M] : make_float2(0.f, 0.f);
    }
    load_tw<GX>(w, a.twx, t);
    const uint32_t s = __builtin_amdgcn_readfirstlane(blk * C / gy), hy = gy / 2u, ny = hy + 1u;
    const uint32_t ky = s ? j - s * gy : pair_ky(j, gy);
    const float sy = ky <= hy ? 1.f : -1.f;
    const float* const nrow = a.N + ((size_t)s * ny + (ky <= hy ? ky : gy - ky)) * 9u + 3u * c;
    const size_t nstr = (size_t)(a.lz + 1u) * ny * 9u;  // per kx
    // mirror signs of the wave's row: components with one x change under kx -> -kx, with one y
    // under ky -> -ky
    const float f0 = c == 1 ? sy : 1.f, f1 = c == 1 ? 1.f : sy, f2 = c == 1 ? sy : 1.f;
    fft_fwd<GX>(v, w, ex, t);
    const uint32_t b1 = c == 0 ? 1 : 0, b2 = c == 2 ? 1 : 2;  // the other components, ascending
#pragma unroll
    for (int q = 0; q < R; ++q) exch[c][q * 64 + lane] = v[q];
    __syncthreads();
    if (s) {
#pragma unroll
        for (int m = 0; m < R / T; ++m)
#pragma unroll
            for (int q = 0; q < T; ++q) {
                const uint32_t k = t + T * m + R * q, i = m * T + q;
                const bool up = q >= T / 2;  // k >= Gx / 2
                const float* const np = nrow + (up ? GX - k : k) * nstr;
                float n0 = np[0] * f0, n1 = np[1] * f1, n2 = np[2] * f2;
                if (up) {
                    if (c == 0) {
                        n1 = -n1;
                        n2 = -n2;
                    } else {
                        n0 = -n0;
                    }
                }
                const c2 s1 = exch[b1][i * 64 + lane], s2 = exch[b2][i * 64 + lane];
                const c2 sx = c == 0 ? v[i] : s1, s_y = c == 1 ? v[i] : (c == 0 ? s1 : s2), sz = c == 2 ? v[i] : s2;
                v[i] = make_float2(n0 * sx.x + n1 * s_y.x + n2 * sz.x, n0 * sx.y + n1 * s_y.y + n2 * sz.y);
            }
    } else {
        const uint32_t pc = j < 2u ? col : col ^ 1u;  // the column of -ky
        const size_t nyq = (size_t)a.lz * ny * 9u;
#pragma unroll
        for (int m = 0; m < R / T; ++m)
#pragma unroll
            for (int q = 0; q < T; ++q) {
                const uint32_t k = t + T * m + R * q;
                const bool up = q >= T / 2;
                const float* const np = nrow + (up ? GX - k : k) * nstr;
                const uint32_t k1 = (GX - k) % GX, i1 = (k1 % R) / T * T + k1 / R, l1 = k1 % R % T * C + pc;
                float f[3] = {f0, f1, f2};
                if (up) {
                    if (c == 0) {
                        f[1] = -f[1];
                        f[2] = -f[2];
                    } else {
                        f[0] = -f[0];
                    }
                }
                float re = 0.f, im = 0.f;
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const float n0 = np[b] * f[b], n1 = np[nyq + b] * f[b], P = 0.5f * (n0 + n1), Q = 0.5f * (n0 - n1);
                    const c2 F = exch[b][(m * T + q) * 64 + lane], F1 = exch[b][i1 * 64 + l1];
                    re += P * F.x + Q * F1.x;
                    im += P * F.y - Q * F1.y;
                }
                v[m * T + q] = make_float2(re, im);
            }
    }
    __syncthreads();
    fft_inv<GX>(v, w, ex, t);
#pragma unroll
    for (int q = 0; q < R / 2; ++q) {
        const uint32_t x = t + T * q;
        if (x < a.lx) sp[(size_t)x * M] = v[q];
    }
}

// One axis of the kernel's transform, FP64: in [6][a][len][b] -> out [6][a][K][b], components
// even in the axis as N(0) + 2 sum_r N(r) cos(2 pi k r / G), odd ones as 2 sum_r N(r) sin.
__global__ __launch_bounds__(kTPB) void k_conv_axis(uint32_t na, uint32_t len, uint32_t nb, uint32_t K, uint32_t G,
                                                    uint32_t odd, const double2* __restrict__ cs,
                                                    const double* __restrict__ in, double* __restrict__ out) {
    const size_t e = (size_t)blockIdx.x * kTPB + threadIdx.x;
    if (e >= (size_t)6 * na * K * nb) return;
    const uint32_t b = (uint32_t)(e % nb), k = (uint32_t)(e / nb % K);
    const size_t ca = e / nb / K;  // component, a
    const bool o = (odd >> (uint32_t)(ca / na)) & 1u;
    const double* const p = in + ca * len * nb + b;
    double s = 0.0;
    uint32_t m = 0;
    for (uint32_t r = 0; r < len; ++r) {
        const double2 w = cs[m];
        s += p[(size_t)r * nb] * (r == 0 ? (o ? 0.0 : 1.0) : 2.0 * (o ? w.y : w.x));
        m += k;
        if (m >= G) m -= G;
    }
    out[e] = s;
}

// [6][kx][ky][kz] -> [kx][kz][ky][3][3] in FP32; the off-diagonal components are odd in two
// axes: (-i)^2.
__global__ __launch_bounds__(kTPB) void k_conv_pack(uint32_t nx, uint32_t ny, uint32_t nz, const double* __restrict__ in,
                                                    float* __restrict__ N) {
    const size_t e = (size_t)blockIdx.x * kTPB + threadIdx.x, V = (size_t)nx * ny * nz;
    if (e >= 9 * V) return;
    const uint32_t ab = (uint32_t)(e % 9), i = ab / 3, j = ab % 3;
    const uint32_t lo = i < j ? i : j, hi = i < j ? j : i, q = lo == 0 ? hi : lo + hi + 1;  // xx xy xz yy yz zz
    const size_t g = e / 9;
    const uint32_t ky = (uint32_t)(g % ny), kz = (uint32_t)(g / ny % nz), kx = (uint32_t)(g / ny / nz);
    const double v = in[q * V + ((size_t)kx * ny + ky) * nz + kz];
    N[e] = (float)(i != j ? -v : v);
}

uint32_t pow2_pad(uint32_t l) {
    uint32_t g = 16;
    while (g < 2 * l) g *= 2;
    return g;
}

// Octants by geometry: replicas of one film share them.
struct ConvKey {
    int device;
    uint32_t l[3];
    double h[3];
    bool operator<(const ConvKey& o) const { return std::memcmp(this, &o, sizeof(ConvKey)) < 0; }
};
std::mutex g_conv_mu;
std::map<ConvKey, std::weak_ptr<DevBuf>> g_conv_cache;

int conv_upload(DevBuf& b, const void* src, size_t bytes) {
    SLLG_TRY(b.alloc(bytes));
    SLLG_HIP(hipMemcpy(b.p, src, bytes, hipMemcpyHostToDevice));
    return 0;
}

// exp(-2 pi i m / g), m < count
int conv_twiddles(DevBuf& b, uint32_t g) {
    std::vector<float2> tw(g);
    for (uint32_t m = 0; m < g; ++m) {
        const double ang = -2.0 * M_PI * (double)m / (double)g;
        tw[m] = make_float2((float)std::cos(ang), (float)std::sin(ang));
    }
    return conv_upload(b, tw.data(), tw.size() * sizeof(float2));
}

// real[6][x][y][z] (octant) -> N
int conv_kernel(const ConvPlan& p, const std::vector<double>& real, DevBuf& N) {
    const uint32_t l[3] = {p.l[0], p.l[1], p.l[2]}, G[3] = {p.gx, p.gy, 2 * p.l[2]};
    const uint32_t K[3] = {G[0] / 2 + 1, G[1] / 2 + 1, l[2] + 1};
    // components xx xy xz yy yz zz odd in x: xy, xz; in y: xy, yz; in z: xz, yz
    const uint32_t odd[3] = {0x06u, 0x12u, 0x14u};
    DevBuf cur, cs;
    SLLG_TRY(conv_upload(cur, real.data(), real.size() * sizeof(double)));
    for (int d = 2; d >= 0; --d) {
        std::vector<double2> t(G[d]);
        for (uint32_t m = 0; m < G[d]; ++m) {
            const double ang = 2.0 * M_PI * (double)m / (double)G[d];
            t[m] = make_double2(std::cos(ang), std::sin(ang));
        }
        SLLG_TRY(conv_upload(cs, t.data(), t.size() * sizeof(double2)));
        uint32_t na = 1, nb = 1;
        for (int a = 0; a < d; ++a) na *= l[a];
        for (int a = d + 1; a < 3; ++a) nb *= K[a];
        const size_t total = (size_t)6 * na * K[d] * nb;
        DevBuf out;
        SLLG_TRY(out.alloc(total * sizeof(double)));
        k_conv_axis<<<blocks_for(total, kTPB), kTPB>>>(na, l[d], nb, K[d], G[d], odd[d], cs.as<double2>(),
                                                       cur.as<double>(), out.as<double>());
        SLLG_HIP(hipGetLastError());
        SLLG_HIP(hipDeviceSynchronize());
        cur = std::move(out);
    }
    const size_t total = (size_t)9 * K[0] * K[1] * K[2];
    SLLG_TRY(N.alloc(total * sizeof(float)));
    k_conv_pack<<<blocks_for(total, kTPB), kTPB>>>(K[0], K[1], K[2], cur.as<double>(), N.as<float>());
    SLLG_HIP(hipGetLastError());
    SLLG_HIP(hipDeviceSynchronize());
    return 0;
}

// N_ab of the exchange list at d >= 0 per axis, added to the octant; false when the list is
// not mirror-symmetric with symmetric tensors.
bool add_exchange(const ConvPlan& p, const llg_fftexch& fx, double mu, std::vector<double>* real) {
    struct Less {
        bool operator()(const std::array<int, 3>& a, const std::array<int, 3>& b) const { return a < b; }
    };
    std::map<std::array<int, 3>, std::array<double, 9>, Less> at;
    for (uint32_t q = 0; q < fx.n_int; ++q) {
        const llg_fft_interaction& it = fx.ints[q];
        bool far = false;  // never joins two spins of the system
        for (int a = 0; a < 3; ++a) far = far || std::abs((int64_t)it.d[a]) >= (int64_t)p.l[a];
        if (far) continue;
        // neighbour at mesh(i) + d: the convolution index is -d
        auto& v = at.emplace(std::array<int, 3>{-it.d[0], -it.d[1], -it.d[2]}, std::array<double, 9>{}).first->second;
        for (int ab = 0; ab < 9; ++ab) v[ab] += it.J[ab] * (1.0 / (mu * LLG_MU_B));
    }
    for (const auto& e : at) {
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 3; ++b)
                if (e.second[a * 3 + b] != e.second[b * 3 + a]) return false;
        for (int d = 0; d < 3; ++d) {
            std::array<int, 3> r = e.first;
            r[d] = -r[d];
            const auto m = at.find(r);
            if (m == at.end()) return false;
            for (int a = 0; a < 3; ++a)
                for (int b = 0; b < 3; ++b) {
                    const double v = e.second[a * 3 + b];
                    if (m->second[a * 3 + b] != (((a == d) != (b == d)) ? -v : v)) return false;
                }
        }
    }
    if (!real) return true;
    const int pairs[6] = {0, 1, 2, 4, 5, 8};
    const size_t V = (size_t)p.l[0] * p.l[1] * p.l[2];
    for (const auto& e : at)
        if (e.first[0] >= 0 && e.first[1] >= 0 && e.first[2] >= 0) {
            const size_t g = ((size_t)e.first[0] * p.l[1] + e.first[1]) * p.l[2] + e.first[2];
            for (int q = 0; q < 6; ++q) (*real)[q * V + g] += e.second[pairs[q]];
        }
    return true;
}

// Dipolar octant, the reference's expression (src/intmat.cpp:263-331) times m.
void add_dipolar(const ConvPlan& p, const double h[3], double m, std::vector<double>& real) {
    const int pairs[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    const size_t V = (size_t)p.l[0] * p.l[1] * p.l[2];
    size_t g = 0;
    for (uint32_t i = 0; i < p.l[0]; ++i)
        for (uint32_t j = 0; j < p.l[1]; ++j)
            for (uint32_t k = 0; k < p.l[2]; ++k, ++g) {
                if (g == 0) continue;
                const double r[3] = {i * h[0], j * h[1], k * h[2]};
                const double mr = std::sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
                const double oo = 1. / (mr * mr * mr);
                const double e[3] = {r[0] / mr, r[1] / mr, r[2] / mr};
                for (int q = 0; q < 6; ++q) {
                    const int a = pairs[q][0], b = pairs[q][1];
                    real[q * V + g] += 1e-7 * ((3.0 * e[a] * e[b]) - (a == b ? 1.0 : 0.0)) * oo * m;
                }
            }
}

// Dynamic LDS of the plane kernels with nw waves; waves: as many as the plane's sequences
// need, within 64 KB.
template <int GY>
size_t plane_lds(bool fwd, uint32_t nw, uint32_t lz) {
    const size_t ex = (size_t)nw * fft_cols(GY) * fft_lds(GY) * sizeof(c2), P = (size_t)(GY / 2) * (lz + 1) * 4;
    const size_t zt = (size_t)lz * lz * sizeof(c2);
    return zt + (fwd ? ex + P : std::max(ex, P) + (size_t)lz * (GY / 2) * sizeof(c2));
}
template <int GY>
uint32_t plane_waves(bool fwd, uint32_t lz) {
    uint32_t nw = std::min<uint32_t>(kConvWaves, (lz + fft_cols(GY) - 1) / fft_cols(GY));
    while (nw > 1 && plane_lds<GY>(fwd, nw, lz) > 64 * 1024) --nw;
    return nw;
}

template <int GY>
void launch_plane(bool fwd, const ConvArgs& a, const float* S, float scale, float* H, hipStream_t s) {
    const uint32_t nw = plane_waves<GY>(fwd, a.lz);
    const size_t lds = plane_lds<GY>(fwd, nw, a.lz);
    if (fwd)
        k_conv_fwd<GY><<<3 * a.lx, nw * 64, lds, s>>>(a, S);
    else
        k_conv_inv<GY><<<3 * a.lx, kConvWaves * 64, lds, s>>>(a, nw, scale, H);
}

template <int GX>
void launch_x(const ConvArgs& a, uint32_t gy, hipStream_t s) {
    k_conv_x<GX><<<a.lz * gy / fft_cols(GX), 192, 0, s>>>(a, gy);
}

}  // namespace

// Extents of at least 4 along x and y keep the padded spectrum and octant within what the
// unpadded whole-grid plan holds (the admission estimate); 128 and 32 are what the register
// transforms and 64 KB of LDS hold.
bool conv_applies(const llg_ctx* c, const llg_dipolar& d, const llg_fftexch* fx) {
    if (c->prec == LLG_FP64_PLAIN || (c->flags & LLG_FLAG_DIPOLAR_FULL_FFT)) return false;
    ConvPlan p;
    for (int a = 0; a < 3; ++a) {
        const uint64_t l = (uint64_t)d.dim[a] * d.nk[a];
        if (l == 0 || l > (a == 2 ? 32u : 128u) || (a < 2 && l < 4)) return false;
        p.l[a] = (uint32_t)l;
    }
    return !fx || (c->ns == 1 && add_exchange(p, *fx, c->mu_sp[0], nullptr));
}

int conv_create(llg_ctx* c, ConvPlan& p, const llg_dipolar& d, const uint32_t* spin_species, const llg_fftexch* fx,
                bool dip_terms) {
    for (int a = 0; a < 3; ++a) p.l[a] = d.dim[a] * d.nk[a];
    p.gx = pow2_pad(p.l[0]);
    p.gy = pow2_pad(p.l[1]);
    const uint32_t n = c->n, lz = p.l[2];
    std::vector<uint32_t> map((size_t)p.l[0] * p.l[1] * lz, 0xFFFFFFFFu);
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t* m = d.mesh + 3 * (size_t)i;
        for (int a = 0; a < 3; ++a)
            if (m[a] >= p.l[a]) SLLG_FAIL(LLG_E_INVALID, "mesh coordinate of spin %u outside dim*nk", i);
        uint32_t& q = map[((size_t)m[0] * p.l[1] + m[1]) * lz + m[2]];
        if (q != 0xFFFFFFFFu) {
            if (fx) SLLG_FAIL(LLG_E_INVALID, "two spins of species 0 share a mesh point (spin %u)", i);
            SLLG_FAIL(LLG_E_INVALID, "two spins share a mesh point (spin %u)", i);
        }
        q = c->perm.to_dev(i);
    }
    p.dense = (size_t)n == map.size();
    for (size_t e = 0; p.dense && e < map.size(); ++e) p.dense = map[e] == (uint32_t)e;
    if (!p.dense) SLLG_TRY(conv_upload(p.map, map.data(), map.size() * sizeof(uint32_t)));
    if (!fx) {
        std::vector<float> mu(n);
        for (uint32_t i = 0; i < n; ++i)
            mu[c->perm.to_dev(i)] = (float)c->mu_sp[spin_species ? spin_species[i] : (i % c->ns)];
        SLLG_TRY(conv_upload(p.mu, mu.data(), n * sizeof(float)));
    }
    SLLG_TRY(conv_twiddles(p.twx, p.gx));
    SLLG_TRY(conv_twiddles(p.twy, p.gy));
    std::vector<float2> zt((size_t)lz * lz);
    for (uint32_t s = 0; s < lz; ++s)
        for (uint32_t z = 0; z < lz; ++z) {
            const double ang = -2.0 * M_PI * (double)((s * z) % (2 * lz)) / (double)(2 * lz);
            zt[s * lz + z] = s == 0 ? make_float2(1.f, (z & 1u) ? -1.f : 1.f)
                                    : make_float2((float)std::cos(ang), (float)std::sin(ang));
        }
    SLLG_TRY(conv_upload(p.zt, zt.data(), zt.size() * sizeof(float2)));
    SLLG_TRY(p.spec.alloc((size_t)3 * p.l[0] * lz * p.gy * sizeof(float2)));
    ConvKey key;
    std::memset(&key, 0, sizeof key);
    key.device = c->device;
    for (int a = 0; a < 3; ++a) {
        key.l[a] = p.l[a];
        key.h[a] = d.abc[a] / (double)d.nk[a];
    }
    if (!fx) {
        std::lock_guard<std::mutex> lk(g_conv_mu);
        const auto it = g_conv_cache.find(key);
        if (it != g_conv_cache.end()) p.N = it->second.lock();
    }
    if (!p.N) {
        std::vector<double> real((size_t)6 * map.size(), 0.0);
        if (fx) add_exchange(p, *fx, c->mu_sp[0], &real);
        if (!fx || dip_terms) add_dipolar(p, key.h, fx ? c->mu_sp[0] * LLG_MU_B : LLG_MU_B, real);
        p.N = std::make_shared<DevBuf>();
        SLLG_TRY(conv_kernel(p, real, *p.N));
        if (!fx) {
            std::lock_guard<std::mutex> lk(g_conv_mu);
            g_conv_cache[key] = p.N;
        }
    }
    return 0;
}

int conv_apply(llg_ctx* c, const ConvPlan& p, const float* S, bool aos3, float* H) {
    ConvArgs a;
    a.n = c->n;
    a.lx = p.l[0];
    a.ly = p.l[1];
    a.lz = p.l[2];
    a.dense = p.dense ? 1u : 0u;
    a.si = aos3 ? 3u : 1u;
    a.sc = aos3 ? 1u : c->n;
    a.map = p.map.as<uint32_t>();
    a.mu = p.mu.as<float>();
    a.twx = p.twx.as<c2>();
    a.twy = p.twy.as<c2>();
    a.zt = p.zt.as<c2>();
    a.N = p.N->as<float>();
    a.spec = p.spec.as<c2>();
    const float scale = (float)(1.0 / ((double)p.gx * p.gy * (2.0 * p.l[2])));
#define SLLG_CONV(G_, L_) \
    case G_: L_; break;
#define SLLG_PLANE(F_)                                                                                             \
    switch (p.gy) {                                                                                                \
        SLLG_CONV(16, launch_plane<16>(F_, a, S, scale, H, c->stream))                                             \
        SLLG_CONV(32, launch_plane<32>(F_, a, S, scale, H, c->stream))                                             \
        SLLG_CONV(64, launch_plane<64>(F_, a, S, scale, H, c->stream))                                             \
        SLLG_CONV(128, launch_plane<128>(F_, a, S, scale, H, c->stream))                                           \
        default: launch_plane<256>(F_, a, S, scale, H, c->stream);                                                 \
    }
    SLLG_PLANE(true)
    SLLG_HIP(hipGetLastError());
    switch (p.gx) {
        SLLG_CONV(16, launch_x<16>(a, p.gy, c->stream))
        SLLG_CONV(32, launch_x<32>(a, p.gy, c->stream))
        SLLG_CONV(64, launch_x<64>(a, p.gy, c->stream))
        SLLG_CONV(128, launch_x<128>(a, p.gy, c->stream))
        default: launch_x<256>(a, p.gy, c->stream);
    }
    SLLG_HIP(hipGetLastError());
    SLLG_PLANE(false)
#undef SLLG_PLANE
#undef SLLG_CONV
    SLLG_HIP(hipGetLastError());
    return 0;
}

}  // namespace sllg
