// k_plain.hip - FP64 plain path: FP64 couplings, state and per-spin parameter arrays (SoA),
// one kernel per field evaluation.  Built with -ffp-contract=off; every operation follows the
// order of the FP64 oracle so that both give the same bits.
//
//   plain_exchange   <- cufields::CSpMV_CSR / _OffDiag / CSpMV_DIA / _OffDiag (src/cufields.cu:97-246)
//   normals3_f64     <- curandGenerateNormal (src/cuda.cu:148), replaced by Philox4x32-10 + Box-Muller
//   k_plain_pred     <- exchange at S, noise, cuint::CHeun1 (src/cuint.cu:60-163)
//   k_plain_corr     <- exchange at Y, cuint::CHeun2 (src/cuint.cu:165-242)
//   k_plain_rk       <- exchange, cuintRK4::CdetRK4k1..k4 (src/cuintRK4.cu:62-434),
//                       cuintRK5::CdetRK5k1..k6 (src/cuintRK5.cu:79-628) with textbook stage
//                       inputs, and CdetSnp1 (src/cuintRK4.cu:436-456, src/cuintRK5.cu:630-651)
//
// The reference launches a kernel for the noise, for each SpMV and for each integrator pass,
// with the field in memory between them.  Here a row's field stays in registers: a Heun step
// is two launches instead of five and moves 72 bytes a spin less (the field written and read
// twice, less the draw's); small systems are bound by the launches (32^3 simple cubic, 500 steps:
// 10.1 ms with five launches a step, 6.7 with two).
#include "field.hpp"
#include "kernels.hpp"
#include "philox.hpp"

namespace sllg {

struct PlainArgs {
    uint32_t n;
    double rdt, T;
    double B[3];
    const double* sigma;
    const double* llgpf;
    const double* lambda;
    const double* k1u;
    const double* k1udir;  // SoA 3n
    const double* kc;      // per spin or null
    const double* stg;     // 3n or null
    const double* dem;     // dipolar field, 3n or null
    double* xi;            // 3n or null (T == 0)
    int draw;              // the kernel draws xi of step t (counter noise) and stores it
    Perm perm;             // device row -> reference spin index, which keys the noise
    uint64_t seed, stream, t;
    AnisG<double> an;
    Exch<double> ex;
};

// Exchange sum of row i at spins S (CSR order), plus the dipolar field and the four-spin term:
// H of the reference's SpMV pass.
template <bool UNI, int NC>
__device__ __forceinline__ void plain_exchange(const Exch<double>& e, uint32_t i, const double* __restrict__ S,
                                               const double* __restrict__ dem, double hx[3]) {
    const uint32_t n = e.n;
    double dot[3];
    if constexpr (UNI)
        exch_row_uni<NC>(e, i, S, dot);
    else
        exch_row_ref<NC, double, double, double>(e, i, S, dot);
    for (int a = 0; a < 3; ++a) hx[a] = (dem ? dem[(size_t)a * n + i] : 0.0) + dot[a];
    if (e.fs_xadj) {  // CH += four-spin field (src/cuda.cu:143-146)
        double h4[3];
        fourspin_row<double, double, double>(e, i, S, h4);
        for (int a = 0; a < 3; ++a) hx[a] = hx[a] + h4[a];
    }
}

// Field at spin i (own spin s, exchange+demag hex): h = ((hex + stg) + th) + B, then local terms
// (th = 0 when noise is false: the deterministic field).
__device__ __forceinline__ void plain_field(const PlainArgs& a, uint32_t i, const double s[3], const double hex[3],
                                            double th[3], double h[3], bool noise = true, bool draw = false) {
    const uint32_t n = a.n;
    if (noise && a.xi) {
        double z[3];
        if (draw) {
            normals3_f64(a.seed, a.stream, a.perm.to_ref(i), a.t, z);
            for (int c = 0; c < 3; ++c) a.xi[(size_t)c * n + i] = z[c];  // for the later passes of the step
        } else {
            for (int c = 0; c < 3; ++c) z[c] = a.xi[(size_t)c * n + i];
        }
        const double TP = sqrt(a.T) * a.sigma[i];
        for (int c = 0; c < 3; ++c) th[c] = z[c] * TP;
    } else {
        th[0] = th[1] = th[2] = 0.0;
    }
    for (int c = 0; c < 3; ++c) {
        const double st = a.stg ? a.stg[(size_t)c * n + i] : 0.0;
        h[c] = ((hex[c] + st) + th[c]) + a.B[c];
    }
    const double d[3] = {a.k1udir[i], a.k1udir[(size_t)n + i], a.k1udir[2 * (size_t)n + i]};
    local_terms<double>(a.k1u[i], d, a.kc ? a.kc[i] : 0.0, a.an, s, h);
}

template <bool UNI, int NC>
__global__ __launch_bounds__(kTPB) void k_plain_pred(PlainArgs a, const double* __restrict__ S, double* __restrict__ Y,
                                                     double* __restrict__ FN) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    const uint32_t n = a.n;
    if (i >= n) return;
    double hex[3], th[3], h[3], f[3];
    plain_exchange<UNI, NC>(a.ex, i, S, a.dem, hex);
    const double s[3] = {S[i], S[(size_t)n + i], S[2 * (size_t)n + i]};
    plain_field(a, i, s, hex, th, h, true, a.draw);
    llg_rhs<double>(a.llgpf[i], a.lambda[i], s, h, f);
    double es[3], mods = 0.0;
    for (int c = 0; c < 3; ++c) {
        FN[(size_t)c * n + i] = f[c];
        es[c] = s[c] + f[c] * a.rdt;
        mods += es[c] * es[c];
    }
    const double nrm = sqrt(mods);
    for (int c = 0; c < 3; ++c) Y[(size_t)c * n + i] = es[c] / nrm;
}

template <bool UNI, int NC>
__global__ __launch_bounds__(kTPB) void k_plain_corr(PlainArgs a, const double* __restrict__ Y, double* __restrict__ S,
                                                     const double* __restrict__ FN, double* __restrict__ DET) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    const uint32_t n = a.n;
    if (i >= n) return;
    double hex[3], th[3], h[3], f[3];
    plain_exchange<UNI, NC>(a.ex, i, Y, a.dem, hex);
    const double s[3] = {Y[i], Y[(size_t)n + i], Y[2 * (size_t)n + i]};
    plain_field(a, i, s, hex, th, h);
    llg_rhs<double>(a.llgpf[i], a.lambda[i], s, h, f);
    double ps[3] = {S[i], S[(size_t)n + i], S[2 * (size_t)n + i]};
    double mods = 0.0;
    for (int c = 0; c < 3; ++c) {
        ps[c] += (0.5 * (FN[(size_t)c * n + i] + f[c]) * a.rdt);
        mods += ps[c] * ps[c];
    }
    const double nrm = sqrt(mods);
    for (int c = 0; c < 3; ++c) {
        S[(size_t)c * n + i] = ps[c] / nrm;
        DET[(size_t)c * n + i] = h[c] - th[c];
    }
}

// RK stage m: k_m = rdt f(Y_m) into K[m]; then the next stage input:
// RK4: Y = S + a_m k_m (a = 1/2, 1/2, 1); Cash-Karp: Y = (((S + b_{m+1,0} k_0) + ...) + b_{m+1,m} k_m).
// The last stage combines instead: S = N(S + sum_m w_m k_m).  Stage inputs alternate between
// two buffers, since neighbouring rows still read the input of this stage.
struct RkTab {
    double b[6][5];
};
__constant__ RkTab c_rk5;

struct RkBufs {
    const double* in;
    double* out;
    double* S;
    double* K[5];
};

template <bool UNI, int NC, int SCHEME>
__global__ __launch_bounds__(kTPB) void k_plain_rk(PlainArgs a, RkBufs r, int m) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    const uint32_t n = a.n;
    if (i >= n) return;
    double hex[3], th[3], h[3], f[3], ls[3];
    plain_exchange<UNI, NC>(a.ex, i, r.in, a.dem, hex);
    const double s[3] = {r.in[i], r.in[(size_t)n + i], r.in[2 * (size_t)n + i]};
    plain_field(a, i, s, hex, th, h, true, a.draw && m == 0);
    llg_rhs<double>(a.llgpf[i], a.lambda[i], s, h, f);
    constexpr int last = SCHEME == LLG_RK4 ? 3 : 5;
    double mods = 0.0;
    for (int c = 0; c < 3; ++c) {
        const size_t o = (size_t)c * n + i;
        const double k = a.rdt * f[c];
        if (m < last) {
            r.K[m][o] = k;
            if constexpr (SCHEME == LLG_RK4) {
                const double am = (m == 2) ? 1.0 : 0.5;
                r.out[o] = r.S[o] + am * k;
            } else {
                double v = r.S[o];
                for (int j = 0; j < m; ++j) v = v + c_rk5.b[m + 1][j] * r.K[j][o];
                r.out[o] = v + c_rk5.b[m + 1][m] * k;
            }
        } else if constexpr (SCHEME == LLG_RK4) {
            const double onesixth = 1.0 / 6.0, onethird = 1.0 / 3.0;
            ls[c] = r.S[o] + r.K[0][o] * onesixth + r.K[1][o] * onethird + r.K[2][o] * onethird + k * onesixth;
            mods += ls[c] * ls[c];
        } else {
            double v = r.S[o];
            v = v + r.K[0][o] * (37.0 / 378.0);
            v = v + r.K[2][o] * (250.0 / 621.0);
            v = v + r.K[3][o] * (125.0 / 594.0);
            ls[c] = v + k * (512.0 / 1771.0);
            mods += ls[c] * ls[c];
        }
    }
    if (m == last) {
        const double nrm = sqrt(mods);
        for (int c = 0; c < 3; ++c) r.S[(size_t)c * n + i] = ls[c] / nrm;
    }
}

// Deterministic field (no thermal part) at spins Sp, FP64 plain layout.
template <bool UNI, int NC>
__global__ __launch_bounds__(kTPB) void k_plain_detfield(PlainArgs a, const double* __restrict__ Sp,
                                                         double* __restrict__ out) {
    const uint32_t i = blockIdx.x * kTPB + threadIdx.x;
    const uint32_t n = a.n;
    if (i >= n) return;
    double hex[3], th[3], h[3];
    plain_exchange<UNI, NC>(a.ex, i, Sp, a.dem, hex);
    const double s[3] = {Sp[i], Sp[(size_t)n + i], Sp[2 * (size_t)n + i]};
    plain_field(a, i, s, hex, th, h, false);
    for (int c = 0; c < 3; ++c) out[(size_t)c * n + i] = h[c];
}

// ---------------------------------------------------------------- host launchers

static PlainArgs plain_args(const llg_ctx* c, bool with_noise, uint64_t t) {
    PlainArgs a;
    a.n = c->n;
    a.rdt = c->rdt;
    a.T = c->T;
    for (int k = 0; k < 3; ++k) a.B[k] = c->B[k];
    a.sigma = c->p_sigma.as<double>();
    a.llgpf = c->p_llgpf.as<double>();
    a.lambda = c->p_lambda.as<double>();
    a.k1u = c->p_k1u.as<double>();
    a.k1udir = c->p_k1udir.as<double>();
    a.kc = c->p_kc.as<double>();
    a.stg = c->stag_set ? c->STG.as<double>() : nullptr;
    a.dem = c->dip ? c->DEM.as<double>() : nullptr;
    a.xi = (with_noise && c->T > 0.0) ? c->XI.as<double>() : nullptr;
    a.draw = c->noise_mode == LLG_NOISE_COUNTER;
    a.perm = c->perm;
    a.seed = c->seed;
    a.stream = c->stream_id;
    a.t = t;
    a.an = c->an64;
    a.ex = c->ex64;
    return a;
}

#define SLLG_PLAIN(EX, MACRO)                                  \
    do {                                                       \
        const bool uni_ = (EX).fmt == FMT_UNI;                 \
        if ((EX).ncomp == 1) {                                 \
            if (uni_) { MACRO(true, 1); } else { MACRO(false, 1); } \
        } else if ((EX).ncomp == 3) {                          \
            if (uni_) { MACRO(true, 3); } else { MACRO(false, 3); } \
        } else {                                               \
            if (uni_) { MACRO(true, 9); } else { MACRO(false, 9); } \
        }                                                      \
    } while (0)

// Predictor of step t: the exchange at S, the step's noise (drawn here in counter mode), Y and f(S).
int plain_heun_pred(llg_ctx* c, uint64_t t) {
    const PlainArgs a = plain_args(c, true, t);
    const dim3 g(blocks_for(c->n, kTPB)), b(kTPB);
#define SLLG_L(U, N) k_plain_pred<U, N><<<g, b, 0, c->stream>>>(a, c->S.as<double>(), c->Y.as<double>(), c->FN.as<double>())
    SLLG_PLAIN(a.ex, SLLG_L);
#undef SLLG_L
    SLLG_HIP(hipGetLastError());
    return 0;
}

int plain_heun_corr(llg_ctx* c, uint64_t t) {
    const PlainArgs a = plain_args(c, true, t);
    const dim3 g(blocks_for(c->n, kTPB)), b(kTPB);
#define SLLG_L(U, N)                                                                                      \
    k_plain_corr<U, N><<<g, b, 0, c->stream>>>(a, c->Y.as<double>(), c->S.as<double>(), c->FN.as<double>(), \
                                            c->DET.as<double>())
    SLLG_PLAIN(a.ex, SLLG_L);
#undef SLLG_L
    SLLG_HIP(hipGetLastError());
    return 0;
}

int plain_rk_init_tables() {
    static bool done = false;
    if (done) return 0;
    RkTab t{};
    const double b2[1] = {0.2};
    const double b3[2] = {3.0 / 40.0, 9.0 / 40.0};
    const double b4[3] = {0.3, -0.9, 1.2};
    const double b5[4] = {-11.0 / 54.0, 2.5, -70.0 / 27.0, 35.0 / 27.0};
    const double b6[5] = {1631.0 / 55296.0, 175.0 / 512.0, 575.0 / 13824.0, 44275.0 / 110592.0, 253.0 / 4096.0};
    const double* rows[6] = {nullptr, b2, b3, b4, b5, b6};
    for (int m = 1; m < 6; ++m)
        for (int j = 0; j < m; ++j) t.b[m][j] = rows[m][j];
    SLLG_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_rk5), &t, sizeof(t)));
    done = true;
    return 0;
}

// Stage m of a Runge-Kutta step: its input is S (m = 0), then Y and H in turn.
double* plain_rk_input(const llg_ctx* c, int m) {
    return m == 0 ? c->S.as<double>() : ((m & 1) ? c->Y.as<double>() : c->H.as<double>());
}

int plain_rk_stage(llg_ctx* c, uint64_t t, int m) {
    const PlainArgs a = plain_args(c, true, t);
    const dim3 g(blocks_for(c->n, kTPB)), b(kTPB);
    RkBufs r;
    r.in = plain_rk_input(c, m);
    r.out = plain_rk_input(c, m + 1);
    r.S = c->S.as<double>();
    for (int k = 0; k < 5; ++k) r.K[k] = c->K[k].as<double>();
#define SLLG_L(U, N)                                                                      \
    do {                                                                               \
        if (c->scheme == LLG_RK4) k_plain_rk<U, N, LLG_RK4><<<g, b, 0, c->stream>>>(a, r, m); \
        else k_plain_rk<U, N, LLG_RK5><<<g, b, 0, c->stream>>>(a, r, m);                  \
    } while (0)
    SLLG_PLAIN(a.ex, SLLG_L);
#undef SLLG_L
    SLLG_HIP(hipGetLastError());
    return 0;
}

int plain_detfield(llg_ctx* c, const double* Sp, double* out) {
    const PlainArgs a = plain_args(c, false, 0);
#define SLLG_L(U, N) k_plain_detfield<U, N><<<blocks_for(c->n, kTPB), kTPB, 0, c->stream>>>(a, Sp, out)
    SLLG_PLAIN(a.ex, SLLG_L);
#undef SLLG_L
    SLLG_HIP(hipGetLastError());
    return 0;
}

// Staggered-field ramp on the device, cufields::CincStagFields (src/cufields.cu:46-56):
// H_stag = r * H0 with H0 the field last given, kept on the device in FP64 (device order,
// SoA).  The product is taken in FP64 and rounded once to the path's precision.
template <class P>
__global__ __launch_bounds__(kTPB) void k_stag_scale(size_t n3, double r, const double* __restrict__ h0,
                                                     P* __restrict__ h) {
    const size_t k = (size_t)blockIdx.x * kTPB + threadIdx.x;
    if (k < n3) h[k] = (P)(r * h0[k]);
}

int stag_scale(llg_ctx* c, double r) {
    const size_t n3 = 3 * (size_t)c->n;
    if (c->prec == LLG_FP64_PLAIN)
        k_stag_scale<double><<<blocks_for(n3, kTPB), kTPB, 0, c->stream>>>(n3, r, c->STG0.as<double>(),
                                                                           c->STG.as<double>());
    else
        k_stag_scale<float><<<blocks_for(n3, kTPB), kTPB, 0, c->stream>>>(n3, r, c->STG0.as<double>(),
                                                                          c->STG.as<float>());
    SLLG_HIP(hipGetLastError());
    return 0;
}

}  // namespace sllg
