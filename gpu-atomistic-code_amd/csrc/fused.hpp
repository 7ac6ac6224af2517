// fused.hpp - what the FP32 Heun kernels share: their arguments, the row a thread takes, the
// thermal field and everything of f(S) after the pair exchange.
#pragma once
#include "field.hpp"
#include "kernels.hpp"
#include "philox.hpp"

namespace sllg {

struct Spin3 {  // one spin of an AoS3 copy
    float x, y, z;
};

// Spins as one raw buffer resource: a neighbour's three components are three buffer loads
// sharing one 32-bit byte offset (scalar component offsets 4n, 8n), so no 64-bit address
// arithmetic per entry; a load outside the 12n bytes returns 0 instead of faulting.
struct SpinBuf {
    __amdgpu_buffer_rsrc_t r;
    uint32_t o1, o2;
};
__device__ __forceinline__ SpinBuf spin_buf(const float* S, uint32_t n) {
    SpinBuf b;
    b.r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(S), 0, (int)(12u * n), 0x00020000);
    b.o1 = 4u * n;
    b.o2 = 8u * n;
    return b;
}

// Coupling record of RW::W words, read with scalar loads by the whole wave.
// Whole 16-byte units, so the record arrives in few wide scalar loads.  CV: through the
// constant view, for kernels whose record loads follow stores, fences or atomics (the
// persistent batched kernel); the per-launch kernels measured slightly faster without it.
template <class RW, bool CV = false>
__device__ __forceinline__ RW load_rec(const uint32_t* __restrict__ p) {
    RW o;
#pragma unroll
    for (int k = 0; k < RW::W / 4; ++k) {
        u32x4 v;
        if constexpr (CV)
            v = cview(reinterpret_cast<const u32x4*>(p))[k];
        else
            v = gview(reinterpret_cast<const u32x4*>(p))[k];
        o.w[4 * k] = v.x;
        o.w[4 * k + 1] = v.y;
        o.w[4 * k + 2] = v.z;
        o.w[4 * k + 3] = v.w;
    }
    return o;
}

struct FusedArgs {
    uint32_t n;
    Perm perm;  // device row -> reference spin index (counter noise is keyed by the latter)
    int noise;  // 0 none (T = 0), 1 counter, 2 injected
    int multi;  // per-spin species index present
    int xcd;    // XCD-aware block remap
    uint32_t il_na;  // > 1: sublattice-interleaved tile order (il_na sublattices of il_cells rows)
    uint32_t il_cells;
    int tile_sub;    // every tile lies in one sublattice block (perm.ncell % blockDim.x == 0)
    int na_sh, ncell_sh;  // log2 of perm.na and perm.ncell when powers of two (shifts), else -1
    float* th_out;   // predictor: store the thermal field it drew (or null)
    const float* th_in;  // corrector: read it instead of drawing again (or null)
    float rdt, half_rdt, sqrtT;
    float B[3];
    uint64_t seed, stream, t;
    const double* xi;
    const float* dem;
    const float* stg;
    const uint8_t* spec;
    const Species<float>* sp;
    Species<float> sp0;
    AnisG<float> an;
    Exch<float> ex;
};

// Block index -> row tile.  Consecutive workgroups are dispatched round-robin over the
// 8 XCDs of the MI355X; the remap gives each XCD a contiguous range of rows so the
// neighbour spins it gathers stay in its own L2.
__device__ __forceinline__ uint32_t tile_index(int xcd) {
    const uint32_t b = blockIdx.x;
    if (!xcd) return b;
    const uint32_t nb = gridDim.x, per = nb >> 3, rem = nb & 7u;
    const uint32_t x = b & 7u, l = b >> 3;
    return x * per + (x < rem ? x : rem) + l;
}

// Row tile of this block in the sublattice-major device order.  With the XCD remap each
// XCD takes a contiguous range of logical tiles; logical tile L is mapped to sublattice
// L % na, cell tile L / na, so an XCD's range covers one cell range of every sublattice and
// the neighbours its rows gather (all sublattices, nearby cells) are fetched into its L2
// once, not once per sublattice.  Requires il_cells % blockDim.x == 0 (checked on the host).
template <int TPB>
__device__ __forceinline__ uint32_t row_tile(const FusedArgs& a) {
    uint32_t L = tile_index(a.xcd);
    if (a.il_na > 1) {
        const uint32_t tps = a.il_cells / TPB;
        if (a.na_sh >= 0)
            L = (L & (a.il_na - 1u)) * tps + (L >> a.na_sh);
        else
            L = (L % a.il_na) * tps + L / a.il_na;
    }
    return L;
}

// Device row of this thread and the reference index that keys its noise.  When a tile
// lies inside one sublattice block, the block's sublattice and first cell are uniform
// (scalar arithmetic once per block) and the lane adds its offset; otherwise the lane
// inverts the permutation itself.
template <int TPB>
__device__ __forceinline__ void row_of_thread(const FusedArgs& a, uint32_t& i, uint32_t& iref) {
    const uint32_t d0 = row_tile<TPB>(a) * TPB;
    i = d0 + threadIdx.x;
    if (a.perm.na <= 1) {
        iref = i;
    } else if (a.tile_sub) {
        const uint32_t t = a.ncell_sh >= 0 ? d0 >> a.ncell_sh : d0 / a.perm.ncell;
        iref = (d0 - t * a.perm.ncell + threadIdx.x) * a.perm.na + t;
    } else {
        iref = a.perm.to_ref(i);
    }
}

// Row in range.  In line mode n is a multiple of 64 and tiles start at multiples of 64, so
// a wave is wholly in or out: the test is made on a wave-uniform value, which keeps the
// line reader out of divergent control flow (its record words stay scalar).
template <int FMT>
__device__ __forceinline__ bool row_live(const FusedArgs& a, uint32_t i) {
    if constexpr (is_line_fmt(FMT))
        return __builtin_amdgcn_readfirstlane(i & ~63u) < a.n;
    else
        return i < a.n;
}

// Species constants of row i: from the kernel arguments (scalar loads) for one species, not
// through a pointer that a per-spin species index would need.
__device__ __forceinline__ Species<float> species_of(const FusedArgs& a, uint32_t i) {
    Species<float> sp = a.sp0;
    if (a.multi) {
        const auto* q = gview(a.sp) + gview(a.spec)[i];
        sp.llgpf = q->llgpf;
        sp.lambda = q->lambda;
        sp.sigma = q->sigma;
        sp.k1u = q->k1u;
        sp.kc = q->kc;
        sp.k1dir[0] = q->k1dir[0];
        sp.k1dir[1] = q->k1dir[1];
        sp.k1dir[2] = q->k1dir[2];
    }
    return sp;
}

// Thermal field of row i at step t (a.noise != 0): counter noise drawn here (and stored for
// the corrector when a.th_out is set) or taken from the predictor (a.th_in), or the injected
// noise of the step.
__device__ __forceinline__ void thermal_field(const FusedArgs& a, uint32_t i, uint32_t iref, const Species<float>& sp,
                                              uint64_t t, float th[3]) {
    const uint32_t n = a.n;
    if (a.noise == 1) {
        if (a.th_in) {
            th[0] = gview(a.th_in)[i];
            th[1] = gview(a.th_in)[n + i];
            th[2] = gview(a.th_in)[2 * (size_t)n + i];
        } else {
            float z[3];
            normals3_f32(a.seed, a.stream, iref, t, z);
            const float TP = a.sqrtT * sp.sigma;
            th[0] = z[0] * TP;
            th[1] = z[1] * TP;
            th[2] = z[2] * TP;
            if (a.th_out) {
                gview(a.th_out)[i] = th[0];
                gview(a.th_out)[n + i] = th[1];
                gview(a.th_out)[2 * (size_t)n + i] = th[2];
            }
        }
    } else {
        const float TP = a.sqrtT * sp.sigma;
        th[0] = (float)gview(a.xi)[i] * TP;
        th[1] = (float)gview(a.xi)[n + i] * TP;
        th[2] = (float)gview(a.xi)[2 * (size_t)n + i] * TP;
    }
}

// Everything of f(S) at row i after the pair exchange h: four-spin term, dipolar field hd
// (already loaded when EDEM), staggered field, thermal field, applied field, anisotropy,
// and the LLG right-hand side.  The thermal field is drawn here, after the exchange: a
// global store (the predictor's hand-off of its draw) before the exchange would make the
// compiler read the read-only coupling streams with vector instead of scalar loads.
// TH: 0 the thermal field is drawn or read here, 1 the same and kept in th, 2 taken from th.
template <bool EDEM, int TH = 0>
__device__ __forceinline__ void fused_tail(const FusedArgs& a, uint32_t i, uint32_t iref, const float* __restrict__ src,
                                           const float s[3], float h[3], float hd[3], float f[3], uint64_t t,
                                           float* keep = nullptr) {
    const uint32_t n = a.n;
    if (a.ex.fs_xadj) {
        float h4[3];
        fourspin_row<float, float, float>(a.ex, i, src, h4);
        h[0] += h4[0];
        h[1] += h4[1];
        h[2] += h4[2];
    }
    if (a.dem) {
        if constexpr (!EDEM) {
            hd[0] = gview(a.dem)[i];
            hd[1] = gview(a.dem)[n + i];
            hd[2] = gview(a.dem)[2 * (size_t)n + i];
        }
        h[0] += hd[0];
        h[1] += hd[1];
        h[2] += hd[2];
    }
    if (a.stg) {
        h[0] += gview(a.stg)[i];
        h[1] += gview(a.stg)[n + i];
        h[2] += gview(a.stg)[2 * (size_t)n + i];
    }
    const Species<float> sp = species_of(a, i);
    if (a.noise) {
        float th[3];
        if constexpr (TH == 2) {
            th[0] = keep[0];
            th[1] = keep[1];
            th[2] = keep[2];
        } else {
            thermal_field(a, i, iref, sp, t, th);
        }
        if constexpr (TH == 1) {
            keep[0] = th[0];
            keep[1] = th[1];
            keep[2] = th[2];
        }
        h[0] += th[0];
        h[1] += th[1];
        h[2] += th[2];
    }
    h[0] += a.B[0];
    h[1] += a.B[1];
    h[2] += a.B[2];
    local_terms<float>(sp.k1u, sp.k1dir, sp.kc, a.an, s, h);
    llg_rhs<float>(sp.llgpf, sp.lambda, s, h, f);
}

// Buffers of a Heun half step.
struct HeunBufs {
    float *S, *S3, *Y, *Y3, *A;
};

// Half step from line blocks (k_block.hip).
void launch_block(bool pred, const FusedArgs& a, const HeunBufs& b, const ExchStore& x, hipStream_t st);

}  // namespace sllg
