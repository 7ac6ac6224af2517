// k_block.hip - Heun half steps of packed encodings whose rows are whole periodic lattice lines
// (any line length), neighbours read from LDS.
//
// The packed reader gathers every neighbour on its own, and a 12-byte gather costs a CU 17 to 19
// cycles whatever its addresses: 42 of them a row are half of its time.  Here a workgroup takes
// a few consecutive lines of every sublattice (build_blocks, encode.hip), stages the lines they
// couple to once in LDS, each with the cells that wrap around its ends, and reads neighbours
// from there (which of the readers a new handle takes: blocks_pay, encode.hip).  In the staged layout an entry's neighbour is the same number of bytes away from
// every row of the workgroup's sublattice, so the entry stream is lane-uniform (scalar loads:
// offset and couplings of four entries a record) where the packed reader loads a word a lane.
// Rows keep their entries' order, so the sums have the packed reader's bits.
//
// us a step (two half steps), packed entries and line blocks, 300 K: fcc, 42 entries, 37 x 45 x 51
// cells 30.7 and 19.8, 59^3 53.4 and 33.0, 20^3 13.1 and 10.4; fcc, 12 entries, 37 x 45 x 51 18.9 and
// 14.0; simple cubic, 56 entries, 60 x 61 x 62 25.2 and 19.4; bct, 8 entries, 50 x 51 x 52 13.6 and
// 11.9.  What is left: the staging loads (every line is fetched by some nine workgroups), the LDS
// reads (two instructions an entry) and the arithmetic follow each other in waves that start
// together, 8 to 32 a CU.
#include <type_traits>

#include "fused.hpp"

namespace sllg {

template <int NC>
struct BlockRecW {  // four entries: LDS byte offsets, then couplings [entry][component]
    static constexpr int W = block_words(NC);
    uint32_t w[W];
};

// Row, own LDS position and stream of a lane.  Lanes past the workgroup's lines repeat its last
// row (the whole wave stays in uniform control flow) and store nothing.
struct BlockRow {
    const uint32_t* ts;
    uint32_t k, lane, t, i, iref, own, nstaged;
    bool live;
};

__device__ __forceinline__ BlockRow block_row(const FusedArgs& a) {
    BlockRow r;
    const uint32_t Z = a.ex.tlps, ws = a.ex.tnw, P = Z + 2u * a.ex.tumax;
    const u32x4 hd = cview(reinterpret_cast<const u32x4*>(a.ex.tgrp))[tile_index(a.xcd)];
    r.ts = a.ex.tent + hd.x;
    r.nstaged = hd.w;
    r.k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    r.lane = threadIdx.x & 63u;
    uint32_t t = 0, k = r.k;
    for (; k >= ws; k -= ws) ++t;
    r.t = t;
    uint32_t p = k * 64u + r.lane;
    const uint32_t last = hd.z * Z - 1u;
    r.live = p <= last;
    p = min(p, last);
    const uint32_t j = (p * r.ts[0]) >> 20;  // line of the workgroup: p / Z
    const uint32_t cell = hd.y * Z + p;
    r.i = t * a.perm.ncell + cell;
    r.iref = cell * a.perm.na + t;
    r.own = r.ts[4 + t] + (j * P + (p - j * Z)) * 12u;
    return r;
}

// The staged lines, [line][cell -H .. Z + H) of 12 bytes.  Lines of at most 32 staged cells: as
// many to a wave load as fit its 64 lanes, four loads in flight; longer ones: a load per line and
// 64 cells with the line's first row in a scalar, eight in flight where that adds no load past the
// list (59^3 fcc cells, 8 lines a wave: 32.9 us a step, 34.7 with four; 40 x 40 x 80, 4 lines:
// 35.1 with eight, 30.5 with four).  One run of cells over all lines (full loads, a row looked up
// by every lane) took 20.5 us a step where this takes 19.5, 37 x 45 x 51 cells, and 26.5 where it
// takes 27.9, 60 x 60 x 33; wrapped cells copied at the LDS store instead of loaded 22.2 for the first.
// Loads past the list or a line's end repeat the last of it (the same value to the same place), so
// that the waves stay out of divergent control flow.
__device__ __forceinline__ void block_stage(const FusedArgs& a, const BlockRow& r, const float* __restrict__ src,
                                            char* lds) {
    const SpinBuf sb = spin_buf(src, a.n);
    const uint32_t nw = blockDim.x >> 6, Z = a.ex.tlps, H = a.ex.tumax, P = Z + 2u * H;
    const uint32_t* __restrict__ ls = r.ts + kBlockHead;
    auto cell_of = [&](uint32_t zz) -> uint32_t {  // cell of the line at staged position zz
        int w = (int)zz - (int)H;
        w += w < 0 ? (int)Z : 0;
        w -= w >= (int)Z ? (int)Z : 0;
        return (uint32_t)w;
    };
    auto put = [&](uint32_t line, uint32_t zz, const auto& v) {
        float* d = reinterpret_cast<float*>(lds + (line * P + zz) * 12u);
        d[0] = __uint_as_float(v[0]);
        d[1] = __uint_as_float(v[1]);
        d[2] = __uint_as_float(v[2]);
    };
    using V3 = decltype(__builtin_amdgcn_raw_buffer_load_b96(sb.r, 0, 0, 0));
    const uint32_t last = r.nstaged - 1u;
    if (P <= 32u) {
        const uint32_t per = r.ts[2], sub = min((r.lane * r.ts[1]) >> 20, per - 1u), zz = min(r.lane - sub * P, P - 1u);
        const uint32_t vo = cell_of(zz) * 12u;
#pragma unroll 1
        for (uint32_t l0 = r.k * per; l0 <= last; l0 += 4u * nw * per) {
            uint32_t row[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) row[u] = gview(ls)[min(l0 + u * nw * per + sub, last)];
            V3 v[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[u] = __builtin_amdgcn_raw_buffer_load_b96(sb.r, row[u] * 12u + vo, 0, 0);
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) put(min(l0 + u * nw * per + sub, last), zz, v[u]);
        }
        return;
    }
#pragma unroll 1
    for (uint32_t z0 = 0; z0 < P; z0 += 64u) {
        const uint32_t zz = min(z0 + r.lane, P - 1u), vo = cell_of(zz) * 12u;
        auto run = [&](auto depth) {
            constexpr uint32_t D = decltype(depth)::value;
#pragma unroll 1
            for (uint32_t l0 = r.k; l0 <= last; l0 += D * nw) {
                V3 v[D];
#pragma unroll
                for (uint32_t u = 0; u < D; ++u)
                    v[u] = __builtin_amdgcn_raw_buffer_load_b96(
                        sb.r, vo, __builtin_amdgcn_readfirstlane(ls[min(l0 + u * nw, last)]) * 12u, 0);
#pragma unroll
                for (uint32_t u = 0; u < D; ++u) put(min(l0 + u * nw, last), zz, v[u]);
            }
        };
        if ((last / nw / 4u) & 1u)  // an even number of fours
            run(std::integral_constant<uint32_t, 8>());
        else
            run(std::integral_constant<uint32_t, 4>());
    }
}

// Pair exchange from LDS, a record ahead (the stream ends with a spare record).
template <int NC>
__device__ __forceinline__ void block_exch(const BlockRow& r, const char* own, float dot[3]) {
    using RW = BlockRecW<NC>;
    const uint32_t* __restrict__ rp = r.ts + (int)__builtin_amdgcn_readfirstlane(r.ts[12 + r.t]);
    const uint32_t nq = __builtin_amdgcn_readfirstlane(r.ts[20 + r.t]);
    dot[0] = dot[1] = dot[2] = 0.0f;
    auto four = [&](const RW& c) {
        Spin3 s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) s[u] = *reinterpret_cast<const Spin3*>(own + (int)c.w[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float v[NC];
#pragma unroll
            for (int k = 0; k < NC; ++k) v[k] = __uint_as_float(c.w[4 + u * NC + k]);
            const float q[3] = {s[u].x, s[u].y, s[u].z};
            accum<NC, float>(v, q, dot);
        }
    };
    RW c0 = load_rec<RW>(rp);
    uint32_t g = 0;
    for (; g + 1 < nq; g += 2) {
        const RW c1 = load_rec<RW>(rp + (size_t)(g + 1) * RW::W);
        four(c0);
        c0 = load_rec<RW>(rp + (size_t)(g + 2) * RW::W);
        four(c1);
    }
    if (g < nq) four(c0);
}

template <int NC, bool PRED>
__global__ __launch_bounds__(1024) void k_heun_block(FusedArgs a, HeunBufs b) {
    extern __shared__ char bl_lds[];
    const BlockRow r = block_row(a);
    const uint32_t n = a.n, i = r.i;
    Spin3 av{0.f, 0.f, 0.f};
    if constexpr (!PRED) av = reinterpret_cast<const Spin3*>(b.A)[i];  // overlaps the staging loads
    block_stage(a, r, PRED ? b.S3 : b.Y3, bl_lds);
    __syncthreads();
    const Spin3 o = *reinterpret_cast<const Spin3*>(bl_lds + r.own);
    const float s[3] = {o.x, o.y, o.z};
    float h[3], f[3], hd[3] = {0.f, 0.f, 0.f};
    block_exch<NC>(r, bl_lds + r.own, h);
    fused_tail<false>(a, i, r.iref, PRED ? b.S : b.Y, s, h, hd, f, a.t);
    if (!r.live) return;
    if constexpr (PRED) {
        const float y[3] = {s[0] + a.rdt * f[0], s[1] + a.rdt * f[1], s[2] + a.rdt * f[2]};
        const float q = rsqrtf(y[0] * y[0] + y[1] * y[1] + y[2] * y[2]);
        reinterpret_cast<Spin3*>(b.A)[i] =
            Spin3{s[0] + a.half_rdt * f[0], s[1] + a.half_rdt * f[1], s[2] + a.half_rdt * f[2]};
        if (b.Y) {
#pragma unroll
            for (int c = 0; c < 3; ++c) b.Y[(size_t)c * n + i] = y[c] * q;
        }
        reinterpret_cast<Spin3*>(b.Y3)[i] = Spin3{y[0] * q, y[1] * q, y[2] * q};
    } else {
        const float p[3] = {av.x + a.half_rdt * f[0], av.y + a.half_rdt * f[1], av.z + a.half_rdt * f[2]};
        const float q = rsqrtf(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
        if (b.S) {
#pragma unroll
            for (int c = 0; c < 3; ++c) b.S[(size_t)c * n + i] = p[c] * q;
        }
        reinterpret_cast<Spin3*>(b.S3)[i] = Spin3{p[0] * q, p[1] * q, p[2] * q};
    }
}

template <int NC>
static void launch_block_nc(bool pred, const FusedArgs& a, const HeunBufs& b, const ExchStore& x, hipStream_t st) {
    const unsigned threads = 64u * x.blk_waves, lds = x.blk_lds;
    if (pred)
        k_heun_block<NC, true><<<x.blk_wgs, threads, lds, st>>>(a, b);
    else
        k_heun_block<NC, false><<<x.blk_wgs, threads, lds, st>>>(a, b);
}

void launch_block(bool pred, const FusedArgs& a, const HeunBufs& b, const ExchStore& x, hipStream_t st) {
    if (a.ex.ncomp == 1)
        launch_block_nc<1>(pred, a, b, x, st);
    else if (a.ex.ncomp == 3)
        launch_block_nc<3>(pred, a, b, x, st);
    else
        launch_block_nc<9>(pred, a, b, x, st);
}

}  // namespace sllg
