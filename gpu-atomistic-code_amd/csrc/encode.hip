// encode.hip - host-side validation of the exchange given in the descriptor and its
// upload in the layout each path reads.
//
// FP64 plain path: CSR as lane-uniform records of 64-row slices where the couplings repeat
// from row to row, else sliced (u32 columns + FP64 values); DIA [ncomp][ndiag][n] and the
// periodic stencil as given.
//
// FP32 path: CSR becomes sliced ELL with 64-row slices (one wavefront) so that every
// load of the coupling stream is a contiguous wave access (1 KB per uint4 load).  When the
// distinct coupling tuples fit the LDS dictionary (kDictLds floats) and every neighbour's
// row offset fits the bits the dictionary index leaves, an entry is one u32: row offset
// << dbits | dictionary index (4 B per nnz; the dictionary is staged in LDS by every
// block), and slices whose entries repeat an earlier slice's are stored once.  Otherwise
// entries are a u32 column plus ncomp FP32 values (M = 4 + 4 ncomp B per nnz).  Rows keep
// their stored order, so the per-row summation order of the reference CSR
// (src/cufields.cu:192-200) is kept.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "kernels.hpp"

namespace sllg {

namespace {

template <class T>
int upload(DevBuf& b, const T* h, size_t count, hipStream_t s) {
    SLLG_TRY(b.alloc(count * sizeof(T)));
    if (count) SLLG_HIP(hipMemcpyAsync(b.p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
    SLLG_HIP(hipStreamSynchronize(s));
    return 0;
}

// The same for a buffer of X, kept on the host while X is encoded away from the device.
template <class T>
int put(ExchStore& X, DevBuf& b, const T* h, size_t count, hipStream_t s) {
    if (!X.host_only) return upload(b, h, count, s);
    const char* p = reinterpret_cast<const char*>(h);
    X.pending.emplace_back(&b, std::vector<char>(p, p + count * sizeof(T)));
    return 0;
}

int validate_and_copy(llg_ctx* c, const llg_exchange& e) {
    ExchStore& X = *c->xs;
    HostExch& h = X.h;
    const uint32_t n = c->n;
    h.fmt = e.format;
    h.ncomp = e.ncomp ? e.ncomp : 1;
    if (h.fmt == LLG_EXCH_NONE) return 0;
    if (h.ncomp != 1 && h.ncomp != 3 && h.ncomp != 9) SLLG_FAIL(LLG_E_INVALID, "exchange ncomp must be 1, 3 or 9");
    const int nc = h.ncomp;
    if (h.fmt == LLG_EXCH_CSR) {
        if (!e.xadj) SLLG_FAIL(LLG_E_INVALID, "CSR exchange without xadj");
        if (e.nnz && (!e.adjncy || !e.csr_vals)) SLLG_FAIL(LLG_E_INVALID, "CSR exchange without adjncy/values");
        if (e.nnz > 0xFFFFFFFFull) SLLG_FAIL(LLG_E_UNSUPPORTED, "nnz above 2^32-1");
        if (e.xadj[0] != 0 || e.xadj[n] != e.nnz)
            SLLG_FAIL(LLG_E_INVALID, "CSR row pointers: xadj[0]=%u xadj[n]=%u nnz=%llu", e.xadj[0], e.xadj[n],
                      (unsigned long long)e.nnz);
        for (uint32_t i = 0; i < n; ++i)
            if (e.xadj[i + 1] < e.xadj[i]) SLLG_FAIL(LLG_E_INVALID, "CSR row pointers decrease at row %u", i);
        for (uint64_t q = 0; q < e.nnz; ++q)
            if (e.adjncy[q] >= n) SLLG_FAIL(LLG_E_INVALID, "CSR column %u out of range at nnz %llu", e.adjncy[q],
                                            (unsigned long long)q);
        h.nnz = e.nnz;
        h.xadj.assign(e.xadj, e.xadj + n + 1);
        h.adj.assign(e.adjncy, e.adjncy + e.nnz);
        h.vals.assign(e.csr_vals, e.csr_vals + (size_t)nc * e.nnz);
    } else if (h.fmt == LLG_EXCH_DIA) {
        if (e.ndiag && (!e.dia_offsets || !e.dia_vals)) SLLG_FAIL(LLG_E_INVALID, "DIA exchange without offsets/values");
        h.ndiag = e.ndiag;
        h.doff.assign(e.dia_offsets, e.dia_offsets + e.ndiag);
        h.vals.assign(e.dia_vals, e.dia_vals + (size_t)nc * e.ndiag * n);
    } else if (h.fmt == LLG_EXCH_STENCIL) {
        if ((uint64_t)e.dims[0] * e.dims[1] * e.dims[2] * e.n_atoms != n || e.n_atoms == 0)
            SLLG_FAIL(LLG_E_INVALID, "stencil dims x n_atoms != n");
        if (e.stencil_k && (!e.stencil_count || !e.stencil_entries || !e.stencil_vals))
            SLLG_FAIL(LLG_E_INVALID, "stencil without counts/entries/values");
        for (int a = 0; a < 3; ++a) { h.dims[a] = e.dims[a]; h.pbc[a] = e.pbc[a] ? 1 : 0; }
        h.na = e.n_atoms;
        h.sk = e.stencil_k;
        h.per_row = e.stencil_vals_per_row ? 1 : 0;
        h.scount.assign(e.stencil_count, e.stencil_count + h.na);
        h.sent.assign(e.stencil_entries, e.stencil_entries + (size_t)h.na * h.sk * 4);
        for (uint32_t t = 0; t < h.na; ++t) {
            if (h.scount[t] > h.sk) SLLG_FAIL(LLG_E_INVALID, "stencil count above stencil_k");
            for (uint32_t q = 0; q < h.scount[t]; ++q) {
                const int32_t* en = &h.sent[((size_t)t * h.sk + q) * 4];
                if (en[3] < 0 || (uint32_t)en[3] >= h.na) SLLG_FAIL(LLG_E_INVALID, "stencil target atom out of range");
                for (int a = 0; a < 3; ++a)
                    if (en[a] <= -(int32_t)h.dims[a] || en[a] >= (int32_t)h.dims[a])
                        SLLG_FAIL(LLG_E_INVALID, "stencil offset reaches beyond one period");
            }
        }
        const size_t nv = h.per_row ? (size_t)nc * h.sk * n : (size_t)nc * h.na * h.sk;
        h.vals.assign(e.stencil_vals, e.stencil_vals + nv);
    } else {
        SLLG_FAIL(LLG_E_INVALID, "unknown exchange format %d", h.fmt);
    }
    return 0;
}

template <class V>
void fill_common(Exch<V>& x, const HostExch& h, uint32_t n) {
    x.fmt = h.fmt;
    x.ncomp = h.ncomp;
    x.n = n;
    x.nnz = h.nnz;
    x.ndiag = h.ndiag;
    for (int a = 0; a < 3; ++a) { x.dims[a] = h.dims[a]; x.pbc[a] = h.pbc[a]; }
    x.na = h.na;
    x.sk = h.sk;
    x.per_row = h.per_row;
}

int upload_stencil_tables(llg_ctx* c) {
    ExchStore& X = *c->xs;
    const HostExch& h = X.h;
    std::vector<int4> ent((size_t)h.na * h.sk);
    for (size_t q = 0; q < ent.size(); ++q)
        ent[q] = make_int4(h.sent[q * 4], h.sent[q * 4 + 1], h.sent[q * 4 + 2], h.sent[q * 4 + 3]);
    SLLG_TRY(upload(X.a, ent.data(), ent.size(), c->stream));
    SLLG_TRY(upload(X.b, h.scount.data(), h.scount.size(), c->stream));
    return 0;
}

// Drop the host copies once the device holds the encoding (scalars stay for llg_get_info).
void release_host(HostExch& h) {
    std::vector<uint32_t>().swap(h.xadj);
    std::vector<uint32_t>().swap(h.adj);
    std::vector<double>().swap(h.vals);
    std::vector<int32_t>().swap(h.doff);
    std::vector<uint32_t>().swap(h.scount);
    std::vector<int32_t>().swap(h.sent);
}

}  // namespace

namespace {

// CSR rows as lane-uniform records (FMT_UNI).  Entry q of the 64 rows of a slice falls into a
// few classes of equal (row offset, couplings): one away from the lattice's boundaries, a
// second where a row's neighbour wraps around a periodic one.  A record holds one coupling and
// two offsets with the lanes that take the second, so a slice is about as many records as its
// rows have entries, each read once a wave, where the CSR reads 12 bytes or more a row and
// entry; rows without an entry q (open boundaries) take the offset "none".  Every row meets its
// own entries in CSR order, and the others load zeros, so the sums are the CSR's bit for bit.
// Slices with equal records are stored once.  False (nothing kept) when the records would be
// more than twice the entries of a row, as for couplings that differ from row to row, when a
// slice of a small system has more than kUniSlice times its entries, when the offsets do not
// fit, or when the caller wants every slice stored.
// The second bound: with few waves in flight a half step lasts as long as its longest slice, a
// record about a third of a sliced-CSR entry.  us a step, records and sliced CSR, by the longest
// slice's records an entry: bct 6^3 12.9 and 13.7 (3.75), fcc 10^3 37.2 and 33.5 (3.9), fcc 7^3 40.1
// and 32.0 (4.1), fcc 100 x 9 x 5 37.8 and 32.2 (4.05), fcc 40 x 5 x 3 45.5 and 29.9 (5.3), bct 3^3 15.3
// and 11.7 (6.75), a random chain of 64 with 4 neighbours 42.8 and 11.2 (64).  From 32,768 spins on
// the waves share the SIMDs, and the sum of the records counts (fcc 30 x 30 x 20, longest 3.7, mean
// 1.1: 43.7 and 65.4).
constexpr uint32_t kUniSlice = 4;
constexpr uint32_t kUniFew = 32768;
bool build_uniform(llg_ctx* c, const HostExch& h, const Perm& P, std::vector<uint2>& table,
                   std::vector<uint32_t>& words, uint32_t& stored) {
    const uint32_t n = c->n, nc = (uint32_t)h.ncomp, nsl = (n + kSlice - 1) / kSlice, BW = uni_words((int)nc);
    if (n > kUniMaxSpins || (c->flags & LLG_FLAG_NO_SLICE_SHARING)) return false;
    struct Rec {
        uint32_t d0, d1;
        uint64_t mask;
        uint32_t entry;  // an entry with the record's couplings
    };
    auto same = [&](uint32_t p, uint32_t q) {
        for (uint32_t k = 0; k < nc; ++k)
            if (std::memcmp(&h.vals[(size_t)k * h.nnz + p], &h.vals[(size_t)k * h.nnz + q], 8)) return false;
        return true;
    };
    const uint32_t sh = P.na > 1 && !(P.na & (P.na - 1)) ? (uint32_t)__builtin_ctz(P.na) : 0u;
    auto to_dev = [&](uint32_t i) { return sh ? (i & (P.na - 1)) * P.ncell + (i >> sh) : P.to_dev(i); };
    table.resize(nsl);
    std::unordered_map<uint64_t, std::vector<uint32_t>> seen;  // hash of a slice's words -> slices
    std::vector<Rec> recs;
    std::vector<uint32_t> st;
    uint64_t nrec = 0, nlen = 0;
    stored = 0;
    for (uint32_t s = 0; s < nsl; ++s) {
        const uint32_t d0 = s * kSlice, rows = std::min<uint32_t>(kSlice, n - d0);
        uint32_t first[kSlice], len[kSlice], most = 0;
        for (uint32_t l = 0; l < rows; ++l) {
            const uint32_t r = P.to_ref(d0 + l);
            first[l] = h.xadj[r];
            len[l] = h.xadj[r + 1] - h.xadj[r];
            most = std::max(most, len[l]);
        }
        recs.clear();
        for (uint32_t q = 0; q < most; ++q) {
            // classes of (offset, couplings) with their lanes; then records: a class and, where
            // there is one, another with the same couplings or the lanes that have none
            struct Cls {
                uint32_t off, entry;
                uint64_t lanes;
            } cls[kSlice];
            uint32_t m = 0;
            uint64_t none = 0;
            for (uint32_t l = 0; l < rows; ++l) {
                if (q >= len[l]) {
                    none |= 1ull << l;
                    continue;
                }
                const uint32_t p = first[l] + q, off = 8u * (to_dev(h.adj[p]) - (d0 + l));
                uint32_t k = 0;
                while (k < m && !(cls[k].off == off && same(cls[k].entry, p))) ++k;
                if (k == m) cls[m++] = Cls{off, p, 0};
                cls[k].lanes |= 1ull << l;
            }
            bool used[kSlice] = {};
            const uint64_t all = rows == kSlice ? ~0ull : (1ull << rows) - 1ull;
            for (uint32_t k = 0; k < m; ++k) {
                if (used[k]) continue;
                used[k] = true;
                uint32_t o = k + 1;
                while (o < m && (used[o] || !same(cls[k].entry, cls[o].entry))) ++o;
                // the lanes outside both classes of a record must read nothing
                if (o < m && (cls[k].lanes | cls[o].lanes) == all) {
                    used[o] = true;
                    recs.push_back(Rec{cls[k].off, cls[o].off, cls[o].lanes, cls[k].entry});
                } else {
                    recs.push_back(Rec{cls[k].off, kUniNone, all & ~cls[k].lanes, cls[k].entry});
                }
            }
        }
        nrec += recs.size();
        nlen += most;
        if (nrec > 2 * nlen + 256 || (n < kUniFew && recs.size() > (size_t)kUniSlice * most)) return false;
        const uint32_t blocks = ((uint32_t)recs.size() + kUniBlock - 1) / kUniBlock;
        st.assign((size_t)blocks * BW, 0u);
        for (uint32_t r = 0; r < blocks * kUniBlock; ++r) {
            uint32_t* const w = st.data() + (size_t)(r / kUniBlock) * BW;
            const uint32_t u = r % kUniBlock;
            const bool pad = r >= recs.size();
            w[u] = pad ? kUniNone : recs[r].d0;
            w[4 + u] = pad ? kUniNone : recs[r].d1;
            if (pad) continue;
            std::memcpy(w + 8 + 2 * u, &recs[r].mask, 8);
            for (uint32_t k = 0; k < nc; ++k)
                std::memcpy(w + 16 + 2 * (u * nc + k), &h.vals[(size_t)k * h.nnz + recs[r].entry], 8);
        }
        uint64_t hsh = 1469598103934665603ull;
        for (uint32_t v : st) hsh = (hsh ^ v) * 1099511628211ull;
        bool found = false;
        for (uint32_t o : seen[hsh])
            if (table[o].y == blocks && !std::memcmp(words.data() + table[o].x, st.data(), st.size() * 4)) {
                table[s] = table[o];
                found = true;
                break;
            }
        if (found) continue;
        if (words.size() + st.size() >= (1ull << 32)) return false;
        table[s] = make_uint2((uint32_t)words.size(), blocks);
        words.insert(words.end(), st.begin(), st.end());
        seen[hsh].push_back(s);
        ++stored;
    }
    return true;
}

// Sublattice-major device order when the caller declares the basis size (spins ordered
// cell * n_atoms + t, as the reference orders them).
Perm csr_order(const llg_ctx* c, uint32_t na) {
    Perm P;
    const bool sub = na > 1 && na <= 16 && c->n % na == 0 && !(c->flags & LLG_FLAG_NO_SUBLATTICE_ORDER);
    P.na = sub ? na : 1;
    P.ncell = sub ? c->n / na : c->n;
    return P;
}

}  // namespace

int build_exchange_fp64(llg_ctx* c, const llg_exchange& e) {
    ExchStore& X = *c->xs;
    SLLG_TRY(validate_and_copy(c, e));
    const HostExch& h = X.h;
    Exch<double>& x = X.ex64;
    fill_common(x, h, c->n);
    X.encoding = "none";
    std::vector<uint2> utable;
    std::vector<uint32_t> uwords;
    uint32_t ustored = 0;
    if (h.fmt == LLG_EXCH_CSR && build_uniform(c, h, csr_order(c, e.n_atoms), utable, uwords, ustored)) {
        X.perm = csr_order(c, e.n_atoms);
        uwords.resize(std::max<size_t>(uwords.size(), 4));
        SLLG_TRY(upload(X.a, utable.data(), utable.size(), c->stream));
        SLLG_TRY(upload(X.b, uwords.data(), uwords.size(), c->stream));
        x.fmt = FMT_UNI;
        x.slice = X.a.as<uint2>();
        x.ent = X.b.as<uint32_t>();
        x.nent = uwords.size();
        char buf[96];
        std::snprintf(buf, sizeof buf, "csr-uniform-t%u-f64-slices%uof%zu", X.perm.na, ustored, utable.size());
        X.encoding = buf;
    } else if (h.fmt == LLG_EXCH_CSR) {
        // The CSR stored by slices of 64 rows: entry q of every row of a slice at [q][lane]
        // (column-major within the slice, the slice as long as its longest row), so one load
        // of entry q by a wave is 64 consecutive words.  Each row keeps its entries in CSR
        // order and the kernels read a row's own count from the row pointers, so the sums are
        // the CSR sums, operation for operation.
        const uint32_t n = c->n, nsl = (n + kSlice - 1) / kSlice, nc = (uint32_t)h.ncomp;
        std::vector<uint2> sl(nsl);
        uint64_t tot = 0;
        for (uint32_t t = 0; t < nsl; ++t) {
            uint32_t len = 0;
            for (uint32_t r = t * kSlice; r < std::min(n, (t + 1) * kSlice); ++r) len = std::max(len, h.xadj[r + 1] - h.xadj[r]);
            sl[t] = make_uint2((uint32_t)tot, len);
            tot += len;
        }
        if (tot > 0xFFFFFFFFull) SLLG_FAIL(LLG_E_INVALID, "exchange too large for the sliced CSR");
        const size_t nent = (size_t)tot * kSlice;
        std::vector<uint32_t> ent(nent);
        std::vector<double> val((size_t)nc * nent, 0.0);
        for (uint32_t r = 0; r < nsl * kSlice; ++r) {
            const uint2 t = sl[r / kSlice];
            const uint32_t rl = r < n ? h.xadj[r + 1] - h.xadj[r] : 0;
            for (uint32_t q = 0; q < t.y; ++q) {
                const size_t o = ((size_t)t.x + q) * kSlice + r % kSlice;
                ent[o] = q < rl ? h.adj[h.xadj[r] + q] : (r < n ? r : 0);  // padding is never read
                if (q < rl)
                    for (uint32_t k = 0; k < nc; ++k) val[(size_t)k * nent + o] = h.vals[(size_t)k * h.nnz + h.xadj[r] + q];
            }
        }
        SLLG_TRY(upload(X.a, h.xadj.data(), h.xadj.size(), c->stream));
        SLLG_TRY(upload(X.b, ent.data(), ent.size(), c->stream));
        SLLG_TRY(upload(X.c, val.data(), val.size(), c->stream));
        SLLG_TRY(upload(X.d, sl.data(), sl.size(), c->stream));
        x.xadj = X.a.as<uint32_t>();
        x.ent = X.b.as<uint32_t>();
        x.vals = X.c.as<double>();
        x.slice = X.d.as<uint2>();
        x.nent = nent;
        X.encoding = "csr-sliced64-u32-f64";
    } else if (h.fmt == LLG_EXCH_DIA) {
        SLLG_TRY(upload(X.a, h.doff.data(), h.doff.size(), c->stream));
        SLLG_TRY(upload(X.c, h.vals.data(), h.vals.size(), c->stream));
        x.doff = X.a.as<int32_t>();
        x.vals = X.c.as<double>();
        X.encoding = "dia-f64";
    } else if (h.fmt == LLG_EXCH_STENCIL) {
        SLLG_TRY(upload_stencil_tables(c));
        SLLG_TRY(upload(X.c, h.vals.data(), h.vals.size(), c->stream));
        x.sent = X.a.as<int4>();
        x.scount = X.b.as<uint32_t>();
        x.vals = X.c.as<double>();
        X.encoding = h.per_row ? "stencil-rowvals-f64" : "stencil-shared-f64";
    }
    release_host(X.h);
    return 0;
}

namespace {

struct TupleKey {
    double v[9];
    int nc;
    bool operator==(const TupleKey& o) const { return std::memcmp(v, o.v, sizeof(double) * nc) == 0; }
};
struct TupleHash {
    size_t operator()(const TupleKey& k) const {
        uint64_t h = 1469598103934665603ull;
        const unsigned char* p = reinterpret_cast<const unsigned char*>(k.v);
        for (size_t i = 0; i < sizeof(double) * (size_t)k.nc; ++i) h = (h ^ p[i]) * 1099511628211ull;
        return (size_t)h;
    }
};

// One neighbour window of a line-mode slice: its first row relative to the slice's, the
// shifts it has couplings for (bit 0/1/2: dz = 0/+1/-1) and the couplings [shift][component].
struct Line {
    int32_t lrel;
    uint32_t mask;
    double v[3][9];
};

// Windows in groups of G: full groups of one shift mask first (masks 7 down to 1), then the
// remainders together under the union of their masks; -1 marks an unused slot.
std::vector<std::vector<int>> group_windows(const std::vector<Line>& lines, int G) {
    std::vector<std::vector<int>> grp;
    std::vector<int> rest;
    for (uint32_t m = 7; m >= 1; --m) {
        std::vector<int> cls;
        for (size_t l = 0; l < lines.size(); ++l)
            if (lines[l].mask == m) cls.push_back((int)l);
        size_t k = 0;
        for (; k + (size_t)G <= cls.size(); k += (size_t)G)
            grp.emplace_back(cls.begin() + (ptrdiff_t)k, cls.begin() + (ptrdiff_t)k + G);
        rest.insert(rest.end(), cls.begin() + (ptrdiff_t)k, cls.end());
    }
    for (size_t k = 0; k < rest.size(); k += (size_t)G) {
        std::vector<int> g(rest.begin() + (ptrdiff_t)k, rest.begin() + (ptrdiff_t)std::min(k + G, rest.size()));
        g.resize((size_t)G, -1);
        grp.push_back(g);
    }
    return grp;
}

// Tile streams of the LDS-staged line reader, made from the line records of a 64-cell line
// encoding in which every slice is a line.  A workgroup takes nw slices: nw / na
// consecutive lines of each of the na sublattice blocks (slice q = w nw + k of workgroup w
// is line q / na of sublattice q % na), so the lines it reads overlap as much as the
// sublattice-major order allows.  Its stream:
//   [0]                 lines staged (nU), [1] nw
//   [2 + k]             slice k's records: first word, relative to the stream
//   [2 + nw + k]        slice k's group count
//   [2 + 2 nw + k]      LDS byte offset of slice k's own line
//   [H, H + nU)         first rows of the staged lines relative to the workgroup's first row
//                       (line q0 / na of sublattice 0, q0 = w nw), int32; H = tile_head(nw)
//   then slice k's records, tile_words(nc) words each: the LDS byte offsets of the record's
//   line_group(nc) windows (kTileLineBytes per line in staging order, so multiples of 8; the
//   first carries the record's shift mask in its low 3 bits), then the couplings
//   [window][dz 0, +1, -1][component] (FP32, zero where a window has none).  The windows are
//   grouped exactly as in the line records (group_windows, line_group(nc) to a group), so
//   both readers form the same sums.
// Streams of equal content are stored once (interior workgroups of a periodic lattice
// repeat); tile_words(nc) zero words follow the last stream, so a reader may fetch one
// record past a slice's last.  kept: the windows of each stored line-record list, by its
// first word.  Chooses nw = 8, else 16: the first that divides the slices evenly
// and stages at most kTileLdsMax bytes.  On failure the encoding keeps no tile streams.
void build_tiles(llg_ctx* c, const std::vector<uint2>& table,
                 const std::unordered_map<uint32_t, std::vector<Line>>& kept) {
    ExchStore& X = *c->xs;
    Exch<float>& x = X.ex32;
    const uint32_t n = c->n, nsl = n / kSlice, na = X.perm.na;
    const int nc = X.h.ncomp, G = line_group(nc), TW = tile_words(nc);
    if (na > 1 && X.perm.ncell % kSlice) return;
    const uint32_t lps = na > 1 ? X.perm.ncell / kSlice : nsl;
    // the groups of each stored window list, as the line records have them
    std::unordered_map<uint32_t, std::vector<std::vector<int>>> groups;
    for (const auto& kv : kept) groups.emplace(kv.first, group_windows(kv.second, G));
    const std::vector<std::vector<int>> nogroups;
    for (uint32_t nw : {8u, 16u}) {
        if (nw % na || nsl % nw || lps % (nw / na)) continue;
        const uint32_t kk = nw / na, nwg = nsl / nw, H = (uint32_t)tile_head((int)nw);
        std::vector<uint32_t> tw, st;
        std::unordered_map<uint64_t, std::vector<uint32_t>> seen;  // stream hash -> workgroups
        std::vector<uint32_t> offs(nwg);
        uint32_t umax = 0;
        bool ok = true;
        std::vector<int64_t> rows;  // staged lines' first rows, staging order
        std::unordered_map<int64_t, uint32_t> slot;
        for (uint32_t w = 0; w < nwg && ok; ++w) {
            const int64_t B = (int64_t)(w * kk) * kSlice;
            rows.clear();
            slot.clear();
            auto slot_of = [&](int64_t r) -> uint32_t {
                auto it = slot.find(r);
                if (it != slot.end()) return it->second;
                const uint32_t u = (uint32_t)rows.size();
                slot.emplace(r, u);
                rows.push_back(r);
                return u;
            };
            st.assign(H, 0u);
            std::vector<uint32_t> recs;
            for (uint32_t k = 0; k < nw; ++k) {
                const uint32_t q = w * nw + k, s = (q % na) * lps + q / na;
                const int64_t base = (int64_t)s * kSlice;
                const uint2 t = table[s];
                const auto gi = t.y ? groups.find(t.x) : groups.end();
                const std::vector<std::vector<int>>& grp = gi != groups.end() ? gi->second : nogroups;
                st[2 + nw + k] = (uint32_t)grp.size();
                st[2 + 2 * nw + k] = slot_of(base) * kTileLineBytes;
                st[2 + k] = (uint32_t)recs.size();  // made relative to the stream below
                if (!grp.empty()) {
                    const std::vector<Line>& lines = kept.at(t.x);
                    for (const std::vector<int>& g : grp) {
                        const size_t o = recs.size();
                        recs.resize(o + (size_t)TW, 0u);
                        uint32_t mask = 0;
                        for (int u = 0; u < G; ++u) {
                            const Line& ln = lines[(size_t)(g[(size_t)u] >= 0 ? g[(size_t)u] : g[0])];
                            recs[o + (size_t)u] = slot_of(base + ln.lrel) * kTileLineBytes;
                            if (g[(size_t)u] < 0) continue;
                            mask |= ln.mask;
                            for (int kz = 0; kz < 3; ++kz)
                                for (int a = 0; a < nc; ++a) {
                                    const float v = (float)ln.v[kz][a];
                                    std::memcpy(&recs[o + (size_t)(G + (u * 3 + kz) * nc + a)], &v, 4);
                                }
                        }
                        recs[o] |= mask;
                    }
                }
            }
            const uint32_t nU = (uint32_t)rows.size();
            if ((uint64_t)nU * kTileLineBytes > kTileLdsMax) {
                ok = false;
                break;
            }
            umax = std::max(umax, nU);
            st[0] = nU;
            st[1] = nw;
            for (int64_t r : rows) st.push_back((uint32_t)(int32_t)(r - B));
            while (st.size() % 4) st.push_back(0u);
            const uint32_t r0 = (uint32_t)st.size();
            for (uint32_t k = 0; k < nw; ++k) st[2 + k] += r0;
            st.insert(st.end(), recs.begin(), recs.end());
            uint64_t hsh = 1469598103934665603ull;
            for (uint32_t v : st) hsh = (hsh ^ v) * 1099511628211ull;
            bool found = false;
            auto& cand = seen[hsh];
            for (uint32_t o : cand)
                if (offs[o] + st.size() <= tw.size() && tw[offs[o]] == st[0] &&
                    std::memcmp(tw.data() + offs[o], st.data(), st.size() * 4) == 0) {
                    // equal prefix of equal length: the stored stream has the same header,
                    // so its length is the same
                    offs[w] = offs[o];
                    found = true;
                    break;
                }
            if (!found) {
                if (tw.size() + st.size() + (size_t)TW >= (1ull << 32)) {  // offsets are 32-bit
                    ok = false;
                    break;
                }
                cand.push_back(w);
                offs[w] = (uint32_t)tw.size();
                tw.insert(tw.end(), st.begin(), st.end());
            }
        }
        if (!ok) continue;
        tw.insert(tw.end(), (size_t)TW, 0u);
        if (put(X, X.f, tw.data(), tw.size(), c->stream)) return;
        if (put(X, X.g, offs.data(), offs.size(), c->stream)) return;
        x.tnw = nw;
        x.tumax = umax;
        x.tlps = lps;
        return;
    }
}

// Line mode of the FP32 path.  When the lattice's fastest cell index runs along lines of
// len = 64 or 16 cells, a 64-row slice is one line (len 64) or four consecutive lines
// (len 16), and neighbour j of lane l is at row
//   L + (l & ~(len - 1)) + ((l + dz) mod len),   dz in {0, +1, -1},
// for periodic lines, or at L + l + dz with no neighbour past a line's ends for open lines,
// of a 64-row window starting at row L (a multiple of len).  Where that holds for every
// lane with one coupling tuple, the couplings of a slice are lane-uniform: per window, one
// load of the spins, and the shifted neighbours come from a rotation (periodic) or a
// zero-filling shift (open) across the wave (len 64) or within each 16-lane row (len 16).  Slices where it does not hold (a window
// that would wrap a periodic boundary inside the slice) keep the packed entries
// (kLineFallback).  A slice becomes a list of group records read with scalar loads,
// G = line_group(ncomp) windows each, line_words(ncomp) words:
//   [0]                  shift mask of the group: bit 0/1/2 = some window of the group has
//                        couplings for dz = 0 / +1 / -1
//   [1, 1 + G)           window starts L - slice base (int32, multiples of len)
//   [1 + G, 1 + G + 3 G nc)  couplings [window][dz 0, +1, -1][component], FP32, zero where
//                        the window has none
//   [W - G, W)           the next group's window starts (zero after the last group); W is
//                        rounded up to whole 16-byte units, the words between are zero
// so the reader issues the next group's window loads before it uses the current group.
// Windows are grouped by their own shift masks (full groups of one mask first, the rest
// together under the union of their masks), so a group tests each shift once for all its
// windows; an unused slot repeats the group's first window with zero couplings.  The reader
// sums each shift's contributions unshifted and rotates the three partial sums once.
// Entries of one row that name the same (window, dz) are summed (in FP64, rounded once).
// Identical record lists are stored once; the first record is a zero record for empty
// slices.  Entries are summed window by window, not in stored CSR order.
bool build_lines(llg_ctx* c, const std::vector<uint32_t>& ref_of, const std::vector<uint32_t>& idx,
                 const std::vector<TupleKey>& tuples, uint32_t len, bool open, uint32_t& stored,
                 uint32_t& lines_row, uint32_t& nfall) {
    ExchStore& X = *c->xs;
    const HostExch& h = X.h;
    const uint32_t n = c->n;
    const int nc = h.ncomp;
    const Perm P = X.perm;
    if (n % kSlice != 0) return false;
    const uint32_t nsl = n / kSlice;
    const int G = line_group(nc), W = line_words(nc);
    std::vector<uint32_t> words((size_t)W, 0u);  // the zero record
    std::vector<uint2> table(nsl);
    std::unordered_map<uint64_t, std::vector<uint32_t>> seen;  // record-list hash -> stored slices
    std::unordered_map<uint32_t, std::vector<Line>> kept;     // windows of each stored record list
    std::vector<uint32_t> st;
    stored = 0;
    nfall = 0;
    uint64_t lines_total = 0, lined = 0;
    const int32_t lm = (int32_t)len - 1;
    // key of one coupling of row d0 + l: window start relative to d0, shift dz, tuple
    using LKey = std::tuple<int64_t, int, uint32_t>;
    // keys of row d0 + l in CSR order (csr, optional) and sorted (out, for comparing lanes)
    auto lane_keys = [&](uint32_t d0, int32_t l, std::vector<LKey>& out, std::vector<LKey>* csr) -> bool {
        out.clear();
        const uint32_t r = ref_of[d0 + (uint32_t)l];
        for (uint32_t qq = h.xadj[r]; qq < h.xadj[r + 1]; ++qq) {
            const int64_t j = P.to_dev(h.adj[qq]);
            bool found = false;
            for (int dz : {0, 1, -1}) {
                int32_t pos = (l & lm) + dz;
                if (open) {
                    if (pos < 0 || pos > lm) continue;
                } else {
                    pos &= lm;
                }
                const int64_t L = j - (int64_t)((l & ~lm) + pos);
                if (L % (int64_t)len == 0 && L >= 0 && L + kSlice <= (int64_t)n) {
                    out.emplace_back(L - (int64_t)d0, dz, idx[qq]);
                    found = true;
                    break;
                }
            }
            if (!found) return false;
        }
        if (csr) *csr = out;
        std::sort(out.begin(), out.end());
        return true;
    };
    std::vector<LKey> ref, ref_csr, lk, first, last;
    for (uint32_t s = 0; s < nsl; ++s) {
        const uint32_t d0 = s * kSlice;
        std::vector<Line> lines;
        // periodic lines: every lane has the same keys; open lines: every interior lane
        // does, and a line's first (last) lane lacks the keys that shift past its start (end)
        bool fits = lane_keys(d0, open ? 1 : 0, ref, &ref_csr);
        if (fits && open) {
            first.clear();
            last.clear();
            for (const LKey& k : ref) {
                if (std::get<1>(k) != -1) first.push_back(k);
                if (std::get<1>(k) != 1) last.push_back(k);
            }
        }
        for (int32_t l = 0; l < kSlice && fits; ++l) {
            fits = lane_keys(d0, l, lk, nullptr);
            if (!fits) break;
            const int32_t p = l & lm;
            const std::vector<LKey>& want = !open ? ref : (p == 0 ? first : (p == lm ? last : ref));
            fits = lk == want;
        }
        if (fits) {
            // windows in the order the CSR row names them; repeated neighbours add up
            for (const LKey& key : ref_csr) {
                const int32_t lrel = (int32_t)std::get<0>(key);
                const int dz = std::get<1>(key);
                Line* g = nullptr;
                for (Line& x : lines)
                    if (x.lrel == lrel) g = &x;
                if (!g) {
                    lines.push_back(Line{lrel, 0u, {}});
                    g = &lines.back();
                }
                const int k = dz == 0 ? 0 : (dz == 1 ? 1 : 2);
                g->mask |= 1u << k;
                for (int a = 0; a < nc; ++a) g->v[k][a] += tuples[std::get<2>(key)].v[a];
            }
        }
        if (!fits) {  // this slice keeps its packed entries
            table[s] = make_uint2(0u, kLineFallback);
            ++nfall;
            continue;
        }
        ++lined;
        st.clear();
        const std::vector<std::vector<int>> grp = group_windows(lines, G);
        const size_t ng = grp.size();
        auto start_of = [&](const std::vector<int>& g, int u) -> uint32_t {
            return (uint32_t)lines[(size_t)(g[(size_t)u] >= 0 ? g[(size_t)u] : g[0])].lrel;
        };
        for (size_t gi = 0; gi < ng; ++gi) {
            const std::vector<int>& g = grp[gi];
            std::vector<uint32_t> rec((size_t)W, 0u);
            for (int u = 0; u < G; ++u) {
                rec[(size_t)(1 + u)] = start_of(g, u);
                if (gi + 1 < ng) rec[(size_t)(W - G + u)] = start_of(grp[gi + 1], u);
                if (g[(size_t)u] < 0) continue;
                const Line& ln = lines[(size_t)g[(size_t)u]];
                rec[0] |= ln.mask;
                for (int k = 0; k < 3; ++k)
                    for (int a = 0; a < nc; ++a) {
                        const float v = (float)ln.v[k][a];
                        std::memcpy(&rec[(size_t)(1 + G + (u * 3 + k) * nc + a)], &v, 4);
                    }
            }
            st.insert(st.end(), rec.begin(), rec.end());
        }
        lines_total += lines.size();
        const uint32_t nrec = (uint32_t)ng;
        if (nrec == 0) {
            table[s] = make_uint2(0u, 0u);
            continue;
        }
        uint64_t hsh = 1469598103934665603ull;
        for (uint32_t w : st) hsh = (hsh ^ w) * 1099511628211ull;
        bool found = false;
        auto& cand = seen[hsh];
        for (uint32_t o : cand)
            if (table[o].y == nrec && std::memcmp(words.data() + table[o].x, st.data(), st.size() * 4) == 0) {
                table[s] = table[o];
                found = true;
                break;
            }
        if (!found) {
            cand.push_back(s);
            table[s] = make_uint2((uint32_t)words.size(), nrec);
            words.insert(words.end(), st.begin(), st.end());
            kept.emplace(table[s].x, lines);
            ++stored;
        }
    }
    // worth it only when most slices are lines
    if (lined == 0 || 4u * nfall > nsl) return false;
    if (put(X, X.d, words.data(), words.size(), c->stream)) return false;
    if (put(X, X.e, table.data(), table.size(), c->stream)) return false;
    Exch<float>& x = X.ex32;
    if (len == 64 && nfall == 0) build_tiles(c, table, kept);
    x.fmt = len == 64 ? (open ? FMT_SELL_LINE_OPEN : FMT_SELL_LINE) : (open ? FMT_SELL_LINE16_OPEN : FMT_SELL_LINE16);
    x.lfall = nfall;
    lines_row = (uint32_t)(lines_total / lined);
    return true;
}

// Line blocks of a packed encoding (read by k_block.hip).  When the rows of a sublattice that
// share a lattice line (len cells, the fastest index) have the same entries, each to the same
// neighbour line with the same shift along the (periodic) line and the same couplings, a
// workgroup of m consecutive lines can stage whole neighbour lines in LDS, and entry q of every
// one of its rows lies at one LDS distance from the row's own spin: the neighbour lines of
// entry q, one per line of the workgroup, form a chain, and chains are staged as consecutive
// lines (overlapping ones share lines: the chains of y - 1, y and y + 1 take m + 2).  Found
// from the couplings alone: the shortest line length that fits.
struct BlockEnt {
    uint32_t t, line, id;  // neighbour's sublattice and line, coupling tuple
    int32_t dz;
    bool like(const BlockEnt& o) const { return t == o.t && id == o.id && dz == o.dz; }
};
constexpr int32_t kBlockShift = 4;  // largest shift along a line

// Entries of line L of sublattice t; false when its rows differ.  Away from the line's ends a
// row's neighbours are the first row's, its distance further: whole rows are compared without a
// branch.  at, id: scratch.
bool block_line(const HostExch& h, const Perm& P, const std::vector<uint32_t>& idx, uint32_t Z, uint32_t t, uint32_t L,
                std::vector<BlockEnt>& out, std::vector<uint32_t>& at, std::vector<uint32_t>& id) {
    out.clear();
    at.clear();
    id.clear();
    const uint32_t r0 = P.to_ref(t * P.ncell + L * Z), q00 = h.xadj[r0], len = h.xadj[r0 + 1] - q00;
    uint32_t reach = 0;  // largest shift along the line
    for (uint32_t q = 0; q < len; ++q) {
        const uint32_t j = P.to_dev(h.adj[q00 + q]), tj = j / P.ncell, cj = j - tj * P.ncell, zj = cj % Z;
        const int32_t dz = 2 * zj > Z ? (int32_t)zj - (int32_t)Z : (int32_t)zj;
        if (std::abs(dz) > kBlockShift || 2 * std::abs(dz) >= (int32_t)Z) return false;
        reach = std::max(reach, (uint32_t)std::abs(dz));
        out.push_back(BlockEnt{tj, cj / Z, idx[q00 + q], dz});
        at.push_back((uint32_t)((int32_t)(cj / Z * Z) + dz) * P.na + tj);  // modulo 2^32 where dz < 0
        id.push_back(idx[q00 + q]);
    }
    for (uint32_t z = 1; z < Z; ++z) {  // reference rows of a line are na apart
        const uint32_t r = r0 + z * P.na, q0 = h.xadj[r];
        if (h.xadj[r + 1] - q0 != len) return false;
        if (z >= reach && z + reach < Z) {  // nothing wraps
            const uint32_t *pa = &h.adj[q0], *pi = &idx[q0];
            uint32_t diff = 0;
            for (uint32_t q = 0; q < len; ++q) diff |= (pa[q] - z * P.na - at[q]) | (pi[q] ^ id[q]);
            if (diff) return false;
            continue;
        }
        for (uint32_t q = 0; q < len; ++q) {
            const BlockEnt& e = out[q];
            int32_t w = (int32_t)z + e.dz;
            w += w < 0 ? (int32_t)Z : 0;
            w -= w >= (int32_t)Z ? (int32_t)Z : 0;
            if (h.adj[q0 + q] != (e.line * Z + (uint32_t)w) * P.na + e.t || idx[q0 + q] != e.id) return false;
        }
    }
    return true;
}

// Lines a workgroup stages: chains of g lines placed on tracks of consecutive lines.
struct BlockLayout {
    struct Track {
        uint32_t t;
        std::vector<uint32_t> lines;
    };
    std::vector<Track> tracks;
    std::map<std::vector<uint32_t>, std::pair<uint32_t, uint32_t>> at;  // chain {t, lines} -> track, first line

    uint32_t staged() const {
        uint32_t k = 0;
        for (const Track& tr : tracks) k += (uint32_t)tr.lines.size();
        return k;
    }
    void build(const std::vector<std::vector<BlockEnt>>& lists, uint32_t na, uint32_t nl, uint32_t L0, uint32_t g) {
        tracks.clear();
        at.clear();
        std::vector<uint32_t> key(g + 1);
        for (uint32_t t = 0; t < na; ++t) {
            key[0] = t;
            for (uint32_t j = 0; j < g; ++j) key[j + 1] = L0 + j;
            at.emplace(key, std::make_pair(0u, 0u));
            const size_t len = lists[(size_t)t * nl + L0].size();
            for (size_t q = 0; q < len; ++q) {
                key[0] = lists[(size_t)t * nl + L0][q].t;
                for (uint32_t j = 0; j < g; ++j) key[j + 1] = lists[(size_t)t * nl + L0 + j][q].line;
                at.emplace(key, std::make_pair(0u, 0u));
            }
        }
        std::vector<std::pair<uint32_t, int64_t>> pos;  // per chain: track, first line (relative to the track's base)
        std::vector<int64_t> base;                      // of each track's first line
        for (auto& c : at) {
            const uint32_t* lines = c.first.data() + 1;
            uint32_t best = 0, track = 0;
            int64_t where = 0;
            for (uint32_t k = 0; k < tracks.size(); ++k) {
                if (tracks[k].t != c.first[0]) continue;
                const std::vector<uint32_t>& tl = tracks[k].lines;
                const int64_t n = (int64_t)tl.size();
                for (int64_t o = 1 - (int64_t)g; o < n; ++o) {
                    uint32_t same = 0;
                    bool ok = true;
                    for (int64_t j = std::max<int64_t>(0, -o); j < (int64_t)g && o + j < n && ok; ++j) {
                        ok = tl[(size_t)(o + j)] == lines[j];
                        ++same;
                    }
                    if (ok && same > best) {
                        best = same;
                        track = k;
                        where = o;
                    }
                }
            }
            if (!best) {
                track = (uint32_t)tracks.size();
                tracks.push_back(Track{c.first[0], {}});
                base.push_back(0);
                where = 0;
            }
            std::vector<uint32_t>& tl = tracks[track].lines;
            if (where < 0) {  // lines before the track's first
                tl.insert(tl.begin(), lines, lines - where);
                base[track] += where;
                where = 0;
            }
            for (uint32_t j = (uint32_t)((int64_t)tl.size() - where); j < g; ++j) tl.push_back(lines[j]);
            pos.emplace_back(track, where + base[track]);
        }
        std::vector<uint32_t> first(tracks.size(), 0);
        for (size_t k = 1; k < tracks.size(); ++k) first[k] = first[k - 1] + (uint32_t)tracks[k - 1].lines.size();
        size_t k = 0;
        for (auto& c : at) {
            c.second = std::make_pair(pos[k].first, first[pos[k].first] + (uint32_t)(pos[k].second - base[pos[k].first]));
            ++k;
        }
    }
};

// Groups of g lines whose entries lead, line by line, to the same lines relative to their own
// first one (with the same couplings) have the same layout, moved along, and the same records:
// both are built once a class of such groups.  Creating a handle, fcc 37 x 45 x 51 x 4 and 60 x 60 x
// 20 x 4: 280 and 250 ms with a layout a group and rows compared entry by entry, 241 and 208 now, 230
// and 189 without blocks.
struct BlockClass {
    uint32_t nst = 0;    // lines staged
    uint32_t group = 0;  // of m lines: how many of them a group takes (group_at), once known
    // of a class with stored records: staged lines {sublattice, line from the group's first}, per
    // sublattice its own first line, first record word and records
    std::vector<std::pair<uint32_t, uint32_t>> lines;
    std::vector<uint32_t> own, where, nrec;
};
constexpr size_t kBlockClasses = 4096;  // remembered at a time
struct BlockSigHash {
    size_t operator()(const std::vector<uint32_t>& v) const {
        uint64_t h = 1469598103934665603ull;
        for (uint32_t w : v) h = (h ^ w) * 1099511628211ull;
        return (size_t)h;
    }
};

// Whether a new handle reads line blocks (lines of Z cells) rather than what it has beside them.
// The blocks stage every line of a workgroup and its neighbours, whole, so they gain with the
// entries a row (read from LDS) and lose with the lines' length, which leaves fewer lines to a
// workgroup and so more staged cells a row.  us a step at 300 K, untuned, blocks last.
// Against packed entries:
//   8 entries (bct): lines of 20 to 63 cells 0.85 to 1.03 of the packed time (64 x 65 x 63 cells 19.2
//     and 18.5), but from 600,000 spins on and past 40 cells 1.01 to 1.13 (100 x 100 x 52 27.3 and 31.0);
//     100 cells 1.02 to 1.24 (100^3 48.6 and 57.0), 200 cells 1.2 to 1.6
//   12 (fcc) and 14 (bct): up to 63 cells 0.67 to 1.06; 80 to 127 cells 0.9 to 1.3 (fcc 64 x 65 x 80
//     38.6 and 48.6); 200 cells 1.1 to 1.5
//   18 (simple cubic): up to 52 cells 0.88 to 1.08, 63 cells 0.97 to 1.2, 80 and 100 cells 0.94 to 1.1
//     and from 400,000 spins on 0.94 to 0.99, 127 cells 1.01 to 1.09
//   26 and 32 (simple cubic): up to 127 cells 0.81 to 1.06; 200 cells 0.99 to 1.13
//   42 (fcc): 0.64 to 0.92 at all lengths measured (7 to 127)
// Against the line reader (encodings of 64- or 16-cell lines without tile streams), which also
// loads a whole line at a time: one sublattice, 64 cells, 1.02 to 1.5 (18 and 26 entries, 8,000 to
// 1,000,000 spins; 262,080 spins 12.9 and 15.8), 16 cells 0.93 to 0.97 at 65,536 spins and 1.05 to 1.09
// at 262,144; bct, 14 entries, from 147,000 spins on 1.05 to 1.25, below 0.93 to 1.01, 8 entries 0.93
// to 0.97 up to 508,000 spins and 1.09 at 991,000; fcc, 12 entries 0.75 to 0.95 throughout, 18 entries
// up to 495,000 spins 0.83 to 0.98, 1,000,000 1.06, 42 entries up to 295,000 0.78 to 1.03, 495,000 and
// more 1.07 to 1.18.
bool blocks_pay(uint32_t n, uint32_t na, uint32_t Z, uint32_t entries, bool lines) {
    if (lines) {
        if (na == 1) return Z < 64 && n < 131072u;
        if (na == 2) return n < (entries > 12 ? 131072u : 750000u);
        return entries <= 12 || (uint64_t)n * entries < 17000000u;
    }
    if (entries >= 40) return true;
    if (entries >= 24) return Z <= 128;
    if (entries < 12 && Z > 40 && n >= 600000u) return false;
    if (na == 1 && entries >= 16 && n >= 400000u) return Z <= 100;
    return Z <= (na == 1 ? 56u : 64u);
}

// Up to this size blocks are built also where a new handle does not read them: about a millisecond
// of its creation, and the autotuner times them.
constexpr uint32_t kBlockSmall = 16384;

bool build_blocks(llg_ctx* c, const std::vector<uint32_t>& idx, const std::vector<TupleKey>& tuples) {
    ExchStore& X = *c->xs;
    const HostExch& h = X.h;
    const Perm P = X.perm;
    const uint32_t na = P.na, ncell = P.ncell, nc = (uint32_t)h.ncomp;
    if (na > kBlockSub || X.len_max < kBlockMinLen || c->n <= kSmallSpins) return false;
    const uint32_t zmax = kBlockWaves / na * 64u;  // a workgroup holds one line of every sublattice
    std::vector<std::vector<BlockEnt>> lists;
    uint32_t Z = 0, nl = 0;
    std::vector<BlockEnt> e;
    std::vector<uint32_t> at, id;
    auto pays = [&](uint32_t z) { return blocks_pay(c->n, na, z, X.len_max, is_line_fmt(X.ex32.fmt)); };
    for (uint32_t z = 4; z <= zmax && z <= ncell && !Z; ++z) {
        if (ncell % z) continue;
        nl = ncell / z;
        if (!block_line(h, P, idx, z, 0, 0, e, at, id) || !block_line(h, P, idx, z, 0, nl / 2, e, at, id)) continue;
        if (c->n > kBlockSmall && !pays(z)) continue;
        lists.assign((size_t)na * nl, {});
        bool ok = true;
        for (uint32_t k = 0; k < na * nl && ok; ++k) ok = block_line(h, P, idx, z, k / nl, k % nl, lists[k], at, id);
        if (ok) Z = z;
    }
    if (!Z) return false;
    uint32_t H = 0;
    for (const auto& l : lists)
        for (const BlockEnt& q : l) H = std::max(H, (uint32_t)std::abs(q.dz));
    const uint32_t len = Z + 2 * H, line_bytes = len * 12u;
    // lines g .. of a group starting at L0 that may follow it: entries alike, line by line
    auto alike = [&](uint32_t L0, uint32_t L) {
        for (uint32_t t = 0; t < na; ++t) {
            const auto &a = lists[(size_t)t * nl + L0], &b = lists[(size_t)t * nl + L];
            if (a.size() != b.size()) return false;
            for (size_t q = 0; q < a.size(); ++q)
                if (!a[q].like(b[q])) return false;
        }
        return true;
    };
    std::unordered_map<std::vector<uint32_t>, BlockClass, BlockSigHash> classes;
    std::vector<uint32_t> sig;
    BlockLayout lay;
    auto class_of = [&](uint32_t L0, uint32_t g) -> BlockClass& {
        sig.assign(1, g);
        for (uint32_t t = 0; t < na; ++t) {
            const size_t cnt = lists[(size_t)t * nl + L0].size();
            sig.push_back((uint32_t)cnt);
            for (size_t q = 0; q < cnt; ++q) {
                const BlockEnt& a = lists[(size_t)t * nl + L0][q];
                sig.insert(sig.end(), {a.t, a.id, (uint32_t)a.dz});
                for (uint32_t j = 0; j < g; ++j) sig.push_back(lists[(size_t)t * nl + L0 + j][q].line - L0);
            }
        }
        BlockClass& b = classes[sig];
        if (b.nst == 0) {
            lay.build(lists, na, nl, L0, g);
            b.nst = lay.staged();
        }
        return b;
    };
    // groups of at most m lines: one more line is taken while it does not stage more than half
    // as many lines as a line alone needs (a step over a lattice boundary does)
    auto group_at = [&](uint32_t L0, uint32_t m) -> uint32_t {
        bool whole = L0 + m <= nl;
        for (uint32_t j = 1; j < m && whole; ++j) whole = alike(L0, L0 + j);
        uint32_t* const known = whole ? &class_of(L0, m).group : nullptr;
        if (known && *known) return *known;
        const uint32_t one = class_of(L0, 1).nst;
        uint32_t g = 1, prev = one;
        while (g < m && L0 + g < nl && alike(L0, L0 + g)) {
            const uint32_t s = class_of(L0, g + 1).nst;
            if (g == 1 ? s > 2 * one : (s - prev) * 2 > one) break;
            if (s * line_bytes > kBlockLdsMax) break;
            prev = s;
            ++g;
        }
        if (known) *known = g;
        return g;
    };
    // Lines of a workgroup: the least estimated time of a cell, from the cycles of a wave (the row
    // itself, its entries, its share of the staging loads), lanes without a row (they cost half:
    // they take no bandwidth) and waves waiting at one barrier; at least three workgroups for
    // two CUs.  us a step of fcc with 42 entries a row, by lines: 37 x 45 x 51 cells 19.8 (1), 22.4
    // (2), 24.8 (5); 60 x 60 x 33 30.9 (1), 27.9 (3), 28.2 (5); 60 x 60 x 20 27.6 (1), 18.7 (3), 21.8
    // (5); 80 x 80 x 12 40.1 (1), 18.8 (5); 20^3, too few lines, 10.4 (1), 11.2 (3).
    uint32_t m = 1;
    double best = 0.0;
    for (uint32_t k = 1; k <= std::min(zmax / Z, 16u); ++k) {
        if (k > 1 && nl / k < 384) break;
        uint32_t nst = 0xFFFFFFFFu;
        for (uint32_t s = 0; s < 4; ++s) {  // the fewest of four places: away from the boundaries
            const uint32_t L0 = (uint32_t)((uint64_t)(nl - k) * s / 3);
            bool same = true;
            for (uint32_t j = 1; j < k && same; ++j) same = alike(L0, L0 + j);
            if (!same) continue;
            nst = std::min(nst, class_of(L0, k).nst);
        }
        if (nst == 0xFFFFFFFFu || nst * line_bytes > kBlockLdsMax) continue;
        const uint32_t wv = (k * Z + 63) / 64;
        const double loads = (len <= 32 ? (double)nst / (64 / len) : (double)nst * ((len + 63) / 64)) / (wv * na);
        const double lanes = wv * 64.0 / (k * Z);
        const double cost = (300.0 + 8.0 * X.len_max + 20.0 * loads) * (0.5 + 0.5 * lanes) *
                            (1.0 + 0.025 * std::max(0.0, (double)(wv * na) - 4.0));
        if (best == 0.0 || cost < best) {
            best = cost;
            m = k;
        }
    }
    if (best == 0.0) return false;
    const uint32_t ws = (m * Z + 63) / 64;
    std::vector<uint32_t> tw, table, st;
    std::unordered_map<uint64_t, std::vector<std::pair<uint32_t, uint32_t>>> seen;  // record lists: first word, words
    uint32_t umax = 0;
    const uint32_t RW = (uint32_t)block_words((int)nc);
    std::vector<uint32_t> key, recs;
    for (uint32_t L0 = 0, g; L0 < nl; L0 += g) {
        if (classes.size() > kBlockClasses) classes.clear();
        g = group_at(L0, m);
        BlockClass& cl = class_of(L0, g);
        const uint32_t nst = cl.nst;
        if (nst * line_bytes > kBlockLdsMax) return false;
        umax = std::max(umax, nst);
        const uint32_t base = (uint32_t)tw.size();
        if ((uint64_t)base + kBlockHead + nst + 16 + (uint64_t)na * (X.len_max + 4) * RW >= (1ull << 31)) return false;
        table.insert(table.end(), {base, L0, g, nst});
        tw.resize(base + kBlockHead, 0u);
        tw[base] = ((1u << 20) + Z - 1) / Z;
        tw[base + 1] = ((1u << 20) + len - 1) / len;
        tw[base + 2] = 64u / len;
        const bool first = cl.own.empty();
        if (first) {
            lay.build(lists, na, nl, L0, g);
            for (const auto& tr : lay.tracks)
                for (uint32_t L : tr.lines) cl.lines.emplace_back(tr.t, L - L0);
        }
        for (const auto& q : cl.lines) tw.push_back(q.first * ncell + (L0 + q.second) * Z);
        while (tw.size() % 4) tw.push_back(0u);
        key.assign(g + 1, 0u);
        for (uint32_t t = 0; first && t < na; ++t) {
            key[0] = t;
            for (uint32_t j = 0; j < g; ++j) key[j + 1] = L0 + j;
            const uint32_t own = lay.at.at(key).second;
            const auto& l0 = lists[(size_t)t * nl + L0];
            const uint32_t nrec = ((uint32_t)l0.size() + 3) / 4;
            recs.assign((size_t)nrec * RW, 0u);  // unused entries: the row itself, zero couplings
            for (size_t q = 0; q < l0.size(); ++q) {
                key[0] = l0[q].t;
                for (uint32_t j = 0; j < g; ++j) key[j + 1] = lists[(size_t)t * nl + L0 + j][q].line;
                uint32_t* rec = &recs[q / 4 * RW];
                const int32_t off = ((int32_t)lay.at.at(key).second - (int32_t)own) * (int32_t)line_bytes + l0[q].dz * 12;
                rec[q % 4] = (uint32_t)off;
                for (uint32_t a = 0; a < nc; ++a) {
                    const float v = (float)tuples[l0[q].id].v[a];
                    std::memcpy(&rec[4 + q % 4 * nc + a], &v, 4);
                }
            }
            uint64_t hsh = 1469598103934665603ull;
            for (uint32_t v : recs) hsh = (hsh ^ v) * 1099511628211ull;
            uint32_t where = 0;
            bool found = false;
            for (const auto& s : seen[hsh])
                if (s.second == recs.size() && std::memcmp(&tw[s.first], recs.data(), recs.size() * 4) == 0) {
                    where = s.first;
                    found = true;
                    break;
                }
            if (!found) {
                where = (uint32_t)tw.size();
                tw.insert(tw.end(), recs.begin(), recs.end());
                seen[hsh].emplace_back(where, (uint32_t)recs.size());
            }
            cl.own.push_back(own);
            cl.where.push_back(where);
            cl.nrec.push_back(nrec);
        }
        for (uint32_t t = 0; t < na; ++t) {
            tw[base + 4 + t] = cl.own[t] * line_bytes + H * 12u;
            tw[base + 12 + t] = cl.where[t] - base;  // modulo 2^32: lists of earlier workgroups lie before
            tw[base + 20 + t] = cl.nrec[t];
        }
    }
    tw.insert(tw.end(), 2 * (size_t)RW, 0u);  // the reader fetches a record or two past a list
    if (put(X, X.f, tw.data(), tw.size(), c->stream)) return false;
    if (put(X, X.g, table.data(), table.size(), c->stream)) return false;
    Exch<float>& x = X.ex32;
    x.tnw = ws;
    x.tumax = H;
    x.tlps = Z;
    X.blk_wgs = (uint32_t)(table.size() / 4);
    X.blk_waves = ws * na;
    X.blk_lds = umax * line_bytes;
    X.blk_first = pays(Z);
    char buf[64];
    std::snprintf(buf, sizeof buf, "-blocks%ux%u", Z, m);
    X.encoding += buf;
    return true;
}

// CSR -> sliced ELL.  Packed layout: per slice, entries in chunks of 4 per lane,
// [chunk][lane][4], so one uint4 load per lane reads 4 entries and a wave reads 1 KB
// contiguous, then a tail of 2 per lane [lane][2] (one uint2 load); slice lengths are
// rounded up to a multiple of 2 with zero-coupling entries
// (offset 0, dictionary tuple 0.0), which add exactly 0 to the field.  Raw layout:
// [entry][lane] u32 columns and [ncomp][entry][lane] FP32 values.
int build_sell(llg_ctx* c) {
    ExchStore& X = *c->xs;
    const HostExch& h = X.h;
    const uint32_t n = c->n;
    const int nc = h.ncomp;
    const Perm P = X.perm;
    const uint32_t ncell = P.ncell;
    const uint32_t nsl = (n + kSlice - 1) / kSlice;
    // device row d holds reference row P.to_ref(d)
    std::vector<uint32_t> ref_of(n);
    for (uint32_t d = 0; d < n; ++d) ref_of[d] = P.to_ref(d);
    std::vector<uint32_t> mx(nsl, 0);
    for (uint32_t s = 0; s < nsl; ++s)
        for (uint32_t d = s * kSlice; d < std::min(n, (s + 1) * kSlice); ++d) {
            const uint32_t r = ref_of[d];
            mx[s] = std::max(mx[s], h.xadj[r + 1] - h.xadj[r]);
        }
    // Packed form: few distinct coupling tuples (the LDS dictionary) and row offsets that
    // fit the bits the dictionary index leaves; 12 n bytes must fit one buffer resource.
    bool pack = (uint64_t)n * 12u < (1ull << 31);
    std::unordered_map<TupleKey, uint32_t, TupleHash> dict;
    std::vector<TupleKey> tuples;
    std::vector<uint32_t> idx;
    if (pack) {
        TupleKey z{};
        z.nc = nc;
        dict.emplace(z, 0u);  // tuple 0 is the zero coupling used for padding
        tuples.push_back(z);
        idx.resize(h.nnz);
        TupleKey last{};
        last.nc = -1;
        uint32_t last_id = 0;
        for (uint64_t q = 0; q < h.nnz && pack; ++q) {
            TupleKey k{};
            k.nc = nc;
            for (int a = 0; a < nc; ++a) k.v[a] = h.vals[(size_t)a * h.nnz + q];
            if (last.nc == nc && k == last) { idx[q] = last_id; continue; }
            auto it = dict.find(k);
            uint32_t id;
            if (it == dict.end()) {
                id = (uint32_t)tuples.size();
                if ((uint64_t)(id + 1) * nc > (uint64_t)kDictLds || id > 0xFFFu) { pack = false; break; }
                dict.emplace(k, id);
                tuples.push_back(k);
            } else {
                id = it->second;
            }
            idx[q] = id;
            last = k;
            last_id = id;
        }
    }
    uint32_t dbits = 1;
    if (pack) {
        while ((1u << dbits) < tuples.size()) ++dbits;
        const int64_t lim = (int64_t)1 << (31 - dbits);
        for (uint32_t r = 0; r < n && pack; ++r) {
            const int64_t dr = P.to_dev(r);
            for (uint32_t q = h.xadj[r]; q < h.xadj[r + 1]; ++q) {
                const int64_t off = (int64_t)P.to_dev(h.adj[q]) - dr;
                if (off < -lim || off >= lim) { pack = false; break; }
            }
        }
    }
    // slice table {first entry / 64, entries per row}
    std::vector<uint2> slice(nsl);
    uint64_t tot = 0;
    for (uint32_t s = 0; s < nsl; ++s) {
        slice[s].y = pack ? (mx[s] + 1u) / 2u * 2u : mx[s];
        X.len_max = std::max(X.len_max, slice[s].y);
        slice[s].x = (uint32_t)tot;
        tot += slice[s].y;
    }
    if (tot > 0xFFFFFFFFull) SLLG_FAIL(LLG_E_INVALID, "exchange too large for the sliced-ELL encoding");
    Exch<float>& x = X.ex32;
    Exch<double>& x64 = X.ex64;
    std::vector<uint32_t> ent;
    uint64_t nent = tot * kSlice;
    if (pack) {
        // Packed entries are relative (sublattice, cell delta, coupling index), so slices of a
        // periodic lattice away from the boundary planes come out identical: each distinct
        // slice block is stored once and the slice table points repeats at it.
        const bool share = !(c->flags & LLG_FLAG_NO_SLICE_SHARING);
        std::unordered_map<uint64_t, std::vector<uint32_t>> seen;  // block hash -> stored slices
        std::vector<uint32_t> blk;
        ent.reserve(share ? 1u << 16 : nent);
        uint64_t used = 0;
        uint32_t stored = 0;
        for (uint32_t s = 0; s < nsl; ++s) {
            const uint32_t len = slice[s].y;
            blk.assign((size_t)len * kSlice, 0u);
            for (uint32_t l = 0; l < kSlice; ++l) {
                const uint32_t d = s * kSlice + l;
                const uint32_t r = d < n ? ref_of[d] : 0;
                for (uint32_t q = 0; q < len; ++q) {
                    uint32_t w = pack_word(0, 0, dbits);  // zero coupling on itself
                    if (d < n && q < h.xadj[r + 1] - h.xadj[r]) {
                        const uint32_t qq = h.xadj[r] + q;
                        w = pack_word((int32_t)((int64_t)P.to_dev(h.adj[qq]) - (int64_t)d), idx[qq], dbits);
                    }
                    blk[pack_pos(q, l, len)] = w;
                }
            }
            uint64_t hsh = 1469598103934665603ull ^ len;  // FNV-1a over the block's words
            for (uint32_t w : blk) hsh = (hsh ^ w) * 1099511628211ull;
            bool found = false;
            if (share) {
                auto& cand = seen[hsh];
                for (uint32_t o : cand)
                    if (slice[o].y == len &&
                        std::memcmp(ent.data() + (size_t)slice[o].x * kSlice, blk.data(), blk.size() * 4) == 0) {
                        slice[s].x = slice[o].x;
                        found = true;
                        break;
                    }
                if (!found) cand.push_back(s);
            }
            if (!found) {
                slice[s].x = (uint32_t)used;
                ent.insert(ent.end(), blk.begin(), blk.end());
                used += len;
                ++stored;
            }
        }
        nent = used * kSlice;
        std::vector<float> d32(tuples.size() * nc);
        std::vector<double> d64(tuples.size() * nc);
        for (size_t t = 0; t < tuples.size(); ++t)
            for (int a = 0; a < nc; ++a) {
                d64[t * nc + a] = tuples[t].v[a];
                d32[t * nc + a] = (float)tuples[t].v[a];
            }
        SLLG_TRY(put(X, X.b, ent.data(), ent.size(), c->stream));
        SLLG_TRY(put(X, X.c, d32.data(), d32.size(), c->stream));
        SLLG_TRY(put(X, X.dict64, d64.data(), d64.size(), c->stream));
        x.fmt = FMT_SELL_PACK;
        x.ndict = (uint32_t)tuples.size();
        char buf[96];
        std::snprintf(buf, sizeof buf, "sell64x4-pack-t%u-dict%u-slices%uof%u", P.na, x.ndict, stored, nsl);
        X.encoding = buf;
    } else {
        ent.assign(nent, 0u);
        std::vector<float> v32((size_t)nc * nent, 0.0f);
        std::vector<double> v64((size_t)nc * nent, 0.0);
        for (uint32_t s = 0; s < nsl; ++s) {
            const uint32_t len = slice[s].y;
            for (uint32_t l = 0; l < kSlice; ++l) {
                const uint32_t d = s * kSlice + l;
                const uint32_t r = d < n ? ref_of[d] : 0;
                for (uint32_t q = 0; q < len; ++q) {
                    const size_t o = ((size_t)slice[s].x + q) * kSlice + l;
                    if (d < n && q < h.xadj[r + 1] - h.xadj[r]) {
                        const uint32_t qq = h.xadj[r] + q;
                        ent[o] = P.to_dev(h.adj[qq]);
                        for (int a = 0; a < nc; ++a) {
                            v64[(size_t)a * nent + o] = h.vals[(size_t)a * h.nnz + qq];
                            v32[(size_t)a * nent + o] = (float)h.vals[(size_t)a * h.nnz + qq];
                        }
                    } else {
                        ent[o] = d < n ? d : 0;
                    }
                }
            }
        }
        SLLG_TRY(put(X, X.b, ent.data(), ent.size(), c->stream));
        SLLG_TRY(put(X, X.c, v32.data(), v32.size(), c->stream));
        SLLG_TRY(put(X, X.dict64, v64.data(), v64.size(), c->stream));
        x.fmt = FMT_SELL_RAW;
        x.ndict = 0;
        X.encoding = P.na > 1 ? "sell64-u32-f32-sublattice-major" : "sell64-u32-f32";
    }
    SLLG_TRY(put(X, X.a, slice.data(), slice.size(), c->stream));
    x.nent = nent;
    x.ncell = ncell;
    x.dbits = pack ? dbits : 0;
    x64 = Exch<double>();
    fill_common(x64, h, n);
    x64.fmt = x.fmt;
    x64.ndict = x.ndict;
    x64.nent = nent;
    x64.ncell = ncell;
    x64.dbits = x.dbits;
    // Line mode replaces only the FP32 kernels' view; the FP64 view (energy, deterministic
    // field) keeps the packed encoding set up above.
    if (pack && !(c->flags & (LLG_FLAG_NO_LINE_MODE | LLG_FLAG_NO_SLICE_SHARING))) {
        uint32_t lstored = 0, lines_row = 0;
        uint32_t nfall = 0;
        bool done = false;
        for (uint32_t len : {64u, 16u})
            for (bool open : {false, true})
                if (!done && build_lines(c, ref_of, idx, tuples, len, open, lstored, lines_row, nfall)) {
                    char buf[128];
                    std::snprintf(buf, sizeof buf, "line%u%s-t%u-slices%uof%u-lines%u-packed%u", len, open ? "o" : "",
                                  P.na, lstored, nsl, lines_row, nfall);
                    if (x.tnw) {  // tile streams: slices per workgroup, most lines staged
                        const size_t l = std::strlen(buf);
                        std::snprintf(buf + l, sizeof buf - l, "-tile%ux%u", x.tnw, x.tumax);
                    }
                    X.encoding = buf;
                    done = true;
                }
        // read by a handle's own Heun steps only (RK and batches read lines or packed entries)
        if (!x.tnw && c->scheme == LLG_HEUN && c->own_stream) (void)build_blocks(c, idx, tuples);
    }
    return 0;
}

}  // namespace

// Point both views of a sliced-ELL store at its device buffers.
static void bind_sell(ExchStore& X) {
    Exch<float>& x = X.ex32;
    Exch<double>& x64 = X.ex64;
    x.slice = x64.slice = X.a.as<uint2>();
    x.ent = x64.ent = X.b.as<uint32_t>();
    x.dict = X.c.as<float>();
    x64.dict = X.dict64.as<double>();
    x.lslice = X.e.as<uint2>();
    x.lent = X.d.as<uint32_t>();
    x.tent = X.f.as<uint32_t>();
    x.tgrp = X.g.as<uint32_t>();
}

int encode_store(const llg_desc& d, std::shared_ptr<ExchStore>& out) {
    if (d.precision != LLG_FP32 || d.exch.format != LLG_EXCH_CSR)
        SLLG_FAIL(LLG_E_UNSUPPORTED, "couplings are encoded on the host for FP32 CSR only");
    auto X = std::make_shared<ExchStore>();
    X->device = d.device;
    X->prec = d.precision;
    X->n = d.n;
    X->host_only = true;
    llg_ctx c;  // what the encoder reads of a batch member; no device state
    c.own_stream = false;
    c.n = d.n;
    c.prec = d.precision;
    c.flags = d.flags;
    c.perm.na = 1;
    c.perm.ncell = d.n;
    X->perm = c.perm;
    c.xs = X;
    SLLG_TRY(build_exchange_fp32(&c, d.exch));
    out = X;
    return 0;
}

int upload_store(ExchStore& X, hipStream_t s) {
    for (auto& p : X.pending) {
        SLLG_TRY(p.first->alloc(p.second.size()));
        if (!p.second.empty())
            SLLG_HIP(hipMemcpyAsync(p.first->p, p.second.data(), p.second.size(), hipMemcpyHostToDevice, s));
    }
    SLLG_HIP(hipStreamSynchronize(s));
    bind_sell(X);
    return 0;
}

void keep_store(ExchStore& X) {
    X.pending.clear();
    X.pending.shrink_to_fit();
    X.host_only = false;
}

void drop_store(ExchStore& X) {
    for (auto& p : X.pending) p.first->release();
    bind_sell(X);
}

int build_exchange_fp32(llg_ctx* c, const llg_exchange& e) {
    ExchStore& X = *c->xs;
    SLLG_TRY(validate_and_copy(c, e));
    const HostExch& h = X.h;
    Exch<float>& x = X.ex32;
    fill_common(x, h, c->n);
    fill_common(X.ex64, h, c->n);
    X.encoding = "none";
    if (h.fmt == LLG_EXCH_CSR) {
        X.perm = csr_order(c, e.n_atoms);
        SLLG_TRY(build_sell(c));
        bind_sell(X);
    } else if (h.fmt == LLG_EXCH_DIA || h.fmt == LLG_EXCH_STENCIL) {
        std::vector<float> v32(h.vals.size());
        for (size_t q = 0; q < v32.size(); ++q) v32[q] = (float)h.vals[q];
        SLLG_TRY(upload(X.c, v32.data(), v32.size(), c->stream));
        SLLG_TRY(upload(X.dict64, h.vals.data(), h.vals.size(), c->stream));
        if (h.fmt == LLG_EXCH_DIA) {
            SLLG_TRY(upload(X.a, h.doff.data(), h.doff.size(), c->stream));
            x.doff = X.ex64.doff = X.a.as<int32_t>();
            X.encoding = "dia-f32";
        } else {
            SLLG_TRY(upload_stencil_tables(c));
            x.sent = X.ex64.sent = X.a.as<int4>();
            x.scount = X.ex64.scount = X.b.as<uint32_t>();
            X.encoding = h.per_row ? "stencil-rowvals-f32" : "stencil-shared-f32";
        }
        x.vals = X.c.as<float>();
        X.ex64.vals = X.dict64.as<double>();
    }
    release_host(X.h);
    return 0;
}

// Four-spin quartets: rows and (j, k, l) in the device order of this path; both exchange
// views (the kernels' precision and the FP64 one of the reductions) point at them.
int build_fourspin(llg_ctx* c, const llg_fourspin& f) {
    ExchStore& X = *c->xs;
    const uint32_t n = c->n;
    if (!f.xadj || !f.jkl) SLLG_FAIL(LLG_E_INVALID, "four-spin term without quartets");
    if (f.xadj[0] != 0 || f.xadj[n] != f.nq) SLLG_FAIL(LLG_E_INVALID, "four-spin row pointers do not span the quartets");
    for (uint32_t i = 0; i < n; ++i)
        if (f.xadj[i + 1] < f.xadj[i]) SLLG_FAIL(LLG_E_INVALID, "four-spin row pointers decrease at row %u", i);
    for (uint64_t q = 0; q < 3 * f.nq; ++q)
        if (f.jkl[q] >= n) SLLG_FAIL(LLG_E_INVALID, "four-spin quartet %llu names spin %u", (unsigned long long)(q / 3),
                                    f.jkl[q]);
    const Perm P = X.perm;
    std::vector<uint32_t> xadj(n + 1, 0);
    std::vector<uint4> q4(std::max<uint64_t>(1, f.nq));
    for (uint32_t d = 0; d < n; ++d) {
        const uint32_t i = P.to_ref(d);
        xadj[d + 1] = xadj[d] + (f.xadj[i + 1] - f.xadj[i]);
    }
    for (uint32_t d = 0; d < n; ++d) {
        const uint32_t i = P.to_ref(d);
        uint32_t o = xadj[d];
        for (uint32_t q = f.xadj[i]; q < f.xadj[i + 1]; ++q, ++o)
            q4[o] = make_uint4(P.to_dev(f.jkl[3 * (size_t)q]), P.to_dev(f.jkl[3 * (size_t)q + 1]),
                               P.to_dev(f.jkl[3 * (size_t)q + 2]), 0u);
    }
    SLLG_TRY(upload(X.fs_x, xadj.data(), xadj.size(), c->stream));
    SLLG_TRY(upload(X.fs_q, q4.data(), q4.size(), c->stream));
    X.ex32.fs_xadj = X.ex64.fs_xadj = X.fs_x.as<uint32_t>();
    X.ex32.fs_jkl = X.ex64.fs_jkl = X.fs_q.as<uint4>();
    X.ex32.fs_jq = (float)f.jq;
    X.ex64.fs_jq = f.jq;
    X.ex32.fs_div3 = X.ex64.fs_div3 = f.cpu_form ? 0 : 1;
    return 0;
}

}  // namespace sllg
