// Dense piecewise-linear encoding (gfx950): the output of the upstream
// PiecewiseLinearEncoding module (rtdl_num_embeddings==0.0.12), restated.
//
// For feature f with n_f bins, bin b = the clamped right-sided search of x
// (as in the fused embedding) and frac = (x - e_b) * iw_b, the n_f
// components written at columns off_f .. off_f + n_f - 1 of the output row are
//     component k = 1 (k < b),  frac (k == b),  0 (k > b)
// which is upstream's clamp pattern: middle bins clamped to [0, 1], the first
// bin only above, the last bin only below, a single bin not at all (the
// component k == b is exactly the one no clamp touches).  A NaN x gives NaN
// components (torch.clamp propagates NaN).
//
// Backward: dx = g[off_f + b] * iw_b, plus g[off_f + b - 1] * iw_{b-1} when
// b > 0 and x == e_b (both neighbouring clamps pass at their bounds) -- the
// same two-term rule as the embedding's dx.
//
// By feature groups: one workgroup per (group of FG adjacent features, chunk of
// samples).  It keeps the group's edges and inverse widths in LDS (searched
// in global memory, a wave's 64 pairs touch up to 64 lines a step, which cost
// more than the searches) and walks its samples in blocks of R rows; a thread
// searches up to kEncPairs pairs of a block side by side, their x loaded a
// block ahead.  Forward: (b, frac) of the block's pairs go to LDS, then the
// threads walk the group's columns of a row in 16-byte vectors -- each finds the
// features of its columns once a block and writes them for every row -- so a
// store instruction covers 1 KiB of one row, and the next block is searched
// while the stores drain.  Bound by those stores, with the table set-up before
// them: 16384 x 128, 48 bins (403 MB written) by whole rows 95 us, by groups 91;
// 700 x 900, 100 bins 244 and 81.  Backward: one or two elements of g per pair,
// each in a line of its own, kEncPairs lines in flight a thread: by pairs 67 and
// 32 us there, by groups 49 and 21.
//
// Without groups, where the tables do not repay their set-up (enc_whole_rows,
// enc_grouped_backward): whole rows in small workgroups, forward; one thread
// per pair, backward.

#include <algorithm>

#include "ple_device.h"
#include "ple_internal.h"

namespace ple {
namespace {

constexpr int kEncRows = 8;      // samples of a workgroup by whole rows
constexpr int kEncBlock = 2 * kBlock;
constexpr int kEncPairs = 4;    // pairs of a block a thread searches, at most
constexpr int kEncBlockPairs = kEncPairs * kEncBlock;
constexpr size_t kEncLdsTarget = 72 * 1024;   // two workgroups per CU

struct EncArgs {
    const float *x, *edges, *iw;
    const int32_t *nbins, *offsets;
    const float *g;      // backward: grad_output [N, T]
    float *out;          // forward: [N, T]; backward: grad_x [N, F]
    int64_t N, NC;       // samples; samples a chunk
    int F, B, T;
    int FG, G, C, R;     // features a group, groups, chunks, rows a block
    int ro_edge, ro_iw, ro_nb, ro_off;   // LDS offsets (bytes); the (b, frac) pairs are first
};

__device__ __forceinline__ float enc_value(int k, int b, float frac) {
    // NaN x: every component NaN (frac is NaN exactly then)
    if (frac != frac) return frac;
    return k < b ? 1.0f : (k == b ? frac : 0.0f);
}

// The value at column p of sample n, whose feature is f or a later one; all
// from global memory.
__device__ __forceinline__ float enc_lookup(const EncArgs &a, int64_t n, int f, int p) {
    while (f + 1 < a.F && a.offsets[f + 1] <= p) ++f;
    const float v = a.x[n * a.F + f];
    const float *e = a.edges + static_cast<int64_t>(f) * (a.B + 1);
    const int b = find_bin(v, e, clamp_nbins(a.nbins[f], a.B));
    return enc_value(p - a.offsets[f], b, (v - e[b]) * a.iw[static_cast<int64_t>(f) * a.B + b]);
}

// The group's tables and its samples' bins, shared by the two kernels.
// TBL: edges and inverse widths in LDS (else read from global memory, see
// plan_encode).
template <bool TBL>
struct EncGroup {
    const EncArgs &a;
    int f0, nf;                  // first feature, features (with the next group's first ones: see the forward)
    int64_t n_begin, n_end;
    float *s_edge, *s_iw;
    int *s_nb, *s_off;
    float xv[kEncPairs];         // x of this thread's pairs of the next block

    __device__ __forceinline__ EncGroup(const EncArgs &args, unsigned char *lds) : a(args) {
        s_edge = reinterpret_cast<float *>(lds + a.ro_edge);
        s_iw = reinterpret_cast<float *>(lds + a.ro_iw);
        s_nb = reinterpret_cast<int *>(lds + a.ro_nb);
        s_off = reinterpret_cast<int *>(lds + a.ro_off);
    }
    __device__ __forceinline__ bool init(int halo) {
        int g, c;
        if (!decode_tile(blockIdx.x, a.G, a.C, g, c)) return false;
        f0 = g * a.FG;
        nf = min(a.F, f0 + a.FG + halo) - f0;
        n_begin = static_cast<int64_t>(c) * a.NC;
        n_end = min(a.N, n_begin + a.NC);
        return n_begin < n_end;
    }
    // x of the pairs of the block at row n0: pair u of thread t is pair
    // t + u kEncBlock of the block, sample-major (pairs past the block read x[0])
    __device__ __forceinline__ void load_x(int64_t n0) {
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) {
            const int i = threadIdx.x + u * kEncBlock;
            const int s = i / nf;
            const int64_t n = n0 + s;
            xv[u] = a.x[s < a.R && n < n_end ? n * a.F + f0 + (i - s * nf) : 0];
        }
    }
    __device__ __forceinline__ void stage() {
        const int tid = threadIdx.x;
        for (int i = tid; i < nf; i += kEncBlock) {
            s_nb[i] = clamp_nbins(a.nbins[f0 + i], a.B);
            s_off[i] = a.offsets[f0 + i];
        }
        if (tid == 0) s_off[nf] = f0 + nf < a.F ? a.offsets[f0 + nf] : a.T;
        if constexpr (TBL) {
            auto copy = [&](float *dst, const float *src, int count) __attribute__((always_inline)) {
                for (int i0 = tid; i0 < count; i0 += 8 * kEncBlock) {
                    float v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = src[min(i0 + u * kEncBlock, count - 1)];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (i0 + u * kEncBlock < count) dst[i0 + u * kEncBlock] = v[u];
                }
            };
            copy(s_edge, a.edges + static_cast<int64_t>(f0) * (a.B + 1), nf * (a.B + 1));
            copy(s_iw, a.iw + static_cast<int64_t>(f0) * a.B, nf * a.B);
        }
        __syncthreads();
    }
    __device__ __forceinline__ const float *edge_row(int fl) const {
        if constexpr (TBL) return s_edge + fl * (a.B + 1);
        else return a.edges + static_cast<int64_t>(f0 + fl) * (a.B + 1);
    }
    __device__ __forceinline__ const float *iw_row(int fl) const {
        if constexpr (TBL) return s_iw + fl * a.B;
        else return a.iw + static_cast<int64_t>(f0 + fl) * a.B;
    }
    // find_bin of the thread's pairs, a step of every search at a time; in
    // global memory until the wave's last one ends, as one feature may be much
    // wider than the others
    __device__ __forceinline__ void find(int (&fl)[kEncPairs], int (&b)[kEncPairs]) const {
        int lo[kEncPairs], hi[kEncPairs], n[kEncPairs];
        const float *e[kEncPairs];
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) {
            fl[u] = static_cast<int>((threadIdx.x + u * kEncBlock) % static_cast<unsigned>(nf));
            n[u] = s_nb[fl[u]];
            e[u] = edge_row(fl[u]);
            lo[u] = 0;
            hi[u] = n[u] + 1;
        }
        auto step = [&]() __attribute__((always_inline)) {
            bool more = false;
#pragma unroll
            for (int u = 0; u < kEncPairs; ++u) {
                const int mid = (lo[u] + hi[u]) >> 1;
                const bool live = lo[u] < hi[u];
                const bool below = xv[u] < e[u][min(mid, n[u])];
                hi[u] = live && below ? mid : hi[u];
                lo[u] = live && !below ? mid + 1 : lo[u];
                more |= lo[u] < hi[u];
            }
            return more;
        };
        if constexpr (TBL) {
            const int steps = 32 - __clz(a.B + 1);
            for (int t = 0; t < steps; ++t) step();
        } else {
            while (__any(step())) {}
        }
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) b[u] = clamp_bin(lo[u] - 1, n[u]);
    }
};

// Forward by whole rows: one workgroup per kEncRows samples, every feature
// searched in global memory, the threads walking the row's columns.  No set-up
// and many small workgroups, whose searches and stores overlap each other's.
template <bool V4>
__global__ __launch_bounds__(kBlock) void ple_encode_rows_kernel(EncArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int F = a.F, B = a.B, T = a.T;
    int *s_off = reinterpret_cast<int *>(lds);                 // [F + 1] column offsets
    int *s_bin = s_off + F + 1;                                // [kEncRows][F]
    float *s_frac = reinterpret_cast<float *>(s_bin + kEncRows * F);
    const int tid = threadIdx.x;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kEncRows;
    const int ns = static_cast<int>(min(static_cast<int64_t>(kEncRows), a.N - n0));

    for (int i = tid; i < F; i += kBlock) s_off[i] = a.offsets[i];
    if (tid == 0) s_off[F] = T;
    for (int i = tid; i < ns * F; i += kBlock) {
        const int s = i / F;
        const int f = i - s * F;
        const float v = a.x[(n0 + s) * F + f];
        const int n = clamp_nbins(a.nbins[f], B);
        const float *e = a.edges + static_cast<int64_t>(f) * (B + 1);
        const int b = find_bin(v, e, n);
        s_bin[i] = b;
        s_frac[i] = (v - e[b]) * a.iw[static_cast<int64_t>(f) * B + b];
    }
    __syncthreads();

    constexpr int W = V4 ? 4 : 1;
    for (int p0 = tid * W; p0 < T; p0 += kBlock * W) {
        // feature of column p0: last f with off[f] <= p0
        int lo = 0, hi = F;          // invariant: off[lo] <= p0 < off[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (s_off[mid] <= p0) lo = mid;
            else hi = mid;
        }
        int fq[W], kq[W];
        int f = lo;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const int p = min(p0 + j, T - 1);
            while (f + 1 < F && p >= s_off[f + 1]) ++f;
            fq[j] = f;
            kq[j] = p - s_off[f];
        }
        for (int s = 0; s < ns; ++s) {
            float v[W];
#pragma unroll
            for (int j = 0; j < W; ++j) v[j] = enc_value(kq[j], s_bin[s * F + fq[j]], s_frac[s * F + fq[j]]);
            store_out<PLE_DTYPE_F32, W>(a.out, (n0 + s) * T + p0, v);
        }
    }
}

// V4: 16-byte stores (T a multiple of 4).  A group owns the vectors whose
// first column is one of its features'; such a vector may end in up to three
// features of the next group, which this one searches too (a vector that goes
// past those, as behind features without columns, is looked up value by value).
template <bool V4, bool TBL>
__global__ __launch_bounds__(kEncBlock) void ple_encode_kernel(EncArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr int W = V4 ? 4 : 1;
    uint2 *s_pair = reinterpret_cast<uint2 *>(lds);   // [R][nf] {bin, frac bits}
    EncGroup<TBL> gr(a, lds);
    if (!gr.init(W - 1)) return;
    const int tid = threadIdx.x;
    const int nf = gr.nf, T = a.T;
    gr.load_x(gr.n_begin);
    gr.stage();
    const int nown = min(a.F - gr.f0, a.FG);
    const int c_begin = gr.f0 == 0 ? 0 : max(0, (gr.s_off[0] + W - 1) / W * W);
    const int c_end = gr.f0 + nown == a.F ? T : min(T, gr.s_off[nown]);
    // short rows: several rows side by side, sets of threads taking rows in turn
    const int vecs = max(1, (c_end - c_begin + W - 1) / W);
    const int sets = max(1, kEncBlock / vecs);
    const int s0 = sets > 1 ? tid / vecs : 0;
    const int v0 = sets > 1 ? (s0 < sets ? tid - s0 * vecs : vecs) : tid;   // (vecs: past the columns)

    for (int64_t n0 = gr.n_begin; n0 < gr.n_end; n0 += a.R) {
        const int ns = static_cast<int>(min(static_cast<int64_t>(a.R), gr.n_end - n0));
        int fl[kEncPairs], b[kEncPairs];
        gr.find(fl, b);
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) {
            const int i = tid + u * kEncBlock;
            const float frac = (gr.xv[u] - gr.edge_row(fl[u])[b[u]]) * gr.iw_row(fl[u])[b[u]];
            if (i < ns * nf) s_pair[i] = make_uint2(static_cast<uint32_t>(b[u]), __float_as_uint(frac));
        }
        if (n0 + a.R < gr.n_end) gr.load_x(n0 + a.R);
        __syncthreads();

        for (int p0 = c_begin + v0 * W; p0 < c_end; p0 += kEncBlock * W) {
            // feature of column p0: the last f with off[f] <= p0
            int lo = 0, hi = nf;          // invariant: off[lo] <= p0 < off[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (gr.s_off[mid] <= p0) lo = mid;
                else hi = mid;
            }
            if (V4 && gr.f0 + nf < a.F && p0 + W - 1 >= gr.s_off[nf]) {
                for (int s = s0; s < ns; s += sets) {
                    for (int j = 0; j < W; ++j)
                        a.out[(n0 + s) * T + p0 + j] = enc_lookup(a, n0 + s, gr.f0 + lo, p0 + j);
                }
                continue;
            }
            int fq[W], kq[W];
            int f = lo;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const int p = min(p0 + j, T - 1);
                while (f + 1 < nf && p >= gr.s_off[f + 1]) ++f;
                fq[j] = f;
                kq[j] = p - gr.s_off[f];
            }
            // the first and last columns' features cover the vector unless a
            // narrower feature lies between them
            const bool two = !V4 || ((fq[W / 2] == fq[0] || fq[W / 2] == fq[W - 1]) &&
                                     (fq[W > 1 ? 1 : 0] == fq[0] || fq[W > 1 ? 1 : 0] == fq[W - 1]));
            const uint2 *first = s_pair + fq[0], *last = s_pair + fq[W - 1];
            for (int s = s0; s < ns; s += sets) {
                float v[W];
                const uint2 pf = first[s * nf];
                const uint2 pl = V4 ? last[s * nf] : pf;
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    const uint2 p = fq[j] == fq[0] ? pf : pl;
                    v[j] = enc_value(kq[j], static_cast<int>(p.x), __uint_as_float(p.y));
                }
                if (!two) {
#pragma unroll
                    for (int j = 0; j < W; ++j) {
                        const uint2 p = s_pair[s * nf + fq[j]];
                        v[j] = enc_value(kq[j], static_cast<int>(p.x), __uint_as_float(p.y));
                    }
                }
                store_out<PLE_DTYPE_F32, W>(a.out, (n0 + s) * T + p0, v);
            }
        }
        __syncthreads();
    }
}

// One thread per (sample, feature) pair, everything from global memory: no
// set-up, and the round trips of one pair for a small call (see
// enc_grouped_backward).
__global__ __launch_bounds__(kBlock) void ple_encode_backward_pair_kernel(EncArgs a) {
    const int F = a.F, B = a.B, T = a.T;
    const int64_t pairs = a.N * F;
    for (int64_t p = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; p < pairs;
         p += static_cast<int64_t>(gridDim.x) * kBlock) {
        const int64_t n = p / F;
        const int f = static_cast<int>(p - n * F);
        const float v = a.x[p];
        const int nb = clamp_nbins(a.nbins[f], B);
        const float *e = a.edges + static_cast<int64_t>(f) * (B + 1);
        const float *iw = a.iw + static_cast<int64_t>(f) * B;
        const int b = find_bin(v, e, nb);
        // column of component b; columns outside [0, T) (offsets that do not
        // match n_bins) read nothing
        const int c = a.offsets[f] + b;
        const float *grow = a.g + n * T;
        float r = (c >= 0 && c < T) ? grow[c] * iw[b] : 0.0f;
        if (b > 0 && v == e[b] && c - 1 >= 0 && c - 1 < T) r = fmaf(grow[c - 1], iw[b - 1], r);
        a.out[p] = r;
    }
}

// Gradients of more bytes than this, the size of the memory-side cache, are
// read past the caches: plain loads take 5 to 15% longer there (22201 x 203,
// 1.6 GB: 104 us against 121).  Smaller ones may still be in that cache from
// the kernel that wrote them, where the hint would not find them (5281 x 568,
// 18 bins, 172 MB, just used: 58 us with it, 41 without; read cold: 58 and 57).
constexpr int64_t kEncStreamBytes = int64_t{1} << 28;
template <bool NT>
__global__ __launch_bounds__(kEncBlock) void ple_encode_backward_kernel(EncArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    EncGroup<true> gr(a, lds);
    if (!gr.init(0)) return;
    const int nf = gr.nf, T = a.T;
    gr.load_x(gr.n_begin);
    gr.stage();
    for (int64_t n0 = gr.n_begin; n0 < gr.n_end; n0 += a.R) {
        const int ns = static_cast<int>(min(static_cast<int64_t>(a.R), gr.n_end - n0));
        int fl[kEncPairs], b[kEncPairs];
        gr.find(fl, b);
        float r[kEncPairs];
        int64_t at[kEncPairs];
        bool ok[kEncPairs], edge[kEncPairs];
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) {
            const int i = threadIdx.x + u * kEncBlock;
            ok[u] = i < ns * nf;
            // column of component b; columns outside [0, T) (offsets that do
            // not match n_bins) read nothing
            const int c = gr.s_off[fl[u]] + b[u];
            const int64_t n = n0 + i / nf;
            at[u] = n * T + c;
            edge[u] = ok[u] && b[u] > 0 && gr.xv[u] == gr.edge_row(fl[u])[b[u]] && c - 1 >= 0 && c - 1 < T;
            const bool in = ok[u] && c >= 0 && c < T;
            const float *gp = a.g + (in ? at[u] : 0);
            const float gv = NT ? __builtin_nontemporal_load(gp) : *gp;
            r[u] = in ? gv * gr.iw_row(fl[u])[b[u]] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u)
            if (edge[u]) r[u] = fmaf(a.g[at[u] - 1], gr.iw_row(fl[u])[b[u] - 1], r[u]);
        if (n0 + a.R < gr.n_end) gr.load_x(n0 + a.R);
#pragma unroll
        for (int u = 0; u < kEncPairs; ++u) {
            const int i = threadIdx.x + u * kEncBlock;
            const int s = i / nf;
            if (ok[u]) a.out[(n0 + s) * a.F + gr.f0 + (i - s * nf)] = r[u];
        }
    }
}

// Features whose tables fit the LDS of a group's workgroup (beside the pairs
// of a forward's block), less the halo; 0: not one feature's.
int64_t enc_table_features(int64_t B, int halo, bool forward) {
    const size_t pair_bytes = forward ? 8 * static_cast<size_t>(kEncBlockPairs) : 0;
    const size_t per_f = 4 * (2 * static_cast<size_t>(B) + 3);   // edges, inverse widths, bin count, offset
    const size_t room = kEncLdsTarget - pair_bytes - 64;
    return std::max<int64_t>(static_cast<int64_t>(room / per_f) - halo, 0);
}

// Entries of the tables per bin in use (all features' have the widest one's size).
int64_t enc_padding(int64_t F, int64_t B, int64_t T) { return F * B / T; }

// Whether the forward leaves tables that are mostly padding in global memory:
// LDS would fill up with a few features' and leave groups of a few columns (817
// x 431, one of 1422 bins among 6: 77 us with tables in LDS, 17 without).
bool enc_global_tables(int64_t F, int64_t B, int64_t T, int halo) {
    return F > 64 && enc_table_features(B, halo, true) < 8 && enc_padding(F, B, T) >= 8;
}

// Features a group: as many as two workgroups' LDS a CU hold (fewer where the
// samples alone do not fill the CUs).  Chunks: one round of workgroups, rounded
// down (a few workgroups of a second round take as long as the first: 11297 x
// 1744, 20 bins: 579 us rounded up, 423 down), their blocks all of one size.
// Rows a block: kEncPairs pairs a thread at most; times the features of a row
// never more than kEncBlockPairs, the pairs that the threads search.  halo:
// further features a group searches.  False: the tables stay in global memory,
// as not one feature's fit LDS, or as they are mostly padding
// (enc_global_tables).
bool plan_encode(EncArgs &a, int halo, bool forward, size_t &lds) {
    const int cus = device_cu_count();
    int64_t fg = enc_table_features(a.B, halo, forward);
    const bool tbl = fg > 0 && !(forward && enc_global_tables(a.F, a.B, a.T, halo));
    if (!tbl) fg = 512;
    fg = std::min<int64_t>({fg, a.F, kEncBlockPairs - halo});
    const int64_t rows = (a.N + 15) / 16;
    while (fg > 16 && (a.F + fg - 1) / fg * rows < cus) fg = (fg + 1) / 2;
    a.FG = static_cast<int>(std::max<int64_t>(1, fg));
    a.G = (a.F + a.FG - 1) / a.FG;
    const int nfh = std::min(a.F, a.FG + halo);
    const int64_t r_max =
        std::max<int64_t>(1, std::min<int64_t>(kEncBlockPairs / nfh, (a.N * a.G + cus - 1) / cus));
    const int64_t round = 2 * static_cast<int64_t>(cus) / a.G;
    const int64_t c = std::max<int64_t>(1, std::min(round, (a.N + r_max - 1) / r_max));
    const int64_t per = (a.N + c - 1) / c;                  // samples a chunk, in blocks of one size
    const int64_t blocks = (per + r_max - 1) / r_max;
    a.R = static_cast<int>((per + blocks - 1) / blocks);
    a.NC = a.R * blocks;
    a.C = static_cast<int>((a.N + a.NC - 1) / a.NC);
    size_t off = forward ? 8 * static_cast<size_t>(a.R) * nfh : 0;
    auto take = [&](int &field, size_t bytes) {
        field = static_cast<int>(off);
        off = align_up(off + bytes, 16);
    };
    take(a.ro_edge, tbl ? 4 * static_cast<size_t>(nfh) * (a.B + 1) : 0);
    take(a.ro_iw, tbl ? 4 * static_cast<size_t>(nfh) * a.B : 0);
    take(a.ro_nb, 4 * static_cast<size_t>(nfh));
    take(a.ro_off, 4 * static_cast<size_t>(nfh + 1));
    lds = off;
    return tbl;
}

// The most features the forward takes: the whole-row kernel's LDS holds every
// feature's offset and kEncRows pairs.
constexpr size_t enc_rows_lds_bytes(int F) {
    return 4 * static_cast<size_t>(F + 1) + 8 * static_cast<size_t>(kEncRows) * F;
}
constexpr int kEncMaxFeatures = 2409;
static_assert(enc_rows_lds_bytes(kEncMaxFeatures) <= kLdsMax && enc_rows_lds_bytes(kEncMaxFeatures + 1) > kLdsMax);

EncArgs enc_args(const EncodeRequest &r) {
    EncArgs a{};
    a.x = r.x; a.edges = r.edges; a.iw = r.iw; a.nbins = r.nbins; a.offsets = r.offsets;
    a.g = r.g; a.out = r.out;
    a.N = r.N; a.F = static_cast<int>(r.F); a.B = static_cast<int>(r.B); a.T = static_cast<int>(r.T);
    return a;
}

// Rows of whole 16-byte vectors.
bool enc_vectors(const EncodeRequest &r) { return r.T % 4 == 0 && reinterpret_cast<uintptr_t>(r.out) % 16 == 0; }

template <typename K>
int enc_launch(K kernel, const EncArgs &a, int halo, size_t lds, hipStream_t s) {
    // (plan_encode's bound: pairs past it would not be searched)
    if (static_cast<int64_t>(a.R) * std::min(a.F, a.FG + halo) > kEncBlockPairs) return PLE_E_UNSUPPORTED;
    const int64_t grid = kNumXcd * tiles_per_xcd(a.G, a.C);
    if (grid > INT32_MAX) return PLE_E_TOO_LARGE;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kEncBlock), lds, s, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? PLE_OK : static_cast<int>(e);
}

// Whether the forward goes by whole rows instead of feature groups (either
// way the same values; times in us, whole rows / groups).
//  * Where LDS holds few features' tables, groups are narrow, most of all when
//    one wide feature pads the others' tables: 16384 x 500, one of 1024 bins
//    among 4: 149 / 890; 16384 x 64, 2 to 235 bins: 57 / 72; 10019 x 160, 217
//    bins: 339 / 402.  Under 32 features; 16 where the row's own searches are
//    many (10687 x 464, one of 341 bins among 11: 152 / 105) or its stores
//    single columns (15937 x 144, one of 304 bins among 19: 90 / 74).  Few
//    samples by whole rows leave CUs idle, which costs more (1024 x 500, 1024
//    bins: 1180 / 610), though less than much padding does from 2048 samples
//    on (3292 x 1074, one of 1040 bins among 10: 111 / 179; but 2339 x 382, up
//    to 1241 bins, 241 on average: 498 / 287), and from 384 to 65536 samples
//    of up to 128 features (444 x 49, one of 3938 bins among 22: 25 / 53; 11907
//    x 118, one of 111 among 1: 16 / 25; but 145625 x 102, one of 96 among 2:
//    193 / 127).
//  * Up to 64 features, a row's searches take a round or two of a workgroup's
//    threads and the groups' tables do not repay their set-up: 50000 x 10, 73
//    bins: 42 / 53; 256 x 8, 48 bins: 5.2 / 7.2; at 16384 x 127, 47 bins, 142 /
//    108.  Not where many samples have few bins, or rows too short for a
//    workgroup (66354 x 26, 15 bins: 41 / 30; 81000 x 4, 230 columns: 30 / 23);
//    nor for long rows of few samples (816 x 42, 530 bins: 51 / 29), of under
//    4096 if they go by single columns (1246 x 62, 497 bins: 130 / 43), unless
//    the tables are padding (826 x 26, one of 3012 bins among 12: 12 / 16).
// (Launches count threads in 32 bits, kBlock for kEncRows samples.)
bool enc_whole_rows(const EncodeRequest &r, int halo) {
    if (r.N > (int64_t{1} << 26)) return false;
    const bool filled = r.N >= 4096;   // two workgroups for each of 256 CUs
    const int64_t padding = enc_padding(r.F, r.B, r.T);
    const int64_t fit = enc_table_features(r.B, halo, true);
    const bool narrow = r.F <= 256 && halo > 0;
    if (filled && fit < std::min<int64_t>(r.F, narrow ? 32 : 16)) return true;
    if (r.N >= 2048 && padding >= 8 && fit < std::min<int64_t>(r.F, narrow ? 32 : 8)) return true;
    if (r.F <= 128 && padding >= 8 && r.N >= 384 && r.N <= 65536) return true;
    if (r.F > 64 || (r.N > 16384 && (r.T < 256 || r.B <= 16))) return false;
    return filled || r.T <= 1280 || r.N >= (padding >= 4 ? 768 : (halo > 0 ? 1536 : 4096));
}

// Whether the backward goes by feature groups (times in us, groups / one
// thread per pair): from 2^21 pairs on (12509 x 324, one of 330 bins among 30:
// 89 / 163; 270000 x 15, 2 bins: 24 / 25), from 2^20 of at least 128 features
// (2821 x 542, one of 115 bins among 5: 22 / 33), or from 2^19 with a gradient
// of 64 MB of at least 32 features (1921 x 448, 143 bins: 26 / 44; but 117000 x
// 5: 17 / 13, and 16 MB, 110000 x 6: 11 / 9).  Below, the tables' set-up costs
// more than it saves (3000 x 5, 256 bins: 6.9 / 4.0), as it does where LDS holds
// but a few features' (8000 x 158, 3220 bins: 42 / 31; none at all, 16384 x 64,
// 8000 bins, searched from global memory: 26 / 14).
bool enc_grouped_backward(const EncodeRequest &r) {
    const int64_t pairs = r.N * r.F, fit = enc_table_features(r.B, 0, false);
    if (fit == 0 || pairs < (1 << 19)) return false;
    if (pairs >= (1 << 21)) return true;
    if (fit < 4) return false;
    return (r.F >= 128 && pairs >= (1 << 20)) || (r.F >= 32 && r.N * r.T >= (1 << 24));
}

}  // namespace

int encode_run(const EncodeRequest &r) {
    if (r.T < 1 || r.T > INT32_MAX / 2) return PLE_E_TOO_LARGE;
    if (r.F > kEncMaxFeatures) return PLE_E_UNSUPPORTED;
    EncArgs a = enc_args(r);
    const bool v4 = enc_vectors(r);
    const int halo = v4 ? 3 : 0;
    if (enc_whole_rows(r, halo)) {
        const dim3 grid(static_cast<unsigned>((r.N + kEncRows - 1) / kEncRows));
        const size_t lds = enc_rows_lds_bytes(a.F);
        if (v4) hipLaunchKernelGGL(ple_encode_rows_kernel<true>, grid, dim3(kBlock), lds, r.stream, a);
        else hipLaunchKernelGGL(ple_encode_rows_kernel<false>, grid, dim3(kBlock), lds, r.stream, a);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? PLE_OK : static_cast<int>(e);
    }
    size_t lds;
    const bool tbl = plan_encode(a, halo, true, lds);
    if (v4) {
        return tbl ? enc_launch(ple_encode_kernel<true, true>, a, halo, lds, r.stream)
                   : enc_launch(ple_encode_kernel<true, false>, a, halo, lds, r.stream);
    }
    return tbl ? enc_launch(ple_encode_kernel<false, true>, a, halo, lds, r.stream)
               : enc_launch(ple_encode_kernel<false, false>, a, halo, lds, r.stream);
}

int encode_backward_run(const EncodeRequest &r) {
    if (r.T < 1 || r.T > INT32_MAX / 2) return PLE_E_TOO_LARGE;
    EncArgs a = enc_args(r);
    if (!enc_grouped_backward(r)) {
        const int64_t blocks = std::min((r.N * r.F + kBlock - 1) / kBlock, static_cast<int64_t>(device_cu_count()) * 32);
        hipLaunchKernelGGL(ple_encode_backward_pair_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0,
                           r.stream, a);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? PLE_OK : static_cast<int>(e);
    }
    size_t lds;
    plan_encode(a, 0, false, lds);
    return 4 * r.N * r.T > kEncStreamBytes ? enc_launch(ple_encode_backward_kernel<true>, a, 0, lds, r.stream)
                                           : enc_launch(ple_encode_backward_kernel<false>, a, 0, lds, r.stream);
}

int encode_plan_info(const EncodeRequest &r, bool backward, ple_encode_plan_info_t *info) {
    if (r.T < 1 || r.T > INT32_MAX / 2) return PLE_E_TOO_LARGE;
    if (!backward && r.F > kEncMaxFeatures) return PLE_E_UNSUPPORTED;
    *info = ple_encode_plan_info_t{};
    EncArgs a = enc_args(r);
    const int halo = !backward && enc_vectors(r) ? 3 : 0;
    if (backward ? !enc_grouped_backward(r) : enc_whole_rows(r, halo)) return PLE_OK;
    size_t lds;
    info->lds_tables = plan_encode(a, halo, !backward, lds) ? 1 : 0;
    info->features_per_group = a.FG;
    info->features_searched = std::min(a.F, a.FG + halo);
    info->groups = a.G;
    info->chunks = a.C;
    info->rows_per_block = a.R;
    info->pairs_per_block = kEncBlockPairs;
    info->lds_bytes = lds;
    return PLE_OK;
}

}  // namespace ple
