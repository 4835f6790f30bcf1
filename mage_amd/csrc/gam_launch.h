// gam_launch.h -- tiling of a launch's points over workgroups, and the two
// launch forms (one context, ensemble) of the step's kernels.
#pragma once
#include "gam_phys.h"
#include "gam_kernels.h"
#include <type_traits>

#define BX 64
#define BY 4

__device__ __forceinline__ bool in_box(const Box &b, int i, int j, int k)
{
    return i >= b.i0 && i <= b.i1 && j >= b.j0 && j <= b.j1 && k >= b.k0 && k <= b.k1;
}

#define THREAD_IJK(b)                                   \
    const int i = (b).i0 + blockIdx.x * BX + threadIdx.x; \
    const int j = (b).j0 + blockIdx.y * BY + threadIdx.y; \
    const int k = (b).k0 + blockIdx.z;                  \
    if (i > (b).i1 || j > (b).j1) return;

// XCD-aware tiling.  A launch covers box b row by row (a row = the points
// of one (j, k) along i) and cuts the rows, i fastest, into chunks of 256
// consecutive points, one per workgroup, so no lane idles however the row
// length falls against 64.  Row order, by ax1:
//   1: j fastest, then k;   2: k fastest, then j;
//   3: slabs of RB j-rows: j fastest within the slab, then k, then the
//      next slab -- the rows at j+1 and at k+1 are both at most RB rows
//      away, for kernels that read neighbours along j and along k.
// The hardware hands workgroup w to XCD w % 8; xcd_tile numbers the chunks
// so that each XCD takes runs of 2^xs consecutive ones: neighbouring chunks,
// which share stencil rows, meet in one L2, while the eight runs in flight
// stay side by side in memory.  Runs of 16 (XCD_RUN): on the 256x256x384
// shell the step takes 17.30 ms with runs of 4, 17.12 with 16 or 32, 17.19
// with 128, 17.40 with 1024 and 17.55 with one run of nb / 8 per XCD (eight
// far-apart streams, each a slower mix of DRAM pages); 96x96x128: 1.037,
// 1.027, 1.068, 1.32 and 1.09.
#define RB 8

// Division by a launch constant d: n / d = umulhi(n, m) >> s for
// 0 <= n < 2^31, with l = ceil(log2 d), m = ceil(2^(31 + l) / d), s = l - 1
// (m d exceeds 2^(31 + l) by less than d <= 2^l, so the quotient is never
// off); d = 1 has m = 0.  Four instructions instead of the ~18 of a 32-bit
// division, of which a point's index takes up to five.
struct FastDiv {
    unsigned d, m, s;
};
static inline FastDiv fast_div(unsigned d)
{
    FastDiv f = {d, 0u, 0u};
    if (d > 1) {
        unsigned l = 0;
        while ((1ul << l) < d) l++;
        f.m = (unsigned)(((1ul << (31 + l)) + d - 1) / d);
        f.s = l - 1;
    }
    return f;
}
__device__ __forceinline__ unsigned operator/(unsigned n, const FastDiv &f)
{
    return f.d == 1 ? n : __umulhi(n, f.m) >> f.s;
}

struct Tile {
    Box b;
    int ax1;
    int ni, nj, nk;   // extents
    FastDiv qi, q1, qt;   // by ni; by nj, nk or RB * nk (ax1 1, 2, 3); by the last slab's rows (ax1 3)
    int nb;           // chunks in all
    int ch;           // points per chunk (= threads per workgroup)
    int xs;           // log2 of an XCD's run of consecutive chunks
};

#define XCD_RUN 4     // log2 of the run length of a large launch
__device__ __forceinline__ int xcd_tile(int w, int xs)
{
    return ((w >> (3 + xs)) << (3 + xs)) + ((w & 7) << xs) + ((w >> 3) & ((1 << xs) - 1));
}
// Run length (log2) of a launch of nb chunks, and its workgroup count: a
// whole number of rounds of eight runs.
static inline int xcd_shift(long nb)
{
    int xs = 0;
    while (xs < XCD_RUN && (16L << xs) <= nb) xs++;
    return xs;
}
static inline unsigned xcd_grid(long nb, int xs)
{
    const long r = 8L << xs;
    return (unsigned)((nb + r - 1) / r * r);
}

// (j, k) of row R
__device__ __forceinline__ void tile_row(const Tile &t, unsigned R, int &j, int &k)
{
    int jj, kk;
    if (t.ax1 == 1) {
        kk = (int)(R / t.q1); jj = (int)R - kk * t.nj;
    } else if (t.ax1 == 2) {
        jj = (int)(R / t.q1); kk = (int)R - jj * t.nk;
    } else {
        const unsigned sb = R / t.q1, nfull = (unsigned)(t.nj / RB);
        if (sb < nfull) {
            const unsigned r = R - sb * (unsigned)(RB * t.nk);
            kk = (int)(r / RB);
            jj = (int)(sb * RB + (r % RB));
        } else {
            const unsigned r = R - nfull * (unsigned)(RB * t.nk);
            kk = (int)(r / t.qt);
            jj = (int)(nfull * RB + (r - (unsigned)kk * t.qt.d));
        }
    }
    j = t.b.j0 + jj;
    k = t.b.k0 + kk;
}

__device__ __forceinline__ bool tile_point(const Tile &t, int w, int &i, int &j, int &k)
{
    const int L = xcd_tile(w, t.xs);
    i = j = k = 0x40000000;
    if (L >= t.nb) return false;
    const unsigned p = (unsigned)L * (unsigned)t.ch + threadIdx.x + BX * threadIdx.y;
    if (p >= (unsigned)t.ni * (unsigned)(t.nj * t.nk)) return false;
    const unsigned R = p / t.qi;
    i = t.b.i0 + (int)(p - R * (unsigned)t.ni);
    tile_row(t, R, j, k);
    return true;
}

#define TILE_IJK(t)                  \
    int i, j, k;                     \
    if (!tile_point((t), (int)bi.x, i, j, k)) return;

static inline Tile tile_of(const Box &b, int ax1, int ch = BX * BY)
{
    Tile t;
    t.b = b;
    t.ax1 = ax1;
    t.ni = b.i1 - b.i0 + 1;
    t.nj = b.j1 - b.j0 + 1;
    t.nk = b.k1 - b.k0 + 1;
    t.qi = fast_div((unsigned)t.ni);
    t.q1 = fast_div((unsigned)(ax1 == 1 ? t.nj : ax1 == 2 ? t.nk : RB * t.nk));
    t.qt = fast_div((unsigned)(t.nj % RB ? t.nj % RB : 1));
    t.ch = ch;
    const long pts = (long)t.ni * t.nj * t.nk;
    t.nb = (int)((pts + ch - 1) / ch);
    t.xs = xcd_shift(t.nb);
    return t;
}

// A launch plan value of a chunk-tiled slot: the row order in its low 3
// bits, the chunk size (threads per workgroup) above them.
static inline int plan_ax(int v) { return v & 7; }
static inline int plan_chunk(int v) { return (v >> 3) == 1 ? 512 : (v >> 3) == 2 ? 128 : BX * BY; }
static inline dim3 tgrid(const Tile &t) { return dim3(xcd_grid(t.nb, t.xs)); }

static inline dim3 grid_of(const Box &b)
{
    return dim3((unsigned)((b.i1 - b.i0 + BX) / BX), (unsigned)((b.j1 - b.j0 + BY) / BY),
                (unsigned)(b.k1 - b.k0 + 1));
}

// ====================================================================
// Launch forms.  Every kernel of the step is a functor whose body takes its
// workgroup's block index bi.  k_one<F> runs F over its own grid (one
// context); k_ens<F> runs F for many contexts in one launch: the
// concatenated grid of the members, each member's workgroups starting at a
// multiple of 8 (so a member's chunk-to-XCD mapping is the same as in its
// own launch) and each with its own argument record.  A table after the
// header names the member of every run of 8 workgroups.
// ====================================================================
// Threads per workgroup of functor F: F::NT where it declares one, else 256.
template <class F, class = void> struct nthreads { static constexpr int v = BX * BY; };
template <class F> struct nthreads<F, std::void_t<decltype(F::NT)>> { static constexpr int v = F::NT; };

// Waves per SIMD that functor F's registers must allow (F::WPS; 1: no bound)
template <class F, class = void> struct nwaves { static constexpr int v = 1; };
template <class F> struct nwaves<F, std::void_t<decltype(F::WPS)>> { static constexpr int v = F::WPS; };

template <class F, class... A>
__global__ __launch_bounds__(nthreads<F>::v, nwaves<F>::v) void k_one(A... a)
{
    F{}(make_uint3(blockIdx.x, blockIdx.y, blockIdx.z), a...);
}

// Pointers read from an argument record are generic pointers to the
// compiler; every one of them addresses device (global) memory, and saying
// so lets it use global instead of flat loads and stores.
template <class T>
__device__ __forceinline__ const T &in_global(const T &v)
{
    return v;
}
template <class T>
__device__ __forceinline__ T *in_global(T *const &p)
{
    __attribute__((address_space(1))) T *q = (__attribute__((address_space(1))) T *)p;
    asm("" : "+s"(q));   // keeps the cast from folding back to a generic pointer
    return (T *)q;
}

// Call F with the record's fields, in order (passed by reference into the
// record, so that arrays in them are read where they lie).
template <class F, class... B>
__device__ __forceinline__ void pcall(const Pack<> &, uint3 bi, const B &...b)
{
    F{}(bi, in_global(b)...);
}
template <class F, class A0, class... A, class... B>
__device__ __forceinline__ void pcall(const Pack<A0, A...> &p, uint3 bi, const B &...b)
{
    pcall<F>(p.r, bi, b..., p.a0);
}

template <class F, class... A>
__global__ __launch_bounds__(nthreads<F>::v, nwaves<F>::v) void k_ens(const EnsHdr *__restrict__ h,
                                             const Pack<A...> *__restrict__ rec)
{
    const unsigned w = blockIdx.x;
    // owner of each run of 8 workgroups, stored right after the header
    const unsigned lo = reinterpret_cast<const unsigned short *>(h + 1)[w >> 3];
    const unsigned gx = h->gx[lo], gy = h->gy[lo], gz = h->gz[lo];
    unsigned l = w - h->wg0[lo];
    if (l >= gx * gy * gz) return;   // padding of the member's range
    uint3 bi;
    bi.x = l % gx;
    l /= gx;
    bi.y = l % gy;
    bi.z = l / gy;
    pcall<F>(rec[lo], bi);
}

template <class F, class... A>
static void launch_ens(hipStream_t s, const void *hdr, const void *rec, unsigned nwg, dim3 block)
{
    hipLaunchKernelGGL((k_ens<F, A...>), dim3(nwg), block, 0, s, (const EnsHdr *)hdr,
                       (const Pack<A...> *)rec);
}

// Batchable launch: issued at once, or appended to this thread's recorder.

template <class F, class... A>
static void launch_f(dim3 grid, dim3 block, hipStream_t s, A... a)
{
    if (std::vector<EnsLaunch> *rec = launch_recorder()) {
        const Pack<A...> p = make_pack(a...);
        EnsLaunch e;
        e.launch = &launch_ens<F, A...>;
        e.grid = grid;
        e.block = block;
        e.rec.resize(sizeof(p));
        memcpy(e.rec.data(), &p, sizeof(p));
        e.stream = s;
        e.mark = 0;
        e.ev = -1;
        rec->push_back(std::move(e));
        return;
    }
    hipLaunchKernelGGL((k_one<F, A...>), grid, block, 0, s, a...);
}
