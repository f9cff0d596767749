// HIP kernels for gfx950 (CDNA4): grouped sub-block permutes, grouped FP64
// MFMA GEMM (and FP32-MFMA hi/lo split variant), trace/normalise, leg
// scaling, grouped parallel-order Jacobi eigensolver for small symmetric
// matrices, column norms, deterministic pseudo-random fill.
//
// Every kernel here is launched with its grid checked on the host against
// the descriptors it reads (see kernels.h); no kernel uses atomics, so every
// reduction has a fixed order and results are bitwise reproducible run to
// run and alone vs batched.
#include "kernels.h"

#include <hip/hip_ext.h>

#include <condition_variable>
#include <map>
#include <mutex>

#include <algorithm>
#include <vector>

namespace tnr {

// Pointers taken from descriptor arrays are generic to the compiler, so plain
// reads through them become flat loads, which also count in lgkmcnt (an LDS
// wait would then also wait for them).  A global-address-space view makes
// them global loads, tracked by vmcnt alone.
using gconst_double = const __attribute__((address_space(1))) double;
using gmut_double = __attribute__((address_space(1))) double;
__device__ __forceinline__ gconst_double* as_global(const double* p) { return (gconst_double*)p; }
__device__ __forceinline__ gmut_double* as_global(double* p) { return (gmut_double*)p; }

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ permute
// dst[sum i_k dstr_k] = src[sum i_k sstr_k] * w0[i_wleg0] * w1[i_wleg1]
// One chunk of COPY_CHUNK consecutive elements (destination order) of one job
// per workgroup iteration.  What bounds it is decoding the index: the host
// merges dims that stay neighbours, divisions are multiplications by
// precomputed reciprocals, offsets take 32 bits where they fit, and the code
// is unrolled for the number of dims left.  Four elements a thread, whose loads
// are issued together: small jobs spread over more CUs than with eight or
// sixteen.  A wave finds its job 64 entries at a time.
template <int ND, class I>
__device__ __forceinline__ void copy_chunk(const CopyDesc& D, uint32_t base, int t) {
    constexpr int G = COPY_CHUNK / 256;
    const int ndim = D.nd;
    uint32_t cnt = 1;
#pragma unroll
    for (int q = 0; q < ND; ++q) cnt *= q < ndim ? (uint32_t)D.dim[q] : 1u;
    gconst_double* src = as_global(D.src);
    gmut_double* dst = as_global(D.dst);
    uint32_t r[G], iw0[G], iw1[G];
    I so[G], dof[G];
    bool ok[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        r[g] = base + (uint32_t)(t + 256 * g);
        ok[g] = r[g] < cnt;
        if (!ok[g]) r[g] = 0;   // element 0: a valid address, not stored
        so[g] = dof[g] = 0;
        iw0[g] = iw1[g] = 0;
    }
#pragma unroll
    for (int q = 0; q < ND; ++q) {
        if (q >= ndim) continue;
        const uint32_t dim = (uint32_t)D.dim[q], mul = D.mul[q];
        const int sh = D.sh[q];
        const I ss = (I)D.sstr[q], ds = (I)D.dstr[q];
        const bool last = q + 1 == ndim, w0 = D.wleg[0] == q, w1 = D.wleg[1] == q;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t n = last ? 0u : __umulhi(r[g], mul) >> sh;
            const uint32_t i = r[g] - n * dim;
            r[g] = n;
            so[g] += (I)i * ss;
            dof[g] += (I)i * ds;
            if (w0) iw0[g] = i;
            if (w1) iw1[g] = i;
        }
    }
    double v[G];
#pragma unroll
    for (int g = 0; g < G; ++g) v[g] = src[so[g]];
    if (D.w[0])
#pragma unroll
        for (int g = 0; g < G; ++g) v[g] *= as_global(D.w[0])[iw0[g]];
    if (D.w[1])
#pragma unroll
        for (int g = 0; g < G; ++g) v[g] *= as_global(D.w[1])[iw1[g]];
#pragma unroll
    for (int g = 0; g < G; ++g)
        if (ok[g]) dst[dof[g]] = v[g];
}

__global__ __launch_bounds__(256) void k_copy(const CopyDesc* __restrict__ descs, int nd,
                                              int64_t chunks) {
    const int t = threadIdx.x, lane = t & 63;
    for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        // the last job that starts at or before chunk c
        int lo = 0, n = nd;
        while (n > 1) {
            const int step = (n + 63) / 64, at = lane * step;
            const bool le = at < n && descs[lo + min(at, n - 1)].start <= c;
            const int k = __builtin_amdgcn_readfirstlane(__popcll(__ballot(le))) - 1;
            lo += k * step;
            n = min(step, n - k * step);
        }
        const CopyDesc& D = descs[lo];
        const uint32_t base = (uint32_t)(c - D.start) * COPY_CHUNK;
        if (D.wide) copy_chunk<MAXLEG, int64_t>(D, base, t);
        else if (D.nd <= 2) copy_chunk<2, uint32_t>(D, base, t);
        else if (D.nd <= 4) copy_chunk<4, uint32_t>(D, base, t);
        else copy_chunk<MAXLEG, uint32_t>(D, base, t);
    }
}

// ------------------------------------------------------- tiled transpose
// One 64 x 64 tile per workgroup iteration: 256 threads read 4 rows of 64
// consecutive source elements per pass (coalesced), and write 4 rows of 64
// consecutive destination elements per pass (coalesced) through LDS.
__global__ __launch_bounds__(256) void k_transpose(const TransDesc* __restrict__ descs, int nd,
                                                   int64_t tiles) {
    // 4096 doubles of LDS hold `sub` sub-tiles of tx (along n0) by ty (along
    // n1), one per consecutive batch index; rows padded by one element
    __shared__ double buf[4096 + 64 * 16];
    __shared__ int64_t soff[64], doff[64];           // batch offsets per sub-tile (-1: none)
    const int t = threadIdx.x;
    int lo = 0;
    for (int64_t tid = blockIdx.x; tid < tiles; tid += gridDim.x) {
        // tiles come in increasing order: continue the search from the last
        // job (usually the same one or the next)
        if (descs[lo].tile_start > tid) lo = 0;
        if (lo + 1 < nd && descs[lo + 1].tile_start <= tid) {
            int hi = nd - 1;
            while (lo < hi) {
                int mid = (lo + hi + 1) >> 1;
                if (descs[mid].tile_start <= tid) lo = mid; else hi = mid - 1;
            }
        }
        const TransDesc& D = descs[lo];
        const int tx = D.tx, ty = D.ty, sub = D.sub, pitch = tx + 1;
        const int lx = __ffs(tx) - 1, ly = __ffs(ty) - 1, la = lx + ly;   // log2 extents
        // a job has fewer than 2^31 tiles and batch entries: 32-bit decode
        int r = (int)(tid - D.tile_start);
        const int i0 = (r % D.t0) * tx;
        r /= D.t0;
        const int i1 = (r % D.t1) * ty;
        r /= D.t1;
        const int b0 = r * sub;                     // first batch index of this tile
        __syncthreads();                            // previous tile done with buf / offsets
        if (t < sub) {
            const int bi = b0 + t;
            int64_t so = -1, dof = -1;
            if (bi < D.nb) {
                int q = bi;
                so = 0;
                dof = 0;
                for (int kk = 0; kk < TR_BATCH; ++kk) {
                    const int ik = q % D.bdim[kk];
                    q /= D.bdim[kk];
                    so += (int64_t)ik * D.bs[kk];
                    dof += (int64_t)ik * D.bd[kk];
                }
            }
            soff[t] = so;
            doff[t] = dof;
        }
        __syncthreads();
        gconst_double* src = as_global(D.src);
        gmut_double* dst = as_global(D.dst);
        // all 16 loads of this thread are issued before the first LDS store
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {              // x along n0 (source-contiguous)
            const int e = t + 256 * u;
            const int s = e >> la, rem = e & ((1 << la) - 1), j = rem >> lx, x = rem & (tx - 1);
            const int a = i0 + x, c = i1 + j;
            const int64_t so = soff[s];
            v[u] = (so >= 0 && a < D.n0 && c < D.n1) ? src[so + a + (int64_t)c * D.ss1] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = t + 256 * u;
            const int s = e >> la, rem = e & ((1 << la) - 1), j = rem >> lx, x = rem & (tx - 1);
            buf[s * ty * pitch + j * pitch + x] = v[u];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 16; ++u) {              // x along n1 (destination-contiguous)
            const int e = t + 256 * u;
            const int s = e >> la, rem = e & ((1 << la) - 1), j = rem >> ly, x = rem & (ty - 1);
            v[u] = buf[s * ty * pitch + x * pitch + j];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = t + 256 * u;
            const int s = e >> la, rem = e & ((1 << la) - 1), j = rem >> ly, x = rem & (ty - 1);
            const int a = i0 + j, c = i1 + x;
            const int64_t dof = doff[s];
            if (dof >= 0 && a < D.n0 && c < D.n1) dst[dof + c + (int64_t)a * D.ds0] = v[u];
        }
    }
}

// --------------------------------------------------------------- FP64 GEMM
// Output tile BM x BN per 256-thread workgroup; 4 waves as 2 x 2, each wave
// owning (BM/2) x (BN/2) = MI x NI blocks of v_mfma_f64_16x16x4_f64 per
// k-step of 4.  The k order of every output element is the same for all
// tile shapes, so results do not depend on the shape chosen.  Operand lane
// layout of the 16x16x4 MFMAs (measured on gfx950): A[i=l%16][k=l/16],
// B[k=l/16][j=l%16]; result register r of lane l holds
//   f64: D[i = l/16 + 4r][j = l%16]   (rows interleaved)
//   f32: D[i = 4(l/16) + r][j = l%16] (rows contiguous).
constexpr int BK = 16;

__device__ __forceinline__ int find_desc_gemm(const GemmDesc* d, int n, int64_t t) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (d[mid].tile_start <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

struct TileCoord {
    int m0, n0, kbeg, kend, kz;
};

// Profiling: the algorithmic flops of one output tile (its rows and columns
// inside M x N, its K range) added to a device counter, so only problems
// that actually ran are counted (a finished problem's tiles return before
// this).  The counts are integers, so the sum does not depend on order.
template <int BM, int BN>
__device__ __forceinline__ void count_tile_flops(unsigned long long* ctr, const GemmDesc& g,
                                                 const TileCoord& tc) {
    if (!ctr || threadIdx.x != 0) return;
    const long long rows = min(BM, g.M - tc.m0), cols = min(BN, g.N - tc.n0);
    const long long kk = tc.kend - tc.kbeg;
    if (rows > 0 && cols > 0 && kk > 0) atomicAdd(ctr, (unsigned long long)(2 * rows * cols * kk));
}

template <int BM, int BN>
__device__ __forceinline__ TileCoord tile_coord(const GemmDesc& g, int64_t local) {
    TileCoord c;
    // Workgroups go round-robin over the 8 XCDs (each with its own L2): the
    // physical ids of one residue class mod 8 get one contiguous range of
    // the tile order, which walks GROUP_M tile rows at a time (then the next
    // tile column), so the tiles an XCD runs together share A and B slices.
    // A bijection on each K chunk's tiles; every tile's arithmetic is the
    // same wherever it runs.
    constexpr int NXCD = 8, GROUP_M = 8;
    const int64_t per_k = (int64_t)g.tiles_m * g.tiles_n;
    const int kz = (int)(local / per_k);
    int64_t r = local - (int64_t)kz * per_k;
    const int64_t F = per_k / NXCD;
    if (r < NXCD * F) r = (r % NXCD) * F + r / NXCD;
    const int64_t width = (int64_t)GROUP_M * g.tiles_n;
    const int64_t grp = r / width, inner = r - grp * width;
    const int first_m = (int)(grp * GROUP_M);
    const int gsz = min(g.tiles_m - first_m, GROUP_M);
    const int tm = first_m + (int)(inner % gsz);
    const int tn = (int)(inner / gsz);
    c.m0 = tm * BM;
    c.n0 = tn * BN;
    if (g.ksplit > 1) {           // one K chunk per workgroup
        c.kbeg = kz * g.kchunk;
        c.kend = min(g.K, (kz + 1) * g.kchunk);
    } else {
        c.kbeg = 0;
        c.kend = g.K;
    }
    c.kz = kz;
    return c;
}

// global -> registers: the tile's BM x KB slab of op(A), KB BM / NT values
// per thread of an NT-thread workgroup
template <int BM, int NT, int KB>
__device__ __forceinline__ void load_a(const GemmDesc& g, int m0, int k0, int t,
                                       double (&ra)[KB * BM / NT]) {
    constexpr int R = KB * BM / NT;
    gconst_double* A = as_global(g.A);
    if (!g.ta) {  // A[i + k*lda], M x K: thread -> (i, k-group)
        const int i = m0 + (t % BM), kk = t / BM;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = k0 + kk + (NT / BM) * r;
            ra[r] = (i < g.M && k < g.K) ? A[(int64_t)i + (int64_t)k * g.lda] : 0.0;
        }
    } else {      // stored K x M: A[k + i*lda]
        const int kk = t % KB, i0 = t / KB;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = m0 + i0 + (NT / KB) * r, k = k0 + kk;
            ra[r] = (i < g.M && k < g.K) ? A[(int64_t)k + (int64_t)i * g.lda] : 0.0;
        }
    }
}

template <int BM, int NT, int KB>
__device__ __forceinline__ void store_a(const GemmDesc& g, int t, const double (&ra)[KB * BM / NT],
                                        double (*As)[BM + 1]) {
    constexpr int R = KB * BM / NT;
    if (!g.ta) {
        const int i = t % BM, kk = t / BM;
#pragma unroll
        for (int r = 0; r < R; ++r) As[kk + (NT / BM) * r][i] = ra[r];
    } else {
        const int kk = t % KB, i0 = t / KB;
#pragma unroll
        for (int r = 0; r < R; ++r) As[kk][i0 + (NT / KB) * r] = ra[r];
    }
}

template <int BN, int NT, int KB>
__device__ __forceinline__ void load_b(const GemmDesc& g, int n0, int k0, int t,
                                       double (&rb)[KB * BN / NT]) {
    constexpr int R = KB * BN / NT;
    gconst_double* B = as_global(g.B);
    if (!g.tb) {  // B[k + j*ldb], K x N
        const int kk = t % KB, j0 = t / KB;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int j = n0 + j0 + (NT / KB) * r, k = k0 + kk;
            rb[r] = (j < g.N && k < g.K) ? B[(int64_t)k + (int64_t)j * g.ldb] : 0.0;
        }
    } else {      // stored N x K: B[j + k*ldb]
        const int j = n0 + (t % BN), kk = t / BN;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = k0 + kk + (NT / BN) * r;
            rb[r] = (j < g.N && k < g.K) ? B[(int64_t)j + (int64_t)k * g.ldb] : 0.0;
        }
    }
}

template <int BN, int NT, int KB>
__device__ __forceinline__ void store_b(const GemmDesc& g, int t, const double (&rb)[KB * BN / NT],
                                        double (*Bs)[BN + 1]) {
    constexpr int R = KB * BN / NT;
    if (!g.tb) {
        const int kk = t % KB, j0 = t / KB;
#pragma unroll
        for (int r = 0; r < R; ++r) Bs[kk][j0 + (NT / KB) * r] = rb[r];
    } else {
        const int j = t % BN, kk = t / BN;
#pragma unroll
        for (int r = 0; r < R; ++r) Bs[kk + (NT / BN) * r][j] = rb[r];
    }
}

template <bool F64_LAYOUT, int MI, int NI>
__device__ __forceinline__ void write_tile(const GemmDesc& g, const TileCoord& tc, int lane,
                                           int wm0, int wn0, const dbl4 (&acc)[MI][NI]) {
    const bool part = g.ksplit > 1;
    gmut_double* out = as_global(part ? g.work + (int64_t)tc.kz * g.M * g.N : g.C);
    const int64_t ld = part ? g.M : g.ldc;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            const int col = tc.n0 + wn0 + ni * 16 + (lane & 15);
            if (col >= g.N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ri = F64_LAYOUT ? (lane >> 4) + 4 * r : (lane >> 4) * 4 + r;
                const int row = tc.m0 + wm0 + mi * 16 + ri;
                if (row >= g.M) continue;
                const double v = acc[mi][ni][r];
                gmut_double* p = out + (int64_t)row + (int64_t)col * ld;
                if (part) *p = v;
                else *p = (g.beta == 0.0) ? g.alpha * v : g.alpha * v + g.beta * *p;
            }
        }
}

// Output through LDS: a register of the FP64 MFMA result holds 4 rows x 16
// columns, which a direct store writes as 16 pieces of 32 bytes.  Instead
// each wave parks 32 x 16 blocks of its result in its own LDS region `ep`
// (EP_REGION doubles, column stride 34: conflict-free both ways) and stores
// whole 256-byte column runs.  Same values and formula as write_tile.
constexpr int EP_LD = 34, EP_REGION = 16 * EP_LD;

template <int MI, int NI>
__device__ __forceinline__ void write_tile_lds(const GemmDesc& g, const TileCoord& tc, int lane,
                                               int wm0, int wn0, const dbl4 (&acc)[MI][NI],
                                               double* ep) {
    static_assert(MI == 2, "32-row wave blocks");
    const bool part = g.ksplit > 1;
    gmut_double* out = as_global(part ? g.work + (int64_t)tc.kz * g.M * g.N : g.C);
    const int64_t ldo = part ? g.M : g.ldc;
    const int row = lane & 31, cpar = lane >> 5;
    const int grow = tc.m0 + wm0 + row;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                ep[(lane & 15) * EP_LD + mi * 16 + (lane >> 4) + 4 * r] = acc[mi][ni][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int col = 2 * c + cpar, gcol = tc.n0 + wn0 + ni * 16 + col;
            const double v = ep[col * EP_LD + row];
            if (grow < g.M && gcol < g.N) {
                gmut_double* p = out + (int64_t)grow + (int64_t)gcol * ldo;
                if (part) *p = v;
                else *p = (g.beta == 0.0) ? g.alpha * v : g.alpha * v + g.beta * *p;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

// WM x WN waves, each owning a (BM/WM) x (BN/WN) block of the tile; k-tiles
// of KB.  Every shape runs the MFMAs over k in the same 4-wide steps.
template <int BM, int BN, int WM, int WN, int KB>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_f64(const GemmDesc* __restrict__ descs,
                                                           int nd, unsigned long long* flop_ctr) {
    constexpr int NT = 64 * WM * WN;
    constexpr int MI = BM / WM / 16, NI = BN / WN / 16;
    // two LDS stages: the next k-tile is stored while the current one is
    // consumed, one barrier per k-tile
    __shared__ double As[2][KB][BM + 1];
    __shared__ double Bs[2][KB][BN + 1];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm0 = (w % WM) * (BM / WM), wn0 = (w / WM) * (BN / WN);
    const GemmDesc g = descs[find_desc_gemm(descs, nd, blockIdx.x)];
    if (g.skip && *g.skip) return;
    const TileCoord tc = tile_coord<BM, BN>(g, (int64_t)blockIdx.x - g.tile_start);
    count_tile_flops<BM, BN>(flop_ctr, g, tc);
    dbl4 acc[MI][NI], tot[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
            tot[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
    double ra[KB * BM / NT], rb[KB * BN / NT];
    if (tc.kbeg < tc.kend) {
        load_a<BM, NT, KB>(g, tc.m0, tc.kbeg, t, ra);
        load_b<BN, NT, KB>(g, tc.n0, tc.kbeg, t, rb);
        store_a<BM, NT, KB>(g, t, ra, As[0]);
        store_b<BN, NT, KB>(g, t, rb, Bs[0]);
    }
    __syncthreads();
    int buf = 0;
    for (int k0 = tc.kbeg; k0 < tc.kend; k0 += KB) {
        const bool more = k0 + KB < tc.kend;
        if (more) {
            load_a<BM, NT, KB>(g, tc.m0, k0 + KB, t, ra);
            load_b<BN, NT, KB>(g, tc.n0, k0 + KB, t, rb);
        }
        // operands of k-step ks + 1 are read from LDS while the MFMAs of
        // k-step ks run (two register sets)
        double a[2][MI], b[2][NI];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) a[0][mi] = As[buf][lane >> 4][wm0 + mi * 16 + (lane & 15)];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) b[0][ni] = Bs[buf][lane >> 4][wn0 + ni * 16 + (lane & 15)];
#pragma unroll
        for (int ks = 0; ks < KB / 4; ++ks) {
            const int cur = ks & 1;
            if (ks + 1 < KB / 4) {
                const int k = (ks + 1) * 4 + (lane >> 4);
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
                    a[cur ^ 1][mi] = As[buf][k][wm0 + mi * 16 + (lane & 15)];
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
                    b[cur ^ 1][ni] = Bs[buf][k][wn0 + ni * 16 + (lane & 15)];
            }
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][mi], b[cur][ni],
                                                                       acc[mi][ni], 0, 0, 0);
        }
        // end of a K chunk: add its sum to the running total (chunk order)
        if ((k0 + KB) % g.kchunk == 0 || !more) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[mi][ni][r] += acc[mi][ni][r];
                    acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
                }
        }
        if (more) {
            store_a<BM, NT, KB>(g, t, ra, As[buf ^ 1]);
            store_b<BN, NT, KB>(g, t, rb, Bs[buf ^ 1]);
        }
        __syncthreads();
        buf ^= 1;
    }
    // the loop's last barrier ends every read of As and Bs
    if constexpr (MI == 2 && 2 * KB * (BM + 1) >= (NT / 64) * EP_REGION)
        write_tile_lds<MI, NI>(g, tc, lane, wm0, wn0, tot, &As[0][0][0] + w * EP_REGION);
    else
        write_tile<true, MI, NI>(g, tc, lane, wm0, wn0, tot);
}

// ------------------------------------------------ FP64 MFMA, LDS-DMA pipeline
// The same products as k_gemm_f64 (same MFMA sequence over k, same K-chunk
// totals, so the same bits), with the operands going from global memory
// straight into LDS (buffer_load_dwordx4 ... lds: lane l of a wave writes its
// 16 bytes at the instruction's LDS base + 16 l) through NS LDS stages (three
// in every launch): the loads of k-tile t + NS - 1 are in flight while
// k-tile t is multiplied, and no registers hold tiles in transit.
//
// Each operand's stage region takes one of two layouts, by storage order:
//  * row layout (operand contiguous along its M / N index: A as stored, B
//    stored transposed): k-row kk holds the D values of that k; even rows
//    are packed from offset 0, odd rows from 8 D + 16, so rows kk and kk + 1
//    sit in opposite halves of the 64 LDS banks;
//  * column layout (contiguous along k): 16-byte slots (i, kp) hold
//    k = 2 kp, 2 kp + 1 of index i, slot i * 8 + (kp ^ ((i >> 1) & 7)): one
//    DMA instruction fetches 8 whole 128-byte lines, and the MFMA operand
//    reads of 16 consecutive i at one k fall in distinct banks.
// Loads go through buffer descriptors rebased per k-tile whose extent ends
// at the operand's last element: reads past it return zero and never fault.
// Rows past M (columns past N) may hold other elements of the operand; they
// only reach output rows (columns) that are not written.  k past K is zeroed
// in LDS before the last k-tile is used, so padded products are 0 * 0 as in
// k_gemm_f64.
// (KB, the k-tile depth, is 16 or 32: KB / 2 k-pairs per index; the column
// layout's XOR mask is (i >> 1) & 7 for 8 pairs and i & 15 for 16, either
// way distinct over 16 consecutive i.  Every launch uses 16: a 32-deep
// 128 x 128 tile on two stages needs more than 256 VGPRs and spills.)
template <int KB>
__host__ __device__ constexpr int dl_region(int d) { return KB * d + 16; }

template <int KB>
__device__ __forceinline__ int dl_mask(int i) { return KB == 16 ? ((i >> 1) & 7) : (i & 15); }

// LDS offset (doubles) of element (i, kk) of a D-wide operand region
template <int KB>
__device__ __forceinline__ int dl_off(bool rowl, int D, int i, int kk) {
    if (rowl) return ((kk & 1) ? (KB / 2) * D + 16 : 0) + (kk >> 1) * D + i;
    return (i * (KB / 2) + ((kk >> 1) ^ dl_mask<KB>(i))) * 2 + (kk & 1);
}

// What DMA instruction u (of D KB / 128) of a D-wide operand region fetches
// for this lane: its LDS base (doubles, uniform), the lane's element (i, k pair)
template <int KB>
__device__ __forceinline__ void dl_slot(bool rowl, int D, int u, int lane, int& base, int& i,
                                        int& kk0, int& kk1) {
    if (rowl) {
        const int half = (KB / 2) * D / 128;   // instructions per row parity
        const int odd = u >= half, uu = odd ? u - half : u;
        const int e = 128 * uu + 2 * lane;
        base = (odd ? (KB / 2) * D + 16 : 0) + 128 * uu;
        i = e % D;
        kk0 = kk1 = 2 * (e / D) + odd;
    } else {
        base = 128 * u;
        i = (128 / KB) * u + lane / (KB / 2);
        const int kp = (lane % (KB / 2)) ^ dl_mask<KB>(i);
        kk0 = 2 * kp;
        kk1 = 2 * kp + 1;
    }
}

template <int BM, int BN, int NW, int KB>
struct DlPlan {
    static constexpr int SA = dl_region<KB>(BM), SB = dl_region<KB>(BN), ST = SA + SB;
    // DMA instructions (1 KB each) per stage: for A, for both, per wave
    static constexpr int QA = BM * KB / 128, Q = (BM + BN) * KB / 128, PER = Q / NW;
    static_assert(Q % NW == 0, "DMA instructions must divide over the waves");
};

// LDS-DMA for one k-tile: this wave's PER instructions into `stage`
template <int BM, int BN, int NW, int KB>
__device__ __forceinline__ void dl_issue(double* stage, __amdgpu_buffer_rsrc_t ra,
                                         __amdgpu_buffer_rsrc_t rb,
                                         const int (&lbase)[DlPlan<BM, BN, NW, KB>::PER],
                                         const int (&vofs)[DlPlan<BM, BN, NW, KB>::PER], int w) {
    using P = DlPlan<BM, BN, NW, KB>;
#pragma unroll
    for (int r = 0; r < P::PER; ++r) {
        const int q = w + NW * r;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(q < P::QA ? ra : rb,
                                                 (__attribute__((address_space(3))) void*)(stage + lbase[r]),
                                                 16, vofs[r], 0, 0, 0);
    }
}

// buffer descriptor over [base, base + n) doubles (n clamped to the 32-bit
// byte range)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dl_rsrc(const double* base, int64_t n) {
    const int64_t bytes = n > 0 ? n * 8 : 0;
    const int nb = (int)(bytes > 0x7fffffffLL ? 0x7fffffffLL : bytes);
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, nb, 0x00020000);
}

// NS LDS stages (3 or 4, each its own array so that the compiler's wait
// for a stage's loads does not include the other stages'); OCC waves per
// SIMD: 4 lets two 128x64 workgroups share a CU (three stages: 73 KB of LDS
// each), 3 fits three 64x64 ones (49 KB each)
template <int BM, int BN, int WM, int WN, int OCC, int NS, int KB>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(OCC)))
void k_gemm_dl(const GemmDesc* __restrict__ descs, int nd, unsigned long long* flop_ctr) {
    static_assert(NS >= 2 && NS <= 4, "two to four LDS stages");
    static_assert(KB == 16 || KB == 32, "16- or 32-deep k-tiles");
    constexpr int NW = WM * WN;
    using P = DlPlan<BM, BN, NW, KB>;
    constexpr int MI = BM / WM / 16, NI = BN / WN / 16;
    __shared__ __align__(16) double S0[P::ST];
    __shared__ __align__(16) double S1[P::ST];
    __shared__ __align__(16) double S2[NS > 2 ? P::ST : 2];
    __shared__ __align__(16) double S3[NS > 3 ? P::ST : 2];
    double* const SS[4] = {S0, S1, S2, S3};
    // the wave index is uniform: keep it (and the LDS bases derived from it)
    // in scalar registers, as the DMA's LDS address must be
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm0 = (w % WM) * (BM / WM), wn0 = (w / WM) * (BN / WN);
    const GemmDesc g = descs[find_desc_gemm(descs, nd, blockIdx.x)];
    if (g.skip && *g.skip) return;
    const TileCoord tc = tile_coord<BM, BN>(g, (int64_t)blockIdx.x - g.tile_start);
    count_tile_flops<BM, BN>(flop_ctr, g, tc);
    if (flop_ctr) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const bool arow = !g.ta, brow = g.tb != 0;

    // per-lane DMA offsets (bytes, relative to the k-tile's descriptors) and
    // LDS bases of this wave's instructions
    int lbase[P::PER], vofs[P::PER];
#pragma unroll
    for (int r = 0; r < P::PER; ++r) {
        const int q = w + NW * r;
        int base, i, kk0, kk1;
        if (q < P::QA) {
            dl_slot<KB>(arow, BM, q, lane, base, i, kk0, kk1);
            lbase[r] = __builtin_amdgcn_readfirstlane(base);
            vofs[r] = 8 * (arow ? i + kk0 * g.lda : kk0 + i * g.lda);
        } else {
            dl_slot<KB>(brow, BN, q - P::QA, lane, base, i, kk0, kk1);
            lbase[r] = __builtin_amdgcn_readfirstlane(P::SA + base);
            vofs[r] = 8 * (brow ? i + kk0 * g.ldb : kk0 + i * g.ldb);
        }
    }
    // the operands' last elements bound the descriptors
    const int64_t extA = arow ? (int64_t)g.lda * (g.K - 1) + g.M : (int64_t)g.lda * (g.M - 1) + g.K;
    const int64_t extB = brow ? (int64_t)g.ldb * (g.K - 1) + g.N : (int64_t)g.ldb * (g.N - 1) + g.K;
    auto rsrc_a = [&](int k0) {
        const int64_t o = arow ? (int64_t)tc.m0 + (int64_t)k0 * g.lda : (int64_t)k0 + (int64_t)tc.m0 * g.lda;
        return dl_rsrc(g.A + o, extA - o);
    };
    auto rsrc_b = [&](int k0) {
        const int64_t o = brow ? (int64_t)tc.n0 + (int64_t)k0 * g.ldb : (int64_t)k0 + (int64_t)tc.n0 * g.ldb;
        return dl_rsrc(g.B + o, extB - o);
    };
    // MFMA operand offsets for each 4-deep k-step (row i / column j at mi,
    // ni = 0; +16 rows is +16 doubles in the row layout, +16 KB doubles in
    // the column one)
    int aoff[KB / 4], boff[KB / 4];
#pragma unroll
    for (int ks = 0; ks < KB / 4; ++ks) {
        const int kk = ks * 4 + (lane >> 4);
        aoff[ks] = dl_off<KB>(arow, BM, wm0 + (lane & 15), kk);
        boff[ks] = P::SA + dl_off<KB>(brow, BN, wn0 + (lane & 15), kk);
    }
    const int astep = arow ? 16 : 16 * KB, bstep = brow ? 16 : 16 * KB;

    dbl4 acc[MI][NI], tot[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
            acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
            tot[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
    const int nt = (tc.kend - tc.kbeg + KB - 1) / KB;
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < nt)
            dl_issue<BM, BN, NW, KB>(SS[s], rsrc_a(tc.kbeg + s * KB), rsrc_b(tc.kbeg + s * KB),
                                 lbase, vofs, w);

    // one k-tile: wait for this wave's loads of tile it, zero k >= K on the
    // last tile, barrier (every wave's loads of tile it have landed and every
    // wave is done with the stage tile it + NS - 1 goes into), issue tile
    // it + NS - 1, multiply
    auto step = [&](double* cur, double* nxt, int it) {
        const int k0 = tc.kbeg + it * KB;
        const int ahead = min(NS - 2, nt - 1 - it);   // tiles issued after this one
        if (NS > 3 && ahead >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P::PER) : "memory");
        else if (ahead >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P::PER) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (k0 + KB > g.K) {
            const int kv = g.K - k0;
#pragma unroll
            for (int r = 0; r < P::PER; ++r) {
                const int q = w + NW * r;
                int base, i, kk0, kk1;
                if (q < P::QA) dl_slot<KB>(arow, BM, q, lane, base, i, kk0, kk1);
                else dl_slot<KB>(brow, BN, q - P::QA, lane, base, i, kk0, kk1);
                double* d = cur + lbase[r] + 2 * lane;
                if (kk0 >= kv) d[0] = 0.0;
                if (kk1 >= kv) d[1] = 0.0;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (it + NS - 1 < nt)
            dl_issue<BM, BN, NW, KB>(nxt, rsrc_a(k0 + (NS - 1) * KB), rsrc_b(k0 + (NS - 1) * KB),
                                 lbase, vofs, w);
        __builtin_amdgcn_sched_barrier(0);
        double a[2][MI], b[2][NI];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) a[0][mi] = cur[aoff[0] + mi * astep];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) b[0][ni] = cur[boff[0] + ni * bstep];
#pragma unroll
        for (int ks = 0; ks < KB / 4; ++ks) {
            const int c = ks & 1;
            if (ks + 1 < KB / 4) {
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) a[c ^ 1][mi] = cur[aoff[ks + 1] + mi * astep];
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) b[c ^ 1][ni] = cur[boff[ks + 1] + ni * bstep];
            }
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[c][mi], b[c][ni],
                                                                       acc[mi][ni], 0, 0, 0);
        }
        if ((k0 + KB) % g.kchunk == 0 || it + 1 == nt) {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int ni = 0; ni < NI; ++ni) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[mi][ni][r] += acc[mi][ni][r];
                    acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
                }
        }
        // the stage's reads are complete before the next barrier lets another
        // wave's DMA overwrite it
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int it = 0; it < nt; it += NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
            if (it + s < nt) step(SS[s], SS[(s + NS - 1) % NS], it + s);
    }
    // the stages are free: the last k-tile waited for every load, and the
    // barrier below for every wave's reads; wave w parks its blocks in slot
    // w / NS of stage w % NS
    static_assert(((NW + NS - 1) / NS) * EP_REGION <= P::ST, "epilogue fits the stages");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int es = w % NS;
    write_tile_lds<MI, NI>(g, tc, lane, wm0, wn0, tot,
                           (es == 0 ? S0 : es == 1 ? S1 : es == 2 ? S2 : S3) + (w / NS) * EP_REGION);
}

// ------------------------------------------------ FP64 MFMA, small launches
// The same products for launches with too few tiles to fill the chip, where
// the chain over K is the time: each wave of a workgroup takes K chunks w,
// w + W, ... of the workgroup's own 16 MI x 16 MI tile, through its own ring
// of NS LDS stages (so the k loop has no barrier), and the chunk sums are
// added in order through LDS.  The sums are those of the other kernels with
// K split or not, bit for bit, without their second launch and workspace.
// Measured alone, copies and events included (64 x 64 tiles with K split and
// its reduction launch -> here): 1024 x 64 x 1024 25.3 -> 15.3 us, 64 x 64 x
// 1024 (a Gram matrix) 24.7 -> 14.4, 2048 x 96 x 2048 40.9 -> 36.4, 256 x 32 x
// 256 (one chunk) 21.1 -> 14.2.
template <int PER, int QA>
__device__ __forceinline__ void kw_issue(double* stage, __amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb,
                                         const int* lbase, const int* vofs) {
#pragma unroll
    for (int r = 0; r < PER; ++r)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r < QA ? ra : rb,
                                                 (__attribute__((address_space(3))) void*)(stage + lbase[r]),
                                                 16, vofs[r], 0, 0, 0);
}

template <int MI, int W, int NS>
__global__ __launch_bounds__(64 * W) void k_gemm_kw(const GemmDesc* __restrict__ descs, int nd,
                                                    unsigned long long* flop_ctr) {
    constexpr int BM = 16 * MI, KB = 16, NT = 64 * W;
    using P = DlPlan<BM, BM, 1, KB>;
    static_assert(NS == 3 || NS == 4, "three or four LDS stages");
    __shared__ __align__(16) double S0[W * P::ST];
    __shared__ __align__(16) double S1[W * P::ST];
    __shared__ __align__(16) double S2[W * P::ST];
    __shared__ __align__(16) double S3[NS > 3 ? W * P::ST : 2];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    double* const SS[4] = {S0 + w * P::ST, S1 + w * P::ST, S2 + w * P::ST, NS > 3 ? S3 + w * P::ST : S3};
    const GemmDesc g = descs[find_desc_gemm(descs, nd, blockIdx.x)];
    if (g.skip && *g.skip) return;
    const TileCoord tc = tile_coord<BM, BM>(g, (int64_t)blockIdx.x - g.tile_start);
    count_tile_flops<BM, BM>(flop_ctr, g, tc);
    if (flop_ctr) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const bool arow = !g.ta, brow = g.tb != 0;
    int lbase[P::PER], vofs[P::PER];
#pragma unroll
    for (int r = 0; r < P::PER; ++r) {
        int base, i, kk0, kk1;
        if (r < P::QA) {
            dl_slot<KB>(arow, BM, r, lane, base, i, kk0, kk1);
            lbase[r] = __builtin_amdgcn_readfirstlane(base);
            vofs[r] = 8 * (arow ? i + kk0 * g.lda : kk0 + i * g.lda);
        } else {
            dl_slot<KB>(brow, BM, r - P::QA, lane, base, i, kk0, kk1);
            lbase[r] = __builtin_amdgcn_readfirstlane(P::SA + base);
            vofs[r] = 8 * (brow ? i + kk0 * g.ldb : kk0 + i * g.ldb);
        }
    }
    const int64_t extA = arow ? (int64_t)g.lda * (g.K - 1) + g.M : (int64_t)g.lda * (g.M - 1) + g.K;
    const int64_t extB = brow ? (int64_t)g.ldb * (g.K - 1) + g.N : (int64_t)g.ldb * (g.N - 1) + g.K;
    auto rsrc_a = [&](int k0) {
        const int64_t o = arow ? (int64_t)tc.m0 + (int64_t)k0 * g.lda : (int64_t)k0 + (int64_t)tc.m0 * g.lda;
        return dl_rsrc(g.A + o, extA - o);
    };
    auto rsrc_b = [&](int k0) {
        const int64_t o = brow ? (int64_t)tc.n0 + (int64_t)k0 * g.ldb : (int64_t)k0 + (int64_t)tc.n0 * g.ldb;
        return dl_rsrc(g.B + o, extB - o);
    };
    auto issue = [&](double* stage, int k0) { kw_issue<P::PER, P::QA>(stage, rsrc_a(k0), rsrc_b(k0), lbase, vofs); };
    int aoff[KB / 4], boff[KB / 4];
#pragma unroll
    for (int ks = 0; ks < KB / 4; ++ks) {
        const int kk = ks * 4 + (lane >> 4);
        aoff[ks] = dl_off<KB>(arow, BM, lane & 15, kk);
        boff[ks] = P::SA + dl_off<KB>(brow, BM, lane & 15, kk);
    }
    const int astep = arow ? 16 : 16 * KB, bstep = brow ? 16 : 16 * KB;
    const int chunks = max(1, (g.K + g.kchunk - 1) / g.kchunk);
    // this thread's elements of the tile
    constexpr int E = BM * BM / NT;
    double sum[E];
#pragma unroll
    for (int i = 0; i < E; ++i) sum[i] = 0.0;
    for (int c0 = 0; c0 < chunks; c0 += W) {
        const int kbeg = (c0 + w) * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
        const int nt = kend > kbeg ? (kend - kbeg + KB - 1) / KB : 0;
        dbl4 acc[MI][MI];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < MI; ++ni) acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < NS - 1; ++s)
            if (s < nt) issue(SS[s], kbeg + s * KB);
        // one k-tile: wait for the loads of tile it, zero k >= K on the last
        // tile, issue tile it + NS - 1 into the stage whose reads were
        // consumed one tile ago, multiply
        auto step = [&](double* cur, double* nxt, int it) {
            const int k0 = kbeg + it * KB;
            const int ahead = min(NS - 2, nt - 1 - it);   // tiles issued after this one
            if (NS > 3 && ahead >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P::PER) : "memory");
            else if (ahead >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P::PER) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (k0 + KB > g.K) {
                const int kv = g.K - k0;
#pragma unroll
                for (int r = 0; r < P::PER; ++r) {
                    int base, i, kk0, kk1;
                    if (r < P::QA) dl_slot<KB>(arow, BM, r, lane, base, i, kk0, kk1);
                    else dl_slot<KB>(brow, BM, r - P::QA, lane, base, i, kk0, kk1);
                    double* d = cur + lbase[r] + 2 * lane;
                    if (kk0 >= kv) d[0] = 0.0;
                    if (kk1 >= kv) d[1] = 0.0;
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (it + NS - 1 < nt) issue(nxt, k0 + (NS - 1) * KB);
            __builtin_amdgcn_sched_barrier(0);
            double a[KB / 4][MI], b[KB / 4][MI];
#pragma unroll
            for (int ks = 0; ks < KB / 4; ++ks)
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) {
                    a[ks][mi] = cur[aoff[ks] + mi * astep];
                    b[ks][mi] = cur[boff[ks] + mi * bstep];
                }
#pragma unroll
            for (int ks = 0; ks < KB / 4; ++ks)
#pragma unroll
                for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                    for (int ni = 0; ni < MI; ++ni)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ks][mi], b[ks][ni], acc[mi][ni], 0,
                                                                           0, 0);
            // the stage's reads are complete (consumed) before the next
            // step's DMA may overwrite it
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int it = 0; it < nt; it += NS) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (it + s < nt) step(SS[s], SS[(s + NS - 1) % NS], it + s);
        }
        // (every load of this wave's stages has landed and been consumed)
        static_assert(BM * (BM + 1) <= P::ST, "the chunk sums fit a stage");
        double* pw = S0 + w * P::ST;
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
            for (int ni = 0; ni < MI; ++ni)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    pw[16 * mi + (lane >> 4) + 4 * r + (16 * ni + (lane & 15)) * (BM + 1)] = acc[mi][ni][r];
        __syncthreads();
        const int here = min(W, chunks - c0);
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const int e = t + NT * i, at = e % BM + (e / BM) * (BM + 1);
            for (int z = 0; z < here; ++z) sum[i] += S0[z * P::ST + at];
        }
        __syncthreads();
    }
    gmut_double* C = as_global(g.C);
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const int e = t + NT * i, row = tc.m0 + e % BM, col = tc.n0 + e / BM;
        if (row < g.M && col < g.N) {
            gmut_double* p = C + (int64_t)row + (int64_t)col * g.ldc;
            *p = (g.beta == 0.0) ? g.alpha * sum[i] : g.alpha * sum[i] + g.beta * *p;
        }
    }
}

// ------------------------------------------------ FP32 MFMA, hi/lo split
// x = hi + lo with hi = fp32(x), lo = fp32(x - hi).  Per k-tile the three
// significant products hi*hi, hi*lo, lo*hi are accumulated on FP32 MFMA
// (v_mfma_f32_16x16x4_f32) in separate accumulators, then flushed into FP64
// registers, so FP32 rounding only acts within one 16-deep k-tile.
__global__ __launch_bounds__(256) void k_gemm_split32(const GemmDesc* __restrict__ descs, int nd,
                                                      unsigned long long* flop_ctr) {
    __shared__ float Ah[BK][65], Al[BK][65];
    __shared__ float Bh[BK][65], Bl[BK][65];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, wm = w & 1, wn = w >> 1;
    const GemmDesc g = descs[find_desc_gemm(descs, nd, blockIdx.x)];
    if (g.skip && *g.skip) return;
    const TileCoord tc = tile_coord<64, 64>(g, (int64_t)blockIdx.x - g.tile_start);
    count_tile_flops<64, 64>(flop_ctr, g, tc);
    dbl4 acc[2][2], tot[2][2];
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
            tot[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
    double ra[4], rb[4];
    for (int k0 = tc.kbeg; k0 < tc.kend; k0 += BK) {
        load_a<64, 256, BK>(g, tc.m0, k0, t, ra);
        load_b<64, 256, BK>(g, tc.n0, k0, t, rb);
        // split and stage
        {
            float ah[4], al[4], bh[4], bl[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ah[r] = (float)ra[r]; al[r] = (float)(ra[r] - (double)ah[r]);
                bh[r] = (float)rb[r]; bl[r] = (float)(rb[r] - (double)bh[r]);
            }
            if (!g.ta) {
                int i = t & 63, kk = t >> 6;
#pragma unroll
                for (int r = 0; r < 4; ++r) { Ah[kk + 4 * r][i] = ah[r]; Al[kk + 4 * r][i] = al[r]; }
            } else {
                int kk = t & 15, i0 = t >> 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) { Ah[kk][i0 + 16 * r] = ah[r]; Al[kk][i0 + 16 * r] = al[r]; }
            }
            if (!g.tb) {
                int kk = t & 15, j0 = t >> 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) { Bh[kk][j0 + 16 * r] = bh[r]; Bl[kk][j0 + 16 * r] = bl[r]; }
            } else {
                int j = t & 63, kk = t >> 6;
#pragma unroll
                for (int r = 0; r < 4; ++r) { Bh[kk + 4 * r][j] = bh[r]; Bl[kk + 4 * r][j] = bl[r]; }
            }
        }
        __syncthreads();
        flt4 hh[2][2], cr[2][2];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) { hh[mi][ni] = flt4{0, 0, 0, 0}; cr[mi][ni] = flt4{0, 0, 0, 0}; }
#pragma unroll
        for (int ks = 0; ks < BK / 4; ++ks) {
            const int k = ks * 4 + (lane >> 4);
            float a0h = Ah[k][wm * 32 + (lane & 15)], a1h = Ah[k][wm * 32 + 16 + (lane & 15)];
            float a0l = Al[k][wm * 32 + (lane & 15)], a1l = Al[k][wm * 32 + 16 + (lane & 15)];
            float b0h = Bh[k][wn * 32 + (lane & 15)], b1h = Bh[k][wn * 32 + 16 + (lane & 15)];
            float b0l = Bl[k][wn * 32 + (lane & 15)], b1l = Bl[k][wn * 32 + 16 + (lane & 15)];
            float ah_[2] = {a0h, a1h}, al_[2] = {a0l, a1l}, bh_[2] = {b0h, b1h}, bl_[2] = {b0l, b1l};
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                for (int ni = 0; ni < 2; ++ni) {
                    hh[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah_[mi], bh_[ni], hh[mi][ni], 0, 0, 0);
                    cr[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(ah_[mi], bl_[ni], cr[mi][ni], 0, 0, 0);
                    cr[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(al_[mi], bh_[ni], cr[mi][ni], 0, 0, 0);
                }
        }
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[mi][ni][r] += (double)hh[mi][ni][r] + (double)cr[mi][ni][r];
        if ((k0 + BK) % g.kchunk == 0 || k0 + BK >= tc.kend) {
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                for (int ni = 0; ni < 2; ++ni) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[mi][ni][r] += acc[mi][ni][r];
                    acc[mi][ni] = dbl4{0.0, 0.0, 0.0, 0.0};
                }
        }
        __syncthreads();
    }
    write_tile<false, 2, 2>(g, tc, lane, wm * 32, wn * 32, tot);
}

// sum ksplit partials in fixed order, apply alpha/beta
__global__ __launch_bounds__(256) void k_gemm_reduce(const GemmDesc* __restrict__ descs, int nd,
                                                     const int64_t* __restrict__ starts,
                                                     int64_t total) {
    // A thread's elements increase, so its job index only moves forward: the
    // search continues from the last job (most steps stay in it or move to
    // the next), and that job's fields stay in registers until it changes.
    int lo = 0, cur = -1;
    const double* work = nullptr;
    double* C = nullptr;
    int64_t mn = 0, base = 0;
    int M = 1, ldc = 1, ks = 1;
    double alpha = 1.0, beta = 0.0;
    bool skip = false;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        if (lo + 1 < nd && starts[lo + 1] <= e) {
            int hi = nd - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (starts[mid] <= e) lo = mid; else hi = mid - 1;
            }
        }
        if (lo != cur) {
            cur = lo;
            const GemmDesc& g = descs[lo];
            skip = g.skip && *g.skip;
            work = g.work;
            C = g.C;
            M = g.M;
            ldc = g.ldc;
            ks = g.ksplit;
            alpha = g.alpha;
            beta = g.beta;
            mn = (int64_t)g.M * g.N;
            base = starts[lo];
        }
        if (skip) continue;
        const int64_t r = e - base;
        double s = 0.0;
        for (int z = 0; z < ks; ++z) s += work[z * mn + r];
        const int row = (int)(r % M), col = (int)(r / M);
        double* p = C + row + (int64_t)col * ldc;
        *p = (beta == 0.0) ? alpha * s : alpha * s + beta * *p;
    }
}

// --------------------------------------------------------- trace / normalise
__device__ __forceinline__ double block_sum_fixed(double v, double* red) {
    // deterministic tree over 256 threads
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (t < s) red[t] += red[t + s];
        __syncthreads();
    }
    double r = red[0];
    __syncthreads();
    return r;
}

// grid (TRACE_PARTS, nprob): partial sums of each problem's weighted trace
__global__ __launch_bounds__(256) void k_trace_partial(const TraceDesc* __restrict__ descs,
                                                       const TraceProb* __restrict__ probs) {
    __shared__ double red[256];
    const TraceProb P = probs[blockIdx.y];
    const TraceDesc* ds = descs + P.first;
    double acc = 0.0;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < P.total;
         e += (int64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = P.count - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (ds[mid].start <= e) lo = mid; else hi = mid - 1;
        }
        const TraceDesc& D = ds[lo];
        int64_t r = e - D.start;
        const int x1 = (int)(r % D.d1);
        r /= D.d1;
        const int x2 = (int)(r % D.d2), x3 = (int)(r / D.d2);
        double v = D.T[x1 * D.s1 + x2 * D.s2 + x3 * D.s3];
        if (D.w1) v *= D.w1[x1];
        if (D.w2) v *= D.w2[x2];
        acc += v;
    }
    double s = block_sum_fixed(acc, red);
    if (threadIdx.x == 0) P.partial[blockIdx.x] = s;
}

// grid (X, nprob): every block re-derives its problem's norm from the
// partials in the same order, block 0 stores it, all scale T by 1/|n|.
__global__ __launch_bounds__(256) void k_normalize(const TraceProb* __restrict__ probs) {
    __shared__ double red[256];
    const TraceProb P = probs[blockIdx.y];
    double v = (threadIdx.x < TRACE_PARTS) ? P.partial[threadIdx.x] : 0.0;
    double s = fabs(block_sum_fixed(v, red));
    if (blockIdx.x == 0 && threadIdx.x == 0) *P.norm_slot = s;
    const double inv = 1.0 / (P.divide_by ? *P.divide_by : s);
    // four elements a grid-stride apart per pass, loaded before they are
    // stored, so each thread keeps four loads in flight
    gmut_double* T = as_global(P.T);
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; e + 3 * stride < P.size; e += 4 * stride) {
        const double x0 = T[e], x1 = T[e + stride], x2 = T[e + 2 * stride], x3 = T[e + 3 * stride];
        T[e] = x0 * inv;
        T[e + stride] = x1 * inv;
        T[e + 2 * stride] = x2 * inv;
        T[e + 3 * stride] = x3 * inv;
    }
    for (; e < P.size; e += stride) T[e] *= inv;
}

// ---------------------------------------------------- linear combinations
__global__ __launch_bounds__(256) void k_lincomb(const LinDesc* __restrict__ descs, int nd,
                                                 int64_t total) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = nd - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (descs[mid].start <= e) lo = mid; else hi = mid - 1;
        }
        const LinDesc& D = descs[lo];
        const int64_t r = e - D.start;
        double v = D.coef[0] * D.in[0][r];
        for (int i = 1; i < D.nin; ++i) v += D.coef[i] * D.in[i][r];
        D.out[r] = v;
    }
}

// ------------------------------------------------------------- Jacobi eigen
// One workgroup per symmetric n x n matrix (n <= LMAX): cyclic two-sided
// Jacobi, G <- J^T G J, W <- W J.  A pair is rotated only while
// |g_pq| > tol sqrt(|g_pp g_qq|) (relative criterion, which keeps the small
// eigenvalues of graded Gram matrices relatively accurate).
//
// The solve is a chain of dependent rounds (n - 1 per sweep), so what counts
// is the latency of one round, not its arithmetic.  A round of M / 2 disjoint
// rotations on an M x M matrix (M <= 32) runs inside ONE wavefront, with no
// workgroup barrier between the rotations and their use: lane x computes the
// rotation of pair x, every lane rotates its one or two off-diagonal 2 x 2
// pair blocks and fetches the other pair's rotation from its lane.  The
// matrix sits in LDS in tournament order: positions t_0 .. t_{M/2-1},
// b_0 .. b_{M/2-1}, pair i = (t_i, b_i), and a round writes its results straight
// to the positions of the next round, so the LDS addresses of a lane never
// change.  A second wave holds the rows of the accumulated Q in registers and
// applies the rotations one round behind (one barrier per round, where the
// first wave has only just consumed its loads).
//   n <= 32: M = 16, 24 or 32, Q is W.
//   n <= 96: block Jacobi over 16-wide blocks.  Each block round pairs the
//   blocks up, every pair's 32 x 32 matrix takes one sweep of rounds in its
//   own two waves (31 rounds in the first block round of a sweep, which
//   also rotates inside the blocks, 16 in the others), then the pairs' Q are
//   applied to the rest of G and, during the next block round, to W on MFMA.
//   W stays in registers as strips of W^T: the MFMA result layout is the B
//   operand layout of the next block round's product.
// Block rounds (or, for n <= 32, sweeps) without a violating pair are
// skipped, and the solve ends with a sweep without one.  The input is
// symmetrised on load ((G + G^T)/2).  Output: eigenvalues by |lambda|
// descending, eigenvectors as columns of W in the same order.
//
// Measured, one Gram matrix of random columns (us a launch), against the
// former kernel (1024 threads, every pair block and W in LDS, two workgroup
// barriers a round): n = 16 / 32 / 64 / 96: 100 / 245 / 754 / 2112 -> 32 / 86
// / 263 / 662; nearly diagonal ones (the block iteration's): 50 / 102 / 274 /
// 696 -> 15 / 43 / 102 / 214.  A round takes 0.28 us at M = 16, 0.35 at 32,
// 0.40 / 0.54 with two / three block pairs side by side (Q in LDS as well:
// 0.49 / 0.56, the LDS pipe was the limit; W's MFMA on the SIMDs of the
// rotations: 0.49); a block round adds 2.8 us at n = 64, 5 us at 96, the
// orthogonal W of final solves 1 / 4 / 14 us at n = 32 / 64 / 96 (|W^T W - 1|
// 1e-14 -> 5e-16).
constexpr int JWAVES = 2;          // per pair of blocks: rotations, Q
constexpr int JB = 16;             // block width for n > 32
constexpr int JM = 2 * JB;
// solves to a tighter threshold than this (final ones, whose W is a factor of
// the result) also get W orthogonal to roundoff
constexpr double JPOLISH_BELOW = 1e-13;

// Position of a round's position x in the next round (t_i = i, b_i = H + i).
// Full tournament: t_0 stays, the others go round the circle t_1 .. t_{H-1},
// b_{H-1} .. b_0 (all pairs in 2H - 1 rounds, which is the identity).  Cross
// rounds: the t_i stay, the b_i go round (all t-b pairs in H rounds, the
// identity again).
__device__ __forceinline__ int jacobi_next(int x, int H, bool cross) {
    if (cross) return x < H ? x : (x == H ? 2 * H - 1 : x - 1);
    if (x < H) return x == 0 ? 0 : (x == H - 1 ? 2 * H - 1 : x + 1);
    return x == H ? 1 : x - 1;
}

// A pair is rotated while g_pq^2 > tol^2 |g_pp g_qq| (the relative
// criterion keeps the small eigenvalues of graded Gram matrices relatively
// accurate); the scans and the rounds use this same predicate.
__device__ __forceinline__ int jacobi_violates(double gpp, double gqq, double gpq, double tol2) {
    return gpq != 0.0 && gpq * gpq > tol2 * fabs(gpp * gqq);
}

// 1 / sqrt(x) from the hardware estimate (v_rsq_f64, ~24 bits) and one
// third-order step, a shorter dependent chain than two Newton steps:
// with e = 1 - x y^2, y (1 + e / 2 + 3 e^2 / 8).
__device__ __forceinline__ double rsqrt_refined(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// Rotation zeroing g_pq by the smaller angle: with a = g_qq - g_pp,
// b = 2 g_pq and r = 1 / sqrt(a^2 + b^2), cos 2x = |a| r and
// sin 2x = sign(a) b r, so c^2 = (1 + cos 2x) / 2, s = sin 2x / (2 c) and
// t = s / c: two reciprocal square roots in a row and no division.
// c^2 + s^2 = 1 to a few ulp.
__device__ __forceinline__ void jacobi_rotation(double gpp, double gqq, double gpq, double& t,
                                                double& c, double& s) {
    const double a = gqq - gpp, b = 2.0 * gpq;
    const double hb = a >= 0.0 ? gpq : -gpq;
    const double r = rsqrt_refined(fma(a, a, b * b));
    const double x = fma(0.5 * fabs(a), r, 0.5);
    const double y = rsqrt_refined(x);
    const double hs = hb * r;
    c = x * y;
    s = hs * y;
    t = s * y;
}

// LDS of one block pair: the M x M matrix (upper triangle by position), Q by
// columns (two for n > 32: the W strips read one while the rounds build the
// other) and the rotations of two rounds.  The strides keep the Q rows'
// rounds and the MFMA operand reads at two lanes per bank or fewer.
template <int M, int NS>
struct JacLds {
    static constexpr int H = M / 2, SL = (H / 2 + 3) / 4;
    static constexpr int LS = M + 1, LQ = M + 4;
    static constexpr int SINK = M * LS;   // for results that go nowhere
    static constexpr int Q = M * LS + 2, NQ = NS > 1 ? 2 : 1, CS = Q + NQ * M * LQ;
    static constexpr int DOUBLES = CS + 4 * H;
    static constexpr int NP = NS > 1 ? M * NS : 0, LG = NP + 2;   // the whole matrix, n > 32
    static constexpr size_t ALL = (size_t)NP * LG + (size_t)NS * DOUBLES;
    // waves: per block pair one for the rotations and one for Q; for n > 32
    // one more per block pair, for two strips of W
    static constexpr int WAVES = NS * (NS > 1 ? JWAVES + 1 : JWAVES);
};

// behind them: the waves' violation flags (two block rounds), the output order
constexpr size_t JTAIL_BYTES = (2 * 3 * JWAVES + LMAX) * sizeof(int);

size_t jacobi_lds_bytes(int n) {
    const size_t d = n <= 16       ? JacLds<16, 1>::ALL
                     : n <= 24     ? JacLds<24, 1>::ALL
                     : n <= JM     ? JacLds<JM, 1>::ALL
                     : n <= 2 * JM ? JacLds<JM, 2>::ALL
                                   : JacLds<JM, 3>::ALL;
    return d * sizeof(double) + JTAIL_BYTES;
}

int jacobi_threads(int n) {
    return 64 * (n <= JM ? JacLds<JM, 1>::WAVES : n <= 2 * JM ? JacLds<JM, 2>::WAVES : JacLds<JM, 3>::WAVES);
}

// compiler and LDS order between this wave's own steps (the LDS unit runs a
// wave's accesses in order)
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double lane_read(int byte_lane, double x) {
    const int lo = __builtin_amdgcn_ds_bpermute(byte_lane, __double2loint(x));
    const int hi = __builtin_amdgcn_ds_bpermute(byte_lane, __double2hiint(x));
    return __hiloint2double(hi, lo);
}

// LDS places of a lane's entries in a round, and of its results for the next
// round (full tournament, cross rounds).  Lane (g, x) of the wave's four rows
// of 16 computes the rotation of pair x (each row again) and rotates the pair
// blocks (x, x + g + 1 + 4 u mod H): its own rotation comes first, while the
// other pair's is fetched from its lane.
template <int M, int NS>
struct JacPlaces {
    using L = JacLds<M, NS>;
    int from[L::SL], rd[L::SL][4], wr[2][L::SL][4], drd[3], dwr[2][3];
    __device__ __forceinline__ explicit JacPlaces(int lane) {
        constexpr int H = L::H;
        auto at = [](int x, int y) { return min(x, y) + max(x, y) * L::LS; };
        const int x0 = lane & 15, x = x0 < H ? x0 : x0 - H;   // spare lanes repeat others
#pragma unroll
        for (int u = 0; u < L::SL; ++u) {
            const int dist = min((lane >> 4) + 1 + 4 * u, H / 2);
            const int y = x + dist < H ? x + dist : x + dist - H;
            // the blocks of distance H / 2 are met from both ends: one end's
            // results go nowhere
            const bool twin = dist == H / 2 && x >= H / 2;
            from[u] = 4 * y;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int p = x + (q >> 1) * H, r = y + (q & 1) * H;
                rd[u][q] = at(p, r);
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    wr[c][u][q] = twin ? L::SINK : at(jacobi_next(p, H, c), jacobi_next(r, H, c));
            }
        }
        drd[0] = at(x, x); drd[1] = at(x + H, x + H); drd[2] = at(x, x + H);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int p = jacobi_next(x, H, c), q = jacobi_next(x + H, H, c);
            dwr[c][0] = at(p, p); dwr[c][1] = at(q, q); dwr[c][2] = at(p, q);
        }
    }
};

// One sweep of R rounds on the matrix in S by one wave, R + 1 barriers.
template <int M, int NS>
__device__ __forceinline__ void jacobi_rounds(const JacPlaces<M, NS>& P, double* S, double2* cs, int lane,
                                              int R, bool cross, double tol2) {
    using L = JacLds<M, NS>;
    constexpr int H = L::H, SL = L::SL;
    int wr[SL][4], dwr[3];
#pragma unroll
    for (int u = 0; u < SL; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) wr[u][q] = cross ? P.wr[1][u][q] : P.wr[0][u][q];
#pragma unroll
    for (int q = 0; q < 3; ++q) dwr[q] = cross ? P.dwr[1][q] : P.dwr[0][q];
    double b[SL][4], d[3];
    auto load = [&] {
#pragma unroll
        for (int k = 0; k < 3; ++k) d[k] = S[P.drd[k]];
#pragma unroll
        for (int u = 0; u < SL; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) b[u][q] = S[P.rd[u][q]];
    };
    load();
    for (int r = 0; r < R; ++r) {
        // the diagonal's arrival means that every LDS access issued before
        // it is done, the last round's rotations among them (a wave's
        // accesses complete in order); what may be in flight are the reads of
        // b, entries of S that no other wave touches during the rounds
        asm volatile("s_barrier" ::"v"(d[0]), "v"(d[1]), "v"(d[2]) : "memory");
        // once a round is run, pairs a hundred times below the threshold are
        // rotated too: close eigenvalues' vectors feel what is left over their
        // gap.  Random and graded spectra take as many sweeps as without the
        // factor; large clusters take more, as the rotations of (nearly) equal
        // diagonals keep stirring up roundoff: with half of the eigenvalues
        // equal, n = 32 / 64 / 96, 11 / 18 / 20 sweeps instead of 8 / 13 / 14
        // (64 problems 153 / 627 / 1568 us instead of 115 / 450 / 1129; the
        // kernel before the block Jacobi 313 / 938 / 2440), with pairs of equal
        // ones 8.8 / 9.9 / 10.5 instead of 7.7 / 8.8 / 9.4.
        const bool on = jacobi_violates(d[0], d[1], d[2], 1e-4 * tol2);
        double c, s, t;
        jacobi_rotation(d[0], d[1], d[2], t, c, s);
        c = on ? c : 1.0;
        s = on ? s : 0.0;
        t = on ? t : 0.0;
        double co[SL], so[SL];
#pragma unroll
        for (int u = 0; u < SL; ++u) {
            co[u] = lane_read(P.from[u], c);
            so[u] = lane_read(P.from[u], s);
        }
        if (lane < H) {
            cs[(r & 1) * H + lane] = make_double2(c, s);
            S[dwr[0]] = d[0] - t * d[2];
            S[dwr[1]] = d[1] + t * d[2];
            S[dwr[2]] = on ? 0.0 : d[2];
        }
#pragma unroll
        for (int u = 0; u < SL; ++u) {
            const double y0 = c * b[u][0] - s * b[u][2], y1 = c * b[u][1] - s * b[u][3];
            const double y2 = s * b[u][0] + c * b[u][2], y3 = s * b[u][1] + c * b[u][3];
            b[u][0] = y0; b[u][1] = y1; b[u][2] = y2; b[u][3] = y3;
        }
#pragma unroll
        for (int u = 0; u < SL; ++u) {
            const double y0 = co[u] * b[u][0] - so[u] * b[u][1], y1 = so[u] * b[u][0] + co[u] * b[u][1];
            const double y2 = co[u] * b[u][2] - so[u] * b[u][3], y3 = so[u] * b[u][2] + co[u] * b[u][3];
            S[wr[u][0]] = y0;
            S[wr[u][1]] = y1;
            S[wr[u][2]] = y2;
            S[wr[u][3]] = y3;
        }
        wave_order();
        load();
    }
    __syncthreads();
}

// Rows of the accumulated Q in one wave's registers, columns in tournament
// order: lane (h, row) holds pairs HP h .. HP h + HP - 1 of row `row` (lanes
// past M hold rows that are never read).
template <int M>
struct JacRows {
    static constexpr int H = M / 2, HP = H / 2;
    double t[HP], b[HP];
    __device__ __forceinline__ void identity(int lane) {
        const int row = lane & 31, p0 = HP * (lane >> 5);
#pragma unroll
        for (int i = 0; i < HP; ++i) {
            t[i] = row == p0 + i ? 1.0 : 0.0;
            b[i] = row == p0 + i + H ? 1.0 : 0.0;
        }
    }
    // R rounds, one behind the rotations' wave, R + 1 barriers; the shifts
    // are jacobi_next on the pairs, between the halves by a lane swap
    template <bool CROSS>
    __device__ __forceinline__ void rounds(const double2* cs, int lane, int R) {
        const bool hi = lane >= 32;
        // (nothing in flight: a __syncthreads came since this wave's last access)
        asm volatile("s_barrier" ::: "memory");
        for (int r = 0; r < R; ++r) {
            // The rotations' wave writes round r's buffer again (round r + 2)
            // behind the next barrier: the reads below are complete by then.
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            const double2* rot = cs + (r & 1) * H + HP * (lane >> 5);
            double2 k[HP];
#pragma unroll
            for (int i = 0; i < HP; ++i) k[i] = rot[i];
            double x[HP], y[HP];
#pragma unroll
            for (int i = 0; i < HP; ++i) {
                x[i] = k[i].x * t[i] - k[i].y * b[i];
                y[i] = k[i].y * t[i] + k[i].x * b[i];
            }
            const double v = CROSS || hi ? y[0] : x[HP - 1];
            const auto lo2 = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
            const auto hi2 = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
            // .x: the lower half's value, .y: the upper half's, in every lane
            const double got = hi ? __hiloint2double(hi2[0], lo2[0]) : __hiloint2double(hi2[1], lo2[1]);
#pragma unroll
            for (int i = 0; i + 1 < HP; ++i) b[i] = y[i + 1];
            if (CROSS) {
                b[HP - 1] = got;
#pragma unroll
                for (int i = 0; i < HP; ++i) t[i] = x[i];
            } else {
                b[HP - 1] = hi ? x[HP - 1] : got;
                t[0] = hi ? got : x[0];
                t[1] = hi ? x[0] : y[0];
#pragma unroll
                for (int i = 2; i < HP; ++i) t[i] = x[i - 1];
            }
        }
    }
    __device__ __forceinline__ void store(double* Q, int ld, int lane) const {
        const int row = lane & 31, p0 = HP * (lane >> 5);
        if (row >= M) return;
#pragma unroll
        for (int i = 0; i < HP; ++i) {
            Q[row + (p0 + i) * ld] = t[i];
            Q[row + (p0 + i + H) * ld] = b[i];
        }
    }
};

// A operand of one k-step of a product with Q^T: rows 16 o .. of Q^T (columns
// of Q), k = 16 k0 + 4 kk ..
__device__ __forceinline__ double jac_qt(const double* Q, int LQ, int lane, int o, int k0, int kk) {
    return Q[16 * k0 + 4 * kk + (lane >> 4) + (16 * o + (lane & 15)) * LQ];
}

// position of slot x of the block tournament in the next block round
constexpr int jac_slot_next(int x, int NS) {
    return x < NS ? (x == 0 ? 0 : (x == NS - 1 ? 2 * NS - 1 : x + 1)) : (x == NS ? 1 : x - 1);
}

template <int M, int NS>
__device__ void jacobi_body(const JacobiDesc& D, double* lds, double tol, int max_sweeps, bool polish) {
    using L = JacLds<M, NS>;
    constexpr int H = L::H, NB = NS > 1 ? 2 * NS : 1, NP = L::NP, LG = L::LG;
    constexpr int NT = 64 * L::WAVES, ST = 64 * JWAVES, PW = NS * JWAVES;
    const int n = D.n, t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (w >= L::WAVES) return;   // a larger problem of the group set the block size
    // The waves' work: per block pair `sub` one wave for the rotations (ROT)
    // and one for Q, for n > 32 also one per block pair with two strips of W.
    // Waves go round the four SIMDs, and FP64 MFMA keeps a SIMD's FP64 unit
    // from its other waves: the rotations' waves get SIMDs of their own
    // (n <= 64), or share one with the least there is (n <= 96).
    enum { ROT, QROWS, STRIPS };
    int role, sub;
    if constexpr (NS == 1) {
        role = w, sub = 0;
    } else if constexpr (NS == 2) {
        role = w < 2 ? QROWS : w < 4 ? ROT : STRIPS, sub = w & 1;
    } else {
        // SIMD 0: strips 0 and 1, Q 0; 1: rotations 0, strips 2; 2, 3: rotations, Q
        role = w == 0 || w == 4 || w == 5 ? STRIPS : w < 4 ? ROT : QROWS;
        sub = w == 0 ? 0 : w == 4 ? 1 : w == 5 ? 2 : w < 4 ? w - 1 : w == 8 ? 0 : w - 5;
    }
    const int slot = JWAVES * sub + role, ts = lane + 64 * role;   // (not the strips)
    double* G = lds;
    double* S0 = lds + NP * LG;
    double* S = S0 + sub * L::DOUBLES;
    double2* cs = (double2*)(S + L::CS);
    int* flags = (int*)(S0 + NS * L::DOUBLES);   // [2][PW]
    int* pos = flags + 2 * 3 * JWAVES;
    // every lane loads (clamped, in bounds), so the loads are not predicated
    // and stay in flight together
    auto entry = [&](int x, int y) {
        const int xc = min(x, n - 1), yc = min(y, n - 1);
        const double v = 0.5 * (D.G[xc + (int64_t)yc * D.ldg] + D.G[yc + (int64_t)xc * D.ldg]);
        return x < n && y < n ? v : 0.0;
    };
    if constexpr (NS == 1) {
#pragma unroll 4
        for (int e = t; e < M * M; e += NT) {
            const int y = e / M, x = e - y * M;
            const double v = entry(x, y);
            if (x <= y) S[x + y * L::LS] = v;
        }
    } else {
#pragma unroll 4
        for (int e = t; e < NP * NP; e += NT) {
            const int y = e / NP, x = e - y * NP;
            G[x + y * LG] = entry(x, y);
        }
    }
    __syncthreads();
    constexpr int ROUNDS = NS > 1 ? NB - 1 : 1;   // block rounds of a sweep
    const double tol2 = tol * tol;
    int sweeps = 0;
    // The sweeps, as every wave of the workgroup goes through them: `scan`
    // writes this wave's flag for a block round, `act` gets `on` (the block
    // pairs with a violating pair, one bit each), whether they are to be
    // rotated, and whether within the blocks too.
    auto drive = [&](auto&& scan, auto&& act) {
        int par = 0;
        for (int sw = 0;; ++sw) {
            bool any = false, stop = false;
#pragma unroll 1
            for (int rnd = 0; rnd < ROUNDS; ++rnd) {
                int* fl = flags + par * PW;
                par ^= 1;
                scan(fl, rnd);
                __syncthreads();
                int on = 0, f = 0;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int v = fl[JWAVES * s] | fl[JWAVES * s + 1];
                    f |= v;
                    on |= v ? 1 << s : 0;
                }
                f = __builtin_amdgcn_readfirstlane(f);
                on = __builtin_amdgcn_readfirstlane(on);
                if (f) {
                    any = true;
                    stop = sw == max_sweeps;
                }
                act(on, f && !stop, !(f & 2));
            }
            if (stop && t == 0 && D.fail) *D.fail = 1.0;   // sweep cap, a rotation still due
            if (stop || !any) break;
            ++sweeps;
        }
    };
    auto rounds_of = [](bool cross) { return cross ? H : M - 1; };
    int qbuf = 0;
    // the blocks in the slots of the block tournament: tops 0 .. NS - 1, then
    // bottoms
    int ids[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) ids[b] = b;
    int I = 0, J = 0;   // first rows of this block pair's blocks (J: less H)
    // violating pairs of this block pair (within the blocks only in the first
    // block round); its matrix into S
    auto scan_pair = [&](int* fl, int rnd) {
        if constexpr (NS > 1) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                if (s == sub) {
                    I = JB * ids[s];
                    J = JB * ids[NS + s] - H;
                }
        }
        int v = 0;
        // entries (x <= y): the cross square, then both blocks' triangles in
        // one square (upper: first block, lower: second), then the second's
        // diagonal
        constexpr int HH = H * H;
#pragma unroll
        for (int k = 0; k < (2 * HH + H + ST - 1) / ST; ++k) {
            const int e = min(ts + k * ST, 2 * HH + H - 1);
            const int sq = e / HH, r = e - sq * HH, c = r / H, a = r - c * H;   // column, row in the square
            int x, y;
            if (sq == 0) x = a, y = c + H;
            else if (sq == 1) x = a <= c ? a : c + H, y = a <= c ? c : a + H;
            else x = y = r + H;
            const double* A = NS > 1 ? G : S;
            constexpr int LA = NS > 1 ? LG : L::LS;
            const int gx = (x < H ? I : J) + x, gy = (y < H ? I : J) + y;
            const double gxy = A[gx + gy * LA], gxx = A[gx + gx * LA], gyy = A[gy + gy * LA];
            if (NS > 1) S[x + y * L::LS] = gxy;
            if (x != y && jacobi_violates(gxx, gyy, gxy, tol2)) v |= sq ? 2 : 1;
        }
        if (NS > 1 && rnd > 0) v &= 1;
        v = (__any(v & 1) ? 1 : 0) | (__any(v & 2) ? 2 : 0);
        if (lane == 0) fl[slot] = v;
    };
    // after the rounds: the block pairs' Q applied to the rest of G
    auto apply = [&](int on) {
        __syncthreads();
        if constexpr (NS > 1) {
            // the 32 x 32 off-diagonal matrix of each two block pairs a < b,
            // G_ab <- Q_a^T G_ab Q_b: H = Q_a^T G_ab (into the Q buffer that
            // the W strips are done with), then Q_b^T H^T, both triangles
            // written.  A unit of either product is one 16 x 16 tile.
            constexpr int UNITS = 2 * NS * (NS - 1);
            auto unit = [&](int u, int* ra, int* rb) {   // first rows of a's and b's blocks; whether to do
                const int a = u < 8 ? 0 : 1, b = u < 4 ? 1 : 2;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    if (s == a) { ra[0] = JB * ids[s]; ra[1] = JB * ids[NS + s]; }
                    if (s == b) { rb[0] = JB * ids[s]; rb[1] = JB * ids[NS + s]; }
                }
                return (on >> a & 1) || (on >> b & 1);
            };
            auto qof = [&](int s, int buf) { return S0 + s * L::DOUBLES + L::Q + buf * M * L::LQ; };
            for (int u = w; u < UNITS; u += L::WAVES) {
                int ra[2], rb[2];
                if (!unit(u, ra, rb)) continue;
                const int o = u & 1, c = u >> 1 & 1;   // tile: rows of a, columns of b
                const double* Qa = qof(u < 8 ? 0 : 1, qbuf);
                const double* col = G + (lane >> 4) + ((c ? rb[1] : rb[0]) + (lane & 15)) * LG;
                dbl4 h = dbl4{0, 0, 0, 0}, h2 = dbl4{0, 0, 0, 0};
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    h = __builtin_amdgcn_mfma_f64_16x16x4f64(jac_qt(Qa, L::LQ, lane, o, 0, kk),
                                                             col[ra[0] + 4 * kk], h, 0, 0, 0);
                    h2 = __builtin_amdgcn_mfma_f64_16x16x4f64(jac_qt(Qa, L::LQ, lane, o, 1, kk),
                                                              col[ra[1] + 4 * kk], h2, 0, 0, 0);
                }
                h = h + h2;
                double* dst = qof(u >> 2, qbuf ^ 1) + 16 * o + (lane >> 4) + (16 * c + (lane & 15)) * L::LQ;
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[4 * r] = h[r];
            }
            // the block pairs' own matrices, both triangles
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (!(on >> s & 1)) continue;
                const int i0 = JB * ids[s], j0 = JB * ids[NS + s] - H;
                const double* Ss = S0 + s * L::DOUBLES;
#pragma unroll
                for (int k = 0; k < (M * M + NT - 1) / NT; ++k) {
                    const int e = min(t + k * NT, M * M - 1), y = e / M, x = e - y * M;
                    G[(x < H ? i0 : j0) + x + ((y < H ? i0 : j0) + y) * LG] = Ss[min(x, y) + max(x, y) * L::LS];
                }
            }
            __syncthreads();
            for (int u = w; u < UNITS; u += L::WAVES) {
                int ra[2], rb[2];
                if (!unit(u, ra, rb)) continue;
                const int o = u & 1, c = u >> 1 & 1;   // tile: columns of b, rows of a
                const double* Qb = qof(u < 4 ? 1 : 2, qbuf);
                const double* hs = qof(u >> 2, qbuf ^ 1) + 16 * c + (lane & 15) + (lane >> 4) * L::LQ;
                dbl4 h = dbl4{0, 0, 0, 0}, h2 = dbl4{0, 0, 0, 0};
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    h = __builtin_amdgcn_mfma_f64_16x16x4f64(jac_qt(Qb, L::LQ, lane, o, 0, kk),
                                                             hs[4 * kk * L::LQ], h, 0, 0, 0);
                    h2 = __builtin_amdgcn_mfma_f64_16x16x4f64(jac_qt(Qb, L::LQ, lane, o, 1, kk),
                                                              hs[(16 + 4 * kk) * L::LQ], h2, 0, 0, 0);
                }
                h = h + h2;
                const int row = (c ? ra[1] : ra[0]) + (lane & 15), cb = (o ? rb[1] : rb[0]) + (lane >> 4);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    G[row + (cb + 4 * r) * LG] = h[r];
                    G[cb + 4 * r + row * LG] = h[r];
                }
            }
            __syncthreads();
            qbuf ^= 1;
        }
    };
    auto next_slots = [&] {
        if constexpr (NS > 1) {
            int nid[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) nid[jac_slot_next(b, NS)] = ids[b];
#pragma unroll
            for (int b = 0; b < NB; ++b) ids[b] = nid[b];
        }
    };
    // (a __syncthreads came since this wave's last LDS access)
    auto idle = [](int R) {
        for (int r = 0; r <= R; ++r) asm volatile("s_barrier" ::: "memory");
    };
    // strips 2 sub, 2 sub + 1 of W^T (16 columns each), by slot
    const int st0 = 2 * sub;
    dbl4 wt[2][NB];
    // (each role's loop is its own code, so that its registers are its own)
    if (NS > 1 && role == STRIPS) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    wt[h][b][r] = (b == st0 + h && 4 * r + (lane >> 4) == (lane & 15)) ? 1.0 : 0.0;
        int owed = 0;   // block pairs whose Q (in the other buffer) W still lacks
        drive([](int*, int) {}, [&](int on, bool go, bool cross) {
            // W^T <- Q^T W^T with the last rotated block round's Q, a few MFMAs
            // per barrier of this one's rounds.  A result is laid out as the
            // next product's B operand, so the strips never leave the registers.
            // (Reads of Qs may be in flight at these barriers: that buffer is
            // written next by apply, behind its __syncthreads.)
            const int R = rounds_of(cross);
            int done = 0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (!(owed >> s & 1)) continue;
                const double* Qs = S0 + s * L::DOUBLES + L::Q + (qbuf ^ 1) * M * L::LQ;
                const int top = NS > 1 ? jac_slot_next(s, NS) : 0, bot = NS > 1 ? jac_slot_next(NS + s, NS) : 0;
                dbl4 x[2][2];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int o = 0; o < 2; ++o) x[h][o] = dbl4{0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        if ((kk & 1) == 0 && go && done <= R) {
                            asm volatile("s_barrier" ::: "memory");
                            ++done;
                        }
#pragma unroll
                        for (int o = 0; o < 2; ++o) {
                            const double a = jac_qt(Qs, L::LQ, lane, o, k, kk);
#pragma unroll
                            for (int h = 0; h < 2; ++h)
                                x[h][o] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    a, wt[h][k == 0 ? top : bot][kk], x[h][o], 0, 0, 0);
                        }
                    }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    wt[h][top] = x[h][0];
                    wt[h][bot] = x[h][1];
                }
            }
            owed = 0;
            if (go) {
                for (; done <= R; ++done) asm volatile("s_barrier" ::: "memory");
                apply(on);
                owed = on;
            }
            next_slots();
            dbl4 nx[2][NB];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) nx[h][NS > 1 ? jac_slot_next(b, NS) : b] = wt[h][b];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) wt[h][b] = nx[h][b];
        });
    } else if (role == ROT) {
        const JacPlaces<M, NS> places(lane);
        drive(scan_pair, [&](int on, bool go, bool cross) {
            if (go) {
                if (on >> sub & 1) jacobi_rounds<M, NS>(places, S, cs, lane, rounds_of(cross), cross, tol2);
                else idle(rounds_of(cross));
                apply(on);
            }
            next_slots();
        });
    } else {
        JacRows<M> rows;
        rows.identity(lane);
        drive(scan_pair, [&](int on, bool go, bool cross) {
            if (go) {
                if (!(on >> sub & 1)) idle(rounds_of(cross));
                else if (cross) rows.template rounds<true>(cs, lane, H);
                else rows.template rounds<false>(cs, lane, M - 1);
                if (NS > 1) {
                    rows.store(S + L::Q + qbuf * M * L::LQ, L::LQ, lane);   // Q = 1 without a rotation
                    rows.identity(lane);
                }
                apply(on);
            }
            next_slots();
        });
        if (NS == 1) rows.store(S + L::Q, L::LQ, lane);
    }
    // (the last sweep rotated nothing, so W lacks no Q; NB - 1 moves are the
    // identity, so slot b holds block b)
    // order by |lambda| descending (stable by index), or keep the diagonal
    // positions, and write out
    const double* dg = NS > 1 ? G : S0;
    constexpr int LD1 = (NS > 1 ? LG : L::LS) + 1;
    if (t < n) {
        const double li = dg[t * LD1], ai = fabs(li);
        int k = t;
        if (!D.natural) {
            k = 0;
            for (int j = 0; j < n; ++j) {
                const double aj = fabs(dg[j * LD1]);
                k += (aj > ai) || (aj == ai && j < t);
            }
        }
        pos[t] = k;
        D.lam[k] = li;
    }
    __syncthreads();
    if (polish && sweeps > 0) {   // (W = 1 without a rotation)
        // One Newton step towards the nearest orthogonal matrix,
        // X <- (3/2 - X X^T / 2) X for X = W^T: a few hundred rotations leave
        // W^T W off by ~1e-14, which singular vectors of close values feel as
        // 1e-14 over their gap; the step leaves ~1e-15.  X takes G's place
        // (n > 32), 3/2 - X X^T / 2 the block pairs' (n > 32) or S's.
        constexpr int NX = NS > 1 ? NP : M, T = (NX + 15) / 16, LC = NS > 1 ? LG : L::LS;
        static_assert(NX * LC <= (NS > 1 ? NS * L::DOUBLES : M * L::LS), "place for X X^T");
        double* X = NS > 1 ? G : S + L::Q;
        double* C = S0;
        if (NS > 1 && role == STRIPS) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        X[JB * b + 4 * q + (lane >> 4) + (JB * (st0 + h) + (lane & 15)) * LG] = wt[h][b][q];
        }
        __syncthreads();
        // entry (i, r) of X, 0 past its edge
        auto x = [&](int i, int r) {
            const int ic = NX % 16 ? min(i, NX - 1) : i, rc = NX % 16 ? min(r, NX - 1) : r;
            const double v = NS > 1 ? X[ic + rc * LG] : X[rc + ic * L::LQ];
            return NX % 16 && (i != ic || r != rc) ? 0.0 : v;
        };
        const int l0 = lane & 15, l1 = lane >> 4;
        for (int u = w; u < T * (T + 1) / 2; u += L::WAVES) {
            int J = 0;
            while ((J + 1) * (J + 2) / 2 <= u) ++J;
            const int I = u - J * (J + 1) / 2;
            dbl4 c = dbl4{0, 0, 0, 0}, c2 = dbl4{0, 0, 0, 0};
#pragma unroll 4
            for (int kk = 0; kk < NX; kk += 8) {
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(x(16 * I + l0, kk + l1), x(16 * J + l0, kk + l1), c,
                                                         0, 0, 0);
                c2 = __builtin_amdgcn_mfma_f64_16x16x4f64(x(16 * I + l0, kk + 4 + l1),
                                                          x(16 * J + l0, kk + 4 + l1), c2, 0, 0, 0);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = 16 * I + 4 * q + l1, j = 16 * J + l0;
                const double v = (i == j ? 1.5 : 0.0) - 0.5 * (c[q] + c2[q]);
                if (NX % 16 == 0 || (i < NX && j < NX)) {
                    C[i + j * LC] = v;
                    C[j + i * LC] = v;
                }
            }
        }
        __syncthreads();
        for (int u = w; u < T * T; u += L::WAVES) {
            const int I = u / T, R = u - I * T;   // eigenvectors 16 I .., rows 16 R ..
            const int ic = NX % 16 ? min(16 * I + l0, NX - 1) : 16 * I + l0;
            dbl4 c = dbl4{0, 0, 0, 0}, c2 = dbl4{0, 0, 0, 0};
#pragma unroll 4
            for (int kk = 0; kk < NX; kk += 8) {
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(C[ic + (kk + l1) * LC], x(kk + l1, 16 * R + l0), c,
                                                         0, 0, 0);
                c2 = __builtin_amdgcn_mfma_f64_16x16x4f64(C[ic + (kk + 4 + l1) * LC],
                                                          x(kk + 4 + l1, 16 * R + l0), c2, 0, 0, 0);
            }
            const int r = 16 * R + l0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = 16 * I + 4 * q + l1;
                if (i < n && r < n) D.W[r + (int64_t)pos[i] * D.ldw] = c[q] + c2[q];
            }
        }
    } else if constexpr (NS == 1) {
        for (int e = t; e < n * M; e += NT) {
            const int i = e / M, r = e - i * M;
            if (r < n) D.W[r + (int64_t)pos[i] * D.ldw] = S[L::Q + r + i * L::LQ];
        }
    } else if (role == STRIPS) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = JB * (st0 + h) + (lane & 15);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = JB * b + 4 * q + (lane >> 4);
                    if (i < n && r < n) D.W[r + (int64_t)pos[i] * D.ldw] = wt[h][b][q];
                }
        }
    }
    if (t == 0 && D.sweeps) *D.sweeps = sweeps;
}

constexpr int JAC_TMAX = 64 * JacLds<JM, 3>::WAVES;

__global__ __launch_bounds__(JAC_TMAX) void k_jacobi(const JacobiDesc* __restrict__ descs,
                                                     int nd, double tol, int max_sweeps, bool polish) {
    extern __shared__ double lds[];
    const JacobiDesc D = descs[blockIdx.x];
    if (D.skip && *D.skip) return;
    // by the problem's own size, never by the rest of its group
    if (D.n <= 16) jacobi_body<16, 1>(D, lds, tol, max_sweeps, polish);
    else if (D.n <= 24) jacobi_body<24, 1>(D, lds, tol, max_sweeps, polish);
    else if (D.n <= JM) jacobi_body<JM, 1>(D, lds, tol, max_sweeps, polish);
    else if (D.n <= 2 * JM) jacobi_body<JM, 2>(D, lds, tol, max_sweeps, polish);
    else jacobi_body<JM, 3>(D, lds, tol, max_sweeps, polish);
}

// ------------------------------------------------ stopping rule
// Stopping rule of the block iteration by one wave, after an iteration whose
// l values (largest first, pivots up to k_cholqr's tolerance) are in sv: the contraction of the top-k subspace,
// (sv_l / sv_k)^2 (or ^1), is accumulated from iteration min_iters on, and the
// problem is done below the target or at max_iters; one that will be
// factorised whole anyway stops once even twice its current rate could not
// reach the target in the iterations left.
__device__ __forceinline__ void conv_step(const ConvDesc& D, const double* sv, const ConvRule& rule,
                                          int lane, bool noisy = false) {
    // the last of the k wanted values above the null threshold
    int kk = 0;
    const double top = sv[0];
    for (int i0 = 0; i0 < D.kmax; i0 += 64) {
        const int i = i0 + lane;
        const unsigned long long b = __ballot(i < D.kmax && sv[min(i, D.kmax - 1)] > rule.null_rtol * top);
        if (b) kk = i0 + 64 - __clzll((long long)b);
    }
    if (lane != 0) return;
    const int it = *D.it + 1;
    double r = 0.0;
    if (kk > 0 && sv[kk - 1] > 0.0) {
        r = sv[D.l - 1] / sv[kk - 1];
        if (D.squared) r *= r;
        r = fmin(r, 1.0);
    }
    // (2 stands for 1 after a first step with columns below its resolution:
    // the next pivots are too small, their ratio does not count)
    double prod = *D.prod;
    if (prod > 1.0) prod = 1.0;
    else if (it >= rule.min_iters) prod *= r;
    if (it == 1 && noisy) prod = 2.0;
    *D.it = it;
    *D.prod = prod;
    if ((it >= rule.min_iters && prod < rule.target) || it >= rule.max_iters) *D.done = 1;
    else if (D.whole_ok && rule.stall_from > 0 && it >= rule.stall_from && it >= rule.min_iters &&
             prod * pow(r, 2.0 * (rule.max_iters - it)) >= rule.target)
        *D.done = 1;
}

// ------------------------------------------------ pivoted Cholesky QR
// One workgroup per n x n Gram matrix G = Y^T Y (n <= LMAX):
// diagonal-pivoted Cholesky G[p, p] = R^T R, stopped where the largest
// remaining diagonal falls to null_rel2 * max diag(G) (numerical rank r),
// then X = R^{-1} (r x r).  Output W = P X (W[perm[i], j] = X[i, j], zero
// columns from r on), so that Y W = Q has orthonormal columns spanning
// span(Y), ordered by decreasing pivot; lam[j] = R[j][j] (the norm of
// column j of Y after projecting out the earlier pivots).
//
// The n pivot steps depend on each other, so their latency is what counts.
// Steps go in panels of 16 (left-looking inside a panel): one wave, lane =
// row, finds the pivot by a 32-bit max over the wave, takes the pivot's column
// of A as the last panel left it, subtracts this panel's earlier columns (the
// lane's own row of L from registers, the pivot's from LDS) and updates the
// remaining diagonal, with no barrier.  After a panel all waves update A by
// L L^T on MFMA.  Rows are never moved: pivoted ones drop out of the search
// and get L = 0.  X comes from the 16 x 16 diagonal blocks' inverses (lane =
// column) and, by distance from the diagonal, X_IJ = -X_II sum_K R_IK X_KJ on
// MFMA, the sum's result layout being the next product's operand layout.
// The pivot search compares the leading 14 (n <= 64) or 13 bits of d's mantissa
// and settles ties by the lowest index: a pivot within 2^-14 (2^-13 = 1.2e-4) of
// the largest serves as well, and the result is a function of G.  So the pivots,
// and lam, descend up to that tolerance only.  G is taken as the
// product of one GEMM, whose two triangles agree bit for bit.
// Measured (average launch in whole runs) against the former kernels, which
// updated all of A and solved for X column by column after every pivot, in one
// wave (n <= 64) or four: 39.6 -> 11.6 us at n = 32, 77 -> 22 at 64, 154 -> 46
// at 96.  A pivot step takes 0.23 us (0.38 with the control flow in vector
// registers and keys converted to single precision).

template <int N>
struct CholLds {
    static constexpr int LD = N + 2;   // A, R, X by columns; L by rows (in X's place)
    static constexpr int ROWS = (N + 63) / 64, BITS = N > 64 ? 7 : 6;
    static constexpr int WAVES = 8;
    static constexpr size_t BYTES =
        2 * (size_t)N * LD * sizeof(double) + 2 * N * sizeof(double) + (3 * N + 2) * sizeof(int);
};

// Largest of x over the wave: within each row of 16 lanes by lane swaps, then
// across rows (the broadcasts of the row before and of lane 31), read from
// lane 63.
template <int CTRL>
__device__ __forceinline__ int max_dpp(int x) {
    return max(x, __builtin_amdgcn_update_dpp(INT32_MIN, x, CTRL, 0xF, 0xF, false));
}

__device__ __forceinline__ int wave_max_i32(int x) {
    x = max_dpp<0xB1>(x);    // quad_perm [1, 0, 3, 2]
    x = max_dpp<0x4E>(x);    // quad_perm [2, 3, 0, 1]
    x = max_dpp<0x141>(x);   // row_half_mirror
    x = max_dpp<0x140>(x);   // row_mirror
    x = max_dpp<0x142>(x);   // row_bcast 15
    x = max_dpp<0x143>(x);   // row_bcast 31
    return __builtin_amdgcn_readlane(x, 63);
}

//
// A small Y (cholqr_fused: its copy fits the LDS beside A and X) comes with the
// job: G = Y^T Y and U = Y W are formed here, without their two launches (5 us
// each and the gaps between).  The one workgroup takes 5 us longer at 128 x 32, 8
// at 256 x 32; larger Y are the GEMM's, which has the whole chip.  Measured: ATRG
// Z2 chi 16 (128 x 32) 23.5 -> 21.0 ms, BTRG Z2 chi 16 11.7 -> 10.9, HOTRG chi 16
// (256 x 32) 12.4 -> 12.0.
//
// SPAN: the basis must keep all n directions.  G resolves a column down to
// 1e-7 of its own norm; what it has left below that (d <= SPAN_FLOOR G_pp) is
// noise, and dropping or eliminating with such a column would lose its direction
// for good (after a random start, every eigenvalue below 1e-8 of the
// largest).  It stays as it is, less the resolved pivots and divided by that
// floor: the next product's columns are graded and resolve it.  lam of such
// a column is the floor, the stopping rule is told.
constexpr double SPAN_FLOOR = 1e-14;

// G into A, zero up to m x m.  Every lane loads (clamped, in bounds), so the
// loads are not predicated and stay in flight together.
template <int N>
__device__ __forceinline__ void chol_load(const JacobiDesc& D, double* A, int n, int m) {
    constexpr int LD = CholLds<N>::LD, NT = 64 * CholLds<N>::WAVES;
    const int t = threadIdx.x;
#pragma unroll 8
    for (int e = t; e < m * N; e += NT) {
        const int c = e / N, r = e - c * N;
        const double v = D.G[min(r, n - 1) + (int64_t)min(c, n - 1) * D.ldg];
        A[r + c * LD] = r < n && c < n ? v : 0.0;
    }
}

// A = Y^T Y (zero beyond n) by way of a copy of Y in LDS, summed over the rows
// in the order of the GEMM kernels (rows < 512: one K chunk).
template <int N>
__device__ __forceinline__ void chol_gram(const CholDesc& D, double* A, double* Yl, int n) {
    constexpr int LD = CholLds<N>::LD, NT = 64 * CholLds<N>::WAVES;
    const int t = threadIdx.x, lane = t & 63, l0 = lane & 15, l1 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int T = (n + 15) / 16, m = 16 * T, ld = cholqr_ldy(D.rows), rows16 = ld - 2;
    gconst_double* Y = as_global(D.Y);
    // 64 rows of a column a wave and load, eight loads in flight (p / rc by a
    // 16-bit reciprocal, exact below 65536 / rc)
    const int rc = (rows16 + 63) / 64, inv = 65536 / rc + 1;
    for (int p0 = w; p0 < m * rc; p0 += 8 * CholLds<N>::WAVES) {
        double v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int p = min(p0 + i * CholLds<N>::WAVES, m * rc - 1), c = (p * inv) >> 16;
            const int r = 64 * (p - c * rc) + lane;
            v[i] = Y[min(r, D.rows - 1) + (int64_t)min(c, n - 1) * D.ldy];
            if (r >= D.rows || c >= n) v[i] = 0.0;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int p = p0 + i * CholLds<N>::WAVES, c = (p * inv) >> 16, r = 64 * (p - c * rc) + lane;
            if (p < m * rc && r < rows16) Yl[r + c * ld] = v[i];
        }
    }
    for (int e = t; e < m * N; e += NT)
        if (e % N >= m) A[e % N + (e / N) * LD] = 0.0;
    __syncthreads();
    for (int u = w; u < T * (T + 1) / 2; u += CholLds<N>::WAVES) {
        int J = 0;
        while ((J + 1) * (J + 2) / 2 <= u) ++J;
        const int I = u - J * (J + 1) / 2;
        dbl4 c = dbl4{0, 0, 0, 0};
        const double *a = Yl + l1 + (16 * I + l0) * ld, *b = Yl + l1 + (16 * J + l0) * ld;
        for (int k = 0; k < rows16; k += 16) {
            double x[4], y[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = a[k + 4 * q], y[q] = b[k + 4 * q];
#pragma unroll
            for (int q = 0; q < 4; ++q) c = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q], y[q], c, 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * I + l1 + 4 * q, s = 16 * J + l0;
            A[r + s * LD] = c[q];
            if (I != J) A[s + r * LD] = c[q];
        }
    }
}

// U = Y W = Y P X from the copy of Y.
template <int N>
__device__ __forceinline__ void chol_rotate(const CholDesc& D, const double* X, const double* Yl, const int* perm,
                                            int rank, int n) {
    constexpr int LD = CholLds<N>::LD;
    const int lane = threadIdx.x & 63, l0 = lane & 15, l1 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int T = (n + 15) / 16, ld = cholqr_ldy(D.rows), RT = (D.rows + 15) / 16;
    for (int u = w; u < RT * T; u += CholLds<N>::WAVES) {
        const int I = u % RT, J = u / RT, row = 16 * I + l0;
        dbl4 c = dbl4{0, 0, 0, 0};
        for (int K = 0; K <= J; ++K)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int k = 16 * K + 4 * kk + l1;
                const double a = k < rank ? Yl[row + perm[min(k, rank - 1)] * ld] : 0.0;
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(a, X[k + (16 * J + l0) * LD], c, 0, 0, 0);
            }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * I + l1 + 4 * q, j = 16 * J + l0;
            if (r < D.rows && j < n) as_global(D.U)[r + (int64_t)j * D.ldu] = c[q];
        }
    }
}

// The pivot steps on A (m columns of N rows in LDS, zero beyond n): perm, piv (pivot values),
// *rank_ and the rows of L in X.  True if a column was noise (SPAN; in the
// panel wave).
template <int N, bool SPAN>
__device__ __forceinline__ bool chol_panels(double* A, double* X, double* piv, int* perm, int* iperm, int* rank_,
                                            int n, double null_rel2) {
    using L = CholLds<N>;
    constexpr int LD = L::LD, ROWS = L::ROWS;
    const int t = threadIdx.x, lane = t & 63, l0 = lane & 15, l1 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int T = (n + 15) / 16;
    if (t < N) iperm[t] = -1;
    if (t == 0) *rank_ = n;
    __syncthreads();
    // what is left of the diagonal (panel wave); -1 in a pivoted row, whose
    // entries of L, A and R-to-be past its own step are not used
    double d[ROWS], dfloor[ROWS];
    double nfloor = 0.0;
    bool noisy = false;
    if (w == 0) {
        double dmax = 0.0;
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
            const int i = lane + 64 * q;
            d[q] = i < n ? A[min(i, n - 1) * (LD + 1)] : -1.0;
            dfloor[q] = i < n ? SPAN_FLOOR * d[q] : -1.0;
            dmax = fmax(dmax, d[q]);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, o, 64));
        nfloor = null_rel2 * dmax;
    }
    for (int pb = 0; pb < T; ++pb) {
        if (w == 0) {
            const int steps = min(16, n - 16 * pb);
            double lr[ROWS][16];
            int pv = 0, vl = 0, vh = 0, stop = 16;   // lane jj: pivot row and value of step jj
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
                if (stop < 16) continue;
                constexpr int LOW = (1 << L::BITS) - 1;
                int key = INT32_MIN;
#pragma unroll
                for (int q = 0; q < ROWS; ++q)
                    key = max(key, (__double2hiint(d[q]) & ~LOW) | (LOW - (lane + 64 * q)));
                // (NaNs spread to the spare lanes' d, and their signs order them
                // at will: a row of the matrix all the same)
                const int p = min(LOW - (wave_max_i32(key) & LOW), n - 1);
                int hi, lo;
                if (ROWS > 1 && p >= 64) {
                    hi = __builtin_amdgcn_readlane(__double2hiint(d[ROWS - 1]), p - 64);
                    lo = __builtin_amdgcn_readlane(__double2loint(d[ROWS - 1]), p - 64);
                } else {
                    hi = __builtin_amdgcn_readlane(__double2hiint(d[0]), p & 63);
                    lo = __builtin_amdgcn_readlane(__double2loint(d[0]), p & 63);
                }
                const double v = __hiloint2double(hi, lo);
                // (a NaN goes on, into the results)
                if (jj >= steps || __builtin_amdgcn_readfirstlane(v <= nfloor)) {
                    stop = jj;
                    continue;
                }
                const double* ap = A + p * LD;
                const double* xp = X + p * LD + 16 * pb;
                double c[ROWS], lp[16];
#pragma unroll
                for (int q = 0; q < ROWS; ++q) c[q] = ap[min(lane + 64 * q, N - 1)];
#pragma unroll
                for (int k = 0; k < jj; ++k) lp[k] = xp[k];
                double rs = rsqrt_refined(v);
                if (SPAN) {   // (a column of noise: nothing is eliminated with it)
                    const double f = lane_read(4 * (p & 63), ROWS > 1 && p >= 64 ? dfloor[ROWS - 1] : dfloor[0]);
                    const bool noise = __builtin_amdgcn_readfirstlane(v <= f);
                    noisy = noisy || noise;
                    rs = noise ? 0.0 : rs;
                }
                pv = lane == jj ? p : pv;
                vh = lane == jj ? hi : vh;
                vl = lane == jj ? lo : vl;
#pragma unroll
                for (int q = 0; q < ROWS; ++q) {
                    const int i = lane + 64 * q;
                    double c2 = 0.0;
#pragma unroll
                    for (int k = 0; k < jj; ++k) {
                        if (k & 1) c2 = fma(-lr[q][k], lp[k], c2);
                        else c[q] = fma(-lr[q][k], lp[k], c[q]);
                    }
                    const double l = (c[q] + c2) * rs;
                    lr[q][jj] = l;
                    d[q] = i == p ? -1.0 : fma(-l, l, d[q]);
                    if (SPAN) {
                        dfloor[q] = i == p ? -1.0 : dfloor[q];
                        d[q] = d[q] < dfloor[q] ? dfloor[q] : d[q];
                    }
                    if (i < N) X[i * LD + 16 * pb + jj] = l;
                }
                wave_order();
            }
            if (lane < stop) {
                perm[16 * pb + lane] = pv;
                piv[16 * pb + lane] = __hiloint2double(vh, vl);
            }
            if (stop < steps && lane == 0) *rank_ = 16 * pb + stop;
            // no step: no column
#pragma unroll
            for (int q = 0; q < ROWS; ++q)
                for (int jj = stop; jj < 16; ++jj)
                    if (lane + 64 * q < N) X[(lane + 64 * q) * LD + 16 * pb + jj] = 0.0;
        }
        __syncthreads();
        if (*rank_ < min(n, 16 * (pb + 1)) || pb + 1 == T) break;   // (the same for every thread)
        for (int u = w; u < T * (T + 1) / 2; u += L::WAVES) {
            int J = 0;
            while ((J + 1) * (J + 2) / 2 <= u) ++J;
            const int I = u - J * (J + 1) / 2;
            dbl4 c;
            double* at = A + 16 * I + l1 + (16 * J + l0) * LD;
#pragma unroll
            for (int q = 0; q < 4; ++q) c[q] = at[4 * q];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(-X[(16 * I + l0) * LD + 16 * pb + 4 * kk + l1],
                                                         X[(16 * J + l0) * LD + 16 * pb + 4 * kk + l1], c, 0,
                                                         0, 0);
            double* ta = A + 16 * J + l0 + (16 * I + l1) * LD;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                at[4 * q] = c[q];
                if (I != J) ta[4 * q * LD] = c[q];
            }
        }
        __syncthreads();
    }
    return noisy;
}

// R in pivot order into A's place, then X = R^{-1} (identity beyond rank);
// piv becomes R[j][j].  Ends with a barrier.
template <int N>
__device__ __forceinline__ void chol_invert(double* A, double* X, double* piv, double* rinv, const int* perm,
                                            int* iperm, int rank, int n) {
    using L = CholLds<N>;
    constexpr int LD = L::LD, NT = 64 * L::WAVES;
    const int t = threadIdx.x, lane = t & 63, l0 = lane & 15, l1 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int T = (n + 15) / 16, m = 16 * T;
    // R in pivot order: R[i + k LD] = R[i][k] for i <= k < rank, else 1 / 0
    // (in A's place)
#pragma unroll 4
    for (int e = t; e < m * N; e += NT) {
        const int c = e / N, r = e - c * N;
        const double v = X[(c < rank ? perm[c] : 0) * LD + r];
        A[r + c * LD] = c < rank && r <= c ? v : (r == c ? 1.0 : 0.0);
    }
    if (t < N) {
        const double rs = t < rank ? rsqrt_refined(piv[t]) : 1.0;
        rinv[t] = rs;
        piv[t] = t < rank ? piv[t] * rs : 0.0;
        if (t < rank) iperm[perm[t]] = t;
    }
    __syncthreads();
    // diagonal blocks of X = R^{-1}, four a wave: lane = (block, column)
    for (int b0 = 4 * w; b0 < T; b0 += 4 * L::WAVES) {
        const int B = min(b0 + l1, T - 1);
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = i == l0 ? 1.0 : 0.0;
#pragma unroll
        for (int kk = 15; kk >= 0; --kk) {
            x[kk] *= rinv[16 * B + kk];
            const double* col = A + 16 * B + (16 * B + kk) * LD;
#pragma unroll
            for (int i = 0; i < kk; ++i) x[i] = fma(-col[i], x[kk], x[i]);
        }
        // (spare lanes repeat the last block)
#pragma unroll
        for (int i = 0; i < 16; ++i) X[16 * B + i + (16 * B + l0) * LD] = x[i];
    }
    __syncthreads();
    for (int dist = 1; dist < T; ++dist) {
        for (int I = w; I + dist < T; I += L::WAVES) {
            const int J = I + dist;
            dbl4 s = dbl4{0, 0, 0, 0};
            for (int K = I + 1; K <= J; ++K)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    s = __builtin_amdgcn_mfma_f64_16x16x4f64(A[16 * I + l0 + (16 * K + 4 * kk + l1) * LD],
                                                             X[16 * K + 4 * kk + l1 + (16 * J + l0) * LD], s,
                                                             0, 0, 0);
            dbl4 x = dbl4{0, 0, 0, 0};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                x = __builtin_amdgcn_mfma_f64_16x16x4f64(-X[16 * I + l0 + (16 * I + 4 * kk + l1) * LD], s[kk],
                                                         x, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) X[16 * I + l1 + 4 * q + (16 * J + l0) * LD] = x[q];
        }
        __syncthreads();
    }
}

template <int N, bool SPAN>
__global__ __launch_bounds__(64 * CholLds<N>::WAVES) void k_cholqr(const CholDesc* __restrict__ descs,
                                                                  int nd, double null_rel2,
                                                                  const ConvDesc* __restrict__ conv,
                                                                  ConvRule rule) {
    using L = CholLds<N>;
    constexpr int LD = L::LD, NT = 64 * L::WAVES;
    extern __shared__ double lds[];
    const CholDesc D = descs[blockIdx.x];
    // (the other sizes of the group are the other kernel's)
    if (D.n > N || (N > CQ64 && D.n <= CQ64) || (D.skip && *D.skip)) return;
    const int n = D.n, t = threadIdx.x, m = 16 * ((n + 15) / 16);
    double* A = lds;              // A[i + k LD]; later R in pivot order
    double* X = A + N * LD;       // L[i][j] at X[i LD + j]; later X[i + j LD]
    double* piv = X + N * LD;     // pivot values, then R[j][j]
    double* rinv = piv + N;       // 1 / R[j][j]
    int* perm = (int*)(rinv + N);
    int* iperm = perm + N;
    int* rank_ = iperm + N;
    double* Yl = lds + CholLds<N>::BYTES / sizeof(double);
    if (D.Y) chol_gram<N>(D, A, Yl, n);
    else chol_load<N>(D, A, n, m);
    const bool noisy = chol_panels<N, SPAN>(A, X, piv, perm, iperm, rank_, n, null_rel2);
    const int rank = *rank_;
    chol_invert<N>(A, X, piv, rinv, perm, iperm, rank, n);
    // W[perm[r]][c] = X[r][c] for r <= c < rank, zero elsewhere
#pragma unroll 4
    for (int e = t; e < n * N; e += NT) {
        const int c = e / N, r = e - c * N;
        const int ip = iperm[r];
        if (r < n)
            D.W[r + (int64_t)c * D.ldw] = ip >= 0 && ip <= c && c < rank ? X[ip + c * LD] : 0.0;
    }
    if (D.Y) chol_rotate<N>(D, X, Yl, perm, rank, n);
    if (t < n) D.lam[t] = piv[t];
    if (t == 0 && D.sweeps) *D.sweeps = 0;
    // (a problem that is done needs no product with W any more)
    if (conv && t < 64) conv_step(conv[blockIdx.x], piv, rule, t, noisy);
}

// ------------------------------------------- basis for a Jacobi solve
// One workgroup per n x n Gram matrix G = Y^T Y (n <= LMAX): an orthogonal Q
// (n x n, into W) for which (Y Q)^T (Y Q) is far closer to diagonal than G, in
// decreasing order.  G = P R^T R P^T by diagonal pivoting; the QR factor of
// R^T, from the Cholesky factor of H = R R^T, gives Q = P R^T P2 R2^{-1}:
// one step of the QR iteration on G, which scales entry (i, j) by about
// sigma_j^2 / sigma_i^2.  The rows of R are graded and well conditioned after
// scaling, so Q is orthogonal to ~1e-14 whatever the spectrum; a Newton
// step Q (3 - Q^T Q) / 2 makes it 1e-16.  What G does not resolve (below
// 1e-8 of the largest singular value) is kept as it is (SPAN) and resolved
// in a second round, on the Gram matrix of the graded columns Y Q.
// Two rounds take the spectra of TRG and BTRG blocks (twelve decades) from
// 20 + 8 Jacobi sweeps in two passes to 4 - 6 in one, and whole solves, copies
// included, from 0.50 to 0.34 ms at n = 32, 1.15 to 0.49 at 64, 2.45 to 0.88 at
// 85; singular values and vectors come out closer to orthogonal than from two
// Jacobi passes.  Like k_cholqr bound by the chain of pivot steps.
template <int N>
__global__ __launch_bounds__(64 * CholLds<N>::WAVES) void k_precond(const JacobiDesc* __restrict__ descs,
                                                                   int nd) {
    using L = CholLds<N>;
    constexpr int LD = L::LD, NT = 64 * L::WAVES, TMAX = N / 16;
    extern __shared__ double lds[];
    const JacobiDesc D = descs[blockIdx.x];
    // (the other sizes of the group are the other kernel's)
    if (D.n > N || (N > CQ64 && D.n <= CQ64) || (D.skip && *D.skip)) return;
    const int n = D.n, t = threadIdx.x, lane = t & 63, l0 = lane & 15, l1 = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int T = (n + 15) / 16, m = 16 * T;
    double* A = lds;
    double* B = A + N * LD;
    double* piv = B + N * LD;
    double* rinv = piv + N;
    int* perm = (int*)(rinv + N);
    int* iperm = perm + N;
    int* rank_ = iperm + N;
    int* perm1 = rank_ + 2;
    chol_load<N>(D, A, n, m);
    chol_panels<N, true>(A, B, piv, perm1, iperm, rank_, n, 0.0);
    const int rank = *rank_;
    // (columns of zeros have no pivot: the rows left over, in order, with R = I)
    if (t < rank) iperm[perm1[t]] = t;
    __syncthreads();
    if (t < n && iperm[t] < 0) {
        int at = rank;
        for (int i = 0; i < t; ++i) at += iperm[i] < 0;
        if (at < n) perm1[at] = t;
    }
    // R[i + c LD], here and in W until Q is formed
#pragma unroll 4
    for (int e = t; e < m * N; e += NT) {
        const int c = e / N, r = e - c * N;
        const double v = B[(c < rank ? perm1[c] : 0) * LD + r];
        const double x = c < rank && r < c ? v : (r != c ? 0.0 : c < rank ? sqrt(piv[c]) : 1.0);
        A[r + c * LD] = x;
        if (r < n && c < n) D.W[r + (int64_t)c * D.ldw] = x;
    }
    __syncthreads();
    // H = R R^T, both triangles, zero below as chol_panels takes it
    for (int e = t; e < m * N; e += NT)
        if (e % N >= m) B[e % N + (e / N) * LD] = 0.0;
    for (int u = w; u < T * (T + 1) / 2; u += L::WAVES) {
        int J = 0;
        while ((J + 1) * (J + 2) / 2 <= u) ++J;
        const int I = u - J * (J + 1) / 2;
        dbl4 c = dbl4{0, 0, 0, 0};
        for (int K = J; K < T; ++K)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int at = (16 * K + 4 * kk + l1) * LD + l0;
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(A[16 * I + at], A[16 * J + at], c, 0, 0, 0);
            }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = 16 * I + l1 + 4 * q, s = 16 * J + l0;
            const double x = r < n && s < n ? c[q] : 0.0;
            B[r + s * LD] = x;
            if (I != J) B[s + r * LD] = x;
        }
    }
    __syncthreads();
    chol_panels<N, true>(B, A, piv, perm, iperm, rank_, n, 0.0);
    chol_invert<N>(B, A, piv, rinv, perm, iperm, *rank_, n);
    // the rows of R in H's pivot order (clamped: perm is not written past a rank
    // below n)
#pragma unroll 4
    for (int e = t; e < m * N; e += NT) {
        const int c = e / N, k = e - c * N;
        const int row = (int)min((unsigned)perm[min(k, n - 1)], (unsigned)(n - 1));
        const double v = D.W[row + (int64_t)min(c, n - 1) * D.ldw];
        B[k + c * LD] = k < n && c < n ? v : 0.0;
    }
    __syncthreads();
    // Q (rows in the order of perm1) = R^T X in tiles of 16, kept until all
    // waves have read B
    constexpr int PER = (TMAX * TMAX + L::WAVES - 1) / L::WAVES;
    dbl4 q[PER];
#pragma unroll
    for (int s = 0; s < PER; ++s) {
        const int u = w + s * L::WAVES;
        q[s] = dbl4{0, 0, 0, 0};
        if (u >= T * T) continue;
        const int I = u % T, J = u / T;
        for (int K = 0; K <= J; ++K)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int at = 16 * K + 4 * kk + l1;
                q[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(B[at + (16 * I + l0) * LD], A[at + (16 * J + l0) * LD],
                                                            q[s], 0, 0, 0);
            }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < PER; ++s) {
        const int u = w + s * L::WAVES;
        if (u >= T * T) continue;
#pragma unroll
        for (int x = 0; x < 4; ++x) B[16 * (u % T) + l1 + 4 * x + (16 * (u / T) + l0) * LD] = q[s][x];
    }
    __syncthreads();
    // S = Q^T Q in A's place
    for (int u = w; u < T * (T + 1) / 2; u += L::WAVES) {
        int J = 0;
        while ((J + 1) * (J + 2) / 2 <= u) ++J;
        const int I = u - J * (J + 1) / 2;
        dbl4 c = dbl4{0, 0, 0, 0};
        for (int k = l1; k < m; k += 4)
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(B[k + (16 * I + l0) * LD], B[k + (16 * J + l0) * LD], c, 0, 0,
                                                     0);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int r = 16 * I + l1 + 4 * x, s = 16 * J + l0;
            A[r + s * LD] = c[x];
            if (I != J) A[s + r * LD] = c[x];
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < PER; ++s) {
        const int u = w + s * L::WAVES;
        if (u >= T * T) continue;
        const int I = u % T, J = u / T;
        dbl4 c = dbl4{0, 0, 0, 0};
        for (int k = l1; k < m; k += 4)
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(B[16 * I + l0 + k * LD], A[k + (16 * J + l0) * LD], c, 0, 0, 0);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int r = 16 * I + l1 + 4 * x, j = 16 * J + l0;
            if (r < n && j < n)
                D.W[min((unsigned)perm1[r], (unsigned)(n - 1)) + (int64_t)j * D.ldw] =
                    fma(-0.5, c[x], 1.5 * q[s][x]);
        }
    }
}

// ------------------------------------------------- column norms / normalise
// sigma_j = ||Y[:, j]||; U[:, j] = Y[:, j] / sigma_j, or 0 when
// sigma_j <= rtol * max_j sigma_j (numerical null direction).  Two launches
// over (problem, group of CN_COLS columns) workgroups, one wave per column,
// so even one problem spreads over many CUs: k_colnorm_part writes the
// raw norms, k_colnorm_scale takes the largest of them and normalises.  A
// lane keeps four partial sums over rows 256 apart (four loads in flight),
// adds them in a fixed order and the wave reduces with a fixed butterfly,
// so the result does not depend on scheduling.
constexpr int CN_COLS = 4;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__global__ __launch_bounds__(64 * CN_COLS) void k_colnorm_part(const ColDesc* __restrict__ descs,
                                                              int nd) {
    const ColDesc D = descs[blockIdx.x];
    const int lane = threadIdx.x & 63, j = blockIdx.y * CN_COLS + (threadIdx.x >> 6);
    if (j >= D.ncol || (D.skip && *D.skip)) return;
    const double* y = D.Y + (int64_t)j * D.ldy;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int i = lane;
    for (; i + 192 < D.nrow; i += 256) {
        const double y0 = y[i], y1 = y[i + 64], y2 = y[i + 128], y3 = y[i + 192];
        a0 = fma(y0, y0, a0); a1 = fma(y1, y1, a1); a2 = fma(y2, y2, a2); a3 = fma(y3, y3, a3);
    }
    for (; i < D.nrow; i += 64) a0 = fma(y[i], y[i], a0);
    const double acc = wave_sum((a0 + a1) + (a2 + a3));
    if (lane == 0) D.sigma[j] = sqrt(acc);   // raw norm
}

// Every workgroup of a problem reads all its raw norms for the largest one;
// a column zeroed as null is never the largest, so the workgroups that
// zero theirs do not change what the others read.
__global__ __launch_bounds__(64 * CN_COLS) void k_colnorm_scale(const ColDesc* __restrict__ descs,
                                                               int nd, double rtol) {
    __shared__ double wmax[CN_COLS];
    const ColDesc D = descs[blockIdx.x];
    if (blockIdx.y * CN_COLS >= D.ncol || (D.skip && *D.skip)) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, j = blockIdx.y * CN_COLS + w;
    double smax = 0.0;
    for (int c = t; c < D.ncol; c += 64 * CN_COLS) smax = fmax(smax, D.sigma[c]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) smax = fmax(smax, __shfl_xor(smax, o, 64));
    if (lane == 0) wmax[w] = smax;
    __syncthreads();
    smax = wmax[0];
    for (int q = 1; q < CN_COLS; ++q) smax = fmax(smax, wmax[q]);
    if (j >= D.ncol) return;
    const double sj = D.sigma[j];
    const bool live = sj > rtol * smax && sj > 0.0;
    const double inv = live ? 1.0 / sj : 0.0;
    const double* y = D.Y + (int64_t)j * D.ldy;
    double* u = D.U + (int64_t)j * D.ldu;
    int i = lane;
    for (; i + 192 < D.nrow; i += 256) {
        const double y0 = y[i], y1 = y[i + 64], y2 = y[i + 128], y3 = y[i + 192];
        u[i] = y0 * inv; u[i + 64] = y1 * inv; u[i + 128] = y2 * inv; u[i + 192] = y3 * inv;
    }
    for (; i < D.nrow; i += 64) u[i] = y[i] * inv;
    if (lane == 0 && !live) D.sigma[j] = 0.0;
}

// ------------------------------------------------ pivoted-row SVD gauge
// One 256-thread workgroup per SVD problem.  For each cluster of columns
// [i0, i0 + d) of U (m x k) the new basis is u_t = U_c c_t with
//   rn(r) = |U_c[r, :]|^2 - sum_{s<t} (U_c[r, :] . c_s)^2   (residual row norm)
//   r_t   = first row with rn(r) >= (1 - tie) * max_r rn(r)
//   c_t   = (U_c[r_t, :]^T - sum_{s<t} c_s (U_c[r_t, :] . c_s)) / sqrt(rn(r_t)),
// i.e. the normalised projection of the coordinate vector e_{r_t} onto the
// part of span(U_c) orthogonal to u_0..u_{t-1}; the c_t are the columns of
// the cluster's diagonal block of Q (a lone vector only gets its sign,
// exactly +-1).  Every column of Q is written once.
constexpr int CNT = 256;

__device__ __forceinline__ double canon_resid(const double* __restrict__ U, int ldu, int r, int i0,
                                              int d, const double* Cq, int tt) {
    double rn = 0.0;
    for (int j = 0; j < d; ++j) {
        const double x = U[r + (int64_t)(i0 + j) * ldu];
        rn += x * x;
    }
    for (int s = 0; s < tt; ++s) {
        double pj = 0.0;
        for (int j = 0; j < d; ++j) pj += U[r + (int64_t)(i0 + j) * ldu] * Cq[j + s * d];
        rn -= pj * pj;
    }
    return rn;
}

__global__ __launch_bounds__(CNT) void k_canon(const CanonDesc* __restrict__ descs, int nd,
                                               double tie) {
    extern __shared__ double lds[];
    __shared__ double rv[CNT / 64];
    __shared__ int ri[CNT / 64];
    __shared__ double s_max, s_rn;
    __shared__ int s_row;
    const CanonDesc D = descs[blockIdx.x];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, k = D.k;
    double* Cq = lds;                   // d x d, column-major, ld d
    double* xr = Cq + (size_t)k * k;    // U_c[r_t, :]
    double* pr = xr + k;                // U_c[r_t, :] . c_s
    for (int c = 0; c < D.nc; ++c) {
        const int i0 = D.cl[c], d = D.cl[c + 1] - i0;
        for (int tt = 0; tt < d; ++tt) {
            double best = -1.0;
            for (int r = t; r < D.m; r += CNT)
                best = fmax(best, canon_resid(D.U, D.ldu, r, i0, d, Cq, tt));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) best = fmax(best, __shfl_xor(best, o, 64));
            if (lane == 0) rv[w] = best;
            __syncthreads();
            if (t == 0) {
                double m = rv[0];
                for (int q = 1; q < CNT / 64; ++q) m = fmax(m, rv[q]);
                s_max = m;
            }
            __syncthreads();
            const double thr = (1.0 - tie) * s_max;
            int first = 0x7fffffff;
            for (int r = t; r < D.m; r += CNT)
                if (canon_resid(D.U, D.ldu, r, i0, d, Cq, tt) >= thr) {
                    first = r;
                    break;
                }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
            if (lane == 0) ri[w] = first;
            __syncthreads();
            if (t == 0) {
                int m = ri[0];
                for (int q = 1; q < CNT / 64; ++q) m = min(m, ri[q]);
                s_row = m;
            }
            __syncthreads();
            const int r = s_row < D.m ? s_row : 0;     // NaN input: no row qualifies
            for (int j = t; j < d; j += CNT) xr[j] = D.U[r + (int64_t)(i0 + j) * D.ldu];
            __syncthreads();
            for (int s = t; s < tt; s += CNT) {
                double pj = 0.0;
                for (int j = 0; j < d; ++j) pj += xr[j] * Cq[j + s * d];
                pr[s] = pj;
            }
            __syncthreads();
            if (t == 0) {
                double rn = 0.0;
                for (int j = 0; j < d; ++j) rn += xr[j] * xr[j];
                for (int s = 0; s < tt; ++s) rn -= pr[s] * pr[s];
                s_rn = rn;
            }
            __syncthreads();
            const double inv = s_rn > 0.0 ? 1.0 / sqrt(s_rn) : 0.0;
            if (d == 1) {                 // a lone vector: only its sign
                if (t == 0) Cq[0] = xr[0] >= 0.0 ? 1.0 : -1.0;
                __syncthreads();
                break;
            }
            for (int j = t; j < d; j += CNT) {
                double cj = xr[j];
                for (int s = 0; s < tt; ++s) cj -= Cq[j + s * d] * pr[s];
                Cq[j + tt * d] = cj * inv;
            }
            __syncthreads();
        }
        for (int e = t; e < k * d; e += CNT) {
            const int jj = e / k, i = e - jj * k;
            D.Q[i + (int64_t)(i0 + jj) * k] = (i >= i0 && i < i0 + d) ? Cq[(i - i0) + jj * d] : 0.0;
        }
        __syncthreads();
    }
    for (int e = t; e < k * (k - D.knn); e += CNT) {
        const int jj = D.knn + e / k, i = e % k;
        D.Q[i + (int64_t)jj * k] = (i == jj) ? 1.0 : 0.0;
    }
}

// ------------------------------------------------------------- dot product
// grid (DOT_PARTS, problems): workgroup b sums the chunk [b c, (b+1) c) with
// c = ceil(n / DOT_PARTS); k_dot_final adds the parts in order
__global__ __launch_bounds__(256) void k_dot_part(const DotDesc* __restrict__ descs, int nd) {
    __shared__ double wpart[4];
    const DotDesc D = descs[blockIdx.y];
    const int t = threadIdx.x;
    const int64_t c = (D.n + DOT_PARTS - 1) / DOT_PARTS;
    const int64_t i0 = (int64_t)blockIdx.x * c, i1 = min(D.n, i0 + c);
    double acc = 0.0;
    for (int64_t i = i0 + t; i < i1; i += 256) acc += D.x[i] * D.y[i];
    acc = wave_sum(acc);
    if ((t & 63) == 0) wpart[t >> 6] = acc;
    __syncthreads();
    if (t == 0) D.part[blockIdx.x] = (wpart[0] + wpart[1]) + (wpart[2] + wpart[3]);
}

__global__ __launch_bounds__(64) void k_dot_final(const DotDesc* __restrict__ descs, int nd) {
    const DotDesc D = descs[blockIdx.x];
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int b = 0; b < DOT_PARTS; ++b) s += D.part[b];
        D.out[0] = s;
    }
}

// ------------------------------------------- eigenvalues of a real matrix
// One 64-lane wavefront per matrix, the matrix in LDS (column-major, ld n+1):
//  1. balancing by powers of two (Parlett & Reinsch): row i / f, column i * f
//     while that brings the off-diagonal row and column norms closer;
//  2. Householder reduction to upper Hessenberg form;
//  3. Francis double-shift QR on the Hessenberg matrix, eigenvalues only
//     (the EISPACK hqr scheme: deflation on a negligible subdiagonal entry,
//     a 2x2 block giving a real pair or a conjugate pair, exceptional shifts
//     after 10 and 20 iterations).
// Every lane runs the same control flow on values read from LDS (the wave
// sums are xor butterflies, identical in every lane); the row and column
// updates of each step are spread over the lanes.
constexpr int EIGT = 64;
constexpr int EIG_MAXITS = 60;   // QR iterations per eigenvalue before giving up

// The solver body; `hf` holds the n x n matrix (ld n+1) and n more values:
// LDS for n <= EIG_NMAX (k_eig_hqr), the problem's workspace in global
// memory above (k_eig_hqr_g: the same code, slower memory).
__device__ __forceinline__ void eig_hqr_body(const EigDesc& D, double* hf) {
    const int nf = D.n, t = threadIdx.x, ld = nf + 1;
    double* v = hf + (size_t)nf * ld;
#define HF(i, j) hf[(i) + (j) * ld]
    for (int e = t; e < nf * nf; e += EIGT) {
        const int j = e / nf, i = e - j * nf;
        HF(i, j) = D.A[i + (int64_t)j * D.lda];
    }
    __syncthreads();
    // 0. permutation (as LAPACK's balancing 'P'): a row with no off-diagonal
    //    entry inside the active window [ilo, ihi] is swapped to ihi, a
    //    column with none to ilo; its diagonal entry is an eigenvalue and
    //    the window shrinks (exact zeros stay exact)
    int ilo = 0, ihi = nf - 1;
    auto swap_idx = [&](int a, int b) {
        if (a == b) return;
        for (int j = t; j < nf; j += EIGT) {
            const double x = HF(a, j);
            HF(a, j) = HF(b, j);
            HF(b, j) = x;
        }
        __syncthreads();
        for (int i = t; i < nf; i += EIGT) {
            const double x = HF(i, a);
            HF(i, a) = HF(i, b);
            HF(i, b) = x;
        }
        __syncthreads();
    };
    for (bool moved = true; moved && ihi >= ilo;) {
        moved = false;
        for (int j = ihi; j >= ilo && !moved; --j) {
            int nz = 0;
            for (int i = ilo + t; i <= ihi; i += EIGT)
                if (i != j && HF(j, i) != 0.0) nz = 1;
            if (!__any(nz)) {
                swap_idx(j, ihi);
                if (t == 0) {
                    D.wr[ihi] = HF(ihi, ihi);
                    D.wi[ihi] = 0.0;
                }
                --ihi;
                moved = true;
            }
        }
        for (int j = ilo; j <= ihi && !moved; ++j) {
            int nz = 0;
            for (int i = ilo + t; i <= ihi; i += EIGT)
                if (i != j && HF(i, j) != 0.0) nz = 1;
            if (!__any(nz)) {
                swap_idx(j, ilo);
                if (t == 0) {
                    D.wr[ilo] = HF(ilo, ilo);
                    D.wi[ilo] = 0.0;
                }
                ++ilo;
                moved = true;
            }
        }
        __syncthreads();
    }
#undef HF
    // the rest works on the window: n x n at (ilo, ilo), eigenvalues to wr/wi + ilo
    const int n = ihi - ilo + 1;
    double* h = hf + (size_t)ilo * (ld + 1);
    double* const wro = D.wr + ilo;
    double* const wio = D.wi + ilo;
#define HH(i, j) h[(i) + (j) * ld]
    // 1. balancing
    for (int sweep = 0; sweep < 100; ++sweep) {
        bool done = true;
        for (int i = 0; i < n; ++i) {
            double c = 0.0, r = 0.0;
            for (int j = t; j < n; j += EIGT)
                if (j != i) {
                    c += fabs(HH(j, i));
                    r += fabs(HH(i, j));
                }
            c = wave_sum(c);
            r = wave_sum(r);
            if (c != 0.0 && r != 0.0) {
                double g = r * 0.5, f = 1.0;
                const double s0 = c + r;
                while (c < g) {
                    f *= 2.0;
                    c *= 4.0;
                }
                g = r * 2.0;
                while (c > g) {
                    f *= 0.5;
                    c *= 0.25;
                }
                if ((c + r) / f < 0.95 * s0) {
                    done = false;
                    const double gi = 1.0 / f;
                    for (int j = t; j < n; j += EIGT) HH(i, j) *= gi;
                    __syncthreads();
                    for (int j = t; j < n; j += EIGT) HH(j, i) *= f;
                }
            }
            __syncthreads();
        }
        if (done) break;
    }
    // 2. Hessenberg reduction
    for (int k = 0; k + 2 < n; ++k) {
        double ss = 0.0;
        for (int i = k + 2 + t; i < n; i += EIGT) ss += HH(i, k) * HH(i, k);
        ss = wave_sum(ss);
        if (ss == 0.0) continue;
        const double x0 = HH(k + 1, k);
        const double alpha = -copysign(sqrt(x0 * x0 + ss), x0);
        const double v0 = x0 - alpha, beta = 2.0 / (v0 * v0 + ss);
        for (int i = k + 1 + t; i < n; i += EIGT) v[i] = (i == k + 1) ? v0 : HH(i, k);
        __syncthreads();
        for (int j = k + t; j < n; j += EIGT) {
            double d = 0.0;
            for (int i = k + 1; i < n; ++i) d += v[i] * HH(i, j);
            d *= beta;
            for (int i = k + 1; i < n; ++i) HH(i, j) -= d * v[i];
        }
        __syncthreads();
        for (int i = t; i < n; i += EIGT) {
            double d = 0.0;
            for (int j = k + 1; j < n; ++j) d += HH(i, j) * v[j];
            d *= beta;
            for (int j = k + 1; j < n; ++j) HH(i, j) -= d * v[j];
        }
        __syncthreads();
        if (t == 0) HH(k + 1, k) = alpha;
        for (int i = k + 2 + t; i < n; i += EIGT) HH(i, k) = 0.0;
        __syncthreads();
    }
    // 3. double-shift QR
    double anorm = 0.0;
    for (int j = t; j < n; j += EIGT)
        for (int i = 0; i <= min(j + 1, n - 1); ++i) anorm += fabs(HH(i, j));
    anorm = wave_sum(anorm);
    int nn = n - 1, info = 0;
    double tsh = 0.0;
    double p = 0.0, q = 0.0, r = 0.0, s = 0.0, w = 0.0, x = 0.0, y = 0.0, z = 0.0;
    while (nn >= 0 && !info) {
        int its = 0, l = 0;
        do {
            for (l = nn; l >= 1; --l) {
                s = fabs(HH(l - 1, l - 1)) + fabs(HH(l, l));
                if (s == 0.0) s = anorm;
                if (fabs(HH(l, l - 1)) + s == s) break;
            }
            __syncthreads();
            if (l >= 1 && t == 0) HH(l, l - 1) = 0.0;
            __syncthreads();
            x = HH(nn, nn);
            if (l == nn) {
                if (t == 0) {
                    wro[nn] = x + tsh;
                    wio[nn] = 0.0;
                }
                --nn;
            } else {
                y = HH(nn - 1, nn - 1);
                w = HH(nn, nn - 1) * HH(nn - 1, nn);
                if (l == nn - 1) {
                    p = 0.5 * (y - x);
                    q = p * p + w;
                    z = sqrt(fabs(q));
                    x += tsh;
                    if (q >= 0.0) z = p + copysign(z, p);
                    if (t == 0) {
                        if (q >= 0.0) {
                            wro[nn - 1] = wro[nn] = x + z;
                            if (z != 0.0) wro[nn] = x - w / z;
                            wio[nn - 1] = wio[nn] = 0.0;
                        } else {
                            wro[nn - 1] = wro[nn] = x + p;
                            wio[nn - 1] = z;
                            wio[nn] = -z;
                        }
                    }
                    nn -= 2;
                } else {
                    if (its == EIG_MAXITS) {
                        info = 1;
                        break;
                    }
                    if (its == 10 || its == 20) {
                        tsh += x;
                        for (int i = t; i <= nn; i += EIGT) HH(i, i) -= x;
                        __syncthreads();
                        s = fabs(HH(nn, nn - 1)) + fabs(HH(nn - 1, nn - 2));
                        y = x = 0.75 * s;
                        w = -0.4375 * s * s;
                    }
                    ++its;
                    int m = nn - 2;
                    for (; m >= l; --m) {
                        z = HH(m, m);
                        r = x - z;
                        s = y - z;
                        p = (r * s - w) / HH(m + 1, m) + HH(m, m + 1);
                        q = HH(m + 1, m + 1) - z - r - s;
                        r = HH(m + 2, m + 1);
                        s = fabs(p) + fabs(q) + fabs(r);
                        p /= s;
                        q /= s;
                        r /= s;
                        if (m == l) break;
                        const double u = fabs(HH(m, m - 1)) * (fabs(q) + fabs(r));
                        const double vv = fabs(p) * (fabs(HH(m - 1, m - 1)) + fabs(z) +
                                                     fabs(HH(m + 1, m + 1)));
                        if (u + vv == vv) break;
                    }
                    __syncthreads();
                    for (int i = m + 2 + t; i <= nn; i += EIGT) {
                        HH(i, i - 2) = 0.0;
                        if (i != m + 2) HH(i, i - 3) = 0.0;
                    }
                    __syncthreads();
                    for (int k = m; k <= nn - 1; ++k) {
                        if (k != m) {
                            p = HH(k, k - 1);
                            q = HH(k + 1, k - 1);
                            r = (k != nn - 1) ? HH(k + 2, k - 1) : 0.0;
                            x = fabs(p) + fabs(q) + fabs(r);
                            if (x != 0.0) {
                                p /= x;
                                q /= x;
                                r /= x;
                            }
                        }
                        s = copysign(sqrt(p * p + q * q + r * r), p);
                        __syncthreads();
                        if (s != 0.0) {
                            if (t == 0) {
                                if (k == m) {
                                    if (l != m) HH(k, k - 1) = -HH(k, k - 1);
                                } else {
                                    HH(k, k - 1) = -s * x;
                                }
                            }
                            p += s;
                            x = p / s;
                            y = q / s;
                            z = r / s;
                            q /= p;
                            r /= p;
                            const bool three = k != nn - 1;
                            for (int j = k + t; j <= nn; j += EIGT) {
                                double pp = HH(k, j) + q * HH(k + 1, j);
                                if (three) {
                                    pp += r * HH(k + 2, j);
                                    HH(k + 2, j) -= pp * z;
                                }
                                HH(k + 1, j) -= pp * y;
                                HH(k, j) -= pp * x;
                            }
                            __syncthreads();
                            const int mmin = nn < k + 3 ? nn : k + 3;
                            for (int i = l + t; i <= mmin; i += EIGT) {
                                double pp = x * HH(i, k) + y * HH(i, k + 1);
                                if (three) {
                                    pp += z * HH(i, k + 2);
                                    HH(i, k + 2) -= pp * r;
                                }
                                HH(i, k + 1) -= pp * q;
                                HH(i, k) -= pp;
                            }
                            __syncthreads();
                        }
                    }
                }
            }
        } while (l < nn - 1 && !info);
    }
#undef HH
    if (t == 0) D.info[0] = info;
}


__global__ __launch_bounds__(EIGT) void k_eig_hqr(const EigDesc* __restrict__ descs, int nd) {
    extern __shared__ double lds[];
    const EigDesc D = descs[blockIdx.x];
    if (D.n > EIG_NMAX) return;
    eig_hqr_body(D, lds);
}

__global__ __launch_bounds__(EIGT) void k_eig_hqr_g(const EigDesc* __restrict__ descs, int nd) {
    const EigDesc D = descs[blockIdx.x];
    if (D.n <= EIG_NMAX) return;
    eig_hqr_body(D, D.work);
}

// conv_step for values that another kernel wrote (Ritz values, where an
// option puts Rayleigh-Ritz steps into the loop), one wave per problem.
__global__ __launch_bounds__(64) void k_conv(const ConvDesc* __restrict__ descs, int nd, ConvRule rule) {
    const ConvDesc D = descs[blockIdx.x];
    if (*D.done) return;
    conv_step(D, D.sigma, rule, threadIdx.x);
}

// in-place (M + M^T)/2 of square blocks (project_hermitian)
__global__ __launch_bounds__(256) void k_symmetrize(const ColDesc* __restrict__ descs, int nd) {
    const ColDesc D = descs[blockIdx.y];
    const int64_t n = D.nrow;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * n;
         e += (int64_t)gridDim.x * blockDim.x) {
        int64_t i = e % n, j = e / n;
        if (i >= j) continue;
        double* a = const_cast<double*>(D.Y);
        double x = a[i + j * D.ldy], y = a[j + i * D.ldy];
        double m = 0.5 * (x + y);
        a[i + j * D.ldy] = m;
        a[j + i * D.ldy] = m;
    }
}

// ------------------------------------------------------ deterministic fill
__device__ __forceinline__ uint64_t splitmix(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ __launch_bounds__(256) void k_randfill(const FillDesc* __restrict__ descs, int nd,
                                                  int64_t total) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = nd - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (descs[mid].start <= e) lo = mid; else hi = mid - 1;
        }
        const FillDesc& D = descs[lo];
        int64_t r = e - D.start;
        int i = (int)(r % D.rows), j = (int)(r / D.rows);
        uint64_t h = splitmix(D.seed ^ splitmix((uint64_t)i * 0x100000001B3ull + (uint64_t)j));
        D.p[i + (int64_t)j * D.ld] = ((double)(h >> 11) * (1.0 / 9007199254740992.0)) * 2.0 - 1.0;
    }
}

// --------------------------------------------------- strided matrix gather
// out[i + j*ldo] = in[(trans ? j + i*ldi : i + j*ldi)] * rw[i] * cw[j]
__global__ __launch_bounds__(256) void k_gather(const GatherDesc* __restrict__ descs, int nd,
                                                int64_t total) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = nd - 1;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (descs[mid].start <= e) lo = mid; else hi = mid - 1;
        }
        const GatherDesc& D = descs[lo];
        int64_t r = e - D.start;
        int i = (int)(r % D.rows), j = (int)(r / D.rows);
        double v = D.trans ? D.in[(int64_t)j + (int64_t)i * D.ldi] : D.in[(int64_t)i + (int64_t)j * D.ldi];
        if (D.rw) v *= D.rw[i];
        if (D.cw) v *= D.cw[j];
        D.out[(int64_t)i + (int64_t)j * D.ldo] = v;
    }
}

// ------------------------------------------------ Frobenius norm of blocks
// Squared Frobenius norm of each problem's nrow x ncol matrix, in a fixed
// order that depends on the matrix alone: grid (FROB_PARTS, problems); part
// q sums columns [q ncol / FROB_PARTS, (q + 1) ncol / FROB_PARTS), each
// thread its rows t + 256 u into four accumulators by u mod 4 (independent
// loads in flight), then a fixed tree; k_frob_final adds the parts in order.
__global__ __launch_bounds__(256) void k_frob_part(const ColDesc* __restrict__ descs,
                                                   double* __restrict__ partial) {
    __shared__ double red[256];
    const ColDesc D = descs[blockIdx.y];
    const int q = blockIdx.x;
    const int j0 = (int)((int64_t)q * D.ncol / FROB_PARTS);
    const int j1 = (int)((int64_t)(q + 1) * D.ncol / FROB_PARTS);
    gconst_double* Y = as_global(D.Y);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int j = j0; j < j1; ++j) {
        gconst_double* y = Y + (int64_t)j * D.ldy;
        int i = threadIdx.x;
        for (; i + 768 < D.nrow; i += 1024) {
            const double a = y[i], b = y[i + 256], c = y[i + 512], d = y[i + 768];
            acc[0] += a * a;
            acc[1] += b * b;
            acc[2] += c * c;
            acc[3] += d * d;
        }
        // fewer than 1024 rows left: at most three more
        if (i < D.nrow) acc[0] += y[i] * y[i];
        if (i + 256 < D.nrow) acc[1] += y[i + 256] * y[i + 256];
        if (i + 512 < D.nrow) acc[2] += y[i + 512] * y[i + 512];
    }
    const double s = block_sum_fixed((acc[0] + acc[1]) + (acc[2] + acc[3]), red);
    if (threadIdx.x == 0) partial[(int64_t)blockIdx.y * FROB_PARTS + q] = s;
}

__global__ __launch_bounds__(64) void k_frob_final(const ColDesc* __restrict__ descs, int nd,
                                                   const double* __restrict__ partial) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nd) return;
    double s = 0.0;
    for (int q = 0; q < FROB_PARTS; ++q) s += partial[(int64_t)p * FROB_PARTS + q];
    descs[p].sigma[0] = s;
}

// ================================================================ profiling
namespace {
struct ProfState {
    std::mutex mu;
    int level = 0;
    struct Rec { hipEvent_t a, b; int kind; double flops, bytes; };
    // a completed launch's times (ms): duration, start and end since `ref`
    struct Times { float ms, t0, t1; };
    std::vector<Rec> recs;
    bool draining = false;   // one thread files a batch of records unlocked
    std::condition_variable idle;   // signalled when that batch is filed
    // with mu held (through lk): wait until no batch is being filed unlocked
    void wait_idle(std::unique_lock<std::mutex>& lk) {
        idle.wait(lk, [this] { return !draining; });
    }
    std::vector<hipEvent_t> spare;
    ProfTotals tot[PK_COUNT];
    // start / end of every filed launch (ms since `ref`), per kind: their
    // union is the kind's device-busy time (launches on different streams
    // overlap)
    hipEvent_t ref = nullptr;
    std::vector<std::pair<float, float>> spans[PK_COUNT];
    // device counters of the GEMM flops that ran (FP64, split), per device
    std::map<int, unsigned long long*> flop_ctr;
    unsigned long long* counters(int dev) {   // with mu held
        auto it = flop_ctr.find(dev);
        if (it != flop_ctr.end()) return it->second;
        unsigned long long* p = nullptr;
        TNR_HIP(hipMalloc(&p, 2 * sizeof(unsigned long long)));
        TNR_HIP(hipMemset(p, 0, 2 * sizeof(unsigned long long)));
        flop_ctr[dev] = p;
        return p;
    }
    hipEvent_t ev() {   // with mu held
        if (!spare.empty()) { hipEvent_t e = spare.back(); spare.pop_back(); return e; }
        hipEvent_t e;
        TNR_HIP(hipEventCreate(&e));
        return e;
    }
    Times times(const Rec& r) const {   // r.b has completed; no lock needed
        Times x{0, 0, 0};
        TNR_HIP(hipEventElapsedTime(&x.ms, r.a, r.b));
        TNR_HIP(hipEventElapsedTime(&x.t0, ref, r.a));
        TNR_HIP(hipEventElapsedTime(&x.t1, ref, r.b));
        return x;
    }
    void file_times(const Rec& r, const Times& x) {   // with mu held
        tot[r.kind].launches++;
        tot[r.kind].ms += x.ms;
        tot[r.kind].flops += r.flops;
        tot[r.kind].bytes += r.bytes;
        spans[r.kind].emplace_back(x.t0, x.t1);
        spare.push_back(r.a);
        spare.push_back(r.b);
    }
    void file(const Rec& r) { file_times(r, times(r)); }   // with mu held; r.b has completed
    void drain() {      // with mu held; waits for every pending launch
        for (auto& r : recs) {
            TNR_HIP(hipEventSynchronize(r.b));
            file(r);
        }
        recs.clear();
    }
};
ProfState& prof() {
    static ProfState p;
    return p;
}
}  // namespace

void prof_enable(int level) {
    ProfState& p = prof();
    std::unique_lock<std::mutex> lk(p.mu);
    p.wait_idle(lk);
    p.drain();
    p.level = level;
    for (auto& t : p.tot) t = ProfTotals();
    for (auto& v : p.spans) v.clear();
    if (level) {
        // the reference point of the launch spans, and zeroed flop counters
        // (outside any timed region: this synchronises the device)
        TNR_HIP(hipDeviceSynchronize());
        if (!p.ref) TNR_HIP(hipEventCreate(&p.ref));
        TNR_HIP(hipEventRecord(p.ref, 0));
        TNR_HIP(hipEventSynchronize(p.ref));
        for (auto& kv : p.flop_ctr) {
            int dev = 0;
            TNR_HIP(hipGetDevice(&dev));
            TNR_HIP(hipSetDevice(kv.first));
            TNR_HIP(hipMemset(kv.second, 0, 2 * sizeof(unsigned long long)));
            TNR_HIP(hipSetDevice(dev));
        }
    }
}

unsigned long long* prof_flop_counter(bool split32) {
    ProfState& p = prof();
    std::lock_guard<std::mutex> lk(p.mu);
    if (!p.level) return nullptr;
    int dev = 0;
    TNR_HIP(hipGetDevice(&dev));
    return p.counters(dev) + (split32 ? 1 : 0);
}

bool prof_enabled() { return prof_level() > 0; }

int prof_level() {
    ProfState& p = prof();
    std::lock_guard<std::mutex> lk(p.mu);
    return p.level;
}

// Launches may come from several host threads (one stream each): the
// events live in the scope object and the record is filed at its end.
ProfScope::ProfScope(hipStream_t s, int k, double f, double b)
    : st(s), kind(k), active(false), flops(f), bytes(b) {
    ProfState& p = prof();
    std::lock_guard<std::mutex> lk(p.mu);
    if (!p.level) return;
    ea = p.ev();
    eb = p.ev();
    active = true;
}

void ProfScope::bracket() {
    if (active && mode == 0) {
        TNR_HIP(hipEventRecord(ea, st));
        mode = 1;
    }
}

void ProfScope::end() {
    if (active && mode == 1 && !ended) {
        (void)hipEventRecord(eb, st);
        ended = true;
    }
}

ProfScope::~ProfScope() {
    if (!active) return;
    end();
    ProfState& p = prof();
    std::unique_lock<std::mutex> lk(p.mu);
    if (mode == 0) {   // nothing was launched
        p.spare.push_back(ea);
        p.spare.push_back(eb);
        return;
    }
    p.recs.push_back(ProfState::Rec{ea, eb, kind, flops, bytes});
    if (p.recs.size() <= 4096 || p.draining) return;
    // File the completed launches.  The event queries take a few ms for
    // thousands of records, so they run without the lock: the other lanes'
    // threads keep launching meanwhile.
    std::vector<ProfState::Rec> batch;
    batch.swap(p.recs);
    p.draining = true;
    lk.unlock();
    std::vector<std::pair<ProfState::Rec, ProfState::Times>> done;
    std::vector<ProfState::Rec> pending;
    try {
        for (const auto& r : batch) {
            if (hipEventQuery(r.b) == hipSuccess) done.emplace_back(r, p.times(r));
            else pending.push_back(r);
        }
    } catch (...) {
        pending = batch;   // try again later
        done.clear();
    }
    lk.lock();
    for (const auto& d : done) p.file_times(d.first, d.second);
    p.recs.insert(p.recs.end(), pending.begin(), pending.end());
    p.draining = false;
    p.idle.notify_all();
}

ProfTotals prof_read(int kind) {
    ProfState& p = prof();
    std::unique_lock<std::mutex> lk(p.mu);
    p.wait_idle(lk);
    p.drain();
    if (kind < 0 || kind >= PK_COUNT) return ProfTotals();
    ProfTotals t = p.tot[kind];
    // union of the launch spans
    auto v = p.spans[kind];
    std::sort(v.begin(), v.end());
    double busy = 0;
    float a = 0, b = -1;
    for (auto& s : v) {
        if (s.first > b) {
            if (b > a) busy += b - a;
            a = s.first;
            b = s.second;
        } else if (s.second > b) {
            b = s.second;
        }
    }
    if (b > a) busy += b - a;
    t.busy_ms = busy;
    if (kind == PK_GEMM_F64 || kind == PK_GEMM_SPLIT32) {
        // flops of the problems that ran, from the device counters
        TNR_HIP(hipDeviceSynchronize());
        double ran = 0;
        for (auto& kv : p.flop_ctr) {
            unsigned long long c[2] = {0, 0};
            int dev = 0;
            TNR_HIP(hipGetDevice(&dev));
            TNR_HIP(hipSetDevice(kv.first));
            TNR_HIP(hipMemcpy(c, kv.second, sizeof(c), hipMemcpyDeviceToHost));
            TNR_HIP(hipSetDevice(dev));
            ran += (double)c[kind == PK_GEMM_SPLIT32 ? 1 : 0];
        }
        t.flops_planned = t.flops;
        t.flops = ran;
    }
    return t;
}

// =================================================================== launch
static int grid_for(int64_t total, int cap = 4096) {
    int64_t g = (total + 255) / 256;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

void launch_copy(hipStream_t st, const CopyDesc* d_descs, int nd, int64_t chunks,
                 int64_t elems) {
    if (chunks <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_COPY, 0.0, 16.0 * (double)elems);
    const int grid = (int)std::min<int64_t>(chunks, 8192);
    TNR_LAUNCH(ps, k_copy, dim3(grid), dim3(256), 0, st, d_descs, nd, chunks);
    TNR_HIP(hipGetLastError());
}

void launch_transpose(hipStream_t st, const TransDesc* d_descs, int nd, int64_t tiles,
                      int64_t elems) {
    if (tiles <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_COPY, 0.0, 16.0 * (double)elems);
    const int grid = (int)std::min<int64_t>(tiles, 4096);
    TNR_LAUNCH(ps, k_transpose, dim3(grid), dim3(256), 0, st, d_descs, nd, tiles);
    TNR_HIP(hipGetLastError());
}

void launch_gemm(hipStream_t st, const GemmDesc* d_descs, int nd, int64_t tiles, bool split32,
                 double flops, int shape, bool dma) {
    if (tiles <= 0 || nd <= 0) return;
    TNR_REQUIRE(split32 || dma || !gemm_shape_kw(shape), TNR_ERR_INTERNAL, "small tiles load through LDS-DMA");
    ProfScope ps(st, split32 ? PK_GEMM_SPLIT32 : PK_GEMM_F64, flops, 0.0);
    unsigned long long* fc = ps.active ? prof_flop_counter(split32) : nullptr;
    if (split32)
        TNR_LAUNCH(ps, k_gemm_split32, dim3((unsigned)tiles), dim3(256), 0, st, d_descs, nd, fc);
    else if (shape == GEMM_KW16x1)
        TNR_LAUNCH(ps, (k_gemm_kw<1, 1, 4>), dim3((unsigned)tiles), dim3(64), 0, st, d_descs, nd, fc);
    else if (shape == GEMM_KW16x4)
        TNR_LAUNCH(ps, (k_gemm_kw<1, 4, 4>), dim3((unsigned)tiles), dim3(256), 0, st, d_descs, nd, fc);
    else if (shape == GEMM_KW32x4)
        TNR_LAUNCH(ps, (k_gemm_kw<2, 4, 4>), dim3((unsigned)tiles), dim3(256), 0, st, d_descs, nd, fc);
    else if (shape == GEMM_128x128 && dma)
        TNR_LAUNCH(ps, (k_gemm_dl<128, 128, 4, 2, 2, 3, 16>), dim3((unsigned)tiles), dim3(512), 0, st,
                           d_descs, nd, fc);
    else if (shape == GEMM_128x64 && dma)
        TNR_LAUNCH(ps, (k_gemm_dl<128, 64, 4, 2, 4, 3, 16>), dim3((unsigned)tiles), dim3(512), 0, st,
                           d_descs, nd, fc);
    else if (shape == GEMM_64x64 && dma)
        TNR_LAUNCH(ps, (k_gemm_dl<64, 64, 2, 2, 3, 3, 16>), dim3((unsigned)tiles), dim3(256), 0, st,
                           d_descs, nd, fc);
    else if (shape == GEMM_128x128)
        TNR_LAUNCH(ps, (k_gemm_f64<128, 128, 4, 2, 16>), dim3((unsigned)tiles), dim3(512), 0,
                           st, d_descs, nd, fc);
    else if (shape == GEMM_128x64)
        TNR_LAUNCH(ps, (k_gemm_f64<128, 64, 4, 2, 16>), dim3((unsigned)tiles), dim3(512), 0,
                           st, d_descs, nd, fc);
    else if (shape == GEMM_64x64_K32)
        TNR_LAUNCH(ps, (k_gemm_f64<64, 64, 2, 2, 32>), dim3((unsigned)tiles), dim3(256), 0,
                           st, d_descs, nd, fc);
    else
        TNR_LAUNCH(ps, (k_gemm_f64<64, 64, 2, 2, 16>), dim3((unsigned)tiles), dim3(256), 0,
                           st, d_descs, nd, fc);
    TNR_HIP(hipGetLastError());
}

void launch_gemm_reduce(hipStream_t st, const GemmDesc* d_descs, int nd, const int64_t* d_starts,
                        int64_t total) {
    if (total <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_GEMM_REDUCE, 0.0, 0.0);
    TNR_LAUNCH(ps, k_gemm_reduce, dim3(grid_for(total, 8192)), dim3(256), 0, st, d_descs, nd,
                       d_starts, total);
    TNR_HIP(hipGetLastError());
}

void launch_trace_normalize(hipStream_t st, const TraceDesc* d_descs, const TraceProb* d_probs,
                            int nprob, int64_t max_size) {
    if (nprob <= 0) return;
    ProfScope ps(st, PK_TRACE, 0.0, 0.0);
    ps.bracket();
    TNR_LAUNCH(ps, k_trace_partial, dim3(TRACE_PARTS, nprob), dim3(256), 0, st, d_descs,
                       d_probs);
    TNR_HIP(hipGetLastError());
    int gx = grid_for(max_size, 1024);
    TNR_LAUNCH(ps, k_normalize, dim3(gx, nprob), dim3(256), 0, st, d_probs);
    TNR_HIP(hipGetLastError());
}

void launch_jacobi(hipStream_t st, const JacobiDesc* d_descs, int nd, int nmax, double tol,
                   int max_sweeps) {
    if (nd <= 0) return;
    // once per process (thread-safe static initialisation)
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_jacobi, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)jacobi_lds_bytes(LMAX));
    TNR_HIP(attr);
    ProfScope ps(st, PK_JACOBI, 0.0, 0.0);
    TNR_LAUNCH(ps, k_jacobi, dim3(nd), dim3(jacobi_threads(nmax)), jacobi_lds_bytes(nmax), st, d_descs, nd,
               tol, max_sweeps, tol < JPOLISH_BELOW);
    TNR_HIP(hipGetLastError());
    if (ps.active && prof_level() >= 2) {
        // profiling only: the work a launch did depends on the sweeps each
        // problem took, read back after the launch (the timing events are
        // already recorded)
        ps.end();
        TNR_HIP(hipStreamSynchronize(st));
        std::vector<JacobiDesc> hd(nd);
        TNR_HIP(hipMemcpy(hd.data(), d_descs, nd * sizeof(JacobiDesc), hipMemcpyDeviceToHost));
        double fl = 0.0, by = 0.0;
        for (const JacobiDesc& d : hd) {
            int sk = 0, sw = 0;
            if (d.skip) TNR_HIP(hipMemcpy(&sk, d.skip, sizeof(int), hipMemcpyDeviceToHost));
            if (sk) continue;
            if (d.sweeps) TNR_HIP(hipMemcpy(&sw, d.sweeps, sizeof(int), hipMemcpyDeviceToHost));
            const double n = d.n;
            // per sweep: (n-1) rounds of n/2 rotations, each 18n flops on
            // G (two rows, two columns) and W (two columns)
            fl += (double)sw * (n - 1.0) * (n / 2.0) * 18.0 * n;
            by += (2.0 * n * n + n) * sizeof(double);
        }
        ps.flops = fl;
        ps.bytes = by;
    }
}


// Problems of at most CQ64 columns run on k_cholqr<64>, larger ones on
// k_cholqr<LMAX> (each kernel skips the other's), so the kernel a problem gets
// depends on its own size only, never on the rest of its launch group.
template <int N, bool SPAN>
static void launch_cholqr_n(hipStream_t st, const CholDesc* d_descs, int nd, double null_rel2,
                            const ConvDesc* d_conv, const ConvRule& rule, int64_t ylds) {
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_cholqr<N, SPAN>, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)(CholLds<N>::BYTES + (N == CQ64 ? CHOLQR_YLDS * sizeof(double) : 0)));
    TNR_HIP(attr);
    ProfScope ps(st, PK_JACOBI, 0.0, 0.0);
    TNR_LAUNCH(ps, (k_cholqr<N, SPAN>), dim3(nd), dim3(64 * CholLds<N>::WAVES),
               CholLds<N>::BYTES + (N == CQ64 ? ylds * sizeof(double) : 0), st, d_descs, nd, null_rel2, d_conv, rule);
    TNR_HIP(hipGetLastError());
}

void launch_cholqr(hipStream_t st, const CholDesc* d_descs, int nd, int nmin, int nmax,
                   double null_rel2, bool span, const ConvDesc* d_conv, const ConvRule& rule, int64_t ylds) {
    if (nd <= 0) return;
    if (nmin <= CQ64) (span ? launch_cholqr_n<CQ64, true> : launch_cholqr_n<CQ64, false>)(
        st, d_descs, nd, null_rel2, d_conv, rule, ylds);
    if (nmax > CQ64) (span ? launch_cholqr_n<LMAX, true> : launch_cholqr_n<LMAX, false>)(
        st, d_descs, nd, null_rel2, d_conv, rule, 0);
}

template <int N>
static void launch_precond_n(hipStream_t st, const JacobiDesc* d_descs, int nd) {
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_precond<N>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CholLds<N>::BYTES);
    TNR_HIP(attr);
    ProfScope ps(st, PK_JACOBI, 0.0, 0.0);
    TNR_LAUNCH(ps, k_precond<N>, dim3(nd), dim3(64 * CholLds<N>::WAVES), CholLds<N>::BYTES, st, d_descs, nd);
    TNR_HIP(hipGetLastError());
}

void launch_precond(hipStream_t st, const JacobiDesc* d_descs, int nd, int nmin, int nmax) {
    if (nd <= 0) return;
    if (nmin <= CQ64) launch_precond_n<CQ64>(st, d_descs, nd);
    if (nmax > CQ64) launch_precond_n<LMAX>(st, d_descs, nd);
}

void launch_lincomb(hipStream_t st, const LinDesc* d_descs, int nd, int64_t total) {
    if (total <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    TNR_LAUNCH(ps, k_lincomb, dim3(grid_for(total, 8192)), dim3(256), 0, st, d_descs, nd,
                       total);
    TNR_HIP(hipGetLastError());
}

void launch_colnorm(hipStream_t st, const ColDesc* d_descs, int nd, int ncol_max, double rtol) {
    if (nd <= 0 || ncol_max <= 0) return;
    const dim3 grid(nd, (ncol_max + CN_COLS - 1) / CN_COLS);
    ProfScope ps(st, PK_COLNORM, 0.0, 0.0);
    ps.bracket();
    TNR_LAUNCH(ps, k_colnorm_part, grid, dim3(64 * CN_COLS), 0, st, d_descs, nd);
    TNR_HIP(hipGetLastError());
    TNR_LAUNCH(ps, k_colnorm_scale, grid, dim3(64 * CN_COLS), 0, st, d_descs, nd, rtol);
    TNR_HIP(hipGetLastError());
}

void launch_canon(hipStream_t st, const CanonDesc* d_descs, int nd, int kmax, double tie) {
    if (nd <= 0) return;
    TNR_REQUIRE(kmax >= 1 && kmax <= LMAX, TNR_ERR_INTERNAL, "gauge block above LMAX");
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_canon, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)(((size_t)LMAX * LMAX + 2 * (size_t)LMAX) * sizeof(double)));
    TNR_HIP(attr);
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    const size_t shm = ((size_t)kmax * kmax + 2 * (size_t)kmax) * sizeof(double);
    TNR_LAUNCH(ps, k_canon, dim3(nd), dim3(CNT), shm, st, d_descs, nd, tie);
    TNR_HIP(hipGetLastError());
}

void launch_dot(hipStream_t st, const DotDesc* d_descs, int nd) {
    if (nd <= 0) return;
    TNR_REQUIRE(nd <= 65535, TNR_ERR_INTERNAL, "too many dot products in one launch");
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    ps.bracket();
    TNR_LAUNCH(ps, k_dot_part, dim3(DOT_PARTS, nd), dim3(256), 0, st, d_descs, nd);
    TNR_HIP(hipGetLastError());
    TNR_LAUNCH(ps, k_dot_final, dim3(nd), dim3(64), 0, st, d_descs, nd);
    TNR_HIP(hipGetLastError());
}

// Problems up to EIG_NMAX run with the matrix in LDS, larger ones (up to
// EIG_NMAX_G, each with its workspace of eig_work_doubles(n)) in global
// memory; each kernel skips the other's, so a problem's kernel depends on
// its own size only.
void launch_eig(hipStream_t st, const EigDesc* d_descs, int nd, int nmin, int nmax) {
    if (nd <= 0) return;
    TNR_REQUIRE(nmin >= 1 && nmax <= EIG_NMAX_G, TNR_ERR_INTERNAL, "eigenproblem above EIG_NMAX_G");
    auto bytes = [](int n) { return (size_t)eig_work_doubles(n) * sizeof(double); };
    static const hipError_t attr = hipFuncSetAttribute(
        (const void*)k_eig_hqr, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes(EIG_NMAX));
    TNR_HIP(attr);
    if (nmin <= EIG_NMAX) {
        ProfScope ps(st, PK_MISC, 0.0, 0.0);
        TNR_LAUNCH(ps, k_eig_hqr, dim3(nd), dim3(EIGT), bytes(std::min(nmax, EIG_NMAX)), st, d_descs,
                   nd);
        TNR_HIP(hipGetLastError());
    }
    if (nmax > EIG_NMAX) {
        ProfScope ps(st, PK_MISC, 0.0, 0.0);
        TNR_LAUNCH(ps, k_eig_hqr_g, dim3(nd), dim3(EIGT), 0, st, d_descs, nd);
        TNR_HIP(hipGetLastError());
    }
}

void launch_symmetrize(hipStream_t st, const ColDesc* d_descs, int nd, int nmax) {
    if (nd <= 0) return;
    int64_t tot = (int64_t)nmax * nmax;
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    TNR_LAUNCH(ps, k_symmetrize, dim3(grid_for(tot, 1024), nd), dim3(256), 0, st, d_descs, nd);
    TNR_HIP(hipGetLastError());
}

void launch_conv(hipStream_t st, const ConvDesc* d_descs, int nd, const ConvRule& rule) {
    if (nd <= 0) return;
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    TNR_LAUNCH(ps, k_conv, dim3(nd), dim3(64), 0, st, d_descs, nd, rule);
    TNR_HIP(hipGetLastError());
}

void launch_frob(hipStream_t st, const ColDesc* d_descs, int nd, double* partial) {
    if (nd <= 0) return;
    ProfScope ps(st, PK_MISC, 0.0, 0.0);
    ps.bracket();
    TNR_LAUNCH(ps, k_frob_part, dim3(FROB_PARTS, nd), dim3(256), 0, st, d_descs, partial);
    TNR_LAUNCH(ps, k_frob_final, dim3((nd + 63) / 64), dim3(64), 0, st, d_descs, nd, partial);
    TNR_HIP(hipGetLastError());
}

void launch_randfill(hipStream_t st, const FillDesc* d_descs, int nd, int64_t total) {
    if (total <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_FILL, 0.0, 0.0);
    TNR_LAUNCH(ps, k_randfill, dim3(grid_for(total, 4096)), dim3(256), 0, st, d_descs, nd, total);
    TNR_HIP(hipGetLastError());
}

void launch_gather(hipStream_t st, const GatherDesc* d_descs, int nd, int64_t total) {
    if (total <= 0 || nd <= 0) return;
    ProfScope ps(st, PK_GATHER, 0.0, 16.0 * (double)total);
    TNR_LAUNCH(ps, k_gather, dim3(grid_for(total, 8192)), dim3(256), 0, st, d_descs, nd, total);
    TNR_HIP(hipGetLastError());
}

}  // namespace tnr
