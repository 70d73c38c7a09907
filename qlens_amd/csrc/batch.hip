// Batched inversion kernels for gfx950: active sets, merged lensing rows, row ordering, block-sparse
// blurred L, F = Lb^T C Lb (FP64 MFMA, or FP16 MFMA with FP32 accumulation), curvature R
// (banded FP64 factorization for ln det R), blocked dense Cholesky of F (FP64 or FP32), solves,
// FP64 iterative refinement and the evidence terms.
//
// Item b of a batch is blockIdx.y (matrix index for the Cholesky kernels); per-item sizes and pool
// offsets come from BatchDev::meta.  Layouts: the blurred L is kept as strips of 64 rows (a chunk) x
// 16 columns, only those a chunk's rows reach, a chunk's one after the other (k_build_lb_b); column n_src
// carries the data vector so the SYRK also yields D = Lb^T C d (row n_src of F).  F is row-major
// ldN x ldN (lower triangle used), R in banded 64 x 64 tiles, padding beyond the source block identity.
//
// Reference behaviour followed:
//   active sets              assign_active_indices / assign_pixel_mappings  pixelgrid.cpp:3586-3626, 12879-12914
//   dense L (merged in CSR)  assign_Lmatrix + convert_Lmatrix_to_dense      pixelgrid.cpp:13196-13321, 13717-13747
//   PSF on L                 PSF_convolution_Lmatrix_dense (direct)         pixelgrid.cpp:14092-14176
//   D, F                     create_lensing_matrices_from_Lmatrix_dense     pixelgrid.cpp:15590-15711
//   curvature R              generate_hmatrices / Rmatrix_from_hmatrices    pixelgrid.cpp:2968-3240
//   F += lambda R            add_regularization_term_to_dense_Fmatrix      pixelgrid.cpp:15808-15818
//   ln det R                 Rmatrix_determinant_dense                      pixelgrid.cpp:18176-18191
//   Cholesky, solve, logdet  Cholesky_dcmp/solve/logdet_lower_packed        pixelgrid.cpp:17071-17246
//   model, chi^2, Es         lens.cpp:12950-13015, pixelgrid.cpp:15821-15863, 18268-18307
#include "qlx_internal.h"

#include <type_traits>
#include <utility>

namespace qlx {

typedef double double2_t __attribute__((ext_vector_type(2)));
typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// 16-byte store marked non-temporal (streamed past the caches): for buffers written once and read
// much later, so that they do not push out lines that are still being re-read
__device__ __forceinline__ void store_nt(uint4* p, const uint4& v)
{
    __builtin_nontemporal_store((u32x4_t){v.x, v.y, v.z, v.w}, (u32x4_t*)p);
}
#define TS 64

// raise the dynamic-LDS limit of a kernel once per process (kernels are told apart by address)
static void allow_big_lds(const void* kernel)
{
    static const void* done[32];
    static int ndone = 0;
    for (int i = 0; i < ndone; i++)
        if (done[i] == kernel) return;
    hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 16 * 1024);
    if (ndone < 32) done[ndone++] = kernel;
}

static inline unsigned grid_for(size_t n, unsigned bs = 256, unsigned cap = 65535u * 4u)
{
    size_t g = (n + bs - 1) / bs;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (unsigned)g;
}

// ------------------------------------------------------------------------------------------------
// utilities
// ------------------------------------------------------------------------------------------------
__global__ void k_fill_i32(int* p, int v, size_t n)
{
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) p[t] = v;
}
__global__ void k_fill_f64(double* p, double v, size_t n)
{
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) p[t] = v;
}
void launch_fill_i32(hipStream_t s, int* p, int v, size_t n)
{
    if (n) hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(n)), dim3(256), 0, s, p, v, n);
}
void launch_fill_f64(hipStream_t s, double* p, double v, size_t n)
{
    if (n) hipLaunchKernelGGL(k_fill_f64, dim3(grid_for(n)), dim3(256), 0, s, p, v, n);
}

__device__ __forceinline__ int wave_incl_scan(int v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int t = __shfl_up(v, off, 64);
        if (lane >= off) v += t;
    }
    return v;
}

// 1024-thread exclusive scan of one flag per thread; returns this thread's exclusive index
__device__ __forceinline__ int block_excl_scan(int flag, int* sh, int& total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = wave_incl_scan(flag);
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    if (w == 0) {
        int v = (lane < 16) ? sh[lane] : 0;
        int s = wave_incl_scan(v);
        if (lane < 16) sh[16 + lane] = s - v;
        if (lane == 15) sh[32] = s;
    }
    __syncthreads();
    int excl = sh[16 + w] + incl - flag;
    total = sh[32];
    __syncthreads();
    return excl;
}

// ------------------------------------------------------------------------------------------------
// active sets: source cells in j-major order, image pixels in j-outer / i-inner order
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) k_compact_b(BatchDev bd)
{
    __shared__ int sh[40];
    const int item = blockIdx.y;
    const int snx = bd.src_n[2 * item], sny = bd.src_n[2 * item + 1];
    const int* cm = bd.cmapped + item * bd.s_cell;
    int* sidx = bd.sidx + item * bd.s_cell;
    const int* pm = bd.pmapped + item * bd.s_pix;
    int* pidx = bd.pidx + item * bd.s_pix;
    int* act = bd.act_pix + item * bd.s_pix;
    int base = 0;
    const int ncell = snx * sny;
    for (int t0 = 0; t0 < ncell; t0 += 1024) {
        int t = t0 + threadIdx.x, c = -1, flag = 0;
        if (t < ncell) {
            c = (t % snx) * sny + t / snx;
            flag = cm[c] ? 1 : 0;
        }
        int tot, ex = block_excl_scan(flag, sh, tot);
        if (c >= 0) sidx[c] = flag ? base + ex : -1;
        base += tot;
    }
    if (threadIdx.x == 0) bd.counts[4 * item] = base;
    __syncthreads();
    // internal order of F's source columns: the same active cells ranked tile by tile
    // (QLX_TILE_W x QLX_TILE_H cells; inside a tile 4 x 4 cells by 4 x 4 cells, all y-major), so that a
    // compact source-plane patch occupies a compact index range, in strips of 16 as in blocks
    {
        int* tix = bd.tix + item * bd.s_cell;
        int* pis = bd.pisrc + item * bd.s_cell;
        const int ntw = (snx + QLX_TILE_W - 1) / QLX_TILE_W, nth = (sny + QLX_TILE_H - 1) / QLX_TILE_H;
        const int tcells = QLX_TILE_W * QLX_TILE_H;
        const int total = ntw * nth * tcells;
        int tbase = 0;
        for (int t0 = 0; t0 < total; t0 += 1024) {
            const int t = t0 + threadIdx.x;
            int c = -1, flag = 0;
            if (t < total) {
                const int tile = t / tcells, wv = t - tile * tcells;
                const int sub = wv >> 4;  // 4 x 4 cells each
                const int i = (tile % ntw) * QLX_TILE_W + 4 * (sub % (QLX_TILE_W / 4)) + wv % 4;
                const int j = (tile / ntw) * QLX_TILE_H + 4 * (sub / (QLX_TILE_W / 4)) + wv % 16 / 4;
                if (i < snx && j < sny) {
                    c = i * sny + j;
                    flag = cm[c] ? 1 : 0;
                }
            }
            int tot, ex = block_excl_scan(flag, sh, tot);
            if (c >= 0) tix[c] = flag ? tbase + ex : -1;
            if (flag) pis[tbase + ex] = sidx[c];
            tbase += tot;
        }
    }
    base = 0;
    const int npix = bd.nx * bd.ny;
    int* apre = bd.apre + item * (bd.s_pix + 1);
    for (int t0 = 0; t0 < npix; t0 += 1024) {
        int t = t0 + threadIdx.x, p = -1, flag = 0;
        if (t < npix) {
            p = (t % bd.nx) * bd.ny + t / bd.nx;
            flag = ((!bd.mask || bd.mask[p]) && pm[p]) ? 1 : 0;
        }
        int tot, ex = block_excl_scan(flag, sh, tot);
        if (p >= 0) {
            pidx[p] = flag ? base + ex : -1;
            apre[t] = base + ex;
            if (flag) act[base + ex] = p;
        }
        base += tot;
    }
    if (threadIdx.x == 0) {
        bd.counts[4 * item + 1] = base;
        apre[npix] = base;
    }
}

void launch_compact_b(hipStream_t s, const BatchDev& bd)
{
    hipLaunchKernelGGL(k_compact_b, dim3(1, bd.B), dim3(1024), 0, s, bd);
}

// merged row of L per active pixel: CSR order, duplicates summed from 0 in that order.  Up to
// nsplit 2 (12 entries) the row is built in registers (predicated, no dynamic indexing) and stored
// once; larger splits build it in place.
__global__ void __launch_bounds__(256) k_merge_lrows_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || r >= M.n_img) return;
    const int nsub = bd.nsub, U = 3 * nsub;
    const long long p = bd.act_pix[item * bd.s_pix + r];
    const int* mcb = bd.map_cell + (size_t)item * bd.s_pix * nsub * 3;
    const double* mwb = bd.map_w + (size_t)item * bd.s_pix * nsub * 3;
    const int* tix = bd.tix + item * bd.s_cell;
    int* uc = bd.ucol + ((size_t)item * bd.s_pix + r) * U;
    double* uv = bd.uval + ((size_t)item * bd.s_pix + r) * U;
    if (nsub <= 4) {
        constexpr int MU = 12;
        int cols[MU];
        double vals[MU];
#pragma unroll
        for (int j = 0; j < MU; j++) {
            cols[j] = -1;
            vals[j] = 0.0;
        }
        // the pixel's nsub x 3 ray entries; with nsub = 4 (2 x 2 split) they are 48 + 96 contiguous,
        // 16-byte aligned bytes, read with six vector loads
        int mcv[MU];
        double mwv[MU];
        if (nsub == 4) {
            const int4* mc4 = (const int4*)(mcb + p * MU);
            const double2* mw2 = (const double2*)(mwb + p * MU);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const int4 t = mc4[j];
                mcv[4 * j] = t.x;
                mcv[4 * j + 1] = t.y;
                mcv[4 * j + 2] = t.z;
                mcv[4 * j + 3] = t.w;
            }
#pragma unroll
            for (int j = 0; j < 6; j++) {
                const double2 t = mw2[j];
                mwv[2 * j] = t.x;
                mwv[2 * j + 1] = t.y;
            }
        } else {
#pragma unroll
            for (int j = 0; j < MU; j++) {
                mcv[j] = (j < 3 * nsub) ? mcb[p * nsub * 3 + j] : -1;
                mwv[j] = (j < 3 * nsub) ? mwb[p * nsub * 3 + j] : 0.0;
            }
        }
        int n = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (mcv[3 * k] < 0) continue;
#pragma unroll
            for (int e = 0; e < 3; e++) {
                const int col = tix[mcv[3 * k + e]];
                const double w = mwv[3 * k + e];
                bool found = false;
#pragma unroll
                for (int j = 0; j < MU; j++)
                    if (!found && j < n && cols[j] == col) {
                        vals[j] += w;
                        found = true;
                    }
                if (!found) {
#pragma unroll
                    for (int j = 0; j < MU; j++)
                        if (j == n) {
                            cols[j] = col;
                            vals[j] = 0.0 + w;
                        }
                    n++;
                }
            }
        }
        if (nsub == 4) {  // the whole 12-slot row with vector stores (slots >= n: col -1, value 0, never read)
#pragma unroll
            for (int j = 0; j < 3; j++) ((int4*)uc)[j] = make_int4(cols[4 * j], cols[4 * j + 1], cols[4 * j + 2], cols[4 * j + 3]);
#pragma unroll
            for (int j = 0; j < 6; j++) ((double2*)uv)[j] = make_double2(vals[2 * j], vals[2 * j + 1]);
        } else {
#pragma unroll
            for (int j = 0; j < MU; j++)
                if (j < n) {
                    uc[j] = cols[j];
                    uv[j] = vals[j];
                }
        }
        bd.ucnt[item * bd.s_pix + r] = n;
        return;
    }
    int cnt = 0;
    for (int k = 0; k < nsub; k++) {
        const int* mc = mcb + (p * nsub + k) * 3;
        const double* mw = mwb + (p * nsub + k) * 3;
        if (mc[0] < 0) continue;
        for (int e = 0; e < 3; e++) {
            int col = tix[mc[e]];
            int q = 0;
            while (q < cnt && uc[q] != col) q++;
            if (q == cnt) {
                uc[cnt] = col;
                uv[cnt] = 0.0 + mw[e];
                cnt++;
            } else {
                uv[q] += mw[e];
            }
        }
    }
    bd.ucnt[item * bd.s_pix + r] = cnt;
}

void launch_merge_lrows_b(hipStream_t s, const BatchDev& bd, int max_img)
{
    if (max_img > 0) hipLaunchKernelGGL(k_merge_lrows_b, dim3((max_img + 255) / 256, bd.B), dim3(256), 0, s, bd);
}

// a merged 12-slot L row (2 x 2 split) as 3 + 6 16-byte loads
__device__ __forceinline__ void load_row12(const int* uc, const double* uv, int (&c)[12], double (&w)[12])
{
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const int4 t = ((const int4*)uc)[j];
        c[4 * j] = t.x;
        c[4 * j + 1] = t.y;
        c[4 * j + 2] = t.z;
        c[4 * j + 3] = t.w;
    }
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const double2 t = ((const double2*)uv)[j];
        w[2 * j] = t.x;
        w[2 * j + 1] = t.y;
    }
}

// ------------------------------------------------------------------------------------------------
// Row order of the blurred lensing matrix: active pixels in image tiles of 8 x 8 pixels (tiles and
// pixels inside a tile y-major), so that the 64 rows of a chunk are image-compact.  Their PSF
// windows then overlap (the Lb build applies each L entry to every row of the chunk it reaches) and
// their blurred supports are one compact source-plane patch (fewer pool blocks and SYRK block pairs
// than rows ordered by source position: 2 780 against 3 767 blocks and 14.6k against 25.8k pairs on
// the 200 x 200 / 60 x 60 workload).  One wave per tile; the order is a pure function of the active
// set, so an item's rows do not depend on its batch.
//   perm[pos] = active row of tile-order position pos, key[r] = tile-order position of row r,
//   tbase[t] = first position of tile t (the eptr buffer, s_pix + 1 ints per item)
// ------------------------------------------------------------------------------------------------
#define RT 8  // row tile side in pixels
__global__ void __launch_bounds__(64) k_tile_count_b(BatchDev bd, int ntx, int nty)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int t = blockIdx.x;
    if (!M.valid || t >= ntx * nty) return;
    const int lane = threadIdx.x;
    const int i = (t % ntx) * RT + (lane % RT), j = (t / ntx) * RT + lane / RT;
    const bool act = i < bd.nx && j < bd.ny && bd.pidx[item * bd.s_pix + (size_t)i * bd.ny + j] >= 0;
    const unsigned long long m = __ballot(act);
    if (lane == 0) bd.eptr[item * (bd.s_pix + 1) + t] = __popcll(m);
}

__global__ void __launch_bounds__(1024) k_tile_scan_b(BatchDev bd, int ntiles)
{
    __shared__ int sh[40];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    int* tb = bd.eptr + item * (bd.s_pix + 1);
    int base = 0;
    for (int t0 = 0; t0 < ntiles; t0 += 1024) {
        const int t = t0 + threadIdx.x;
        const int v = t < ntiles ? tb[t] : 0;
        int tot, ex = block_excl_scan(v, sh, tot);
        if (t < ntiles) tb[t] = base + ex;
        base += tot;
    }
    if (threadIdx.x == 0) tb[ntiles] = base;
}

__global__ void __launch_bounds__(64) k_tile_scatter_b(BatchDev bd, int ntx, int nty)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int t = blockIdx.x;
    if (!M.valid || t >= ntx * nty) return;
    const int lane = threadIdx.x;
    const int i = (t % ntx) * RT + (lane % RT), j = (t / ntx) * RT + lane / RT;
    const int r = (i < bd.nx && j < bd.ny) ? bd.pidx[item * bd.s_pix + (size_t)i * bd.ny + j] : -1;
    const unsigned long long m = __ballot(r >= 0);
    if (r < 0) return;
    const int rank = __popcll(m & ((1ull << lane) - 1ull));
    const int pos = bd.eptr[item * (bd.s_pix + 1) + t] + rank;
    bd.perm[item * bd.s_pix + pos] = r;
    bd.key[item * bd.s_pix + r] = pos;
}

void launch_sort_rows_b(hipStream_t s, const BatchDev& bd, int max_img, int max_src)
{
    (void)max_src;
    if (max_img <= 0) return;
    const int ntx = (bd.nx + RT - 1) / RT, nty = (bd.ny + RT - 1) / RT;
    hipLaunchKernelGGL(k_tile_count_b, dim3(ntx * nty, bd.B), dim3(64), 0, s, bd, ntx, nty);
    hipLaunchKernelGGL(k_tile_scan_b, dim3(1, bd.B), dim3(1024), 0, s, bd, ntx * nty);
    hipLaunchKernelGGL(k_tile_scatter_b, dim3(ntx * nty, bd.B), dim3(64), 0, s, bd, ntx, nty);
}

// ------------------------------------------------------------------------------------------------
// L by columns (CSC) for the Lb build: for every internal source column c, the entries (pixel, value)
// of the merged L rows, ordered by the rows' tile-order position (a fixed order, so every sum over a
// column's entries is reproducible): cpix (pixel i << 16 | j) and cval, with the column sizes and
// first entries in bcnt and boff (s_cell + 2 ints per item).
// ------------------------------------------------------------------------------------------------
// The columns are built in row-position order directly (a stable counting sort of the entries by
// column): the positions are cut into segments of QLX_CSC_SEG; k_csc_hist_b counts each segment's
// entries per column, k_csc_base_b turns the counts into each segment's first slot within the
// column (segments in order) and the column's size, k_csc_scan_b places the columns, and
// k_csc_place_b lets one wave per segment walk its rows in position order, each entry taking the
// next slot of its column.
__global__ void __launch_bounds__(256) k_csc_hist_b(BatchDev bd)
{
    extern __shared__ int hs[];  // n_src counters
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int seg = blockIdx.x, k0 = seg * QLX_CSC_SEG;
    if (!M.valid || k0 >= M.n_img) return;
    const int n = M.n_src, U = 3 * bd.nsub, tid = threadIdx.x;
    for (int c = tid; c < n; c += 256) hs[c] = 0;
    __syncthreads();
    const int k1 = min(k0 + QLX_CSC_SEG, M.n_img);
    const int* perm = bd.perm + item * bd.s_pix;
    const int* ucnt = bd.ucnt + item * bd.s_pix;
    const int* ucol = bd.ucol + (size_t)item * bd.s_pix * U;
    for (int k = k0 + tid; k < k1; k += 256) {
        const int r = perm[k], nu = ucnt[r];
        for (int e = 0; e < nu; e++) atomicAdd(&hs[ucol[(size_t)r * U + e]], 1);
    }
    __syncthreads();
    int* H = bd.csh + ((size_t)item * csc_segments(bd.s_pix) + seg) * bd.s_cell;
    for (int c = tid; c < n; c += 256) H[c] = hs[c];
}

__global__ void __launch_bounds__(256) k_csc_base_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || c >= M.n_src) return;
    const int nsg = (M.n_img + QLX_CSC_SEG - 1) / QLX_CSC_SEG;
    int* H = bd.csh + (size_t)item * csc_segments(bd.s_pix) * bd.s_cell + c;
    int run = 0;
    for (int sg = 0; sg < nsg; sg++) {
        const int v = H[(size_t)sg * bd.s_cell];
        H[(size_t)sg * bd.s_cell] = run;
        run += v;
    }
    bd.bcnt[item * (bd.s_cell + 2) + c] = run;
}

__global__ void __launch_bounds__(1024) k_csc_scan_b(BatchDev bd)
{
    __shared__ int sh[40];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const int* cnt = bd.bcnt + item * (bd.s_cell + 2);
    int* off = bd.boff + item * (bd.s_cell + 2);
    int* fill = bd.bfill + item * (bd.s_cell + 2);
    int base = 0;
    for (int t0 = 0; t0 < M.n_src; t0 += 1024) {
        const int t = t0 + threadIdx.x;
        const int v = t < M.n_src ? cnt[t] : 0;
        int tot, ex = block_excl_scan(v, sh, tot);
        if (t < M.n_src) {
            off[t] = base + ex;
            fill[t] = 0;
        }
        base += tot;
    }
    if (threadIdx.x == 0) off[M.n_src] = base;
}

// one wave per segment: the column cursors start at the segment's first slots; 64 rows at a time
// are staged in LDS (lane l: row k + l's entries and pixel), then the rows are walked in order, lane
// e placing entry e of the row (a merged row's columns are distinct)
__global__ void __launch_bounds__(64) k_csc_place_b(BatchDev bd)
{
    // dynamic LDS: the staged rows' values (64 x U doubles), columns (64 x U ints), then the n_src
    // column cursors
    extern __shared__ double place_raw[];
    __shared__ int scnt[64];
    __shared__ unsigned spk[64];
    const int U = 3 * bd.nsub;
    double* sval = place_raw;
    int* scol = (int*)(place_raw + 64 * U);
    int* cur = scol + 64 * U;
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int seg = blockIdx.x, k0 = seg * QLX_CSC_SEG;
    if (!M.valid || k0 >= M.n_img) return;
    const int n = M.n_src, lane = threadIdx.x;
    const int* H = bd.csh + ((size_t)item * csc_segments(bd.s_pix) + seg) * bd.s_cell;
    const int* off = bd.boff + item * (bd.s_cell + 2);
    for (int c = lane; c < n; c += 64) cur[c] = off[c] + H[c];
    const int k1 = min(k0 + QLX_CSC_SEG, M.n_img);
    const int* perm = bd.perm + item * bd.s_pix;
    const int* act = bd.act_pix + item * bd.s_pix;
    const int* ucnt = bd.ucnt + item * bd.s_pix;
    const int* ucol = bd.ucol + (size_t)item * bd.s_pix * U;
    const double* uval = bd.uval + (size_t)item * bd.s_pix * U;
    const size_t eb = (size_t)item * bd.s_pix * U;
    unsigned* cpix = bd.cpix + eb;
    double* cval = bd.cval + eb;
    for (int kb = k0; kb < k1; kb += 64) {
        const int k = kb + lane;
        int nu = 0;
        unsigned pk = 0;
        if (k < k1) {
            const int r = perm[k], p = act[r];
            nu = ucnt[r];
            pk = ((unsigned)(p / bd.ny) << 16) | (unsigned)(p - (p / bd.ny) * bd.ny);
            for (int e = 0; e < nu; e++) {
                scol[lane * U + e] = ucol[(size_t)r * U + e];
                sval[lane * U + e] = uval[(size_t)r * U + e];
            }
        }
        scnt[lane] = nu;
        spk[lane] = pk;
        __syncthreads();
        const int nrow = min(64, k1 - kb);
        for (int l = 0; l < nrow; l++) {
            for (int e = lane; e < scnt[l]; e += 64) {  // U <= 48 entries per row
                const int c = scol[l * U + e];
                const int slot = cur[c];
                cur[c] = slot + 1;
                cpix[slot] = spk[l];
                cval[slot] = sval[l * U + e];
            }
        }
        __syncthreads();
    }
}

void launch_lcols_b(hipStream_t s, const BatchDev& bd, int max_img, int max_src)
{
    if (max_img <= 0 || max_src <= 0) return;
    const int nsg = (max_img + QLX_CSC_SEG - 1) / QLX_CSC_SEG;
    const size_t lds = (size_t)bd.s_cell * 4;
    allow_big_lds((const void*)k_csc_hist_b);
    allow_big_lds((const void*)k_csc_place_b);
    hipLaunchKernelGGL(k_csc_hist_b, dim3(nsg, bd.B), dim3(256), lds, s, bd);
    hipLaunchKernelGGL(k_csc_base_b, dim3((max_src + 255) / 256, bd.B), dim3(256), 0, s, bd);
    hipLaunchKernelGGL(k_csc_scan_b, dim3(1, bd.B), dim3(1024), 0, s, bd);
    const size_t U = 3 * (size_t)bd.nsub;
    hipLaunchKernelGGL(k_csc_place_b, dim3(nsg, bd.B), dim3(64), 64 * U * 12 + lds, s, bd);
}

// ------------------------------------------------------------------------------------------------
// chunk support (one workgroup per chunk): the columns of L with an entry in the PSF reach of the
// chunk's 64 rows (a bit per column, which the Lb build also reads), the strips of 16 columns that
// hold one (the pool holds these and only these), then per item the strips' slots and, per column
// block of the SYRK, which strips of a chunk it holds and where they start.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int wave_min_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_max_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
// a chunk whose rows span at most LB_SPAN + 1 pixels each way is scanned as one rectangle, and the
// padded tap table of the Lb build covers it
#define LB_SPAN 15

__global__ void __launch_bounds__(256) k_chunk_cols_b(BatchDev bd)
{
    extern __shared__ unsigned colbits[];  // M.ncw words, then per wave the rows' reach in one image column
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int kt = blockIdx.x;
    if (!M.valid || kt >= M.nkt) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int rows = min(TS, M.n_img - kt * TS);
    for (int t = tid; t < M.ncw; t += 256) colbits[t] = 0u;
    int k = 0, l = 0;
    if (lane < rows) {
        const int p = bd.act_pix[item * bd.s_pix + bd.perm[item * bd.s_pix + kt * TS + lane]];
        k = p / bd.ny;
        l = p - (p / bd.ny) * bd.ny;
    }
    const bool row = lane < rows;
    const int kmin = wave_min_i(row ? k : 1 << 30), kmax = wave_max_i(row ? k : -(1 << 30));
    const int lmin = wave_min_i(row ? l : 1 << 30), lmax = wave_max_i(row ? l : -(1 << 30));
    __syncthreads();
    const int U = 3 * bd.nsub, pnx = bd.pnx, pny = bd.pny;
    const int* pidx = bd.pidx + item * bd.s_pix;
    const int* ucnt = bd.ucnt + item * bd.s_pix;
    const int* ucol = bd.ucol + (size_t)item * bd.s_pix * U;
    auto mark = [&](int i, int j) {  // a pixel of the image
        const int r = pidx[(size_t)i * bd.ny + j];
        if (r < 0) return;
        const int nu = ucnt[r];
        for (int e = 0; e < nu; e++) {
            const int c = ucol[(size_t)r * U + e];
            atomicOr(&colbits[c >> 5], 1u << (c & 31));
        }
    };
    // pixels (i, j) whose tap (k + hx - i, l + hy - j) lies in the PSF for a row (k, l): of a compact
    // chunk the rectangle of all its rows' windows.  Of another (a chunk of the last tiles of two image
    // rows spans the image, not its pixels; a scattered mask's chunks span many tiles) the union of the
    // windows, each pixel once: a wave takes an image column, its lanes' rows set the column's stretch they
    // reach in a bit map, and the pixels set are marked.  (Window by window a pixel was marked once per
    // row that reaches it, 64 x taps a chunk.  The stages ahead of the pool's build, 200 x 200 pixels on
    // 60 x 60 cells: one item with a 121 x 121 PSF 4.34 -> 0.34 ms, 32 with 41 x 41 taps 2.34 -> 0.77, on
    // every third image column 2.97 -> 0.38; one with 21 x 21 taps 0.35 -> 0.25.)
    const int i0 = pnx / 2 - pnx + 1, j0 = pny / 2 - pny + 1;
    const int ilo = max(0, kmin + i0), ihi = min(bd.nx - 1, kmax + i0 + pnx - 1);
    const int jlo = max(0, lmin + j0), jhi = min(bd.ny - 1, lmax + j0 + pny - 1);
    if (kmax - kmin <= LB_SPAN && lmax - lmin <= LB_SPAN) {
        const int wj = jhi - jlo + 1, n = (ihi - ilo + 1) * wj;
        for (int t = tid; t < n; t += 256) mark(ilo + t / wj, jlo + t % wj);
    } else {
        const int njw = (bd.ny + 31) / 32;
        unsigned* const jb = colbits + M.ncw + (tid >> 6) * njw;
        const int ja = max(0, l + j0), je = min(bd.ny - 1, l + j0 + pny - 1);
        for (int i = ilo + (tid >> 6); i <= ihi; i += 4) {
            const bool in = row && (unsigned)(i - k - i0) < (unsigned)pnx;
            if (!__ballot(in)) continue;
            for (int t = (jlo >> 5) + lane; t <= jhi >> 5; t += 64) jb[t] = 0u;
            wave_lds_sync();
            if (in)
                for (int t = ja >> 5; t <= je >> 5; t++)
                    atomicOr(&jb[t], (t == ja >> 5 ? ~0u << (ja & 31) : ~0u) & (t == je >> 5 ? ~0u >> (31 - (je & 31)) : ~0u));
            wave_lds_sync();
            for (int j = jlo + lane; j <= jhi; j += 64)
                if (jb[j >> 5] >> (j & 31) & 1u) mark(i, j);
            wave_lds_sync();
        }
    }
    __syncthreads();
    unsigned* cb = bd.colb + M.col_off + (size_t)kt * M.ncw;
    for (int t = tid; t < M.ncw; t += 256) cb[t] = colbits[t];
    // strip s = columns 16 s .. 16 s + 15; the data column's strip is in every chunk
    if (tid < M.nsw) {
        unsigned m = 0;
        for (int q = 0; q < 16 && 16 * tid + q < M.ncw; q++) {
            const unsigned c = colbits[16 * tid + q];
            m |= ((c & 0xffffu) ? 1u : 0u) << (2 * q) | ((c >> 16) ? 1u : 0u) << (2 * q + 1);
        }
        const int sd = M.n_src >> 4;
        if ((sd >> 5) == tid) m |= 1u << (sd & 31);
        bd.nz[M.nz_off + (size_t)kt * M.nsw + tid] = m;
    }
}

// the chunks' first slots in the item's pool (in strips), the item's strips and the strip pairs that its SYRK
// multiplies
__global__ void __launch_bounds__(1024) k_block_scan_b(BatchDev bd)
{
    __shared__ int sh[40];
    __shared__ unsigned long long sp[1024];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const unsigned* nz = bd.nz + M.nz_off;
    int* bb = bd.bbase + M.bb_off;
    int base = 0;
    unsigned long long pairs = 0;
    for (int t0 = 0; t0 < M.nkt; t0 += 1024) {
        const int t = t0 + threadIdx.x;
        int v = 0;
        if (M.cbs == 6) {  // FP64: the SYRK multiplies the pairs held
            if (t < M.nkt)
                for (int w = 0; w < M.nsw; w++) v += __popc(nz[(size_t)t * M.nsw + w]);
            pairs += (unsigned long long)v * (v + 1) / 2;
        } else if (t < M.nkt) {
            // FP16: a wave takes four column strips together, absent ones as zeros: per four of which one is
            // held, the strips held from their first on, times four
            unsigned long long fours = 0, before = 0;
            for (int w = 0; w < M.nsw; w++)
                for (unsigned x = nz[(size_t)t * M.nsw + w], q = 0; q < 8; q++, x >>= 4)
                    if (x & 15u) {
                        fours++;
                        before += v;
                        v += __popc(x & 15u);
                    }
            pairs += 4 * (fours * v - before);
        }
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        int incl = wave_incl_scan(v);
        if (lane == 63) sh[wv] = incl;
        __syncthreads();
        if (wv == 0) {
            int x = (lane < 16) ? sh[lane] : 0;
            int sx = wave_incl_scan(x);
            if (lane < 16) sh[16 + lane] = sx - x;
            if (lane == 15) sh[32] = sx;
        }
        __syncthreads();
        if (t < M.nkt) bb[t] = base + sh[16 + wv] + incl - v;
        const int tot = sh[32];
        __syncthreads();
        base += tot;
    }
    sp[threadIdx.x] = pairs;
    __syncthreads();
    for (int st = 512; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sp[threadIdx.x] += sp[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        bb[M.nkt] = base;
        bd.counts[4 * item + 2] = base;
        bd.npairs[item] = sp[0];
    }
}

// sup[I * nkt + kt]: of chunk kt's strips those in column block I (1 << cbs columns): mask in the low
// byte, their first strip's rank in the chunk above it; 0 where there is none
__global__ void __launch_bounds__(256) k_sup_table_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (!M.valid || t >= (long long)M.ncb * M.nkt) return;
    const int I = (int)(t / M.nkt), kt = (int)(t - (long long)I * M.nkt);
    const unsigned* m = bd.nz + M.nz_off + (size_t)kt * M.nsw;
    const int sb = 1 << (M.cbs - 4), s0 = I * sb;  // 4 or 8 strips a block: within one word
    unsigned rank = 0;
    for (int w = 0; w < (s0 >> 5); w++) rank += __popc(m[w]);
    const unsigned word = m[s0 >> 5];
    rank += __popc(word & ((1u << (s0 & 31)) - 1u));
    const unsigned mask = (word >> (s0 & 31)) & ((1u << sb) - 1u);
    bd.sup[M.sup_off + t] = mask ? rank << 8 | mask : 0u;
}

void launch_row_support_b(hipStream_t s, const BatchDev& bd, int max_nkt, int max_ld, int max_sup)
{
    if (max_nkt <= 0) return;
    hipLaunchKernelGGL(k_chunk_cols_b, dim3(max_nkt, bd.B), dim3(256), (size_t)max_ld / 8 + (size_t)16 * ((bd.ny + 31) / 32), s, bd);
    hipLaunchKernelGGL(k_block_scan_b, dim3(1, bd.B), dim3(1024), 0, s, bd);
    hipLaunchKernelGGL(k_sup_table_b, dim3((max_sup + 255) / 256, bd.B), dim3(256), 0, s, bd);
}

// ------------------------------------------------------------------------------------------------
// Blurred rows of one 64-row chunk into the chunk's support strips (PSF_convolution_Lmatrix_dense,
// direct branch, pixelgrid.cpp:14092-14176): Lb[r][c] = sum over pixels (i, j) of the chunk's PSF
// reach of psf[k_r + hx - i][l_r + hy - j] * L[(i, j)][c], taps inside the PSF only, (i, j) active.
// One workgroup per chunk; lane l of every wave owns chunk row l (the rows are image-compact, so an
// L entry of a pixel near the chunk reaches most of its rows), and a wave takes every fourth of the
// chunk's strips of 16 columns.  Per column with an entry in the reach (colb) it walks the column's
// entries in L's CSC form, keeps those whose pixel lies in the reach (a ballot over 64 entries at a
// time), broadcasts each kept entry and every lane adds its own tap weight times the value: the output
// element is summed in registers in a fixed order and written once, with no atomics.  A strip's values
// go to the wave's LDS tile and from there to the pool with 16-byte stores; waves share no barrier.
//   T = double: FP64 pool, unscaled (the FP64 SYRK applies C), a strip's element (row k, column i) at
//               ((k >> 1) * 16 + i) * 2 + (k & 1): a lane's 16 bytes are two rows of its column;
//   T = float:  FP16 pool, ((k >> 3) * 16 + i) * 8 + (k & 7): a lane's 16 bytes are the eight rows of
//               an MFMA operand; entries x = Lb sqrt(c_r) s16 rounded once (s16 a power of two, |x| <=
//               2^14).
// Column n_src carries the data: d (FP64) or d sqrt(c_r) s16 (FP16).  256 items of the 200 x 200 / 60 x 60
// workload, FP16: 10.0 ms with half blocks of 64 columns shared by the four waves and stored whole (13.0 GB) and
// the columns found in this kernel; 6.9 on strips (6.0 GB) after 1.1 in k_chunk_cols_b.  Bound by its LDS
// traffic (a broadcast and 64 tap reads per kept entry).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint16_t f32_to_f16_rne(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

__device__ __forceinline__ double readlane_f64(double v, int l)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ float readlane_f32(float v, int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
template <typename T> __device__ __forceinline__ T readlane_t(T v, int l);
template <> __device__ __forceinline__ double readlane_t<double>(double v, int l) { return readlane_f64(v, l); }
template <> __device__ __forceinline__ float readlane_t<float>(float v, int l) { return readlane_f32(v, l); }

// Tap table in LDS: tap (tp, tq) of the PSF at (tp + toff) * tpc + tq.  Padded form (toff =
// LB_SPAN + 1, tpc >= pny + LB_SPAN + 1, pnx + 2 LB_SPAN + 2 rows, zero outside the PSF): for a chunk
// whose rows span at most LB_SPAN + 1 pixels in each direction, every kept L entry (i, j) of the
// chunk's reach and every row (k, l) of it give tp = k + hx - i in [-LB_SPAN, pnx - 1 + LB_SPAN] and
// tq = l + hy - j in [-LB_SPAN, pny - 1 + LB_SPAN], so the flat index K(k, l) - E(i, j), with
// K = (k + hx + toff) tpc + l + hy and E = i tpc + j, lands on the tap when it lies in the PSF and
// on a zero otherwise (a tq past either edge falls on the zero columns of that row or the one
// before): no bounds test, and the zero products add exact zeros, so the sums are the bounds-tested
// ones bit for bit.  Other chunks (and PSFs too large for the padded table: compact form, toff = 0,
// tpc = pny) test the bounds per entry.

template <typename T>
struct LbEnt {
    int e;
    T v;
};

// LDS tile of a wave: eight columns of a strip as runs of eight 16-byte pieces (one per FP64 row pair or
// FP16 group of eight rows), 16 bytes of padding a run: at a multiple of 128 bytes the lanes' stores of a
// column fell on the same banks
template <typename T>
struct LbTile {
    static constexpr int RPR = 16 / (sizeof(T) == 8 ? 8 : 2);  // rows per run
    static constexpr int NRUN = TS / RPR;
    static constexpr int HC = 8;                               // columns per tile
    static constexpr int PITCH = 128 + 16;                     // bytes
    static constexpr int BYTES = NRUN * PITCH;
};

template <typename T>
__global__ void __launch_bounds__(256) k_build_lb_b(BatchDev bd, int tab_bytes, int toff, int tpc, int trows)
{
    extern __shared__ double lds_raw[];
    const int item = blockIdx.y, kt = blockIdx.x;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || kt >= M.nkt) return;
    constexpr bool F64 = sizeof(T) == 8;
    typedef LbTile<T> LT;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int pnx = bd.pnx, pny = bd.pny;
    T* tab = (T*)lds_raw;
    LbEnt<T>* ent = (LbEnt<T>*)((char*)lds_raw + tab_bytes) + 64 * w;
    char* tile = (char*)lds_raw + tab_bytes + 4 * 64 * sizeof(LbEnt<T>) + w * LT::BYTES;
    for (int t = tid; t < trows * tpc; t += 256) {
        const int tr = t / tpc, tq = t - tr * tpc, tp = tr - toff;
        tab[t] = (tp >= 0 && tp < pnx && tq < pny) ? (T)bd.psf[tp * pny + tq] : (T)0;
    }
    // this lane's row
    const int rs = kt * TS + lane;
    const int p = rs < M.n_img ? bd.act_pix[item * bd.s_pix + bd.perm[item * bd.s_pix + rs]] : -1;
    const int kr = p >= 0 ? p / bd.ny : 0, lr = p >= 0 ? p - (p / bd.ny) * bd.ny : 0;
    // the chunk's PSF reach: pixels (i, j) with i in [kmin + hx - pnx + 1, kmax + hx], likewise j
    const int hx = pnx / 2, hy = pny / 2;
    const int kmin = wave_min_i(p >= 0 ? kr : 1 << 30), kmax = wave_max_i(p >= 0 ? kr : -(1 << 30));
    const int lmin = wave_min_i(p >= 0 ? lr : 1 << 30), lmax = wave_max_i(p >= 0 ? lr : -(1 << 30));
    const int i_lo = kmin + hx - pnx + 1, j_lo = lmin + hy - pny + 1;
    const unsigned i_span = (unsigned)(kmax - kmin + pnx - 1), j_span = (unsigned)(lmax - lmin + pny - 1);
    const int kr2 = kr + hx, lr2 = lr + hy;  // tap (kr2 - i, lr2 - j) of pixel (i, j)
    const bool fast = toff > 0 && kmax - kmin <= LB_SPAN && lmax - lmin <= LB_SPAN;
    int K = (kr2 + toff) * tpc + lr2;
    K = p >= 0 ? K : __builtin_amdgcn_readlane(K, 0);  // lane 0 holds a row of every chunk
    double sc = 0.0, dv = 0.0;
    if (p >= 0) {
        if constexpr (F64) {
            dv = bd.data[p];
        } else {
            sc = sqrt(bd.covinv[p]) * bd.s16;
            dv = bd.data[p] * sc;
        }
    }
    const unsigned* m = bd.nz + M.nz_off + (size_t)kt * M.nsw;
    const unsigned* cb = bd.colb + M.col_off + (size_t)kt * M.ncw;
    const size_t eb = (size_t)item * bd.s_pix * 3 * bd.nsub;
    const unsigned* cpix = bd.cpix + eb;
    const double* cval = bd.cval + eb;
    const int* cptr = bd.boff + item * (bd.s_cell + 2);
    // a strip's 64 x 16 elements are 128 16-byte pieces (FP16) or 512 (FP64)
    uint4* dst0 = (uint4*)((char*)bd.lb + M.lb_off * (F64 ? 8 : 2)) + (size_t)bd.bbase[M.bb_off + kt] * (F64 ? 512 : 128);
    const char* const tb = (const char*)tab + K * (int)sizeof(T);  // byte offsets: tap at tb - E
    __syncthreads();  // the table
    int q = 0;
    for (int wd = 0; wd < M.nsw; wd++) {
        unsigned bits = m[wd];
        while (bits) {
            const int strip = wd * 32 + __builtin_ctz(bits);
            bits &= bits - 1;
            if ((q++ & 3) != w) continue;
            const int c0 = 16 * strip;
            const unsigned live16 = (cb[strip >> 1] >> (16 * (strip & 1))) & 0xffffu;
            int lb0 = 0, lb1 = 0;
            if (lane < 16 && c0 + lane < M.n_src) {
                lb0 = cptr[c0 + lane];
                lb1 = cptr[c0 + lane + 1];
            }
#pragma unroll 1
            for (int h = 0; h < 16; h += LT::HC) {
                unsigned lmask = (live16 >> h) & ((1u << LT::HC) - 1u);
                int nxt = lmask ? __builtin_ctz(lmask) : LT::HC;
                int ce0 = 0, ce1 = 0;
                unsigned pk = 0;
                double vd = 0.0;
                if (nxt < LT::HC) {
                    ce0 = __builtin_amdgcn_readlane(lb0, h + nxt);
                    ce1 = __builtin_amdgcn_readlane(lb1, h + nxt);
                    if (ce0 + lane < ce1) {
                        pk = cpix[ce0 + lane];
                        vd = cval[ce0 + lane];
                    }
                }
                // columns without an entry in the reach are zero
                for (int t = lane; t < LT::NRUN * 8; t += 64) *(uint4*)(tile + (t >> 3) * LT::PITCH + (t & 7) * 16) = make_uint4(0, 0, 0, 0);
                wave_lds_sync();
                while (nxt < LT::HC) {
                    const int ii = nxt;
                    lmask &= lmask - 1;
                    nxt = lmask ? __builtin_ctz(lmask) : LT::HC;
                    const int e0c = ce0, e1c = ce1;
                    unsigned pkc = pk;
                    double vc = vd;
                    pk = 0;
                    vd = 0.0;
                    if (nxt < LT::HC) {  // the next live column's first entries
                        ce0 = __builtin_amdgcn_readlane(lb0, h + nxt);
                        ce1 = __builtin_amdgcn_readlane(lb1, h + nxt);
                        if (ce0 + lane < ce1) {
                            pk = cpix[ce0 + lane];
                            vd = cval[ce0 + lane];
                        }
                    }
                    T acc = (T)0;
                    for (int e0 = e0c; e0 < e1c; e0 += 64) {
                        if (e0 != e0c) {
                            pkc = 0;
                            vc = 0.0;
                            if (e0 + lane < e1c) {
                                pkc = cpix[e0 + lane];
                                vc = cval[e0 + lane];
                            }
                        }
                        const bool rel = e0 + lane < e1c && (unsigned)((int)(pkc >> 16) - i_lo) <= i_span &&
                                         (unsigned)((int)(pkc & 0xffffu) - j_lo) <= j_span;
                        const T v = (T)vc;
                        unsigned long long bal = __ballot(rel);
                        if (fast) {
                            if (rel) {
                                const int pos = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
                                ent[pos].e = ((int)(pkc >> 16) * tpc + (int)(pkc & 0xffffu)) * (int)sizeof(T);
                                ent[pos].v = v;
                            }
                            wave_lds_sync();
                            const int n = __popcll(bal);
                            int k = 0;
                            if constexpr (sizeof(T) == 4) {
                                // two entries per 16-byte LDS read (the same value in every lane)
                                for (; k + 4 <= n; k += 4) {
                                    const uint4 q0 = *(const uint4*)&ent[k], q1 = *(const uint4*)&ent[k + 2];
                                    const T t0 = *(const T*)(tb - (int)q0.x), t1 = *(const T*)(tb - (int)q0.z);
                                    const T t2 = *(const T*)(tb - (int)q1.x), t3 = *(const T*)(tb - (int)q1.z);
                                    acc += t0 * __uint_as_float(q0.y);
                                    acc += t1 * __uint_as_float(q0.w);
                                    acc += t2 * __uint_as_float(q1.y);
                                    acc += t3 * __uint_as_float(q1.w);
                                }
                            }
                            for (; k + 4 <= n; k += 4) {  // four entries' reads in flight together, summed in order
                                const LbEnt<T> x0 = ent[k], x1 = ent[k + 1], x2 = ent[k + 2], x3 = ent[k + 3];
                                const T t0 = *(const T*)(tb - x0.e), t1 = *(const T*)(tb - x1.e);
                                const T t2 = *(const T*)(tb - x2.e), t3 = *(const T*)(tb - x3.e);
                                acc += t0 * x0.v;
                                acc += t1 * x1.v;
                                acc += t2 * x2.v;
                                acc += t3 * x3.v;
                            }
                            for (; k < n; k++) acc += *(const T*)(tb - ent[k].e) * ent[k].v;
                            wave_lds_sync();
                        } else {
                            while (bal) {
                                const int b = __builtin_ctzll(bal);
                                bal &= bal - 1;
                                const unsigned pkb = (unsigned)__builtin_amdgcn_readlane((int)pkc, b);
                                const T vb = readlane_t<T>(v, b);
                                const int tp = kr2 - (int)(pkb >> 16), tq = lr2 - (int)(pkb & 0xffffu);
                                if (p >= 0 && (unsigned)tp < (unsigned)pnx && (unsigned)tq < (unsigned)pny) acc += tab[(tp + toff) * tpc + tq] * vb;
                            }
                        }
                    }
                    if (p < 0) acc = (T)0;  // rows past the image: the fast path read row 0's taps for them
                    char* d = tile + lane / LT::RPR * LT::PITCH + ii * 16 + lane % LT::RPR * (16 / LT::RPR);
                    if constexpr (F64) *(double*)d = acc;
                    else *(uint16_t*)d = f32_to_f16_rne((float)((double)acc * sc));
                }
                if (M.n_src - c0 - h >= 0 && M.n_src - c0 - h < LT::HC) {  // the data column
                    char* d = tile + lane / LT::RPR * LT::PITCH + (M.n_src - c0 - h) * 16 + lane % LT::RPR * (16 / LT::RPR);
                    if constexpr (F64) *(double*)d = dv;
                    else *(uint16_t*)d = f32_to_f16_rne((float)dv);
                }
                wave_lds_sync();
                uint4* dst = dst0 + (size_t)(q - 1) * (F64 ? 512 : 128) + h;
#pragma unroll
                for (int t = lane; t < LT::NRUN * 8; t += 64)
                    store_nt(&dst[(t >> 3) * 16 + (t & 7)], *(const uint4*)(tile + (t >> 3) * LT::PITCH + (t & 7) * 16));
                wave_lds_sync();
            }
        }
    }
}

int launch_build_lb_b(hipStream_t s, const BatchDev& bd, int max_rows, int mixed)
{
    if (max_rows <= 0) return 0;
    const int max_nkt = (max_rows + TS - 1) / TS;
    const size_t esz = mixed ? 4 : 8;
    // padded tap table when it fits in 32 KB, else the compact PSF (bounds tested everywhere)
    int tpc = bd.pny + LB_SPAN + 1;
    tpc = (tpc + 7) / 16 * 16 + 8;  // odd multiple of 8: the rows of an 8 x 8 pixel tile's taps on distinct banks
    int toff = LB_SPAN + 1, trows = bd.pnx + 2 * LB_SPAN + 2;
    if ((size_t)trows * tpc * esz > 32 * 1024) {
        tpc = bd.pny;
        toff = 0;
        trows = bd.pnx;
    }
    const size_t tab_bytes = ((size_t)trows * tpc * esz + 15) / 16 * 16;
    if (tab_bytes > 64 * 1024) return -1;  // PSF beyond the LDS budget
    if (mixed) {
        const size_t lds = tab_bytes + 4 * (64 * sizeof(LbEnt<float>) + LbTile<float>::BYTES);
        allow_big_lds((const void*)k_build_lb_b<float>);
        hipLaunchKernelGGL(k_build_lb_b<float>, dim3(max_nkt, bd.B), dim3(256), lds, s, bd, (int)tab_bytes, toff, tpc, trows);
    } else {
        const size_t lds = tab_bytes + 4 * (64 * sizeof(LbEnt<double>) + LbTile<double>::BYTES);
        allow_big_lds((const void*)k_build_lb_b<double>);
        hipLaunchKernelGGL(k_build_lb_b<double>, dim3(max_nkt, bd.B), dim3(256), lds, s, bd, (int)tab_bytes, toff, tpc, trows);
    }
    return 0;
}

__global__ void k_gather_cvec_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || r >= M.nrows) return;
    bd.cvec[M.cvec_off + r] =
        (r < M.n_img) ? bd.covinv[bd.act_pix[item * bd.s_pix + bd.perm[item * bd.s_pix + r]]] : 0.0;
}

void launch_gather_cvec_b(hipStream_t s, const BatchDev& bd, int max_rows)
{
    if (max_rows > 0) hipLaunchKernelGGL(k_gather_cvec_b, dim3((max_rows + 255) / 256, bd.B), dim3(256), 0, s, bd);
}

__device__ __forceinline__ void tri_decode(int t, int& I, int& J)
{
    int i = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((i + 1) * (i + 2) / 2 <= t) i++;
    while (i * (i + 1) / 2 > t) i--;
    I = i;
    J = t - i * (i + 1) / 2;
}

// Tile order of the SYRK and Cholesky-update grids.  Workgroups are dealt to the 8 XCDs
// round-robin by linear index, and each XCD has its own L2.  The lower-triangular tile set is cut
// into SUPER x SUPER super-tiles (all slots of a super-tile are launched; slots above the
// diagonal or past the matrix exit at once) and the grid is arranged so that every super-tile
// lands whole on one XCD: its SUPER^2 workgroups run together there and share SUPER row blocks
// and SUPER column blocks in that L2.  Super-tiles go to XCDs round-robin, starting at an XCD
// rotated by the item (blockIdx.y), so small triangles of many items still spread over all XCDs.
#define SUPER 8
#define NXCD 8
// Extents below one super-tile get a plain triangular grid (g -> tri_decode(g)); larger ones whole
// super-tile rounds.  syrk_tile tells the two apart by the grid size.
static unsigned syrk_grid(int max_ncb)
{
    if (max_ncb < SUPER) return (unsigned)std::max(1, max_ncb * (max_ncb + 1) / 2);
    const unsigned nS = (max_ncb + SUPER - 1) / SUPER;
    const unsigned nsup = nS * (nS + 1) / 2;
    const unsigned rounds = (nsup + NXCD - 1) / NXCD;
    return rounds * NXCD * SUPER * SUPER;
}

__device__ __forceinline__ bool syrk_tile(int ncb, int& I, int& J)
{
    const unsigned g = blockIdx.x;
    if (gridDim.x < NXCD * SUPER * SUPER) {
        tri_decode((int)g, I, J);
        return I < ncb;
    }
    const unsigned x = g % NXCD, k = g / NXCD;
    const unsigned w = k % (SUPER * SUPER), r = k / (SUPER * SUPER);
    const unsigned vx = (x + NXCD - (blockIdx.y % NXCD)) % NXCD;
    int SI, SJ;
    tri_decode((int)(r * NXCD + vx), SI, SJ);
    I = SI * SUPER + (int)(w / SUPER);
    J = SJ * SUPER + (int)(w % SUPER);
    return I < ncb && J <= I;
}

// Loads of a column block's strips of one chunk, all issued whatever the mask holds, so that the loads
// behind them can be counted and stay in flight: a strip that is absent gets an offset past the buffer
// resource's `bytes` and reads zero without touching memory.
#define NO_STRIP 0x40000000
__device__ __forceinline__ __amdgpu_buffer_rsrc_t strips_rsrc(const void* pool, unsigned first, int strip_bytes, int nstrip)
{
    return __builtin_amdgcn_make_buffer_rsrc((char*)pool + (size_t)first * strip_bytes, 0, strip_bytes * nstrip, 0x00020000);
}
// byte offset of strip a (asked in order, `next` from 0), or NO_STRIP
__device__ __forceinline__ int strip_off(unsigned mask, int a, int strip_bytes, int& next)
{
    const bool has = mask >> a & 1;
    const int o = has ? next : NO_STRIP;
    next += has ? strip_bytes : 0;
    return o;
}
__device__ __forceinline__ u32x4_t load_strip(__amdgpu_buffer_rsrc_t rs, int off) { return __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0); }

// The chunks k0 .. k0 + SYRK_LIST - 1 holding strips of both column blocks I and J, in order, as
// {first strip of I's, of J's (slots in the pool), masks I | J << 8, chunk}; returns how many.  Called by
// the 256 threads of a workgroup; `list` may be read after it and rewritten after a barrier.
#define SYRK_LIST 512
__device__ __forceinline__ int chunk_list(const BatchDev& bd, const ItemMeta& M, int I, int J, int k0, uint4* list, int* cnt)
{
    const unsigned* sI = bd.sup + M.sup_off + (size_t)I * M.nkt;
    const unsigned* sJ = bd.sup + M.sup_off + (size_t)J * M.nkt;
    const int* bb = bd.bbase + M.bb_off;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    unsigned e[2], f[2];
    unsigned long long bal[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {  // group g = w + 4 u: chunks k0 + 64 g ..
        const int k = k0 + 64 * (w + 4 * u) + lane;
        e[u] = k < M.nkt ? sI[k] : 0u;
        f[u] = k < M.nkt ? sJ[k] : 0u;
        bal[u] = __ballot(e[u] && f[u]);
        if (lane == 0) cnt[w + 4 * u] = __popcll(bal[u]);
    }
    __syncthreads();
    int n = 0, off[2] = {0, 0};
#pragma unroll
    for (int g = 0; g < 8; g++) {
        if (g == w) off[0] = n;
        if (g == w + 4) off[1] = n;
        n += cnt[g];
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int k = k0 + 64 * (w + 4 * u) + lane;
        if (e[u] && f[u]) {
            const unsigned b = (unsigned)bb[k];
            list[off[u] + __popcll(bal[u] & ((1ull << lane) - 1ull))] =
                make_uint4(b + (e[u] >> 8), b + (f[u] >> 8), (e[u] & 255u) | (f[u] & 255u) << 8, (unsigned)k);
        }
    }
    __syncthreads();
    return n;
}

// ------------------------------------------------------------------------------------------------
// F = Lb^T C Lb, FP64 MFMA (v_mfma_f64_16x16x4f64; accumulator register v of lane l holds
// D[l/16 + 4v][l%16] on gfx950).  One workgroup per lower 64 x 64 tile; only chunks with strips in both
// blocks, and of their 4 x 4 pairs of 16-column strips only those held (a chunk's rows reach 33 strips on
// the 200 x 200 / 60 x 60 workload, 12.3 blocks of 64 columns: 44 % of the blocks' products).  Wave w takes
// rows 16 w .. 16 w + 15 of every chunk for the whole tile, straight from the pool into operand registers
// (a lane's 16 bytes are two rows of its column), so there is no staging and no barrier; its second
// half's loads and the next chunk's first half's are in flight during the products.  The four waves'
// sums are added in a fixed order at the end.  100 items of the workload: 44.9 ms on whole 64-blocks
// staged in LDS, now 17.9 (10.2 ms of MFMA issue; 104 GB from beyond the L2s, 5.8 TB/s); one item 1.69 ->
// 0.5 ms, one of 900 columns 0.27 -> 0.08.
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_syrk_f64_b(BatchDev bd)
{
    __shared__ uint4 list[SYRK_LIST];
    __shared__ int cnt[8];
    __shared__ double red[2][TS * TS];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    int I, J;
    if (!syrk_tile(M.ncb, I, J)) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool dg = I == J;
    // rows 16 w .. of a strip: 128 16-byte pieces from 128 w on, half h of them 64
    const double* const pool = (const double*)bd.lb + M.lb_off;
    const int vo = (128 * w + lane) * 16;
    const double2_t* const cvec = (const double2_t*)(bd.cvec + M.cvec_off) + 8 * w + (lane >> 4);
    double4_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[a][c] = (double4_t){0, 0, 0, 0};
    for (int k0 = 0; k0 < M.nkt; k0 += SYRK_LIST) {
        const int n = chunk_list(bd, M, I, J, k0, list, cnt);
        double2_t A[2][4], Bq[2][4], C[2];
        unsigned mk = 0;
        auto entry = [&](int i) {
            const uint4 v = list[i];
            return make_uint4((unsigned)__builtin_amdgcn_readfirstlane((int)v.x), (unsigned)__builtin_amdgcn_readfirstlane((int)v.y),
                              (unsigned)__builtin_amdgcn_readfirstlane((int)v.z), (unsigned)__builtin_amdgcn_readfirstlane((int)v.w));
        };
        auto load = [&](const uint4& e, int h) {
            const __amdgpu_buffer_rsrc_t sa = strips_rsrc(pool, e.x, 8192, 4), sb = strips_rsrc(pool, e.y, 8192, 4);
            C[h] = cvec[(size_t)e.w * 32 + 4 * h];
            int na = 0, nb = 0;
#pragma unroll
            for (int a = 0; a < 4; a++) A[h][a] = __builtin_bit_cast(double2_t, load_strip(sa, vo + 1024 * h + strip_off(e.z, a, 8192, na)));
#pragma unroll
            for (int c = 0; c < 4; c++) Bq[h][c] = __builtin_bit_cast(double2_t, load_strip(sb, vo + 1024 * h + strip_off(e.z, 8 + c, 8192, nb)));
        };
        auto mul = [&](int h) {
            double2_t B[4];
#pragma unroll
            for (int c = 0; c < 4; c++) B[c] = Bq[h][c] * C[h];
#pragma unroll
            for (int a = 0; a < 4; a++)
                if (mk >> a & 1)
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        if ((mk >> (8 + c) & 1) && !(dg && c > a)) {
                            acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[h][a].x, B[c].x, acc[a][c], 0, 0, 0);
                            acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[h][a].y, B[c].y, acc[a][c], 0, 0, 0);
                        }
        };
        if (n) {
            uint4 e = entry(0);
            load(e, 0);
            __builtin_amdgcn_sched_barrier(0);  // in this order, as in the loop: the waits count them
            load(e, 1);
            for (int i = 0; i < n; i++) {  // (after the last chunk the loads repeat it, for a fixed number in flight)
                mk = e.z;
                e = entry(min(i + 1, n - 1));
                mul(0);
                __builtin_amdgcn_sched_barrier(0);
                load(e, 0);
                __builtin_amdgcn_sched_barrier(0);
                mul(1);
                __builtin_amdgcn_sched_barrier(0);
                load(e, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();  // the list is rewritten
    }
    // ((w0 + w2) + (w1 + w3)); element (a, c, v) of a lane at ((a * 4 + c) * 4 + v) * 64 + lane
    auto put = [&](double* d) {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) d[((a * 4 + c) * 4 + v) * 64 + lane] = acc[a][c][v];
    };
    auto add = [&](const double* d) {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[a][c][v] += d[((a * 4 + c) * 4 + v) * 64 + lane];
    };
    if (w >= 2) put(red[w - 2]);
    __syncthreads();
    if (w < 2) add(red[w]);
    if (w == 1) put(red[1]);
    __syncthreads();
    if (w) return;
    add(red[1]);
    double* F = (bd.Fraw ? bd.Fraw : bd.F) + M.f_off;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = I * TS + a * 16 + (lane >> 4) + 4 * v, q = J * TS + c * 16 + (lane & 15);
                F[(size_t)r * M.ldN + q] = r > M.n_src ? (r == q ? 1.0 : 0.0) : acc[a][c][v];  // identity beyond the data row
            }
}

void launch_syrk_f64_b(hipStream_t s, const BatchDev& bd, int max_ncb)
{
    hipLaunchKernelGGL(k_syrk_f64_b, dim3(syrk_grid(max_ncb), bd.B), dim3(256), 0, s, bd);
}

// ------------------------------------------------------------------------------------------------
// F32 = Lb^T Lb on the mixed path: one FP16 pool of sqrt(c) s16-scaled rows in strips of 16 columns,
// v_mfma_f32_16x16x32_f16 accumulated in FP32, scaled back by s16^-2 (exact) at the store.  One
// workgroup per 128 x 128 lower tile of F.  A operand lane l holds A[i = l%16][8 consecutive k], B the
// same with j; accumulator register v of lane l holds D[4*(l/16) + v][l%16].  Only the strips a chunk
// holds are read (33 of 16 columns a chunk on the 200 x 200 / 60 x 60 workload against 8.5 blocks of
// 128); each row strip held is multiplied by all four of the wave's column strips if one of them is held,
// the absent ones as zeros (1.5 times the products of the pairs held).  As in the FP64 kernel the operands come straight from the pool into registers,
// SYRK_D chunks ahead, with no staging and no barrier: wave (kh, jh) takes rows 32 kh .. of every chunk for
// the tile's columns 64 jh .. (16-byte loads: a wave's load occupies the L1 for 16 cycles whatever its
// width, and four waves of 16 rows with 8-byte ones took 14.4 ms).  The two row halves' sums are added
// at the end, each wave finishing 64 x 64.  256 items of the workload: 15.3 ms on whole 128-blocks staged
// in LDS (114 GB from beyond the L2s), 15.6 with the strips staged there, now 10.1 (36 GB; 7 of them are
// issue: the masks' offsets and branches).
// ------------------------------------------------------------------------------------------------
#define SCB 128  // column-block width of the mixed path
__device__ __forceinline__ double item_lambda(const BatchDev& bd, int item) { return bd.lam ? bd.lam[item] : bd.lambda; }

// R entry (r, c), c <= r, of the banded curvature tiles (reference order, |r - c| within the band)
__device__ __forceinline__ double* rtile(const BatchDev& bd, const ItemMeta& M, int r, int c)
{
    const int I = r >> 6, J = c >> 6;
    return bd.R + M.r_off + ((size_t)I * (M.bwb + 1) + (I - J)) * TS * TS + (r & 63) * TS + (c & 63);
}
// the same entry of an item's R as read: R is built once per distinct R, by the item rrep names
__device__ __forceinline__ double rget(const BatchDev& bd, int item, int r, int c)
{
    return *rtile(bd, bd.meta[bd.rrep[item]], r, c);
}

// The FP16 SYRK's store: scaled back, the data row n kept with a large pivot (the refined solve never
// reads it), identity beyond n.  k_add_reg_b then adds lambda R.  The tiles go to Ff32 (F as formed); the
// Cholesky kernels that touch a block first (the first part's diagonal and panel kernels, the first
// strip and trailing updates) read it there and write the factor buffer F32.  A diagonal 64-tile is
// held whole (the refinement residual reads its upper half).  acc: 64 rows r0 .., 64 columns c0 ..
__device__ __forceinline__ void syrk_f16_store(const BatchDev& bd, const ItemMeta& M, int r0, int c0, const float4_t (&acc)[4][4])
{
    const int lane = threadIdx.x & 63;
    const float unscale = (float)(1.0 / (bd.s16 * bd.s16));
    const int ld = M.ldN, n = M.n_src;
    float* C = bd.Ff32 + M.f_off;
    r0 += 4 * (lane >> 4);
    c0 += lane & 15;
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = r0 + a * 16 + v, cg = c0 + c * 16;
                float x = acc[a][c][v] * unscale;
                if (r > n || cg > n) x = (r == cg) ? 1.0f : 0.0f;
                else if (r == n && cg == n) x = 1e30f;  // the rest of row n (D) is kept
                __builtin_nontemporal_store(x, &C[(size_t)r * ld + cg]);
            }
}

#define SYRK_D 2
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_syrk_f16_b(BatchDev bd)
{
    __shared__ uint4 list[SYRK_LIST];
    __shared__ int cnt[8];
    __shared__ float4_t red[4][16 * 64];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    int I, J;
    if (!syrk_tile(M.ncb, I, J)) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = w >> 1, jh = w & 1;
    // rows 32 kh .. of a strip: its 16-byte pieces 64 kh ..
    const uint16_t* const pool = (const uint16_t*)bd.lb + M.lb_off;
    const int vo = (64 * kh + lane) * 16;
    const unsigned rowsel = I == J && jh ? 0xf0u : 0xffu;  // (above the diagonal: not needed)
    float4_t acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[a][c] = (float4_t){0, 0, 0, 0};
    for (int k0 = 0; k0 < M.nkt; k0 += SYRK_LIST) {
        const int n = chunk_list(bd, M, I, J, k0, list, cnt);
        f16x8_t A[SYRK_D][8], B[SYRK_D][4];
        unsigned mk[SYRK_D];  // strips of the rows, of the wave's 64 columns << 8
        auto load = [&](int i, int s) {
            const uint4 v = list[i];
            const unsigned m = (unsigned)__builtin_amdgcn_readfirstlane((int)v.z);
            const unsigned mj = m >> (8 + 4 * jh) & 15u, mi = mj ? m & rowsel : 0u;
            const __amdgpu_buffer_rsrc_t sa = strips_rsrc(pool, (unsigned)__builtin_amdgcn_readfirstlane((int)v.x), 2048, 8);
            const __amdgpu_buffer_rsrc_t sb = strips_rsrc(pool, (unsigned)__builtin_amdgcn_readfirstlane((int)v.y), 2048, 8);
            int na = 2048 * __popc(m & 255u & ~rowsel), nb = jh ? 2048 * __popc(m >> 8 & 15u) : 0;
            mk[s] = mi;
#pragma unroll
            for (int a = 0; a < 8; a++) A[s][a] = __builtin_bit_cast(f16x8_t, load_strip(sa, vo + strip_off(mi, a, 2048, na)));
#pragma unroll
            for (int c = 0; c < 4; c++) B[s][c] = __builtin_bit_cast(f16x8_t, load_strip(sb, vo + strip_off(mj, c, 2048, nb)));
        };
        // SYRK_D chunks at a time; past the last one the loads repeat it and the products are left out, so
        // that the number of loads behind each product is fixed
        if (n) {
#pragma unroll
            for (int s = 0; s < SYRK_D; s++) {
                load(min(s, n - 1), s);
                __builtin_amdgcn_sched_barrier(0);  // in this order, as in the loop: the waits count them
            }
            for (int i0 = 0; i0 < n; i0 += SYRK_D)
#pragma unroll
                for (int s = 0; s < SYRK_D; s++) {
                    const unsigned m = i0 + s < n ? mk[s] : 0u;
#pragma unroll
                    for (int a = 0; a < 8; a++)
                        if (m >> a & 1)
#pragma unroll
                            for (int c = 0; c < 4; c++)
                                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[s][a], B[s][c], acc[a][c], 0, 0, 0);
                    load(min(i0 + s + SYRK_D, n - 1), s);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        __syncthreads();  // the list is rewritten
    }
    // wave (kh, jh) finishes the tile's rows 64 kh .. of its columns: its own sums and wave (1 - kh, jh)'s
    float4_t o[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            o[a][c] = kh ? acc[4 + a][c] : acc[a][c];
            red[w][(a * 4 + c) * 64 + lane] = kh ? acc[a][c] : acc[4 + a][c];
        }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float4_t t = red[w ^ 2][(a * 4 + c) * 64 + lane];
            o[a][c] = kh ? t + o[a][c] : o[a][c] + t;
        }
    if (I == J && jh > kh) return;  // above the diagonal
    syrk_f16_store(bd, M, I * SCB + 64 * kh, J * SCB + 64 * jh, o);
}

void launch_syrk_f16_b(hipStream_t s, const BatchDev& bd, int max_ncb)
{
    hipLaunchKernelGGL(k_syrk_f16_b, dim3(syrk_grid(max_ncb), bd.B), dim3(256), 0, s, bd);
}

// ------------------------------------------------------------------------------------------------
// curvature R (exact small integers) in banded tiles.  In the active (j-major) order an R entry
// couples cells at most two source rows apart, |a - b| <= 2*snx, so the lower band in 64-blocks is
// bwb = (2*snx)/64 + 1 and the Cholesky factor stays inside it.
// ------------------------------------------------------------------------------------------------

__global__ void __launch_bounds__(256) k_zero_r_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || bd.rrep[item] != item) return;  // an earlier item holds this R
    // 16-byte stores: the band holds whole 64 x 64 tiles and starts on a tile boundary
    double2* R2 = (double2*)(bd.R + M.r_off);
    const size_t n2 = (size_t)(M.ldN / TS) * (M.bwb + 1) * TS * TS / 2;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n2; t += (size_t)gridDim.x * blockDim.x)
        R2[t] = make_double2(0.0, 0.0);
}

__global__ void __launch_bounds__(256) k_curvature_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || bd.rrep[item] != item) return;  // an earlier item holds this R
    if (c >= M.snx * M.sny) {
        // identity on the padding rows (the data row of F's augmented matrix has no R entries)
        const int r = c - M.snx * M.sny + M.n_src;
        if (r < M.ldN && c - M.snx * M.sny < M.ldN - M.n_src) *rtile(bd, M, r, r) = 1.0;
        return;
    }
    const int* sidx = bd.sidx + item * bd.s_cell;
    const int a = sidx[c];
    if (a < 0) return;
    const int snx = M.snx, sny = M.sny;
    const int i = c / sny, j = c % sny;
    for (int l = 0; l < 2; l++) {
        int ids[3];
        double h[3];
        int m = 0;
        ids[m] = a;
        h[m++] = -2.0;
        int nb0, nb1;
        if (l == 0) {
            nb0 = (i < snx - 1) ? sidx[(i + 1) * sny + j] : -1;
            nb1 = (i > 0) ? sidx[(i - 1) * sny + j] : -1;
        } else {
            nb0 = (j < sny - 1) ? sidx[i * sny + j + 1] : -1;
            nb1 = (j > 0) ? sidx[i * sny + j - 1] : -1;
        }
        if (nb0 >= 0) { ids[m] = nb0; h[m++] = 1.0; }
        if (nb1 >= 0) { ids[m] = nb1; h[m++] = 1.0; }
        for (int x = 0; x < m; x++)
            for (int y = x; y < m; y++) {
                const int r0 = ids[x] > ids[y] ? ids[x] : ids[y];
                const int c0 = ids[x] > ids[y] ? ids[y] : ids[x];
                atomicAdd(rtile(bd, M, r0, c0), h[x] * h[y]);
            }
    }
}

// R is a function of the grid's shape (snx, sny) and the item's active-index map (sidx): its entries
// are sums of small integers, exact in any order.  Items with equal shapes and maps share one
// factorization: k_rhash_b keys each item (an order-free sum of mixed (cell, index) words),
// k_rdup_b compares an item with the earlier items of equal key, entry by entry, and takes the first
// equal one as its representative (whose own representative is itself).
__device__ __forceinline__ unsigned long long mix64(unsigned long long x)
{
    x ^= x >> 30;
    x *= 0xbf58476d1ce4e5b9ULL;
    x ^= x >> 27;
    x *= 0x94d049bb133111ebULL;
    x ^= x >> 31;
    return x;
}

__global__ void __launch_bounds__(256) k_rhash_b(BatchDev bd)
{
    __shared__ unsigned long long sh[256];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int tid = threadIdx.x;
    unsigned long long h = 0;
    if (M.valid) {
        const int* sidx = bd.sidx + item * bd.s_cell;
        const int n = M.snx * M.sny;
        for (int c = tid; c < n; c += 256) h += mix64(((unsigned long long)c << 32) ^ (unsigned)(sidx[c] + 1));
    }
    sh[tid] = h;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) sh[tid] += sh[tid + st];
        __syncthreads();
    }
    if (tid == 0) bd.rkey[item] = M.valid ? sh[0] ^ mix64(((unsigned long long)M.snx << 32) | (unsigned)M.sny) : 0ULL;
}

__global__ void __launch_bounds__(256) k_rdup_b(BatchDev bd)
{
    __shared__ int eq;
    const int b = blockIdx.y;
    const ItemMeta& M = bd.meta[b];
    int rep = b;
    if (M.valid) {
        const int n = M.snx * M.sny;
        const int* sb = bd.sidx + b * bd.s_cell;
        for (int a = 0; a < b; a++) {
            const ItemMeta& A = bd.meta[a];
            if (!A.valid || bd.rkey[a] != bd.rkey[b] || A.snx != M.snx || A.sny != M.sny || A.n_src != M.n_src) continue;
            const int* sa = bd.sidx + a * bd.s_cell;
            if (threadIdx.x == 0) eq = 1;
            __syncthreads();
            for (int c = threadIdx.x; c < n; c += 256)
                if (sa[c] != sb[c]) eq = 0;
            __syncthreads();
            const int same = eq;
            __syncthreads();
            if (same) {
                rep = a;
                break;
            }
        }
    }
    if (threadIdx.x == 0) bd.rrep[b] = rep;
}

void launch_rdup_b(hipStream_t s, const BatchDev& bd)
{
    hipLaunchKernelGGL(k_rhash_b, dim3(1, bd.B), dim3(256), 0, s, bd);
    hipLaunchKernelGGL(k_rdup_b, dim3(1, bd.B), dim3(256), 0, s, bd);
}

void launch_curvature_b(hipStream_t s, const BatchDev& bd, int max_cells, int max_rtiles)
{
    hipLaunchKernelGGL(k_zero_r_b, dim3(grid_for((size_t)max_rtiles * TS * TS, 256, 2048), bd.B), dim3(256), 0, s, bd);
    const int n = max_cells + QLX_MAX_LD;
    hipLaunchKernelGGL(k_curvature_b, dim3((n + 255) / 256, bd.B), dim3(256), 0, s, bd);
}

// regparam optimisation: F's lower tiles from F as formed (Fraw), for the next lambda
__global__ void __launch_bounds__(256) k_copy_f_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const int nb = M.ldN / TS;
    if ((int)blockIdx.x >= nb * (nb + 1) / 2) return;
    int I, J;
    tri_decode(blockIdx.x, I, J);
    const size_t o = M.f_off + (size_t)I * TS * M.ldN + (size_t)J * TS;
#pragma unroll
    for (int e = 2 * threadIdx.x; e < TS * TS; e += 512) {
        const size_t t = o + (size_t)(e >> 6) * M.ldN + (e & 63);
        *(double2_t*)&bd.F[t] = *(const double2_t*)&bd.Fraw[t];
    }
}

// F += lambda R.  R couples a cell with itself and the cells one and two away along each axis, so a
// thread takes a cell's five pairs that lie ahead of it: a pass over those entries instead of one over F
// that gathered an R entry for each of its own (FP16 SYRK's store 17.7 -> 13.8 ms of the kernel per 256
// items of 3600 cells, the FP64 pass 2.45 ms per 100).  R is held in the reference order, F in the
// internal one.  FP32: the diagonal 64-tiles' upper halves too, and the diagonal, as rounded to FP32, into Fdiag.
template <typename T>
__global__ void __launch_bounds__(256) k_add_reg_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (!M.valid || c >= M.snx * M.sny) return;
    const int* sidx = bd.sidx + item * bd.s_cell;
    const int* tix = bd.tix + item * bd.s_cell;
    if (sidx[c] < 0) return;
    const int i = c / M.sny, j = c - i * M.sny;
    T* F = (sizeof(T) == 8 ? (T*)bd.F : (T*)bd.Ff32) + M.f_off;
    double* fdiag = bd.vec + M.vec_off + 3 * (size_t)M.ldN;
    const double lam = item_lambda(bd, item);
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const int di = k == 1 ? 1 : k == 2 ? 2 : 0, dj = k == 3 ? 1 : k == 4 ? 2 : 0;
        if (i + di >= M.snx || j + dj >= M.sny) continue;
        const int d = c + di * M.sny + dj;
        if (sidx[d] < 0) continue;
        const int pa = sidx[c], pb = sidx[d], a = tix[c], b = tix[d];
        const int r = a > b ? a : b, q = a > b ? b : a;
        T* f = &F[(size_t)r * M.ldN + q];
        const T x = (T)((double)*f + lam * rget(bd, item, pa > pb ? pa : pb, pa > pb ? pb : pa));
        *f = x;
        if (sizeof(T) == 4) {
            if (k == 0) fdiag[r] = (double)x;
            else if ((r >> 6) == (q >> 6)) F[(size_t)q * M.ldN + r] = x;
        }
    }
}

void launch_add_reg_b(hipStream_t s, const BatchDev& bd, int max_ld, int max_cells, int f32)
{
    const dim3 grid((max_cells + 255) / 256, bd.B);
    if (f32) {
        hipLaunchKernelGGL(k_add_reg_b<float>, grid, dim3(256), 0, s, bd);
        return;
    }
    const int nb = max_ld / TS;
    if (bd.Fraw) hipLaunchKernelGGL(k_copy_f_b, dim3(nb * (nb + 1) / 2, bd.B), dim3(256), 0, s, bd);
    hipLaunchKernelGGL(k_add_reg_b<double>, grid, dim3(256), 0, s, bd);
}

// ------------------------------------------------------------------------------------------------
// Batched blocked Cholesky (lower, 64x64 tiles) of many matrices, FP64 or FP32 per matrix, dense
// or banded per matrix: diagonal blocks (factor + block inverse W), left-looking panel steps
// (A_ib,kb <- (A_ib,kb - earlier blocks) W^T) and trailing updates (A_IJ -= P_I P_J^T), products on MFMA.
// Matrices with fewer blocks skip the step; the upper triangle is never written.
// Restates Cholesky_dcmp_packed (pixelgrid.cpp:17071-17105) blockwise: a pivot of a row < n that
// is not positive (negative, zero or NaN) sets *status and the factorization continues with
// sqrt(|a|) as that routine does; the item is then reported as not positive definite (the
// reference's non-MKL caller dies there, pixelgrid.cpp:17384).
// ------------------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T* tile_ptr(const MatDesc& D, int I, int J, int& ld)
{
    if (D.bwb > 0) {
        ld = TS;
        return (T*)D.A + ((size_t)I * (D.bwb + 1) + (I - J)) * TS * TS;
    }
    ld = D.ld;
    return (T*)D.A + (size_t)I * TS * D.ld + (size_t)J * TS;
}

__device__ __forceinline__ int band_last(const MatDesc& D, int kb)
{
    return D.bwb > 0 ? min(D.nb - 1, kb + D.bwb) : D.nb - 1;
}

// MFMA operand/accumulator types: FP64 v_mfma_f64_16x16x4f64 (accumulator register v of lane l
// holds D[l/16 + 4v][l%16]) and FP32 v_mfma_f32_16x16x4f32 (D[4(l/16) + v][l%16])
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
    typedef double4_t acc_t;
    typedef double2 vec_t;
    __device__ static acc_t op(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mfma16<float> {
    typedef float4_t acc_t;
    typedef float4 vec_t;
    __device__ static acc_t op(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// value of lane `src` in every lane (src is a constant of the unrolled loops that call this)
__device__ __forceinline__ float lane_bcast(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

// 64x64x64 MFMA product acc = sum_q A(i, q) B(j, q) with A and B stored "row holds the k-vector"
// (the panel blocks as they lie in the factor), staged into LDS unchanged ([i][k], row pitch
// LDT) and read as MFMA operands A[i = lane%16][k = kk + lane/16].
#define LDT 68
template <typename T>
__device__ __forceinline__ void stage64(const T* P, int sp, T (*S)[LDT])
{
    typedef typename Mfma16<T>::vec_t V;
    constexpr int VW = sizeof(V) / sizeof(T);
    for (int e = threadIdx.x * VW; e < TS * TS; e += 256 * VW) {
        const int i = e >> 6, k = e & 63;
        *(V*)&S[i][k] = *(const V*)&P[(size_t)i * sp + k];
    }
}

template <typename T>
__device__ __forceinline__ void mma64_add(T (*As)[LDT], T (*Bs)[LDT], typename Mfma16<T>::acc_t acc[2][2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll 4
    for (int kk = 0; kk < TS; kk += 4) {
        const int kq = kk + (lane >> 4);
        T a0 = As[wr * 32 + (lane & 15)][kq];
        T a1 = As[wr * 32 + 16 + (lane & 15)][kq];
        T b0 = Bs[wc * 32 + (lane & 15)][kq];
        T b1 = Bs[wc * 32 + 16 + (lane & 15)][kq];
        acc[0][0] = Mfma16<T>::op(a0, b0, acc[0][0]);
        acc[0][1] = Mfma16<T>::op(a0, b1, acc[0][1]);
        acc[1][0] = Mfma16<T>::op(a1, b0, acc[1][0]);
        acc[1][1] = Mfma16<T>::op(a1, b1, acc[1][1]);
    }
}

template <typename T>
__device__ __forceinline__ void mma64(T (*As)[LDT], T (*Bs)[LDT], typename Mfma16<T>::acc_t acc[2][2])
{
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c] = (typename Mfma16<T>::acc_t){0, 0, 0, 0};
    mma64_add<T>(As, Bs, acc);
}

// C (64x64 at row pitch ldc) = acc
template <typename T>
__device__ __forceinline__ void store64(T* C, int ldc, const typename Mfma16<T>::acc_t acc[2][2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int rr = wr * 32 + a * 16 + Mfma16<T>::row(lane, v);
                const int cc = wc * 32 + c * 16 + (lane & 15);
                C[(size_t)rr * ldc + cc] = acc[a][c][v];
            }
}

// the 16 C values of a lane (store64's layout), loaded before the staging barrier so their latency
// overlaps the operand loads
template <typename T>
__device__ __forceinline__ void load64c(const T* C, int ldc, T (&cv)[16])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int rr = wr * 32 + a * 16 + Mfma16<T>::row(lane, v);
                const int cc = wc * 32 + c * 16 + (lane & 15);
                cv[(a * 2 + c) * 4 + v] = C[(size_t)rr * ldc + cc];
            }
}

#define TT 128  // tile side of the trailing updates
// FP32 matrices (mixed path): the trailing update C(I, J) -= sum over the panel's column blocks of
// L(I, q) L(J, q)^T on 128 x 128 tiles, with the panel operands split x = hi + lo
// into BF16 while they are staged (hi = bf16(x), lo = bf16(x - hi): 2^-17 of each entry, with the
// hardware round-to-nearest conversion) and all four products hi*hi + hi*lo + lo*hi + lo*lo on
// v_mfma_f32_16x16x32_bf16, accumulated in FP32.  The accumulators start from the C tile and the A
// operand is negated while staging, so the MFMAs form C - A B^T directly.  Loads go through a buffer
// resource (32-bit offsets: one VGPR per lane, row offsets in SGPRs).  Operands are staged 32 k at
// a time (LDS: A hi, A lo, B hi, B lo as 128 rows x TBP BF16, 40 KB; 80-byte rows put the 16 rows
// of an operand read on distinct bank groups), which with 150 registers allows three waves per SIMD.
// The update covers the 128 x 128 tiles of rows and columns >= k0 + nq (64-blocks) from the nq panel
// blocks k0 .. k0+nq-1; ncolt > 0 restricts it to the first ncolt tile columns (a strip).
#define TBP 40
static_assert((long long)QLX_MAX_LD * QLX_MAX_LD * 4 < (1LL << 31), "trailing-update byte offsets must fit in 31 bits");
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void chol_diag_f32_4w(const MatDesc& D, int kb, float* tile, int ld, float (&a)[16],
                                                 float (*Lt)[TS], float (*X)[TS], float* Rd);

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3)))
k_chol_trail_bf16(const MatDesc* mats, int k0, int nq, int ncolt, int fdiag)
{
    typedef float P __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(1))) float gfloat;
    extern __shared__ double trail_raw[];
    __bf16* Ah = (__bf16*)trail_raw;
    __bf16* Al = Ah + TT * TBP;
    __bf16* Bh = Al + TT * TBP;
    __bf16* Bl = Bh + TT * TBP;
    const MatDesc D = mats[blockIdx.y];
    const int r0b = k0 + nq;
    if (r0b >= D.nb) return;
    const int nt = (D.nb - r0b) / 2;
    int I2 = -1, J2 = -1;
    if (ncolt == 0) {
        if (!syrk_tile(nt, I2, J2)) return;
    } else {
        int t = blockIdx.x;
        for (int j = 0; j < ncolt && j < nt; j++) {
            if (t < nt - j) {
                J2 = j;
                I2 = j + t;
                break;
            }
            t -= nt - j;
        }
        if (J2 < 0) return;
    }
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wr = w >> 1, wc = w & 1;
    const int ld = D.ld;  // ld <= QLX_MAX_LD: byte offsets within the matrix fit in 31 bits
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(D.A, 0, ld * ld * 4, 0x00020000);
    // C tiles: from F as formed (A0) in the first update, which thereby moves them into A
    const __amdgpu_buffer_rsrc_t rc = (k0 == 0 && D.A0) ? __builtin_amdgcn_make_buffer_rsrc(D.A0, 0, ld * ld * 4, 0x00020000) : rs;
    const int rI = (r0b + 2 * I2) * TS, rJ = (r0b + 2 * J2) * TS;
    // byte offsets: the lane's part in a VGPR, the uniform part in an SGPR.  Staging step st covers
    // columns 32 st .. 32 st + 31 of the panel; piece h of a thread: row srow + 32 h, columns
    // 4 (tid & 7) .. +3 of the step.  The 16 lanes of each group of tid stage rows r and r + 4,
    // whose 64-byte LDS pieces (row pitch 80 bytes) fall on disjoint banks
    const int g16 = tid >> 4;
    const int srow = (g16 & 3) + 8 * (g16 >> 2) + 4 * ((tid >> 3) & 1);
    const int vp = (srow * ld + 4 * (tid & 7)) * 4;
    const int sA = (rI * ld + k0 * TS) * 4, sB = (rJ * ld + k0 * TS) * 4;
    const int vc = ((wr * 64 + 4 * (lane >> 4)) * ld + wc * 64 + (lane & 15)) * 4;
    const int sC = (rI * ld + rJ) * 4;
    float4_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                acc[a][c][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rc, vc + c * 64, sC + (a * 16 + v) * ld * 4, 0));
    P pa[4], pb[4];
#define TRAIL_LOAD_BF(st)                                                                                          \
    {                                                                                                              \
        _Pragma("unroll") for (int h = 0; h < 4; h++)                                                              \
        {                                                                                                          \
            pa[h] = __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b128(rs, vp, sA + (32 * h * ld + (st) * 32) * 4, 0)); \
            pb[h] = __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b128(rs, vp, sB + (32 * h * ld + (st) * 32) * 4, 0)); \
        }                                                                                                          \
    }
    TRAIL_LOAD_BF(0);
    const int nst = 2 * nq;
    for (int st = 0; st < nst; st++) {
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 4; h++) {
            const int i = srow + 32 * h, k = 4 * (tid & 7);
            const P xa = -pa[h], xb = pb[h];
            const bf16x4_t ah = __builtin_convertvector(xa, bf16x4_t);
            const bf16x4_t bh = __builtin_convertvector(xb, bf16x4_t);
            const bf16x4_t al = __builtin_convertvector(xa - __builtin_convertvector(ah, P), bf16x4_t);
            const bf16x4_t bl = __builtin_convertvector(xb - __builtin_convertvector(bh, P), bf16x4_t);
            *(bf16x4_t*)&Ah[i * TBP + k] = ah;
            *(bf16x4_t*)&Al[i * TBP + k] = al;
            *(bf16x4_t*)&Bh[i * TBP + k] = bh;
            *(bf16x4_t*)&Bl[i * TBP + k] = bl;
        }
        __syncthreads();
        if (st + 1 < nst) TRAIL_LOAD_BF(st + 1);
        const int kq = 8 * (lane >> 4);
        bf16x8_t bhv[4], blv[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int jb = (wc * 64 + t * 16 + (lane & 15)) * TBP + kq;
            bhv[t] = *(const bf16x8_t*)&Bh[jb];
            blv[t] = *(const bf16x8_t*)&Bl[jb];
        }
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int ia = (wr * 64 + a * 16 + (lane & 15)) * TBP + kq;
            const bf16x8_t ahv = *(const bf16x8_t*)&Ah[ia];
            const bf16x8_t alv = *(const bf16x8_t*)&Al[ia];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahv, bhv[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahv, blv[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alv, bhv[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alv, blv[c], acc[a][c], 0, 0, 0);
            }
        }
    }
#undef TRAIL_LOAD_BF
    // plain global stores (the buffer-store form stored one register for all four rows of a
    // 16 x 16 block under the diagonal predicate with this compiler)
    const bool diag = (I2 == J2);
    gfloat* Cg = (gfloat*)D.A + (size_t)rI * ld + rJ;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int rr = wr * 64 + a * 16 + 4 * (lane >> 4) + v;
                const int cc = wc * 64 + c * 16 + (lane & 15);
                if (!diag || cc <= rr) Cg[(size_t)rr * ld + cc] = acc[a][c][v];
            }
    // fdiag: the workgroup of tile (0, 0) also factors diagonal block r0b, now up to date (wave 0's
    // quadrant), so the part that starts there needs no diagonal launch; through LDS (S, 64 x 65,
    // over the operand tiles) into rows per lane, as the panel kernel does
    if (fdiag && I2 == 0 && J2 == 0) {
        float* S = (float*)trail_raw;
        float(*Lt)[TS] = (float(*)[TS])(S + TS * 65);
        float* Rd = S + TS * 65 + TS * TS;
        __syncthreads();
        if (w == 0) {
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int c = 0; c < 4; c++)
#pragma unroll
                    for (int v = 0; v < 4; v++) S[(a * 16 + 4 * (lane >> 4) + v) * 65 + c * 16 + (lane & 15)] = acc[a][c][v];
        }
        __syncthreads();
        float av[16];
#pragma unroll
        for (int j = 0; j < 16; j++) av[j] = S[lane * 65 + 16 * w + j];
        chol_diag_f32_4w(D, r0b, (float*)D.A + (size_t)rI * ld + rJ, ld, av, Lt, (float(*)[TS])S, Rd);  // X over S: read before its first barrier
    }
}

// The left-looking panel step for FP32 matrices (the FP64 one's schedule) with the
// products on v_mfma_f32_16x16x32_bf16: every operand is split x = hi + lo into BF16 as it is
// staged (as in k_chol_trail_bf16) and the four products hi*hi + hi*lo + lo*hi + lo*lo are summed
// in FP32 (1.9 ms faster than FP32 MFMA per batch of 256 3712 x 3712 matrices; |delta lnE| against
// FP64 unchanged).  The workgroup of row block kb + 1, having brought diagonal block kb + 1 up to
// date, also factors it (chol_diag_f32_4w: the same bits as the diagonal kernel), so within a part
// only the first column block needs a diagonal launch; the grid is (matrices, row blocks) so that
// these workgroups are dispatched first (dispatched last, their serial factorization prolonged
// every launch).  LDS: A hi, A lo, B hi, B lo, 64 rows x LPB BF16 each (144-byte rows: the 16 rows
// of an operand read start on distinct 16-byte bank groups).
#define LPB 72
typedef float f32x4_t __attribute__((ext_vector_type(4)));
// a 64 x 64 FP32 block (row pitch sp) into registers: thread piece h holds row e >> 6, columns
// e & 63 .. +3 of e = (tid + 256 h) * 4
__device__ __forceinline__ void load64_regs(const float* P, int sp, f32x4_t (&r)[4])
{
#pragma unroll
    for (int h = 0; h < 4; h++) {
        const int e = (threadIdx.x + 256 * h) * 4;
        r[h] = *(const f32x4_t*)&P[(size_t)(e >> 6) * sp + (e & 63)];
    }
}
// those registers split x = hi + lo into BF16 rows of an operand
__device__ __forceinline__ void split64_store(const f32x4_t (&r)[4], __bf16* H, __bf16* L)
{
#pragma unroll
    for (int h = 0; h < 4; h++) {
        const int e = (threadIdx.x + 256 * h) * 4;
        const int i = e >> 6, k = e & 63;
        const bf16x4_t xh = __builtin_convertvector(r[h], bf16x4_t);
        *(bf16x4_t*)&H[i * LPB + k] = xh;
        *(bf16x4_t*)&L[i * LPB + k] = __builtin_convertvector(r[h] - __builtin_convertvector(xh, f32x4_t), bf16x4_t);
    }
}

// an accumulator tile (mma64's layout: wave (wr, wc) holds quadrant rows wr*32.., columns wc*32..)
// split into H / L as the rows of an operand
__device__ __forceinline__ void acc64_split(const float4_t (&acc)[2][2], __bf16* H, __bf16* L)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int rr = wr * 32 + a * 16 + 4 * (lane >> 4) + v;
                const int cc = wc * 32 + c * 16 + (lane & 15);
                const float x = acc[a][c][v];
                const __bf16 xh = (__bf16)x;
                H[rr * LPB + cc] = xh;
                L[rr * LPB + cc] = (__bf16)(x - (float)xh);
            }
}

// acc(i, j) += sum_q A(i, q) B(j, q) over the 64 staged q, A = Ah + Al, B = Bh + Bl
__device__ __forceinline__ void mma64_bf16(const __bf16* Ah, const __bf16* Al, const __bf16* Bh, const __bf16* Bl,
                                           float4_t (&acc)[2][2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll
    for (int ks = 0; ks < TS; ks += 32) {
        const int kq = ks + 8 * (lane >> 4);
        bf16x8_t ah[2], al[2], bh[2], bl[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int ia = (wr * 32 + t * 16 + (lane & 15)) * LPB + kq;
            const int ib = (wc * 32 + t * 16 + (lane & 15)) * LPB + kq;
            ah[t] = *(const bf16x8_t*)&Ah[ia];
            al[t] = *(const bf16x8_t*)&Al[ia];
            bh[t] = *(const bf16x8_t*)&Bh[ib];
            bl[t] = *(const bf16x8_t*)&Bl[ib];
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], bh[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a], bl[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[a], bh[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[a], bl[c], acc[a][c], 0, 0, 0);
            }
    }
}

// The FP32 diagonal block factored by the four waves of a workgroup (one wave per 16-column panel;
// the earlier one-wave form held 256 registers and its 64 column steps ran serially): lane r of wave
// w holds a[j] = A(r, 16 w + j).  d = |p| rsqrt|p| and l = a rsqrt|p| for the pivot p.  Column c: its pivot is lane c's entry (readlane), the
// column goes to Lt[c] (Lt[c][i] = L(i, c)) and 1/sqrt of the pivot to Rd[c], and every entry right
// of c takes the rank-1 update.  L^-1 by the right-looking substitution, lane r of wave w holding
// rows 16 w .. 16 w + 15 of column r (row q scaled by Rd[q], published in X[q], then the rows below
// updated).  Both blocked by 16-column (row) panels, one per wave, one barrier per panel: wave p
// does its own panel's steps, the waves after it then apply the panel's 16 updates in order.  Writes
// L's lower triangle into the block (row pitch ld), the pivots and W.  LDS: Lt and X 64 x 64 each,
// Rd 64.
__device__ __forceinline__ void chol_diag_f32_4w(const MatDesc& D, int kb, float* tile, int ld, float (&a)[16],
                                                 float (*Lt)[TS], float (*X)[TS], float* Rd)
{
    typedef float T;
    const int r = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long base = (long long)kb * TS;
    bool bad = false;
    // factor, by 16-column panels: wave p factors its own panel (its columns' pivots, the columns into
    // Lt, the rank-1 updates of its later columns), then the waves right of it apply the panel's 16
    // updates in column order: each element sees the updates of columns 0, 1, ... in turn
#pragma unroll
    for (int p = 0; p < 4; p++) {
        if (w == p) {
#pragma unroll
            for (int cc = 0; cc < 16; cc++) {
                const int c = 16 * p + cc;
                const T piv = lane_bcast(a[cc], c);
                bad |= (!(piv > 0) && base + c < D.n);  // negative, zero or NaN pivot
                const T pa = fabs(piv);
                const T rd = rsqrtf(pa);
                const T d = (pa > 0) ? pa * rd : (T)0;
                const T l = (r > c) ? a[cc] * rd : d;
                a[cc] = l;
                Lt[c][r] = l;
                if (r == c) Rd[c] = rd;
                wave_lds_sync();
#pragma unroll
                for (int j = cc + 1; j < 16; j++) a[j] = fma(-l, Lt[c][16 * p + j], a[j]);
            }
        }
        __syncthreads();
        if (w > p) {
#pragma unroll
            for (int cc = 0; cc < 16; cc++) {
                const int c = 16 * p + cc;
                const T l = Lt[c][r];
#pragma unroll
                for (int j = 0; j < 16; j++) a[j] = fma(-l, Lt[c][16 * w + j], a[j]);
            }
        }
    }
    if (r == 0 && bad) atomicOr(D.status, 1);  // bad is uniform in a wave (the pivots are broadcast)
    // row r of the lower triangle
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
        const int q = 16 * w + j;
        T* dst = tile + (size_t)r * ld + q;
        if (q + 3 <= r) {
            *(float4*)dst = make_float4(a[j], a[j + 1], a[j + 2], a[j + 3]);
        } else if (q <= r) {
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (q + u <= r) dst[u] = a[j + u];
        }
    }
    if (w == 0) ((T*)D.diag)[base + r] = Lt[r][r];
    // L^-1 by 16-row panels in the same way: wave p finalizes its rows (scale by 1/L(q, q), then the
    // updates of its later rows), publishes them in X, and the waves below apply them in row order
    T x[16];
#pragma unroll
    for (int j = 0; j < 16; j++) x[j] = (16 * w + j == r) ? (T)1 : (T)0;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        if (w == p) {
#pragma unroll
            for (int qq = 0; qq < 16; qq++) {
                const int q = 16 * p + qq;
                x[qq] *= Rd[q];
                X[q][r] = x[qq];
#pragma unroll
                for (int j = qq + 1; j < 16; j++) x[j] = fma(-Lt[q][16 * p + j], x[qq], x[j]);
            }
        }
        __syncthreads();
        if (w > p) {
#pragma unroll
            for (int qq = 0; qq < 16; qq++) {
                const int q = 16 * p + qq;
                const T xq = X[q][r];
#pragma unroll
                for (int j = 0; j < 16; j++) x[j] = fma(-Lt[q][16 * w + j], xq, x[j]);
            }
        }
    }
    T* W = (T*)D.W + (size_t)kb * TS * TS;
#pragma unroll
    for (int j = 0; j < 16; j++) W[(16 * w + j) * TS + r] = x[j];
}

// 1 / sqrt(p) of a positive FP64 p: the hardware estimate (about 2^-23) and one third-order step
// (r e (1/2 + 3/8 e) with e = 1 - p r^2 leaves an error of order e^3, below the last place)
__device__ __forceinline__ double rsqrt_f64(double p)
{
    const double r = __builtin_amdgcn_rsq(p);
    const double e = fma(-(p * r), r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
// a / d for r = 1 / d to within an ulp: one correction from the exact remainder
__device__ __forceinline__ double div_r(double a, double d, double r)
{
    const double q = a * r;
    return fma(fma(-q, d, a), r, q);
}

// 1 / p of an FP64 p > 0 likewise (e = 1 - p r, r (1 + e + e^2))
__device__ __forceinline__ double rcp_f64(double p)
{
    const double r = __builtin_amdgcn_rcp(p);
    const double e = fma(-p, r, 1.0);
    return fma(r * e, 1.0 + e, r);
}

// lane C of each 16-lane row in all of the row's lanes
template <int C>
__device__ __forceinline__ double row_bcast_f64(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x150 + C, 0xf, 0xf, false);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x150 + C, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// x (row m of four columns of the identity) through the elimination's steps c = 0 .. 14
template <int... C>
__device__ __forceinline__ void z_steps(double (&x)[4], const double (&mc)[15], std::integer_sequence<int, C...>)
{
    auto step = [&](auto c) {
        constexpr int cc = decltype(c)::value;
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = fma(-mc[cc], row_bcast_f64<cc>(x[j]), x[j]);
    };
    (step(std::integral_constant<int, C>()), ...);
}

// The FP64 diagonal block and its inverse by four waves, in 16 x 16 blocks.  It is the serial chain of
// every FP64 factorization, so it is arranged for latency (34 us a launch on one
// matrix as rank-1 updates with a square root and a division a column, now 16):
//   * wave t factors panel t (columns 16 t .. 16 t + 15), one row per lane, without square roots
//     (A = M P M^T, M unit lower): a column's chain is its pivot's reciprocal, one product and the next
//     pivot's update, with the next two columns' entries broadcast by readlane; the other columns take
//     theirs from LDS a column later, and the sixteen 1 / sqrt(p) are formed at once afterwards;
//   * the waves after t then update their panels' blocks with v_mfma_f64_16x16x4f64 (operands M |P| and
//     M), held in the accumulator layout until their turn;
//   * wave j owns column block j of M^-1: Z_jj by eliminating the identity while wave j + 1 factors,
//     then Z_ij = -Z_ii sum_k M_ik Z_kj on MFMA as the Z_ii appear (an accumulator is a B operand as it
//     lies); L^-1 = P^-1/2 M^-1 and L = M P^1/2 are scaled on the way out.
// Phases 0 .. 4 end with a barrier; in phase t wave t factors, wave t - 1 forms Z_(t-1)(t-1), the waves
// before finish row t - 2 and sum for row t - 1.  acc[i] holds rows 16 i .. of the wave's 16 columns
// (i >= w; the accumulator layout).  LDS: DGL doubles.
#define DGP 74                      // row pitch: rows and columns of 16 spread over the banks, pairs aligned
#define DGL (2 * TS * DGP + 2 * TS) // Mt[c][r] = M(r, c), Z by rows, the pivots, their 1 / sqrt
__device__ __forceinline__ void chol_diag_f64_4w(const MatDesc& D, int kb, double* tile, int ld, double4_t (&acc)[4], double* sm)
{
    typedef double T;
    T(*Z)[DGP] = (T(*)[DGP])sm;
    T(*Mt)[DGP] = (T(*)[DGP])(sm + TS * DGP);
    T* const Pv = sm + 2 * TS * DGP;
    T* const Rs = Pv + TS;
    const int r = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = r & 15, g = r >> 4;
    const int w16 = 16 * w;
    const long long base = (long long)kb * TS;
    T* const W = (T*)D.W + (size_t)kb * TS * TS;
    // panel t's update of the blocks i >= I0 (= w, known to the compiler: no branch between the MFMAs)
    auto update = [&](int t, auto I0) {
        constexpr int i0 = decltype(I0)::value;
        T b[4], av[4][4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int c = 16 * t + 4 * s + g;
            b[s] = Mt[c][w16 + m];
            const T pc = -fabs(Pv[c]);  // L L^T with sqrt|p|, as within the panel
#pragma unroll
            for (int i = i0; i < 4; i++) av[s][i] = Mt[c][16 * i + m] * pc;
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = i0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s][i], b[s], acc[i], 0, 0, 0);
    };
#pragma unroll 1
    for (int t = 0; t < w; t++) {
        __syncthreads();
        if (w == 1) update(t, std::integral_constant<int, 1>());
        else if (w == 2) update(t, std::integral_constant<int, 2>());
        else update(t, std::integral_constant<int, 3>());
    }
    // ---- phase w: the panel, one row per lane ----
    T a[16];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) Mt[w16 + m][16 * i + 4 * v + g] = i >= w ? acc[i][v] : (T)0;
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < 16; j++) a[j] = Mt[w16 + j][r];
    wave_lds_sync();
    {
        T p = readlane_f64(a[0], w16);
        T ap = (T)0, myp = (T)1;  // the previous column; the lane's own pivot
        double2_t vp[8];          // its multipliers of columns >= c + 2, still to be applied
        int mo;                   // &Mt[w16][w16] in a vector register: every broadcast read is an immediate offset away
        asm("v_mov_b32 %0, %1" : "=v"(mo) : "s"((TS + w16) * DGP + w16));
#pragma unroll
        for (int c = 0; c < 16; c++) {
            const T rp = rcp_f64(fabs(p));
            myp = (r == w16 + c) ? a[c] : myp;
            const T v = a[c] * rp;
            Mt[w16 + c][r] = v;
            if (c < 15) {
                a[c + 1] = fma(-a[c], readlane_f64(v, w16 + c + 1), a[c + 1]);
                p = readlane_f64(a[c + 1], w16 + c + 1);
            }
            if (c < 14) a[c + 2] = fma(-a[c], readlane_f64(v, w16 + c + 2), a[c + 2]);
#pragma unroll
            for (int j = c + 2; j < 16; j++)
                if (c > 0) a[j] = fma(-ap, vp[j >> 1][j & 1], a[j]);
            wave_lds_sync();
#pragma unroll
            for (int j = (c + 3) / 2; j < 8; j++) vp[j] = *(const double2_t*)&sm[mo + c * DGP + 2 * j];
            ap = a[c];
        }
        if (g == w) Pv[r] = myp;
    }
    __syncthreads();
    // ---- phase w + 1: Z_ww by the same elimination of the identity ----
    const T pv = Pv[w16 + m];  // pivot of the lane's row within the block, its square root and inverse
    const T pa = fabs(pv);
    const T rs = rsqrt_f64(pa);
    T dg = pa * rs;
    dg = fma(fma(-dg, dg, pa), 0.5 * rs, dg);
    const bool own = g == w;  // lanes of the panel's own rows
    {
        // lane (m, g): row m, columns 4 g .. 4 g + 3; row c's entries come from lane c of the 16-lane row
        T x[4], mc[15];
#pragma unroll
        for (int j = 0; j < 4; j++) x[j] = (m == 4 * g + j) ? (T)1 : (T)0;
#pragma unroll
        for (int c = 0; c < 15; c++) mc[c] = m > c ? Mt[w16 + c][w16 + m] : (T)0;
        z_steps(x, mc, std::make_integer_sequence<int, 15>());
        if (g == 0) Rs[w16 + m] = rs;
#pragma unroll
        for (int j = 0; j < 4; j++) Z[w16 + m][w16 + 4 * g + j] = x[j];
#pragma unroll
        for (int j = 0; j < 4; j += 2)
            *(double2_t*)&W[(w16 + m) * TS + w16 + 4 * g + j] = (double2_t){x[j] * rs, x[j + 1] * rs};
    }
    // L's panel (M P^1/2 below the diagonal) and what lies above it in L^-1
    auto finish = [&]() {
#pragma unroll
        for (int c = 0; c < 16; c++) a[c] = (r == w16 + c) ? dg : div_r(a[c], readlane_f64(dg, c), readlane_f64(rs, c));
#pragma unroll
        for (int j = 0; j < 16; j += 2) {
            const int q = w16 + j;
            T* dst = tile + (size_t)r * ld + q;
            if (q + 1 <= r) {
                *(double2_t*)dst = (double2_t){a[j], a[j + 1]};
            } else if (q <= r) {
                dst[0] = a[j];
            }
        }
        if (g < w) {
#pragma unroll
            for (int j = 0; j < 16; j += 2) *(double2_t*)&W[r * TS + w16 + j] = (double2_t){0, 0};
        }
        if (own) {
            ((T*)D.diag)[base + r] = dg;
            if (!(pv > 0) && base + r < D.n) atomicOr(D.status, 1);  // negative, zero or NaN pivot
        }
    };
    // ---- phases w + 2 .. 5: the sum of row t - 1, and row t - 2 of the sum formed a phase earlier ----
    double4_t S = {0, 0, 0, 0};
#pragma unroll 1
    for (int t = w + 1; t <= 5; t++) {
        if (t - 2 > w) {  // Z_iw = -Z_ii S, i = t - 2
            const int i = t - 2;
            double4_t o = {0, 0, 0, 0};
            T av[4];
#pragma unroll
            for (int s = 0; s < 4; s++) av[s] = -Z[16 * i + m][16 * i + 4 * s + g];
#pragma unroll
            for (int s = 0; s < 4; s++) o = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], S[s], o, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                Z[16 * i + 4 * v + g][w16 + m] = o[v];
                W[(16 * i + 4 * v + g) * TS + w16 + m] = o[v] * Rs[16 * i + 4 * v + g];
            }
            wave_lds_sync();
        }
        if (t - 1 > w && t <= 4) {  // S_iw = sum_(k = w)^(i - 1) M_ik Z_kw, i = t - 1
            const int i = t - 1;
            S = (double4_t){0, 0, 0, 0};
#pragma unroll 1
            for (int k = w; k < i; k++) {
                T av[4], bv[4];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    av[s] = Mt[16 * k + 4 * s + g][16 * i + m];
                    bv[s] = Z[16 * k + 4 * s + g][w16 + m];
                }
#pragma unroll
                for (int s = 0; s < 4; s++) S = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s], S, 0, 0, 0);
            }
        }
        if (t == w + 2) finish();  // (the last wave's comes in phase 5)
        if (t < 5) __syncthreads();
    }
}

// one diagonal block per matrix (blockIdx.y), four waves; FP32 blocks of the first column read F as
// formed (A0), when the matrix has it
template <typename T>
__global__ void __launch_bounds__(256) k_chol_diag4_m(const MatDesc* mats, int kb)
{
    const MatDesc D = mats[blockIdx.y];
    if (kb >= D.nb) return;
    int ld;
    T* tile = tile_ptr<T>(D, kb, kb, ld);
    const T* src = (sizeof(T) == 4 && kb == 0 && D.A0) ? (const T*)D.A0 + (tile - (T*)D.A) : tile;
    const int r = threadIdx.x & 63, w = threadIdx.x >> 6;
    if constexpr (sizeof(T) == 8) {
        __shared__ __align__(16) double sm[DGL];
        double4_t acc[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[i][v] = i >= w ? src[(size_t)(16 * i + 4 * v + (r >> 4)) * ld + 16 * w + (r & 15)] : 0.0;
        chol_diag_f64_4w(D, kb, tile, ld, acc, sm);
    } else {
        __shared__ __align__(16) float Lt[TS][TS];
        __shared__ float X[TS][TS];
        __shared__ float Rd[TS];
        float a[16];
#pragma unroll
        for (int j = 0; j < 16; j += 4) {
            const float4_t v = *(const float4_t*)&src[(size_t)r * ld + 16 * w + j];
            a[j] = v.x;
            a[j + 1] = v.y;
            a[j + 2] = v.z;
            a[j + 3] = v.w;
        }
        chol_diag_f32_4w(D, kb, tile, ld, a, Lt, X, Rd);
    }
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) k_chol_lpanel_bf16(const MatDesc* mats, int kb, int k0, int kend)
{
    __shared__ __attribute__((aligned(16))) __bf16 sm[4 * TS * LPB];
    __bf16* const Ah = sm;
    __bf16* const Al = sm + TS * LPB;
    __bf16* const Bh = sm + 2 * TS * LPB;
    __bf16* const Bl = sm + 3 * TS * LPB;
    typedef float T;
    // grid (matrices, row blocks): the workgroups of the first row block, which also factor the next
    // diagonal block, are dispatched first
    const MatDesc D = mats[blockIdx.x];
    if (kb >= D.nb) return;
    const int ib = kb + 1 + blockIdx.y;
    if (ib > band_last(D, kb)) return;
    int ld, lp;
    T* blk = tile_ptr<T>(D, ib, kb, ld);
    const bool first = (k0 == 0 && D.A0);
    // operand blocks are loaded into registers one step ahead of their use (the first with the C
    // block, W_kb during the last step), so their latency overlaps the barriers and products
    T cv[16];
    load64c<T>(first ? (const T*)D.A0 + (blk - (T*)D.A) : blk, ld, cv);
    f32x4_t ra[4], rb[4];
    const T* const Wkb = (const T*)D.W + (size_t)kb * TS * TS;
    if (k0 < kb) {
        load64_regs(tile_ptr<T>(D, ib, k0, lp), lp, ra);
        load64_regs(tile_ptr<T>(D, kb, k0, lp), lp, rb);
    } else {
        load64_regs(Wkb, TS, ra);
    }
    float4_t acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c] = (float4_t){0, 0, 0, 0};
    for (int kp = k0; kp < kb; kp++) {
        __syncthreads();
        split64_store(ra, Ah, Al);
        split64_store(rb, Bh, Bl);
        __syncthreads();
        if (kp + 1 < kb) {
            load64_regs(tile_ptr<T>(D, ib, kp + 1, lp), lp, ra);
            load64_regs(tile_ptr<T>(D, kb, kp + 1, lp), lp, rb);
        } else {
            load64_regs(Wkb, TS, ra);
        }
        mma64_bf16(Ah, Al, Bh, Bl, acc);
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[a][c][v] = cv[(a * 2 + c) * 4 + v] - acc[a][c][v];
    __syncthreads();
    acc64_split(acc, Ah, Al);
    split64_store(ra, Bh, Bl);  // W_kb
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c] = (float4_t){0, 0, 0, 0};
    mma64_bf16(Ah, Al, Bh, Bl, acc);  // L_ib,kb(i, j) = sum_q A'(i, q) W_kb(j, q)
    store64<T>(blk, ld, acc);
    if (ib != kb + 1 || ib >= kend) return;
    T* dg = tile_ptr<T>(D, ib, ib, ld);
    load64c<T>(first ? (const T*)D.A0 + (dg - (T*)D.A) : dg, ld, cv);
    if (k0 < kb) load64_regs(tile_ptr<T>(D, ib, k0, lp), lp, ra);
    __syncthreads();
    acc64_split(acc, Ah, Al);
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c] = (float4_t){0, 0, 0, 0};
    mma64_bf16(Ah, Al, Ah, Al, acc);
    for (int kp = k0; kp < kb; kp++) {
        __syncthreads();
        split64_store(ra, Ah, Al);
        __syncthreads();
        if (kp + 1 < kb) load64_regs(tile_ptr<T>(D, ib, kp + 1, lp), lp, ra);
        mma64_bf16(Ah, Al, Ah, Al, acc);
    }
    // the block, now up to date, is factored here, so the next column step needs no diagonal
    // launch: through LDS (S, 64 x 65, over the operand tiles) into rows per lane
    float* S = (float*)sm;
    float(*Lt)[TS] = (float(*)[TS])((float*)sm + TS * 65);
    float* Rd = (float*)sm + TS * 65 + TS * TS;
    {
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        const int wr = w >> 1, wc = w & 1;
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int rr = wr * 32 + a * 16 + 4 * (lane >> 4) + v;
                    const int cc = wc * 32 + c * 16 + (lane & 15);
                    S[rr * 65 + cc] = cv[(a * 2 + c) * 4 + v] - acc[a][c][v];
                }
        __syncthreads();
        float av[16];
#pragma unroll
        for (int j = 0; j < 16; j++) av[j] = S[lane * 65 + 16 * w + j];
        chol_diag_f32_4w(D, ib, dg, ld, av, Lt, (float(*)[TS])S, Rd);  // X over S: read before the first barrier
    }
}

// acc += A B^T over nst stages of 16 k, 64 rows of A and of B: wave (wr, wc) of four holds 32 rows of each
// as 2 x 2 accumulators.  Rows lie lda (ldb) apart; 64-column block q of a row starts q * ba
// (bb) after the first (64 in a dense matrix, -4096 along a banded row).  Operands go through two LDS
// buffers, one barrier a stage, loaded a stage ahead; rows 144 bytes apart put the 16 rows of an operand
// read on distinct 16-byte slots.
#define TFP 18
__device__ __forceinline__ void gemm_f64(const double* A, size_t lda, long long ba, const double* B, size_t ldb, long long bb, int nst,
                                         double* lds, double4_t (&acc)[2][2])
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wr = w >> 1, wc = w & 1;
    // piece h of a thread: row (tid >> 3) + 32 h, columns 2 (tid & 7) and the next of the stage
    const double* const pA = A + (tid >> 3) * lda + 2 * (tid & 7);
    const double* const pB = B + (tid >> 3) * ldb + 2 * (tid & 7);
    double* const st0 = lds + (tid >> 3) * TFP + 2 * (tid & 7);
    const double* const a0 = lds + (wr * 32 + (lane & 15)) * TFP + 2 * (lane >> 4);
    const double* const b0 = lds + (TS + wc * 32 + (lane & 15)) * TFP + 2 * (lane >> 4);
    double2_t ra[2], rb[2];
    auto load = [&](int st) {
        const long long oa = (st >> 2) * ba + (st & 3) * 16, ob = (st >> 2) * bb + (st & 3) * 16;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ra[h] = *(const double2_t*)(pA + (size_t)(32 * h) * lda + oa);
            rb[h] = *(const double2_t*)(pB + (size_t)(32 * h) * ldb + ob);
        }
    };
    auto stage = [&](int buf) {
        double* const d = st0 + buf * 2 * TS * TFP;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            *(double2_t*)(d + 32 * h * TFP) = ra[h];
            *(double2_t*)(d + (TS + 32 * h) * TFP) = rb[h];
        }
    };
    load(0);
    stage(0);
    for (int st = 0; st < nst; st++) {
        __syncthreads();  // stage st is in its buffer, and the other buffer's readers are done
        if (st + 1 < nst) load(st + 1);
        const double* const as = a0 + (st & 1) * 2 * TS * TFP;
        const double* const bs = b0 + (st & 1) * 2 * TS * TFP;
#pragma unroll
        for (int kk = 0; kk < 16; kk += 8) {
            double2_t av[2], bv[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                av[t] = *(const double2_t*)(as + t * 16 * TFP + kk);
                bv[t] = *(const double2_t*)(bs + t * 16 * TFP + kk);
            }
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int c = 0; c < 2; c++) acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a].x, bv[c].x, acc[a][c], 0, 0, 0);
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int c = 0; c < 2; c++) acc[a][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a].y, bv[c].y, acc[a][c], 0, 0, 0);
        }
        if (st + 1 < nst) stage((st + 1) & 1);
    }
}
// the accumulators of a tile at C (row pitch ldc): -C read, -acc written (its lower triangle only)
__device__ __forceinline__ void load_neg(const double* C, size_t ldc, double4_t (&acc)[2][2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double* const c0 = C + ((w >> 1) * 32 + (lane >> 4)) * ldc + (w & 1) * 32 + (lane & 15);
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[a][c][v] = -c0[(a * 16 + 4 * v) * ldc + c * 16];
}
__device__ __forceinline__ void store_neg(double* C, size_t ldc, const double4_t (&acc)[2][2], bool lower)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r0 = (w >> 1) * 32 + (lane >> 4), q0 = (w & 1) * 32 + (lane & 15);
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (!lower || q0 + c * 16 <= r0 + a * 16 + 4 * v) C[(r0 + a * 16 + 4 * v) * ldc + q0 + c * 16] = -acc[a][c][v];
}
// the diagonal block in sm's first 64 rows of DGP into the blocks of 16 columns, factored
__device__ __forceinline__ void chol_diag_f64_lds(const MatDesc& D, int kb, double* tile, int ld, double* sm)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    double4_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[i][v] = i >= w ? sm[(16 * i + 4 * v + (lane >> 4)) * DGP + 16 * w + (lane & 15)] : 0.0;
    chol_diag_f64_4w(D, kb, tile, ld, acc, sm);
}

// Left-looking FP64 panel step: column block kb of the part that starts at k0, dense or banded (there
// every earlier block of the row inside the band, so a banded factorization is one launch per column
// block).  Workgroup y takes row block ib = kb + 1 + y and forms
// L_ib,kb = (A_ib,kb - sum_k' L_ib,k' L_kb,k'^T) W_kb^T; the part's diagonal blocks (in a band, every
// one of the launch) take this column's product at once, and the workgroup of ib = kb + 1 factors the
// next one, so a column needs this one launch instead of a diagonal, a panel and a panel-update one.
// Alone, a step is bound by that workgroup's serial chain (its 64^3 products at 1.7 us each on one CU,
// then the diagonal block); the grid is (matrices, row blocks), so it is dispatched first.
// One 3712 matrix alone: 4.3 -> 2.15 ms for the factorization, R's banded chain of 58 steps 3.0 -> 1.6.
__global__ void __launch_bounds__(256) k_chol_lpanel_f64(const MatDesc* mats, int kb, int k0, int kend)
{
    __shared__ __attribute__((aligned(16))) double sm[DGL];  // stages, operand tiles, the diagonal block's buffers
    static_assert(2 * 2 * 64 * TFP <= DGL && 2 * TS * LDT <= DGL, "the stages and the operand tiles fit");
    double(*As)[LDT] = (double(*)[LDT])sm;
    double(*Bs)[LDT] = (double(*)[LDT])(sm + TS * LDT);
    const MatDesc D = mats[blockIdx.x];
    if (kb >= D.nb) return;
    const int ib = kb + 1 + blockIdx.y;
    if (ib > band_last(D, kb)) return;
    const int ks = D.bwb > 0 ? max(0, ib - D.bwb) : k0;
    int ld, lp;
    double* blk = tile_ptr<double>(D, ib, kb, ld);
    double4_t acc[2][2];
    load_neg(blk, ld, acc);
    if (ks < kb) {
        const long long bs = D.bwb > 0 ? -TS * TS : TS;
        const double* Pa = tile_ptr<double>(D, ib, ks, lp);
        gemm_f64(Pa, lp, bs, tile_ptr<double>(D, kb, ks, lp), lp, bs, 4 * (kb - ks), sm, acc);
        __syncthreads();
    }
    stage64<double>((const double*)D.W + (size_t)kb * TS * TS, TS, Bs);
    store_neg(&As[0][0], LDT, acc, false);
    const bool upd = D.bwb > 0 || ib < kend;
    double* dg = tile_ptr<double>(D, ib, ib, lp);
    const int ldd = lp;
    double4_t dacc[2][2];
    if (upd) load_neg(dg, ldd, dacc);
    __syncthreads();
    mma64<double>(As, Bs, acc);  // L_ib,kb(i, j) = sum_q A'(i, q) W_kb(j, q)
    store64<double>(blk, ld, acc);
    if (!upd) return;
    __syncthreads();
    store64<double>(&As[0][0], LDT, acc);
    __syncthreads();
    mma64_add<double>(As, As, dacc);
    if (ib != kb + 1) {
        store_neg(dg, ldd, dacc, true);
        return;
    }
    __syncthreads();
    store_neg(sm, DGP, dacc, false);
    chol_diag_f64_lds(D, ib, dg, ldd, sm);
}

// FP64 trailing update C(I, J) -= sum over the panel's nq column blocks of L(I, q) L(J, q)^T on the
// 64-tiles of rows and columns >= k0 + nq; ncolt > 0: the first ncolt tile columns only, a strip.  The
// accumulators start from -C and are stored negated, so each element takes its products in k order
// whatever the panel's width.  Two LDS stages of 37 KB leave four workgroups a CU, so
// that some multiply while others wait for their C tiles or store them: 52 TFLOP/s on 100 matrices of
// 3712 (the 128-tile form with one workgroup of 139 KB a CU, whose C traffic stood beside the products:
// 32; 128-tiles on the same two stages, two workgroups a CU: 50, and slower by 0.5 ms on one matrix).
// fdiag (the diagonal block's buffers: two workgroups a CU) factors block k0 + nq in tile (0, 0)'s
// workgroup; it saves the diagonal launch and its wait where the tiles do not fill those two anyway
// (TRAIL_FUSED; 100 matrices of 3712: 38.5 ms fused, 34.9 apart; one: 2.15 against 2.23).
#define TRAIL_F64_LDS (DGL * 8)
#define TRAIL_F64_LDS0 (2 * 2 * 64 * TFP * 8)
#define TRAIL_FUSED 512
__global__ void __launch_bounds__(256) k_chol_trail_f64(const MatDesc* mats, int k0, int nq, int ncolt, int fdiag)
{
    extern __shared__ double trail_raw[];
    const MatDesc D = mats[blockIdx.y];
    const int r0b = k0 + nq;
    if (r0b >= D.nb) return;
    const int nt = D.nb - r0b;
    int I = -1, J = -1;
    if (ncolt == 0) {
        if (!syrk_tile(nt, I, J)) return;
    } else {
        int t = blockIdx.x;
        for (int j = 0; j < ncolt && j < nt; j++) {
            if (t < nt - j) {
                J = j;
                I = j + t;
                break;
            }
            t -= nt - j;
        }
        if (J < 0) return;
    }
    const size_t ld = D.ld;
    double* const A = (double*)D.A;
    const size_t rI = (size_t)(r0b + I) * TS, rJ = (size_t)(r0b + J) * TS;
    double4_t acc[2][2];
    load_neg(A + rI * ld + rJ, ld, acc);
    gemm_f64(A + rI * ld + (size_t)k0 * TS, ld, TS, A + rJ * ld + (size_t)k0 * TS, ld, TS, 4 * nq, trail_raw, acc);
    store_neg(A + rI * ld + rJ, ld, acc, I == J);
    // fdiag: the workgroup of tile (0, 0) also factors diagonal block r0b, now up to date, so the part
    // that starts there needs no diagonal launch
    if (fdiag && I == 0 && J == 0) {
        __syncthreads();
        store_neg(trail_raw, DGP, acc, false);
        chol_diag_f64_lds(D, r0b, A + rI * ld + rJ, (int)ld, trail_raw);
    }
}

// Dense matrices (padded to a multiple of 128), panel by panel of panel_blocks 64-blocks: each panel
// in 256-wide left-looking parts, each part after the first brought up to date by a strip update from
// the earlier parts, then one trailing update of the rest.  Only the first diagonal block has a launch
// of its own: the others are factored by the panel step or the update before them.  FP32 (the mixed
// path): per batch of 256 3600 x 3600 matrices the factorization took 33.7 ms with a rank-256 update
// per 256 columns, 30.0 ms with 512-wide panels and 29.4 ms with 1024-wide ones (2048: 29.1, one panel:
// 30.1; FP32 MFMA in the panel kernel then).  FP64: 1024-wide panels where there are many matrices (100
// of 3712: 36.7 ms with 1024, 37.8 with 512, 40.1 with 256, which reads and writes the trailing matrix four
// times as often), 256-wide ones for few (one of 3712: 2.15, 2.21 and 2.31 ms with 256, 512 and 1024: the
// strips are launches on the serial chain).  The line counts the trailing tiles, so that one large matrix is on
// the wide side; 256 against 1024: one of 8192 7.55 / 7.53 ms, one of 10 112 11.34 / 11.29, four of these 29.8 /
// 28.4, eight of 3712 4.38 / 4.35, 32 of them 12.3 / 11.7.  (Right-looking panels: 100 of 3712 60.9 ms, one
// 4.3.)  The schedule's arithmetic does not depend on the panel's width or on the batch, so an item's
// factor is the same bits alone and in any.
#define CHOL_WIDE 16384  // matrices x blocks^2 from which FP64 panels are wide
#define QLX_CHOL_SUB 4  // 256-wide left-looking parts per panel by default
template <typename T>
static void chol_two_level(hipStream_t s, const MatDesc* mats, int nmat, int max_nb, int panel_blocks)
{
    constexpr bool F32 = sizeof(T) == 4;
    const size_t lds = (size_t)4 * TT * TBP * sizeof(uint16_t);
    allow_big_lds(F32 ? (const void*)k_chol_trail_bf16 : (const void*)k_chol_trail_f64);
    // the update of everything from block k0 + nq on, or (strip) of the first 256 columns there
    auto trail = [&](int k0, int nq, bool strip) {
        const int n = max_nb - k0 - nq, nt = n / 2;
        if (F32) {
            hipLaunchKernelGGL(k_chol_trail_bf16, dim3(strip ? 2 * nt - 1 : syrk_grid(nt), nmat), dim3(256), lds, s, mats, k0, nq, strip ? 2 : 0, 1);
        } else {
            const int grid = strip ? (n >= 4 ? 4 * n - 6 : n * (n + 1) / 2) : (int)syrk_grid(n);
            const bool fused = (long long)(strip ? grid : n * (n + 1) / 2) * nmat <= TRAIL_FUSED;
            hipLaunchKernelGGL(k_chol_trail_f64, dim3(grid, nmat), dim3(256), fused ? (size_t)TRAIL_F64_LDS : (size_t)TRAIL_F64_LDS0, s, mats,
                               k0, nq, strip ? 4 : 0, fused ? 1 : 0);
            if (!fused) hipLaunchKernelGGL(k_chol_diag4_m<T>, dim3(1, nmat), dim3(256), 0, s, mats, k0 + nq);
        }
    };
    // panel width in 64-blocks
    const int NB = panel_blocks > 0 ? panel_blocks : F32 || (long long)nmat * max_nb * max_nb >= CHOL_WIDE ? 4 * QLX_CHOL_SUB : 4;
    hipLaunchKernelGGL(k_chol_diag4_m<T>, dim3(1, nmat), dim3(256), 0, s, mats, 0);
    for (int k0 = 0; k0 < max_nb; k0 += NB) {
        for (int ks = k0; ks < k0 + NB && ks < max_nb; ks += 4) {
            if (ks > k0) trail(k0, ks - k0, true);  // the part's columns, from the panel's earlier parts
            for (int kb = ks; kb < ks + 4 && kb + 1 < max_nb; kb++) {
                const dim3 grid(nmat, max_nb - kb - 1);
                if (F32) hipLaunchKernelGGL(k_chol_lpanel_bf16, grid, dim3(256), 0, s, mats, kb, ks, ks + 4);
                else hipLaunchKernelGGL(k_chol_lpanel_f64, grid, dim3(256), 0, s, mats, kb, ks, ks + 4);
            }
        }
        if (k0 + NB >= max_nb) break;
        trail(k0, NB, false);
    }
}

// nmat matrices of one element type (f32): dense ones (all of the launch) by the two-level schedule,
// banded ones (FP64, lower band <= max_bwb blocks) by one left-looking launch per column block
void cholesky_batched(hipStream_t s, const MatDesc* d_mats, int n32, int n64, int max_nb, int dense, int max_bwb, int panel_blocks)
{
    if (dense) {
        if (n32) chol_two_level<float>(s, d_mats, n32, max_nb, panel_blocks);
        if (n64) chol_two_level<double>(s, d_mats + n32, n64, max_nb, 0);
        return;
    }
    if (!n64) return;
    hipLaunchKernelGGL(k_chol_diag4_m<double>, dim3(1, n64), dim3(256), 0, s, d_mats + n32, 0);
    for (int kb = 0; kb + 1 < max_nb; kb++)
        hipLaunchKernelGGL(k_chol_lpanel_f64, dim3(n64, std::min(max_nb - kb - 1, max_bwb)), dim3(256), 0, s, d_mats + n32, kb, 0, max_nb);
}

// 2 sum log(diag) in a fixed order (Cholesky_logdet_lower_packed, pixelgrid.cpp:17201-17210)
template <typename T>
__device__ double block_sum_log(const T* diag, int n, double* sh)
{
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += log(fabs((double)diag[i]));
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    double r = 2.0 * sh[0];
    __syncthreads();
    return r;
}

template <typename T>
__global__ void __launch_bounds__(256) k_logdets_b(BatchDev bd)
{
    __shared__ double sh[256];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const double* v = bd.vec + M.vec_off;
    const T* diagF = (const T*)(v + M.ldN);
    // R's pivots: those of the item whose factorization serves this one (the same R)
    const int rr = bd.rrep[item];
    const double* diagR = bd.vec + bd.meta[rr].vec_off + 2 * (size_t)M.ldN;
    const double lf = block_sum_log<T>(diagF, M.n_src, sh);
    const double lr = block_sum_log<double>(diagR, M.n_src, sh);
    if (threadIdx.x == 0) {
        bd.out[QLX_OUT_STRIDE * item + 2] = lf;
        bd.out[QLX_OUT_STRIDE * item + 3] = lr;
        if (rr != item) bd.status[4 * item + 1] = bd.status[4 * rr + 1];
    }
}

void launch_logdets_b(hipStream_t s, const BatchDev& bd, int f32)
{
    if (f32) hipLaunchKernelGGL(k_logdets_b<float>, dim3(1, bd.B), dim3(256), 0, s, bd);
    else hipLaunchKernelGGL(k_logdets_b<double>, dim3(1, bd.B), dim3(256), 0, s, bd);
}

// ------------------------------------------------------------------------------------------------
// Triangular solves with the stored block inverses.
// y = L^-1 D is row n of the augmented factor, so the first solve is backward only: x = L^-T y.
// ------------------------------------------------------------------------------------------------
// Each block step: a strip product over the solved part of the vector (16 B loads, eight in flight
// per lane), then the 64x64 block inverse applied by all 1024 threads, 16 lanes per output.
template <typename T>
__device__ __forceinline__ T sum16(T v)
{
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 4, 64);
    v += __shfl_xor(v, 8, 64);
    return v;
}

// forward: x_kb = W_kb (b_kb - L[kb, 0:kb] x_{0:kb}); wave w owns rows w, w+16, w+32, w+48 of the block
template <typename T>
__device__ void tri_fwd(const T* L, int ld, int nb, const T* W, T* sx, T* rhs)
{
    constexpr int VW = 16 / sizeof(T);
    typedef T P __attribute__((ext_vector_type(VW)));
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int orow = tid >> 4, oq = 4 * (tid & 15);
    for (int kb = 0; kb < nb; kb++) {
        const int r0 = kb * TS;
        T wv[4];
        {
            const T* Wr = W + (size_t)kb * TS * TS + orow * TS + oq;
            P a = *(const P*)Wr;
            if constexpr (VW == 4) {
                wv[0] = a.x; wv[1] = a.y; wv[2] = a.z; wv[3] = a.w;
            } else {
                const P b = *(const P*)(Wr + 2);
                wv[0] = a.x; wv[1] = a.y; wv[2] = b.x; wv[3] = b.y;
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (oq + j > orow) wv[j] = (T)0;
        }
        const T* L0 = L + (size_t)(r0 + w) * ld;
        const size_t s16 = (size_t)16 * ld;
        P acc[4];
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] = (P)0;
        int c = VW * lane;
        for (; c + 64 * VW < r0; c += 128 * VW) {
            P v[8];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                v[q] = *(const P*)(L0 + q * s16 + c);
                v[4 + q] = *(const P*)(L0 + q * s16 + c + 64 * VW);
            }
            const P sa = *(const P*)(sx + c), sb = *(const P*)(sx + c + 64 * VW);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[q] = __builtin_elementwise_fma(v[4 + q], sb, __builtin_elementwise_fma(v[q], sa, acc[q]));
        }
        if (c < r0) {
            const P sa = *(const P*)(sx + c);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[q] = __builtin_elementwise_fma(*(const P*)(L0 + q * s16 + c), sa, acc[q]);
        }
        T a[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            a[q] = acc[q].x + acc[q].y;
            if constexpr (VW == 4) a[q] += acc[q].z + acc[q].w;
        }
        // 4 row sums over 64 lanes: halve the set twice, then a 16-lane sum
        const bool h5 = lane & 32, h4 = lane & 16;
        const T k0 = (h5 ? a[2] : a[0]) + __shfl_xor(h5 ? a[0] : a[2], 32, 64);
        const T k1 = (h5 ? a[3] : a[1]) + __shfl_xor(h5 ? a[1] : a[3], 32, 64);
        const T k = sum16<T>((h4 ? k1 : k0) + __shfl_xor(h4 ? k0 : k1, 16, 64));
        if ((lane & 15) == 0) {
            const int r = w + 16 * (lane >> 4);
            rhs[r] = sx[r0 + r] - k;
        }
        __syncthreads();
        T y = wv[0] * rhs[oq];
#pragma unroll
        for (int j = 1; j < 4; j++) y = fma(wv[j], rhs[oq + j], y);
        y = sum16<T>(y);
        if ((tid & 15) == 0) sx[r0 + orow] = y;
        __syncthreads();
    }
}

// backward: x_kb = W_kb^T (b_kb - L[kb+1:, kb]^T x_{kb+1:}); lanes cover the block's 64 columns with
// 16 B loads, the rest of the wave and the 16 waves split the rows
template <typename T>
__device__ void tri_bwd(const T* L, int ld, int nb, const T* W, T* sx, T (*part)[TS + 1], T* rhs)
{
    constexpr int VW = 16 / sizeof(T);
    constexpr int LPR = TS / VW;   // lanes per row
    constexpr int RPW = 64 / LPR;  // rows per wave per pass
    constexpr int RPP = 16 * RPW;  // rows per pass over the workgroup
    typedef T P __attribute__((ext_vector_type(VW)));
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int ocol = tid >> 4, oq = 4 * (tid & 15);
    const int cv = VW * (lane % LPR), rsub = lane / LPR;
    const int rend = nb * TS;
    for (int kb = nb - 1; kb >= 0; kb--) {
        const int r0 = kb * TS;
        T wv[4];
        {
            const T* Wc = W + (size_t)kb * TS * TS + (size_t)oq * TS + ocol;
#pragma unroll
            for (int j = 0; j < 4; j++) wv[j] = (oq + j >= ocol) ? Wc[j * TS] : (T)0;
        }
        P acc = (P)0;
        int rr = r0 + TS + RPW * w + rsub;
        for (; rr + 7 * RPP < rend; rr += 8 * RPP) {
            P v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = *(const P*)(L + (size_t)(rr + u * RPP) * ld + r0 + cv);
#pragma unroll
            for (int u = 0; u < 8; u++) acc = __builtin_elementwise_fma(v[u], (P)sx[rr + u * RPP], acc);
        }
        for (; rr < rend; rr += RPP) acc = __builtin_elementwise_fma(*(const P*)(L + (size_t)rr * ld + r0 + cv), (P)sx[rr], acc);
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) {
            acc.x += __shfl_xor(acc.x, off, 64);
            acc.y += __shfl_xor(acc.y, off, 64);
            if constexpr (VW == 4) {
                acc.z += __shfl_xor(acc.z, off, 64);
                acc.w += __shfl_xor(acc.w, off, 64);
            }
        }
        if (rsub == 0) {
            part[w][cv] = acc.x;
            part[w][cv + 1] = acc.y;
            if constexpr (VW == 4) {
                part[w][cv + 2] = acc.z;
                part[w][cv + 3] = acc.w;
            }
        }
        __syncthreads();
        if (tid < TS) {
            T s = sx[r0 + tid];
#pragma unroll
            for (int q = 0; q < 16; q++) s -= part[q][tid];
            rhs[tid] = s;
        }
        __syncthreads();
        T y = wv[0] * rhs[oq];
#pragma unroll
        for (int j = 1; j < 4; j++) y = fma(wv[j], rhs[oq + j], y);
        y = sum16<T>(y);
        if ((tid & 15) == 0) sx[r0 + ocol] = y;
        __syncthreads();
    }
}

// Solves by panels of 256 rows: the panel's triangle (block by block, tri_bwd / tri_fwd), then its products
// off every panel still to be solved.  Two forms of the same arithmetic, so the same bits:
//   * a launch per panel (k_solve_bwd_b, k_solve_fwd_b), each panel still to be solved a workgroup, so
//     that an item's factor is read by many CUs: workgroup g of step s takes panel P -/+ g, subtracts
//     the products of the panel solved by the launch before, and workgroup 0 solves P's triangle;
//   * one workgroup per item for the whole solve (k_solve_one_b), where the items fill the GPU by
//     themselves and the launches' tails would only idle it.
// A solve reads its factor once; one workgroup gets the 55-110 GB/s of its CU, a launch per panel costs a
// chain of a triangle and a product (~20 us) each.  The stage, one workgroup -> launches: 6 items of 10 000
// mixed 12.2 -> 3.0 ms, one of 3712 mixed 1.21 -> 0.65, FP64 0.62 -> 0.31; one -> launches: 256 items of
// 3712 mixed 6.6 -> 7.9 ms, 100 FP64 1.34 -> 1.42, so these keep the one workgroup.  The line, by panels
// against one workgroup each: of 3712, 64 items mixed 2.38 against 2.84 ms, 96 3.28 / 3.45, 128 4.00 / 3.70
// (FP64 0.92 / 1.25, 1.29 / 1.35, 1.56 / 1.47); of 1024 the one workgroup is the better form at every
// count, by at most 0.05 ms (8 items mixed 0.232 / 0.222, 96 0.552 / 0.508), so the size does not enter.
// The vector stands in slot 6 of the item's vectors, in the factor's type.
#define PAN 256
#define SOLVE_ONE_B 96      // items from which one workgroup each is the better form,
// for factors up to QLX_SOLVE_ONE_LD, whose vector fits LDS beside the partial sums (107 KB of FP64)
#define SOLVE_ONE_LDS(ld) (16 * PAN + 16 * (TS + 1) + TS + (size_t)(ld))
template <typename T>
__device__ __forceinline__ T* solve_vec(const BatchDev& bd, const ItemMeta& M) { return (T*)(bd.vec + M.vec_off + 6 * (size_t)M.ldN); }

// part[w][c]: wave w's sum over its rows (w, w + 16, ..) of the panel's L(r, c) x(r); Lp = the panel's
// first row at the target panel's first column, nr rows (a multiple of 128), x their values
template <typename T>
__device__ __forceinline__ void bwd_tile(const T* Lp, int ld, int nr, const T* x, T (*part)[PAN])
{
    constexpr int VW = 16 / sizeof(T);
    typedef T P __attribute__((ext_vector_type(VW)));
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int h = 0; h < PAN; h += 64 * VW) {
        const T* Lw = Lp + (size_t)w * ld + h + VW * lane;
        P acc = (P)0;
#pragma unroll 1
        for (int k0 = 0; 16 * k0 < nr; k0 += 8) {  // eight rows in flight
            P t[8];
#pragma unroll
            for (int k = 0; k < 8; k++) t[k] = *(const P*)(Lw + (size_t)(16 * (k0 + k)) * ld);
#pragma unroll
            for (int k = 0; k < 8; k++) acc = __builtin_elementwise_fma(t[k], (P)x[w + 16 * (k0 + k)], acc);
        }
        *(P*)&part[w][h + VW * lane] = acc;
    }
}
template <typename T>
__device__ __forceinline__ T part_sum(const T (*part)[PAN], int c)
{
    T t = part[0][c];
#pragma unroll
    for (int w = 1; w < 16; w++) t += part[w][c];
    return t;
}

// row w + 16 (lane >> 2) of the target panel (nq rows, a multiple of 128): its sum of L(r, c) x(c) over the
// 256 columns of a solved panel (all four lanes of a row); Lp = its first row at that panel's first column
__device__ __forceinline__ float fwd_tile(const float* Lp, int ld, int nq, const float* x)
{
    typedef float T;
    typedef float4_t P;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const P xc = *(const P*)(x + 4 * lane);
    const T* Lw = Lp + (size_t)w * ld + 4 * lane;
    T a[16];
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 8) {
        P t[8];
        if (16 * k0 < nq)
#pragma unroll
            for (int k = 0; k < 8; k++) t[k] = *(const P*)(Lw + (size_t)(16 * (k0 + k)) * ld);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const P m = t[k] * xc;
            a[k0 + k] = 16 * k0 < nq ? (m.x + m.y) + (m.z + m.w) : 0;
        }
    }
    // 16 row sums over 64 lanes: four halvings, then a 4-lane sum
    T b[8], c[4], d[2];
    const bool h5 = lane & 32, h4 = lane & 16, h3 = lane & 8, h2 = lane & 4;
#pragma unroll
    for (int j = 0; j < 8; j++) b[j] = (h5 ? a[8 + j] : a[j]) + __shfl_xor(h5 ? a[j] : a[8 + j], 32, 64);
#pragma unroll
    for (int j = 0; j < 4; j++) c[j] = (h4 ? b[4 + j] : b[j]) + __shfl_xor(h4 ? b[j] : b[4 + j], 16, 64);
#pragma unroll
    for (int j = 0; j < 2; j++) d[j] = (h3 ? c[2 + j] : c[j]) + __shfl_xor(h3 ? c[j] : c[2 + j], 8, 64);
    T e = (h2 ? d[1] : d[0]) + __shfl_xor(h2 ? d[0] : d[1], 4, 64);
    e += __shfl_xor(e, 2, 64);
    return e + __shfl_xor(e, 1, 64);
}

// mode 0: x = L^-T y, y = row n of the factor, to s.  mode 1: y = the vector (of items not yet
// converged), s += x
template <typename T>
__global__ void __launch_bounds__(1024) k_solve_bwd_b(BatchDev bd, int s, int mode)
{
    __shared__ T part[16][PAN];
    __shared__ __align__(16) T sx[PAN];
    __shared__ T tpart[16][TS + 1];
    __shared__ T rhs[TS];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || (mode && bd.status[4 * item + 3])) return;
    const int ld = M.ldN, n = M.n_src, np = (ld + PAN - 1) / PAN;
    const int Pn = np - 1 - s, Q = Pn - (int)blockIdx.x;  // an item's steps count from its own last panel
    if (Q < 0) return;
    const T* L = (sizeof(T) == 8) ? (const T*)(bd.F + M.f_off) : (const T*)(bd.F32 + M.f_off);
    T* v = solve_vec<T>(bd, M);
    const int q0 = Q * PAN, nq = min(PAN, ld - q0), c = threadIdx.x;
    if (s > 0) {
        const int r0 = (Pn + 1) * PAN;
        bwd_tile<T>(L + (size_t)r0 * ld + q0, ld, min(PAN, ld - r0), v + r0, part);
        __syncthreads();
    }
    if (c < nq) {
        // mode 0: until its first update a panel's y stands in row n of the factor
        T a = (mode || s > 1) ? v[q0 + c] : q0 + c < n ? L[(size_t)n * ld + q0 + c] : (T)0;
        if (s > 0) a -= part_sum<T>(part, c);
        sx[c] = a;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        tri_bwd<T>(L + (size_t)q0 * ld + q0, ld, nq / TS, (const T*)(bd.winv + M.w_off) + (size_t)q0 * TS, sx, tpart, rhs);
        double* so = bd.vec + M.vec_off + q0;
        if (c < nq) {
            if (mode == 0) so[c] = q0 + c < n ? (double)sx[c] : 0.0;
            else if (q0 + c < n) so[c] += (double)sx[c];
        }
    }
    if (c < nq) v[q0 + c] = sx[c];
}

// x = L^-1 b in place in the vector, of items not yet converged (FP32)
__global__ void __launch_bounds__(1024) k_solve_fwd_b(BatchDev bd, int s)
{
    __shared__ __align__(16) float sx[PAN];
    __shared__ float rhs[TS];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || bd.status[4 * item + 3]) return;
    const int ld = M.ldN, np = (ld + PAN - 1) / PAN;
    const int Q = s + (int)blockIdx.x;
    if (Q >= np) return;
    const float* L = bd.F32 + M.f_off;
    float* v = solve_vec<float>(bd, M);
    const int q0 = Q * PAN, nq = min(PAN, ld - q0), c = threadIdx.x;
    const int r = (c >> 6) + 16 * ((c & 63) >> 2);
    if (s > 0) {
        const int c0 = (s - 1) * PAN;
        const float e = fwd_tile(L + (size_t)q0 * ld + c0, ld, nq, v + c0);
        if ((c & 3) == 0 && r < nq) sx[r] = v[q0 + r] - e;
    } else if (c < nq) {
        sx[c] = v[q0 + c];
    }
    __syncthreads();
    if (blockIdx.x == 0) tri_fwd<float>(L + (size_t)q0 * ld + q0, ld, nq / TS, (const float*)(bd.winv + M.w_off) + (size_t)q0 * TS, sx, rhs);
    if (c < nq) v[q0 + c] = sx[c];
}

// mode 0: x = L^-T y to s.  mode 1 (FP32): s += (L L^T)^-1 of the vector, of items not yet converged
template <typename T>
__global__ void __launch_bounds__(1024) k_solve_one_b(BatchDev bd, int mode)
{
    extern __shared__ __align__(16) double one_lds[];
    T(*part)[PAN] = (T(*)[PAN])one_lds;
    T(*tpart)[TS + 1] = (T(*)[TS + 1])(part + 16);
    T* rhs = (T*)(tpart + 16);
    T* sx = rhs + TS;  // the vector
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || (mode && bd.status[4 * item + 3])) return;
    const int ld = M.ldN, n = M.n_src, np = (ld + PAN - 1) / PAN, tid = threadIdx.x;
    const T* L = (sizeof(T) == 8) ? (const T*)(bd.F + M.f_off) : (const T*)(bd.F32 + M.f_off);
    const T* W = (const T*)(bd.winv + M.w_off);
    const T* v = solve_vec<T>(bd, M);
    for (int c = tid; c < ld; c += 1024) sx[c] = mode ? v[c] : c < n ? L[(size_t)n * ld + c] : (T)0;
    __syncthreads();
    if constexpr (sizeof(T) == 4)
        if (mode)
            for (int P = 0; P < np; P++) {
                const int p0 = P * PAN;
                tri_fwd<T>(L + (size_t)p0 * ld + p0, ld, min(PAN, ld - p0) / TS, W + (size_t)p0 * TS, sx + p0, rhs);
                const int r = (tid >> 6) + 16 * ((tid & 63) >> 2);
                for (int q0 = p0 + PAN; q0 < ld; q0 += PAN) {
                    const int nq = min(PAN, ld - q0);
                    const float e = fwd_tile(L + (size_t)q0 * ld + p0, ld, nq, sx + p0);
                    if ((tid & 3) == 0 && r < nq) sx[q0 + r] -= e;
                }
                __syncthreads();
            }
    for (int P = np - 1; P >= 0; P--) {
        const int p0 = P * PAN, npr = min(PAN, ld - p0);
        tri_bwd<T>(L + (size_t)p0 * ld + p0, ld, npr / TS, W + (size_t)p0 * TS, sx + p0, tpart, rhs);
        for (int Q = P - 1; Q >= 0; Q--) {
            bwd_tile<T>(L + (size_t)p0 * ld + Q * PAN, ld, npr, sx + p0, part);
            __syncthreads();
            if (tid < PAN) sx[Q * PAN + tid] -= part_sum<T>(part, tid);
            __syncthreads();
        }
    }
    double* s = bd.vec + M.vec_off;
    for (int c = tid; c < ld; c += 1024) {
        if (mode == 0) s[c] = (c < n) ? (double)sx[c] : 0.0;
        else if (c < n) s[c] += (double)sx[c];
    }
}

template <typename T>
static void launch_solve(hipStream_t s, const BatchDev& bd, int max_ld, int mode, bool one)
{
    const int np = (max_ld + PAN - 1) / PAN;
    if (one && max_ld <= QLX_SOLVE_ONE_LD) {
        allow_big_lds((const void*)k_solve_one_b<T>);
        hipLaunchKernelGGL(k_solve_one_b<T>, dim3(1, bd.B), dim3(1024), SOLVE_ONE_LDS(max_ld) * sizeof(T), s, bd, mode);
        return;
    }
    if (mode)
        for (int k = 0; k < np; k++) hipLaunchKernelGGL(k_solve_fwd_b, dim3(np - k, bd.B), dim3(1024), 0, s, bd, k);
    for (int k = 0; k < np; k++) hipLaunchKernelGGL(k_solve_bwd_b<T>, dim3(np - k, bd.B), dim3(1024), 0, s, bd, k, mode);
}

void launch_trisolve_b(hipStream_t s, const BatchDev& bd, int max_ld, int f32)
{
    const bool one = bd.B >= SOLVE_ONE_B;
    if (f32) launch_solve<float>(s, bd, max_ld, 0, one);
    else launch_solve<double>(s, bd, max_ld, 0, one);
}

// ------------------------------------------------------------------------------------------------
// FP64 iterative refinement of the mixed-precision solve (classical mixed-precision refinement,
// Wilkinson / Moler): r = D - F s in FP64 arithmetic on the FP32 F as formed (Ff32 + Fdiag),
// dx = F^-1 r with the FP32 factor, s += dx.  The residual kernel writes per-row-block partial
// sums of r^2 and D^2; the refine kernel stops an item once ||r|| <= tol ||D||.
// status[4*item+2] counts steps; status[4*item+3] marks a finished item: 1 converged, 2 stopped after
// the last allowed step with the residual still above the tolerance.
// ------------------------------------------------------------------------------------------------
// sum of a[k] over the 64 lanes for 16 values at once: four halvings, then a 4-lane sum; lane l ends
// with the total of a[(l >> 2) & 15]
__device__ __forceinline__ double lane_sum16(const double* a)
{
    const int lane = threadIdx.x & 63;
    double b[8], c[4], d[2];
    const bool h5 = lane & 32, h4 = lane & 16, h3 = lane & 8, h2 = lane & 4;
#pragma unroll
    for (int j = 0; j < 8; j++) b[j] = a[(h5 ? 8 : 0) + j] + __shfl_xor(a[(h5 ? 0 : 8) + j], 32, 64);
#pragma unroll
    for (int j = 0; j < 4; j++) c[j] = b[(h4 ? 4 : 0) + j] + __shfl_xor(b[(h4 ? 0 : 4) + j], 16, 64);
#pragma unroll
    for (int j = 0; j < 2; j++) d[j] = c[(h3 ? 2 : 0) + j] + __shfl_xor(c[(h3 ? 0 : 2) + j], 8, 64);
    double e = d[h2 ? 1 : 0] + __shfl_xor(d[h2 ? 0 : 1], 4, 64);
    e += __shfl_xor(e, 2, 64);
    e += __shfl_xor(e, 1, 64);
    return e;
}

// r = D - F s on F as formed (Ff32, lower 128-tiles; a diagonal tile is held whole), reading each
// lower element once: k_resid_rows_b takes row block I (64 rows): its row strip (columns c < 64 I
// of rows i) gives the rows' sums, and the same loads give the strip's transposed products
// z_I(c) = sum_i F(i, c) s(i), stored per row block (zres); with the diagonal tile (through LDS, its
// upper half) the rows' partial sums go to the slot Yp.  k_resid_cols_b adds, for the rows of block
// J, the column strip sum_{I > J} z_I in order of I, then r = D - (Fdiag s + that + Yp); D(i) =
// F(n, i).  Products are formed and summed in FP64; rows >= n take no part.
__global__ void __launch_bounds__(256) k_resid_rows_b(BatchDev bd)
{
    __shared__ float tile[TS][TS + 1];
    __shared__ double dacc[4][TS];
    __shared__ double racc[TS];
    __shared__ double zs[2][4][256];  // column partials of passes it (even / odd)
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || bd.status[4 * item + 3]) return;
    const int ld = M.ldN, n = M.n_src, nb = ld / TS;
    const int I = (int)gridDim.x - 1 - (int)blockIdx.x;  // the longest row strips are dispatched first
    if (I >= nb || I * TS >= n) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const float* U = bd.Ff32 + M.f_off;
    double* v = bd.vec + M.vec_off;
    const double* s = v;
    double* yp = v + 7 * (size_t)ld;
    double* Z = bd.zres + M.f_off / 128 + (size_t)TS * I * (I - 1) / 2;  // z_I: c0 values
    const int c0 = I * TS;
    // diagonal tile
#pragma unroll
    for (int e = tid; e < TS * TS / 4; e += 256) {
        const int row = e >> 4, cc = 4 * (e & 15);
        const float4_t t = *(const float4_t*)(U + (size_t)(c0 + row) * ld + c0 + cc);
        tile[row][cc] = t.x;
        tile[row][cc + 1] = t.y;
        tile[row][cc + 2] = t.z;
        tile[row][cc + 3] = t.w;
    }
    // row strip: F(i,c) = U[i][c] for c < c0; wave w owns rows c0 + w + 4k, k = 0..15, lane the four
    // columns 256 it + 4 lane .. + 3 of pass it (every thread runs every pass: the passes' barrier).
    // A pass's loads are issued before the previous pass's barrier and column sums; the column
    // partials alternate between two LDS buffers, so one barrier per pass orders them
    {
        double ra[16], si[16];
#pragma unroll
        for (int k = 0; k < 16; k++) {
            ra[k] = 0.0;
            const int row = c0 + w + 4 * k;
            si[k] = row < n ? s[row] : 0.0;
        }
        const float* Ur = U + (size_t)(c0 + w) * ld;
        const int npass = (c0 + 255) / 256;
        float4_t t[16];
        if (4 * lane < c0) {  // c0 is a multiple of 64, so c + 3 < c0 for every c < c0 below
#pragma unroll
            for (int k = 0; k < 16; k++) t[k] = *(const float4_t*)(Ur + (size_t)(4 * k) * ld + 4 * lane);
        }
        for (int it = 0; it < npass; it++) {
            const int c = 256 * it + 4 * lane;
            double z0 = 0.0, z1 = 0.0, z2 = 0.0, z3 = 0.0;
            if (c < c0) {
                const double s0 = s[c], s1 = s[c + 1], s2 = s[c + 2], s3 = s[c + 3];
#pragma unroll
                for (int k = 0; k < 16; k++) {
                    ra[k] = fma((double)t[k].x, s0, fma((double)t[k].y, s1, fma((double)t[k].z, s2, fma((double)t[k].w, s3, ra[k]))));
                    z0 = fma((double)t[k].x, si[k], z0);
                    z1 = fma((double)t[k].y, si[k], z1);
                    z2 = fma((double)t[k].z, si[k], z2);
                    z3 = fma((double)t[k].w, si[k], z3);
                }
            }
            double* zb = &zs[it & 1][0][0];
            zb[w * 256 + 4 * lane] = z0;
            zb[w * 256 + 4 * lane + 1] = z1;
            zb[w * 256 + 4 * lane + 2] = z2;
            zb[w * 256 + 4 * lane + 3] = z3;
            if (c + 256 < c0) {
#pragma unroll
                for (int k = 0; k < 16; k++) t[k] = *(const float4_t*)(Ur + (size_t)(4 * k) * ld + c + 256);
            }
            __syncthreads();
            if (256 * it + tid < c0) Z[256 * it + tid] = ((zb[tid] + zb[256 + tid]) + zb[512 + tid]) + zb[768 + tid];
        }
        const double tot = lane_sum16(ra);
        if ((lane & 3) == 0) racc[w + 4 * (lane >> 2)] = tot;
    }
    __syncthreads();
    // diagonal tile: thread (i, g) sums c in [16 g, 16 g + 16), c != i, c0 + c < n
    {
        const int i = tid & 63, g = tid >> 6;
        double a = 0.0;
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int c = 16 * g + q;
            if (c != i && c0 + c < n) a = fma((double)(c > i ? tile[i][c] : tile[c][i]), s[c0 + c], a);
        }
        dacc[g][i] = a;
    }
    __syncthreads();
    if (tid < TS && c0 + tid < n)
        yp[c0 + tid] = ((dacc[0][tid] + dacc[1][tid]) + (dacc[2][tid] + dacc[3][tid])) + racc[tid];
}

__global__ void __launch_bounds__(64) k_resid_cols_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || bd.status[4 * item + 3]) return;
    const int ld = M.ldN, n = M.n_src, nb = ld / TS;
    const int J = blockIdx.x;
    if (J >= nb || J * TS >= n) return;
    const int nbr = (n + TS - 1) / TS;
    const int tid = threadIdx.x;
    const float* U = bd.Ff32 + M.f_off;
    double* v = bd.vec + M.vec_off;
    const double* s = v;
    const double* fdiag = v + 3 * (size_t)ld;
    double* r = v + 4 * (size_t)ld;
    double* part = v + 5 * (size_t)ld;
    const double* yp = v + 7 * (size_t)ld;
    const double* Zb = bd.zres + M.f_off / 128;
    const int i = J * TS + tid;
    double rr = 0.0, dd = 0.0;
    if (i < n) {
        double cs = 0.0;
        for (int I = J + 1; I < nbr; I++) cs += Zb[(size_t)TS * I * (I - 1) / 2 + i];
        const double D = (double)U[(size_t)n * ld + i];
        const double Fs = fdiag[i] * s[i] + cs + yp[i];
        rr = D - Fs;
        r[i] = rr;
        rr = rr * rr;
        dd = D * D;
    }
    for (int off = 32; off > 0; off >>= 1) {
        rr += __shfl_xor(rr, off, 64);
        dd += __shfl_xor(dd, off, 64);
    }
    if (tid == 0) {
        part[J] = rr;
        part[nb + J] = dd;
    }
}

// convergence of the item from the residual partials; an item that goes on gets the residual into its vector
__global__ void __launch_bounds__(1024) k_refine_check_b(BatchDev bd, int final_check, double tol)
{
    __shared__ double red[2][64];
    __shared__ int done;
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid || bd.status[4 * item + 3]) return;
    const int ld = M.ldN, nb = ld / TS, n = M.n_src;
    const int tid = threadIdx.x;
    const double* pr = bd.vec + M.vec_off + 5 * (size_t)ld;
    const int nbr = (n + TS - 1) / TS;
    if (tid < 64) {
        double a = 0.0, b = 0.0;
        for (int k = tid; k < nbr; k += 64) {
            a += pr[k];
            b += pr[nb + k];
        }
        red[0][tid] = a;
        red[1][tid] = b;
    }
    __syncthreads();
    if (tid == 0) {
        double a = 0.0, b = 0.0;
        for (int k = 0; k < 64; k++) {
            a += red[0][k];
            b += red[1][k];
        }
        const double rel = (b > 0) ? sqrt(a / b) : 0.0;
        bd.out[QLX_OUT_STRIDE * item + 6] = rel;
        done = (rel <= tol || final_check) ? 1 : 0;
        if (done) bd.status[4 * item + 3] = (rel <= tol) ? 1 : 2;  // 2: stopped above the tolerance
        else bd.status[4 * item + 2] += 1;
    }
    __syncthreads();
    if (done) return;
    float* v = solve_vec<float>(bd, M);
    const double* r = bd.vec + M.vec_off + 4 * (size_t)ld;
    for (int c = tid; c < ld; c += 1024) v[c] = (c < n) ? (float)r[c] : 0.0f;
}

void launch_refine_check_b(hipStream_t s, const BatchDev& bd, int max_ld, int final_check, double tol)
{
    const int nb = max_ld / TS;
    hipLaunchKernelGGL(k_resid_rows_b, dim3(nb, bd.B), dim3(256), 0, s, bd);
    hipLaunchKernelGGL(k_resid_cols_b, dim3(nb, bd.B), dim3(64), 0, s, bd);
    hipLaunchKernelGGL(k_refine_check_b, dim3(1, bd.B), dim3(1024), 0, s, bd, final_check, tol);
}

void launch_refine_step_b(hipStream_t s, const BatchDev& bd, int max_ld, int step)
{
    // steps after the first are for the few items still above the tolerance: one workgroup each, in one
    // launch, up to QLX_SOLVE_ONE_LD
    launch_solve<float>(s, bd, max_ld, 1, step > 0 || bd.B >= SOLVE_ONE_B);
}

// ------------------------------------------------------------------------------------------------
// evidence: v = L s per active pixel, model = PSF (x) v over active taps, chi^2 over the mask,
// Es = sum_l ||H_l s||^2 (= s^T R s), -2 ln E = ((0 + regterms) + ln det F) + chi^2
// ------------------------------------------------------------------------------------------------
// s in the reference order: s_ref[pisrc[p]] = s[p]
__global__ void __launch_bounds__(256) k_unpermute_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || p >= M.n_src) return;
    const double* s = bd.vec + M.vec_off;
    double* sref = bd.vec + M.vec_off + 6 * (size_t)M.ldN;
    sref[bd.pisrc[item * bd.s_cell + p]] = s[p];
}

__global__ void __launch_bounds__(256) k_Ls_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || r >= M.n_img) return;
    const int U = 3 * bd.nsub;
    const int* ucol = bd.ucol + ((size_t)item * bd.s_pix + r) * U;
    const double* uval = bd.uval + ((size_t)item * bd.s_pix + r) * U;
    const double* s = bd.vec + M.vec_off;
    double acc = 0.0;
    const int cnt = bd.ucnt[item * bd.s_pix + r];
    if (U == 12) {  // 2 x 2 split: all 12 slots written by the merge, same summation order
        int c[12];
        double w[12];
        load_row12(ucol, uval, c, w);
#pragma unroll
        for (int e = 0; e < 12; e++)
            if (e < cnt) acc += w[e] * s[c[e]];
    } else {
        for (int e = 0; e < cnt; e++) acc += uval[e] * s[ucol[e]];
    }
    // the unblurred model as a dense image (pixel index; inactive pixels keep the zero fill)
    bd.model[(size_t)item * 2 * bd.s_pix + bd.s_pix + bd.act_pix[item * bd.s_pix + r]] = acc;
}

// blurred model of every active pixel: the PSF taps over the dense unblurred image (zero outside
// the active set, which is what skipping inactive neighbours gives).  A lane takes MKB pixels
// (k0 .. k0+MKB-1, l) and lanes of a wave consecutive l, so the lanes of one load read consecutive
// pixels; each image value it loads serves every one of its pixels that the tap reaches
// ((pnx + MKB - 1) pny loads for MKB pixels instead of MKB pnx pny).  Image rows go in descending
// order, so each pixel still sums its taps pk ascending, pl ascending: the result is the
// one-pixel-per-lane gather's, bit for bit.
#define MKB 4
__global__ void __launch_bounds__(256) k_model_b(BatchDev bd)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    const int nx = bd.nx, ny = bd.ny;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (!M.valid || t >= (nx + MKB - 1) / MKB * ny) return;
    const int kb = t / ny, l = t - kb * ny, k0 = kb * MKB;
    const int* pidx = bd.pidx + item * bd.s_pix;
    bool any = false;
#pragma unroll
    for (int a = 0; a < MKB; a++) any |= (k0 + a < nx) && pidx[(k0 + a) * ny + l] >= 0;
    if (!any) return;
    const int nxh = bd.pnx / 2, nyh = bd.pny / 2, pnx = bd.pnx, pny = bd.pny;
    double* model = bd.model + (size_t)item * 2 * bd.s_pix;
    const double* v = model + bd.s_pix;
    double acc[MKB];
#pragma unroll
    for (int a = 0; a < MKB; a++) acc[a] = 0.0;
    for (int ii = k0 + MKB - 1 + nxh; ii >= k0 + nxh - pnx + 1; ii--) {
        if (ii < 0 || ii >= nx) continue;
        const double* vr = v + (size_t)ii * ny;
        for (int pl = 0; pl < pny; pl++) {
            const int jj = l + nyh - pl;
            if (jj < 0 || jj >= ny) continue;
            const double x = vr[jj];
#pragma unroll
            for (int a = 0; a < MKB; a++) {
                const int pk = k0 + a + nxh - ii;
                if (pk >= 0 && pk < pnx) acc[a] += bd.psf[pk * pny + pl] * x;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < MKB; a++) {
        const int pa = (k0 + a) * ny + l;
        if (k0 + a < nx && pidx[pa] >= 0) model[pa] = acc[a];
    }
}

__global__ void __launch_bounds__(1024) k_evidence_b(BatchDev bd)
{
    __shared__ double sh[1024];
    __shared__ double sh2[1024];
    __shared__ double sh3[1024];
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const int npix = bd.nx * bd.ny;
    const int* pm = bd.pmapped + item * bd.s_pix;
    const double* model = bd.model + (size_t)item * 2 * bd.s_pix;
    const int* sidx = bd.sidx + item * bd.s_cell;
    const double* s = bd.vec + M.vec_off + 6 * (size_t)M.ldN;  // reference order
    double chi = 0.0, chia = 0.0;  // all mask pixels; active pixels only (chisq_regparam_dense's Ed)
    for (int p = threadIdx.x; p < npix; p += 1024) {
        if (bd.mask && !bd.mask[p]) continue;
        const double d = bd.data[p];
        if (pm[p]) {
            const double r = model[p] - d;
            chi += (r * r) * bd.covinv[p];
            chia += (r * r) * bd.covinv[p];
        } else {
            chi += (d * d) * bd.covinv[p];
        }
    }
    double es = 0.0;
    const int snx = M.snx, sny = M.sny;
    for (int c = threadIdx.x; c < snx * sny; c += 1024) {
        const int a = sidx[c];
        if (a < 0) continue;
        const int i = c / sny, j = c % sny;
        const double sa = s[a];
        int n0 = (i < snx - 1) ? sidx[(i + 1) * sny + j] : -1;
        int n1 = (i > 0) ? sidx[(i - 1) * sny + j] : -1;
        double h = -2.0 * sa + (n0 >= 0 ? s[n0] : 0.0) + (n1 >= 0 ? s[n1] : 0.0);
        es += h * h;
        n0 = (j < sny - 1) ? sidx[i * sny + j + 1] : -1;
        n1 = (j > 0) ? sidx[i * sny + j - 1] : -1;
        h = -2.0 * sa + (n0 >= 0 ? s[n0] : 0.0) + (n1 >= 0 ? s[n1] : 0.0);
        es += h * h;
    }
    sh[threadIdx.x] = chi;
    sh2[threadIdx.x] = es;
    sh3[threadIdx.x] = chia;
    __syncthreads();
    for (int st = 512; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            sh[threadIdx.x] += sh[threadIdx.x + st];
            sh2[threadIdx.x] += sh2[threadIdx.x + st];
            sh3[threadIdx.x] += sh3[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        double* o = bd.out + QLX_OUT_STRIDE * item;
        const double chisq = sh[0], Es = sh2[0];
        const double logdetF = o[2], logdetR = o[3];
        const double lam = item_lambda(bd, item);
        double loglike = 0.0, regterms = 0.0;
        if (lam != 0) {
            regterms = lam * Es - M.n_src * log(lam) - logdetR;
            loglike += regterms;
        }
        loglike += logdetF;
        loglike += chisq;
        o[0] = loglike;
        o[1] = chisq;
        o[4] = Es;
        o[5] = regterms;
        o[7] = (double)bd.status[4 * item + 2];
        o[8] = (sh3[0] + regterms) + logdetF;  // chisq_regparam_dense: Ed + loglike_reg, then + logdet
    }
}

__global__ void __launch_bounds__(256) k_keep_b(BatchDev bd, char* keep)
{
    const int item = blockIdx.y;
    const ItemMeta& M = bd.meta[item];
    if (!M.valid) return;
    const int ncell = M.snx * M.sny;
    double* ks = (double*)(keep + M.keep_off);
    double* km = ks + ncell;
    int* ki = (int*)(km + bd.s_pix);
    const double* sref = bd.vec + M.vec_off + 6 * (size_t)M.ldN;
    const double* model = bd.model + (size_t)item * 2 * bd.s_pix;
    const int* sidx = bd.sidx + (size_t)item * bd.s_cell;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < bd.s_pix; t += stride) {
        km[t] = model[t];
        if (t < ncell) ki[t] = sidx[t];
        if (t < M.n_src) ks[t] = sref[t];
    }
    for (long long t = bd.s_pix + (long long)blockIdx.x * blockDim.x + threadIdx.x; t < ncell; t += stride) {
        ki[t] = sidx[t];
        if (t < M.n_src) ks[t] = sref[t];
    }
}

void launch_keep_b(hipStream_t s, const BatchDev& bd, void* keep, int max_cells)
{
    const long long n = std::max<long long>(bd.s_pix, max_cells);
    const unsigned nb = (unsigned)std::min<long long>((n + 255) / 256, 64);
    hipLaunchKernelGGL(k_keep_b, dim3(nb, bd.B), dim3(256), 0, s, bd, (char*)keep);
}

void launch_evidence_b(hipStream_t st, const BatchDev& bd, int max_img, int max_src)
{
    launch_fill_f64(st, bd.model, 0.0, (size_t)bd.B * 2 * bd.s_pix);
    if (max_src > 0) hipLaunchKernelGGL(k_unpermute_b, dim3((max_src + 255) / 256, bd.B), dim3(256), 0, st, bd);
    if (max_img > 0) {
        hipLaunchKernelGGL(k_Ls_b, dim3((max_img + 255) / 256, bd.B), dim3(256), 0, st, bd);
        const long long nlane = (long long)(bd.nx + MKB - 1) / MKB * bd.ny;
        hipLaunchKernelGGL(k_model_b, dim3((unsigned)((nlane + 255) / 256), bd.B), dim3(256), 0, st, bd);
    }
    hipLaunchKernelGGL(k_evidence_b, dim3(1, bd.B), dim3(1024), 0, st, bd);
}

// ------------------------------------------------------------------------------------------------
// MFMA layout self-tests (fixed operands, results per lane/register)
// ------------------------------------------------------------------------------------------------
__global__ void k_selftest_mfma(double* out)
{
    const int lane = threadIdx.x;
    // f64 16x16x4: A[i][k] = i + 1 + 0.01 k, B[k][j] = 1 + k + 0.1 j
    {
        const int i = lane & 15, k = lane >> 4;
        double a = i + 1 + 0.01 * k, b = 1 + k + 0.1 * (lane & 15);
        double4_t acc = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        for (int v = 0; v < 4; v++) out[lane * 4 + v] = acc[v];
    }
    // f32 16x16x4: same operands in float
    {
        const int i = lane & 15, k = lane >> 4;
        float a = i + 1 + 0.01f * k, b = 1 + k + 0.1f * (lane & 15);
        float4_t acc = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
        for (int v = 0; v < 4; v++) out[256 + lane * 4 + v] = acc[v];
    }
    // bf16 16x16x32: lane holds k = 8*(lane/16) .. +8 of row/col lane%16;
    // A[i][k] = (i+1) * (k%4+1) / 4, B[k][j] = (j+1) * ((k/4)%8 + 1) / 8
    {
        bf16x8_t a, b;
        for (int t = 0; t < 8; t++) {
            const int k = 8 * (lane >> 4) + t;
            a[t] = (__bf16)((float)((lane & 15) + 1) * (float)(k % 4 + 1) * 0.25f);
            b[t] = (__bf16)((float)((lane & 15) + 1) * (float)((k / 4) % 8 + 1) * 0.125f);
        }
        float4_t acc = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        for (int v = 0; v < 4; v++) out[512 + lane * 4 + v] = acc[v];
    }
    // f16 16x16x32: the same operand values and lane layout in FP16
    {
        f16x8_t a, b;
        for (int t = 0; t < 8; t++) {
            const int k = 8 * (lane >> 4) + t;
            a[t] = (_Float16)((float)((lane & 15) + 1) * (float)(k % 4 + 1) * 0.25f);
            b[t] = (_Float16)((float)((lane & 15) + 1) * (float)((k / 4) % 8 + 1) * 0.125f);
        }
        float4_t acc = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
        for (int v = 0; v < 4; v++) out[768 + lane * 4 + v] = acc[v];
    }
}

void launch_selftest_mfma(hipStream_t s, double* out)
{
    hipLaunchKernelGGL(k_selftest_mfma, dim3(1), dim3(64), 0, s, out);
}

}  // namespace qlx
