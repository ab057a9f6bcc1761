// levels.hip -- batched apply of fields stored side by side per cell (field
// stride 1: the row-major x[n, k] of a model column, src/regridder/regrid.jl's
// NDSliceLoop over the trailing axes).
//
// A cell's k values are one contiguous run, so no staging of fields is needed
// for coalescing: LPR = ceil(k / V) neighbouring threads own one row, V fields
// (16 bytes) each, and read a source cell's run with 16-byte loads.  LPR is any
// integer (19 threads for 37 FP64 levels), so a block of 256 threads works on
// 256 / LPR rows at a time and few lanes idle; an odd last lane takes the last
// V fields again (it stores the values its neighbour stores).  A block's
// matrix entries are one contiguous run too: they are read into LDS first, so
// the loads of a row's source runs wait for nothing but their own latency.
// Bound: HBM for the fields plus the L2 traffic of the source runs (each is read
// by the ~4 rows that touch it; consecutive rows share a block, and every XCD
// owns a contiguous range of rows, so most of those reads hit a cache).
//
// A thread group runs through a short row by itself.  Wide rows (cells at a
// pole, or every row of a coarsening regridder) are summed by the whole block,
// its groups taking segments of the row side by side.
//
// Measured: 50 FP32 levels, 1440 x 721 -> HEALPix 256 (nnz 4.36 M) 1638 us in
// the tile kernel (which reads each field with a stride) -> 137 us, 3.1 TB/s of
// the 428 MB it needs; without poles (C416 -> C362) 106 us, 4.1 TB/s; 37 FP64
// levels, 721 x 361 -> C90 157 -> 34 us.  Occupancy is what counts (110 us with
// 6 waves a SIMD, 137 with 4): hence at most 6 source runs in flight a thread
// and 18 KB of entries a block; more rows a block widen the sources in use past
// an XCD's 4 MB of L2 (2 rows a thread group 141 us, 4 191, 8 268).
//
// FP32 fields: products and sums in FP64 from the FP64 A, one rounding at the
// end.  No plan is needed: a block takes a fixed number of rows, and the wide
// rows come from the regridder's list, a block each, the launch's first blocks
// (left inside the blocks of their neighbours they were its tail: all the
// pole's rows are neighbours).
//
// FP64 fields (EVEN): the segments of the kEven tile plan -- a row is cut where
// its tile's non-zeros cross a multiple of TileDesc::ent, each segment is summed
// with FMAs, the segments are added in order and divided by the area -- so the
// result equals the single-field tile kernel's bit for bit.  A block takes the
// rows of a tile that start in one run of its non-zeros, so blocks are even
// however long the rows are.
#include <algorithm>

#include "regridder.hpp"
#include "tileplan.hpp"

namespace cr {

namespace {

constexpr int kLevelThreads = 256;
constexpr int kStage = 1536;   // matrix entries a block holds in LDS
constexpr int kStageEven = 1280;
constexpr int kWideSeg = 16;   // longest segment of a wide row for FP32 fields
constexpr int kUnroll = 6;     // source runs in flight per thread

template <class T, int V>
struct Vec {
    typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T))));
};

// The sum of V fields over non-zeros [k, ke) in order: segments end where
// `left` more entries have been added (then every E), each summed on its own.
template <class T, int V, bool EVEN>
__device__ __forceinline__ void sum_row(double (&tot)[V], int k, int ke, const int32_t *col, const double *val,
                                        const T *__restrict__ x, int64_t xc, int left, int E) {
    using X = typename Vec<T, V>::type;
    double acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.0;
    for (; k < ke; k += kUnroll) {
        X xv[kUnroll];
#pragma unroll
        for (int j = 0; j < kUnroll; ++j)
            if (k + j < ke) xv[j] = *(const X *)(x + (int64_t)col[k + j] * xc);
#pragma unroll
        for (int j = 0; j < kUnroll; ++j)
            if (k + j < ke) {
                const double a = val[k + j];
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] = fma(a, (double)xv[j][v], acc[v]);
                if constexpr (EVEN) {
                    if (--left == 0) {
                        left = E;
#pragma unroll
                        for (int v = 0; v < V; ++v) {
                            tot[v] += acc[v];
                            acc[v] = 0.0;
                        }
                    }
                }
            }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) tot[v] += acc[v];
}

template <class T, int V>
__device__ __forceinline__ void store_row(const double (&tot)[V], T *__restrict__ y, const double *__restrict__ scale,
                                          int64_t row) {
    typename Vec<T, V>::type o;
    const double a = scale ? scale[row] : 1.0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        if constexpr (sizeof(T) == 4) o[v] = (float)(scale ? tot[v] * a : tot[v]);  // scale = 1 / area
        else o[v] = scale ? tot[v] / a : tot[v];                                    // scale = area
    }
    __builtin_nontemporal_store(o, (typename Vec<T, V>::type *)y);
}

// A wide row of `len` non-zeros at col, val by the whole block: segment g of
// the row is its entries [g * E - off, (g + 1) * E - off).  FP64: segment sums
// side by side, added in the segments' order.  FP32: a thread group runs through
// its share and the shares are added once.  Every thread of the block calls it;
// part: kLevelThreads * V sums.
template <class T, int V, bool EVEN>
__device__ __forceinline__ void wide_row(double (&tot)[V], int len, const int32_t *col, const double *val,
                                         const T *__restrict__ x, int64_t xc, int E, int off, int lpr,
                                         double (*part)[V]) {
    const int tid = threadIdx.x, groups = kLevelThreads / lpr, g = tid / lpr, l = tid - g * lpr;
    const int nseg = (len + off + E - 1) / E;
#pragma unroll
    for (int v = 0; v < V; ++v) tot[v] = 0.0;
    for (int s0 = 0; s0 < nseg; s0 += EVEN ? groups : nseg) {
        double acc[V];
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = 0.0;
        for (int sg = s0 + g; g < groups && sg < nseg; sg += groups) {
            sum_row<T, V, false>(acc, max(0, sg * E - off), min(len, (sg + 1) * E - off), col, val, x, xc, 0, 0);
            if (EVEN) break;
        }
        if (g < groups) {
#pragma unroll
            for (int v = 0; v < V; ++v) part[tid][v] = acc[v];
        }
        __syncthreads();
        if (g == 0) {
            const int m = min(groups, nseg - s0);
#pragma unroll 4
            for (int j = 0; j < m; ++j)
#pragma unroll
                for (int v = 0; v < V; ++v) tot[v] += part[j * lpr + l][v];
        }
        __syncthreads();
    }
}

// EVEN: block u takes the parts u % parts, u % parts + parts, ... of tile
// u / parts: the rows that start in that run of `run` of the tile's non-zeros.
// Else: rows [u * run, (u+1) * run), and blocks [0, wide_blocks) take the listed
// wide rows.  blockIdx.y: a chunk of the fields.
template <class T, int V, bool EVEN>
__global__ void __launch_bounds__(kLevelThreads) k_levels(
    const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col, const double *__restrict__ val,
    int64_t nrows, const T *__restrict__ x, int64_t xc, T *__restrict__ y, int64_t yc, int64_t nf, int lpr,
    int64_t chunk, const double *__restrict__ scale, int64_t units, int64_t units_per_xcd, int run,
    const TileDesc *__restrict__ tiles, int parts, const int32_t *__restrict__ wide,
    const int32_t *__restrict__ nwide, int wide_blocks, int wide_over) {
    constexpr int kRowsMax = EVEN ? GeomS::kRows : kLevelThreads;
    // entries of the block, and a wide row's partial sums: behind the entries
    // (EVEN), or in their last places (a listed row may use fewer places)
    constexpr int kPartAt = EVEN ? kStageEven : kStage - kLevelThreads * V;
    constexpr int kPlaces = EVEN ? kStageEven : kStage;
    __shared__ double sval[kPartAt + kLevelThreads * V];
    __shared__ int32_t scol[kPlaces];
    __shared__ int32_t srow[kRowsMax + 1];  // first entry of each row, from row r0's
    __shared__ int range[2];
    const int tid = threadIdx.x;
    const int groups = kLevelThreads / lpr;
    const int g = tid / lpr, l = tid - g * lpr;
    const int64_t c0 = (int64_t)blockIdx.y * chunk;
    const int64_t f = c0 + min((int64_t)l * V, min(chunk, nf - c0) - V);
    const T *xf = x + f;
    double(*part)[V] = (double(*)[V])(sval + kPartAt);

    if (!EVEN && (int)blockIdx.x < wide_blocks) {
        const int n = *nwide;
        for (int i = blockIdx.x; i < n; i += wide_blocks) {
            const int64_t r = wide[i], k0 = rowptr[r];
            const int len = (int)(rowptr[r + 1] - k0);
            if (len <= wide_over) continue;
            const bool staged = len <= kPartAt;
            if (staged)
                for (int q = tid; q < len; q += kLevelThreads) {
                    scol[q] = col[k0 + q];
                    sval[q] = val[k0 + q];
                }
            __syncthreads();
            const int E = max(2, min(kWideSeg, (len + groups - 1) / groups));
            double tot[V];
            if (staged) wide_row<T, V, false>(tot, len, scol, sval, xf, xc, E, 0, lpr, part);
            else wide_row<T, V, false>(tot, len, col + k0, val + k0, xf, xc, E, 0, lpr, part);
            if (g == 0) store_row<T, V>(tot, y + r * yc + f, scale, r);
        }
        return;
    }

    const int64_t b = (int64_t)blockIdx.x - wide_blocks;  // wide_blocks is a multiple of 8: b % 8 is the XCD
    const int64_t u = (b & 7) * units_per_xcd + (b >> 3);
    if (u >= units) return;
    int64_t r0, kb;         // the row of srow[0], its first non-zero
    int nr, E = 1, p = 0;   // rows of srow; EVEN: segment length, part
    bool huge = false;      // EVEN: the tile holds huge rows, which have no place in its runs
    auto run_start = [&](int i) {  // EVEN: row i's first place in the tile's runs
        int q = srow[i];
        if (huge)
            for (int h = 0; h < i; ++h) {
                const int n = srow[h + 1] - srow[h];
                if (n > GeomS::kCols) q -= n;
            }
        return q;
    };
    if constexpr (EVEN) {
        const TileDesc &t = tiles[u / parts];
        p = (int)(u % parts);
        E = t.ent;
        if (p * run > E * GeomS::kThreads) return;  // past the tile's last non-zero
        r0 = t.row0;
        nr = t.nrows;
    } else {
        r0 = u * run;
        nr = (int)min((int64_t)run, nrows - r0);
    }
    kb = rowptr[r0];
    for (int i = tid; i <= nr; i += kLevelThreads) {
        const int64_t k = rowptr[r0 + i];
        srow[i] = (int32_t)(k - kb);
        if (EVEN) huge |= i < nr && rowptr[r0 + i + 1] - k > GeomS::kCols;
    }
    if (EVEN) huge = __syncthreads_or(huge);
    else __syncthreads();

    // one pass, or (EVEN) one per part
    for (const int end = EVEN ? E * GeomS::kThreads : 0; p * run <= end; p += parts) {
        int i0 = 0, i1 = nr;  // this pass's rows r0 + [i0, i1)
        if constexpr (EVEN) {
            if (tid < 2) range[tid] = 0;
            __syncthreads();
            for (int i = tid; i < nr; i += kLevelThreads) {
                if (run_start(i) / run != p) continue;
                if (i == 0 || run_start(i - 1) / run != p) range[0] = i;
                if (i + 1 == nr || run_start(i + 1) / run != p) range[1] = i + 1;
            }
            __syncthreads();
            i0 = range[0];
            i1 = range[1];
            if (i0 == i1) continue;
        }
        const int first = srow[i0], total = srow[i1] - first;
        const bool staged = total <= kPlaces;
        const int32_t *gcol = col + kb + first;
        const double *gval = val + kb + first;
        if (staged) {
            for (int i = tid; i < total; i += kLevelThreads) {
                scol[i] = gcol[i];
                sval[i] = gval[i];
            }
        }
        __syncthreads();
        bool any_wide = false;
        for (int i = i0 + g; g < groups && i < i1; i += groups) {
            const int k0 = srow[i] - first, k1 = srow[i + 1] - first;
            if (k1 - k0 > wide_over) {
                any_wide = true;
                continue;
            }
            int left = 0;
            if constexpr (EVEN) left = E - (int)((uint32_t)run_start(i) % (uint32_t)E);
            double tot[V];
#pragma unroll
            for (int v = 0; v < V; ++v) tot[v] = 0.0;
            if (staged) sum_row<T, V, EVEN>(tot, k0, k1, scol, sval, xf, xc, left, E);
            else sum_row<T, V, EVEN>(tot, k0, k1, gcol, gval, xf, xc, left, E);
            store_row<T, V>(tot, y + (r0 + i) * yc + f, scale, r0 + i);
        }
        if constexpr (EVEN) {
            if (!__syncthreads_or(any_wide)) continue;
            for (int i = i0; i < i1; ++i) {
                const int k0 = srow[i] - first, len = srow[i + 1] - srow[i];
                if (len <= wide_over || len > GeomS::kCols) continue;  // done, or left to the long-row kernel
                const int off = (int)((uint32_t)run_start(i) % (uint32_t)E);
                double tot[V];
                if (staged) wide_row<T, V, true>(tot, len, scol + k0, sval + k0, xf, xc, E, off, lpr, part);
                else wide_row<T, V, true>(tot, len, gcol + k0, gval + k0, xf, xc, E, off, lpr, part);
                if (g == 0) store_row<T, V>(tot, y + (r0 + i) * yc + f, scale, r0 + i);
            }
        } else {
            break;
        }
    }
}

template <class T, int V, bool EVEN>
void launch(const Csr &A, const TilePlan *P, const T *x, int64_t xc, T *y, int64_t yc, int64_t nf, const double *scale,
            hipStream_t s) {
    // threads per row: at most a wave's worth, the fields split evenly over chunks of that size
    const int64_t lanes = (nf + V - 1) / V, chunks = (lanes + 63) / 64;
    const int lpr = (int)((lanes + chunks - 1) / chunks);
    const int64_t chunk = (int64_t)lpr * V;
    const int64_t gy = (nf + chunk - 1) / chunk;
    CR_REQUIRE(gy <= 65535, CR_UNSUPPORTED, "too many fields for one launch");
    // two rows a thread group where their entries fit the stage (FP32: one where two
    // would leave fewer than 1024 blocks: 37 fields of 360 x 180 -> C48 14.7 -> 9.1
    // us, of 2592 rows 3.9 -> 3.3)
    const int groups = kLevelThreads / lpr;
    const int64_t mean = (A.nnz + A.nrows - 1) / A.nrows;
    int run, parts = 1, wide_blocks = 0;
    // the pole's rows of an otherwise even matrix are worth a block each from
    // kWideRow on; where most rows are that long a thread group per row is better
    const int wide_over = EVEN || mean > 16 ? 2 * kWideRow : kWideRow;
    int64_t units;
    if (EVEN) {
        // every part's block reads its tile's row starts (4 KB), so runs are long
        // where that leaves enough blocks: 33 fields of 786 k rows take 201 us
        // with runs of 128, 163 with 256, 151 with 512.  Where 128 leaves few
        // blocks they are shorter, down to two rows a thread group: 64 fields of
        // 2592 rows take 21.5 us with runs of 128, 10.6 with 8; 100 fields of C24
        // -> 180 x 90 23.5 with 128, 14.1 with 36
        const int64_t even =
            std::min<int64_t>(512, std::max<int64_t>(std::min<int64_t>(128, A.nnz * gy / 1024), A.nnz / 4096));
        run = (int)std::min<int64_t>(kStageEven / 4 * 3, std::max<int64_t>(even, 2 * groups * mean));
        parts = (int)((A.nnz / P->ntiles + run - 1) / run);  // of a tile with the mean number of non-zeros
        parts = std::max(1, parts);
        units = P->ntiles * parts;
    } else {
        run = (int)std::min<int64_t>(A.nrows < 2048 * (int64_t)groups ? groups : 2 * groups, kLevelThreads);
        if (run * mean > kStage / 4 * 3) run = std::max<int>(std::min<int64_t>(groups, kStage / 4 * 3 / mean), 1);
        units = (A.nrows + run - 1) / run;
        wide_blocks = (int)std::min<int64_t>(8192, (A.wide_cap + 7) / 8 * 8);  // 0 when no row can be wide
    }
    const int64_t per_xcd = (units + 7) / 8;
    CR_REQUIRE(per_xcd * 8 + wide_blocks < (int64_t)1 << 31, CR_UNSUPPORTED, "too many rows for one launch");
    hipLaunchKernelGGL((k_levels<T, V, EVEN>), dim3((unsigned)(per_xcd * 8 + wide_blocks), (unsigned)gy),
                       dim3(kLevelThreads), 0, s, A.rowptr.p, A.col.p, A.val.p, A.nrows, x, xc, y, yc, nf, lpr, chunk,
                       scale, units, per_xcd, run, EVEN ? P->tiles.p : nullptr, parts, A.wide, A.nwide, wide_blocks,
                       wide_over);
}

}  // namespace

// y[row, 0..nf) = A x[:, 0..nf) with field stride 1 on both sides (nf >= 4).
// scale: 1/area (FP32 fields) or area (FP64 fields), nullptr: none.  FP64
// fields leave the plan's huge rows to the long-row kernel.
void launch_levels(const Csr &A, const float *x, int64_t xc, float *y, int64_t yc, int64_t nf, const double *scale,
                   hipStream_t s) {
    launch<float, 4, false>(A, nullptr, x, xc, y, yc, nf, scale, s);
}
void launch_levels(const Csr &A, const TilePlan &P, const double *x, int64_t xc, double *y, int64_t yc, int64_t nf,
                   const double *scale, hipStream_t s) {
    if (P.ntiles) launch<double, 2, true>(A, &P, x, xc, y, yc, nf, scale, s);
}

}  // namespace cr
