// kernels_column.hip -- the pressure system in the column layout
// (column_types.h): building the layout and its matrix, the fused matrix
// product, and the MIC(0) application as one launch per triangular sweep
// (column_sweep.h).
//
// Why this layout: the rows' own order (k, j, i) gives a sweep 64 lines to
// gather from per hyperplane and a neighbour id per term.  In columns a wave's
// operands of one hyperplane are one slice of consecutive slots, and every
// neighbour is at a fixed place of an adjacent slice, so the sweeps and the
// product load whole slices at addresses known ahead of time.  The price is
// the slots without rows: 22 hyperplanes of skew per column and the gaps.
#include <stdexcept>
#include <vector>

#include "kernels.h"

#include "column_hw.h"
#include "column_sweep.h"

namespace ff {

namespace {

// Steps whose operands, and whose neighbours' words, are in flight.  A forward
// sweep FP32 / FP64, us:
//             24^3       64^3      96x160x256
//    6, 3  20.0/26.4  52.4/70.4   151/203   taken (the fewest registers)
//    6, 2  23.3/27.2  60.5/71.9   160/198
//    6, 4  19.9/27.0  52.0/72.0   153/210
//    8, 3  19.6/26.0  51.4/69.4   150/202
//    8, 4  19.9/26.8  52.4/71.8   154/211
//   12, 3  21.5/28.4  53.6/72.5   151/205
constexpr int CPF = 6, CPX = 3;
// A wait's limit.  A look takes the latency of LDS (a ring) or of device memory (a
// word), some 0.05 to 0.7 us: 1 s at least, where a whole sweep takes 1 ms.
constexpr int WAIT_LOOKS = 20000000;
constexpr int EMPTY_LO = 0x3fffffff;

int ceilDiv(int a, int b) { return (a + b - 1) / b; }

// lowest and highest hyperplane of the pressure cells of each column: one
// workgroup per column, a wave per line
__global__ __launch_bounds__(256) void columnRangeKernel(Grid g, const int *mask, int ncj, ColumnRange *cols) {
    __shared__ int sLo[4], sHi[4];
    const int ni = g.ni, nj = g.nj, nk = g.nk;
    const int J0 = (blockIdx.x % ncj) * COL_J, K0 = (blockIdx.x / ncj) * COL_K;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    int lo = EMPTY_LO, hi = -1;
    for (int line = wave; line < COL_SLICE; line += 4) {
        const int j = J0 + line % COL_J, k = K0 + line / COL_J;
        if (j >= nj || k >= nk) continue;
        const int *m = mask + (size_t)ni * (j + (size_t)nj * k);
        for (int i = lane; i < ni; i += 64)
            if (m[i]) {
                lo = min(lo, i + j + k);
                hi = max(hi, i + j + k);
            }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if (lane == 0) {
        sLo[wave] = lo;
        sHi[wave] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        cols[blockIdx.x] = ColumnRange{min(min(sLo[0], sLo[1]), min(sLo[2], sLo[3])),
                                       max(max(sHi[0], sHi[1]), max(sHi[2], sHi[3])), 0, 0};
}

// the columns' slots in column order (one workgroup) and the total slice count
__global__ __launch_bounds__(1024) void columnScanKernel(ColumnRange *cols, int nc, int *totalSlices) {
    __shared__ int s[1024];
    const int t = threadIdx.x, per = (nc + 1023) / 1024;
    int sum = 0;
    for (int q = 0; q < per; q++) {
        const int c = t * per + q;
        if (c < nc && cols[c].hi >= cols[c].lo) sum += cols[c].hi - cols[c].lo + 1;
    }
    s[t] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int add = t >= off ? s[t - off] : 0;
        __syncthreads();
        s[t] += add;
        __syncthreads();
    }
    int run = s[t] - sum;
    for (int q = 0; q < per; q++) {
        const int c = t * per + q;
        if (c >= nc || cols[c].hi < cols[c].lo) continue;
        cols[c].base = COL_SLICE * (run - cols[c].lo);
        run += cols[c].hi - cols[c].lo + 1;
    }
    if (t == 1023) *totalSlices = s[t];
}

// the slices' links: one workgroup per column
__global__ __launch_bounds__(256) void columnLinksKernel(const ColumnRange *cols, int ncj, int nck, SliceLinks *links) {
    const int c = blockIdx.x, cj = c % ncj, ck = c / ncj;
    const ColumnRange own = cols[c], none{EMPTY_LO, -1, 0, 0};
    const ColumnRange jm = cj > 0 ? cols[c - 1] : none, jp = cj + 1 < ncj ? cols[c + 1] : none;
    const ColumnRange km = ck > 0 ? cols[c - ncj] : none, kp = ck + 1 < nck ? cols[c + ncj] : none;
    auto at = [](const ColumnRange &r, int h) { return h >= r.lo && h <= r.hi ? r.base + COL_SLICE * h : -1; };
    for (int h = own.lo + (int)threadIdx.x; h <= own.hi; h += 256)
        links[(own.base + COL_SLICE * h) / COL_SLICE] =
            SliceLinks{at(own, h - 1), at(own, h + 1), at(jm, h - 1), at(jp, h + 1),
                       at(km, h - 1),  at(kp, h + 1),  c,             h};
}

// slot -> row, and the matrix and right-hand side in slots; two slices per
// workgroup
template <class T>
__global__ __launch_bounds__(256) void columnFillKernel(Grid g, PressureSys S, int slices, const SliceLinks *links,
                                                        int ncj, int *slotRow, double *rhs, double *diag, double *ox,
                                                        double *oy, double *oz, T *fdiag, T *fox, T *foy, T *foz) {
    const int slice = blockIdx.x * (256 / COL_SLICE) + threadIdx.x / COL_SLICE, place = threadIdx.x % COL_SLICE;
    if (slice >= slices) return;
    const int c = links[slice].col, h = links[slice].h;
    const int j = (c % ncj) * COL_J + columnLineJ(place), k = (c / ncj) * COL_K + columnLineK(place), i = h - j - k;
    int r = -1;
    if (j < g.nj && k < g.nk && i >= 0 && i < g.ni) r = S.cellRow[i + (size_t)g.ni * (j + (size_t)g.nj * k)];
    const size_t e = (size_t)slice * COL_SLICE + place;
    const bool has = r >= 0;
    const double d = has ? S.diag[r] : 0.0, x = has ? S.ox[r] : 0.0, y = has ? S.oy[r] : 0.0, z = has ? S.oz[r] : 0.0;
    slotRow[e] = r;
    rhs[e] = has ? S.rhs[r] : 0.0;
    diag[e] = d;
    ox[e] = x;
    oy[e] = y;
    oz[e] = z;
    if (fdiag) {
        fdiag[e] = (T)d;
        fox[e] = (T)x;
        foy[e] = (T)y;
        foz[e] = (T)z;
    }
}

// the sweeps' records from the factor's rows: forward the L entries of the
// -x/-y/-z neighbour rows toward the row, backward the row's own
template <class T>
__global__ void columnRecordsKernel(PressureSys S, size_t slots, const int *slotRow, MicRec<T> *fwd, MicRec<T> *bwd) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= slots) return;
    const int r = slotRow[e];
    MicRec<T> f{T(0), T(0), T(0), T(0)}, b = f;
    if (r >= 0) {
        const int *nb = S.nbr + (size_t)6 * r;
        f.inv = b.inv = (T)S.invdiag[r];
        f.a = nb[0] >= 0 ? (T)S.lx[nb[0]] : T(0);
        f.b = nb[2] >= 0 ? (T)S.ly[nb[2]] : T(0);
        f.c = nb[4] >= 0 ? (T)S.lz[nb[4]] : T(0);
        b.a = (T)S.lx[r];
        b.b = (T)S.ly[r];
        b.c = (T)S.lz[r];
    }
    fwd[e] = f;
    bwd[e] = b;
}

// A vector between the slots' order and the rows' (the row-ordered schedules'
// applications and dots).  A slice's slots are 128 different lines, a line's rows
// lie together: a workgroup turns TURN slices over in LDS, so both sides move
// whole runs.  Bound by memory: 94 MB there in 22 us and back in 25 us FP64 at
// 256^3 (5.2M slots), 58 MB in 19 and 21 us FP32; a thread a slot, its row wherever
// that lies, took about 80 and 62 us both ways.  8 slices a workgroup 23 / 26 and 18
// / 21 us, 32 (FP32) 25 / 30.
constexpr int TURN = 16;
template <class T>
__global__ __launch_bounds__(256) void rowsFromSlotsKernel(size_t slots, const int *slotRow, const T *in, T *rows) {
    constexpr int N = TURN, P = N + 1;  // an odd pitch spreads a line over the banks
    __shared__ T v[COL_SLICE * P];
    __shared__ int r[COL_SLICE * P];
    const size_t e0 = (size_t)blockIdx.x * (COL_SLICE * N);
#pragma unroll
    for (int q = 0; q < COL_SLICE * N / 256; q++) {
        const int c = q * 256 + (int)threadIdx.x, a = c % COL_SLICE * P + c / COL_SLICE;
        const size_t e = e0 + c;
        r[a] = e < slots ? slotRow[e] : -1;
        v[a] = e < slots ? in[e] : T(0);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < COL_SLICE * N / 256; q++) {
        const int c = q * 256 + (int)threadIdx.x, a = c / N * P + c % N;
        if (r[a] >= 0) rows[r[a]] = v[a];
    }
}
template <class T>
__global__ __launch_bounds__(256) void slotsFromRowsKernel(size_t slots, const int *slotRow, const T *rows, T *out) {
    constexpr int N = TURN, P = N + 1;  // an odd pitch spreads a line over the banks
    __shared__ T v[COL_SLICE * P];
    __shared__ int r[COL_SLICE * P];
    const size_t e0 = (size_t)blockIdx.x * (COL_SLICE * N);
#pragma unroll
    for (int q = 0; q < COL_SLICE * N / 256; q++) {
        const int c = q * 256 + (int)threadIdx.x;
        r[c % COL_SLICE * P + c / COL_SLICE] = e0 + c < slots ? slotRow[e0 + c] : -1;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < COL_SLICE * N / 256; q++) {
        const int c = q * 256 + (int)threadIdx.x, a = c / N * P + c % N;
        v[a] = r[a] >= 0 ? rows[r[a]] : T(0);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < COL_SLICE * N / 256; q++) {
        const int c = q * 256 + (int)threadIdx.x;
        if (e0 + c < slots) out[e0 + c] = v[c % COL_SLICE * P + c / COL_SLICE];
    }
}
// cells' values at the slots' rows (a float grid), and back
__global__ void slotsFromCellsKernel(size_t slots, const int *slotRow, const int *rows, const float *cells, double *out) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < slots) out[e] = slotRow[e] >= 0 ? (double)cells[rows[slotRow[e]]] : 0.0;
}
template <class T>
__global__ void cellsFromSlotsKernel(size_t slots, const int *slotRow, const int *rows, const double *x, T *cells) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < slots && slotRow[e] >= 0) cells[rows[slotRow[e]]] = (T)x[e];
}

// (A x) of one slot in the reference's order (sparsematrix.h:174-215: -z, -y,
// -x, diagonal, +x, +y, +z).  The -x/-y/-z coefficients are the neighbour
// slots' +x/+y/+z ones (the assembly computes both from the shared face by
// the same expression).  A missing neighbour's term is left out.
template <class T>
struct ColumnMatrix {
    const T *diag, *ox, *oy, *oz;
};
template <class T, class X>
__device__ __forceinline__ T columnProduct(const SliceLinks &L, size_t e, int place, const ColumnMatrix<T> &A,
                                           const X &x) {
    const int lj = columnLineJ(place), lk = columnLineK(place);
    // first slot of the neighbour's slice and the place in it
    const int bym = lj > 0 ? L.im : L.jm, byp = lj < COL_J - 1 ? L.ip : L.jp;
    const int bzm = lk > 0 ? L.im : L.km, bzp = lk < COL_K - 1 ? L.ip : L.kp;
    const bool hxm = L.im >= 0, hxp = L.ip >= 0, hym = bym >= 0, hyp = byp >= 0, hzm = bzm >= 0, hzp = bzp >= 0;
    const int exm = hxm ? L.im + place : (int)e, exp = hxp ? L.ip + place : (int)e;
    const int eym = hym ? bym + columnPlace(lj + COL_J - 1, lk) : (int)e;
    const int eyp = hyp ? byp + columnPlace(lj + 1, lk) : (int)e;
    const int ezm = hzm ? bzm + columnPlace(lj, lk + COL_K - 1) : (int)e;
    const int ezp = hzp ? bzp + columnPlace(lj, lk + 1) : (int)e;
    const T cmz = A.oz[ezm], cmy = A.oy[eym], cmx = A.ox[exm], cd = A.diag[e], cox = A.ox[e], coy = A.oy[e],
            coz = A.oz[e];
    const T xzm = x[ezm], xym = x[eym], xxm = x[exm], xr = x[e], xxp = x[exp], xyp = x[eyp], xzp = x[ezp];
    T s = 0;
    if (hzm) s += cmz * xzm;
    if (hym) s += cmy * xym;
    if (hxm) s += cmx * xxm;
    s += cd * xr;
    if (hxp) s += cox * xxp;
    if (hyp) s += coy * xyp;
    if (hzp) s += coz * xzp;
    return s;
}

// q = A s with the partials of s . q, over the spans of the reductions (a span
// is whole slices, a wave handles half a slice at a time)
static_assert(REDUCE_THREADS % COL_SLICE == 0 && COL_SLICE % 64 == 0, "spans are whole slices, slices whole waves");
constexpr int COL_SPMV_PARTS = 4;
template <class T>
__global__ __launch_bounds__(REDUCE_THREADS) void columnSpmvDotKernel(size_t slots, const SliceLinks *links,
                                                                      ColumnMatrix<T> A, const T *__restrict__ x,
                                                                      T *__restrict__ y, double *partial) {
    const unsigned L = reduceLogicalBlock();
    const size_t span = reduceSpan(slots, gridDim.x);
    const size_t lo = (size_t)L * span, hi = lo + span < slots ? lo + span : slots;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    double acc = 0.0;
    for (size_t b = lo + (size_t)wave * 64; b < hi; b += COL_SPMV_PARTS * REDUCE_THREADS) {
        T s[COL_SPMV_PARTS];
#pragma unroll
        for (int u = 0; u < COL_SPMV_PARTS; u++) {
            size_t e = b + (size_t)u * REDUCE_THREADS;
            if (e >= hi) e = b;
            s[u] = columnProduct<T>(links[e / COL_SLICE], e + lane, (int)(e % COL_SLICE) + lane, A, x);
        }
#pragma unroll
        for (int u = 0; u < COL_SPMV_PARTS; u++) {
            const size_t e = b + (size_t)u * REDUCE_THREADS + lane;
            if (b + (size_t)u * REDUCE_THREADS < hi) {
                y[e] = s[u];
                acc += (double)x[e] * (double)s[u];
            }
        }
    }
    acc = reduceFold<0>(acc);
    if (threadIdx.x == 0) partial[L] = acc;
}

// The same for the next direction z + a s, which each slot forms for itself and
// for its neighbours as it needs them (from cache), so no pass over the vectors
// and no launch comes between the preconditioner and the product.  Bound by
// memory at large sizes, by its launch at small ones.  A solve, with a launch of
// its own for the direction before: 64^3 7.0 -> 6.8 ms, 128^3 17.8 -> 17.1, 256^3
// 77.0 -> 77.4 (the same).  Two slots a lane in flight changed nothing.
template <class T, class Z>
struct NextDirection {
    const Z *__restrict__ z;
    const T *__restrict__ s;
    T a;
    __device__ __forceinline__ T operator[](size_t e) const {
        T v = (T)z[e];
        v += a * s[e];
        return v;
    }
};
template <class T, class Z>
__global__ __launch_bounds__(REDUCE_THREADS) void columnDirectionSpmvDotKernel(
    size_t slots, const SliceLinks *links, ColumnMatrix<T> A, const Z *__restrict__ z, const T *__restrict__ s,
    T *__restrict__ t, T *__restrict__ y, const double *zrPartial, int nzr, const double *rho, double *rhoNew,
    double *partial) {
    const double num = foldPartials<0>(zrPartial, nzr);
    __syncthreads();  // the second fold below takes the same LDS
    if (blockIdx.x == 0 && threadIdx.x == 0) *rhoNew = num;
    const NextDirection<T, Z> x{z, s, (T)(float)(num / *rho)};
    const unsigned L = reduceLogicalBlock();
    const size_t span = reduceSpan(slots, gridDim.x);
    const size_t lo = (size_t)L * span, hi = lo + span < slots ? lo + span : slots;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
    double acc = 0.0;
    for (size_t b = lo + (size_t)wave * 64; b < hi; b += REDUCE_THREADS) {
        const size_t e = b + lane;
        const T p = columnProduct<T>(links[b / COL_SLICE], e, (int)(b % COL_SLICE) + lane, A, x);
        const T v = x[e];
        t[e] = v;
        y[e] = p;
        acc += (double)v * (double)p;
    }
    acc = reduceFold<0>(acc);
    if (threadIdx.x == 0) partial[L] = acc;
}

// y = A x (b null) or y = b - A x
template <class T>
__global__ __launch_bounds__(256) void columnResidualKernel(size_t slots, const SliceLinks *links, ColumnMatrix<T> A,
                                                            const T *b, const T *x, T *y) {
    const unsigned g = gridDim.x, lb = g % XCDS == 0 ? (blockIdx.x % XCDS) * (g / XCDS) + blockIdx.x / XCDS : blockIdx.x;
    const size_t e0 = (size_t)lb * 256 + (size_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x / 64) * 64;
    const int lane = threadIdx.x % 64;
    if (e0 >= slots) return;
    const T s = columnProduct<T>(links[e0 / COL_SLICE], e0 + lane, (int)(e0 % COL_SLICE) + lane, A, x);
    y[e0 + lane] = b ? b[e0 + lane] - s : s;
}

template <class T, bool FWD>
__global__ __launch_bounds__(COL_LANES *COL_WAVES) void columnSweepKernel(ColumnArgs<T, MicRec<T>> a,
                                                                          ColumnPublish pub) {
    if (pub.rmax && blockIdx.x == 0) {
        publishMax(pub.rmax, pub.n, pub.host);
        return;
    }
    columnSweep<T, MicRec<T>, CPF, CPX, FWD>(a, (int)threadIdx.x);
}

template <class T, bool FWD>
void columnSweepLaunch(ColumnPlan &cp, const T *in, T *out, const MicRec<T> *rec, ColumnPublish pub, hipStream_t st) {
    const unsigned tiles = (unsigned)cp.ntj * cp.ntk;
    if (++cp.epoch == 0) cp.epoch = 1;  // 0 tags the cleared buffer
    ColumnArgs<T, MicRec<T>> a{cp.ncj, cp.nck,     cp.ntj,     cp.ntk,   cp.cols,  cp.order, in,           out,         rec,
                               cp.exJ, cp.exK,     cp.exSteps, cp.counter, cp.error, cp.base,  cp.epoch,     WAIT_LOOKS};
    cp.base += tiles;
    // the publishing workgroup takes no ticket
    hipLaunchKernelGGL((columnSweepKernel<T, FWD>), dim3(tiles + (pub.rmax ? 1 : 0)), dim3(COL_LANES * COL_WAVES), 0, st,
                       a, pub);
    hipCheck(hipGetLastError(), "MIC(0) column sweep launch");
}

unsigned slotBlocks(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

void columnShape(Grid g, ColumnPlan &cp) {
    cp.ncj = ceilDiv(g.nj, COL_J);
    cp.nck = ceilDiv(g.nk, COL_K);
    cp.ntj = cp.ncj;
    cp.ntk = ceilDiv(cp.nck, COL_WAVES);
    cp.exSteps = g.ni + COL_SKEW;
    cp.maxSlices = (size_t)cp.ncj * cp.nck * cp.exSteps;
    // four 32-bit parts: a double's two words
    cp.exJWords = (size_t)cp.ncj * cp.ntk * COL_WAVES * cp.exSteps * COL_K * 4;
    cp.exKWords = (size_t)cp.ntj * cp.ntk * cp.exSteps * COL_J * 4;
}

void columnOrder(const ColumnPlan &cp, std::vector<int> &order) {
    order.clear();
    for (int d = 0; d <= cp.ntj + cp.ntk - 2; d++)
        for (int pj = 0; pj < cp.ntj; pj++)
            if (d - pj >= 0 && d - pj < cp.ntk) order.push_back(pj + (d - pj) * cp.ntj);
}

void columnRanges(Grid g, const int *mask, ColumnPlan &cp, hipStream_t s) {
    hipLaunchKernelGGL(columnRangeKernel, dim3(cp.ncj * cp.nck), dim3(256), 0, s, g, mask, cp.ncj, cp.cols);
    hipLaunchKernelGGL(columnScanKernel, dim3(1), dim3(1024), 0, s, cp.cols, cp.ncj * cp.nck, cp.total);
}

void columnFill(Grid g, const PressureSys &S, ColumnPlan &cp, ColumnSys &C, bool floats, hipStream_t s) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(columnLinksKernel, dim3(cp.ncj * cp.nck), dim3(256), 0, s, cp.cols, cp.ncj, cp.nck, cp.links);
    hipLaunchKernelGGL(columnFillKernel<float>, dim3(slotBlocks(cp.slots())), dim3(256), 0, s, g, S, cp.slices, cp.links,
                       cp.ncj, cp.slotRow, C.rhs, C.diag, C.ox, C.oy, C.oz, floats ? C.fdiag : nullptr, C.fox, C.foy,
                       C.foz);
}

void columnRecords(const PressureSys &S, const ColumnPlan &cp, ColumnSys &C, bool fp64, hipStream_t s) {
    if (cp.slices == 0) return;
    if (fp64)
        hipLaunchKernelGGL(columnRecordsKernel<double>, dim3(slotBlocks(cp.slots())), dim3(256), 0, s, S, cp.slots(),
                           cp.slotRow, C.recFwd, C.recBwd);
    else
        hipLaunchKernelGGL(columnRecordsKernel<float>, dim3(slotBlocks(cp.slots())), dim3(256), 0, s, S, cp.slots(),
                           cp.slotRow, C.frecFwd, C.frecBwd);
}

template <class T>
void slotsFromRows(const ColumnPlan &cp, const T *rows, T *slots, hipStream_t s) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(slotsFromRowsKernel<T>, dim3(ceilDiv(cp.slices, TURN)), dim3(256), 0, s, cp.slots(), cp.slotRow,
                       rows, slots);
}
template <class T>
void rowsFromSlots(const ColumnPlan &cp, const T *slots, T *rows, hipStream_t s) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(rowsFromSlotsKernel<T>, dim3(ceilDiv(cp.slices, TURN)), dim3(256), 0, s, cp.slots(), cp.slotRow,
                       slots, rows);
}
template void slotsFromRows<float>(const ColumnPlan &, const float *, float *, hipStream_t);
template void slotsFromRows<double>(const ColumnPlan &, const double *, double *, hipStream_t);
template void rowsFromSlots<float>(const ColumnPlan &, const float *, float *, hipStream_t);
template void rowsFromSlots<double>(const ColumnPlan &, const double *, double *, hipStream_t);

void slotsFromCells(const PressureSys &S, const ColumnPlan &cp, const float *cells, double *slots, hipStream_t s) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(slotsFromCellsKernel, dim3(slotBlocks(cp.slots())), dim3(256), 0, s, cp.slots(), cp.slotRow,
                       S.rows, cells, slots);
}
template <class T>
void cellsFromSlots(const PressureSys &S, const ColumnPlan &cp, const double *slots, T *cells, hipStream_t s) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(cellsFromSlotsKernel<T>, dim3(slotBlocks(cp.slots())), dim3(256), 0, s, cp.slots(), cp.slotRow,
                       S.rows, slots, cells);
}
template void cellsFromSlots<float>(const PressureSys &, const ColumnPlan &, const double *, float *, hipStream_t);
template void cellsFromSlots<double>(const PressureSys &, const ColumnPlan &, const double *, double *, hipStream_t);

template <class T>
static void launchColumnSpmvDot(const ColumnPlan &cp, ColumnMatrix<T> A, const T *x, T *y, double *partial,
                                hipStream_t st) {
    if (cp.slices == 0) return;
    hipLaunchKernelGGL(columnSpmvDotKernel<T>, dim3(reduceBlocks(cp.slots())), dim3(REDUCE_THREADS), 0, st, cp.slots(),
                       cp.links, A, x, y, partial);
}
void columnSpmvDot(const ColumnPlan &cp, const ColumnSys &C, const double *x, double *y, double *partial,
                   hipStream_t st) {
    launchColumnSpmvDot<double>(cp, ColumnMatrix<double>{C.diag, C.ox, C.oy, C.oz}, x, y, partial, st);
}
void columnSpmvDotF(const ColumnPlan &cp, const ColumnSys &C, const float *x, float *y, double *partial,
                    hipStream_t st) {
    launchColumnSpmvDot<float>(cp, ColumnMatrix<float>{C.fdiag, C.fox, C.foy, C.foz}, x, y, partial, st);
}
template <class T, class Z>
void columnDirectionSpmvDot(const ColumnPlan &cp, const ColumnSys &C, const Z *z, const T *s, T *t, T *q,
                            const double *zr, int nzr, const double *rho, double *rhoNew, double *partial,
                            hipStream_t st) {
    if (cp.slices == 0) return;
    ColumnMatrix<T> A;
    if constexpr (sizeof(T) == 8)
        A = ColumnMatrix<T>{C.diag, C.ox, C.oy, C.oz};
    else
        A = ColumnMatrix<T>{C.fdiag, C.fox, C.foy, C.foz};
    hipLaunchKernelGGL((columnDirectionSpmvDotKernel<T, Z>), dim3(reduceBlocks(cp.slots())), dim3(REDUCE_THREADS), 0, st,
                       cp.slots(), cp.links, A, z, s, t, q, zr, nzr, rho, rhoNew, partial);
}
template void columnDirectionSpmvDot(const ColumnPlan &, const ColumnSys &, const double *, const double *, double *,
                                     double *, const double *, int, const double *, double *, double *, hipStream_t);
template void columnDirectionSpmvDot(const ColumnPlan &, const ColumnSys &, const float *, const double *, double *,
                                     double *, const double *, int, const double *, double *, double *, hipStream_t);
template void columnDirectionSpmvDot(const ColumnPlan &, const ColumnSys &, const float *, const float *, float *,
                                     float *, const double *, int, const double *, double *, double *, hipStream_t);
void columnResidual(const ColumnPlan &cp, const ColumnSys &C, const double *b, const double *x, double *r,
                    hipStream_t st) {
    if (cp.slices == 0) return;
    const unsigned nb = (slotBlocks(cp.slots()) + XCDS - 1) / XCDS * XCDS;
    hipLaunchKernelGGL(columnResidualKernel<double>, dim3(nb), dim3(256), 0, st, cp.slots(), cp.links,
                       ColumnMatrix<double>{C.diag, C.ox, C.oy, C.oz}, b, x, r);
}

void columnForward(ColumnPlan &cp, const ColumnSys &C, const double *r, double *y, hipStream_t s, ColumnPublish pub) {
    if (cp.slices > 0) columnSweepLaunch<double, true>(cp, r, y, C.recFwd, pub, s);
}
void columnForward(ColumnPlan &cp, const ColumnSys &C, const float *r, float *y, hipStream_t s, ColumnPublish pub) {
    if (cp.slices > 0) columnSweepLaunch<float, true>(cp, r, y, C.frecFwd, pub, s);
}
void columnBackward(ColumnPlan &cp, const ColumnSys &C, const double *y, double *z, hipStream_t s) {
    if (cp.slices > 0) columnSweepLaunch<double, false>(cp, y, z, C.recBwd, ColumnPublish{}, s);
}
void columnBackward(ColumnPlan &cp, const ColumnSys &C, const float *y, float *z, hipStream_t s) {
    if (cp.slices > 0) columnSweepLaunch<float, false>(cp, y, z, C.frecBwd, ColumnPublish{}, s);
}

}  // namespace ff
