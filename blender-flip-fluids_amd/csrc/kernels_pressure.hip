// kernels_pressure.hip -- the variational pressure solve of the FLIP substep:
// pressure-cell rows, divergence and 7-point ghost-fluid assembly, the MIC(0)
// factor, its hyperplane-scheduled triangular solves and the PCG vector ops.
// (The solver's matrix product and sweeps: kernels_column.hip.)
//
// Rows keep the reference's order (interior liquid cells in k,j,i order,
// pressuresolver.cpp:118-159).  The factor and both triangular sweeps depend
// only on the -x/-y/-z (or +x/+y/+z) neighbours, which sit on the previous
// (next) i+j+k hyperplane, so running the rows hyperplane by hyperplane
// performs the reference's own serial recurrences (pcgsolver.h:68-241) with
// identical operations per row.
#include "kernels.h"

namespace ff {

namespace {

unsigned blocksFor(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }
constexpr int TPB = 256;

__global__ void maskKernel(Grid g, const float *phi, int *mask) {
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t n = (size_t)g.ni * g.nj * g.nk;
    if (c > n) return;
    if (c == n) {
        mask[n] = 0;
        return;
    }
    int i = (int)(c % g.ni), j = (int)((c / g.ni) % g.nj), k = (int)(c / ((size_t)g.ni * g.nj));
    bool interior = i >= 1 && j >= 1 && k >= 1 && i < g.ni - 1 && j < g.nj - 1 && k < g.nk - 1;
    mask[c] = (interior && phi[c] < 0) ? 1 : 0;
}

__global__ void rowsKernel(size_t n, const int *mask, const int *rowOf, int *rows, int *cellRow) {
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    int row = mask[c] ? rowOf[c] : -1;
    cellRow[c] = row;
    if (row >= 0) rows[row] = (int)c;
}

// _calculateNegativeDivergenceVectorThread (pressuresolver.cpp:624-713) and
// _calculateMatrixCoefficientsThread (767-867).  Static solids have zero face
// velocity, so the divergence's solid terms add +-0.0 to a sum that is never
// -0.0 and are left out; a moving solid's (T.us given) are added with the
// cell weight.  Density is 1 (fluidsimulation.cpp:6214).  An
// off-diagonal entry exists when the neighbour is liquid and a pressure row
// (SparseMatrix::add ignores -1, sparsematrix.h:94-96).
__global__ void assembleKernel(Grid g, double dt, const float *u, const float *v, const float *w,
                               const float *wu, const float *wv, const float *ww, const float *phi,
                               const int *mask, const int *rowOf, PressureSys S, SolidTerms T,
                               TensionView tv) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= S.m) return;
    const int ni = g.ni, nj = g.nj;
    int c = S.rows[r];
    int i = c % ni, j = (c / ni) % nj, k = c / (ni * nj);
    const double factor = 1.0 / g.dx;
    const double mfactor = dt / (g.dx * g.dx);
    const double eps = 1e-9, maxtheta = 25;
    double volRight = wu[flat(i + 1, j, k, ni + 1, nj)], volLeft = wu[flat(i, j, k, ni + 1, nj)];
    double volTop = wv[flat(i, j + 1, k, ni, nj + 1)], volBottom = wv[flat(i, j, k, ni, nj + 1)];
    double volFront = ww[flat(i, j, k + 1, ni, nj)], volBack = ww[flat(i, j, k, ni, nj)];
    double div = 0.0;
    div += -factor * volRight * (double)u[flat(i + 1, j, k, ni + 1, nj)];
    div += factor * volLeft * (double)u[flat(i, j, k, ni + 1, nj)];
    div += -factor * volTop * (double)v[flat(i, j + 1, k, ni, nj + 1)];
    div += factor * volBottom * (double)v[flat(i, j, k, ni, nj + 1)];
    div += -factor * volFront * (double)w[flat(i, j, k + 1, ni, nj)];
    div += factor * volBack * (double)w[flat(i, j, k, ni, nj)];
    if (T.us) {
        const double volCenter = T.wc[c];
        div += factor * (volRight - volCenter) * (double)T.us[flat(i + 1, j, k, ni + 1, nj)];
        div += -factor * (volLeft - volCenter) * (double)T.us[flat(i, j, k, ni + 1, nj)];
        div += factor * (volTop - volCenter) * (double)T.vs[flat(i, j + 1, k, ni, nj + 1)];
        div += -factor * (volBottom - volCenter) * (double)T.vs[flat(i, j, k, ni, nj + 1)];
        div += factor * (volFront - volCenter) * (double)T.ws[flat(i, j, k + 1, ni, nj)];
        div += -factor * (volBack - volCenter) * (double)T.ws[flat(i, j, k, ni, nj)];
    }
    if (tv.status) {  // surface tension (pressuresolver.cpp:659-710)
        const double stfactor = dt / (g.dx * g.dx);
        const double pc = phi[c];
        auto add = [&](int a, int b, int e, double vol) {
            const double pn = phi[flat(a, b, e, ni, nj)];
            if (pn >= 0.0) {
                const double t = tensionTerm(g, tv, i, j, k, a, b, e);
                double theta = (pc - pn) / (pc + eps);
                theta = fmax(-maxtheta, fmin(theta, maxtheta));
                div += stfactor * vol * theta * t;
            }
        };
        add(i + 1, j, k, volRight);
        add(i - 1, j, k, volLeft);
        add(i, j + 1, k, volTop);
        add(i, j - 1, k, volBottom);
        add(i, j, k + 1, volFront);
        add(i, j, k - 1, volBack);
    }
    S.rhs[r] = div;

    const double rho = (1.0 + 1.0) / 2.0;
    double phiC = phi[c];
    const size_t sx = 1, sy = (size_t)ni, sz = (size_t)ni * nj;
    double diag = (volRight / rho + volLeft / rho + volTop / rho + volBottom / rho + volFront / rho +
                   volBack / rho) * mfactor;
    int *nb = S.nbr + (size_t)6 * r;
    double off[6] = {0, 0, 0, 0, 0, 0};
    const double vols[6] = {volLeft, volRight, volBottom, volTop, volBack, volFront};
    const long long steps[6] = {-(long long)sx, (long long)sx, -(long long)sy, (long long)sy,
                                -(long long)sz, (long long)sz};
    // reference neighbour order: +x, -x, +y, -y, +z, -z
    const int order[6] = {1, 0, 3, 2, 5, 4};
#pragma unroll
    for (int q = 0; q < 6; q++) {
        int sl = order[q];
        size_t nc = (size_t)((long long)c + steps[sl]);
        double phiN = phi[nc];
        nb[sl] = -1;
        if (phiN < 0.0) {
            if (mask[nc]) {
                nb[sl] = rowOf[nc];
                off[sl] = -(vols[sl] / rho) * mfactor;
            }
        } else {
            double theta = phiN / (phiC + eps);
            theta = fmax(-maxtheta, fmin(theta, maxtheta));
            diag -= (vols[sl] / rho) * mfactor * theta;
        }
    }
    diag = fmax(diag, 0.0);
    S.diag[r] = diag;
    // the -x/-y/-z entries are the neighbour rows' +x/+y/+z ones: both rows
    // compute -(weight / rho) * dt / dx^2 from the shared face
    S.ox[r] = off[1];
    S.oy[r] = off[3];
    S.oz[r] = off[5];
}

__global__ void levelCountKernel(Grid g, PressureSys S) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= S.m) return;
    int c = S.rows[r];
    int l = c % g.ni + (c / g.ni) % g.nj + c / (g.ni * g.nj);
    atomicAdd(&S.levelCount[l], 1);
}
__global__ void levelScatterKernel(Grid g, PressureSys S) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= S.m) return;
    int c = S.rows[r];
    int l = c % g.ni + (c / g.ni) % g.nj + c / (g.ni * g.nj);
    int slot = atomicAdd(&S.levelFill[l], 1);
    S.levelRows[S.levelStart[l] + slot] = r;
}

// factorModifiedIncompleteColesky0 (pcgsolver.h:68-205), omega 0.97, min
// diagonal ratio 0.25, one hyperplane of rows: every row pulls its updates
// from the -z, -y, -x neighbour columns (ascending column order); within a
// column the "missing" sum runs over the column's other rows in ascending row
// order (+x, +y, +z).  A row whose diagonal is below 1e-9 is null: it keeps
// its updated diagonal and contributes nothing as a column.
__global__ void mic0LevelKernel(PressureSys S, const int *rows, int count) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    int j = rows[t];
    const int *nb = S.nbr + (size_t)6 * j;
    double a = S.diag[j];
    if (a < 1e-9) a = 0;
    double d = a;
    const int cslots[3] = {4, 2, 0};
#pragma unroll
    for (int q = 0; q < 3; q++) {
        int k = nb[cslots[q]];
        if (k < 0) continue;
        if (S.diag[k] < 1e-9) continue;
        int jslot = cslots[q] + 1;
        const int *kb = S.nbr + (size_t)6 * k;
        double ik = S.invdiag[k];
        double okx = S.ox[k], oky = S.oy[k], okz = S.oz[k];
        double Ljk = (jslot == 1 ? okx : (jslot == 3 ? oky : okz)) * ik;
        d -= Ljk * Ljk;
        double missing = 0;
        if (jslot != 1 && kb[1] >= 0) missing += okx * ik;
        if (jslot != 3 && kb[3] >= 0) missing += oky * ik;
        if (jslot != 5 && kb[5] >= 0) missing += okz * ik;
        d -= 0.97 * Ljk * missing;
    }
    double inv;
    if (a == 0)
        inv = d;
    else if (d < 0.25 * a)
        inv = 1 / sqrt(a);
    else
        inv = 1 / sqrt(d);
    S.invdiag[j] = inv;
}

// L entries toward +x/+y/+z: A * invdiag, or A itself for a null column
__global__ void lfactorKernel(PressureSys S) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= S.m) return;
    bool null = S.diag[r] < 1e-9;
    double iv = S.invdiag[r];
    S.lx[r] = null ? S.ox[r] : S.ox[r] * iv;
    S.ly[r] = null ? S.oy[r] : S.oy[r] * iv;
    S.lz[r] = null ? S.oz[r] : S.oz[r] * iv;
}

// solveLower (pcgsolver.h:211-224), one hyperplane: subtractions in column
// order -z, -y, -x, then the scaling by invdiag
template <class T>
__global__ void forwardLevelKernel(const int *nbr, const T *invdiag, const T *lx, const T *ly,
                                   const T *lz, const int *rows, int count, const T *rv, T *z) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    int j = rows[t];
    const int *nb = nbr + (size_t)6 * j;
    T y = rv[j];
    int k = nb[4];
    if (k >= 0) y -= lz[k] * z[k];
    k = nb[2];
    if (k >= 0) y -= ly[k] * z[k];
    k = nb[0];
    if (k >= 0) y -= lx[k] * z[k];
    z[j] = y * invdiag[j];
}
// solveLowerTransposeInPlace (pcgsolver.h:227-241), one hyperplane
template <class T>
__global__ void backwardLevelKernel(const int *nbr, const T *invdiag, const T *lx, const T *ly,
                                    const T *lz, const int *rows, int count, T *z) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= count) return;
    int i = rows[t];
    const int *nb = nbr + (size_t)6 * i;
    T x = z[i];
    int r = nb[1];
    if (r >= 0) x -= lx[i] * z[r];
    r = nb[3];
    if (r >= 0) x -= ly[i] * z[r];
    r = nb[5];
    if (r >= 0) x -= lz[i] * z[r];
    z[i] = x * invdiag[i];
}

// x += a s; r -= a q with a = rho / (s . q) the float-rounded step, and the
// partial max |r|
template <class TX, class T>
__global__ __launch_bounds__(REDUCE_THREADS) void pcgStepKernel(TX *x, const T *s, T *r, const T *q, size_t n,
                                                                const double *rho, const double *sqPartial, int nsq,
                                                                double *partial, float *rf) {
    const double a = *rho / foldPartials<0>(sqPartial, nsq);
    const float fa = (float)a, fna = (float)(-a);
    const unsigned L = reduceLogicalBlock();
    const size_t span = reduceSpan(n, gridDim.x);
    const size_t lo = (size_t)L * span, hi = lo + span < n ? lo + span : n;
    double acc = 0.0;
    for (size_t i = lo + threadIdx.x; i < hi; i += REDUCE_THREADS) {
        x[i] += (TX)fa * (TX)s[i];
        const T ri = r[i] + (T)fna * q[i];
        r[i] = ri;
        if (rf) rf[i] = (float)ri;  // FP32 copy for an FP32 preconditioner
        acc = fmax(acc, fabs((double)ri));
    }
    acc = reduceFold<1>(acc);
    if (threadIdx.x == 0) partial[L] = acc;
}

// the search direction z + (float)(rhoNew / rho) s, into z; rhoNew = z . r from
// its partials, stored for the next step
__global__ __launch_bounds__(REDUCE_THREADS) void pcgDirectionKernel(double *z, const double *s, size_t n,
                                                                     const double *zrPartial, int nzr,
                                                                     const double *rho, double *rhoNew) {
    const double num = foldPartials<0>(zrPartial, nzr);
    const float fa = (float)(num / *rho);
    const size_t span = reduceSpan(n, gridDim.x);
    const size_t lo = (size_t)reduceLogicalBlock() * span, hi = lo + span < n ? lo + span : n;
    for (size_t q = lo + threadIdx.x; q < hi; q += REDUCE_THREADS) z[q] += (double)fa * s[q];
    if (blockIdx.x == 0 && threadIdx.x == 0) *rhoNew = num;
}

__global__ void gatherRowsKernel(int m, const int *rows, const double *cells, double *rhs) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < m) rhs[r] = cells[rows[r]];
}
__global__ void castKernel(const double *a, float *b, size_t n) {
    size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) b[q] = (float)a[q];
}
__global__ void addFloatKernel(double *x, const float *d, size_t n) {
    size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) x[q] += (double)d[q];
}

}  // namespace

void pressureMask(Grid g, const float *phi, int *mask, hipStream_t s) {
    size_t n = (size_t)g.ni * g.nj * g.nk;
    hipLaunchKernelGGL(maskKernel, dim3(blocksFor(n + 1, TPB)), dim3(TPB), 0, s, g, phi, mask);
}

void pressureRows(Grid g, const int *mask, const int *rowOf, int *rows, int *cellRow, hipStream_t s) {
    size_t n = (size_t)g.ni * g.nj * g.nk;
    hipLaunchKernelGGL(rowsKernel, dim3(blocksFor(n, TPB)), dim3(TPB), 0, s, n, mask, rowOf, rows, cellRow);
}

void pressureAssemble(Grid g, double dt, const float *u, const float *v, const float *w,
                      const float *wu, const float *wv, const float *ww, const float *phi,
                      PressureSys &S, hipStream_t s, SolidTerms solid, TensionView tension) {
    if (S.m == 0) return;
    hipLaunchKernelGGL(assembleKernel, dim3(blocksFor(S.m, TPB)), dim3(TPB), 0, s, g, dt, u, v, w, wu,
                       wv, ww, phi, S.mask, S.rowOf, S, solid, tension);
}

void pressureLevels(Grid g, PressureSys &S, int *scanScratch, hipStream_t s) {
    S.nLevels = g.ni + g.nj + g.nk - 2;
    hipCheck(hipMemsetAsync(S.levelCount, 0, sizeof(int) * (S.nLevels + 1), s), "hipMemsetAsync");
    if (S.m > 0)
        hipLaunchKernelGGL(levelCountKernel, dim3(blocksFor(S.m, TPB)), dim3(TPB), 0, s, g, S);
    exclusiveScan(S.levelCount, S.levelStart, S.nLevels, scanScratch, s);
}

void pressureLevelRows(Grid g, PressureSys &S, hipStream_t s) {
    hipCheck(hipMemsetAsync(S.levelFill, 0, sizeof(int) * S.nLevels, s), "hipMemsetAsync");
    if (S.m > 0)
        hipLaunchKernelGGL(levelScatterKernel, dim3(blocksFor(S.m, TPB)), dim3(TPB), 0, s, g, S);
}

void mic0Factor(PressureSys &S, const int *hs, hipStream_t s) {
    for (int l = 0; l < S.nLevels; l++) {
        int cnt = hs[l + 1] - hs[l];
        if (cnt == 0) continue;
        hipLaunchKernelGGL(mic0LevelKernel, dim3(blocksFor(cnt, TPB)), dim3(TPB), 0, s, S,
                           S.levelRows + hs[l], cnt);
    }
    mic0LFactor(S, s);
}

void mic0LFactor(PressureSys &S, hipStream_t s) {
    if (S.m > 0) hipLaunchKernelGGL(lfactorKernel, dim3(blocksFor(S.m, TPB)), dim3(TPB), 0, s, S);
}

template <class T>
static void micApply(const PressureSys &S, const int *hs, const T *invdiag, const T *lx, const T *ly,
                     const T *lz, const T *r, T *z, hipStream_t s) {
    for (int l = 0; l < S.nLevels; l++) {
        int cnt = hs[l + 1] - hs[l];
        if (cnt == 0) continue;
        hipLaunchKernelGGL(forwardLevelKernel<T>, dim3(blocksFor(cnt, TPB)), dim3(TPB), 0, s, S.nbr,
                           invdiag, lx, ly, lz, S.levelRows + hs[l], cnt, r, z);
    }
    for (int l = S.nLevels - 1; l >= 0; l--) {
        int cnt = hs[l + 1] - hs[l];
        if (cnt == 0) continue;
        hipLaunchKernelGGL(backwardLevelKernel<T>, dim3(blocksFor(cnt, TPB)), dim3(TPB), 0, s, S.nbr,
                           invdiag, lx, ly, lz, S.levelRows + hs[l], cnt, z);
    }
}

void mic0Apply(const PressureSys &S, const int *hs, const double *r, double *z, hipStream_t s) {
    micApply<double>(S, hs, S.invdiag, S.lx, S.ly, S.lz, r, z, s);
}
void mic0ApplyF(const PressureSys &S, const int *hs, const float *r, float *z, hipStream_t s) {
    micApply<float>(S, hs, S.finvdiag, S.flx, S.fly, S.flz, r, z, s);
}

template <class TX, class T>
static void launchPcgStep(TX *x, const T *s, T *r, const T *q, size_t n, const double *rho, const double *sq, int nsq,
                          double *rmax, hipStream_t st, float *rf = nullptr) {
    if (n == 0) return;
    hipLaunchKernelGGL((pcgStepKernel<TX, T>), dim3(reduceBlocks(n)), dim3(REDUCE_THREADS), 0, st, x, s, r, q, n, rho,
                       sq, nsq, rmax, rf);
}
void pcgStep(double *x, const double *s, double *r, const double *q, size_t n, const double *rho, const double *sq,
             int nsq, double *rmax, hipStream_t st, float *rf) {
    launchPcgStep<double, double>(x, s, r, q, n, rho, sq, nsq, rmax, st, rf);
}
void pcgStepF(float *x, const float *s, float *r, const float *q, size_t n, const double *rho, const double *sq, int nsq,
              double *rmax, hipStream_t st) {
    launchPcgStep<float, float>(x, s, r, q, n, rho, sq, nsq, rmax, st);
}
void pcgStepMixed(double *x, const float *s, float *r, const float *q, size_t n, const double *rho, const double *sq,
                  int nsq, double *rmax, hipStream_t st) {
    launchPcgStep<double, float>(x, s, r, q, n, rho, sq, nsq, rmax, st);
}

void pcgDirection(double *z, const double *s, size_t n, const double *zr, int nzr, const double *rho, double *rhoNew,
                  hipStream_t st) {
    if (n == 0) return;
    hipLaunchKernelGGL(pcgDirectionKernel, dim3(reduceBlocks(n)), dim3(REDUCE_THREADS), 0, st, z, s, n, zr, nzr, rho,
                       rhoNew);
}

void gatherRows(const PressureSys &S, const double *cells, double *rhs, hipStream_t s) {
    if (S.m == 0) return;
    hipLaunchKernelGGL(gatherRowsKernel, dim3(blocksFor(S.m, TPB)), dim3(TPB), 0, s, S.m, S.rows, cells, rhs);
}
void castToFloat(const double *a, float *b, size_t n, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(castKernel, dim3(blocksFor(n, TPB)), dim3(TPB), 0, s, a, b, n);
}
void addFloatToDouble(double *x, const float *d, size_t n, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(addFloatKernel, dim3(blocksFor(n, TPB)), dim3(TPB), 0, s, x, d, n);
}
void mic0ToFloat(PressureSys &S, hipStream_t s) {
    size_t m = S.m;
    castToFloat(S.invdiag, S.finvdiag, m, s);
    castToFloat(S.lx, S.flx, m, s);
    castToFloat(S.ly, S.fly, m, s);
    castToFloat(S.lz, S.flz, m, s);
}

}  // namespace ff
