// pressure.hip -- host side of the GPU pressure solve.
#include "pressure.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>

namespace ff {

void hipCheck(hipError_t e, const char *what);

PressureSolver::~PressureSolver() {
    dropGraph();
    if (_block) (void)hipFree(_block);
    if (_rowBlock) (void)hipFree(_rowBlock);
    if (_hostScal) (void)hipHostFree(_hostScal);
}

namespace {
// consecutive 256-byte aligned parts of one allocation
struct Carver {
    size_t bytes = 0;
    size_t take(size_t n) {
        const size_t off = bytes;
        bytes += (n + 255) / 256 * 256;
        return off;
    }
};
}  // namespace

void PressureSolver::allocate(Grid g) {
    _g = g;
    if (!_hostScal) {
        hipCheck(hipHostMalloc((void **)&_hostScal, 64, hipHostMallocMapped), "hipHostMalloc");
        hipCheck(hipHostGetDevicePointer((void **)&_hostScalDev, _hostScal, 0), "hipHostGetDevicePointer");
    }
    if (_block) (void)hipFree(_block);
    if (_rowBlock) (void)hipFree(_rowBlock);
    _block = _rowBlock = nullptr;
    const size_t N = (size_t)g.ni * g.nj * g.nk;
    const size_t M = maxRows(), L = (size_t)g.ni + g.nj + g.nk;
    Carver b;
    size_t oMask = b.take(4 * (N + 1)), oRowOf = b.take(4 * (N + 1)), oRows = b.take(4 * M), oNbr = b.take(24 * M);
    size_t oCellRow = b.take(4 * N), oError = b.take(4);
    _bandTilesMax = std::max(mic0BandTiles(g, true), mic0BandTiles(g, false));
    size_t oTileLo = b.take(4 * (size_t)_bandTilesMax), oTileHi = b.take(4 * (size_t)_bandTilesMax);
    size_t oLc = b.take(4 * (L + 1)), oLs = b.take(4 * (L + 1));
    size_t oD[9];
    for (auto &o : oD) o = b.take(8 * M);
    columnShape(g, _cp);
    const size_t E = _cp.maxSlices * COL_SLICE;
    size_t oCols = b.take(sizeof(ColumnRange) * (size_t)_cp.ncj * _cp.nck);
    size_t oOrder = b.take(4 * (size_t)_cp.ntj * _cp.ntk);
    size_t oLinks = b.take(sizeof(SliceLinks) * _cp.maxSlices), oSlotRow = b.take(4 * E), oTotal = b.take(4);
    size_t oExJ = b.take(4 * _cp.exJWords), oExK = b.take(4 * _cp.exKWords), oCounter = b.take(4);
    size_t oC[5], oCF[4], oV[6], oFV[4];
    for (auto &o : oC) o = b.take(8 * E);
    for (auto &o : oCF) o = b.take(4 * E);
    for (auto &o : oV) o = b.take(8 * E);
    for (auto &o : oFV) o = b.take(4 * E);
    // one solve's sweeps are of one precision: the FP32 records share the FP64 ones' place
    size_t oRec[2];
    for (auto &o : oRec) o = b.take(sizeof(MicRec<double>) * E);
    size_t oPart = b.take(8 * 4 * 1024), oScal = b.take(8 * 16);
    hipCheck(hipMalloc(&_block, b.bytes), "hipMalloc pressure");
    char *m = (char *)_block;
    _S.mask = (int *)(m + oMask);
    _S.rowOf = (int *)(m + oRowOf);
    _S.rows = (int *)(m + oRows);
    _S.nbr = (int *)(m + oNbr);
    _S.levelCount = (int *)(m + oLc);
    _S.levelStart = (int *)(m + oLs);
    _S.cellRow = (int *)(m + oCellRow);
    _tileLo = (int *)(m + oTileLo);
    _tileHi = (int *)(m + oTileHi);
    _hTileLo.assign(_bandTilesMax, 0);
    _hTileHi.assign(_bandTilesMax, 0);
    double *d[9];
    for (int q = 0; q < 9; q++) d[q] = (double *)(m + oD[q]);
    _S.rhs = d[0]; _S.diag = d[1]; _S.ox = d[2]; _S.oy = d[3]; _S.oz = d[4];
    _S.invdiag = d[5]; _S.lx = d[6]; _S.ly = d[7]; _S.lz = d[8];
    _cp.cols = (ColumnRange *)(m + oCols);
    _cp.order = (int *)(m + oOrder);
    _cp.links = (SliceLinks *)(m + oLinks);
    _cp.slotRow = (int *)(m + oSlotRow);
    _cp.total = (int *)(m + oTotal);
    _cp.exJ = (unsigned *)(m + oExJ);
    _cp.exK = (unsigned *)(m + oExK);
    _cp.counter = (unsigned *)(m + oCounter);
    _cp.error = (int *)(m + oError);
    _cp.base = _cp.epoch = 0;
    _cp.slices = 0;
    _C.rhs = (double *)(m + oC[0]); _C.diag = (double *)(m + oC[1]);
    _C.ox = (double *)(m + oC[2]); _C.oy = (double *)(m + oC[3]); _C.oz = (double *)(m + oC[4]);
    _C.fdiag = (float *)(m + oCF[0]); _C.fox = (float *)(m + oCF[1]);
    _C.foy = (float *)(m + oCF[2]); _C.foz = (float *)(m + oCF[3]);
    _C.recFwd = (MicRec<double> *)(m + oRec[0]); _C.recBwd = (MicRec<double> *)(m + oRec[1]);
    _C.frecFwd = (MicRec<float> *)(m + oRec[0]); _C.frecBwd = (MicRec<float> *)(m + oRec[1]);
    _x = (double *)(m + oV[0]); _r = (double *)(m + oV[1]); _z = (double *)(m + oV[2]); _s = (double *)(m + oV[3]);
    _y = (double *)(m + oV[4]);
    _t0 = (double *)(m + oV[5]);
    _fr = (float *)(m + oFV[0]); _fz = (float *)(m + oFV[1]); _fs = (float *)(m + oFV[2]);
    _fy = (float *)(m + oFV[3]);
    // of no use to the modes with FP32 vectors: places of theirs
    _fd = (float *)_t0;
    _fq = _fd + E;
    _ft = (float *)_s;
    _S.ni = g.ni;
    _S.nj = g.nj;
    _S.nk = g.nk;
    {
        // epoch 0 marks a word no launch has published; the counter starts at
        // 0.  The copy comes last: it waits for the fills, which the solver's
        // own stream would not.
        hipCheck(hipMemset(_cp.exJ, 0, 4 * _cp.exJWords), "clear exchange words");
        hipCheck(hipMemset(_cp.exK, 0, 4 * _cp.exKWords), "clear exchange words");
        hipCheck(hipMemset(_cp.counter, 0, 4), "clear ticket counter");
        std::vector<int> order;
        columnOrder(_cp, order);
        hipCheck(hipMemcpy(_cp.order, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice),
                 "H2D tile order");
    }
    _partial = (double *)(m + oPart);
    _pSq = _partial + 1024;
    _pRmax = _partial + 2048;
    _pZr = _partial + 3072;
    _scal = (double *)(m + oScal);
    _S.m = 0;
    _S.nLevels = g.ni + g.nj + g.nk - 2;
    int dev = 0, wallKHz = 0;
    hipCheck(hipGetDevice(&dev), "hipGetDevice");
    hipCheck(hipDeviceGetAttribute(&wallKHz, hipDeviceAttributeWallClockRate, dev), "device attribute");
    _waitTicks = 2000LL * std::max(wallKHz, 1);  // 2 s
}

size_t PressureSolver::maxRows() const {
    // pressure rows live on interior cells only
    return (size_t)std::max(_g.ni - 2, 1) * std::max(_g.nj - 2, 1) * std::max(_g.nk - 2, 1);
}

// The buffers of the row-ordered schedules, made when one of them is first
// used.
void PressureSolver::ensureRowSchedules() {
    if (_rowBlock) return;
    const Grid g = _g;
    const size_t M = maxRows(), L = (size_t)g.ni + g.nj + g.nk;
    int ti, tj, tk;
    micTileCounts(g, std::min(micTileDepth(true), micTileDepth(false)), ti, tj, tk);
    _maxTiles = ti * tj * tk;
    Carver b;
    size_t oOrder = b.take(4 * (size_t)_maxTiles), oTileRows = b.take(4 * (size_t)_maxTiles);
    size_t oFlags = b.take(4 * (size_t)_maxTiles), oCounter = b.take(4);
    size_t oLf = b.take(4 * L), oLr = b.take(4 * M);
    size_t oD[6], oF[10];
    for (auto &o : oD) o = b.take(8 * M);
    for (auto &o : oF) o = b.take(4 * M);
    size_t oRec64[2], oRec32[2];
    for (auto &o : oRec64) o = b.take(sizeof(MicRec<double>) * M);
    for (auto &o : oRec32) o = b.take(sizeof(MicRec<float>) * M);
    pencilShape(g, _pp.npj, _pp.npk, _pp.nw);
    _pp.np = _pp.npj * _pp.npk;
    size_t oPOrder = b.take(4 * (size_t)_pp.np), oPWords = b.take(sizeof(LineWord) * (size_t)g.nj * g.nk * _pp.nw);
    const size_t exWords = pencilExchangeWords(g);
    size_t oPEx = b.take(8 * exWords), oPCounter = b.take(4);
    int dev = 0, cus = 0, lds = 0;
    hipCheck(hipGetDevice(&dev), "hipGetDevice");
    hipCheck(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "device attribute");
    hipCheck(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev), "device attribute");
    const size_t pencilLds = pencilLdsBytes(g) + 8448;
    if ((size_t)lds < pencilLds)
        throw std::runtime_error("the MIC(0) line pipeline needs " + std::to_string(pencilLds) +
                                 " bytes of LDS per workgroup at this grid size; the device offers " +
                                 std::to_string(lds));
    if ((size_t)lds < micTileLds(true))
        throw std::runtime_error("the MIC(0) tile kernel needs " + std::to_string(micTileLds(true)) +
                                 " bytes of LDS per workgroup; the device offers " + std::to_string(lds));
    hipCheck(hipMalloc(&_rowBlock, b.bytes), "hipMalloc pressure (row schedules)");
    char *m = (char *)_rowBlock;
    _ms.g = g;
    _ms.order = (int *)(m + oOrder);
    _ms.tileRows = (int *)(m + oTileRows);
    _ms.flags = (int *)(m + oFlags);
    _ms.counter = (int *)(m + oCounter);
    _ms.error = _cp.error;
    _ms.grid = std::max(cus, 1);
    _ms.waitTicks = _waitTicks;
    _S.levelFill = (int *)(m + oLf);
    _S.levelRows = (int *)(m + oLr);
    double *d[6];
    for (int q = 0; q < 6; q++) d[q] = (double *)(m + oD[q]);
    _S.lmx = d[0]; _S.lmy = d[1]; _S.lmz = d[2];
    _rowR = d[3]; _rowY = d[4]; _rowZ = d[5];
    float *f[10];
    for (int q = 0; q < 10; q++) f[q] = (float *)(m + oF[q]);
    _S.finvdiag = f[0]; _S.flx = f[1]; _S.fly = f[2]; _S.flz = f[3];
    _S.flmx = f[4]; _S.flmy = f[5]; _S.flmz = f[6];
    _rowFR = f[7]; _rowFY = f[8]; _rowFZ = f[9];
    _S.recFwd = (MicRec<double> *)(m + oRec64[0]);
    _S.recBwd = (MicRec<double> *)(m + oRec64[1]);
    _S.frecFwd = (MicRec<float> *)(m + oRec32[0]);
    _S.frecBwd = (MicRec<float> *)(m + oRec32[1]);
    _pp.order = (int *)(m + oPOrder);
    _pp.words = (LineWord *)(m + oPWords);
    _pp.ex = (unsigned long long *)(m + oPEx);
    _pp.counter = (unsigned *)(m + oPCounter);
    _pp.error = _cp.error;
    _pp.waitTicks = _waitTicks;
    _pp.base = _pp.epoch = 0;
    hipCheck(hipMemset(_pp.ex, 0, 8 * exWords), "clear exchange words");
    hipCheck(hipMemset(_pp.counter, 0, 4), "clear ticket counter");
    std::vector<int> order;
    pencilOrder(g, order);
    hipCheck(hipMemcpy(_pp.order, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice),
             "H2D pencil order");
}

// Non-empty tiles of the preconditioner's tile wavefront, listed by tile
// level (any order inside a level), with the flags, ticket counter and error
// word cleared for a new system.
void PressureSolver::buildSchedule(bool fp64, hipStream_t s) {
    _ms.depth = micTileDepth(fp64);
    micTileCounts(_g, _ms.depth, _ms.ti, _ms.tj, _ms.tk);
    _ms.nTiles = _ms.ti * _ms.tj * _ms.tk;
    micMarkTiles(_g, _S, _ms.depth, _ms.tileRows, s);
    _hTileRows.resize(_ms.nTiles);
    hipCheck(hipMemcpyAsync(_hTileRows.data(), _ms.tileRows, sizeof(int) * _ms.nTiles, hipMemcpyDeviceToHost, s),
             "D2H tiles");
    hipCheck(hipStreamSynchronize(s), "sync");
    const int nl = _ms.ti + _ms.tj + _ms.tk;
    std::vector<int> count(nl + 1, 0);
    for (int t = 0; t < _ms.nTiles; t++)
        if (_hTileRows[t]) count[t % _ms.ti + (t / _ms.ti) % _ms.tj + t / (_ms.ti * _ms.tj) + 1]++;
    for (int l = 0; l < nl; l++) count[l + 1] += count[l];
    _hOrder.assign(count[nl], 0);
    for (int t = 0; t < _ms.nTiles; t++)
        if (_hTileRows[t]) _hOrder[count[t % _ms.ti + (t / _ms.ti) % _ms.tj + t / (_ms.ti * _ms.tj)]++] = t;
    _ms.nActive = (int)_hOrder.size();
    if (_ms.nActive > 0)
        hipCheck(hipMemcpyAsync(_ms.order, _hOrder.data(), sizeof(int) * _ms.nActive, hipMemcpyHostToDevice, s),
                 "H2D tile order");
    hipCheck(hipMemsetAsync(_ms.flags, 0, sizeof(int) * _ms.nTiles, s), "memset flags");
    hipCheck(hipMemsetAsync(_ms.counter, 0, sizeof(int), s), "memset counter");
    _ms.base = 0;
    _ms.epoch = 0;
}

// hyperplane range of each band tile's rows, on the device and (after the
// stream's next synchronisation) in _hTileLo/_hTileHi
void PressureSolver::enqueueTileRanges(bool fp64, hipStream_t s) {
    const int nt = mic0BandTiles(_g, fp64);
    mic0BandTileRanges(_g, _S, fp64, _tileLo, _tileHi, s);
    hipCheck(hipMemcpyAsync(_hTileLo.data(), _tileLo, sizeof(int) * nt, hipMemcpyDeviceToHost, s), "D2H tiles");
    hipCheck(hipMemcpyAsync(_hTileHi.data(), _tileHi, sizeof(int) * nt, hipMemcpyDeviceToHost, s), "D2H tiles");
}

void PressureSolver::checkError(hipStream_t s) {
    int e = 0;
    hipCheck(hipMemcpyAsync(&e, _cp.error, sizeof(int), hipMemcpyDeviceToHost, s), "D2H error word");
    hipCheck(hipStreamSynchronize(s), "sync");
    if (e) throw std::runtime_error("MIC(0) preconditioner: a wait for a neighbour's results exceeded its limit");
}

void PressureSolver::setSchedule(int schedule) {
    if (schedule != 2 && schedule != 4 && schedule != 5)
        throw std::domain_error(
            "the solver's preconditioner schedule must be 2 (columns), 4 (line pipeline) or 5 (bands from a graph)");
    _sched = schedule;
}

void PressureSolver::dropGraph() {
    if (_graph) (void)hipGraphExecDestroy(_graph);
    _graph = nullptr;
}

// The band launches of one application are the same for every application
// of a solve (same plan, same buffers), so they are recorded once by stream
// capture and replayed with one hipGraphLaunch.  The capture holds kernel
// launches only.
template <class T>
void PressureSolver::graphApply(const T *r, T *y, T *z, hipStream_t s) {
    if (_S.m == 0) return;
    if (!_graph) {
        hipGraph_t graph = nullptr;
        hipCheck(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed), "begin capture");
        try {
            if constexpr (sizeof(T) == 8)
                mic0ApplyBands(_g, _S, _plan, _tileLo, _tileHi, r, y, z, s);
            else
                mic0ApplyBandsF(_g, _S, _plan, _tileLo, _tileHi, r, y, z, s);
        } catch (...) {
            (void)hipStreamEndCapture(s, &graph);
            if (graph) (void)hipGraphDestroy(graph);
            throw;
        }
        hipCheck(hipStreamEndCapture(s, &graph), "end capture");
        const hipError_t e = hipGraphInstantiate(&_graph, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) _graph = nullptr;
        hipCheck(e, "instantiate the band graph");
    }
    hipCheck(hipGraphLaunch(_graph, s), "launch the band graph");
}

// the row-ordered schedules' operands of the current factor
void PressureSolver::prepareRowSchedule(int schedule, bool fp64, hipStream_t s) {
    ensureRowSchedules();
    if (!fp64) mic0ToFloat(_S, s);
    mic0LowerEntries(_S, fp64, s);
    if (schedule == 4) {
        pencilLineWords(_g, _S, _pp, s);
    } else if (schedule == 0) {
        pressureLevelRows(_g, _S, s);
    } else if (schedule != 1) {
        const bool host = schedule != 3;
        mic0BandPlan(_g, _S, _hLevelStart.data(), fp64, host ? _hTileLo.data() : nullptr,
                     host ? _hTileHi.data() : nullptr, _plan);
        _bandLaunches = (int)_plan.l0.size();
    }
    dropGraph();  // recorded with the previous system's plan
}

// An application in two halves.  The forward half also publishes the largest
// of the PCG step's |r| partials to the host (rmax: those partials, or null):
// a workgroup of its own does it beside the forward sweep, so the host learns
// whether the solve has converged while the sweep runs and enqueues the rest
// of the iteration, or nothing more, before the GPU is through with it.
// Against a stream synchronize and a one-block reduction there: 4.67 -> 4.32 ms
// a frame of a 24^3 pool (30 iterations), 22.7 -> 19.9 ms for two 56^3 solves.
template <class T>
void PressureSolver::precondForward(const T *r, T *y, const double *rmax, hipStream_t s) {
    const int nb = reduceBlocks(_cp.slots());
    if (_sched == 2) {
        columnForward(_cp, _C, r, y, s, rmax ? ColumnPublish{rmax, nb, _hostScalDev} : ColumnPublish{});
        return;
    }
    if (rmax) publishMaximum(rmax, nb, _hostScalDev, s);
    if constexpr (sizeof(T) == 8)
        rowsFromSlots(_cp, r, _rowR, s);
    else
        rowsFromSlots(_cp, r, _rowFR, s);
}
template <class T>
void PressureSolver::precondBackward(const T *y, T *z, hipStream_t s) {
    if (_sched == 2) {
        columnBackward(_cp, _C, y, z, s);
        return;
    }
    if constexpr (sizeof(T) == 8) {
        if (_sched == 4)
            pencilApply(_g, _S, _pp, _rowR, _rowY, _rowZ, s);
        else
            graphApply(_rowR, _rowY, _rowZ, s);
        slotsFromRows(_cp, _rowZ, z, s);
    } else {
        if (_sched == 4)
            pencilApplyF(_g, _S, _pp, _rowFR, _rowFY, _rowFZ, s);
        else
            graphApply(_rowFR, _rowFY, _rowFZ, s);
        slotsFromRows(_cp, _rowFZ, z, s);
    }
}
template <class T>
void PressureSolver::precond(const T *r, T *y, T *z, hipStream_t s) {
    _t->begin(T_MIC0_APPLY, s, applyLaunches(false));
    precondForward<T>(r, y, nullptr, s);
    precondBackward<T>(y, z, s);
    _t->end(T_MIC0_APPLY, s);
}

void PressureSolver::applyPreconditioner(const double *r, double *z, int schedule, hipStream_t s) {
    if (schedule == 2) {
        columnRecords(_S, _cp, _C, true, s);
        slotsFromRows(_cp, r, _r, s);
        columnForward(_cp, _C, _r, _y, s);
        columnBackward(_cp, _C, _y, _z, s);
        rowsFromSlots(_cp, _z, z, s);
        return;
    }
    prepareRowSchedule(schedule, true, s);
    if (schedule == 4) {
        pencilApply(_g, _S, _pp, r, _rowY, z, s);
    } else if (schedule == 1) {
        buildSchedule(true, s);
        micApplyTiles(_S, _ms, r, z, s);
    } else if (schedule == 3 || schedule == 5) {
        mic0ApplyBands(_g, _S, _plan, _tileLo, _tileHi, r, _rowY, z, s);
    } else {
        mic0Apply(_S, _hLevelStart.data(), r, z, s);
    }
}
void PressureSolver::applyPreconditionerF(const float *r, float *z, int schedule, hipStream_t s) {
    if (schedule == 2) {
        columnRecords(_S, _cp, _C, false, s);
        slotsFromRows(_cp, r, _fr, s);
        columnForward(_cp, _C, _fr, _fy, s);
        columnBackward(_cp, _C, _fy, _fz, s);
        rowsFromSlots(_cp, _fz, z, s);
        return;
    }
    prepareRowSchedule(schedule, false, s);
    if (schedule == 4) {
        pencilApplyF(_g, _S, _pp, r, _rowFY, z, s);
    } else if (schedule == 1) {
        buildSchedule(false, s);
        micApplyTilesF(_S, _ms, r, z, s);
    } else if (schedule == 3 || schedule == 5) {
        mic0ApplyBandsF(_g, _S, _plan, _tileLo, _tileHi, r, _rowFY, z, s);
    } else {
        mic0ApplyF(_S, _hLevelStart.data(), r, z, s);
    }
}

// Reads one device scalar.
double PressureSolver::hostScalar(const double *d, hipStream_t s) {
    double h = 0.0;
    hipCheck(hipMemcpyAsync(&h, d, sizeof(double), hipMemcpyDeviceToHost, s), "D2H scalar");
    hipCheck(hipStreamSynchronize(s), "sync");
    return h;
}

namespace {
// what the host's slot holds while no residual has arrived: a NaN that no
// reduction produces
constexpr unsigned long long NO_RESIDUAL = 0x7ff8dead0badbeefull;
}  // namespace

void PressureSolver::armResidual() { *(volatile unsigned long long *)_hostScal = NO_RESIDUAL; }

// The |r|_inf that the forward half of the application publishes to mapped
// pinned host memory while it runs.  The host looks for it without waiting for
// the stream; the stream is asked now and then, so a failed launch ends the
// wait.
double PressureSolver::awaitResidual(hipStream_t s) {
    const volatile unsigned long long *slot = (const volatile unsigned long long *)_hostScal;
    for (unsigned tries = 1;; tries++) {
        const unsigned long long v = *slot;
        if (v != NO_RESIDUAL) {
            double d;
            memcpy(&d, &v, sizeof d);
            return d;
        }
        if (tries % 65536 == 0) {
            const hipError_t e = hipStreamQuery(s);
            if (e == hipErrorNotReady) continue;
            hipCheck(e, "pressure solve");
            if (*slot == NO_RESIDUAL) throw std::runtime_error("the pressure solve's residual did not arrive");
        }
    }
}

// PressureSolver::solve (pressuresolver.cpp:52-92) and _solveLinearSystem (869-916)
PressureResult PressureSolver::solve(double dt, const float *u, const float *v, const float *w,
                                     const float *wu, const float *wv, const float *ww, const float *phi,
                                     double tol, int maxIter, int mode, double innerTol, float *pressure,
                                     int *scanScratch, hipStream_t s, hipEvent_t afterAssembly,
                                     KernelTimers *timers, int referenceDots, const double *cellRhs,
                                     double *cellSolution) {
    PressureResult res;
    _refDots = referenceDots;
    if (cellSolution)
        hipCheck(hipMemsetAsync(cellSolution, 0, sizeof(double) * (size_t)_g.ni * _g.nj * _g.nk, s), "memset");
    _t = timers ? timers : &_noTimers;
    hipCheck(hipMemsetAsync(_cp.error, 0, sizeof(int), s), "memset error word");
    _t->begin(T_ASSEMBLE, s);
    const size_t N = (size_t)_g.ni * _g.nj * _g.nk;
    pressureMask(_g, phi, _S.mask, s);
    exclusiveScan(_S.mask, _S.rowOf, N, scanScratch, s);
    columnRanges(_g, _S.mask, _cp, s);
    int m = 0;
    hipCheck(hipMemcpyAsync(&m, _S.rowOf + N, sizeof(int), hipMemcpyDeviceToHost, s), "D2H");
    hipCheck(hipMemcpyAsync(&_cp.slices, _cp.total, sizeof(int), hipMemcpyDeviceToHost, s), "D2H");
    hipCheck(hipStreamSynchronize(s), "sync");
    _S.m = m;
    res.unknowns = m;
    pressureRows(_g, _S.mask, _S.rowOf, _S.rows, _S.cellRow, s);
    pressureAssemble(_g, dt, u, v, w, wu, wv, ww, phi, _S, s, _solid, _tension);
    if (cellRhs) gatherRows(_S, cellRhs, _S.rhs, s);
    pressureLevels(_g, _S, scanScratch, s);
    columnFill(_g, _S, _cp, _C, mode == 1 || mode == 2, s);
    _t->end(T_ASSEMBLE, s);
    _hLevelStart.resize(_S.nLevels + 1);
    hipCheck(hipMemcpyAsync(_hLevelStart.data(), _S.levelStart, sizeof(int) * (_S.nLevels + 1),
                            hipMemcpyDeviceToHost, s), "D2H levels");
    enqueueTileRanges(mode == 0, s);
    double maxAbs = 0.0;
    if (m > 0) {
        absMax(_C.rhs, _cp.slots(), _partial, _scal + 1, s);
        maxAbs = hostScalar(_scal + 1, s);  // also waits for the level table and the tile ranges
    } else {
        hipCheck(hipStreamSynchronize(s), "sync");
    }
    res.rhsInf = maxAbs;
    if (afterAssembly) hipCheck(hipEventRecord(afterAssembly, s), "event");
    _levelLaunches = mic0FactorBandLaunches(_S, _hLevelStart.data());
    // The forward solve skips a right-hand side below the tolerance as an
    // absolute threshold, as the reference does (pressuresolver.cpp:69-75).  A
    // given right-hand side (the adjoint's) is solved unless it is exactly 0,
    // so the solution stays linear in it at every scale.
    if (cellRhs ? maxAbs == 0.0 : maxAbs < tol) {
        hipCheck(hipMemsetAsync(pressure, 0, sizeof(float) * N, s), "memset");
        res.success = true;
        res.iterations = 0;
        res.error = 0.0;
        return res;
    }
    int iters = 0;
    double resid = -1.0;
    _prevPressure = pressure;
    bool conv = mode == 0   ? pcgFP64(tol, maxIter, maxAbs, iters, resid, s)
                : mode == 1 ? pcgMixed(tol, maxIter, maxAbs, innerTol, iters, resid, s)
                : mode == 2 ? pcgReliable(tol, maxIter, maxAbs, innerTol, iters, resid, s)
                            : pcgPrecond32(tol, maxIter, maxAbs, iters, resid, s);
    checkError(s);
    hipCheck(hipMemsetAsync(pressure, 0, sizeof(float) * N, s), "memset");
    cellsFromSlots(_S, _cp, _x, pressure, s);
    if (cellSolution) cellsFromSlots(_S, _cp, _x, cellSolution, s);
    float e = (float)resid;
    res.success = conv || (iters == maxIter && e < 1.0);
    res.iterations = iters;
    res.error = e;
    return res;
}

// PCGSolver<double>::solve (pcgsolver.h:268-322): x0 = 0, MIC(0), float step
// lengths, |r|_inf stop test against min(tol * |b|_inf, 1.0)
void PressureSolver::initialGuess(hipStream_t st) {
    const size_t n = _cp.slots();
    if (_warm && _prevPressure) {
        slotsFromCells(_S, _cp, _prevPressure, _x, st);
        columnResidual(_cp, _C, _C.rhs, _x, _r, st);
    } else {
        hipCheck(hipMemcpyAsync(_r, _C.rhs, sizeof(double) * n, hipMemcpyDeviceToDevice, st), "copy");
        hipCheck(hipMemsetAsync(_x, 0, sizeof(double) * n, st), "memset");
    }
}

// MIC(0) factor and the operands of the solver's sweeps in fp64 or FP32
void PressureSolver::factor(bool fp64, hipStream_t st) {
    _t->begin(T_MIC0_FACTOR, st, _levelLaunches + 2);
    mic0FactorBands(_g, _S, _hLevelStart.data(), _hTileLo.data(), _hTileHi.data(), _tileLo, _tileHi, st);
    mic0LFactor(_S, st);
    if (_sched == 2)
        columnRecords(_S, _cp, _C, fp64, st);
    else
        prepareRowSchedule(_sched, fp64, st);
    _t->end(T_MIC0_FACTOR, st);
}

void PressureSolver::factorSystem(bool fp64, hipStream_t s) {
    if (_S.m > 0) factor(fp64, s);
}

// a . b in the reference's summation order: over the rows
void PressureSolver::rowDot(const double *a, const double *b, double *out, hipStream_t st) {
    ensureRowSchedules();
    rowsFromSlots(_cp, a, _rowR, st);
    rowsFromSlots(_cp, b, _rowY, st);
    dotReference(_rowR, _rowY, _S.m, _refDots, _partial, out, st);
}

bool PressureSolver::pcgFP64(double tolFactor, int maxIter, double resid0, int &iters, double &resid,
                             hipStream_t st) {
    const size_t n = _cp.slots();
    if (tolFactor < 1e-30) tolFactor = 1e-30;
    initialGuess(st);
    resid = resid0;
    double tol = tolFactor * resid;
    factor(true, st);
    precond(_r, _y, _z, st);
    double *rho = _scal + 2, *rhoNew = _scal + 3;
    // dot products: the reference's order (one partial), or the deterministic tree
    const int nb = _refDots > 0 ? 1 : reduceBlocks(n);
    if (_refDots > 0)
        rowDot(_z, _r, rho, st);
    else
        dot(_z, _r, n, _partial, rho, st);
    double hrho = hostScalar(rho, st);
    if (hrho == 0 || hrho != hrho) {
        iters = 0;
        return false;
    }
    hipCheck(hipMemcpyAsync(_s, _z, sizeof(double) * n, hipMemcpyDeviceToDevice, st), "copy");
    // q shares the forward sweep's place: it is read before the sweep
    double *s = _s, *z = _z, *t = _t0, *q = _y;
    int it;
    for (it = 0; it < maxIter; it++) {
        // s = z + (float)beta s with beta = rhoNew / rho, and q = A s
        _t->begin(T_SPMV, st);
        if (_refDots > 0) {
            if (it > 0) {
                pcgDirection(z, s, n, _pZr, nb, rho, rhoNew, st);
                std::swap(s, z);
                std::swap(rho, rhoNew);
            }
            columnResidual(_cp, _C, nullptr, s, q, st);
            rowDot(s, q, _pSq, st);
        } else if (it == 0) {
            columnSpmvDot(_cp, _C, s, q, _pSq, st);
        } else {
            columnDirectionSpmvDot(_cp, _C, z, s, t, q, _pZr, nb, rho, rhoNew, _pSq, st);
            std::swap(s, t);
            std::swap(rho, rhoNew);
        }
        _t->end(T_SPMV, st);
        armResidual();
        pcgStep(_x, s, _r, q, n, rho, _pSq, nb, _pRmax, st);
        _t->begin(T_MIC0_APPLY, st, applyLaunches(true));
        precondForward<double>(_r, _y, _pRmax, st);
        resid = awaitResidual(st);
        if (resid <= std::min(tol, 1.0)) {
            _t->end(T_MIC0_APPLY, st, forwardLaunches(true));
            iters = it + 1;
            return true;
        }
        precondBackward<double>(_y, z, st);
        _t->end(T_MIC0_APPLY, st);
        if (_refDots > 0)
            rowDot(z, _r, _pZr, st);
        else
            dotPartials(z, _r, n, _pZr, st);
    }
    iters = it;
    return false;
}

// FP64 PCG (pcgsolver.h:268-322) whose MIC(0) application runs on the FP32
// copy of the factor: the step that updates r also rounds it to float for the
// sweeps, and their result is widened into the search-direction update.  The
// SpMV, the dot products, the step lengths and every vector stay FP64, so the
// iteration follows the FP64 solve except for the preconditioner's rounding.
bool PressureSolver::pcgPrecond32(double tolFactor, int maxIter, double resid0, int &iters, double &resid,
                                  hipStream_t st) {
    const size_t n = _cp.slots();
    if (tolFactor < 1e-30) tolFactor = 1e-30;
    initialGuess(st);
    resid = resid0;
    double tol = tolFactor * resid;
    factor(false, st);
    castToFloat(_r, _fr, n, st);
    precond(_fr, _fy, _fz, st);
    double *rho = _scal + 2, *rhoNew = _scal + 3;
    const int nb = reduceBlocks(n);
    dotfd(_fz, _r, n, _partial, rho, st);
    double hrho = hostScalar(rho, st);
    if (hrho == 0 || hrho != hrho) {
        iters = 0;
        return false;
    }
    hipCheck(hipMemsetAsync(_s, 0, sizeof(double) * n, st), "memset");
    addFloatToDouble(_s, _fz, n, st);
    double *s = _s, *t = _z, *q = _y;
    int it;
    for (it = 0; it < maxIter; it++) {
        // s = (double)fz + (float)beta s with beta = rhoNew / rho, and q = A s
        _t->begin(T_SPMV, st);
        if (it == 0) {
            columnSpmvDot(_cp, _C, s, q, _pSq, st);
        } else {
            columnDirectionSpmvDot(_cp, _C, _fz, s, t, q, _pZr, nb, rho, rhoNew, _pSq, st);
            std::swap(s, t);
            std::swap(rho, rhoNew);
        }
        _t->end(T_SPMV, st);
        armResidual();
        pcgStep(_x, s, _r, q, n, rho, _pSq, nb, _pRmax, st, _fr);
        _t->begin(T_MIC0_APPLY, st, applyLaunches(true));
        precondForward<float>(_fr, _fy, _pRmax, st);
        resid = awaitResidual(st);
        if (resid <= std::min(tol, 1.0)) {
            _t->end(T_MIC0_APPLY, st, forwardLaunches(true));
            iters = it + 1;
            return true;
        }
        precondBackward<float>(_fy, _fz, st);
        _t->end(T_MIC0_APPLY, st);
        dotfdPartials(_fz, _r, n, _pZr, st);
    }
    iters = it;
    return false;
}

// The FP32 modes' direction s (fz + (float)beta s after the first) and fq = A s.
void PressureSolver::nextProduct(float *&s, float *&t, bool &first, double *&rho, double *&rhoNew, hipStream_t st) {
    if (first) {
        columnSpmvDotF(_cp, _C, s, _fq, _pSq, st);
        first = false;
        return;
    }
    columnDirectionSpmvDot(_cp, _C, _fz, s, t, _fq, _pZr, reduceBlocks(_cp.slots()), rho, rhoNew, _pSq, st);
    std::swap(s, t);
    std::swap(rho, rhoNew);
}

// FP32 PCG inside FP64 iterative refinement.  The outer loop keeps the FP64
// solution and its true residual r = b - A x; each inner solve runs PCG with
// the same MIC(0) factor rounded to FP32 on FP32 vectors (FP64 dot products)
// to a relative tolerance on its own right-hand side.  The stop test is the
// reference's |r|_inf <= min(tol * |b|_inf, 1.0), on the true residual.
bool PressureSolver::pcgMixed(double tolFactor, int maxIter, double resid0, double innerRel, int &iters,
                              double &resid, hipStream_t st) {
    const size_t n = _cp.slots();
    if (tolFactor < 1e-30) tolFactor = 1e-30;
    double tol = std::min(tolFactor * resid0, 1.0);
    hipCheck(hipMemcpyAsync(_r, _C.rhs, sizeof(double) * n, hipMemcpyDeviceToDevice, st), "copy");
    hipCheck(hipMemsetAsync(_x, 0, sizeof(double) * n, st), "memset");
    factor(false, st);
    double *rho = _scal + 2, *rhoNew = _scal + 3, *rn = _scal + 5;
    const int nb = reduceBlocks(n);
    resid = resid0;
    iters = 0;
    int outer = 0;
    while (resid > tol && iters < maxIter && outer < 100) {
        outer++;
        castToFloat(_r, _fr, n, st);
        absMaxf(_fr, n, _partial, rn, st);
        double innerTol = innerRel * hostScalar(rn, st);
        hipCheck(hipMemsetAsync(_fd, 0, sizeof(float) * n, st), "memset");
        precond(_fr, _fy, _fz, st);
        dotf(_fz, _fr, n, _partial, rho, st);
        double hrho = hostScalar(rho, st);
        if (hrho == 0 || hrho != hrho) return false;
        hipCheck(hipMemcpyAsync(_fs, _fz, sizeof(float) * n, hipMemcpyDeviceToDevice, st), "copy");
        float *s = _fs, *t = _ft;
        bool first = true;
        while (iters < maxIter) {
            _t->begin(T_SPMV, st);
            nextProduct(s, t, first, rho, rhoNew, st);
            _t->end(T_SPMV, st);
            armResidual();
            pcgStepF(_fd, s, _fr, _fq, n, rho, _pSq, nb, _pRmax, st);
            iters++;
            _t->begin(T_MIC0_APPLY, st, applyLaunches(true));
            precondForward<float>(_fr, _fy, _pRmax, st);
            if (awaitResidual(st) <= innerTol) {
                _t->end(T_MIC0_APPLY, st, forwardLaunches(true));
                break;
            }
            precondBackward<float>(_fy, _fz, st);
            _t->end(T_MIC0_APPLY, st);
            dotfPartials(_fz, _fr, n, _pZr, st);
        }
        addFloatToDouble(_x, _fd, n, st);
        columnResidual(_cp, _C, _C.rhs, _x, _r, st);
        absMax(_r, n, _partial, rn, st);
        resid = hostScalar(rn, st);
    }
    return resid <= tol;
}

// FP32 PCG whose FP64 solution is kept exact by reliable updates (Sleijpen &
// van der Vorst, 1996).  The search directions, the FP32 residual, SpMV and the
// preconditioner run in FP32; x accumulates in FP64 with the float-rounded
// step length; dot products accumulate in FP64.  Whenever the FP32 residual
// has dropped by `delta` since the last update (or meets the tolerance), the
// true residual r = b - A x is recomputed in FP64, tested against the
// reference's stop rule |r|_inf <= min(tol * |b|_inf, 1.0), and replaces the
// FP32 residual; the search direction is kept, so the Krylov space is not
// restarted.  Iterations counts every FP32 PCG step.
bool PressureSolver::pcgReliable(double tolFactor, int maxIter, double resid0, double delta, int &iters,
                                 double &resid, hipStream_t st) {
    const size_t n = _cp.slots();
    if (tolFactor < 1e-30) tolFactor = 1e-30;
    const double tol = std::min(tolFactor * resid0, 1.0);
    hipCheck(hipMemsetAsync(_x, 0, sizeof(double) * n, st), "memset");
    factor(false, st);
    double *rho = _scal + 2, *rhoNew = _scal + 3, *rn = _scal + 5;
    const int nb = reduceBlocks(n);
    castToFloat(_C.rhs, _fr, n, st);
    double sinceUpdate = resid0;
    resid = resid0;
    iters = 0;
    precond(_fr, _fy, _fz, st);
    dotf(_fz, _fr, n, _partial, rho, st);
    double hrho = hostScalar(rho, st);
    if (hrho == 0 || hrho != hrho) return false;
    hipCheck(hipMemcpyAsync(_fs, _fz, sizeof(float) * n, hipMemcpyDeviceToDevice, st), "copy");
    float *s = _fs, *t = _ft;
    bool first = true;
    bool trueKnown = true;  // resid holds the true residual of the current x
    while (iters < maxIter) {
        _t->begin(T_SPMV, st);
        nextProduct(s, t, first, rho, rhoNew, st);
        _t->end(T_SPMV, st);
        armResidual();
        pcgStepMixed(_x, s, _fr, _fq, n, rho, _pSq, nb, _pRmax, st);
        iters++;
        trueKnown = false;
        _t->begin(T_MIC0_APPLY, st, applyLaunches(true));
        precondForward<float>(_fr, _fy, _pRmax, st);
        const double rf = awaitResidual(st);
        if (rf <= delta * sinceUpdate || rf <= tol) {
            _t->end(T_MIC0_APPLY, st, forwardLaunches(true));
            columnResidual(_cp, _C, _C.rhs, _x, _r, st);
            absMax(_r, n, _partial, rn, st);
            resid = hostScalar(rn, st);
            trueKnown = true;
            if (resid <= tol) return true;
            castToFloat(_r, _fr, n, st);
            sinceUpdate = resid;
            _t->begin(T_MIC0_APPLY, st, applyLaunches(false));
            precondForward<float>(_fr, _fy, nullptr, st);  // again, from the replaced residual
        }
        precondBackward<float>(_fy, _fz, st);
        _t->end(T_MIC0_APPLY, st);
        dotfPartials(_fz, _fr, n, _pZr, st);
    }
    if (!trueKnown) {
        columnResidual(_cp, _C, _C.rhs, _x, _r, st);
        absMax(_r, n, _partial, rn, st);
        resid = hostScalar(rn, st);
    }
    return resid <= tol;
}

}  // namespace ff
