// pressure.h -- GPU pressure solve of the FLIP substep (host side).
//
// PressureSolver mirrors the reference's PressureSolver::solve +
// _solveLinearSystem (pressuresolver.cpp:52-92, 869-916) and
// PCGSolver<double>::solve (pcgsolver.h:268-322), with an additional
// mixed-precision mode.  It owns the system buffers for one grid size.
#pragma once

#include <vector>

#include "kernels.h"
#include "timers.h"

namespace ff {

struct PressureResult {
    bool success = true;  // after the acceptable-tolerance rule
    int iterations = 0;
    double error = 0.0;   // |r|_inf at exit (the reference rounds it to float)
    double rhsInf = 0.0;  // |b|_inf of the right-hand side
    int unknowns = 0;
};

class PressureSolver {
public:
    PressureSolver() = default;
    ~PressureSolver();
    PressureSolver(const PressureSolver &) = delete;
    PressureSolver &operator=(const PressureSolver &) = delete;

    void allocate(Grid g);
    // Builds the system from the current fields, solves it and writes the
    // float pressure grid.  cellRhs (N doubles, optional) replaces the
    // assembled right-hand side by its values at the rows' cells (the matrix
    // still comes from phi and the weights); cellSolution (N doubles,
    // optional) receives the FP64 solution on the rows' cells and 0 elsewhere.
    // referenceDots > 0 makes the FP64 solve (mode 0)
    // take its dot products in the reference's order for that thread count.
    // mode 0 = FP64 PCG; 1 = FP32 PCG restarted inside
    // FP64 iterative refinement (innerTol = relative tolerance of each inner
    // solve); 2 = FP32 PCG with FP64 reliable updates (innerTol = drop of the
    // FP32 residual between true-residual updates); 3 = FP64 PCG with the
    // MIC(0) application in FP32 (innerTol unused).
    PressureResult solve(double dt, const float *u, const float *v, const float *w, const float *wu,
                         const float *wv, const float *ww, const float *phi, double tol, int maxIter,
                         int mode, double innerTol, float *pressure, int *scanScratch, hipStream_t s,
                         hipEvent_t afterAssembly, KernelTimers *timers = nullptr, int referenceDots = 0,
                         const double *cellRhs = nullptr, double *cellSolution = nullptr);
    const PressureSys &system() const { return _S; }
    // FP64 PCG (modes 0 and 3): start from the pressure grid's values at
    // the rows (the previous solve's result) instead of 0.  The stopping
    // test keeps the zero-start threshold, tolerance x |b|_inf.
    void setWarmStart(bool on) { _warm = on; }
    // the moving solid's face velocities and cell weights for the divergence
    // of the following solves (all null: a static solid)
    void setSolidTerms(SolidTerms t) { _solid = t; }
    // the surface tension terms of the following solves' divergence (status
    // null: none)
    void setTension(TensionView t) { _tension = t; }
    // the solver's MIC(0) application: 2 = columns of lines, one launch per
    // sweep; 4 = the line pipeline on the row order (two launches per
    // application), 5 = bands of hyperplanes on the row order, replayed from a
    // HIP graph captured once per solve
    void setSchedule(int schedule);
    int schedule() const { return _sched; }
    const std::vector<int> &levelTable() const { return _hLevelStart; }
    // the MIC(0) factor of the last solve()'s system, which a solve that had
    // nothing to solve did not need
    void factorSystem(bool fp64, hipStream_t s);
    // one preconditioner application z = (L L^T)^-1 r on the current factor
    // (after solve()); FP64 or the FP32 copy; r and z in row order.
    // schedule 0 = one launch per hyperplane, 1 = tile wavefront (switched
    // off: raises an error), 2 = columns (the solver's), 3 = bands of
    // hyperplanes with the tile ranges checked on the device, 4 = the line
    // pipeline, 5 = bands of the tiles the host lists.  0, 3 and 5 leave the term
    // of a missing neighbour out; 2 and 4 subtract 0 times it, the same for finite
    // values only.
    void applyPreconditioner(const double *r, double *z, int schedule, hipStream_t s);
    void applyPreconditionerF(const float *r, float *z, int schedule, hipStream_t s);
    // throws when a preconditioner launch gave up waiting (waits for the stream)
    void checkError(hipStream_t s);

private:
    Grid _g{};
    PressureSys _S{};
    void *_block = nullptr;     // one allocation for the system, its columns and the vectors
    void *_rowBlock = nullptr;  // and one for the row-ordered schedules, made when one is used
    ColumnPlan _cp;
    ColumnSys _C{};
    // the PCG's vectors, in slots
    double *_x = nullptr, *_r = nullptr, *_z = nullptr, *_s = nullptr, *_y = nullptr, *_t0 = nullptr;
    float *_fr = nullptr, *_fz = nullptr, *_fs = nullptr, *_fd = nullptr, *_fq = nullptr, *_fy = nullptr, *_ft = nullptr;
    // an application's operands in row order (row-ordered schedules and dots)
    double *_rowR = nullptr, *_rowY = nullptr, *_rowZ = nullptr;
    float *_rowFR = nullptr, *_rowFY = nullptr, *_rowFZ = nullptr;
    double *_partial = nullptr, *_scal = nullptr;
    double *_pSq = nullptr, *_pRmax = nullptr, *_pZr = nullptr;  // partials of s . q, |r|_inf and z . r
    double *_hostScal = nullptr, *_hostScalDev = nullptr;  // mapped pinned host slot and its device alias
    std::vector<int> _hLevelStart;
    MicSchedule _ms;
    int _maxTiles = 0;
    int *_tileLo = nullptr, *_tileHi = nullptr;  // band schedule: hyperplane range of each tile's rows
    int _bandTilesMax = 0;
    std::vector<int> _hTileLo, _hTileHi;  // host copies of the tile ranges
    BandPlan _plan;                       // band launches of the current system
    std::vector<int> _hTileRows, _hOrder;
    KernelTimers *_t = nullptr;
    KernelTimers _noTimers;
    int _levelLaunches = 0, _bandLaunches = 0;
    PencilPlan _pp;  // line-pipeline buffers (inside _rowBlock)
    long long _waitTicks = 0;  // the row-ordered schedules' longest wait, wall-clock ticks
    int _sched = 2;
    // z = M^-1 r with the solver's schedule (y: forward result), whole or in
    // its two halves
    template <class T>
    void precond(const T *r, T *y, T *z, hipStream_t s);
    template <class T>
    void precondForward(const T *r, T *y, const double *rmax, hipStream_t s);
    template <class T>
    void precondBackward(const T *y, T *z, hipStream_t s);
    // launches of its halves: the row-ordered schedules convert before and after,
    // and publish in a launch of its own
    int forwardLaunches(bool publish) const { return _sched == 2 ? 1 : publish ? 2 : 1; }
    int applyLaunches(bool publish) const {
        return forwardLaunches(publish) + (_sched == 2 ? 1 : (_sched == 5 ? _bandLaunches : 2) + 1);
    }
    size_t maxRows() const;
    void ensureRowSchedules();
    void prepareRowSchedule(int schedule, bool fp64, hipStream_t s);
    void factor(bool fp64, hipStream_t st);
    void rowDot(const double *a, const double *b, double *out, hipStream_t st);
    // schedule 5: the band launches of an application as an executable graph,
    // recorded at the first application of a system (every application of it
    // has the same operands), dropped when a new system is prepared
    hipGraphExec_t _graph = nullptr;
    void dropGraph();
    template <class T>
    void graphApply(const T *r, T *y, T *z, hipStream_t s);
    int _refDots = 0;  // thread count of the reference's dot order, or 0 for the tree reductions
    bool _warm = false;
    SolidTerms _solid{};
    TensionView _tension{};
    const float *_prevPressure = nullptr;  // the pressure grid at solve() entry
    // x = 0, r = b; or, warm, x from the pressure grid and r = b - A x
    void initialGuess(hipStream_t st);

    double hostScalar(const double *d, hipStream_t s);
    void nextProduct(float *&s, float *&t, bool &first, double *&rho, double *&rhoNew, hipStream_t st);
    void armResidual();
    double awaitResidual(hipStream_t s);
    void enqueueTileRanges(bool fp64, hipStream_t s);
    // tile schedule of the preconditioner application for this system
    void buildSchedule(bool fp64, hipStream_t s);
    bool pcgFP64(double tolFactor, int maxIter, double resid0, int &iters, double &resid, hipStream_t s);
    bool pcgMixed(double tolFactor, int maxIter, double resid0, double innerTol, int &iters,
                  double &resid, hipStream_t s);
    bool pcgReliable(double tolFactor, int maxIter, double resid0, double delta, int &iters, double &resid,
                     hipStream_t s);
    bool pcgPrecond32(double tolFactor, int maxIter, double resid0, int &iters, double &resid, hipStream_t s);
};

}  // namespace ff
