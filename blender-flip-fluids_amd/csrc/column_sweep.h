// column_sweep.h -- one triangular sweep of the MIC(0) preconditioner
// application z = (L L^T)^-1 r (solveLower / solveLowerTransposeInPlace,
// pcgsolver.h:211-241) in the column layout (column_types.h), as one launch.
//
// Work split.  One wave runs one column over the hyperplanes that hold its
// rows, in order: a step is one hyperplane.  The x neighbour is the line's own
// result of the previous step, the z neighbour inside a lane its other
// line's, and the neighbours in other lanes are moved by cross-lane register
// operations.  COL_WAVES columns along k, a wave each, make a workgroup's tile;
// they never meet at a barrier.  A wave hands its last line row to the next
// wave through a ring in LDS, and its face lines to the neighbour tiles
// through exchange words.
//
// What bounds it: the chain of hyperplanes (a step is some fifty instructions
// of one wave, the only one on its SIMD) and the hand-off between tiles along j
// and k.  So a step keeps to registers: its operands are whole slices at
// addresses that follow from the step alone, loaded PF steps ahead through
// buffer descriptors of the column's extent (a step past either end loads
// zeros and stores nothing, so no step is a special case), and the words read
// across a face are loaded PX steps ahead, about the latency of a load: more
// would only add to the lag between tiles.
//
// Hand-off.  A published value is one 64-bit word {32 value bits, epoch} (two
// words for a double), written and read with device-coherent accesses: the
// value and its validity travel in one single-copy-atomic access, so no fence
// orders them.  The epoch changes with every launch, so the buffer is never
// cleared.  A reader re-polls a word until it carries the launch's epoch.
//
// Progress.  Each workgroup first takes a ticket from a device counter and
// runs the tile of that rank in dependency order (tiles by PJ+PK, reversed for
// the backward sweep).  A tile reads only from tiles of a lower rank, whose
// workgroups took their tickets earlier and are running or done, and a wave
// waits for the next wave of its tile only while that one holds unread ring
// entries, so the launch drains for any number of resident workgroups.  Every
// wait is bounded, in looks and not by a clock, which would go on while the
// device runs another process: past the limit the wave raises the error word
// (which every other waiting wave also gives up on) and the launch still
// finishes; the host turns the word into an error.
//
// Arithmetic.  Every slot performs the reference's operations in its order
// (forward: subtract the -z, -y, -x terms, then scale by invdiag; backward:
// +x, +y, +z).  A missing neighbour's coefficient and value are zero, so its
// term subtracts +0 and leaves every bit.  (Values must be finite: an infinity
// times a missing coefficient is NaN.  PCG's dot products spread either;
// FFAMD_mic0_apply answers such a call in bands.)
//
// Measured, one application (both sweeps) FP64 / FP32, against launches over
// bands of 8 / 12 hyperplanes: 24^3 99 / 86 -> 42 / 35 us, 64^3 237 / 201 ->
// 108 / 80, 128^3 513 / 441 -> 217 / 162, 256^3 dam break 1267 / 1058 -> 473 /
// 353.  A forward sweep FP32 / FP64 by (lines a lane, waves a tile), us:
//              24^3       64^3       100^3       96x160x256
//   (2, 2)  20.0/26.5  52.3/70.5   85.3/114.3   151/204   taken
//   (2, 1)  18.8/34.9  48.9/95.9   79.9/147.9   142/264
//   (2, 4)  20.8/27.9  53.4/85.7   86.6/137.4   153/238
//   (1, 2)  19.6/23.6  53.4/64.3   87.1/102.1   165/198
//   (1, 4)  20.5/25.3  55.1/66.2   91.3/105.4   169/199
// One shape serves both precisions, since FP64 vectors and FP32 sweeps share a
// layout; (4, 1) and (4, 2) were slower still.  A 16 x 16 tile with an LDS plane
// and a barrier per step took 0.22 us a step against 0.15.
//
// This header holds only the sweep's body; its includer supplies the hardware
// operations as macros: column_hw.h the GPU's, tests/emu/column_emu.cpp ones
// that run it on the CPU and grant a ring value no more ordering than asked for.
#pragma once

#include "column_types.h"

namespace ff {

// Rec: {inv, a, b, c} -- invdiag and the L entries the sweep multiplies the
// -x/-y/-z (forward) or +x/+y/+z (backward) neighbours' results by
template <class T, class Rec>
struct ColumnArgs {
    int ncj, nck;             // columns along j and k
    int ntj, ntk;             // tiles along j and k (ntj = ncj)
    const ColumnRange *cols;  // ncj * nck
    const int *order;         // tiles by PJ + PK (forward ranks)
    const T *in;              // slots: right-hand side (forward) or forward result (backward)
    T *out;                   // slots
    const Rec *rec;           // slots
    unsigned *exJ, *exK;      // words: column x step x COL_K lines; tile x step x COL_J lines
    int exSteps;              // steps of a column's words (the hyperplanes it can span)
    unsigned *counter;        // ticket counter
    int *error;               // raised when a wait exceeded waitLooks
    unsigned base;            // counter value when this launch started
    unsigned epoch;           // tag of this launch's published words (never 0)
    int waitLooks;            // longest wait, looks at what is waited for
};

// a value's words as four (double) or two (float) 32-bit parts
template <class T>
struct ColumnWord;
template <>
struct ColumnWord<float> {
    static constexpr int N = 2;
    static FF_CS_DEVICE void pack(float v, unsigned epoch, unsigned (&w)[2]) {
        w[0] = FF_CS_F2U(v);
        w[1] = epoch;
    }
    static FF_CS_DEVICE float value(const unsigned (&w)[2]) { return FF_CS_U2F(w[0]); }
    static FF_CS_DEVICE bool fresh(const unsigned (&w)[2], unsigned epoch) { return w[1] == epoch; }
};
template <>
struct ColumnWord<double> {
    static constexpr int N = 4;
    static FF_CS_DEVICE void pack(double v, unsigned epoch, unsigned (&w)[4]) {
        const unsigned long long u = FF_CS_D2U(v);
        w[0] = (unsigned)u;
        w[1] = epoch;
        w[2] = (unsigned)(u >> 32);
        w[3] = epoch;
    }
    static FF_CS_DEVICE double value(const unsigned (&w)[4]) {
        return FF_CS_U2D((unsigned long long)w[0] | ((unsigned long long)w[2] << 32));
    }
    static FF_CS_DEVICE bool fresh(const unsigned (&w)[4], unsigned epoch) { return w[1] == epoch && w[3] == epoch; }
};

// a wave's results of its last steps, in LDS, for the next wave of the tile
constexpr int COL_RING = 32;  // steps; a power of two
template <class T>
struct ColumnRing {
    T v[COL_RING][COL_LANES];
    int made, taken;  // steps written; steps the reader is done with
};

constexpr int COL_DONE = 0x7fffffff;
constexpr int COL_AHEAD = 2;  // steps a wave waits for at once

// what the variants of a wave's loop share
template <class T>
struct ColumnWave {
    int lane, n;      // hyperplanes (steps) of the column
    int offJ, lenJ;   // step u reads step u + offJ of the column across the j face (lenJ steps, 0: none)
    int offK, lenK;   // and of the column across the k face
    FF_CS_BUFFER in, rec, out, fromJ, fromK, toJ, toK;
    unsigned toJ0, toK0;   // this lane's first words, out of the buffer unless it is on the face
    ColumnRing<T> *up, *own;  // the previous wave's ring and this wave's
};

// FIRST: the lines before the column's first row are another tile's (or
// none), otherwise the previous wave's; LAST: another tile reads its last row.
template <class T, class Rec, int PF, int PX, bool FWD, bool FIRST, bool LAST>
FF_CS_DEVICE void columnSteps(const ColumnArgs<T, Rec> &a, const ColumnWave<T> &w) {
    static_assert(PX <= PF && PF + COL_AHEAD < COL_RING, "the words' ring is the operands'");
    constexpr int N = ColumnWord<T>::N;
    using Word = ColumnWord<T>;
    constexpr int R = COL_R;
    struct Slot {
        T in[R];
        Rec rec[R];
        unsigned j[R][N], k[N];
    };
    const int lane = w.lane, lj = lane % COL_J, lk = lane / COL_J, n = w.n;
    constexpr unsigned SLICE = COL_SLICE * sizeof(T), RSLICE = COL_SLICE * sizeof(Rec);
    constexpr unsigned JSTEP = COL_K * N * 4, KSTEP = COL_J * N * 4;
    // the backward sweep starts at the last slice
    auto slice = [&](int u) { return (unsigned)(FWD ? u : n - 1 - u); };
    // looks at the error word only now and then: that takes as long as a look at
    // what it waits for
    auto wait = [&](auto &&ready) {
#pragma unroll 1
        for (int looks = 0;; looks++) {
            FF_CS_REREAD();
            if (ready()) return;
            if ((looks & 63) == 63 && (FF_CS_LOAD32(a.error) != 0 || looks >= a.waitLooks)) {
                FF_CS_RAISE(a.error);
                return;
            }
        }
    };
    auto loadJ = [&](unsigned (&q)[R][N], int u) {
        FF_CS_LOAD_WORDS(q, w.fromJ, lk * (R * N * 4) + (unsigned)(u + w.offJ) * JSTEP);
    };
    auto loadK = [&](unsigned (&q)[N], int u) {
        FF_CS_LOAD_WORDS(q, w.fromK, lj * (N * 4) + (unsigned)(u + w.offK) * KSTEP);
    };
    auto operands = [&](Slot &q, int u) {
        FF_CS_LOAD(q.in, w.in, lane * (unsigned)(R * sizeof(T)) + slice(u) * SLICE);
        FF_CS_LOAD(q.rec, w.rec, lane * (unsigned)(R * sizeof(Rec)) + slice(u) * RSLICE);
    };
    auto staleJ = [&](const unsigned (&q)[R][N]) {
        bool fresh = true;
#pragma unroll
        for (int r = 0; r < R; r++) fresh = fresh && Word::fresh(q[r], a.epoch);
        return FF_CS_ANY(!fresh);
    };
    // the line row before the column's, of step u, from the previous wave's
    // ring.  A wave that runs into the writer waits for a few steps at once,
    // so that it looks again every few steps only.
    const int ringLane = lj + (FWD ? COL_LANES - COL_J : 0);
    int made = 0;
    auto ringK = [&](int u) {
        T v = T(0);
        const int x = u + w.offK;
        if ((unsigned)x < (unsigned)w.lenK) {
            if (FF_CS_RARE(made <= x)) {
                const int want = x + COL_AHEAD < w.lenK ? x + COL_AHEAD : w.lenK;
                wait([&]() { return (made = FF_CS_UNIFORM(FF_CS_LDS_LOAD(&w.up->made))) >= want; });
                FF_CS_WAVE_ORDER();  // the entries are read after the count that promised them
            }
            v = FF_CS_LDS_LOAD(&w.up->v[x & (COL_RING - 1)][ringLane]);
        }
        return v;
    };
    auto store = [&](const T (&v)[R], int u) {
        unsigned p[R][N];
#pragma unroll
        for (int r = 0; r < R; r++) Word::pack(v[r], a.epoch, p[r]);
        FF_CS_STORE_WORDS(p, w.toJ, w.toJ0 + (unsigned)u * JSTEP);
        if (LAST) FF_CS_STORE_WORDS(p[FWD ? R - 1 : 0], w.toK, w.toK0 + (unsigned)u * KSTEP);
        FF_CS_STORE(v, w.out, lane * (unsigned)(R * sizeof(T)) + slice(u) * SLICE);
    };
    int taken = 0;
    T prev[R];  // the lines' results of the previous step
#pragma unroll
    for (int r = 0; r < R; r++) prev[r] = T(0);
    Slot ring[PF];
    // The accesses of the PF steps before the first, in a step's order: stores
    // that go nowhere, words past the ends.  The counter a wave waits on counts
    // loads and stores alike, and at the loop's head the compiler takes the
    // smaller distance of the two ways in: with a head of loads only, every
    // step waited for all but its last 11 accesses, some of them stores to
    // memory (96 x 160 x 256: 168 us FP32, 224 us FP64 a sweep; so 151, 205).
#pragma unroll
    for (int q = 0; q < PF; q++) {
        store(prev, q - PF);
        loadJ(ring[(q + PX) % PF].j, q - PF + PX);
        if (FIRST) loadK(ring[(q + PX) % PF].k, q - PF + PX);
        operands(ring[q], q);
    }
    T nextK = T(0);
    if (!FIRST) nextK = ringK(0);
    // whole rounds of PF steps: a step past the last one reads zeros and
    // writes nothing but the (unread) ring
    for (int u0 = 0; u0 < n; u0 += PF) {
#pragma unroll
        for (int q = 0; q < PF; q++) {
            const int u = u0 + q;
            Slot &c = ring[q];
            // A word that is not there yet: the words in flight were read
            // before it and are not there either, so wait for the last of
            // them and read them all again.  From then on the wave stays
            // behind the writer by what it reads ahead.
            if ((unsigned)(u + w.offJ) < (unsigned)w.lenJ && FF_CS_RARE(staleJ(c.j))) {
                const int end = w.lenJ - 1 - w.offJ, far = u + PX - 1 < end ? u + PX - 1 : end;
                unsigned t[R][N];
                wait([&]() {
                    loadJ(t, far);
                    return !staleJ(t);
                });
#pragma unroll
                for (int x = 1; x < PX; x++) loadJ(ring[(q + x) % PF].j, u + x);
                wait([&]() {
                    loadJ(c.j, u);
                    return !staleJ(c.j);
                });
            }
            T extK;
            if (FIRST) {
                if ((unsigned)(u + w.offK) < (unsigned)w.lenK && FF_CS_RARE(FF_CS_ANY(!Word::fresh(c.k, a.epoch)))) {
                    const int end = w.lenK - 1 - w.offK, far = u + PX - 1 < end ? u + PX - 1 : end;
                    unsigned t[N];
                    wait([&]() {
                        loadK(t, far);
                        return !FF_CS_ANY(!Word::fresh(t, a.epoch));
                    });
#pragma unroll
                    for (int x = 1; x < PX; x++) loadK(ring[(q + x) % PF].k, u + x);
                    wait([&]() {
                        loadK(c.k, u);
                        return !FF_CS_ANY(!Word::fresh(c.k, a.epoch));
                    });
                }
                extK = Word::value(c.k);
            } else {
                extK = nextK;
                nextK = ringK(u + 1);
            }
            T vy[R], vz[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                vy[r] = FF_CS_ROW_SHIFT(FWD, prev[r], Word::value(c.j[r]));
                if (FWD ? r > 0 : r < R - 1) vz[r] = prev[FWD ? r - 1 : r + 1];
            }
            vz[FWD ? 0 : R - 1] = FF_CS_LINE_SHIFT(FWD, prev[FWD ? R - 1 : 0], extK);
#pragma unroll
            for (int r = 0; r < R; r++) {
                T y = c.in[r];
                if (FWD) {
                    y -= c.rec[r].c * vz[r];
                    y -= c.rec[r].b * vy[r];
                    y -= c.rec[r].a * prev[r];
                } else {
                    y -= c.rec[r].a * prev[r];
                    y -= c.rec[r].b * vy[r];
                    y -= c.rec[r].c * vz[r];
                }
                prev[r] = y * c.rec[r].inv;
            }
            const T face = prev[FWD ? R - 1 : 0];  // the line the next lane row reads
            if (!LAST) {
                if (FF_CS_RARE(u - taken >= COL_RING))
                    wait([&]() { return u - (taken = FF_CS_UNIFORM(FF_CS_LDS_LOAD(&w.own->taken))) < COL_RING; });
                FF_CS_LDS_STORE(&w.own->v[u & (COL_RING - 1)][lane], face);
                FF_CS_WAVE_ORDER();
                FF_CS_LDS_STORE(&w.own->made, u + 1);
            }
            store(prev, u);
            loadJ(ring[(q + PX) % PF].j, u + PX);
            if (FIRST) loadK(ring[(q + PX) % PF].k, u + PX);
            operands(ring[q], u + PF);
        }
        // entries up to the one in nextK are read
        if (!FIRST) {
            FF_CS_WAVE_ORDER();
            const int x = u0 + PF + w.offK;
            if (x > 0) FF_CS_LDS_STORE(&w.up->taken, x);
        }
    }
    if (!FIRST) FF_CS_LDS_STORE(&w.up->taken, (int)COL_DONE);
}

template <class T, class Rec, int PF, int PX, bool FWD>
FF_CS_DEVICE void columnSweep(const ColumnArgs<T, Rec> &a, const int tid) {
    constexpr int s = FWD ? 1 : -1, N = ColumnWord<T>::N;
    FF_CS_SHARED ColumnRing<T> rings[COL_WAVES > 1 ? COL_WAVES - 1 : 1];
    FF_CS_SHARED unsigned sTicket;
    if (tid == 0) sTicket = FF_CS_TICKET(a.counter) - a.base;
    const int wave = FF_CS_UNIFORM(tid / COL_LANES), lane = tid % COL_LANES;
    const int pos = FWD ? wave : COL_WAVES - 1 - wave;  // place in the order of the waves
    if (lane == 0 && pos > 0) {
        rings[pos - 1].made = 0;
        rings[pos - 1].taken = 0;
    }
    FF_CS_BARRIER();
    const int nt = a.ntj * a.ntk;
    const int ticket = FF_CS_UNIFORM((int)sTicket);
    if (ticket < 0 || ticket >= nt) return;  // the grid has nt workgroups: never taken
    const int p = FF_CS_UNIFORM(a.order[FWD ? ticket : nt - 1 - ticket]);
    const int PJ = p % a.ntj, PK = p / a.ntj;
    const int ck = PK * COL_WAVES + wave;
    auto column = [&](int cj, int k) {
        ColumnRange r{1, 0, 0, 0};
        if (cj >= 0 && cj < a.ncj && k >= 0 && k < a.nck) r = a.cols[k * a.ncj + cj];
        return ColumnRange{FF_CS_UNIFORM(r.lo), FF_CS_UNIFORM(r.hi), FF_CS_UNIFORM(r.base), 0};
    };
    auto steps = [](const ColumnRange &r) { return r.hi >= r.lo ? r.hi - r.lo + 1 : 0; };
    const ColumnRange own = column(PJ, ck);
    ColumnWave<T> w;
    w.lane = lane;
    w.n = steps(own);
    // a wave without rows publishes nothing and nobody waits for it
    if (w.n == 0) return;
    // the columns read from (forward: -j, -k) and read by; a step of this
    // column at h reads the step of the other one at h - s
    const ColumnRange fj = column(PJ - s, ck), fk = column(PJ, ck - s), tj = column(PJ + s, ck), tk = column(PJ, ck + s);
    auto offset = [&](const ColumnRange &r) { return FWD ? own.lo - 1 - r.lo : r.hi - (own.hi + 1); };
    w.lenJ = steps(fj);
    w.lenK = steps(fk);
    w.offJ = w.lenJ > 0 ? offset(fj) : 0;
    w.offK = w.lenK > 0 ? offset(fk) : 0;
    const bool first = pos == 0, last = pos == COL_WAVES - 1;
    w.up = first ? nullptr : &rings[pos - 1];
    w.own = last ? nullptr : &rings[pos];
    // a ring nobody reads is never full; entries before the first one read are
    // done with
    if (!last && steps(tk) == 0) FF_CS_LDS_STORE(&w.own->taken, (int)COL_DONE);
    if (!first && w.lenK > 0 && w.offK > 0) FF_CS_LDS_STORE(&w.up->taken, w.offK);
    // buffers of exactly the column's slots and of the steps the neighbours publish
    const long long slot0 = (long long)own.base + (long long)COL_SLICE * own.lo;
    const unsigned slots = (unsigned)w.n * COL_SLICE;
    w.in = FF_CS_MAKE_BUFFER(a.in + slot0, slots * (unsigned)sizeof(T));
    w.rec = FF_CS_MAKE_BUFFER(a.rec + slot0, slots * (unsigned)sizeof(Rec));
    w.out = FF_CS_MAKE_BUFFER(a.out + slot0, slots * (unsigned)sizeof(T));
    const long long jWords = (long long)a.exSteps * COL_K * N, kWords = (long long)a.exSteps * COL_J * N;
    const long long c = (long long)ck * a.ncj + PJ;
    w.fromJ = FF_CS_MAKE_BUFFER(a.exJ + (w.lenJ > 0 ? c - s : c) * jWords, (unsigned)w.lenJ * (COL_K * N * 4));
    w.toJ = FF_CS_MAKE_BUFFER(a.exJ + c * jWords, (unsigned)(steps(tj) > 0 ? w.n : 0) * (COL_K * N * 4));
    const bool readK = first && w.lenK > 0, writeK = last && steps(tk) > 0;
    w.fromK = FF_CS_MAKE_BUFFER(a.exK + (long long)(readK ? p - s * a.ntj : p) * kWords,
                                (unsigned)(readK ? w.lenK : 0) * (COL_J * N * 4));
    w.toK = FF_CS_MAKE_BUFFER(a.exK + (long long)p * kWords, (unsigned)(writeK ? w.n : 0) * (COL_J * N * 4));
    const int lj = lane % COL_J, lk = lane / COL_J;
    constexpr unsigned OUTSIDE = 0x80000000u;
    w.toJ0 = lj == (FWD ? COL_J - 1 : 0) ? lk * (unsigned)(COL_R * N * 4) : OUTSIDE;
    w.toK0 = lk == (FWD ? COL_LANES / COL_J - 1 : 0) ? lj * (unsigned)(N * 4) : OUTSIDE;
    if (first)
        columnSteps<T, Rec, PF, PX, FWD, true, COL_WAVES == 1>(a, w);
    else if (last)
        columnSteps<T, Rec, PF, PX, FWD, false, true>(a, w);
    else if (COL_WAVES > 2)
        columnSteps<T, Rec, PF, PX, FWD, false, false>(a, w);
}

}  // namespace ff
