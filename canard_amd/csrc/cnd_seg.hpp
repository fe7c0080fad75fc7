// Segmented pencil sweeps: the pentadiagonal solves of the compact
// derivative (src/mo_numerics.f90:709-886) and compact filter
// (src/mo_numerics.f90:890-987) with every pencil split into S segments of
// at most L points, one lane per (pencil, segment, variable), so a lane keeps
// its whole segment in registers and the sweep reads each source point once
// and writes each result once (no forward-value scratch in HBM).
//
// The LU factors of the line (xl, xu of init_penta/penta) are the ones the
// sequential sweep uses.  Each lane runs each recurrence twice over its own
// rows: first with zero incoming values, which gives the two values the
// segment would pass on; a short scan over the segments of the pencil
// through LDS (a 2x2 transfer per segment, built from the homogeneous
// solutions phi1, phi2 / psi1, psi2 at the segment's ends) turns them into
// the true incoming values; the second run starts from those and is the
// sequential recurrence itself, so the result equals it up to rounding.
// Segments are held right-aligned in L registers; the registers in front of
// a shorter segment are pass-through rows (LU coefficients that swap the
// recurrence state exactly), so every lane runs the same branch-free code.
//
// Workgroup: NV * P * SP threads.  Thread t: variable v = t / (P * SP),
// pencil p = t % P, segment s = (t / P) % SP.  xi tiles (P contiguous
// pencils) are staged whole into LDS with consecutive threads on consecutive
// points; eta/zeta sweeps, of one plain field a workgroup, load each lane's
// rows directly (the lanes of a wave hold P neighbouring pencils, so every
// load reads runs of P consecutive points).  The lanes near a pencil end keep the 13
// source values next to it in LDS (xi: they stay in the staged tile); the
// closure rows are formed from them after the stream (and, for a block that
// is its own periodic partner, the partner sums too, so no extra loads).
#pragma once

#include <type_traits>

#include "cnd_dev.hpp"
#include "cnd_kernels.hpp"

namespace cnd {

// Points of a pencil end used by the closure rows (12) plus the face point.
constexpr int kSegEnd = 12;
constexpr int kSegEndRows = kSegEnd + 1;

// Compiled segment lengths (coefficient tables).
constexpr int kNumL = 3, kLs[kNumL] = {17, 33, 9};
__host__ __device__ constexpr int l_index(int L) { return L == 17 ? 0 : (L == 33 ? 1 : 2); }

// Fewest rows of a segment of at most L (seg_count); a whole pencil has 13 or
// more.
__host__ __device__ constexpr int seg_min_rows(int L) { return L < 17 ? 6 : 12; }

// Doubles in front of and behind a xi tile in LDS: a lane reads its rows
// without clamping those outside its line (they only reach rows that the
// closure rows replace), at most 33 - 12 + 3 of them.
constexpr int kTilePad = 24;

// LU values a thread stages per round trip.
constexpr int kLuBatch = 12;

// Points whose sources a thread reads back together at a xi store.
constexpr int kOutBatch = 8;

// Segments of an n-point pencil for lanes of at most L points: 0 when one of
// them would have fewer than seg_min_rows(L) rows.  The closure rows of an end
// lie inside one segment that way; the source values they are formed from may
// come from several lanes.  Segments are as even as possible.
__host__ __device__ inline int seg_count(int n, int L)
{
    const int S = (n + L - 1) / L;
    if (S > 1 && n / S < seg_min_rows(L)) return 0;
    return S;
}

__host__ __device__ inline void seg_bounds(int n, int, int S, int s, int &a, int &len)
{
    const int q = n / S, r = n % S;
    a = s * q + (s < r ? s : r);
    len = q + (s < r ? 1 : 0);
}


template <int NV, int SCH, int L, int P, bool XI>
struct SegShape {
    static constexpr int H = SCH == 0 ? 2 : 3;          // stencil half width
    static constexpr int NB = SCH == 0 ? 2 : 3;         // closure rows per end
    static constexpr int KR = L + 2 * H;                // rows streamed per lane
    // xi tiles in LDS: pencil after pencil, each n | 1 points long (an odd
    // stride puts the lanes of neighbouring pencils in different banks),
    // variable after variable; for odd n a point's place is its index in
    // the tile
    __host__ __device__ static constexpr int pencil_stride(int n) { return n | 1; }
    // LDS.  eta/zeta: the pencil-end values [2][13][P], and over them, once the
    // closure rows are formed, the exchange buffer [2][SP][P]; the segment
    // transfer values [SP][8]; the LU rows of the launch's SP segments as
    // their lanes hold them [SP][L][5].  xi: the whole tile's sources
    // [NV][P][nmax | 1], and over them, once the closure rows are formed, the
    // LU rows and the exchange buffer [2][NV][SP][P] (kTilePad doubles on
    // either side of the tile); the transfer values.
    // Last, both, and only when some block has another block as its partner
    // along the sweep direction: the partner points [2][13][NV][P].
    // Total bytes: seg_lds_bytes.  (With a staging chunk, partner points and
    // both buffers side by side eta and zeta took twice as much: the filters
    // of 257^3 points 354 and 377 us, with this 329 and 347.)
};

// xi sweeps (XI shapes run along xi only): the P pencils of a tile are
// consecutive rows of the block, so point e of the tile (pencil e / n, row
// e % n) sits at g0 + e, g0 the tile's first point; the LDS tile keeps the
// same order (pencils n | 1 points apart), so staging and stores address
// both by e.

// One lane's segment s of the S of its line, held right-aligned in
// Y[kb .. L - 1]; Y[0 .. kb - 1] are pass-through registers.  exi: the lane's
// place in the exchange buffer, segments P apart, the second value of a pair
// exs further on; ok: the lane has a segment.
struct SegLane {
    int kb, s, S, ok, exi, exs, P;
};

// LU row of a pass-through register: the forward step y = (Y - l0 ya) - l1 yb
// with Y = 0 gives y = ya, the backward step x = (l2 Y - l3 xa) - l4 xb
// gives x = xb; either way the recurrence state (two values) is swapped
// exactly, and two such rows leave it unchanged.
__host__ __device__ constexpr double seg_pass_row(int c) { return c == 0 || c == 4 ? -1.0 : 0.0; }

// Solve the line for the lane's segment held in Y (right-hand side in,
// solution out; Y[0 .. kb - 1] must be zero).  LUs: the
// LU rows of every segment as the lanes hold them, [SP][L][5] in LDS
// (pass-through rows in front); SM: per-segment transfer values in LDS
// (phi1, phi2 at the segment's last two rows, psi1, psi2 at its first two);
// ex: LDS room for 2 x NV x SP x P doubles.  All threads must call it.
//
// Each recurrence runs twice over the lane's registers: first with zero
// incoming values, keeping only the two values that leave the segment;
// after the scan over the segments has turned those into the true incoming
// values, again from them, which is the sequential recurrence itself.  All
// passes run over all L registers with no branches: the segment's last row
// is always register L - 1, and the kb pass-through registers carry the
// state across the front of the segment (swapped kb times, which the start
// or end values undo).  A pencil of one segment (S is the same for the whole
// workgroup) needs no pass 1: with it, and with the block's codes read in the
// first round of loads, a step of 16^3 points went from 252 to 228 us.
template <int L>
__device__ __forceinline__ void seg_solve(double (&Y)[L], const SegLane &ln, const double *LUs, const double *SM,
                                          double *ex)
{
    const int s = ln.s;
    const bool odd = (ln.kb & 1) != 0;
    const double *lu = LUs + 5 * L * s;
    double t0 = 0.0, t1 = 0.0;
    if (ln.S > 1) {
        // forward, pass 1: zero incoming values, outgoing values only
        {
            double ya = 0.0, yb = 0.0;
#pragma unroll
            for (int k = 0; k < L; ++k) {
                const double y = (Y[k] - lu[5 * k] * ya) - lu[5 * k + 1] * yb;
                ya = yb;
                yb = y;
            }
            __syncthreads();
            ex[ln.exi] = ya;
            ex[ln.exs + ln.exi] = yb;
            __syncthreads();
        }
        // incoming values y(a-2), y(a-1): scan over the segments before this one
        if (ln.ok) {
            for (int sp = 0; sp < s; ++sp) {
                const double *m = SM + 8 * sp;
                const int xi = ln.exi + (sp - s) * ln.P;
                const double n0 = (m[0] * t0 + m[1] * t1) + ex[xi];
                const double n1 = (m[2] * t0 + m[3] * t1) + ex[ln.exs + xi];
                t0 = n0;
                t1 = n1;
            }
        }
    }
    // forward, pass 2: from the true incoming values
    {
        double ya = odd ? t1 : t0, yb = odd ? t0 : t1;
#pragma unroll
        for (int k = 0; k < L; ++k) {
            const double y = (Y[k] - lu[5 * k] * ya) - lu[5 * k + 1] * yb;
            Y[k] = y;
            ya = yb;
            yb = y;
        }
    }
    double h0 = 0.0, h1 = 0.0;
    if (ln.S > 1) {
        // backward, pass 1: zero incoming values, outgoing values only
        {
            double xa = 0.0, xb = 0.0;
#pragma unroll
            for (int k = L - 1; k >= 0; --k) {
                const double x = (lu[5 * k + 2] * Y[k] - lu[5 * k + 3] * xa) - lu[5 * k + 4] * xb;
                xb = xa;
                xa = x;
            }
            __syncthreads();
            ex[ln.exi] = odd ? xb : xa;
            ex[ln.exs + ln.exi] = odd ? xa : xb;
            __syncthreads();
        }
        // incoming values x(b), x(b+1): scan over the segments after this one
        if (ln.ok) {
            for (int sp = ln.S - 1; sp > s; --sp) {
                const double *m = SM + 8 * sp + 4;
                const int xi = ln.exi + (sp - s) * ln.P;
                const double n0 = (m[0] * h0 + m[1] * h1) + ex[xi];
                const double n1 = (m[2] * h0 + m[3] * h1) + ex[ln.exs + xi];
                h0 = n0;
                h1 = n1;
            }
        }
    }
    // backward, pass 2
    {
        double xa = h0, xb = h1;
#pragma unroll
        for (int k = L - 1; k >= 0; --k) {
            const double x = (lu[5 * k + 2] * Y[k] - lu[5 * k + 3] * xa) - lu[5 * k + 4] * xb;
            Y[k] = x;
            xb = xa;
            xa = x;
        }
    }
    // the solution is complete here: keep the compiler from sinking the
    // recurrence into the (per-lane conditional) stores that consume it
#pragma unroll
    for (int k = 0; k < L; ++k) asm volatile("" : "+v"(Y[k]));
}

// Coefficients of the segmented sweeps of one segment length L: at
// BlkDev.pk, per block, scheme and direction, the LU rows as the lanes hold
// them [S][L][5] (pass-through rows in front of a short segment's), then the
// transfer values [S][8].  Laid out once by the host: formed entry by entry
// in the sweep they took 400 of the 3500 instructions of a xi wave.
struct SegTabs {
    const double *pk;
};

// Sinks that read operands of their own at each point (type Pre, filled by
// pre(g, Pre&), written with put_pre(g, x, Pre)): eta/zeta sweeps load them
// for kOutBatch points before storing any.
template <class S, class = void> struct sink_pre : std::false_type {};
template <class S> struct sink_pre<S, std::void_t<typename S::Pre>> : std::true_type {};

// One tile of P pencils of block tile.b along d.
//  Src: load(g, b, Raw&), finish(Raw, b, double (&)[NV])
//  Sink: ends(side, pencil, v, x) and, by sweep and kind,
//        store(g, b, const double (&)[NV]): xi sweeps, all variables of a point;
//        fold(f, x): the value to write given the source f and the result x,
//        put_raw(g, b, v, y): write such a value (eta/zeta sweeps, which still
//        hold the source in registers, and xi ones with kReadBack, which read
//        it back with src(g, v));
//        Pre, pre and put_pre (sink_pre) instead of these
template <int NV, int SCH, int L, int P, bool XI, class Src, class Sink>
__device__ __forceinline__ void seg_tile(const BlkDev *__restrict__ blks, const TabDev *__restrict__ tabs,
                                         const SegTabs &tb, Tile tile, int d, int n45, int SP, const Src &src,
                                         Sink &sink, double *lds)
{
    using Sh = SegShape<NV, SCH, L, P, XI>;
    constexpr int H = Sh::H;
    const int nthr = NV * P * SP;
    const int t = threadIdx.x;
    // (one variable: t < P SP, so v = 0 and s = t / P without dividing by
    // the run-time SP)
    const int v = NV == 1 ? 0 : t / (P * SP), p = t % P, s = NV == 1 ? t / P : (t / P) % SP;
    const int b = tile.b;
    const BlkDev &B = blks[b];
    const TabDev &T = tabs[B.inst];
    const double fa = SCH == 1 ? T.fa : 0.0, fb = SCH == 1 ? T.fb : 0.0, fc = SCH == 1 ? T.fc : 0.0;
    const int npen = npencils(B, d);
    const int n = B.n[d], N = n - 1;
    // (read here, with the first round of loads, not at the uses behind the barriers)
    const int qds[2] = {B.qd[d][0], B.qd[d][1]}, parts[2] = {B.part[d][0], B.part[d][1]};
    const int codes[2] = {B.bc[d][0], B.bc[d][1]};
    const int S = seg_count(n, L);
    const double *PK = tb.pk + B.pk[l_index(L)][SCH][d];
    const int nlu = 5 * L * SP, nluS = 5 * L * S;   // (idle lanes' rows are not set)
    double *buf = lds;   // xi: the tile
    double *ends = nullptr, *part = nullptr, *LUs = nullptr, *ex = nullptr;
    double *SM = nullptr;   // [SP][8]
    const int exs2 = 2 * NV * SP * P;
    if constexpr (XI) {
        const int fsz = NV * P * Sh::pencil_stride(n) + 2 * kTilePad;
        buf = lds + kTilePad;
        LUs = lds;
        ex = lds + nlu;
        SM = lds + (fsz > nlu + exs2 ? fsz : nlu + exs2);
        part = SM + 8 * SP;
    } else {
        static_assert(NV == 1, "an eta or zeta workgroup sweeps one field");
        constexpr int esz = 2 * kSegEndRows * P;
        ends = lds;
        ex = lds;
        SM = lds + (esz > exs2 ? esz : exs2);
        LUs = SM + 8 * SP;
        part = LUs + nlu;
    }
    // xi: staged source of the lane's variable and pencil at row; the place
    // of tile point e (pencil e / n, row e % n) of variable 0; variable m
    // follows FS doubles further on
    const int NS = Sh::pencil_stride(n), FS = P * NS;
    auto F = [&](int row) { return buf[(v * P + p) * NS + row]; };
    // (e + e / n for even n: exact for e < 2^32 / n, one multiplication)
    const unsigned inv_n = (n & 1) ? 0u : 0xffffffffu / unsigned(n) + 1u;
    auto place = [&](int e) { return e + int(__umulhi(unsigned(e), inv_n)); };
    const bool pen_ok = tile.q0 + p < npen;
    const bool lane_ok = pen_ok && s < S;
    int a, len;   // (lanes without a segment: the last one's, so that what they load is in the block)
    seg_bounds(n, L, S, s < S ? s : S - 1, a, len);
    const int kb = L - len;                 // row a - kb + k is held in Y[k], kb <= k < L
    // (a segment has at least seg_min_rows(L) rows)
    auto have = [&](int k) { return k >= L - seg_min_rows(L) || k >= kb; };
    auto pt = [&](int pp, int i) -> int64_t {
        int64_t pb, st;
        pencil_of(B, d, tile.q0 + pp, pb, st);
        return pb + int64_t(i) * st;
    };
    auto eidx = [&](int side, int i, int m, int pp) { return ((side * kSegEndRows + i) * NV + m) * P + pp; };

    // ---- 0. every segment's LU rows as its lanes hold them ([SP][L][5]:
    //         pass-through rows, then the segment's rows; a thread's loads are
    //         issued together, kLuBatch per round trip) and the segments'
    //         transfer values into LDS
    // xi: the first KPRE values per thread are loaded once the tile is
    // staged (their latency overlaps the right-hand sides and closure rows)
    // and written over the tile afterwards
    constexpr int KPRE0 = (5 * L + NV * P - 1) / (NV * P);
    constexpr int KPRE = KPRE0 < kLuBatch ? KPRE0 : kLuBatch;
    double lv[KPRE];
    auto lu_fetch = [&]() {
#pragma unroll
        for (int u = 0; u < KPRE; ++u) lv[u] = PK[t + u * nthr < nluS ? t + u * nthr : nluS - 1];
    };
    auto lu_store = [&]() {
#pragma unroll
        for (int u = 0; u < KPRE; ++u)
            if (t + u * nthr < nluS) LUs[t + u * nthr] = lv[u];
        if constexpr (KPRE0 > kLuBatch)
            for (int i0 = t + KPRE * nthr; i0 < nluS; i0 += kLuBatch * nthr) {
                double w2[kLuBatch];
#pragma unroll
                for (int u = 0; u < kLuBatch; ++u) w2[u] = PK[i0 + u * nthr < nluS ? i0 + u * nthr : nluS - 1];
#pragma unroll
                for (int u = 0; u < kLuBatch; ++u)
                    if (i0 + u * nthr < nluS) LUs[i0 + u * nthr] = w2[u];
            }
    };
    if constexpr (!XI) {
        lu_fetch();
        lu_store();
    }
    for (int i = t; i < 8 * S; i += nthr) SM[i] = PK[nluS + i];

    // ---- 1. stream the segment (with H halo points each side): interior
    //         right-hand sides into registers, end values into LDS
    double Y[L];
#pragma unroll
    for (int k = 0; k < L; ++k) Y[k] = 0.0;
    double W[Sh::KR];   // eta/zeta: the lane's source rows
    int64_t pb = 0, st = 0;   // and its pencil
    double w[2 * H + 1];
#pragma unroll
    for (int m = 0; m <= 2 * H; ++m) w[m] = 0.0;
    if constexpr (XI) {
        // stage all points of the tile at once, consecutive threads on
        // consecutive points: a thread has P n / (NV P SP) <= L / NV points
        // (segments hold at most L), so BX slots take them in one round
        constexpr int BX = (L + NV - 1) / NV;
        const int tot = P * n;
        const int64_t g0 = pt(0, 0);
        const int elim = (npen - tile.q0 < P ? npen - tile.q0 : P) * n;   // points of the tile inside the block
        __syncthreads();
        for (int e0 = t; e0 < tot; e0 += nthr * BX) {
            typename Src::Raw raw[BX];
            int dst[BX];
#pragma unroll
            for (int kk = 0; kk < BX; ++kk) {
                const int e = e0 + kk * nthr;
                const bool ok = e < elim;
                src.load(ok ? g0 + e : g0, b, raw[kk]);
                dst[kk] = ok ? place(e) : -1;
            }
#pragma unroll
            for (int kk = 0; kk < BX; ++kk) {
                if (dst[kk] < 0) continue;
                double f[NV];
                src.finish(raw[kk], b, f);
#pragma unroll
                for (int m = 0; m < NV; ++m) buf[dst[kk] + m * FS] = f[m];
            }
        }
        __syncthreads();
        lu_fetch();
        const double *rows_in = &buf[(v * P + p) * NS + (a - kb - H)];
#pragma unroll
        for (int kr = 0; kr < Sh::KR; ++kr) {
            const double fv = rows_in[kr];
#pragma unroll
            for (int m = 0; m < 2 * H; ++m) w[m] = w[m + 1];
            w[2 * H] = fv;
            const int k = kr - 2 * H;
            if (k < 0 || k >= L) continue;
            // interior rows; the closure rows are replaced below and the
            // pass-through registers cleared
            double rr;
            if constexpr (SCH == 0) {
                rr = kAa * (w[3] - w[1]) + kAb * (w[4] - w[0]);
            } else {
                const double resk = w[3] + w[3];
                rr = (fa * ((w[2] + w[4]) - resk) + fb * ((w[1] + w[5]) - resk)) +
                     fc * ((w[0] + w[6]) - resk);
            }
            Y[k] = rr;
        }
    } else {
        // eta/zeta: each lane loads its own rows, all at once.
        // The lanes of a wave hold P neighbouring pencils, so one load
        // instruction reads runs of P consecutive points.  Rows outside the
        // lane's window are clamped into it (loaded but never used); those of
        // the fewest rows a segment has need no clamp, and their places differ
        // by the same offsets in all lanes.
        const int ppc = tile.q0 + p < npen ? p : npen - 1 - tile.q0;
        pencil_of(B, d, tile.q0 + ppc, pb, st);
        const int r0 = a - kb - H;                 // row held in W[0]
        const int rlo = (a - H) > 0 ? a - H : 0;
        const int rhi = (a + len + H - 1) < N ? a + len + H - 1 : N;
        const int64_t g0 = pb + int64_t(r0) * st;
#pragma unroll
        for (int kr = 0; kr < Sh::KR; ++kr) {
            if (kr >= L - seg_min_rows(L) + H && kr < L + H) {
                W[kr] = src.field(g0 + int64_t(kr) * st, v);
            } else {
                // (n >= 13 along the other directions: st < 2^31)
                int row = r0 + kr;
                row = row < rlo ? rlo : (row > rhi ? rhi : row);
                W[kr] = src.field(pb + int64_t(uint64_t(unsigned(row)) * unsigned(st)), v);
            }
        }
        // the 13 points next to each pencil end, for the closure rows, from the
        // lanes whose rows they are
        if (lane_ok && (a <= kSegEnd || N - (a + len - 1) <= kSegEnd)) {
#pragma unroll
            for (int k = 0; k < L; ++k) {
                const int row = a - kb + k;
                if (k < kb) continue;
                if (row <= kSegEnd) ends[eidx(0, row, v, p)] = W[k + H];
                if (N - row <= kSegEnd) ends[eidx(1, N - row, v, p)] = W[k + H];
            }
        }
        // row a - kb + k: stencil W[k .. k + 2H] (interior rows; the closure
        // rows are replaced below and the pass-through registers cleared)
#pragma unroll
        for (int k = 0; k < L; ++k) {
            double rr;
            if constexpr (SCH == 0) {
                rr = kAa * (W[k + 3] - W[k + 1]) + kAb * (W[k + 4] - W[k]);
            } else {
                const double resk = W[k + 3] + W[k + 3];
                rr = (fa * ((W[k + 2] + W[k + 4]) - resk) + fb * ((W[k + 1] + W[k + 5]) - resk)) +
                     fc * ((W[k] + W[k + 6]) - resk);
            }
            Y[k] = rr;
        }
    }

    // the pass-through registers start at zero (a segment has at least
    // seg_min_rows(L) rows, so only the first L - seg_min_rows(L) can be such)
#pragma unroll
    for (int k = 0; k < L - seg_min_rows(L); ++k)
        if (k < kb) Y[k] = 0.0;

    // ---- 2. partner points of interfaces with another block (one round) ------
    bool self[2];
    for (int side = 0; side < 2; ++side) self[side] = qds[side] != 0 && parts[side] == b;
    const bool stage_part = (qds[0] != 0 && !self[0]) || (qds[1] != 0 && !self[1]);
    __syncthreads();
    if (stage_part) {
        for (int slot = t; slot < 2 * kSegEndRows * P; slot += nthr) {
            const int pp = slot % P, o = (slot / P) % kSegEndRows, side = slot / (P * kSegEndRows);
            if (tile.q0 + pp >= npen || qds[side] == 0 || self[side]) continue;
            const int Pb = parts[side];
            const BlkDev &BP = blks[Pb];
            const int ps = 1 - side, code = codes[side];
            const int iik = code == 40 ? 0 : 1;
            const int NP = BP.n[d] - 1;
            const int idx = o == kSegEnd ? (ps == 0 ? 0 : NP) : (ps == 0 ? o + iik : NP - (o + iik));
            int64_t pb, pst;
            pencil_of(BP, d, tile.q0 + pp, pb, pst);
            typename Src::Raw raw;
            src.load(pb + int64_t(idx) * pst, Pb, raw);
            double f[NV];
            src.finish(raw, Pb, f);
#pragma unroll
            for (int m = 0; m < NV; ++m) part[eidx(side, o, m, pp)] = f[m];
        }
        __syncthreads();
    }

    // ---- 3. closure rows at both ends (same arithmetic as the sequential sweep)
    double lo[3] = {0.0, 0.0, 0.0}, hi[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        if (!(lane_ok && s == (side == 0 ? 0 : S - 1))) continue;
        // distance i from this end
        auto f = [&](int i) { return XI ? F(side == 0 ? i : N - i) : ends[eidx(side, i, v, p)]; };
        const bool qd = qds[side] != 0;
        double rows[3] = {0.0, 0.0, 0.0};
        if (qd) {
            const int ps = 1 - side, code = codes[side];   // the partner's opposite face has the same
            const int iik = code == 40 ? 0 : 1;
            const double ra0k = code == 45 ? double(n45) : 0.0;
            // partner point o (o = 12: the partner's face point)
            auto g = [&](int o) {
                if (self[side]) {
                    const int i = o == kSegEnd ? 0 : o + iik;   // distance from the partner's end ps
                    return XI ? F(ps == 0 ? i : N - i) : ends[eidx(ps, i, v, p)];
                }
                return part[eidx(side, o, v, p)];
            };
            double r0 = 0.0, r1 = 0.0, sap0 = 0.0;
            for (int i = 0; i < kSegEnd; ++i) {
                const double fp = g(i);
                if (i == 0) sap0 = fp;
                r0 = r0 + T.qout[SCH][0][i] * fp;
                r1 = r1 + T.qout[SCH][1][i] * fp;
            }
            const double resk = ra0k != 0.0 ? ra0k * g(kSegEnd) : 0.0;
            r0 = r0 - resk * T.qsum[SCH][0];
            r1 = r1 - resk * T.qsum[SCH][1];
            double r2 = sap0 - resk;
            if (n45 == 1 && codes[side] == 45) {
                const double fo = f(0);
                r0 = r0 + fo * T.qsum[SCH][0];
                r1 = r1 + fo * T.qsum[SCH][1];
                r2 = r2 + double(SCH) * fo;
            }
            double a0 = 0.0, a1 = 0.0;
            for (int i = 0; i < kSegEnd; ++i) {
                a0 = a0 + T.qin[SCH][0][i] * f(i);
                a1 = a1 + T.qin[SCH][1][i] * f(i);
            }
            if (SCH == 0) {
                rows[0] = side == 0 ? a0 + r0 : -a0 - r0;
                rows[1] = side == 0 ? a1 + r1 : -a1 - r1;
            } else {
                rows[0] = a0 + r0;
                rows[1] = a1 + r1;
                const double ra2k = f(2) + f(2);
                if (side == 0)
                    rows[2] = (fa * ((f(1) + f(3)) - ra2k) + fb * ((f(0) + f(4)) - ra2k)) +
                              fc * ((r2 + f(5)) - ra2k);
                else
                    rows[2] = (fa * ((f(3) + f(1)) - ra2k) + fb * ((f(4) + f(0)) - ra2k)) +
                              fc * ((f(5) + r2) - ra2k);
            }
        } else if (SCH == 0) {
            double sum = 0.0;
            if (side == 0) {
                sum = sum + kA01 * (f(1) - f(0)); sum = sum + kA02 * (f(2) - f(0));
                sum = sum + kA03 * (f(3) - f(0)); sum = sum + kA04 * (f(4) - f(0));
                rows[0] = sum;
                sum = 0.0;
                sum = sum + kA10 * (f(0) - f(1)); sum = sum + kA12 * (f(2) - f(1));
                sum = sum + kA13 * (f(3) - f(1)); sum = sum + kA14 * (f(4) - f(1));
                rows[1] = sum;
            } else {
                sum = sum + kA01 * (f(0) - f(1)); sum = sum + kA02 * (f(0) - f(2));
                sum = sum + kA03 * (f(0) - f(3)); sum = sum + kA04 * (f(0) - f(4));
                rows[0] = sum;
                sum = 0.0;
                sum = sum + kA10 * (f(1) - f(0)); sum = sum + kA12 * (f(1) - f(2));
                sum = sum + kA13 * (f(1) - f(3)); sum = sum + kA14 * (f(1) - f(4));
                rows[1] = sum;
            }
        } else {
            const int o0[5] = {1, 2, 3, 4, 5}, o1[5] = {0, 2, 3, 4, 5}, o2[5] = {0, 1, 3, 4, 5};
            double sum = 0.0;
            for (int cc = 0; cc < 5; ++cc) sum = sum + T.fbc[0][cc] * (f(o0[cc]) - f(0));
            rows[0] = sum;
            sum = 0.0;
            for (int cc = 0; cc < 5; ++cc) sum = sum + T.fbc[1][cc] * (f(o1[cc]) - f(1));
            rows[1] = sum;
            sum = 0.0;
            for (int cc = 0; cc < 5; ++cc) sum = sum + T.fbc[2][cc] * (f(o2[cc]) - f(2));
            rows[2] = sum;
        }
        for (int r = 0; r < 3; ++r) (side == 0 ? lo : hi)[r] = rows[r];
    }
    // closure rows: rows 0..NB-1 open segment 0; rows N-r close the last one
    if (lane_ok && s == 0) {       // row r is Y[kb + r]
#pragma unroll
        for (int r = 0; r < Sh::NB; ++r)
#pragma unroll
            for (int k = 0; k <= L - seg_min_rows(L) + r; ++k)
                if (k == kb + r) Y[k] = lo[r];
    }
    if (lane_ok && s == S - 1) {   // row N is Y[L - 1]
#pragma unroll
        for (int r = 0; r < Sh::NB; ++r) Y[L - 1 - r] = hi[r];
    }

    if constexpr (XI) {   // the tile is no longer read: LU rows over it
        __syncthreads();
        lu_store();
        __syncthreads();
    }

    // ---- 4. solve ---------------------------------------------------------------
    const SegLane ln{kb, s, S, lane_ok, (v * SP + s) * P + p, NV * SP * P, P};
    seg_solve<L>(Y, ln, LUs, SM, ex);
    if (lane_ok && s == 0) {
        double x0 = 0.0;
#pragma unroll
        for (int k = 0; k <= L - seg_min_rows(L); ++k)
            if (k == kb) x0 = Y[k];
        sink.ends(0, p, v, x0);
    }
    if (lane_ok && s == S - 1) sink.ends(1, p, v, Y[L - 1]);

    // ---- 5. results ------------------------------------------------------------
    if constexpr (!XI) {
        // eta/zeta: lanes of a wave hold P neighbouring pencils, stores coalesce
        if (lane_ok) {
            pb += int64_t(a - kb) * st;
            if constexpr (sink_pre<Sink>::value) {
                static_assert(!Sink::kReadBack, "prefetching sinks write results as they are");
#pragma unroll
                for (int k0 = 0; k0 < L; k0 += kOutBatch) {
                    typename Sink::Pre pr[kOutBatch];
#pragma unroll
                    for (int kk = 0; kk < kOutBatch; ++kk)
                        if (k0 + kk < L && have(k0 + kk)) sink.pre(pb + int64_t(k0 + kk) * st, pr[kk]);
#pragma unroll
                    for (int kk = 0; kk < kOutBatch; ++kk)
                        if (k0 + kk < L && have(k0 + kk)) sink.put_pre(pb + int64_t(k0 + kk) * st, Y[k0 + kk], pr[kk]);
                }
            } else {
#pragma unroll
                for (int k = 0; k < L; ++k)
                    if (have(k)) sink.put_raw(pb + int64_t(k) * st, b, v, sink.fold(W[k + H], Y[k]));
            }
        }
    } else {
        // xi: results into the tile buffer, then stored along the pencils
        // (the filter's sink adds them to the sources it reads back)
        __syncthreads();
        if (lane_ok) {
#pragma unroll
            for (int k = 0; k < L; ++k)
                if (have(k)) {
                    buf[(v * P + p) * NS + (a - kb + k)] = Y[k];
                }
        }
        __syncthreads();
        const int tot = P * n;
        const int64_t g0 = pt(0, 0);
        const int elim = (npen - tile.q0 < P ? npen - tile.q0 : P) * n;   // points of the tile inside the block
        if constexpr (Sink::kReadBack) {
            // the sink adds the results to its sources: read those back for
            // kOutBatch points at a time, all loads in flight together
            for (int e0 = t; e0 < tot; e0 += kOutBatch * nthr) {
                double fs[kOutBatch][NV];
                int li[kOutBatch];   // LDS place of the point's results, -1: none
#pragma unroll
                for (int kk = 0; kk < kOutBatch; ++kk) {
                    const int e = e0 + kk * nthr;
                    const bool ok = e < elim;
                    li[kk] = ok ? place(e) : -1;
#pragma unroll
                    for (int m = 0; m < NV; ++m) fs[kk][m] = sink.src(ok ? g0 + e : g0, m);
                }
#pragma unroll
                for (int kk = 0; kk < kOutBatch; ++kk) {
                    if (li[kk] < 0) continue;
                    const int64_t g = g0 + (e0 + kk * nthr);
#pragma unroll
                    for (int m = 0; m < NV; ++m) sink.put_raw(g, b, m, sink.fold(fs[kk][m], buf[li[kk] + m * FS]));
                }
            }
        } else if constexpr (sink_pre<Sink>::value) {
            // the sink's own operands of kOutBatch points in flight together
            static_assert(NV == 1, "prefetching sinks take one variable");
            for (int e0 = t; e0 < tot; e0 += kOutBatch * nthr) {
                typename Sink::Pre pr[kOutBatch];
                int li[kOutBatch];
#pragma unroll
                for (int kk = 0; kk < kOutBatch; ++kk) {
                    const int e = e0 + kk * nthr;
                    const bool ok = e < elim;
                    li[kk] = ok ? place(e) : -1;
                    sink.pre(ok ? g0 + e : g0, pr[kk]);
                }
#pragma unroll
                for (int kk = 0; kk < kOutBatch; ++kk)
                    if (li[kk] >= 0) sink.put_pre(g0 + (e0 + kk * nthr), buf[li[kk]], pr[kk]);
            }
        } else {
            for (int e = t; e < elim; e += nthr) {
                const int li = place(e);
                double x[NV];
#pragma unroll
                for (int m = 0; m < NV; ++m) x[m] = buf[li + m * FS];
                sink.store(g0 + e, b, x);
            }
        }
    }

}

}  // namespace cnd
