// LDS-resident FFT pass kernels for CDNA4 (gfx950).
//
// One workgroup owns a tile of C lines of length L.  The tile is loaded from
// HBM once (coalesced along the line for row passes, across adjacent lines for
// column passes), every radix stage of the length-L transform runs out of
// LDS through VGPRs, and the tile is written back once -- one HBM round trip
// per pass.  Element-wise work that the reference runs as separate sweeps
// (ele_mul, fused_twiddle_transpose, recombine/separate) is folded into the
// load or store of the adjacent pass.
//
// The first stage takes its operands straight from HBM and the last stage
// stores straight to it.  In between a line sits in LDS as mixed-radix digits
// and stage s transforms digit s in place: a butterfly writes the positions
// that it read, so a stage needs one barrier, one set of addresses, no
// registers held across a barrier and no particular number of butterflies per
// thread (threads loop over the line's butterflies).  The output order comes
// from the last stage's numbering of its butterflies.  What bounds it: vector
// issue and LDS latency rather than HBM, at 75 VALU instructions per element
// for three stages (a self-sorting form with its results moved and guarded
// took 112).  Measured, before -> after: 3001 complex64 lines of 1200
// (12 x 10 x 10) 26.7 -> 17.9 us; 9 lines of 1,000,000, then planned as three
// passes of 100, 187 -> 112 us; 1500 complex128 lines of 1009 (Bluestein, M =
// 2048) 37.1 -> 30.8 us; 2000 uneven items 2.87 -> 2.32 ms.  (The reference's
// self-sorting geometry, core/solvers/complex/pow2_iterative_solver_dft.c:27-78,
// moves every stage's results instead.)
//
// Included by the instantiation units kernels_pass_{f32,f64}_{mixed,pow2,light}.hip,
// kernels_pass_f64_to8.hip and kernels_batch_{f32,f64}_{small,medium,large}.hip (compiled in
// parallel); kernels.hip holds the launch-table dispatch.
#pragma once

#include <hip/hip_runtime.h>

#include "codelets.h"
#include "kernels.h"
#include "pass.h"

namespace fftz {

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f)
{
    return (__umulhi(n, f.mul) + n) >> f.shift;
}

struct LineIdx {
    int64_t ioff, ooff;
    uint32_t l0;
    int64_t gin, gout;  // sequence index of the line's element 0 (kChirpFlags)
};

// The buffers and line set a pass body works on: the descriptor's own for a
// single-size pass, the queue entry's for the uneven-batch kernel (which reads
// its size class's descriptor in place and never patches it).
struct TileIo {
    const void* in;
    void* out;
    int64_t nlines;
    int64_t ils0, ols0;  // line strides of level 0
};

__device__ __forceinline__ TileIo io_of(const PassDesc& p)
{
    return TileIo{p.in, p.out, p.nlines, p.ils[0], p.ols[0]};
}

__device__ __forceinline__ LineIdx line_index(const PassDesc& p, const TileIo& io, uint32_t l)
{
    uint32_t r = fdiv(l, p.ln0);
    uint32_t l0 = l - r * p.ln0.d;
    uint32_t l2 = fdiv(r, p.ln1);
    uint32_t l1 = r - l2 * p.ln1.d;
    LineIdx li;
    li.ioff = (int64_t)l0 * io.ils0 + (int64_t)l1 * p.ils[1] + (int64_t)l2 * p.ils[2];
    li.ooff = (int64_t)l0 * io.ols0 + (int64_t)l1 * p.ols[1] + (int64_t)l2 * p.ols[2];
    li.l0 = l0;
    li.gin = li.gout = 0;
    if (p.flags & kChirpFlags) {
        li.gin = p.gin_base + (int64_t)l0 * p.gin[0] + (int64_t)l1 * p.gin[1] + (int64_t)l2 * p.gin[2];
        li.gout = p.gout_base + (int64_t)l0 * p.gout[0] + (int64_t)l1 * p.gout[1] + (int64_t)l2 * p.gout[2];
    }
    return li;
}

// Line held by tile slot c (l_base = tile index x C): line l_base + c for
// flat tiles; for ragged column tiles the slot's row and position in the row
// (PassDesc::vrow), live only below the row length.
struct SlotLine {
    uint32_t l;
    bool live;
};

__device__ __forceinline__ SlotLine slot_line(const PassDesc& p, const TileIo& io, int64_t l_base, int c)
{
    const int64_t v = l_base + c;
    if (p.vrow.d == 0) return SlotLine{(uint32_t)v, v < io.nlines};
    const uint32_t row = fdiv((uint32_t)v, p.vrow);
    const uint32_t cc = (uint32_t)v - row * p.vrow.d;
    const uint32_t l = row * p.ln0.d + cc;
    return SlotLine{l, cc < p.ln0.d && (int64_t)l < io.nlines};
}

// w_N^p from the two-level FP64 table: hi[p >> b] * lo[p & (2^b - 1)].
__device__ __forceinline__ cplx<double> tw4_root(const PassDesc& p, int64_t q)
{
    const cplx<double>* t = reinterpret_cast<const cplx<double>*>(p.tw4);
    const int64_t lo_n = (int64_t)1 << p.tw4_lobits;
    cplx<double> lo = t[q & (lo_n - 1)];
    cplx<double> hi = t[lo_n + (q >> p.tw4_lobits)];
    return cmul(hi, lo);
}

__device__ __forceinline__ uint32_t sdiv(uint32_t n, const SmallDiv& f) { return __umul24(n, f.mul) >> f.shift; }

// Workgroup barrier that waits only for this wave's LDS traffic (the stages
// exchange data through LDS alone; twiddle loads and result stores in flight
// are not waited for).  Lines that sit in one wavefront each need no barrier:
// a wave's own LDS operations complete in order once counted down.
__device__ __forceinline__ void stage_sync(bool wave_local)
{
    if (wave_local)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---------------------------------------------------------------------------
// LDS positions.  A line is kept as mixed-radix digits: position
// d0 A0 + d1 A1 + ... + d(S-1), As = p.st[s].lst, where digit s holds the input
// digit n_s before stage s and the output digit k_s after it (input index
// n0 L/R0 + n1 L/(R0 R1) + ..., output index k0 + R0 k1 + R0 R1 k2 + ...).
// Stage s transforms digit s, so it reads and writes the same R_s positions.
// ---------------------------------------------------------------------------

// Leg 0 of butterfly j of the last stage (j = k0 + R0 k1 + ..., so that the
// outputs j + i L/R of neighbouring lanes are neighbours); legs are adjacent.
__device__ __forceinline__ int last_base(const PassDesc& p, int j)
{
    const int S = p.nst;
    uint32_t rem = (uint32_t)j, base = 0;
    for (int s = 0; s + 2 < S; s++) {
        const uint32_t q = sdiv(rem, p.st[s].rdiv);
        base += __umul24(rem - __umul24(q, (uint32_t)p.st[s].radix), (uint32_t)p.st[s].lst);
        rem = q;
    }
    return (int)(base + __umul24(rem, (uint32_t)p.st[S - 2].lst));
}

// Leg 0 of butterfly j of a middle stage s; m is the index below digit s
// (the stage's twiddle column).  Digit 0 runs fastest over the lanes: its odd
// stride spreads them over the LDS banks whatever the later radices are, and
// neighbouring lanes share a twiddle.
__device__ __forceinline__ int mid_base(const PassDesc& p, int s, int j, uint32_t& m)
{
    const uint32_t q = sdiv((uint32_t)j, p.st[0].rdiv);
    const uint32_t d0 = (uint32_t)j - __umul24(q, (uint32_t)p.st[0].radix);
    const uint32_t o = sdiv(q, p.st[s].mdiv);
    m = q - __umul24(o, (uint32_t)p.st[s].lst);
    return (int)(__umul24(d0, (uint32_t)p.st[0].lst) + __umul24(o, (uint32_t)(p.st[s].radix * p.st[s].lst)) + m);
}

// Stage twiddles, one row per output digit k >= 1 and one column per index m
// below the digit: w_{Rs As}^(k m).
template <typename R>
__device__ __forceinline__ const cplx<R>* stage_tw(const PassDesc& p, int s)
{
    return reinterpret_cast<const cplx<R>*>(p.stw) + p.st[s].twoff;
}

template <typename R, int RAD>
__device__ __forceinline__ void load_twiddles(const cplx<R>* tw, uint32_t m, int cols, cplx<R> (&w)[RAD - 1])
{
#pragma unroll
    for (int i = 0; i < RAD - 1; i++) w[i] = tw[m + (uint32_t)(i * cols)];
}

template <typename R, int RAD>
__device__ __forceinline__ void apply_twiddles(cplx<R> (&v)[RAD], const cplx<R> (&w)[RAD - 1])
{
#pragma unroll
    for (int i = 1; i < RAD; i++) v[i] = cmul(v[i], w[i - 1]);
}

// Whether a stage asks for its twiddles only after its DFT.  Radix 11, 13 and 16
// in complex128 hold 44 to 64 registers of operands and nearly as many of
// twiddles, which decided the registers of every plain pass of kRadAll (199, two
// wavefronts per SIMD, or 66 spilled at three; now 167) and made kRadLight spill
// (168 and 4; now 161).  2666 lines of 1573 (13 x 11 x 11) 34.6 -> 30.8 us, the
// 100 x 120 x 144 grid (16 x 9) there and back 85.5 -> 80.9, 104 chirp-z
// transforms of 20011 (passes of 220 and 182) 177 -> 166.
template <typename R, int RADSET, int RAD>
constexpr bool kLateTw = sizeof(R) == 8 && (RADSET == kRadAll || RADSET == kRadLight) &&
                         (RAD == 11 || RAD == 13 || RAD == 16);

// Middle stage in place: DFT then twiddle (decimation in frequency), or, for
// the second transform of a Bluestein pass, twiddle then DFT with the same
// table (decimation in time: digits return from output to input order).
// Addresses and twiddles of the first butterfly are fetched before the
// barrier that makes the previous stage's results visible: their latency
// (tables of long lines live in the L2 or beyond) overlaps the barrier.
// LATE: twiddles after the DFT (kLateTw).
template <typename R, int RAD, bool DIT, bool LATE>
__device__ __forceinline__ void mid_stage(const PassDesc& p, cplx<R>* line, int t, int s, bool live, bool wave_local)
{
    const int nbl = live ? p.st[s].nbl : 0, step = p.st[s].lst;
    const cplx<R>* tw = stage_tw<R>(p, s);
    static_assert(!(DIT && LATE));
    int j = t, base = 0;
    uint32_t m = 0;
    cplx<R> w[RAD - 1];
    auto fetch = [&]() {
        if (j < nbl) {
            base = mid_base(p, s, j, m);
            if constexpr (!LATE) load_twiddles<R, RAD>(tw, m, step, w);
        }
    };
    fetch();
    stage_sync(wave_local);
#pragma unroll 1
    while (j < nbl) {
        cplx<R>* q = line + base;
        cplx<R> v[RAD];
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = q[i * step];
        if constexpr (DIT) apply_twiddles<R, RAD>(v, w);
        Dft<RAD, R>::run(v);
        if constexpr (LATE) {
            __builtin_amdgcn_sched_barrier(0);
            load_twiddles<R, RAD>(tw, m, step, w);
        }
        if constexpr (!DIT) apply_twiddles<R, RAD>(v, w);
#pragma unroll
        for (int i = 0; i < RAD; i++) q[i * step] = v[i];
        j += p.TL;
        fetch();
    }
}

#define FFTZ_RADIX_CASE(RADSET, r, CALL)            \
    case r:                                         \
        if constexpr (rad_in_set((RADSET), r)) {    \
            constexpr int RAD = r;                  \
            CALL;                                   \
        }                                           \
        break;

#define FFTZ_RADIX_SWITCH(rad, RADSET, CALL)        \
    switch (rad) {                                  \
        FFTZ_RADIX_CASE(RADSET, 2, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 3, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 4, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 5, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 6, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 7, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 8, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 9, CALL)            \
        FFTZ_RADIX_CASE(RADSET, 10, CALL)           \
        FFTZ_RADIX_CASE(RADSET, 11, CALL)           \
        FFTZ_RADIX_CASE(RADSET, 12, CALL)           \
        FFTZ_RADIX_CASE(RADSET, 13, CALL)           \
        FFTZ_RADIX_CASE(RADSET, 16, CALL)           \
        default: break;                             \
    }

// Radices of the stage that holds mirrored butterfly pairs (kRealPair: up to
// 10, kRealWide: 11 and 13, and 12 and 16 where a tuned order asks for them).
#define FFTZ_PAIR_CASE(RADSET, r, CALL)             \
    case r:                                         \
        if constexpr (rad_in_pairs((RADSET), r)) {  \
            constexpr int RAD = r;                  \
            CALL;                                   \
        }                                           \
        break;

#define FFTZ_PAIR_SWITCH(rad, RADSET, REAL, CALL)   \
    if constexpr (REAL == kRealWide) {              \
        switch (rad) {                              \
            FFTZ_RADIX_CASE(kRadAll, 11, CALL)      \
            FFTZ_RADIX_CASE(kRadAll, 12, CALL)      \
            FFTZ_RADIX_CASE(kRadAll, 13, CALL)      \
            FFTZ_RADIX_CASE(kRadAll, 16, CALL)      \
            default: break;                         \
        }                                           \
    } else {                                        \
        switch (rad) {                              \
            FFTZ_PAIR_CASE(RADSET, 2, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 3, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 4, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 5, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 6, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 7, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 8, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 9, CALL)         \
            FFTZ_PAIR_CASE(RADSET, 10, CALL)        \
            default: break;                         \
        }                                           \
    }

// ---------------------------------------------------------------------------
// HBM side.  The first stage loads its butterflies' operands x[i nbl + j]
// straight into registers and the last stage stores y[i nbl + j] straight from
// them, both coalesced over j.
// ---------------------------------------------------------------------------

// Two adjacent real elements as one complex value; a real line may start at
// an odd element, so only the real type's alignment is assumed.
template <typename R>
struct RealPair {
    typedef R vec __attribute__((ext_vector_type(2), aligned(sizeof(R))));
};

template <typename R>
__device__ __forceinline__ cplx<R> load_pair(const R* s, int64_t es)
{
    if (es == 1) {
        const auto w = *reinterpret_cast<const typename RealPair<R>::vec*>(s);
        return {w.x, w.y};
    }
    return {s[0], s[es]};
}

template <typename R>
__device__ __forceinline__ void store_pair(R* d, int64_t es, cplx<R> v)
{
    if (es == 1) {
        typename RealPair<R>::vec w;
        w.x = v.x;
        w.y = v.y;
        *reinterpret_cast<typename RealPair<R>::vec*>(d) = w;
    } else {
        d[0] = v.x;
        d[es] = v.y;
    }
}

// Whether the backward direction's conjugation of the operands waits until the
// stage's twiddles are asked for (conj_operands): conjugating waits for the
// operands, and the twiddles' latency then comes on top.  3001 complex64 lines
// of 1200 backward 14.3 us, 12.6 this way, as forward.  Complex128 has no
// registers to spare for both: either direction loses 1-3%.
template <typename R>
constexpr bool kConjLate = sizeof(R) == 4;

// Operands of butterfly j of stage 0, conjugated for the backward direction
// unless kConjLate.  src is the line's element 0; for the flags that read reals
// it points at real elements.
template <typename R, int RAD, bool REAL>
__device__ __forceinline__ void load_butterfly(const PassDesc& p, const cplx<R>* src, int j, int64_t gbase,
                                               cplx<R> (&v)[RAD])
{
    const int nbl = p.st[0].nbl;
    if constexpr (REAL) {
        const R* s = reinterpret_cast<const R*>(src);
        if (p.flags & kRealIn) {
            const R* q = s + (int64_t)(2 * j) * p.ies;
            const int64_t step = (int64_t)(2 * nbl) * p.ies;
#pragma unroll
            for (int i = 0; i < RAD; i++) v[i] = load_pair<R>(q + i * step, p.ies);
            return;
        }
        if (p.flags & kRealPromote) {
            const R* q = s + (int64_t)j * p.ies;
            const int64_t step = (int64_t)nbl * p.ies;
#pragma unroll
            for (int i = 0; i < RAD; i++) v[i] = {q[i * step], R(0)};
            return;
        }
        if (p.flags & kHermIn) {
            // bins 0..n/2 are stored; bin e > n/2 is conj(bin n - e)
            const int n = p.nvalid_in;
#pragma unroll
            for (int i = 0; i < RAD; i++) {
                const int e = i * nbl + j;
                const bool up = 2 * e > n;
                v[i] = src[(int64_t)(up ? n - e : e) * p.ies];
                if (up) v[i].y = -v[i].y;
            }
        }
    } else if (p.flags & kChirpIn) {
        // x * chirp[g] for g < nchirp, 0 beyond (the input holds only nchirp elements)
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int e = i * nbl + j;
            const int64_t g = gbase + (int64_t)e * p.gin[3];
            v[i] = {R(0), R(0)};
            if (g < p.nchirp) {
                v[i] = src[(int64_t)e * p.ies];
                if (p.flags & kConjIn) v[i].y = -v[i].y;
                v[i] = cmul(v[i], reinterpret_cast<const cplx<R>*>(p.chirp)[g]);
            }
        }
        return;
    }
    if (!REAL || !(p.flags & kHermIn)) {
        const cplx<R>* q = src + (int64_t)j * p.ies;
        const int64_t step = (int64_t)nbl * p.ies;
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = q[i * step];
    }
    if (!kConjLate<R> && (p.flags & kConjIn)) {
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i].y = -v[i].y;
    }
}

// The conjugation that load_butterfly left out (not of kChirpIn's products, nor
// of reals).
template <typename R, int RAD>
__device__ __forceinline__ void conj_operands(const PassDesc& p, cplx<R> (&v)[RAD])
{
    if (kConjLate<R> && (p.flags & (kConjIn | kRealIn | kRealPromote | kChirpIn)) == kConjIn) {
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i].y = -v[i].y;
    }
}

// One result; NT: past the L2's write-back (kNtStore).  A kernel's parameter
// rather than a branch: both forms of the store in one kernel measured 2-3%
// slower (3001 lines of 1200: 16.9 against 16.5 us).
template <typename R, bool NT>
__device__ __forceinline__ void put(cplx<R>* d, cplx<R> v)
{
    if constexpr (NT)
        store_nt<R>(d, v);
    else
        *d = v;
}

// Results y[i nbl + j] of butterfly j of the last stage: fused four-step
// twiddle, scale, Bluestein products, conjugation, store.
template <typename R, int RAD, bool REAL, bool NT>
__device__ __forceinline__ void store_butterfly(const PassDesc& p, cplx<R> (&v)[RAD], int j, int nbl, cplx<R>* dst,
                                                uint32_t l0, int64_t gbase)
{
    if (!REAL && (p.flags & kTw4)) {
        // w_N^(l0 e), e = i*nbl + j: two table products, then an FP64
        // recurrence over i
        cplx<double> wc = tw4_root(p, (int64_t)l0 * j);
        const cplx<double> ws = tw4_root(p, (int64_t)l0 * nbl);
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            cplx<double> vd = {double(v[i].x), double(v[i].y)};
            vd = cmul(vd, wc);
            v[i] = {R(vd.x), R(vd.y)};
            wc = cmul(wc, ws);
        }
    }
    if (p.flags & kScale) {
        const R sc = R(sizeof(R) == 4 ? p.scale_f : p.scale_d);
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = cscale(v[i], sc);
    }
    if (!REAL && (p.flags & (kSpecOut | kChirpOut))) {
        // multi-pass Bluestein: Z = conj(A) * spec after the first M-point
        // transform; conj(chirp) * W after the second (stored for g < n only)
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int64_t g = gbase + (int64_t)(i * nbl + j) * p.gout[3];
            if (p.flags & kSpecOut) {
                v[i] = cmul(cconj(v[i]), reinterpret_cast<const cplx<R>*>(p.spec)[g]);
            } else if (g < p.nchirp) {
                v[i] = cmul(cconj(reinterpret_cast<const cplx<R>*>(p.chirp)[g]), v[i]);
            }
        }
    }
    if (p.flags & kConjOut) {
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i].y = -v[i].y;
    }
    if constexpr (REAL) {
        R* d = reinterpret_cast<R*>(dst);
        if (p.flags & kRealOut) {
            R* q = d + (int64_t)(2 * j) * p.oes;
            const int64_t step = (int64_t)(2 * nbl) * p.oes;
#pragma unroll
            for (int i = 0; i < RAD; i++) store_pair<R>(q + i * step, p.oes, v[i]);
            return;
        }
        if (p.flags & kRealPart) {
#pragma unroll
            for (int i = 0; i < RAD; i++) d[(int64_t)(i * nbl + j) * p.oes] = v[i].x;
            return;
        }
        // promoted real input: only bins 0..n/2 are stored
        const int nvo = p.nvalid_out;
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int e = i * nbl + j;
            if (e < nvo) dst[(int64_t)e * p.oes] = v[i];
        }
        return;
    }
    if (p.flags & kChirpOut) {
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int e = i * nbl + j;
            if (gbase + (int64_t)e * p.gout[3] < p.nchirp) dst[(int64_t)e * p.oes] = v[i];
        }
        return;
    }
    cplx<R>* q = dst + (int64_t)j * p.oes;
    const int64_t step = (int64_t)nbl * p.oes;
#pragma unroll
    for (int i = 0; i < RAD; i++) put<R, NT>(q + i * step, v[i]);
}

// Stage 0 on loaded operands: DFT, twiddle, write digit 0 (lanes contiguous).
// CONJ: v comes from load_butterfly.  LATE: twiddles after the DFT (kLateTw).
template <typename R, int RAD, bool CONJ, bool LATE>
__device__ __forceinline__ void first_to_lds(const PassDesc& p, cplx<R>* line, int j, cplx<R> (&v)[RAD])
{
    cplx<R> w[RAD - 1];
    if constexpr (!LATE) load_twiddles<R, RAD>(stage_tw<R>(p, 0), (uint32_t)j, p.st[0].nbl, w);
    if constexpr (CONJ) conj_operands<R, RAD>(p, v);
    Dft<RAD, R>::run(v);
    if constexpr (LATE) {
        __builtin_amdgcn_sched_barrier(0);
        load_twiddles<R, RAD>(stage_tw<R>(p, 0), (uint32_t)j, p.st[0].nbl, w);
    }
    apply_twiddles<R, RAD>(v, w);
    const int step = p.st[0].lst;
#pragma unroll
    for (int i = 0; i < RAD; i++) line[j + i * step] = v[i];
}

template <typename R, int RAD, bool REAL, bool LATE>
__device__ __forceinline__ void first_stage(const PassDesc& p, cplx<R>* line, int t, const cplx<R>* src, int64_t gbase)
{
    const int nbl = p.st[0].nbl;
#pragma unroll 1
    for (int j = t; j < nbl; j += p.TL) {
        cplx<R> v[RAD];
        load_butterfly<R, RAD, REAL>(p, src, j, gbase, v);
        first_to_lds<R, RAD, true, LATE>(p, line, j, v);
    }
}

template <typename R, int RAD>
__device__ __forceinline__ void last_from_lds(const PassDesc& p, const cplx<R>* line, int j, cplx<R> (&v)[RAD])
{
    const cplx<R>* q = line + last_base(p, j);
#pragma unroll
    for (int i = 0; i < RAD; i++) v[i] = q[i];
    Dft<RAD, R>::run(v);
}

template <typename R, int RAD, bool REAL, bool NT>
__device__ __forceinline__ void last_stage(const PassDesc& p, const cplx<R>* line, int t, cplx<R>* dst, uint32_t l0,
                                           int64_t gbase)
{
    // small radices: several butterflies at a time, for the LDS reads in flight
    constexpr int U = RAD <= 3 ? 4 : RAD <= 5 ? 2 : 1;
    const int nbl = p.st[p.nst - 1].nbl;
#pragma unroll 1
    for (int j = t; j < nbl; j += U * p.TL) {
        cplx<R> v[U][RAD];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (u == 0 || j + u * p.TL < nbl) last_from_lds<R, RAD>(p, line, j + u * p.TL, v[u]);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (u == 0 || j + u * p.TL < nbl)
                store_butterfly<R, RAD, REAL, NT>(p, v[u], j + u * p.TL, nbl, dst, l0, gbase);
    }
}

// One-stage lengths (L <= 16): load, DFT, store, no LDS.
template <typename R, int RAD, bool REAL, bool NT>
__device__ __forceinline__ void single_stage(const PassDesc& p, const cplx<R>* src, cplx<R>* dst, uint32_t l0,
                                             int64_t gin, int64_t gout)
{
    cplx<R> v[RAD];
    load_butterfly<R, RAD, REAL>(p, src, 0, gin, v);
    conj_operands<R, RAD>(p, v);
    Dft<RAD, R>::run(v);
    store_butterfly<R, RAD, REAL, NT>(p, v, 0, 1, dst, l0, gout);
}

// ---------------------------------------------------------------------------
// Real-packed transforms (core/kernels/non_dft/real_packed/packed_rdft_common.h:19-60).
// Bin k and its mirror L - k of the L-point complex transform belong to legs
// i and R-1-i of butterflies j and nbl - j, so one thread that holds both
// butterflies recombines (R2C) or separates (C2R) them in registers: no LDS
// round trip, no further barrier.  Butterflies 0 and nbl/2 are their own
// mirrors; lane 0 takes them both, so nbl butterflies are (nbl + 1) / 2 items.
// The planner gives that stage a radix of at most 10 (11 and 13, for lengths
// that have no other, run in a kernel of their own): the pair's registers set
// the whole kernel's VGPR count.
// ---------------------------------------------------------------------------

// Slot i of an item: the bins (k, L - k) that it pairs.  An ordinary lane pairs
// v[i] with u[R-1-i].  Lane 0 pairs v[i] with v[R-i] in slots 1.., then u[q]
// with u[R-1-q]; slot 0 is bin 0 (with L), and bin L/2, its own mirror, stands
// apart: v[R/2] when R is even, the middle leg of u when it is odd.
template <int RAD>
struct PairSlots {
    static constexpr int U0 = (RAD + 1) / 2;  // first slot of u's pairs in lane 0
    static __device__ __forceinline__ int bin(int i, int j, int nbl)
    {
        if (i < U0) return i * nbl + j;
        return j == 0 ? (i - U0) * nbl + (nbl >> 1) : i * nbl + j;
    }
};

template <typename R>
__device__ __forceinline__ cplx<R> pick(bool first, cplx<R> a, cplx<R> b)
{
    return {first ? a.x : b.x, first ? a.y : b.y};
}

template <typename R, int RAD>
__device__ __forceinline__ void r2c_last_stage(const PassDesc& p, const cplx<R>* line, int t, cplx<R>* dst,
                                               const cplx<R>* src)
{
    using PS = PairSlots<RAD>;
    const int nbl = p.st[p.nst - 1].nbl, L = p.L;
    const bool even = (nbl & 1) == 0;
    const cplx<R>* rtw = reinterpret_cast<const cplx<R>*>(p.rtw);
    const R half = R(0.5);
    const R sc = (p.flags & kScale) ? R(sizeof(R) == 4 ? p.scale_f : p.scale_d) : R(1);
#pragma unroll 1
    for (int j = t; 2 * j < nbl; j += p.TL) {
        cplx<R> v[RAD], u[RAD];
        if (p.nst == 1) {
            if (j != 0) return;  // one butterfly
            load_butterfly<R, RAD, true>(p, src, 0, 0, v);
            Dft<RAD, R>::run(v);
#pragma unroll
            for (int i = 0; i < RAD; i++) u[i] = v[i];
        } else {
            last_from_lds<R, RAD>(p, line, j, v);
            last_from_lds<R, RAD>(p, line, j == 0 ? nbl >> 1 : nbl - j, u);
        }
        const bool z = j == 0;
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int k = PS::bin(i, j, nbl);
            cplx<R> zk = v[i], zm = u[RAD - 1 - i];
            if (i < PS::U0) {
                zm = pick<R>(z, v[(RAD - i) % RAD], zm);
            } else {
                zk = pick<R>(z, u[i - PS::U0], zk);
                zm = pick<R>(z, u[RAD - 1 - (i - PS::U0)], zm);
            }
            const cplx<R> w = rtw[k];
            const R sum_re = zk.x + zm.x, diff_im = zk.y - zm.y;
            const R ra_re = zk.y + zm.y, ra_im = zm.x - zk.x;
            // rot = (0.5 w) * (ra_re + i ra_im)
            const R rot_re = half * (w.x * ra_re - w.y * ra_im);
            const R rot_im = half * (w.x * ra_im + w.y * ra_re);
            const R h_re = half * sum_re, h_im = half * diff_im;
            cplx<R> xk = {h_re + rot_re, h_im + rot_im};
            cplx<R> xm = {h_re - rot_re, rot_im - h_im};
            if (i == 0 && z) {
                xk = {zk.x + zk.y, R(0)};
                xm = {zk.x - zk.y, R(0)};
            }
            if (i < PS::U0 || !z || even) {
                dst[(int64_t)k * p.oes] = cscale(xk, sc);
                dst[(int64_t)(L - k) * p.oes] = cscale(xm, sc);
            }
            // four twiddles in flight at a time (all RAD would cost a wave per SIMD)
            if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
        if (z && (L & 1) == 0) {
            // X_{L/2} = conj(Z_{L/2})
            const cplx<R> h = (RAD & 1) == 0 ? v[RAD / 2] : u[RAD / 2];
            dst[(int64_t)(L >> 1) * p.oes] = cscale(cconj(h), sc);
        }
    }
}

// Z_k = E_k + i O_k,  E_k = X_k + conj(X_{L-k}),
// O_k = (X_k - conj(X_{L-k})) exp(+2 pi i k / 2L), and the mirror Z_{L-k};
// conjugated, so the forward stages compute the inverse transform.
template <typename R>
__device__ __forceinline__ void separate(cplx<R> xk, cplx<R> xm, cplx<R> w, cplx<R>& zk, cplx<R>& zm)
{
    const cplx<R> ek = {xk.x + xm.x, xk.y - xm.y};
    const cplx<R> dk = {xk.x - xm.x, xk.y + xm.y};
    const cplx<R> ok = cmul(dk, cconj(w));
    zk = {ek.x - ok.y, -(ek.y + ok.x)};
    // L-k side: E = conj(ek), O = (X_{L-k} - conj(X_k)) * (-w)
    const cplx<R> dm = {xm.x - xk.x, xm.y + xk.y};
    const cplx<R> om = cmul(dm, cplx<R>{-w.x, -w.y});
    zm = {ek.x - om.y, ek.y - om.x};
}

template <typename R, int RAD>
__device__ __forceinline__ void c2r_first_stage(const PassDesc& p, cplx<R>* line, int t, const cplx<R>* src,
                                                cplx<R>* dst)
{
    using PS = PairSlots<RAD>;
    const int nbl = p.st[0].nbl, L = p.L;
    const bool even = (nbl & 1) == 0;
    const cplx<R>* rtw = reinterpret_cast<const cplx<R>*>(p.rtw);
#pragma unroll 1
    for (int j = t; 2 * j < nbl; j += p.TL) {
        const bool z = j == 0;
        cplx<R> a[RAD], b[RAD], h = {R(0), R(0)};
        // (an odd nbl has no butterfly nbl/2: lane 0 reads in range and drops it)
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            const int k = PS::bin(i, j, nbl);
            a[i] = src[(int64_t)k * p.ies];
            b[i] = src[(int64_t)(L - k) * p.ies];
        }
        if (z && (L & 1) == 0) h = src[(int64_t)(L >> 1) * p.ies];
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            cplx<R> zk, zm;
            separate<R>(a[i], b[i], rtw[PS::bin(i, j, nbl)], zk, zm);
            a[i] = zk;
            b[i] = zm;
            if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
        h = {h.x + h.x, h.y + h.y};  // conj(Z_{L/2}) = 2 X_{L/2}
        // slots back to the legs of butterflies j (v) and nbl - j (u), or 0 and nbl/2
        cplx<R> v[RAD], u[RAD];
#pragma unroll
        for (int i = 0; i < RAD; i++) {
            // v[i] is slot i's k side; lane 0's upper legs are the mirror sides of slots R - i
            v[i] = i < PS::U0 ? a[i] : pick<R>(z, i == RAD - i ? h : b[RAD - i], a[i]);
            // u[r] is slot R-1-r's mirror side; in lane 0 u[q] / u[R-1-q] are slot U0 + q's two sides
            constexpr int NU = RAD - PS::U0;  // pairs of u in lane 0
            const cplx<R> lane0 = i < NU ? a[PS::U0 + (i < NU ? i : 0)]
                                  : RAD - 1 - i < NU ? b[PS::U0 + (RAD - 1 - i < NU ? RAD - 1 - i : 0)]
                                                     : h;
            u[i] = pick<R>(z, lane0, b[RAD - 1 - i]);
        }
        if (p.nst == 1) {
            if (j != 0) return;  // one butterfly
            Dft<RAD, R>::run(v);
            store_butterfly<R, RAD, true, false>(p, v, 0, 1, dst, 0, 0);
            return;
        }
        first_to_lds<R, RAD, false, false>(p, line, j, v);
        __builtin_amdgcn_sched_barrier(0);
        if (!z || even) first_to_lds<R, RAD, false, false>(p, line, z ? nbl >> 1 : nbl - j, u);
    }
}

// The pass descriptor read in place from the kernel-argument segment (the
// kernels take it as their only argument, at offset 0).  A by-value copy
// whose arrays are indexed by the runtime stage number would be materialised
// in per-lane scratch memory.
__device__ __forceinline__ const PassDesc& kernarg_desc()
{
    return *(const PassDesc*)__builtin_amdgcn_kernarg_segment_ptr();  // address-space cast
}

__device__ __forceinline__ uint32_t tile_of_block(const PassDesc& p)
{
    uint32_t tile = blockIdx.x;
    if (p.flags & kXcdRemap) {
        // Workgroups are dispatched round-robin over the 8 XCDs; give each XCD
        // a contiguous run of tiles so column tiles that share cache lines
        // meet in the same L2.
        const uint32_t G = gridDim.x;
        const uint32_t per = G >> 3;
        if (tile < (per << 3)) tile = (tile & 7u) * per + (tile >> 3);
    }
    return tile;
}

// Length-1 lines: the transform is the identity.
template <typename R, bool REAL>
__device__ __forceinline__ void identity_line(const PassDesc& p, const cplx<R>* src, cplx<R>* dst, uint32_t l0,
                                              int64_t gin, int64_t gout)
{
    cplx<R> v[1];
    if constexpr (REAL) {
        // real-packed with L = 1: (x0, x1) <-> bins 0 and 1
        const R* s = reinterpret_cast<const R*>(src);
        R* d = reinterpret_cast<R*>(dst);
        const R sc = (p.flags & kScale) ? R(sizeof(R) == 4 ? p.scale_f : p.scale_d) : R(1);
        if (p.flags & kR2CPost) {
            v[0] = load_pair<R>(s, p.ies);
            dst[0] = {(v[0].x + v[0].y) * sc, R(0)};
            dst[p.oes] = {(v[0].x - v[0].y) * sc, R(0)};
        } else if (p.flags & kC2RPre) {
            const cplx<R> a = src[0], b = src[p.ies];
            cplx<R> zk, zm;
            separate<R>(a, b, cplx<R>{R(1), R(0)}, zk, zm);
            v[0] = zk;
            store_butterfly<R, 1, true, false>(p, v, 0, 1, dst, 0, 0);
        } else if (p.flags & kRealPromote) {
            dst[0] = {s[0] * sc, R(0)};
        } else {
            d[0] = src[0].x * sc;  // kHermIn | kRealPart
        }
    } else {
        v[0] = src[0];
        if (p.flags & kConjIn) v[0].y = -v[0].y;
        store_butterfly<R, 1, false, false>(p, v, 0, 1, dst, l0, gout);
    }
}

// Every middle stage begins with the barrier that ends the stage before it.
template <typename R, int RADSET, bool DIT, bool LATE>
__device__ __forceinline__ void mid_stage_any(const PassDesc& p, cplx<R>* line, int t, int s, bool live,
                                              bool wave_local)
{
    FFTZ_RADIX_SWITCH(p.st[s].radix, RADSET, (mid_stage<R, RAD, DIT, LATE && kLateTw<R, RADSET, RAD>>(p, line, t, s, live, wave_local)))
}

// Forms of the generic pass kernel: complex on both sides; a real side, with
// pair stages of radix <= 10; the same with wider pair stages.
enum RealForm : int { kRealNone = 0, kRealPair = 1, kRealWide = 2 };

// One tile: C lines, threads (c, t) per side's mapping -- row (a wavefront
// walks along a line) or column (it walks the same element of adjacent lines).
// REAL passes carry the real-packed and promoted forms and are row-mapped.
// LATE: wide radices may ask for their twiddles after the DFT (kLateTw).
template <typename R, int RADSET, int REALK, bool NT, bool LATE>
__device__ __forceinline__ void pass_body(const PassDesc& p, const TileIo& io, cplx<R>* lds, int64_t l_base, int tid)
{
    constexpr bool REAL = REALK != kRealNone;
    const bool in_col = !REAL && (p.flags & kInCol) != 0, out_col = !REAL && (p.flags & kOutCol) != 0;
    const int cr = tid >> p.tl_shift, tr = tid & (p.TL - 1);
    const int cc = tid & (p.C - 1), tc = tid >> p.c_shift;
    const int ci = in_col ? cc : cr, ti = in_col ? tc : tr;
    const int co = out_col ? cc : cr, to = out_col ? tc : tr;
    const SlotLine sli = slot_line(p, io, l_base, ci);
    const bool live_in = ci < p.C && sli.live;
    const cplx<R>* src = nullptr;
    cplx<R>* dst = nullptr;
    uint32_t l0 = 0;
    int64_t gin = 0, gout = 0;
    const bool real_in = REAL && (p.flags & (kRealIn | kRealPromote));
    const bool real_out = REAL && (p.flags & (kRealOut | kRealPart));
    bool live_out = live_in;
    if (live_in) {
        const LineIdx li = line_index(p, io, sli.l);
        src = real_in ? reinterpret_cast<const cplx<R>*>(reinterpret_cast<const R*>(io.in) + li.ioff)
                      : reinterpret_cast<const cplx<R>*>(io.in) + li.ioff;
        dst = real_out ? reinterpret_cast<cplx<R>*>(reinterpret_cast<R*>(io.out) + li.ooff)
                       : reinterpret_cast<cplx<R>*>(io.out) + li.ooff;
        l0 = li.l0;
        gin = li.gin;
        gout = li.gout;
    }
    const int S = p.nst;
    if (S <= 1) {
        // the loading thread stores
        if (!live_in || ti != 0) return;
        if (S == 0) {
            identity_line<R, REAL>(p, src, dst, l0, gin, gout);
            return;
        }
        if constexpr (REAL) {
            if (p.flags & kR2CPost) {
                FFTZ_PAIR_SWITCH(p.st[0].radix, RADSET, REALK, (r2c_last_stage<R, RAD>(p, lds, 0, dst, src)))
                return;
            }
            if (p.flags & kC2RPre) {
                FFTZ_PAIR_SWITCH(p.st[0].radix, RADSET, REALK, (c2r_first_stage<R, RAD>(p, lds, 0, src, dst)))
                return;
            }
        }
        FFTZ_RADIX_SWITCH(p.st[0].radix, RADSET, (single_stage<R, RAD, REAL, NT>(p, src, dst, l0, gin, gout)))
        return;
    }
    const bool wave_local = p.TL <= 64 && !in_col && !out_col;
    if (live_in) {
        cplx<R>* line = lds + ci * p.LP;
        bool packed = false;
        if constexpr (REAL) {
            packed = (p.flags & kC2RPre) != 0;
            if (packed) {
                FFTZ_PAIR_SWITCH(p.st[0].radix, RADSET, REALK, (c2r_first_stage<R, RAD>(p, line, ti, src, dst)))
            }
        }
        if (!packed) {
            FFTZ_RADIX_SWITCH(p.st[0].radix, RADSET, (first_stage<R, RAD, REAL, LATE && kLateTw<R, RADSET, RAD>>(p, line, ti, src, gin)))
        }
    }
    for (int s = 1; s + 1 < S; s++)
        mid_stage_any<R, RADSET, false, LATE>(p, lds + cr * p.LP, tr, s, cr < p.C, wave_local);
    stage_sync(wave_local);
    if (in_col != out_col) {
        const SlotLine slo = slot_line(p, io, l_base, co);
        live_out = co < p.C && slo.live;
        if (live_out) {
            const LineIdx li = line_index(p, io, slo.l);
            dst = reinterpret_cast<cplx<R>*>(io.out) + li.ooff;
            l0 = li.l0;
            gout = li.gout;
        }
    }
    if (!live_out) return;
    const cplx<R>* line = lds + co * p.LP;
    if constexpr (REAL) {
        if (p.flags & kR2CPost) {
            FFTZ_PAIR_SWITCH(p.st[S - 1].radix, RADSET, REALK, (r2c_last_stage<R, RAD>(p, line, to, dst, src)))
            return;
        }
    }
    FFTZ_RADIX_SWITCH(p.st[S - 1].radix, RADSET, (last_stage<R, RAD, REAL, NT>(p, line, to, dst, l0, gout)))
}

template <typename R, int RADSET, int REALK, bool NT, int MAXT>
__global__ void __launch_bounds__(MAXT)
    __attribute__((amdgpu_waves_per_eu(REALK == kRealNone ? (sizeof(R) == 8 && (RADSET == kRadLight || RADSET == kRadAll) ? 3 : 1) : REALK == kRealWide ? 1 : sizeof(R) == 4 ? 4 : RADSET == kRadTo8 ? 3 : 2))) k_fft_pass(const PassDesc p_arg)
{
    (void)p_arg;
    const PassDesc& p = kernarg_desc();
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    cplx<R>* lds = reinterpret_cast<cplx<R>*>(smem_raw);
    const int64_t l_base = (int64_t)tile_of_block(p) * p.C;
    pass_body<R, RADSET, REALK, NT, REALK == kRealNone>(p, io_of(p), lds, l_base, threadIdx.x);
}

// ---------------------------------------------------------------------------
// Bluestein (chirp-z) for one or more lines of prime length n, fused into a
// single pass over an M-point LDS tile (M = smooth length >= 2n-1, the
// reference's get_extended_length, core/common/bluestein_utils.c:39-70):
//   a = x * conj(B) zero-padded to M     (load)
//   A = FFT_M(a)                         (stages 0 .. S-1)
//   Z = conj(A) * conj(FFT_M(B)) / M      (in registers)
//   W = FFT_M(Z) = conj(IFFT_M(A * FFT_M(B)) / M)   (stages S-1 .. 0)
//   X = conj(B * W)                       (store)
// which is core/solvers/complex/bluestein_solver_dft.c:137-234 with its five
// sweeps (pre_mul, memset, FFT, mul, IFFT, post_mul) in one HBM round trip.
// The first transform leaves its digits in output order and the second runs
// the stages backwards, so nothing is reordered between them and the last
// stage of the first, the product and the first stage of the second share one
// butterfly's registers: 2 S - 2 LDS exchanges for the two transforms.
// ---------------------------------------------------------------------------
template <typename R, int RAD>
__device__ __forceinline__ void bs_first(const PassDesc& p, cplx<R>* line, int t, const cplx<R>* src)
{
    const int nbl = p.st[0].nbl;
    const int n = p.nvalid_in;
    const cplx<R>* chirp = reinterpret_cast<const cplx<R>*>(p.chirp);
    const bool cj = (p.flags & kConjIn) != 0;
#pragma unroll 1
    for (int j = t; j < nbl; j += p.TL) {
        cplx<R> v[RAD];
        if (p.flags & (kRealPromote | kHermIn)) {
#pragma unroll
            for (int i = 0; i < RAD; i++) {
                const int e = i * nbl + j;
                v[i] = {R(0), R(0)};
                if (e < n) {
                    if (p.flags & kRealPromote) {
                        v[i] = {reinterpret_cast<const R*>(src)[(int64_t)e * p.ies], R(0)};
                    } else {
                        const bool up = 2 * e > n;
                        v[i] = src[(int64_t)(up ? n - e : e) * p.ies];
                        if (up) v[i].y = -v[i].y;
                    }
                    if (cj) v[i].y = -v[i].y;
                    v[i] = cmul(v[i], chirp[e]);
                }
            }
        } else {
            // at most (R + 1) / 2 legs hold data (n <= (M + 1) / 2)
            constexpr int H = (RAD + 1) / 2;
            const cplx<R>* q = src + (int64_t)j * p.ies;
            const int64_t step = (int64_t)nbl * p.ies;
#pragma unroll
            for (int i = 0; i < RAD; i++) v[i] = {R(0), R(0)};
#pragma unroll
            for (int i = 0; i < H; i++) {
                const int e = i * nbl + j;
                if (e < n) {
                    v[i] = q[i * step];
                    if (cj) v[i].y = -v[i].y;
                    v[i] = cmul(v[i], chirp[e]);
                }
            }
        }
        first_to_lds<R, RAD, false, false>(p, line, j, v);
    }
}

template <typename R, int RAD>
__device__ __forceinline__ void bs_center(const PassDesc& p, cplx<R>* line, int t, bool live, bool wave_local)
{
    const int full = p.st[p.nst - 1].nbl, nbl = live ? full : 0;
    const cplx<R>* spec = reinterpret_cast<const cplx<R>*>(p.spec);
    int j = t, base = 0;
    cplx<R> w[RAD];
    auto fetch = [&]() {
        if (j < nbl) {
            base = last_base(p, j);
#pragma unroll
            for (int i = 0; i < RAD; i++) w[i] = spec[(uint32_t)(i * full + j)];
        }
    };
    fetch();
    stage_sync(wave_local);
#pragma unroll 1
    while (j < nbl) {
        cplx<R>* q = line + base;
        cplx<R> v[RAD];
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = q[i];
        Dft<RAD, R>::run(v);
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = cmul(cconj(v[i]), w[i]);
        Dft<RAD, R>::run(v);
#pragma unroll
        for (int i = 0; i < RAD; i++) q[i] = v[i];
        j += p.TL;
        fetch();
    }
}

template <typename R, int RAD, bool NT>
__device__ __forceinline__ void bs_final(const PassDesc& p, const cplx<R>* line, int t, cplx<R>* dst, bool live,
                                         bool wave_local)
{
    const int full = p.st[0].nbl, nbl = live ? full : 0, step = p.st[0].lst;
    const int n = p.nvalid_out;
    const cplx<R>* chirp = reinterpret_cast<const cplx<R>*>(p.chirp);
    const cplx<R>* tw = stage_tw<R>(p, 0);
    const bool fwd = !(p.flags & kConjOut);
    const bool part = (p.flags & kRealPart) != 0;
    constexpr int H = (RAD + 1) / 2;  // outputs beyond n <= (M + 1) / 2 are not wanted
    int j = t;
    cplx<R> w[RAD - 1];
    if (j < nbl) load_twiddles<R, RAD>(tw, (uint32_t)j, full, w);
    stage_sync(wave_local);
#pragma unroll 1
    while (j < nbl) {
        cplx<R> v[RAD];
#pragma unroll
        for (int i = 0; i < RAD; i++) v[i] = line[j + i * step];
        apply_twiddles<R, RAD>(v, w);
        Dft<RAD, R>::run(v);
#pragma unroll
        for (int i = 0; i < H; i++) {
            const int e = i * full + j;
            if (e < n) {
                v[i] = cmul(cconj(chirp[e]), v[i]);  // B * W
                if (fwd) v[i].y = -v[i].y;            // forward result is conj(B W)
            }
        }
        if (part) {
            R* d = reinterpret_cast<R*>(dst);
#pragma unroll
            for (int i = 0; i < H; i++)
                if (i * full + j < n) d[(int64_t)(i * full + j) * p.oes] = v[i].x;
        } else {
#pragma unroll
            for (int i = 0; i < H; i++)
                if (i * full + j < n) put<R, NT>(dst + (int64_t)(i * full + j) * p.oes, v[i]);
        }
        j += p.TL;
        if (j < nbl) load_twiddles<R, RAD>(tw, (uint32_t)j, full, w);
    }
}

template <typename R, int RADSET, bool NT>
__device__ __forceinline__ void bluestein_body(const PassDesc& p, const TileIo& io, cplx<R>* lds, int64_t l_base, int tid)
{
    const int c = tid >> p.tl_shift;
    const int t = tid & (p.TL - 1);
    const SlotLine sl = slot_line(p, io, l_base, c);
    const bool live = c < p.C && sl.live;
    const cplx<R>* src = nullptr;
    cplx<R>* dst = nullptr;
    if (live) {
        LineIdx li = line_index(p, io, sl.l);
        // real-side lines are offset in real elements (and then only read /
        // written through real pointers)
        src = (p.flags & kRealPromote)
                  ? reinterpret_cast<const cplx<R>*>(reinterpret_cast<const R*>(io.in) + li.ioff)
                  : reinterpret_cast<const cplx<R>*>(io.in) + li.ioff;
        dst = (p.flags & kRealPart) ? reinterpret_cast<cplx<R>*>(reinterpret_cast<R*>(io.out) + li.ooff)
                                    : reinterpret_cast<cplx<R>*>(io.out) + li.ooff;
    }
    const int S = p.nst;
    const bool wave_local = p.TL <= 64;
    cplx<R>* line = lds + c * p.LP;
    if (live) {
        FFTZ_RADIX_SWITCH(p.st[0].radix, RADSET, (bs_first<R, RAD>(p, line, t, src)))
    }
    for (int s = 1; s + 1 < S; s++) mid_stage_any<R, RADSET, false, false>(p, line, t, s, live, wave_local);
    FFTZ_RADIX_SWITCH(p.st[S - 1].radix, RADSET, (bs_center<R, RAD>(p, line, t, live, wave_local)))
    for (int s = S - 2; s >= 1; s--) mid_stage_any<R, RADSET, true, false>(p, line, t, s, live, wave_local);
    FFTZ_RADIX_SWITCH(p.st[0].radix, RADSET, (bs_final<R, RAD, NT>(p, line, t, dst, live, wave_local)))
}

template <typename R, int RADSET, bool NT, int MAXT>
__global__ void __launch_bounds__(MAXT) k_bluestein(const PassDesc p_arg)
{
    (void)p_arg;
    const PassDesc& p = kernarg_desc();
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    cplx<R>* lds = reinterpret_cast<cplx<R>*>(smem_raw);
    bluestein_body<R, RADSET, NT>(p, io_of(p), lds, (int64_t)blockIdx.x * p.C, threadIdx.x);
}

// ---------------------------------------------------------------------------
// Uneven batches in one persistent launch.  A device work queue lists tiles
// (size class, first line, line count, offsets); each workgroup takes the
// next tile from an atomic counter, reads the size class's pass descriptor in
// place, and runs the same pass or Bluestein body as the single-size kernels.
// Tiles are sorted by cost on the host, largest first.  The arithmetic of a
// tile does not depend on the workgroup that runs it, so results are bitwise
// identical run to run.
// ---------------------------------------------------------------------------
template <typename R, int MAXT, bool NT>
__global__ void __launch_bounds__(MAXT) k_batch(const BatchArgs a)
{
    // dynamic LDS: [tile index | tile data].  The tile index is made uniform
    // with readfirstlane, and the queue entry and its size class's descriptor
    // are read in place from the plan tables through the constant address
    // space (read-only for the whole launch), i.e. with scalar loads.
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    int& s_tile = *reinterpret_cast<int*>(smem_raw);
    cplx<R>* lds = reinterpret_cast<cplx<R>*>(smem_raw + kBatchHdrBytes);
    const int tid = threadIdx.x;
    const int esz = 2 * (int)sizeof(R);
    if (tid == 0) s_tile = (int)atomicAdd(a.counter, 1u);
    __syncthreads();
    for (;;) {
        const int t = __builtin_amdgcn_readfirstlane(s_tile);
        if (t >= a.ntiles) break;
        // the next tile's index is fetched now and published at the end, so
        // the atomic's round trip overlaps this tile's work
        int nxt = 0;
        if (tid == 0) nxt = (int)atomicAdd(a.counter, 1u);
        const BatchTile& bt = *(const BatchTile*)((const __attribute__((address_space(4))) BatchTile*)a.tiles + t);
        const PassDesc& p = *(const PassDesc*)((const __attribute__((address_space(4))) PassDesc*)a.descs + bt.desc);
        const TileIo io{reinterpret_cast<const char*>(a.in) + bt.in_off * esz,
                        reinterpret_cast<char*>(a.out) + bt.out_off * esz, (int64_t)bt.nlines, bt.dist, bt.dist};
        const bool blue = bt.bluestein != 0;
        const int C = p.C;
        // a queue entry covers one or more rounds of C lines
        for (int64_t lb = 0; lb < io.nlines; lb += C) {
            if (blue)
                bluestein_body<R, kRadAll, NT>(p, io, lds, lb, tid);
            else
                pass_body<R, kRadAll, kRealNone, NT, false>(p, io, lds, lb, tid);
            __syncthreads();
        }
        if (tid == 0) s_tile = nxt;
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Launch table: precision x radix set x block limit.  The larger block is
// 1024 threads in complex64 and 512 in complex128, half of that for real passes:
// they hold a butterfly and its mirror.
// ---------------------------------------------------------------------------
template <typename R>
constexpr int kBigBlock = sizeof(R) == 4 ? 1024 : 512;

template <typename R, int A, int T>
inline const void* sym(KernelKind kind, bool nt)
{
    constexpr int TR = T > kBigBlock<R> / 2 ? kBigBlock<R> / 2 : T;
    switch (kind) {
        case KernelKind::Pass:
            return nt ? (const void*)&k_fft_pass<R, A, kRealNone, true, T>
                      : (const void*)&k_fft_pass<R, A, kRealNone, false, T>;
        case KernelKind::Real:
            if constexpr (A != kRadLight) return (const void*)&k_fft_pass<R, A, kRealPair, false, TR>;
            return nullptr;
        case KernelKind::RealWide:
            if constexpr (A == kRadAll) return (const void*)&k_fft_pass<R, A, kRealWide, false, TR>;
            return nullptr;
        default: return nt ? (const void*)&k_bluestein<R, A, true, T> : (const void*)&k_bluestein<R, A, false, T>;
    }
}

template <typename R, int A>
inline const void* sym_t(KernelKind kind, bool nt, int maxt)
{
    return maxt <= 256 ? sym<R, A, 256>(kind, nt) : sym<R, A, kBigBlock<R>>(kind, nt);
}

}  // namespace fftz
