// mpcf_kernels.hip -- CDNA4 kernels of one LSRK3 stage and the dt reduction.
//
// Built four times (see build.py):
//   MPCF_FAST=0, -ffp-contract=off  -> namespace mpcf::parity  (bit-exact scheme)
//   MPCF_FAST=1, -ffp-contract=on   -> namespace mpcf::fast
//   MPCF_FAST=1, MPCF_P64=1         -> namespace mpcf::fastp   (fast + binary64
//                                      pressure recovery and speed-of-sound reduction)
//   MPCF_F64=1,  -ffp-contract=off  -> namespace mpcf::f64     (the scheme in binary64:
//                                      storage, arithmetic and reductions)
//
// One RK stage (GPUlab::process_all, source/GPUlab.cpp:703-793) is
//   ghost fill -> x sweep -> y sweep -> z sweep (+ register update)
// Each sweep marches its direction with a rolling five-cell primitive window
// in registers: every cell is converted to primitives once, reconstructed
// once (both face states), and every face is solved once.  The x sweep
// stages x-runs of 64 pencils through LDS so its loads stay contiguous; the
// y and z sweeps put the 64 lanes of a wave along x and march a strided axis.
// Accumulators carry the partial flux sums between sweeps in the reference's
// summation order (((((fxp-fxm)+fyp)-fym)+fzp)-fzm) (GPUkernels.cu:1111).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "mpcf_scheme.h"
#include "mpcf_launch.h"

#ifndef MPCF_FAST
#define MPCF_FAST 0
#endif
#ifndef MPCF_P64
#define MPCF_P64 0
#endif
#ifndef MPCF_F64
#define MPCF_F64 0
#endif
#ifndef MPCF_EPAIR
#define MPCF_EPAIR 0
#endif

#if MPCF_F64
#define MPCF_NS f64
#elif MPCF_EPAIR
#define MPCF_NS fastpe
#elif MPCF_P64
#define MPCF_NS fastp
#elif MPCF_FAST
#define MPCF_NS fast
#else
#define MPCF_NS parity
#endif

namespace mpcf {
namespace MPCF_NS {

#if MPCF_F64
typedef double Real;
#else
typedef float Real;
#endif
typedef PrimT<Real> Prim;
constexpr bool kP64 = MPCF_P64 != 0;
// E stored as a binary32 pair: the solution buffers hold an eighth field,
// the low part of E (E = E[hi] + E[lo], exact in binary64), read wherever E
// is read and written wherever E is written
constexpr bool kEPair = MPCF_EPAIR != 0;
constexpr int NU = 7 + (kEPair ? 1 : 0);   // fields of a solution buffer
constexpr int FELO = 7;                   // the low part of E
// the speed-of-sound reduction and dt/h run in binary64
constexpr bool kSosD = MPCF_P64 != 0 || MPCF_F64 != 0 || MPCF_EPAIR != 0;
// scalar type of the speed-of-sound reduction
typedef std::conditional<kSosD, double, float>::type SosT;

// c + max(|rho u|, |rho v|, |rho w|) / rho of one cell (GPUkernels.cu:1206-1212,
// or MaxSpeedOfSound.cpp:43-47 with 0.5/rho in binary64 for CPU_FORM).  bad:
// the cell fails one of the reference's assertions (rho > 0, E > 0, G > 0,
// c > 0, no NaN: GPUkernels.cu:1171-1173, MaxSpeedOfSound.cpp:31-48) or its
// speed is infinite.  The update's P >= 0 (GPUkernels.cu:1174) is left out:
// rounding leaves P a few ulp of the neighbouring water's P below zero in air
// cells next to a sharp interface in one arithmetic and at +0 in another, and
// a P negative enough to matter drives c^2 <= 0, which is flagged.  Every comparison is false for a NaN, and a NaN
// in any field reaches p and c, so a NaN cell is always flagged -- the maximum
// itself drops NaN operands (fmax) and would not show it.
// QUICK (binary32, GPU form): the quotients and the root by div_rn and sqrt_rn,
// which round like the IEEE operations; `odd` is set where an operand is
// outside [2^-40, 2^40] (all but the momentum's quotient, which a momentum too
// small for div_rn leaves without effect on the sum), and sos_cell then
// evaluates the cell again without QUICK.  29 instructions instead of 72.
template <bool QUICK>
__device__ __forceinline__ SosT sos_cell_as(const bool cpu_form, const SosT r, const SosT mu, const SosT mv,
                                            const SosT mw, const SosT E, const SosT G, const SosT P, bool& bad, bool* odd)
{
    SosT c, s;
    const SosT mm = mmax(mmax(fabs(mu), fabs(mv)), fabs(mw));
    if constexpr (QUICK) {
        const SosT ir = rcp_rn(r), iG = rcp_rn(G);
        const SosT p = div_rn(E - (mu*mu + mv*mv + mw*mw)*div_rn(SosT(0.5f), r, ir) - P, G, iG);
        const SosT x = div_rn(p + P, G, iG) + p;
        const SosT c2 = div_rn(x, r, ir);
        c = sqrt_rn(c2);
        s = c + div_rn(mm, r, ir);
        const SosT lo = mmin3(mmin3(r, G, p + P), mmin3(x, c2, fabs(p)), fabs(p));
        const SosT hi = mmax3(mmax3(r, G, p + P), mmax3(x, c2, fabs(p)), mm);
        *odd = !(lo >= SosT(0x1p-40f) && hi <= SosT(0x1p40f));
    } else {
        SosT p;
        if (cpu_form) p = (SosT)((E - (mu*mu + mv*mv + mw*mw)*(0.5/r) - P)/G);
        else          p = (E - (mu*mu + mv*mv + mw*mw)*(SosT(0.5f)/r) - P) / G;
        c = msqrt(((p + P) / G + p) / r);
        s = c + mm / r;
    }
    const SosT huge = kSosD ? SosT(__DBL_MAX__) : SosT(__FLT_MAX__);
    bad = !(r > SosT(0) && E > SosT(0) && G > SosT(0) && c > SosT(0) && s <= huge);
    return s;
}

__device__ __forceinline__ SosT sos_cell(const bool cpu_form, const SosT r, const SosT mu, const SosT mv,
                                         const SosT mw, const SosT E, const SosT G, const SosT P, bool& bad)
{
    if constexpr (!kSosD) {
        bool odd = cpu_form;
        if (!cpu_form) {
            const SosT s = sos_cell_as<true>(false, r, mu, mv, mw, E, G, P, bad, &odd);
            if (__builtin_expect(!any_lane(odd), 1)) return s;
        }
    }
    return sos_cell_as<false>(cpu_form, r, mu, mv, mw, E, G, P, bad, nullptr);
}

// a maximum speed of sound and its flag as a reduction or a step's last stage
// left them
struct SosIn { SosT sos; unsigned bad; };

// the maximum and flag folded into the previous step's last stage.  Relaxed
// loads at device scope, which go past the caches: the values come from other
// XCDs' atomics in earlier kernels
__device__ __forceinline__ SosIn take_folded(const StepState* st)
{
    SosIn in;
    if constexpr (kSosD)
        in.sos = __longlong_as_double((long long)__hip_atomic_load(&st->next_sos_bits_d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    else
        in.sos = __uint_as_float(__hip_atomic_load(&st->next_sos_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    in.bad = __hip_atomic_load(&st->next_bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return in;
}

struct DtArgs
{
    int with_dt;                  // 0: only the maximum (mpcf_max_sos)
    double cfl, h, dt_max;
};

__device__ __forceinline__ void sos_finalize(StepState* st, const DtArgs& d, const SosIn& in)
{
    const double sos = in.sos;
    st->sos_d = sos;
    st->sos = (float)sos;
    st->sos_is_d = kSosD ? 1 : 0;
    st->bad = in.bad;
    // the folded maximum (and flag) of the next step starts from zero
    __hip_atomic_store(&st->next_sos_bits, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&st->next_sos_bits_d, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&st->next_bad, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d.with_dt) {
        // binary64 dt from the binary32 (or binary64) maximum
        double dt = d.cfl*d.h/sos;
        dt = d.dt_max < dt ? d.dt_max : dt;
        st->dt = dt;
        st->h = d.h; st->cfl = d.cfl; st->dt_max = d.dt_max;
        st->dtinvh = (float)(dt/d.h);
        st->dtinvh_d = dt/d.h;
    }
}

typedef FaceFluxT<Real> FaceFlux;
typedef CellRecT<Real> CellRec;
typedef RecT<Real> Rec;
constexpr bool kFast = MPCF_FAST != 0;
// FAST builds fold the x and y parts of a stage into R as soon as they are
// known, R <- a R - dtinvh (x+y flux differences), and keep only the three
// G/P accumulators (sum G, sum P, div u) for the z sweep, which then finishes
// R <- R - dtinvh (z flux differences - div u sum G / 6 ...).  The same
// algebra as the reference's single update, rounded in two parts; it moves
// the R read from the bandwidth-bound z sweep to the x+y sweep, which has
// bandwidth to spare, and drops 7 accumulator fields from the z sweep's
// reads.  The bit-exact builds keep the reference's single update.
constexpr bool kFold = kFast;
// In a stage with a = 0 (the first stage of a step) the folded x+y part is
// stored unscaled, R' = a R - (x+y flux differences), and the z sweep scales
// it: R = dtinvh * R' - dtinvh (z part).  dtinvh * (-t) rounds to exactly
// -(dtinvh * t), so the results are bit for bit those of scaling in the x+y
// sweep -- but the x+y sweep of a step's first stage no longer needs dt, and
// can run while the previous step's last z sweeps (which fold the maximum
// speed of sound dt is taken from) are still in flight.
__device__ __forceinline__ bool unscaled_stage(const Real a) { return kFold && a == Real(0.0f); }
// accelerator complex dies of an MI355X; workgroups are dispatched to them in
// turn by linear workgroup id
constexpr int kXCDs = 8;
// the fused x+y march unrolled by five in the binary32 FAST builds (in the
// bit-exact and binary64 builds the unrolled march spills)
constexpr bool kUnrollXY = kFast && !MPCF_F64;
// the waves of a workgroup of the binary32 x+y sweeps keep phase (keep_phase)
// (single-case and batched flat launches: FAST 512^3 step 19.45 -> 18.61 ms, a
// 24-case ensemble 1.76 -> 1.72 ms, bit-exact 256^3 6.58 -> 6.45 ms; the
// persistent launches' item loop has barriers of its own that a wave without
// work reaches early, and does not).  The z sweep gains 0.5 % at most and is
// left alone; a wave that evaluates a window or face again without QUICK does
// so between two barriers
constexpr bool kSyncXY = !MPCF_F64;
// likewise the y / z marches (a separate switch: their register budget differs)
constexpr bool kUnrollMarch = kFast && !MPCF_F64;

// MODE_STAGE_NOR: a stage whose R is not stored -- the last stage of a step
// that another step of the same mpcf_steps call follows (that step's first
// stage multiplies R by a = 0), 28 B/cell less for the bandwidth-bound z sweep
enum { MODE_FIRST = 0, MODE_ACC = 1, MODE_CONV = 2, MODE_STAGE = 3, MODE_STAGE_NOR = 4 };
constexpr bool is_stage(const int mode) { return mode == MODE_STAGE || mode == MODE_STAGE_NOR; }

struct StageArgs
{
    const Real* __restrict__ u;    // input solution (7 fields, ghosts filled)
    Real* __restrict__ R;          // RK register (7 fields), updated in place
    Real* __restrict__ acc;        // sweep accumulators (10 fields)
    Real* __restrict__ uo;         // output solution (MODE_STAGE)
    int64_t fs;                    // field stride (elements)
    Real a, b, dtinvh;
    const StepState* st;           // if non-null, dtinvh is read from st->dtinvh
    StepState* sos_next;           // non-null: fold the max speed of sound of the written u into
                                   // sos_next->next_sos_bits[_d] (last stage of a step)
    int sos_cpu;                   // its form: MaxSpeedOfSound_CPP (1) or the GPU kernel's (0)
    int z0, z1;                    // the z range of interior cells this launch covers: the planes
                                   // of the x, y and x+y sweeps, the marched rows of the z sweep
                                   // (a slab of a pipelined step; 0, nz otherwise)
    int bcmask;                    // bit f: face f reflecting; bit 8+f: face f a halo
                                   // face (ghost band imported); else absorbing
};

// Boundary conditions at load time (BoundaryConditions.h:60-109).  A stencil
// read at index i outside [0, n) along an axis is served by the cell its
// ghost would copy: absorbing -- the boundary cell; reflecting -- the mirror
// cell (-1-i on the low face, 2n-1-i on the high face) with the axis' normal
// momentum negated (sg = -1).  The values are the ghost values bit for bit,
// so no kernel fills or reads a ghost band -- except on a halo face, whose
// ghost band holds a neighbouring block's cells (imported by k_halo) and is
// read as it is.
__device__ __forceinline__ int bc_index(const int i, const int n, const int bcmask, const int face_lo, Real& sg)
{
    sg = Real(1.0f);
    if (i < 0) {
        if ((bcmask >> (8 + face_lo)) & 1) return i;
        if ((bcmask >> face_lo) & 1) { sg = Real(-1.0f); return -1 - i; }
        return 0;
    }
    if (i >= n) {
        if ((bcmask >> (9 + face_lo)) & 1) return i;
        if ((bcmask >> (face_lo + 1)) & 1) { sg = Real(-1.0f); return 2 * n - 1 - i; }
        return n - 1;
    }
    return i;
}

// A lane's element index split into a part that is the same for every lane of
// the wave (base, a scalar: the element of a row the march starts from) and
// the lane's byte offset from it (lo, small and non-negative).
// An access is a global load or store of a scalar base and a 32-bit vector
// offset, `ld_lane(p, off)`: the sweeps keep one scalar base per field for the
// whole march and add the row's bytes to the lane's offset, one vector add
// that all fields of the row share.  Buffer resources rebuilt per access took
// 165 scalar instructions a row in the x+y sweep (30 now), 64-bit flat
// addresses 29 64-bit vector adds a row in the z sweep (none now; its E-pair
// instance fits two waves per SIMD again).  100 steps of 128^3 with transfers
// 44.2 -> 43.6 ms, 30 steps of 512^3 661 -> 656 ms.
struct LaneIdx { int64_t base; uint32_t lo; };

// e: the lane's element; floor_e: an element no greater than the element of
// any active lane of the wave (the first active lane's value is taken);
// shift: wave-uniform elements from there to the row the march starts from
__device__ __forceinline__ LaneIdx lane_idx(const int e, const int floor_e, const int64_t shift)
{
    const int b = __builtin_amdgcn_readfirstlane(floor_e);
    return LaneIdx{b + shift, (uint32_t)(e - b) * (uint32_t)sizeof(Real)};
}

// wave-uniform pointers of the first N fields at p, fs elements apart, each in
// a scalar register pair of its own: hidden from the optimizer, which would
// otherwise add the lane offset once and then every field's distance with a
// 64-bit vector add
#define MPCF_GLOBAL __attribute__((address_space(1)))
template <int N, typename V> struct Bases
{
    V MPCF_GLOBAL* p[N];
    __device__ __forceinline__ Bases(V* const p0, const int64_t fs)
    {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            // uniform by construction; a pointer read from a table in memory may
            // sit in a vector register
            const uint64_t a = (uint64_t)(p0 + q * fs);
            const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
            const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
            uint64_t b = ((uint64_t)hi << 32) | lo;
            asm("" : "+s"(b));
            p[q] = (V MPCF_GLOBAL*)b;
        }
    }
};

// the element `off` bytes after the wave-uniform pointer p
template <typename V>
__device__ __forceinline__ V ld_lane(const V MPCF_GLOBAL* p, const uint32_t off)
{
    return *(const V MPCF_GLOBAL*)((const char MPCF_GLOBAL*)p + off);
}

// store; STREAM: non-temporal, for data that no kernel reads again soon --
// the solution and register written by the z sweep (read by the next stage, a
// whole block later) and the G/P accumulators of the x+y sweep (read once by
// the z sweep of the slab).  The hint keeps these streams from displacing
// lines in the caches; at 512^3 it takes the pipelined step from 20.66 to
// 20.0 ms.
template <bool STREAM = false, typename V>
__device__ __forceinline__ void st_lane(V MPCF_GLOBAL* p, uint32_t off, const V v)
{
    // the address is formed here, not shared with a load of the same element:
    // across a branch it would be kept as a 64-bit vector sum
    asm("" : "+v"(off));
    V MPCF_GLOBAL* const q = (V MPCF_GLOBAL*)((char MPCF_GLOBAL*)p + off);
    if (STREAM) __builtin_nontemporal_store(v, q);
    else        *q = v;
}

// raw conserved values of the cell at index `row` of a marched column, boundary-
// mapped: U.p[q] + the lane's byte offset lo is field q's element of row r0, s
// the element stride of the axis.  Returns the sign the axis' normal momentum
// takes; the caller applies it where the values are consumed, so that a
// prefetch is not waited on when it is issued.
__device__ __forceinline__ Real load_row(const StageArgs& A, const Bases<NU, const Real>& U, const uint32_t lo, const int r0,
                                         const int row, const int n, const int s, const int face_lo, Real* out)
{
    Real sg;
    const int r = bc_index(row, n, A.bcmask, face_lo, sg) - r0;
    const uint32_t off = lo + (uint32_t)(r * s) * (uint32_t)sizeof(Real);
#pragma unroll
    for (int q = 0; q < NU; ++q) out[q] = ld_lane(U.p[q], off);
    return sg;
}
// the same for the z axis, whose rows may lie further apart than 32-bit offsets
// reach (the planes of the largest blocks): u0 + lo is field 0's element of
// row r0, and the row's distance goes into the scalar pointers
__device__ __forceinline__ Real load_row_far(const StageArgs& A, const Real* u0, const uint32_t lo, const int r0,
                                             const int row, const int n, const int s, const int face_lo, Real* out)
{
    Real sg;
    const int r = bc_index(row, n, A.bcmask, face_lo, sg) - r0;
    const Bases<NU, const Real> U(u0 + (int64_t)r * s, A.fs);
    uint32_t off = lo;
    asm volatile("" : "+v"(off));   // kept 32-bit: widened once before the loop it would be a vector add per field
#pragma unroll
    for (int q = 0; q < NU; ++q) out[q] = ld_lane(U.p[q], off);
    return sg;
}

// primitives of a loaded row of NU conserved values
__device__ __forceinline__ Prim prim_of(const Real* w)
{
    return to_prim<Real, kFast, kP64, kEPair>(w[0], w[1], w[2], w[3], w[4], w[5], w[6], kEPair ? w[FELO] : Real(0));
}

// operands of one cell's accumulator update, loaded one step ahead
template <int MODE>
struct EmitIn
{
    Real acc[NACC];
    Real R[NVAR];
    Real u[NU];
};

// fields of a y / z sweep at the march's first row, as wave-uniform pointers
template <int MODE>
struct EmitPtr
{
    static constexpr bool kR = MODE == MODE_CONV || is_stage(MODE) || (kFold && MODE == MODE_ACC);
    static constexpr bool kAll = MODE == MODE_FIRST || MODE == MODE_ACC || !kFold;   // all accumulators
    Bases<kAll ? A_SUMG : 1, Real> acc;
    Bases<3, Real> gp;                     // the G/P accumulators
    Bases<kR ? NVAR : 1, Real> R;
    Bases<is_stage(MODE) ? NU : 1, Real> uo;
    __device__ __forceinline__ EmitPtr(const StageArgs& A, const int64_t base)
        : acc(A.acc + base, A.fs), gp(A.acc + base + A_SUMG * A.fs, A.fs), R(A.R + base, A.fs), uo(A.uo + base, A.fs) {}
};

template <int MODE>
__device__ __forceinline__ void emit_load(const EmitPtr<MODE>& E, const uint32_t off, EmitIn<MODE>& in)
{
    if constexpr (MODE != MODE_FIRST) {
        if constexpr (EmitPtr<MODE>::kAll) {
#pragma unroll
            for (int q = 0; q < NVAR; ++q) in.acc[q] = ld_lane(E.acc.p[q], off);
        }
        // folded: only the G/P accumulators remain
#pragma unroll
        for (int q = 0; q < 3; ++q) in.acc[A_SUMG + q] = ld_lane(E.gp.p[q], off);
        if constexpr (EmitPtr<MODE>::kR) {
#pragma unroll
            for (int q = 0; q < NVAR; ++q) in.R[q] = ld_lane(E.R.p[q], off);
        }
    }
}

// write the contribution of one cell, at byte offset `off` from the first
// row of each field.  F = flux at the cell's right face, Fl = flux at its left
// face; cG/cP = plus-state + minus-state of G/P.
template <int MODE>
__device__ __forceinline__ void emit(const StageArgs& A, const EmitPtr<MODE>& E, const Real dtinvh, const uint32_t off,
                                     const EmitIn<MODE>& in,
                                     const FaceFlux& F, const FaceFlux& Fl, const Real cG, const Real cP,
                                     SosT& smax, bool& bad)
{
    if constexpr (MODE == MODE_FIRST) {
        // _xflux + _xextraterm_hllc ("=" assignment, GPUkernels.cu:57-59)
#pragma unroll
        for (int q = 0; q < NVAR; ++q) st_lane(E.acc.p[q], off, F.f[q] - Fl.f[q]);
        st_lane(E.gp.p[0], off, cG);
        st_lane(E.gp.p[1], off, cP);
        st_lane(E.gp.p[2], off, F.vel - Fl.vel);
    } else if constexpr (MODE == MODE_ACC) {
        // _yextraterm_hllc ("+=", GPUkernels.cu:439-441)
#pragma unroll
        for (int q = 0; q < NVAR; ++q) {
            const Real t = (in.acc[q] + F.f[q]) - Fl.f[q];
            if constexpr (kFold) st_lane(E.R.p[q], off, unscaled_stage(A.a) ? A.a*in.R[q] - t : A.a*in.R[q] - dtinvh*t);
            else       st_lane(E.acc.p[q], off, t);
        }
        st_lane(E.gp.p[0], off, in.acc[A_SUMG] + cG);
        st_lane(E.gp.p[1], off, in.acc[A_SUMP] + cP);
        st_lane(E.gp.p[2], off, in.acc[A_DIVU] + (F.vel - Fl.vel));
    } else {
        // _zextraterm_hllc + _divergence (+ _update), GPUkernels.cu:812-814,1104-1136,1164-1170
        const Real sG = in.acc[A_SUMG] + cG;
        const Real sP = in.acc[A_SUMP] + cP;
        const Real dU = in.acc[A_DIVU] + (F.vel - Fl.vel);
        const Real factor6 = Real(1.0f) / Real(6.0f);
        Real un[NVAR];
        double Eun = 0.0;   // E + b R in binary64 (E pair builds)
#pragma unroll
        for (int q = 0; q < NVAR; ++q) {
            // folded: R already holds a R - dtinvh (x+y part)
            const Real t = kFold ? F.f[q] - Fl.f[q] : (in.acc[q] + F.f[q]) - Fl.f[q];
            Real rhs;
            if (q == FG)      rhs = dtinvh*(t - dU * sG * factor6);
            else if (q == FP) rhs = dtinvh*(t - dU * sP * factor6);
            else              rhs = dtinvh*t;
            // folded: R holds a R - dtinvh (x+y part), or a R - (x+y part)
            // when unscaled (an explicit product: no contraction into the
            // subtraction, so it rounds as the x+y sweep's product would)
            const Real Rx = !kFold ? A.a*in.R[q] : unscaled_stage(A.a) ? __fmul_rn(dtinvh, in.R[q]) : in.R[q];
            const Real Rn = Rx - rhs;
            if constexpr (MODE != MODE_STAGE_NOR) st_lane<true>(E.R.p[q], off, Rn);
            if constexpr (is_stage(MODE)) {
                if (kEPair && q == FE) {
                    // E + b R in binary64, stored as the rounded sum and its
                    // remainder (exact: |remainder| <= half an ulp of the sum)
                    const double Ed = (double(in.u[FE]) + double(in.u[FELO])) + double(A.b) * double(Rn);
                    const Real hi = Real(Ed);
                    un[q] = hi;
                    st_lane<true>(E.uo.p[q], off, hi);
                    st_lane<true>(E.uo.p[FELO], off, Real(Ed - double(hi)));
                    Eun = Ed;
                } else {
                    un[q] = A.b*Rn + in.u[q];
                    st_lane<true>(E.uo.p[q], off, un[q]);
                }
            }
        }
        // the next step's speed of sound, from the values just stored
        if (is_stage(MODE) && A.sos_next) {
            bool b;
            smax = mmax(smax, sos_cell(A.sos_cpu != 0, un[0], un[1], un[2], un[3], kEPair ? SosT(Eun) : SosT(un[4]),
                                       un[5], un[6], b));
            bad = bad || b;
        }
    }
}

// marching state along direction D
template <int D, int MODE>
struct March
{
    Prim w0, w1, w2, w3, w4;   // primitives of cells k-2 .. k+2
    Prim pm;                   // minus-state (face k-1/2) of cell k-1
    Real pGp, pPp;             // plus-state G,P (face k-3/2) of cell k-1
    FaceFlux Fl;               // flux at face k-3/2
    SosT smax = 0;             // running max speed of sound of the emitted cells (folded step)
    bool bad = false;          // an emitted cell is non-finite or non-physical (folded step)

    __device__ __forceinline__ void push(const Prim& q) { w0 = w1; w1 = w2; w2 = w3; w3 = w4; w4 = q; }

    // reconstruct cell k, solve face k-1/2 (FLUX: k >= c0), emit cell k-1
    // (EMIT: k >= c0 + 1; operands in `in`).  FLUX and EMIT are bools or
    // std::bool_constant (the peeled steps of an unrolled march)
    template <class FLUX, class EMIT>
    __device__ __forceinline__ void step(const StageArgs& A, const Real dtinvh, const FLUX flux, const EMIT em,
                                         const EmitPtr<MODE>& E, const uint32_t off_km1, const EmitIn<MODE>& in)
    {
        const CellRec r = reconstruct<Real, kFast>(w0, w1, w2, w3, w4);
        if (flux) {
            const FaceFlux F = riemann<D, Real, kFast>(pm, r.p);
            if (em) emit<MODE>(A, E, dtinvh, off_km1, in, F, Fl, pGp + pm.G, pPp + pm.P, smax, bad);
            Fl = F;
        }
        pm = r.m; pGp = r.p.G; pPp = r.p.P;
    }
};

__device__ __forceinline__ Prim load_prim(const Real* __restrict__ u, const int64_t fs, const int e)
{
    return to_prim<Real, kFast, kP64, kEPair>(u[e], u[fs + e], u[2*fs + e], u[3*fs + e], u[4*fs + e], u[5*fs + e],
                                              u[6*fs + e], kEPair ? u[FELO*fs + e] : Real(0));
}

__device__ __forceinline__ Real stage_dtinvh(const StageArgs& A)
{
    if (!A.st) return A.dtinvh;
    return MPCF_F64 ? Real(A.st->dtinvh_d) : Real(A.st->dtinvh);
}

// ---------------------------------------------------------------------------
// y / z sweeps: block of 256 lanes over the flattened (x, transverse) columns,
// blockIdx.y = chunk of the marched axis.
// ---------------------------------------------------------------------------
// one column of a y / z sweep; returns the running max speed of sound of the
// cells it wrote and sets bad if one of them is non-finite or non-physical
// (zero / false unless A.sos_next)
template <int D, int MODE>
__device__ __forceinline__ SosT sweep_yz_column(const Geom& g, const StageArgs& A, const int chunk, const int x,
                                                const int row, const int bz, bool& bad)
{
    const int nd = D == 1 ? g.ny : g.nz;
    // the y sweep's columns lie in the launch's planes [z0, z1); the z sweep
    // marches its launch's rows [z0, z1) (boundary conditions still use the
    // whole extent nd)
    const int t = (D == 1 ? A.z0 : 0) + row;
    const int c0 = (D == 2 ? A.z0 : 0) + bz * chunk;
    const int c1 = min(c0 + chunk, D == 2 ? A.z1 : nd);
    const int s = g.stride(D);
    const int e0 = D == 1 ? g.idx(x, 0, t) : g.idx(x, t, 0);
    // the columns of a wave are consecutive: the first active lane's element is the least
    const LaneIdx L = lane_idx(e0, e0, (int64_t)c0 * s);
    constexpr int NEGQ = D == 1 ? FV : FW;   // normal momentum of the marched axis
    constexpr int FLO = 2 * D;               // its low face
    const Real* const u0 = A.u + L.base;   // row c0
    const Bases<NU, const Real> U(u0 - GHOST * (int64_t)s, A.fs);   // row c0 - 3 (y sweep)
    const EmitPtr<MODE> E(A, L.base);
    // byte offset of row k (c0 <= k < c1: the launch keeps chunks within 32 bits)
    auto off = [&](const int k) { return L.lo + (uint32_t)(k - c0) * (uint32_t)s * (uint32_t)sizeof(Real); };
    // the y sweep of a first stage stores its part unscaled and does not read dt
    const Real dtinvh = (MODE == MODE_ACC && unscaled_stage(A.a)) ? Real(0.0f) : stage_dtinvh(A);
    const int64_t fs = A.fs;
    auto load = [&](const int row, Real* out) {
        if constexpr (D == 2) return load_row_far(A, u0, L.lo, c0, row, nd, s, FLO, out);
        else                  return load_row(A, U, L.lo, c0 - GHOST, row, nd, s, FLO, out);
    };
    constexpr bool kRaw = is_stage(MODE);   // the update needs the raw u of the emitted cell

    March<D, MODE> m;
    // raw conserved values of cells k-1 .. k+2 (kept for the register update;
    // the emitted cell k-1 is always interior, so its raw values are exact)
    Real r0[NU], r1[NU], r2[NU], r3[NU], w[NU];
    r1[NEGQ] *= load(c0 - 2, r1);
    r2[NEGQ] *= load(c0 - 1, r2);
    r3[NEGQ] *= load(c0, r3);
    w[NEGQ] *= load(c0 - 3, w);
    m.w1 = prim_of(w);
    m.w2 = prim_of(r1);
    m.w3 = prim_of(r2);
    m.w4 = prim_of(r3);
    // software pipeline: raw values of the next incoming cell and the emit
    // operands of the next step are loaded one step ahead
    Real nxt[NU];
    Real nsg = load(c0 + 1, nxt);
    EmitIn<MODE> ein, ein_next;
    // one march step at row k.  FLUX: face k-1/2 is solved (k >= c0); EMIT:
    // cell k-1 is written (k >= c0 + 1); PF: row k+3 is prefetched and the
    // emit operands of cell k are loaded (k < c1; the latter from k >= c0)
    auto step = [&](auto FLUX, auto EMIT, auto PF, const int k) {
        nxt[NEGQ] *= nsg;   // boundary sign of the prefetched row
        // rotate the raw ring: r0 = cell k-1, r3 = cell k+2
#pragma unroll
        for (int q = 0; q < NU; ++q) { r0[q] = r1[q]; r1[q] = r2[q]; r2[q] = r3[q]; r3[q] = nxt[q]; }
        const Prim q = prim_of(nxt);  // cell k+2
        if (PF) nsg = load(k + 3, nxt);
        if (PF && FLUX) emit_load<MODE>(E, off(k), ein_next);   // emitted at step k+1
        if (kRaw) {
#pragma unroll
            for (int f = 0; f < NU; ++f) ein.u[f] = r0[f];                   // cell k-1
        }
        m.push(q);
        // The stages' z sweeps of the P64 builds, whose folded speed of sound is
        // binary64, take 257 to 260 VGPRs and run one wave per SIMD unless a
        // row's instructions keep out of the next row's (246 to 253 VGPRs): z
        // sweep of 128^3 63.1 -> 55.2 us, 192^3 180.6 -> 157.1, E pair 65.7 ->
        // 57.8 and 189.4 -> 167.3
        if constexpr (kEPair && is_stage(MODE)) __builtin_amdgcn_sched_barrier(0);
        m.step(A, dtinvh, FLUX, EMIT, E, off(k - 1), ein);
        if constexpr (kP64 && is_stage(MODE)) __builtin_amdgcn_sched_barrier(0);
        ein = ein_next;
    };
    if constexpr (kUnrollMarch) {
        using T_ = std::true_type;
        using F_ = std::false_type;
        step(F_{}, F_{}, T_{}, c0 - 1);
        step(T_{}, F_{}, T_{}, c0);
        int k = c0 + 1;
        // five steps per trip, the period of the window of primitives
        for (; k + 5 <= c1; k += 5) {
            step(T_{}, T_{}, T_{}, k);
            step(T_{}, T_{}, T_{}, k + 1);
            step(T_{}, T_{}, T_{}, k + 2);
            step(T_{}, T_{}, T_{}, k + 3);
            step(T_{}, T_{}, T_{}, k + 4);
        }
        for (; k < c1; ++k) step(T_{}, T_{}, T_{}, k);
        step(T_{}, T_{}, F_{}, c1);      // c1 >= c0 + 1: every chunk has a row
    } else {
        for (int k = c0 - 1; k <= c1; ++k) step(k >= c0, k >= c0 + 1, k < c1, k);
    }
    bad = m.bad;
    return m.smax;
}

// column `col` of the columns (x, t) flattened x-fastest, `width` of them a row
// (nx, or z_width's for a z sweep): consecutive lanes are consecutive x
// (coalesced); the columns x >= nx idle.  Every thread of the workgroup (256 threads, unless PER_WAVE) takes
// part (the fold reduction)
// PER_WAVE: the fold's atomics are issued by every wave, with no barrier (the
// persistent kernels, whose item loop keeps its barriers in calls of their own)
template <int D, int MODE, bool PER_WAVE = false>
__device__ __forceinline__ void sweep_yz_body(const Geom& g, const StageArgs& A, const int chunk,
                                              const int width, const int col, const int bz)
{
    const int nt = D == 1 ? A.z1 - A.z0 : g.ny;
    SosT smax = 0;
    bool bad = false;
    const int row = col / width, x = col - row * width;
    if (row < nt && x < g.nx) smax = sweep_yz_column<D, MODE>(g, A, chunk, x, row, bz, bad);   // no barriers in the body
    if (is_stage(MODE) && A.sos_next) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) smax = mmax(smax, __shfl_xor(smax, off, 64));
        int anybad = __ballot(bad) != 0;
        const int wave = threadIdx.x >> 6;
        bool first = (threadIdx.x & 63) == 0;
        if constexpr (!PER_WAVE) {
            // one atomic max (and, for a bad cell, one atomic or) per workgroup:
            // they take turns at one address, and one per wave took 5 us of
            // the 12 us of a 32^3 block's last sweep
            __shared__ SosT wmax[4];
            __shared__ int wbad[4];
            if (first) { wmax[wave] = smax; wbad[wave] = anybad; }
            __syncthreads();
            smax = mmax(mmax(wmax[0], wmax[1]), mmax(wmax[2], wmax[3]));
            anybad = wbad[0] | wbad[1] | wbad[2] | wbad[3];
            first = threadIdx.x == 0;
        }
        if (first) {
            if (smax > SosT(0)) {
                if (kSosD) atomicMax(&A.sos_next->next_sos_bits_d, (unsigned long long)__double_as_longlong((double)smax));
                else       atomicMax(&A.sos_next->next_sos_bits, __float_as_uint((float)smax));
            }
            if (anybad) atomicOr(&A.sos_next->next_bad, 1u);
        }
    }
}

template <int D, int MODE>
__global__ __launch_bounds__(256)
void k_sweep_yz(const Geom g, const StageArgs A, const int chunk, const int width)
{
    sweep_yz_body<D, MODE>(g, A, chunk, width, blockIdx.x * 256 + threadIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------
// x sweep: one wave per block, lane = pencil (y,z) flattened.  x-runs of SX
// cells of the block's 64 pencils are loaded with contiguous segments,
// converted to primitives and staged in LDS; each lane then marches its own
// pencil through the run.  The run's outputs are staged in LDS as well and
// stored back as contiguous segments (lane-per-pencil stores would touch 64
// cache lines per instruction).  The raw values of the next run are loaded
// into registers while the current run is computed.
// ---------------------------------------------------------------------------
enum { SX = 8 };

struct XStage
{
    Real in[NVAR][64][SX + 1];     // primitives of the current run
    Real out[NACC][64][SX + 1];    // outputs of cells xs-3 .. xs+SX-4
};

// x-sweep output for one cell, written to LDS instead of global memory
__device__ __forceinline__ void emit_first_lds(XStage& S, const int lane, const int slot, const FaceFlux& F,
                                               const FaceFlux& Fl, const Real cG, const Real cP)
{
#pragma unroll
    for (int q = 0; q < NVAR; ++q) S.out[q][lane][slot] = F.f[q] - Fl.f[q];
    S.out[A_SUMG][lane][slot] = cG;
    S.out[A_SUMP][lane][slot] = cP;
    S.out[A_DIVU][lane][slot] = F.vel - Fl.vel;
}

__global__ __launch_bounds__(64)
void k_sweep_x(const Geom g, const StageArgs A, const int chunk)
{
    __shared__ XStage S;
    const int lane = threadIdx.x;
    const int npen = g.ny * (A.z1 - A.z0);     // pencils (y, z) of the launch's planes [z0, z1)
    const int pb = blockIdx.x * 64;
    const int c0 = blockIdx.y * chunk;
    const int c1 = min(c0 + chunk, g.nx);
    const int64_t fs = A.fs;
    const int xl = lane % SX;

    // element index of x = 0 for the 8 pencils this lane stages/stores
    int sbase[8];
    bool sok[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int p = pb + i * 8 + lane / SX;
        sok[i] = p < npen;
        const int pc = sok[i] ? p : npen - 1;
        sbase[i] = g.idx(0, pc % g.ny, A.z0 + pc / g.ny);
    }
    const bool active = pb + lane < npen;

    // raw values of the next run: cell xs + xl of the lane's 8 staging pencils
    Real pre[8][NVAR];
    Real pre_sg;   // boundary sign of the prefetched run's x-momentum, applied when it is staged
    auto load_run = [&](const int xs) {
        const int xc = min(xs + xl, c1 + 2);   // reads past the run end are clamped to the stencil reach
        const int xm = bc_index(xc, g.nx, A.bcmask, 0, pre_sg);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int q = 0; q < NVAR; ++q) pre[i][q] = A.u[q * fs + sbase[i] + xm];
    };

    March<0, MODE_FIRST> m;
    int xs = c0 - 3;
    load_run(xs);
    for (; xs <= c1 + 2; xs += SX) {
        // stage the run (previous run's consumers and storers are past the barrier below)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const Prim q = to_prim<Real, kFast, kP64>(pre[i][0], pre[i][1] * pre_sg, pre[i][2], pre[i][3], pre[i][4],
                                                      pre[i][5], pre[i][6]);
            const int pl = i * 8 + lane / SX;
            S.in[FR][pl][xl] = q.r; S.in[FU][pl][xl] = q.u; S.in[FV][pl][xl] = q.v; S.in[FW][pl][xl] = q.w;
            S.in[FE][pl][xl] = q.p; S.in[FG][pl][xl] = q.G; S.in[FP][pl][xl] = q.P;
        }
        if (xs + SX <= c1 + 2) load_run(xs + SX);
        __syncthreads();
        const int nj = min(SX, c1 + 3 - xs);
        for (int j = 0; j < nj; ++j) {
            Prim q;
            q.r = S.in[FR][lane][j]; q.u = S.in[FU][lane][j]; q.v = S.in[FV][lane][j]; q.w = S.in[FW][lane][j];
            q.p = S.in[FE][lane][j]; q.G = S.in[FG][lane][j]; q.P = S.in[FP][lane][j];
            m.push(q);
            const int k = xs + j - 2;              // cell reconstructed at this step
            if (k >= c0 - 1) {
                const CellRec r = reconstruct<Real, kFast>(m.w0, m.w1, m.w2, m.w3, m.w4);
                if (k >= c0) {
                    const FaceFlux F = riemann<0, Real, kFast>(m.pm, r.p);
                    if (k >= c0 + 1) emit_first_lds(S, lane, j, F, m.Fl, m.pGp + m.pm.G, m.pPp + m.pm.P);
                    m.Fl = F;
                }
                m.pm = r.m; m.pGp = r.p.G; m.pPp = r.p.P;
            }
        }
        __syncthreads();
        // outputs of this run are cells xs-3+j for the slots j written above
        const int xo = xs - 3 + xl;
        if (xo >= c0 && xo < c1 && xl < nj) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!sok[i]) continue;
                const int pl = i * 8 + lane / SX;
#pragma unroll
                for (int q = 0; q < NACC; ++q) A.acc[q * fs + sbase[i] + xo] = S.out[q][pl][xl];
            }
        }
    }
    (void)active;
}

// ---------------------------------------------------------------------------
// fused x + y sweep: lanes along x, marching y.  A wave covers 64 consecutive
// x-cells.  FAST: it writes the 58 whose x-stencils lie inside the wave (lanes
// 3..60), and neighbouring tiles overlap by six cells.  The other builds: it
// writes the 62 whose faces' two cells lie inside the wave (lanes 1..62); the
// primitives of two cells beside the wave on either side come from LDS, and
// neighbouring tiles overlap by two cells.  The x-direction of row k-1 is computed from the rolling window's
// row k-1 with wave-shifted copies (DPP wave_shr/wave_shl) for the five-point
// windows, the left face state and the right face flux; the y-direction is
// the same register march as the y sweep.  The accumulators leave this kernel
// already summed in the x-then-y order of the reference (GPUkernels.cu:1111),
// so the x sweep's accumulator round trip disappears.
// ---------------------------------------------------------------------------
// The bit-exact and binary64 builds take the two positions beside a wave on
// either side from LDS and store 62 of its 64 lanes; the FAST builds keep them
// inside the wave and store 58.  The row's edge values cost FAST 14 differences
// and the registers of the LDS reads against 6.5 % fewer waves: 512^3 19.4 ms a
// step against 18.8, 256^3 whole-block 2.69 against 2.60; the bit-exact build,
// with 3 times the arithmetic per cell, gains (while it solved its x faces
// twice): 256^3 6.32 against 6.45, a 600x300x6 block 0.545 against 0.565;
// binary64 128^3 1.42 against 1.43.
constexpr bool kHaloLDS = !kFast;
enum { XY_TILE = kHaloLDS ? 62 : 58 };
static_assert(!kHaloLDS || !kUnrollXY, "the unrolled march does not refill the rows in LDS");
constexpr int kHaloRows = 16;   // rows of edge primitives a wave keeps in LDS: 16 x 4 positions fill its lanes

// value of lane l-1 / lane l+1.  The wave's edge lanes (no source lane) read
// zero: they are halo positions whose results are never stored, and with no
// old value to keep the shift is one v_mov_b32_dpp (no copy of the operand),
// which the compiler can also fold into the consuming VALU instruction
template <int CTRL>
__device__ __forceinline__ float dpp_move(const float v)
{
    const int b = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(b, CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(const double v)
{
    // the two 32-bit halves move with the same lane shift
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = (int)(b & 0xffffffffLL), hi = (int)(b >> 32);
    const int lo2 = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true);
    const int hi2 = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((long long)hi2 << 32) | (long long)(unsigned)lo2);
}
__device__ __forceinline__ Real from_left(const Real v) { return dpp_move<0x138>(v); }    // wave_shr:1
__device__ __forceinline__ Real from_right(const Real v) { return dpp_move<0x130>(v); }   // wave_shl:1
// the same, the wave's edge lane taking `edge` (its value in that lane)
template <int CTRL>
__device__ __forceinline__ float dpp_move(const float edge, const float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v),
                                                                 CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(const double edge, const double v)
{
    const long long b = __builtin_bit_cast(long long, v), o = __builtin_bit_cast(long long, edge);
    const int lo = __builtin_amdgcn_update_dpp((int)(o & 0xffffffffLL), (int)(b & 0xffffffffLL), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ Real from_left(const Real edge, const Real v) { return dpp_move<0x138>(edge, v); }
__device__ __forceinline__ Real from_right(const Real edge, const Real v) { return dpp_move<0x130>(edge, v); }

// One primitive at the four positions beside a wave, as the x reconstruction
// of its edge lanes needs it: two and one left of lane 0, one and two right of
// lane 63 (kHaloLDS)
typedef Real Halo4 __attribute__((ext_vector_type(4)));

// orders the wave's LDS accesses before it against those after it, for all its
// lanes: LDS serves one wave's accesses in order, so it holds the compiler back
// and costs no instruction
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The x faces of a wave, each lane's face to its left: lane 0 has no left state
// (it reads zeros), and its face is not used.  Counted among the faces whose
// operands decide on the quick quotients, it had every wave solve every x face
// of the bit-exact build twice
constexpr uint64_t kXFaceLanes = ~uint64_t(1);

__device__ __forceinline__ Prim prim_from_left(const Prim& q)
{
    Prim o;
    o.r = from_left(q.r); o.u = from_left(q.u); o.v = from_left(q.v); o.w = from_left(q.w);
    o.p = from_left(q.p); o.G = from_left(q.G); o.P = from_left(q.P);
    return o;
}

// workgroups go to the XCDs round-robin by linear id; this maps linear id
// `lin` of a grid of n to a tile index such that each XCD takes a contiguous
// run of tiles, so that neighbouring tiles of the fused x+y sweep (which
// overlap by 64 - XY_TILE positions and share partial cache lines) meet in one L2.
// For grids of equal-cost tiles (one block)
__device__ __forceinline__ int xcd_order(const int lin, const int n)
{
    const int xcd = lin % kXCDs, k = lin / kXCDs;
    const int per = n / kXCDs, extra = n % kXCDs;
    return xcd * per + min(xcd, extra) + k;
}

// x-direction reconstruction of each lane's cell from its lane neighbours (and,
// kHaloLDS, at the wave's edges the positions beside it).
// FAST: the second difference is formed once per lane and shifted (a lane's Db
// is its left neighbour's Dc, the same subtractions of the same values)
template <bool SYNC, bool QUICK>
__device__ __forceinline__ RecT<Real> weno_lanes(const Real c, const Halo4 h, bool* odd)
{
    if constexpr (kFast) {
        const Real b = from_left(c), d = from_right(c);
        const Real dbc = c - b, dcd = d - c;
        const Real D = dcd - dbc;
        const Real Db = from_left(D), Dd = from_right(D);
        keep_phase<SYNC>();
        return weno_fast_core<Real, SYNC>(b, c, d, dbc, dcd, Db, D, Dd, weno_kD<Real>(Db), weno_kD<Real>(D), weno_kD<Real>(Dd));
    } else {
        const Real b = from_left(h[1], c), d = from_right(h[2], c);
        return weno_cell<Real, kFast, QUICK, SYNC>(from_left(h[0], b), b, c, d, from_right(h[3], d), odd);
    }
}
// halo: the row's Halo4 of the seven primitives
template <bool SYNC, bool QUICK>
__device__ __forceinline__ CellRec reconstruct_lanes_as(const Prim& c, const Halo4* halo, bool* odd)
{
    constexpr bool S = SYNC && (kFast || QUICK);
    CellRec o;
    RecT<Real> t;
    t = weno_lanes<S, QUICK>(c.r, halo[0], odd); o.m.r = t.m; o.p.r = t.p;
    t = weno_lanes<S, QUICK>(c.u, halo[1], odd); o.m.u = t.m; o.p.u = t.p;
    t = weno_lanes<S, QUICK>(c.v, halo[2], odd); o.m.v = t.m; o.p.v = t.p;
    t = weno_lanes<S, QUICK>(c.w, halo[3], odd); o.m.w = t.m; o.p.w = t.p;
    t = weno_lanes<S, QUICK>(c.p, halo[4], odd); o.m.p = t.m; o.p.p = t.p;
    t = weno_lanes<S, QUICK>(c.G, halo[5], odd); o.m.G = t.m; o.p.G = t.p;
    t = weno_lanes<S, QUICK>(c.P, halo[6], odd); o.m.P = t.m; o.p.P = t.p;
    return o;
}
// as reconstruct(): the bit-exact builds take the quick quotients, and the
// IEEE ones where a lane's window needs them
template <bool SYNC>
__device__ __forceinline__ CellRec reconstruct_lanes(const Prim& c, const Halo4* halo, bool* again = nullptr)
{
    if constexpr (!kFast) {
        bool odd = false;
        CellRec o = reconstruct_lanes_as<SYNC, true>(c, halo, &odd);
        if (again) *again = any_lane(odd);
        if (__builtin_expect(any_lane(odd), 0)) o = reconstruct_lanes_as<SYNC, false>(c, halo, nullptr);
        return o;
    } else {
        return reconstruct_lanes_as<SYNC, false>(c, halo, nullptr);
    }
}

// what a FAST march along y carries of one primitive besides the window: the
// second differences of the two cells before the newest and their products
struct Diff2 { Real D0, D1, k0, k1; };

// y-direction reconstruction of row k of one primitive from rows k-1 .. k+2
// (b, c, d, e); s holds rows k-1 and k on entry, rows k and k+1 on return
template <bool SYNC>
__device__ __forceinline__ Rec weno_march(const Real b, const Real c, const Real d, const Real e, Diff2& s)
{
    const Real dbc = c - b, dcd = d - c, dde = e - d;
    const Real D2 = dde - dcd, k2 = weno_kD<Real>(D2);
    const Rec r = weno_fast_core<Real, SYNC>(b, c, d, dbc, dcd, s.D0, s.D1, D2, s.k0, s.k1, k2);
    s.D0 = s.D1; s.D1 = D2;
    s.k0 = s.k1; s.k1 = k2;
    return r;
}

// the y reconstruction of the x+y march: FAST carries the second differences,
// the other builds evaluate the window as it stands
template <bool SYNC>
struct YRec
{
    Diff2 r, u, v, w, p, G, P;

    // rows c0-3 .. c0 (a, b, c, d): the state for the first row, c0 - 1
    static __device__ __forceinline__ Diff2 first(const Real a, const Real b, const Real c, const Real d)
    {
        Diff2 s;
        s.D0 = (c - b) - (b - a); s.k0 = weno_kD<Real>(s.D0);
        s.D1 = (d - c) - (c - b); s.k1 = weno_kD<Real>(s.D1);
        return s;
    }
    __device__ __forceinline__ void start(const Prim& a, const Prim& b, const Prim& c, const Prim& d)
    {
        if constexpr (!kFast) return;
        r = first(a.r, b.r, c.r, d.r); u = first(a.u, b.u, c.u, d.u); v = first(a.v, b.v, c.v, d.v);
        w = first(a.w, b.w, c.w, d.w); p = first(a.p, b.p, c.p, d.p); G = first(a.G, b.G, c.G, d.G);
        P = first(a.P, b.P, c.P, d.P);
    }
    __device__ __forceinline__ CellRec row(const Prim& A, const Prim& B, const Prim& C, const Prim& D, const Prim& E)
    {
        if constexpr (!kFast) return reconstruct<Real, kFast, SYNC>(A, B, C, D, E);
        CellRec o;
        Rec t;
        t = weno_march<SYNC>(B.r, C.r, D.r, E.r, r); o.m.r = t.m; o.p.r = t.p;
        t = weno_march<SYNC>(B.u, C.u, D.u, E.u, u); o.m.u = t.m; o.p.u = t.p;
        t = weno_march<SYNC>(B.v, C.v, D.v, E.v, v); o.m.v = t.m; o.p.v = t.p;
        t = weno_march<SYNC>(B.w, C.w, D.w, E.w, w); o.m.w = t.m; o.p.w = t.p;
        t = weno_march<SYNC>(B.p, C.p, D.p, E.p, p); o.m.p = t.m; o.p.p = t.p;
        t = weno_march<SYNC>(B.G, C.G, D.G, E.G, G); o.m.G = t.m; o.p.G = t.p;
        t = weno_march<SYNC>(B.P, C.P, D.P, E.P, P); o.m.P = t.m; o.p.P = t.p;
        return o;
    }
};

// wave `wv` of the x+y sweep over rows [bz * chunk, bz * chunk + chunk).
// FIRST (folded builds, a = 0 known at launch): R is not read -- the stage
// multiplies it by zero -- which takes 28 B/cell from that stage's traffic
// SYNC: the waves of the workgroup keep phase (keep_phase); all of them run
// rows of the same chunk, and a wave past the end leaves the kernel
template <bool FIRST = false, bool SYNC = false>
__device__ __forceinline__ void sweep_xy_body(const Geom& g, const StageArgs& A, const int chunk,
                                              const int wv, const int wib, const int bz)
{
    // positions q along the padded rows (x = -3 .. nx+2) of all z-planes,
    // flattened; ghost positions are computed but never stored.  Wave w (wib:
    // its place in the workgroup) of the FAST builds covers q = 58 w .. 58 w +
    // 63 and stores lanes 3..60, so consecutive waves overlap by six positions.
    // kHaloLDS: it covers q = 62 w + 2 .. 62 w + 65 and stores lanes 1..62: a
    // stored cell's faces need the reconstruction of its lane neighbours, and
    // theirs the primitives of two positions beside the wave on either side.
    // Those come from LDS, where the wave puts them for 16 rows at a time, a
    // lane per row and position (one conversion of 64 lanes, then 7 broadcast
    // reads a row), bit for bit what the neighbouring wave computes.
    const int lane = threadIdx.x & 63;
    const int rowlen = g.nx + 6;
    const int nzr = A.z1 - A.z0;                  // planes of this launch
    const int q = wv * XY_TILE + (kHaloLDS ? 2 : 0) + lane;
    int z = q / rowlen;
    const int x = q - z * rowlen - 3;
    const bool store = lane >= (kHaloLDS ? 1 : 3) && lane <= (kHaloLDS ? 62 : 60) && x >= 0 && x < g.nx && z < nzr;
    if (wv * XY_TILE >= rowlen * nzr) return;     // whole wave past the end
    z = A.z0 + min(z, nzr - 1);                   // lanes past the last plane read its last row
    // lanes outside [0, nx) read the cell their x-ghost copies
    Real sgx;
    const int xm = bc_index(x, g.nx, A.bcmask, 0, sgx);
    const bool xmirror = (A.bcmask & 3) != 0;
    const int c0 = bz * chunk;
    const int c1 = min(c0 + chunk, g.ny);
    const int s = g.px;
    const int e0 = g.idx(xm, 0, z);
    // every lane's element is at least that of the first ghost column of lane
    // 0's plane (lanes left of x = 0 read it on a halo face)
    const int r0 = c0 - GHOST;             // the first row of the chunk's stencils
    const LaneIdx L = lane_idx(e0, g.idx(-GHOST, 0, z), (int64_t)r0 * s);
    const int64_t fs = A.fs;
    // row r0 of the fields; a plane is well under 4 GB, so the rows of a chunk
    // are within 32-bit offsets
    const Bases<NU, const Real> U(A.u + L.base, fs);
    const Bases<NVAR, Real> R((kFold ? A.R : A.acc) + L.base, fs);
    const Bases<3, Real> gp(A.acc + L.base + A_SUMG * fs, fs);
    // boundary signs of a loaded row: y-momentum by the row's mapping,
    // x-momentum by the lane's (applied where the values are consumed)
    auto fix = [&](Real* o, const Real sgy) {
        o[FV] *= sgy;
        if (xmirror) o[FU] *= sgx;
    };

    // scalars, a Halo4 each: four lanes write the four positions of one, and a
    // store into an element of a vector reads and writes the whole vector
    __shared__ alignas(sizeof(Halo4)) Real sh_halo[kHaloLDS ? 4 : 1][kHaloLDS ? kHaloRows : 1][NVAR][4];
    // primitives beside the wave of rows [h0, h0 + kHaloRows), interior rows
    int h0 = c0 - kHaloRows;
    auto fill_halo = [&](const int row0) {
        wave_sync();   // the wave's lanes have read the rows that go
        h0 = row0;
        const int j = lane >> 2, side = lane & 3;
        const int row = min(row0 + j, c1 - 1);
        // a position left of the wave's first plane is never needed (it reads
        // that plane's first ghost)
        const int qh = max(wv * XY_TILE + (side < 2 ? side : 64 + side), (wv * XY_TILE + 2) / rowlen * rowlen);
        const int zq = qh / rowlen;
        Real sx;
        const int xh = bc_index(qh - zq * rowlen - 3, g.nx, A.bcmask, 0, sx);
        const uint32_t off = (uint32_t)(g.idx(xh, row, A.z0 + min(zq, nzr - 1)) - L.base) * (uint32_t)sizeof(Real);
        Real w[NU];
#pragma unroll
        for (int f = 0; f < NU; ++f) w[f] = ld_lane(U.p[f], off);
        if (xmirror) w[FU] *= sx;
        const Prim p = prim_of(w);
        const Real v[NVAR] = {p.r, p.u, p.v, p.w, p.p, p.G, p.P};
#pragma unroll
        for (int f = 0; f < NVAR; ++f) sh_halo[wib][j][f][side] = v[f];
        wave_sync();   // the rows are there for every lane
    };

    March<1, MODE_ACC> m;
    Real w[NU];
    fix(w, load_row(A, U, L.lo, r0, c0 - 3, g.ny, s, 2, w)); m.w1 = prim_of(w);
    fix(w, load_row(A, U, L.lo, r0, c0 - 2, g.ny, s, 2, w)); m.w2 = prim_of(w);
    fix(w, load_row(A, U, L.lo, r0, c0 - 1, g.ny, s, 2, w)); m.w3 = prim_of(w);
    fix(w, load_row(A, U, L.lo, r0, c0, g.ny, s, 2, w));     m.w4 = prim_of(w);
    YRec<SYNC> yrec;
    yrec.start(m.w1, m.w2, m.w3, m.w4);
    Real nxt[NU];
    Real nsg = load_row(A, U, L.lo, r0, c0 + 1, g.ny, s, 2, nxt);
    // a first stage stores its x+y part unscaled and does not read dt
    const bool unscaled = FIRST || unscaled_stage(A.a);
    const Real dtinvh = unscaled ? Real(0.0f) : stage_dtinvh(A);
    // one march step at row k.  FLUX: the face below row k is solved
    // (k >= c0); EMIT: row k-1 is finished and written (k >= c0 + 1); PF: row
    // k+3 is prefetched (k < c1)
    auto step = [&](auto FLUX, auto EMIT, auto PF, const int k) {
        fix(nxt, nsg);
        const Prim q = prim_of(nxt);  // row k+2
        if (PF) nsg = load_row(A, U, L.lo, r0, k + 3, g.ny, s, 2, nxt);
        // folded builds: R of row k-1, emitted below (every lane's address is
        // an interior cell, stored or not)
        const uint32_t off_km1 = L.lo + (uint32_t)((k - 1 - r0) * s) * (uint32_t)sizeof(Real);
        Real Ro[NVAR];
        if (kFold && EMIT && !FIRST) {
#pragma unroll
            for (int f = 0; f < NVAR; ++f) Ro[f] = ld_lane(R.p[f], off_km1);
        }
        m.push(q);
        const CellRec ry = yrec.row(m.w0, m.w1, m.w2, m.w3, m.w4);              // row k, y-direction
        if (FLUX) {
            const FaceFlux Fy = riemann<1, Real, kFast, SYNC>(m.pm, ry.p);          // face k-1/2
            if (EMIT) {
                // x-direction of row k-1 (window slot w1)
                Halo4 halo[NVAR];
#pragma unroll
                for (int f = 0; f < NVAR; ++f)
                    if constexpr (kHaloLDS) halo[f] = *(const Halo4*)sh_halo[wib][k - 1 - h0][f];
                const CellRec rx = reconstruct_lanes<SYNC>(m.w1, halo);
                const Prim Lm = prim_from_left(rx.m);
                const FaceFlux Fxl = riemann<0, Real, kFast, SYNC, kXFaceLanes>(Lm, rx.p);      // face x-1/2
                FaceFlux Fxr;                                                        // face x+1/2
#pragma unroll
                for (int f = 0; f < NVAR; ++f) Fxr.f[f] = from_right(Fxl.f[f]);
                Fxr.vel = from_right(Fxl.vel);
                if (store) {
                    const Real cGy = m.pGp + m.pm.G, cPy = m.pPp + m.pm.P;
#pragma unroll
                    for (int f = 0; f < NVAR; ++f) {
                        const Real t = ((Fxr.f[f] - Fxl.f[f]) + Fy.f[f]) - m.Fl.f[f];
                        // first stage: -t, which is 0 R - t up to the sign of a zero
                        if (kFold) st_lane(R.p[f], off_km1, unscaled ? -t : A.a*Ro[f] - dtinvh*t);
                        else       st_lane(R.p[f], off_km1, t);
                    }
                    st_lane<true>(gp.p[0], off_km1, (rx.p.G + rx.m.G) + cGy);
                    st_lane<true>(gp.p[1], off_km1, (rx.p.P + rx.m.P) + cPy);
                    st_lane<true>(gp.p[2], off_km1, (Fxr.vel - Fxl.vel) + (Fy.vel - m.Fl.vel));
                }
            }
            m.Fl = Fy;
        }
        m.pm = ry.m; m.pGp = ry.p.G; m.pPp = ry.p.P;
    };
    if constexpr (kUnrollXY) {
        using T_ = std::true_type;
        using F_ = std::false_type;
        step(F_{}, F_{}, T_{}, c0 - 1);
        step(T_{}, F_{}, T_{}, c0);
        int k = c0 + 1;
        // five steps per trip, the period of the window of primitives: the
        // window then rotates by register renaming instead of ~50 moves a step
        for (; k + 5 <= c1; k += 5) {
            step(T_{}, T_{}, T_{}, k);
            step(T_{}, T_{}, T_{}, k + 1);
            step(T_{}, T_{}, T_{}, k + 2);
            step(T_{}, T_{}, T_{}, k + 3);
            step(T_{}, T_{}, T_{}, k + 4);
        }
        for (; k < c1; ++k) step(T_{}, T_{}, T_{}, k);
        step(T_{}, T_{}, F_{}, c1);      // c1 >= c0 + 1: every chunk has a row
    } else {
        for (int k = c0 - 1; k <= c1; ++k) {
            if (kHaloLDS && k > c0 && k > h0 + kHaloRows) fill_halo(k - 1);
            step(k >= c0, k >= c0 + 1, k < c1, k);
        }
    }
}

// the unrolled FAST march could take more than 256 VGPRs (one wave per SIMD);
// two waves per SIMD with a few spills outside the march run faster
#if MPCF_FAST && !MPCF_F64
#define MPCF_XY_WAVES __attribute__((amdgpu_waves_per_eu(2, 2)))
#else
#define MPCF_XY_WAVES
#endif
// DT (a step's first stage, which needs no dt): one wave, of the tile that is
// least often full, also turns the maximum that the previous step folded into
// dt, for the z sweep that follows.  A launch of its own took 5 us with the gap
// before it (16^3 40.3 -> 37.8 us a step, 64^3 93.5 -> 92.7, bit-exact 64^3
// 201.4 -> 200.5; a step by itself 66 -> 52 us at 16^3)
template <bool FIRST, bool DT>
__global__ __launch_bounds__(256) MPCF_XY_WAVES
void k_sweep_xy(const Geom g, const StageArgs A, const int chunk, StepState* dt_st, const DtArgs d)
{
    // where a pipelined step's z sweep shares a SIMD with these waves, they
    // issue first (wave priority, not a queue priority): 512^3 19.92 ->
    // 19.85 ms a step; the z sweep's waves first instead was 7 % slower
    __builtin_amdgcn_s_setprio(2);
    const int gx = gridDim.x;
    const int t = xcd_order(blockIdx.x + blockIdx.y * gx, gx * gridDim.y);
    if constexpr (DT) {
        if (t == gx - 1 && threadIdx.y == 3 && threadIdx.x == 0) sos_finalize(dt_st, d, take_folded(dt_st));
    }
    sweep_xy_body<FIRST, kSyncXY>(g, A, chunk, (t % gx) * 4 + threadIdx.y, threadIdx.y, t / gx);
}

// ---------------------------------------------------------------------------
// ghost fill (BoundaryConditions.h:60-109 applied to the padded band).
// blockIdx.y = face = 2*dir + side.  kind: 0 absorbing, 1 reflecting, 2 halo
// (left as imported).
// ---------------------------------------------------------------------------
struct BCSet { int kind[6]; };

__device__ __forceinline__ void ghosts_body(const Geom& g, Real* __restrict__ u, const int64_t fs, const int* bc,
                                            const int bx, const int face)
{
    const int dir = face >> 1, side = face & 1;
    const int na = dir == 0 ? g.ny : g.nx;
    const int nb = dir == 2 ? g.ny : g.nz;
    const int t = bx * 256 + threadIdx.x;
    if (t >= na * nb) return;
    const int ta = t % na, tb = t / na;
    const int n = g.n(dir);
    const int kind = bc[face];
    if (kind == 2) return;
#pragma unroll
    for (int gl = 0; gl < 3; ++gl) {
        const int dst = side == 0 ? gl - 3 : n + gl;
        const int src = kind == 0 ? (side == 0 ? 0 : n - 1) : (side == 0 ? 2 - gl : n - 1 - gl);
        int ed, es;
        if (dir == 0)      { ed = g.idx(dst, ta, tb); es = g.idx(src, ta, tb); }
        else if (dir == 1) { ed = g.idx(ta, dst, tb); es = g.idx(ta, src, tb); }
        else               { ed = g.idx(ta, tb, dst); es = g.idx(ta, tb, src); }
#pragma unroll
        for (int q = 0; q < NVAR; ++q) {
            const Real v = u[q*fs + es];
            u[q*fs + ed] = (kind == 1 && q == 1 + dir) ? -v : v;
        }
    }
}

__global__ __launch_bounds__(256)
void k_ghosts(const Geom g, Real* __restrict__ u, const int64_t fs, const BCSet bc)
{
    ghosts_body(g, u, fs, bc.kind, blockIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------
// face halos of a decomposed domain (GPUlab::_copysend_halos,
// GPUlab.cpp:76-112, and the receive side that becomes the ghost band,
// GPUlab.cpp:636-641).  The buffer holds the 7 fields one after the other,
// each in the reference's ghost map order (Types.h:31-69): x faces
// [NZ][NY][3], y faces [NZ][3][NX], z faces [3][NY][NX], layer l = the l-th
// of the three cells in increasing index.  MODE 0 (export) reads the three
// boundary cells (0..2 on the low face, n-3..n-1 on the high face), MODE 1
// (import) writes the ghost band (-3..-1 low, n..n+2 high): a high face's
// export is the high neighbour's low-face import and vice versa.  MODE 2
// reads the ghost band back in the same order (the halo buffers GPUlab's
// load_ghosts leaves, GPUlab.cpp:622-644).
// ---------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256)
void k_halo(const Geom g, Real* __restrict__ u, const int64_t fs, const int face, Real* __restrict__ buf)
{
    constexpr bool IMPORT = MODE == 1;
    constexpr bool BAND = MODE != 0;   // the ghost band, not the boundary cells
    const int dir = face >> 1, side = face & 1;
    const int area = dir == 0 ? g.ny * g.nz : dir == 1 ? g.nx * g.nz : g.nx * g.ny;
    const int count = 3 * area;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= count) return;
    int x, y, z, layer;
    if (dir == 0)      { layer = t % 3;                 y = (t / 3) % g.ny;    z = t / (3 * g.ny); x = 0; }
    else if (dir == 1) { x = t % g.nx;                  layer = (t / g.nx) % 3; z = t / (3 * g.nx); y = 0; }
    else               { x = t % g.nx;                  y = (t / g.nx) % g.ny;  layer = t / area;   z = 0; }
    const int n = g.n(dir);
    const int cell = BAND ? (side == 0 ? layer - 3 : n + layer) : (side == 0 ? layer : n - 3 + layer);
    if (dir == 0) x = cell; else if (dir == 1) y = cell; else z = cell;
    const int e = g.idx(x, y, z);
#pragma unroll
    for (int q = 0; q < NVAR; ++q) {
        if (IMPORT) u[q * fs + e] = buf[(int64_t)q * count + t];
        else        buf[(int64_t)q * count + t] = u[q * fs + e];
    }
}

// ---------------------------------------------------------------------------
// max speed of sound and dt in one launch (GPUkernels.cu:1182-1222,
// MaxSpeedOfSound.cpp:18-55, LSRK3_IntegratorMPI.cpp:37-38): every block
// folds its maximum into the step state with an atomic max, then counts
// itself done; the last block reads the maximum, derives dt and dt/h, and puts
// the reduction target and the counter back to zero for the next step.
// ---------------------------------------------------------------------------

// the finished reduction's targets, put back to zero with its counter
__device__ __forceinline__ SosIn take_reduction(StepState* st)
{
    SosIn in;
    if constexpr (kSosD) in.sos = __longlong_as_double((long long)atomicExch(&st->sos_bits_d, 0ull));
    else                 in.sos = __uint_as_float(atomicExch(&st->sos_bits, 0u));
    in.bad = atomicExch(&st->bad_bits, 0u);
    atomicExch(&st->sos_count, 0u);
    return in;
}

// rows a wave of the reduction reads at a time
constexpr int kSosRows = 4;

// the reduction over the rows of a block, blocks b = 0..nb-1 of it in this
// launch; returns true in the one thread that finalized (thread (0, 0) of the
// last block to finish).  DENSE: the fields are in the host layout, cell
// (x, y, z) at x + nx*(y + ny*z), instead of the padded one
template <int CPU_FORM, bool DENSE = false>
__device__ __forceinline__ bool sos_body(const Geom& g, const Real* __restrict__ u, const int64_t fs, StepState* st,
                                         const int b, const int nb, SosT* wmax, int* wbad, const DtArgs& d)
{
    const int rows = g.ny * g.nz;
    SosT sos = 0.0f;
    bool bad = false;
    // four rows at a time, all their loads in flight; a row past the end
    // repeats the wave's first one
    const int step = nb * 4;
    for (int row = b * 4 + threadIdx.y; row < rows; row += kSosRows * step) {
        int e0[kSosRows];
#pragma unroll
        for (int k = 0; k < kSosRows; ++k) {
            const int r = row < rows - k * step ? row + k * step : row;
            e0[k] = DENSE ? r * g.nx : g.idx(0, r % g.ny, r / g.ny);
        }
        for (int x = threadIdx.x; x < g.nx; x += 64) {
            Real w[kSosRows][NU];
#pragma unroll
            for (int k = 0; k < kSosRows; ++k)
#pragma unroll
                for (int q = 0; q < (DENSE ? NVAR : NU); ++q) w[k][q] = u[q*fs + e0[k] + x];
#pragma unroll
            for (int k = 0; k < kSosRows; ++k) {
                bool cb;
                const SosT Ec = (kEPair && !DENSE) ? SosT(double(w[k][FE]) + double(w[k][NU - 1])) : SosT(w[k][FE]);
                sos = mmax(sos, sos_cell(CPU_FORM != 0, w[k][0], w[k][1], w[k][2], w[k][3], Ec, w[k][5], w[k][6], cb));
                bad = bad || cb;
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sos = mmax(sos, __shfl_xor(sos, off, 64));
    const int anybad = __ballot(bad) != 0;
    if (threadIdx.x == 0) { wmax[threadIdx.y] = sos; wbad[threadIdx.y] = anybad; }
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        const SosT m = mmax(mmax(wmax[0], wmax[1]), mmax(wmax[2], wmax[3]));
        // Nothing but these atomics passes between the blocks, so they are all
        // that the count has to follow: the values they return say that they
        // have been performed.  A device-scope fence here writes back and
        // invalidates the XCD's L2 once per block (see sos_blocks).
        unsigned seen = wbad[0] | wbad[1] | wbad[2] | wbad[3] ? atomicOr(&st->bad_bits, 1u) : 0u;
        if (kSosD) seen += (unsigned)atomicMax(&st->sos_bits_d, (unsigned long long)__double_as_longlong((double)m));
        else       seen += atomicMax(&st->sos_bits, __float_as_uint((float)m));
        asm volatile("" : : "v"(seen) : "memory");
        if (atomicAdd(&st->sos_count, 1u) == (unsigned)nb - 1u) {
            sos_finalize(st, d, take_reduction(st));
            return true;
        }
    }
    return false;
}

// dt from the maximum folded into the previous step's last z sweep
__global__ __launch_bounds__(64)
void k_sos_folded(StepState* st, const DtArgs d)
{
    if (threadIdx.x == 0) sos_finalize(st, d, take_folded(st));
}

template <int CPU_FORM>
__global__ __launch_bounds__(256)
void k_sos(const Geom g, const Real* __restrict__ u, const int64_t fs, StepState* st, const DtArgs d)
{
    __shared__ SosT wmax[4];
    __shared__ int wbad[4];
    sos_body<CPU_FORM>(g, u, fs, st, blockIdx.x, gridDim.x, wmax, wbad, d);
}

// the same reduction over fields in the host layout (cell x + nx*(y + ny*z),
// field q at u + q*fs), with st a caller-provided reduction state that must
// hold zeros in sos_bits[_d], bad_bits and sos_count; the finalizing thread
// copies the maximum (binary64), dt and the flag to the outputs (any may be
// null)
template <int CPU_FORM>
__global__ __launch_bounds__(256)
void k_sos_dense(const Geom g, const Real* __restrict__ u, const int64_t fs, StepState* st, const DtArgs d,
                 double* sos_out, double* dt_out, int* bad_out)
{
    __shared__ SosT wmax[4];
    __shared__ int wbad[4];
    if (sos_body<CPU_FORM, true>(g, u, fs, st, blockIdx.x, gridDim.x, wmax, wbad, d)) {
        if (sos_out) *sos_out = st->sos_d;
        if (dt_out) *dt_out = st->dt;
        if (bad_out) *bad_out = (int)st->bad;
    }
}

// ---------------------------------------------------------------------------
// Update_CUDA (GPUkernels.cu:1164-1170): u <- b*R + u, in place
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void k_update(const Geom g, Real* __restrict__ u, const Real* __restrict__ R, const int64_t fs, const Real b)
{
    const int rows = g.ny * g.nz;
    for (int row = blockIdx.x * 4 + threadIdx.y; row < rows; row += gridDim.x * 4) {
        const int e0 = g.idx(0, row % g.ny, row / g.ny);
        for (int x = threadIdx.x; x < g.nx; x += 64) {
            const int e = e0 + x;
#pragma unroll
            for (int q = 0; q < NVAR; ++q) {
                if (kEPair && q == FE) {
                    const double Ed = (double(u[FE*fs + e]) + double(u[FELO*fs + e])) + double(b) * double(R[FE*fs + e]);
                    const Real hi = Real(Ed);
                    u[FE*fs + e] = hi;
                    u[FELO*fs + e] = Real(Ed - double(hi));
                } else {
                    u[q*fs + e] = b*R[q*fs + e] + u[q*fs + e];
                }
            }
        }
    }
}

// E of an E-pair solution <-> a dense host field: to the device, hi = the
// value rounded to binary32 and lo = the remainder (zero for binary32 host
// values); from the device, hi + lo (binary64), rounded once for binary32
template <int TO_PADDED, typename Dense>
__global__ __launch_bounds__(256)
void k_pack_epair(const Geom g, Real* __restrict__ hi, Real* __restrict__ lo, Dense* __restrict__ dense)
{
    const int rows = g.ny * g.nz;
    for (int row = blockIdx.x * 4 + threadIdx.y; row < rows; row += gridDim.x * 4) {
        const int e0 = g.idx(0, row % g.ny, row / g.ny);
        const int64_t d0 = (int64_t)g.nx * row;
        for (int x = threadIdx.x; x < g.nx; x += 64) {
            if (TO_PADDED) {
                const double v = (double)dense[d0 + x];
                const Real h = Real(v);
                hi[e0 + x] = h;
                lo[e0 + x] = Real(v - double(h));
            } else {
                dense[d0 + x] = (Dense)(double(hi[e0 + x]) + double(lo[e0 + x]));
            }
        }
    }
}

// dense reference SoA (NX*NY*NZ per field, Types.h:31) <-> padded layout;
// the dense side may be binary32 or binary64 (converted on the way)
template <int TO_PADDED, typename Dense>
__global__ __launch_bounds__(256)
void k_pack(const Geom g, Real* __restrict__ pad, Dense* __restrict__ dense, const int64_t fs, const int nq)
{
    const int rows = g.ny * g.nz;
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    for (int row = blockIdx.x * 4 + threadIdx.y; row < rows; row += gridDim.x * 4) {
        const int y = row % g.ny, z = row / g.ny;
        const int e0 = g.idx(0, y, z);
        const int64_t d0 = (int64_t)g.nx * row;
        for (int x = threadIdx.x; x < g.nx; x += 64)
            for (int q = 0; q < nq; ++q) {
                if (TO_PADDED) pad[q*fs + e0 + x] = (Real)dense[q*n + d0 + x];
                else           dense[q*n + d0 + x] = (Dense)pad[q*fs + e0 + x];
            }
    }
}

// Streamers of the reference's dumps (Types.h:188-280) between the padded
// state and a dense channel-interleaved binary32 array [Z][Y][X][C]
// (HDF5Dumper_MPI.h:118-141):
//   KIND 0 myTensorialStreamer, 9 channels: rho, u, v, w, p, G, P, 0, 0 with
//          u = rho u / rho in the storage type and p = (E - 0.5 |rho u|^2 / rho
//          - P) / G evaluated in binary64 from the stored values (the
//          reference's 0.5 is a double literal)
//   KIND 1 mySaveStreamer, 7 channels: the conserved fields (also read back)
//   KIND 2 myScalarStreamer, 1 channel: rho
template <int KIND, int OUT>
__global__ __launch_bounds__(256)
void k_stream(const Geom g, Real* __restrict__ u, float* __restrict__ dense, const int64_t fs)
{
    constexpr int NC = KIND == 0 ? 9 : KIND == 1 ? 7 : 1;
    const int rows = g.ny * g.nz;
    for (int row = blockIdx.x * 4 + threadIdx.y; row < rows; row += gridDim.x * 4) {
        const int e0 = g.idx(0, row % g.ny, row / g.ny);
        const int64_t d0 = (int64_t)g.nx * row;
        for (int x = threadIdx.x; x < g.nx; x += 64) {
            const int e = e0 + x;
            float* o = dense + (d0 + x) * NC;
            if (!OUT) {
#pragma unroll
                for (int q = 0; q < NVAR; ++q) u[q*fs + e] = (Real)o[q];
                continue;
            }
            const Real r = u[e], ru = u[fs + e], rv = u[2*fs + e], rw = u[3*fs + e];
            const Real E = u[4*fs + e], G = u[5*fs + e], P = u[6*fs + e];
            if (KIND == 2) { o[0] = (float)r; continue; }
            if (KIND == 1) {
                o[0] = (float)r; o[1] = (float)ru; o[2] = (float)rv; o[3] = (float)rw;
                o[4] = (float)E; o[5] = (float)G; o[6] = (float)P;
                continue;
            }
            const Real ss = ru*ru + rv*rv + rw*rw;
            o[0] = (float)r;
            o[1] = (float)(ru / r);
            o[2] = (float)(rv / r);
            o[3] = (float)(rw / r);
            o[4] = (float)(((double)E - 0.5*(double)ss/(double)r - (double)P) / (double)G);
            o[5] = (float)G;
            o[6] = (float)P;
            o[7] = 0.0f;
            o[8] = 0.0f;
        }
    }
}

// device-function test hooks (the counterpart of GPU::TestKernel,
// GPUkernels.cu:1354-1382): run weno_cell / riemann on arrays
__global__ void k_test_weno(const int n, const Real* __restrict__ in5, Real* __restrict__ m, Real* __restrict__ p)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Real* a = in5 + 5*(int64_t)i;
    // as the sweeps do: quick quotients, and the IEEE ones where a lane's window needs them
    bool odd = false;
    Rec r = weno_cell<Real, kFast, !kFast>(a[0], a[1], a[2], a[3], a[4], &odd);
    if (any_lane(odd)) r = weno_cell<Real, kFast>(a[0], a[1], a[2], a[3], a[4]);
    m[i] = r.m; p[i] = r.p;
}

// st: n x 7 x 6 conserved values at stencil points i-3..i+2 of face i-1/2;
// out: n x 12 (7 fluxes, vel, Gm, Gp, Pm, Pp)
template <int D>
__global__ void k_test_face(const int n, const Real* __restrict__ st, Real* __restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Real* s = st + 42*(int64_t)i;
    Prim c[6];
    for (int k = 0; k < 6; ++k)
        c[k] = to_prim<Real, kFast, kP64>(s[0*6+k], s[1*6+k], s[2*6+k], s[3*6+k], s[4*6+k], s[5*6+k], s[6*6+k]);
    const CellRec left = reconstruct<Real, kFast>(c[0], c[1], c[2], c[3], c[4]);   // cell i-1
    const CellRec right = reconstruct<Real, kFast>(c[1], c[2], c[3], c[4], c[5]);  // cell i
    const FaceFlux F = riemann<D, Real, kFast>(left.m, right.p);
    Real* o = out + 12*(int64_t)i;
    for (int q = 0; q < NVAR; ++q) o[q] = F.f[q];
    o[7] = F.vel; o[8] = left.m.G; o[9] = right.p.G; o[10] = left.m.P; o[11] = right.p.P;
}

// st: n rows x 7 fields x 68 cells, conserved; row i is what a wave of the x+y
// sweep holds in x (its 64 lanes' cells and two beside them on either side).
// again[i]: bit 0, the wave evaluated its windows, bit 1, its faces a second
// time with the IEEE quotients
__global__ void k_test_rows(const Real* __restrict__ st, int* __restrict__ again)
{
    const int lane = threadIdx.x;
    const Real* const s = st + (int64_t)blockIdx.x * NVAR * 68;
    auto prim = [&](const int cell) {
        Real w[NU] = {};
#pragma unroll
        for (int f = 0; f < NVAR; ++f) w[f] = s[f * 68 + cell];
        return prim_of(w);
    };
    Halo4 halo[NVAR];
#pragma unroll
    for (int side = 0; side < 4; ++side) {
        const Prim p = prim(side < 2 ? side : 64 + side);
        const Real v[NVAR] = {p.r, p.u, p.v, p.w, p.p, p.G, p.P};
#pragma unroll
        for (int f = 0; f < NVAR; ++f) halo[f][side] = v[f];
    }
    bool windows = false, faces = false;
    const CellRec rx = reconstruct_lanes<false>(prim(2 + lane), halo, &windows);
    const Prim Lm = prim_from_left(rx.m);
    (void)riemann<0, Real, kFast, false, kXFaceLanes>(Lm, rx.p, &faces);
    if (lane == 0) again[blockIdx.x] = (windows ? 1 : 0) | (faces ? 2 : 0);
}

#if !MPCF_FAST && !MPCF_F64
// the quick operations by themselves (mpcf_scheme.h): OP 0 rcp_rn(b), 1
// div_rn(a, b), 2 sqrt_rn(a), all binary32, 3 rcp_rn(b) in binary64
template <int OP, typename V>
__global__ void k_test_quotient(const int n, const V* __restrict__ a, const V* __restrict__ b, V* __restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if constexpr (OP == 1)      out[i] = div_rn(a[i], b[i], rcp_rn(b[i]));
    else if constexpr (OP == 2) out[i] = sqrt_rn(a[i]);
    else                        out[i] = rcp_rn(b[i]);
}
#endif

// ---------------------------------------------------------------------------
// batched ensemble: one launch per kernel kind advances every live case.  A
// flat block index is mapped to (case, local block) by a binary search over
// the per-case prefix offsets; the local block runs the same body as the
// single-case kernel, so every case gets exactly the arithmetic it gets
// alone.  The cases' current-buffer indices live on the device and are
// flipped after each stage, so a whole step can be captured in a graph.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int find_case(const int* __restrict__ off, const int n, const int b)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ StageArgs case_args(const CaseDesc& C, const int cur, const Real a, const Real b)
{
    StageArgs A;
    A.sos_next = nullptr; A.sos_cpu = 0;
    A.bcmask = 0;
    for (int f = 0; f < 6; ++f) A.bcmask |= (C.bc[f] == 1) << f;
    A.z0 = 0; A.z1 = C.g.nz;
    A.u = (const Real*)C.u[cur]; A.R = (Real*)C.R; A.acc = (Real*)C.acc; A.uo = (Real*)C.u[1 - cur];
    A.fs = C.g.fstride;
    A.a = a; A.b = b; A.dtinvh = Real(0.0f); A.st = C.st;
    return A;
}

template <int CPU_FORM>
__global__ __launch_bounds__(256)
void kb_sos(const BatchDev B, const double cfl, const double dt_max)
{
    __shared__ SosT wmax[4];
    __shared__ int wbad[4];
    const int c = find_case(B.off_sos, B.n, blockIdx.x);
    const CaseDesc& C = B.cases[c];
    const DtArgs d{1, cfl, C.h, dt_max};
    const int local = blockIdx.x - B.off_sos[c];
    if (C.st->folded) {
        // the previous step's last z sweep folded this state's maximum: only
        // dt remains, done by the case's first block
        if (local == 0 && threadIdx.x == 0 && threadIdx.y == 0) sos_finalize(C.st, d, take_folded(C.st));
        return;
    }
    sos_body<CPU_FORM>(C.g, (const Real*)C.u[B.cur[c]], C.g.fstride, C.st, local, C.nb_sos, wmax, wbad, d);
}

template <bool FIRST>
__global__ __launch_bounds__(256) MPCF_XY_WAVES
void kb_sweep_xy(const BatchDev B, const Real a, const Real b)
{
    // round-robin over the XCDs as dispatched: the tiles of different cases
    // differ in cost, and an even mix per XCD balances them (contiguous runs
    // per XCD, as in k_sweep_xy, were slower here)
    const int c = find_case(B.off_xy, B.n, blockIdx.x);
    const CaseDesc& C = B.cases[c];
    const int local = blockIdx.x - B.off_xy[c];
    const StageArgs A = case_args(C, B.cur[c], a, b);
    sweep_xy_body<FIRST, kSyncXY>(C.g, A, C.chunk_xy, (local % C.nbx_xy) * 4 + threadIdx.y, threadIdx.y, local / C.nbx_xy);
}

// the z sweep finishes the stage; the last block of each case to finish
// flips the case's current-buffer index (every block has read it before it
// counts itself: no fence is needed, and a device-scope fence here would
// write back and invalidate the XCD's L2 once per block).
// fold != 0 (a step's last stage): the sweep also folds the maximum speed of
// sound of the state it writes, for the next step's kb_sos.  MODE_STAGE_NOR:
// R is not stored (a caller that never reads R after a step)
template <int MODE>
__global__ __launch_bounds__(256)
void kb_sweep_z(const BatchDev B, const Real a, const Real b, const int fold, const int cpu_form)
{
    const int c = find_case(B.off_z, B.n, blockIdx.x);
    const CaseDesc& C = B.cases[c];
    const int local = blockIdx.x - B.off_z[c];
    StageArgs A = case_args(C, B.cur[c], a, b);
    if (fold) { A.sos_next = C.st; A.sos_cpu = cpu_form; }
    sweep_yz_body<2, MODE>(C.g, A, C.chunk_z, C.width_z, (local % C.nbx_z) * 256 + threadIdx.x, local / C.nbx_z);
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned nblk = (unsigned)(B.off_z[c + 1] - B.off_z[c]);
        if (atomicAdd(&C.st->z_count, 1u) == nblk - 1u) {
            atomicExch(&B.cur[c], 1 - B.cur[c]);
            if (fold) atomicExch(&C.st->folded, 1);
            atomicExch(&C.st->z_count, 0u);
        }
    }
}

// ---------------------------------------------------------------------------
// persistent batched stage: two launches per RK stage for every case, one for
// the x+y items of all cases, then one for their z items (a z item reads the
// R and accumulators the x+y items of its case wrote; the launch boundary
// orders them -- inside one launch that order would take a device-scope
// release and acquire per item, an L2 write-back and invalidation of the XCD,
// which measured 1.7x slower than flat launches).  Each workgroup pulls items
// from a device queue (an atomic counter) until it is empty; an item is one
// workgroup's share of one case's x+y sweep (W = blockDim.x / 64 consecutive
// tiles of XY_TILE positions over one y-chunk) or z sweep (blockDim.x columns over one
// z-chunk), running the single-case bodies, so every case gets exactly the
// arithmetic it gets alone.  The queue holds the items of the larger cases
// first, so the small ones fill the launch's tail.
// ---------------------------------------------------------------------------
// Thread 0 alone takes an item or counts a finished one; those steps are
// calls of their own, bracketed by barriers.  Written inline, the compiler
// may restructure the item loop around such a branch so that thread 0 leaves
// the loop body on its own while the other threads of its wave go round
// again, which breaks the barriers and lets those threads run an item twice;
// a call is convergent, so the loop body the compiler sees has no branch that
// splits the workgroup.
__device__ __attribute__((noinline)) unsigned take_item(PCtl* ctl)
{
    __shared__ unsigned s_item;
    if (threadIdx.x == 0) s_item = atomicAdd(&ctl->head, 1u);
    __syncthreads();
    const unsigned i = s_item;
    __syncthreads();                              // read everywhere before the next take
    return i;
}

// a z item is finished; the case's last one flips its current-buffer index
// (every z item of the case has read it by then: each reads it before it
// counts itself) and clears the count for the next stage
__device__ __attribute__((noinline)) void count_z(unsigned* done, const unsigned items_z, int* cur_c,
                                                  const int cur, int* folded, const int fold)
{
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(done, 1u) == items_z - 1u) {
        atomicExch(cur_c, 1 - cur);
        if (fold) atomicExch(folded, 1);
        atomicExch(done, 0u);
    }
}

// PHASE 0: the x+y items (queue items [0, seg[nxy].first)); PHASE 1: the z
// items (the rest).  Two kernels, so that each holds only its own sweep's
// registers
template <int PHASE>
__device__ __forceinline__ void kp_stage_body(const PersistDev& P, const Real a, const Real b, const int fold,
                                              const int cpu_form)
{
    constexpr int phase = PHASE;
    const int W = (int)(blockDim.x >> 6);        // waves per item
    const int wib = (int)(threadIdx.x >> 6);     // this wave's place in the item
    const int s0 = phase == 0 ? 0 : P.nxy, s1 = phase == 0 ? P.nxy : P.nseg;
    const unsigned first = P.seg[s0].first, end = P.seg[s1].first;
    for (;;) {
        // the same value in every thread: readfirstlane only makes it scalar
        const unsigned i = first + (unsigned)__builtin_amdgcn_readfirstlane((int)take_item(P.ctl));
        if (i >= end) break;
        int lo = s0, hi = s1 - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (P.seg[mid].first <= i) lo = mid; else hi = mid - 1;
        }
        const PSeg S = P.seg[lo];
        const CaseDesc& C = P.cases[S.c];
        const int j = (int)(i - S.first);
        const int cur = P.cur[S.c];
        StageArgs A = case_args(C, cur, a, b);
        if constexpr (phase == 0) {
            (void)fold; (void)cpu_form;
            sweep_xy_body(C.g, A, C.chunk_xy, (j % C.wxy) * W + wib, wib, j / C.wxy);
        } else {
            if (fold) { A.sos_next = C.st; A.sos_cpu = cpu_form; }
            sweep_yz_body<2, MODE_STAGE, true>(C.g, A, C.chunk_z, C.width_z, (j % C.wz) * (int)blockDim.x + (int)threadIdx.x, j / C.wz);
            count_z(P.done + S.c, C.items_z, &P.cur[S.c], cur, &C.st->folded, fold);
        }
    }
    // the last workgroup out puts the queue back for the next launch
    if (threadIdx.x == 0 && atomicAdd(&P.ctl->exited, 1u) == P.nblocks - 1u) {
        atomicExch(&P.ctl->head, 0u);
        atomicExch(&P.ctl->exited, 0u);
    }
}

__global__ __launch_bounds__(256) MPCF_XY_WAVES
void kp_stage_xy(const PersistDev P, const Real a, const Real b)
{
    kp_stage_body<0>(P, a, b, 0, 0);
}

__global__ __launch_bounds__(256)
void kp_stage_z(const PersistDev P, const Real a, const Real b, const int fold, const int cpu_form)
{
    kp_stage_body<1>(P, a, b, fold, cpu_form);
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
// march length of a launch that shares the chip: a slab of a pipelined step
// (the other stream's sweep fills its tail) and the split x / y sweeps
static int pick_chunk(const int nd, const int64_t columns)
{
    // enough marching threads for ~4 waves per SIMD (256 CUs x 4 SIMDs)
    const int64_t target_threads = 256LL * 4 * 4 * 64;
    int nchunks = (int)((target_threads + columns - 1) / columns);
    if (nchunks < 1) nchunks = 1;
    int chunk = (nd + nchunks - 1) / nchunks;
    if (chunk < 16) chunk = nd < 16 ? nd : 16;
    return chunk;
}

// March length of a fused x+y (dir 3) or z (dir 2) sweep launch that runs
// alone: the one with the least modelled time.  `blocks` four-wave workgroups
// cover the marching columns; cut into chunks of L rows, the busiest of the
// 256 CUs runs n = ceil(blocks * chunks / 256) of them, two at a time, and a
// chunk costs its rows plus `ov` rows of start-up (window fill and the rows
// whose flux is recomputed at the chunk's first face; for the z sweep also
// the five extra rows of u it reads).  `lat` rows pass once per launch before
// the first row is done.  A workgroup alone on its CU takes 1.2 times its
// share.  Measured on MI355X over L = 1..64 for blocks from 16^3 to 192^3, the
// model is within 10 % in every arithmetic build.  Chunks of at least 16 rows
// (four waves per SIMD and more) left small blocks to a few dozen waves
// marching 16 rows each: FAST x+y / z sweep 42 / 27 us at 32^3, 45 / 29 at
// 64^3 and 100 / 54 at 128^3, against 9 / 10, 22 / 17 and 96 / 53 here.
// lone: one wave holds the x+y sweep's columns.  The workgroup's other three waves
// leave at once, and three such workgroups run on a CU side by side (one in
// the binary64 build, whose waves take a whole SIMD): us for (5, ny, 5) counted as
// above / so, FAST 300 10.8 / 9.5, 3000 22.8 / 18.9, 9000 48.6 / 38.3, 20000
// 97.3 / 75.7; bit-exact 22.5 / 17.2, 48.1 / 36.7, 117 / 82, 242 / 169.
static int whole_march(const int nd, const int64_t blocks, const int dir, const bool lone = false)
{
    const double lat = dir == 3 ? 3.0 : 1.0;
    const double ov = dir == 3 ? 1.0 : kFast ? 3.0 : 2.0;
    int best = nd;
    double least = 0.0;
    for (int L = nd; L >= 1;) {
        const int nch = (nd + L - 1) / L;
        const int64_t n = lone ? (nch + 767) / 768 : (blocks * nch + 255) / 256;
        if (L < nd && n > 64) break;     // the tail no longer matters
        const double t = lat + (n == 1 && !lone ? 1.2 : (double)n) * (L + ov);
        if (L == nd || t < least) { least = t; best = L; }
        const int next = (nd + nch) / (nch + 1);   // the longest march with more chunks
        L = next < L ? next : L - 1;
    }
    return best;
}

// March length of a FAST slab's fused x+y (dir 3) or z (dir 2) sweep where the
// slab's launch is only a few workgroups a CU and runs beside the other sweep's
// (SweepParams::fit: queued steps of blocks below 2^25 cells): the least rows on
// the busiest of the 256 CUs, as in whole_march, with at most five workgroups a
// CU -- longer marches than pick_chunk's have fewer start-up rows, and counts
// just over a multiple of 256 cost a round.  The x+y sweep keeps two workgroups
// a CU (a lone wave's instructions do not pair: slabs of (216, 189, 62) with one
// takes 1.6 times as long a step).  Three slabs, FAST, ms a step, pick_chunk / this:
// (216,189,186) 1.20 / 1.15, (227,270,156) 1.56 / 1.50, 240^3 2.15 / 1.99,
// (221,248,290) 2.59 / 2.30, (270,235,266) 2.57 / 2.53, 256^3 2.56 / 2.32,
// 320^3 4.53 / 4.49.  Larger blocks keep pick_chunk: 384^3 7.77 / 7.80, 448^3
// 12.24 / 12.40; so do other slab counts, which it suits less evenly (four slabs,
// 256^3 2.50 / 2.27, (270,235,266) 2.64 / 2.87).
static int slab_march(const int nd, const int64_t blocks, const int dir)
{
    const double ov = dir == 3 ? 1.0 : 3.0;
    const int nmin = dir == 3 ? 2 : 1, nmax = 5;
    int best = nd;
    double least = 0.0;
    for (int L = nd; L >= 8;) {
        const int nch = (nd + L - 1) / L;
        const int64_t n = (blocks * nch + 255) / 256;
        if (n > nmax && least > 0.0) break;
        const double t = (double)n * (L + ov);
        // fewer than nmin only with the longest marches: a slab of two million
        // cells or more always reaches it
        if (n >= nmin && (least == 0.0 || t < least)) { least = t; best = L; }
        const int next = (nd + nch) / (nch + 1);   // the longest march with more chunks
        L = next < L ? next : L - 1;
    }
    return best;
}
// columns of a z sweep's rows of nx, in a launch (or a batch's launches) over
// `cells` cells.  The FAST builds' z sweep runs at the memory's rate: rows
// rounded up to 32 columns give every half wave one whole 128-byte line a
// field, where the packed columns of an odd nx read and write each line in
// parts, from two waves.  Smaller blocks stay in the L2s and only feel the idle
// lanes, and so do rows of up to 48 columns, most of whose lanes may idle, until
// the padded rows fill some 8 M elements a field; of those, rows of whole
// 64-byte halves of a line never gain.  Time of the rounded against the packed z
// sweep: below 2^19 cells 0.99-1.20; nx 56-161, 0.6 to 4 M cells, 0.75-1.07
// (161^3 126 / 103 us, 193^3 234 / 185); nx 5-44 below 15 2^19 padded elements
// 0.95-1.18, above 0.81-1.01; nx 16 and 48 0.95-1.21.  Alike in the P64 and
// E-pair builds.  The bit-exact and binary64 sweeps are bound by their
// arithmetic and lose what the idle lanes cost (193^3 335 / 373)
int z_width(const int nx, const long long cells)
{
    if (!kFast || cells < 1LL << 19) return nx;
    const long long padded = cells / nx * ((nx + XOFF + GHOST + 31) / 32 * 32);
    if (nx <= 48 && (nx % 16 == 0 || padded < 15LL << 19)) return nx;
    return (nx + 31) / 32 * 32;
}
static int z_width(const Geom& g) { return z_width(g.nx, (long long)g.nx * g.ny * g.nz); }

// four-wave workgroups of one chunk of the x+y sweep over nz planes / of the
// z sweep's flattened (x, y) columns, `width` of them a row
static int xy_waves(const Geom& g, const int nz) { return ((g.nx + 6) * nz + XY_TILE - 1) / XY_TILE; }
static int xy_blocks(const Geom& g, const int nz) { return (xy_waves(g, nz) + 3) / 4; }
static bool xy_lone(const Geom& g, const int nz) { return !MPCF_F64 && xy_waves(g, nz) == 1; }
static int z_blocks(const Geom& g, const int width) { return (width * g.ny + 255) / 256; }

static int rows_grid(const Geom& g)
{
    const int rows = g.ny * g.nz;
    int blocks = (rows + 3) / 4;
    return blocks < 8192 ? blocks : 8192;
}

void launch_ghosts(const Geom& g, void* uv, const int bc[6], hipStream_t s)
{
    BCSet b;
    for (int i = 0; i < 6; ++i) b.kind[i] = bc[i];
    int tmax = g.ny * g.nz;
    if (g.nx * g.nz > tmax) tmax = g.nx * g.nz;
    if (g.nx * g.ny > tmax) tmax = g.nx * g.ny;
    hipLaunchKernelGGL(k_ghosts, dim3((tmax + 255) / 256, 6), dim3(256), 0, s, g, (Real*)uv, g.fstride, b);
}

// mode 0: export the boundary cells, 1: import into the ghost band, 2: read the ghost band
void launch_halo(const Geom& g, void* uv, void* buf, const int face, const int mode, hipStream_t s)
{
    const int dir = face >> 1;
    const int count = 3 * (dir == 0 ? g.ny * g.nz : dir == 1 ? g.nx * g.nz : g.nx * g.ny);
    const dim3 grid((count + 255) / 256);
    if (mode == 1)
        hipLaunchKernelGGL(k_halo<1>, grid, dim3(256), 0, s, g, (Real*)uv, g.fstride, face, (Real*)buf);
    else if (mode == 2)
        hipLaunchKernelGGL(k_halo<2>, grid, dim3(256), 0, s, g, (Real*)uv, g.fstride, face, (Real*)buf);
    else
        hipLaunchKernelGGL(k_halo<0>, grid, dim3(256), 0, s, g, (Real*)uv, g.fstride, face, (Real*)buf);
}

void launch_sos(const Geom& g, const void* uv, StepState* st, const int cpu_form, const int with_dt, const double cfl,
                const double h, const double dt_max, hipStream_t s)
{
    const Real* u = (const Real*)uv;
    const int nb = mpcf::sos_blocks(g);
    const DtArgs d{with_dt, cfl, h, dt_max};
    if (cpu_form) hipLaunchKernelGGL(k_sos<1>, dim3(nb), dim3(64, 4), 0, s, g, u, g.fstride, st, d);
    else          hipLaunchKernelGGL(k_sos<0>, dim3(nb), dim3(64, 4), 0, s, g, u, g.fstride, st, d);
}

void launch_sos_dense(const Geom& g, const void* uv, const int64_t fs, StepState* st, const int cpu_form,
                      const double cfl, const double h, const double dt_max, double* sos_out, double* dt_out,
                      int* bad_out, hipStream_t s)
{
    const Real* u = (const Real*)uv;
    const int nb = mpcf::sos_blocks(g);
    const DtArgs d{1, cfl, h, dt_max};
    if (cpu_form)
        hipLaunchKernelGGL(k_sos_dense<1>, dim3(nb), dim3(64, 4), 0, s, g, u, fs, st, d, sos_out, dt_out, bad_out);
    else
        hipLaunchKernelGGL(k_sos_dense<0>, dim3(nb), dim3(64, 4), 0, s, g, u, fs, st, d, sos_out, dt_out, bad_out);
}

void launch_sos_folded(StepState* st, const double cfl, const double h, const double dt_max, hipStream_t s)
{
    const DtArgs d{1, cfl, h, dt_max};
    hipLaunchKernelGGL(k_sos_folded, dim3(1), dim3(64), 0, s, st, d);
}

// one direction sweep.  dir 0 (x) assigns the accumulators, dir 1 (y)
// accumulates, dir 3 does x and y fused (assigns), dir 2 (z) finishes the
// register update (stage == 0: R only, as Convection; stage == 1: R and the
// new solution, as process_all; stage == 2: the new solution only, R not
// stored).
void launch_sweep(const Geom& g, const int dir, const SweepParams& p, const int stage, hipStream_t s)
{
    StageArgs A;
    A.u = (const Real*)p.u; A.R = (Real*)p.R; A.acc = (Real*)p.acc; A.uo = (Real*)p.uo; A.fs = g.fstride;
    A.a = (Real)p.a; A.b = (Real)p.b; A.dtinvh = (Real)p.dtinvh; A.st = p.st;
    A.bcmask = p.bcmask;
    A.sos_next = p.sos_next; A.sos_cpu = p.sos_cpu;
    A.z0 = p.z0; A.z1 = p.z1 < 0 ? g.nz : p.z1;
    const int nzr = A.z1 - A.z0;
    const bool whole = A.z0 == 0 && A.z1 == g.nz;   // not a slab
    if (dir == 3) {
        const int nb = xy_blocks(g, nzr);
        const int chunk = whole ? whole_march(g.ny, nb, 3, xy_lone(g, nzr)) : p.fit ? slab_march(g.ny, nb, 3)
                                                                            : pick_chunk(g.ny, (int64_t)g.nx * nzr);
        const dim3 grid(nb, (g.ny + chunk - 1) / chunk);
        // a first stage of a folded build does not read R
        const bool first = kFold && A.a == Real(0.0f);
        const DtArgs d{1, p.cfl, p.h, p.dt_max};
        const dim3 block(64, 4);
        if (p.dt_st) hipLaunchKernelGGL((k_sweep_xy<kFold, true>), grid, block, 0, s, g, A, chunk, p.dt_st, d);
        else if (first) hipLaunchKernelGGL((k_sweep_xy<kFold, false>), grid, block, 0, s, g, A, chunk, p.dt_st, d);
        else hipLaunchKernelGGL((k_sweep_xy<false, false>), grid, block, 0, s, g, A, chunk, p.dt_st, d);
    } else if (dir == 0) {
        const int npen = g.ny * nzr;
        const int chunk = pick_chunk(g.nx, npen);
        dim3 grid((npen + 63) / 64, (g.nx + chunk - 1) / chunk);
        hipLaunchKernelGGL(k_sweep_x, grid, dim3(64), 0, s, g, A, chunk);
    } else if (dir == 1) {
        const int chunk = pick_chunk(g.ny, (int64_t)g.nx * nzr);
        dim3 grid((g.nx * nzr + 255) / 256, (g.ny + chunk - 1) / chunk);
        hipLaunchKernelGGL((k_sweep_yz<1, MODE_ACC>), grid, dim3(256), 0, s, g, A, chunk, g.nx);
    } else {
        const int width = z_width(g);
        const int nb = z_blocks(g, width);
        const int march = whole ? whole_march(nzr, nb, 2) : p.fit ? slab_march(nzr, nb, 2)
                                                                           : pick_chunk(nzr, (int64_t)g.nx * g.ny);
        const int chunk = std::min(z_march_limit(g), march);
        const dim3 grid(nb, (nzr + chunk - 1) / chunk);
        if (stage == 2)      hipLaunchKernelGGL((k_sweep_yz<2, MODE_STAGE_NOR>), grid, dim3(256), 0, s, g, A, chunk, width);
        else if (stage == 1) hipLaunchKernelGGL((k_sweep_yz<2, MODE_STAGE>), grid, dim3(256), 0, s, g, A, chunk, width);
        else                 hipLaunchKernelGGL((k_sweep_yz<2, MODE_CONV>), grid, dim3(256), 0, s, g, A, chunk, width);
    }
}

void launch_update(const Geom& g, void* u, const void* R, const double b, hipStream_t s)
{
    hipLaunchKernelGGL(k_update, dim3(rows_grid(g)), dim3(64, 4), 0, s, g, (Real*)u, (const Real*)R, g.fstride, (Real)b);
}

void launch_pack(const Geom& g, void* pad, void* dense, const int to_padded, const int nq, const int dense_f64,
                 hipStream_t s)
{
    Real* P = (Real*)pad;
    const dim3 grid(rows_grid(g)), block(64, 4);
    if (dense_f64) {
        if (to_padded) hipLaunchKernelGGL((k_pack<1, double>), grid, block, 0, s, g, P, (double*)dense, g.fstride, nq);
        else           hipLaunchKernelGGL((k_pack<0, double>), grid, block, 0, s, g, P, (double*)dense, g.fstride, nq);
    } else {
        if (to_padded) hipLaunchKernelGGL((k_pack<1, float>), grid, block, 0, s, g, P, (float*)dense, g.fstride, nq);
        else           hipLaunchKernelGGL((k_pack<0, float>), grid, block, 0, s, g, P, (float*)dense, g.fstride, nq);
    }
}

void launch_pack_epair(const Geom& g, void* hi, void* lo, void* dense, const int to_padded, const int dense_f64,
                       hipStream_t s)
{
    Real* H = (Real*)hi;
    Real* L = (Real*)lo;
    const dim3 grid(rows_grid(g)), block(64, 4);
    if (dense_f64) {
        if (to_padded) hipLaunchKernelGGL((k_pack_epair<1, double>), grid, block, 0, s, g, H, L, (double*)dense);
        else           hipLaunchKernelGGL((k_pack_epair<0, double>), grid, block, 0, s, g, H, L, (double*)dense);
    } else {
        if (to_padded) hipLaunchKernelGGL((k_pack_epair<1, float>), grid, block, 0, s, g, H, L, (float*)dense);
        else           hipLaunchKernelGGL((k_pack_epair<0, float>), grid, block, 0, s, g, H, L, (float*)dense);
    }
}

void launch_stream(const Geom& g, void* pad, float* dense, const int kind, const int out, hipStream_t s)
{
    Real* P = (Real*)pad;
    const dim3 grid(rows_grid(g)), block(64, 4);
    if (!out)           hipLaunchKernelGGL((k_stream<1, 0>), grid, block, 0, s, g, P, dense, g.fstride);
    else if (kind == 0) hipLaunchKernelGGL((k_stream<0, 1>), grid, block, 0, s, g, P, dense, g.fstride);
    else if (kind == 1) hipLaunchKernelGGL((k_stream<1, 1>), grid, block, 0, s, g, P, dense, g.fstride);
    else                hipLaunchKernelGGL((k_stream<2, 1>), grid, block, 0, s, g, P, dense, g.fstride);
}

void launch_test_weno(const int n, const void* in5v, void* mv, void* pv, hipStream_t s)
{
    const Real* in5 = (const Real*)in5v;
    Real* m = (Real*)mv;
    Real* p = (Real*)pv;
    hipLaunchKernelGGL(k_test_weno, dim3((n + 255) / 256), dim3(256), 0, s, n, in5, m, p);
}

#if !MPCF_FAST && !MPCF_F64
void launch_test_quotient(const int op, const int n, const void* a, const void* b, void* out, hipStream_t s)
{
    const dim3 grid((n + 255) / 256), block(256);
    const float *af = (const float*)a, *bf = (const float*)b;
    if (op == 0)      hipLaunchKernelGGL((k_test_quotient<0, float>), grid, block, 0, s, n, af, bf, (float*)out);
    else if (op == 1) hipLaunchKernelGGL((k_test_quotient<1, float>), grid, block, 0, s, n, af, bf, (float*)out);
    else if (op == 2) hipLaunchKernelGGL((k_test_quotient<2, float>), grid, block, 0, s, n, af, bf, (float*)out);
    else hipLaunchKernelGGL((k_test_quotient<3, double>), grid, block, 0, s, n, (const double*)a, (const double*)b, (double*)out);
}
#endif

void launch_test_rows(const int n, const void* st, int* again, hipStream_t s)
{
    hipLaunchKernelGGL(k_test_rows, dim3(n), dim3(64), 0, s, (const Real*)st, again);
}

void launch_test_face(const int n, const int dir, const void* stv, void* outv, hipStream_t s)
{
    const Real* st = (const Real*)stv;
    Real* out = (Real*)outv;
    dim3 grid((n + 127) / 128), block(128);
    if (dir == 0)      hipLaunchKernelGGL(k_test_face<0>, grid, block, 0, s, n, st, out);
    else if (dir == 1) hipLaunchKernelGGL(k_test_face<1>, grid, block, 0, s, n, st, out);
    else               hipLaunchKernelGGL(k_test_face<2>, grid, block, 0, s, n, st, out);
}

// the march length of a whole-block x+y (dir 3) or z (dir 2) launch that runs alone
int whole_chunk(const Geom& g, const int dir)
{
    return dir == 3 ? whole_march(g.ny, xy_blocks(g, g.nz), 3, xy_lone(g, g.nz))
                    : whole_march(g.nz, z_blocks(g, z_width(g)), 2);
}

// positions a wave of the fused x+y sweep stores
int xy_tile() { return XY_TILE; }

// grid of the fused x+y sweep: dims[0] blocks of four waves over the padded
// rows of all planes, dims[2] y-chunks (dims[1] = 1)
void xy_grid(const Geom& g, const int chunk, int dims[3])
{
    dims[0] = xy_blocks(g, g.nz); dims[1] = 1; dims[2] = (g.ny + chunk - 1) / chunk;
}

// grid of the z sweep: dims[0] blocks of 256 flattened (x, y) columns, `width` a
// row, dims[2] z-chunks
void z_grid(const Geom& g, const int width, const int chunk, int dims[3])
{
    dims[0] = z_blocks(g, width); dims[1] = 1; dims[2] = (g.nz + chunk - 1) / chunk;
}

void batch_sos(const BatchDev& B, const int blocks, const int cpu_form, const double cfl, const double dt_max,
               hipStream_t s)
{
    if (cpu_form) hipLaunchKernelGGL(kb_sos<1>, dim3(blocks), dim3(64, 4), 0, s, B, cfl, dt_max);
    else          hipLaunchKernelGGL(kb_sos<0>, dim3(blocks), dim3(64, 4), 0, s, B, cfl, dt_max);
}

void batch_xy(const BatchDev& B, const int blocks, const double a, const double b, hipStream_t s)
{
    if (kFold && a == 0.0) hipLaunchKernelGGL(kb_sweep_xy<true>, dim3(blocks), dim3(64, 4), 0, s, B, (Real)a, (Real)b);
    else                   hipLaunchKernelGGL(kb_sweep_xy<false>, dim3(blocks), dim3(64, 4), 0, s, B, (Real)a, (Real)b);
}

// storeR == 0: R is not stored (MODE_STAGE_NOR)
void batch_z(const BatchDev& B, const int blocks, const double a, const double b, const int fold, const int cpu_form,
             const int storeR, hipStream_t s)
{
    if (storeR) hipLaunchKernelGGL(kb_sweep_z<MODE_STAGE>, dim3(blocks), dim3(256), 0, s, B, (Real)a, (Real)b, fold, cpu_form);
    else        hipLaunchKernelGGL(kb_sweep_z<MODE_STAGE_NOR>, dim3(blocks), dim3(256), 0, s, B, (Real)a, (Real)b, fold, cpu_form);
}
// the two launches of one stage; blocks[0] workgroups for the x+y items,
// blocks[1] for the z items
void persist_stage(const PersistDev& P, const int blocks[2], const int threads, const double a, const double b,
                   const int fold, const int cpu_form, hipStream_t s)
{
    PersistDev Q = P;
    Q.nblocks = (unsigned)blocks[0];
    hipLaunchKernelGGL(kp_stage_xy, dim3(blocks[0]), dim3(threads), 0, s, Q, (Real)a, (Real)b);
    Q.nblocks = (unsigned)blocks[1];
    hipLaunchKernelGGL(kp_stage_z, dim3(blocks[1]), dim3(threads), 0, s, Q, (Real)a, (Real)b, fold, cpu_form);
}
// resident workgroups of `threads` threads per CU of the x+y (phase 0) or z
// (phase 1) launch
int persist_occupancy(const int threads, const int phase)
{
    int n = 0;
    const hipError_t e = phase == 0 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kp_stage_xy, threads, 0)
                                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kp_stage_z, threads, 0);
    return e == hipSuccess ? n : 0;
}

} // namespace MPCF_NS
} // namespace mpcf
