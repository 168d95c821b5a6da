// Element-local volume right-hand side of the hydrostatic primitive
// equations on gfx950 (MI355X), sum-factorised.
//
// Replaces PrimitiveEquationsSolver::compute_rhs
// (src/physics/primitive_equations.cpp:428-442) and everything below it:
// update_derived (:12-29), compute_momentum_rhs (:154-199), compute_tracer_rhs
// (:201-227), compute_eta_rhs (:229-273), with the reference-coordinate
// derivatives of DG3DElementOperator::{gradient,divergence}_reference
// (src/dg/operators_3d.cpp:58-79) applied by sum factorisation instead of
// dense Kronecker mat-vecs (D_xi = D (x) I (x) I, src/dg/basis_hexahedron.cpp:321-357).
// Second derivatives are applied as D (D u) in FP64, two line contractions
// as the reference applies its Kronecker gradient twice (only D then sits in
// SGPRs), and as (D D) u with D^2 formed once on the host in FP32.
//
// Work decomposition.  A workgroup owns EPB elements per batch; every element
// is handled by n^2 threads, each owning one grid line of n nodes.  Line
// ownership rotates xi -> eta -> zeta -> xi through LDS twice per batch, once
// for the momentum terms and once for the tracers, so that seven staged
// values per node suffice (phases P1 .. P4b at the kernel).  Each value
// crosses LDS once per direction instead of once per derivative tap.
// Workgroups are persistent: while a batch is computed, the state lines of
// the workgroup's next batch are already being loaded into registers, so HBM
// traffic overlaps the FP64 arithmetic.  A workgroup holds 128, 256 or 512
// grid lines (at N = 4: 5, 10 or 20 elements per batch, 8 waves per CU in
// every case, as registers and LDS allow); wider workgroups read longer
// contiguous runs of each field plane.
//
// Index quirk reproduced on purpose: the free-surface tendency integrates
// Hu, Hv over the xi index (d % n) and differentiates the column integrals
// along eta and zeta, replicating the result along xi
// (primitive_equations.cpp:244-272).  omega is identically 0 in the RHS
// (src/solver/simulation_driver.cpp:222 -> primitive_equations.cpp:47-48), so
// zeta fluxes vanish.
#pragma once
#include <type_traits>

#include "drf_internal.hpp"
#include "interface.hpp"

namespace drf {
namespace vol {

// LDS slots per element node, used in two rounds (see the kernel).
enum : int { S_A = 0, S_B, S_C, S_D, S_E, S_F, S_G, S_NF };
static_assert(S_NF == kVolSlots, "the batch geometry counts the kernel's LDS slots");

// LW: grid lines per workgroup (128, 256 or 512), the workgroup size; the
// elements per batch EPB follow from it and from the LDS budget
// (vol_batch_elements, shared with the blocked layout's block size).
template <int N, int LW> struct Cfg {
    static constexpr int n = N + 1, n2 = n * n, n3 = n2 * n;
    static constexpr int EPB = vol_batch_elements(N, LW);
    static constexpr int NT = EPB * n2;
    static constexpr int BLOCK = ((NT + 63) / 64) * 64;
    // minimum waves per SIMD the register allocation must allow
    template <class TS, int EPI> static constexpr int wpe()
    {
        return sizeof(TS) == 8 ? (N <= 4 ? 2 : 1) : (N <= 4 ? 3 : 2);
    }
};

// LDS placement of the staged values.  Node (i, j, k) of a slot sits at
// i + j SJ + k SK, slots SS apart, elements ES apart.  The LDS serves 32 banks
// of 4 bytes a clock, so B = 32 float or 16 double lanes at a time: SJ, SK and
// ES (mod B) are such that B consecutive xi-lines lie in distinct banks where
// some padding can do it (odd n need none, n = 6 in FP64 has no LDS to spare),
// and the eta- and zeta-lines are dealt to the lanes by line_order, so that
// theirs do too.  Naturally placed and dealt, the accesses took 3.2 (N = 3),
// 1.6 (N = 4) and 4.5 (N = 7) times their conflict-free clocks in FP64, and
// 3.5, 2.0 and 5.0 times in FP32; now 1.0 to 1.3 (n = 2 and FP64 n = 6: 1.5).
// RK4 of 4 M nodes in FP64: N = 3 205 -> 174 us, N = 4 204 -> 196 us, N = 7
// 450 -> 405 us; in FP32 N = 3 97.6 -> 88.7 us, N = 4 110.9 -> 100.0 us.
template <int n, int BYTES> struct Place {
    static constexpr int B = 128 / BYTES;
    static constexpr bool D = BYTES == 8;
    static constexpr int SJ = n == 6 ? (D ? 6 : 7) : n == 8 ? 9 : n;
    static constexpr int SK = n == 4 ? (D ? 17 : 19) : n == 6 ? (D ? 36 : 42) : n == 8 ? 72 : n * n;
    // element stride modulo B
    static constexpr int EM = (n == 2   ? 9
                               : n == 4 ? (D ? 68 : 80)
                               : n == 6 ? (D ? 219 : 252)
                               : n == 8 ? (D ? 584 : 583)
                                        : n * n * n) % B;
    static constexpr int SS = (n - 1) * (1 + SJ + SK) + 1;
    static constexpr int ES = S_NF * SS + (EM + B - S_NF * SS % B) % B;
};

// The eta- and zeta-lines of a batch in the order the lanes take them: entry t
// packs the first node's place (element part included) of lane t's eta-line
// (low half) and zeta-line.  Each group of B lanes takes one line from each of
// the fullest banks in turn.
template <int NT> struct LineOrder {
    uint32_t v[NT];
};
template <int n, int EPB, int BYTES> constexpr LineOrder<EPB * n * n> line_order()
{
    using P = Place<n, BYTES>;
    constexpr int NT = EPB * n * n, B = P::B;
    static_assert(EPB * P::ES < 65536, "line places are packed in 16 bits");
    LineOrder<NT> r{};
    for (int z = 0; z < 2; ++z) {
        int place[NT] = {}, left[B] = {};
        bool used[NT] = {};
        for (int t = 0; t < NT; ++t) {
            const int e = t / (n * n), L = t % (n * n);
            place[t] = e * P::ES + L % n + (L / n) * (z ? P::SJ : P::SK);
            ++left[place[t] % B];
        }
        int out = 0;
        while (out < NT) {
            const int end = out + B < NT ? out + B : NT;
            while (out < end) {
                // one pass over the banks, fullest first
                bool taken[B] = {};
                for (int pass = 0; pass < B && out < end; ++pass) {
                    int best = -1;
                    for (int b = 0; b < B; ++b)
                        if (!taken[b] && left[b] > 0 && (best < 0 || left[b] > left[best]))
                            best = b;
                    if (best < 0)
                        break;
                    taken[best] = true;
                    int t = 0;
                    while (used[t] || place[t] % B != best)
                        ++t;
                    used[t] = true;
                    --left[best];
                    r.v[out++] |= (uint32_t)place[t] << (16 * z);
                }
            }
        }
    }
    return r;
}
template <int n, int EPB, int BYTES> struct LineTable {
    static constexpr LineOrder<EPB * n * n> order = line_order<n, EPB, BYTES>();
};

// Operators sized for one order, passed by value (kernel-argument SGPRs).
template <int n, class TC> struct KOps {
    TC D[n * n];   // 1D derivative matrix, row-major
    TC D2[n * n];  // D * D (second derivative; read by the FP32 kernel only)
    double Dc[n * n]; // FP64 D for the free-surface column integrals
    double sw[n];     // 0.5 * LGL weights
};

template <class TS, class TC> __device__ __forceinline__ TC ld(const TS *p) { return (TC)(*p); }

// Addresses are split into a wave-uniform base (pointer + field and xi
// offsets, all from kernel arguments: SGPRs) and a 32-bit per-lane byte offset
// (element and line), so that an access can be one `saddr` load or store with a
// single VGPR offset.  In the line and blocked layouts the compiler forms most
// addresses by a 64-bit vector add of base and offset all the same: 41 of them in
// the right-hand side at N = 1, 95 at N = 4, 159 at N = 8.  Offsets within one
// field must stay below 4 GiB (checked on the host).
template <class TS, class TC> __device__ __forceinline__ TC ldo(const TS *ubase, uint32_t off)
{
    return (TC)(*(const TS *)((const char *)ubase + off));
}
// NT: a streaming store, for a result that nothing reads back soon.
template <class TS, bool NT = false>
__device__ __forceinline__ void sto(TS *ubase, uint32_t off, TS v)
{
    if constexpr (NT)
        __builtin_nontemporal_store(v, (TS *)((char *)ubase + off));
    else
        *(TS *)((char *)ubase + off) = v;
}
// The n adjacent nodes of a xi-line (ADJ: the packed and structure-of-arrays
// layouts), moved in accesses of up to 16 bytes: with one per node every access
// of a wavefront touches all the cache lines that the n share, and the L1
// serves them n times over.
template <class T> struct Chunk {
    static constexpr int W = 16 / (int)sizeof(T);
    typedef T V __attribute__((ext_vector_type(W), aligned(sizeof(T))));
    typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};
template <int n, class TS, class TC>
__device__ __forceinline__ void ld_run(const TS *ubase, uint32_t off, TC (&v)[n])
{
    using C = Chunk<TS>;
    const char *p = (const char *)ubase + off;
    constexpr int nw = n / C::W * C::W, n2 = nw + (C::W == 4 && n - nw >= 2 ? 2 : 0);
#pragma unroll
    for (int i = 0; i < nw; i += C::W) {
        const typename C::V c = *(const typename C::V *)(p + i * sizeof(TS));
#pragma unroll
        for (int k = 0; k < C::W; ++k)
            v[i + k] = (TC)c[k];
    }
    if constexpr (n2 > nw) {
        const typename C::V2 c = *(const typename C::V2 *)(p + nw * sizeof(TS));
        v[nw] = (TC)c[0];
        v[nw + 1] = (TC)c[1];
    }
    if constexpr (n > n2)
        v[n2] = (TC)(*(const TS *)(p + n2 * sizeof(TS)));
}
template <int n, class TS, class TC>
__device__ __forceinline__ void st_run(TS *ubase, uint32_t off, const TC (&v)[n])
{
    using C = Chunk<TS>;
    char *p = (char *)ubase + off;
    constexpr int nw = n / C::W * C::W, n2 = nw + (C::W == 4 && n - nw >= 2 ? 2 : 0);
#pragma unroll
    for (int i = 0; i < nw; i += C::W) {
        typename C::V c;
#pragma unroll
        for (int k = 0; k < C::W; ++k)
            c[k] = (TS)v[i + k];
        *(typename C::V *)(p + i * sizeof(TS)) = c;
    }
    if constexpr (n2 > nw) {
        typename C::V2 c;
        c[0] = (TS)v[nw];
        c[1] = (TS)v[nw + 1];
        *(typename C::V2 *)(p + nw * sizeof(TS)) = c;
    }
    if constexpr (n > n2)
        *(TS *)(p + n2 * sizeof(TS)) = (TS)v[n2];
}

// Byte offsets of (element, line) pairs.  32-bit arithmetic is exact: the
// host checks that every offset of the launch fits in 32 bits.
//
// A view without blocks: the bathymetry and Coriolis lines (always in the
// line layout, no larger than one field of the state).
template <class T> __device__ __forceinline__ uint32_t flat_off(const View<T> &v, int64_t e, int L)
{
    return ((uint32_t)e * (uint32_t)v.es + (uint32_t)L * (uint32_t)v.ls) * (uint32_t)sizeof(T);
}
// Element e of batch b in a state view.  All state views of one launch share
// the layout and its strides.  In the blocked layout a batch never straddles
// a block (a block's element count is a multiple of the batch's, checked at
// launch), so the block is b / (bb / EPB): a division of uniform values, once
// per batch, none per lane.  Lanes that repeat element E - 1 sit in the last
// batch, in that element's block.  Without blocks (bb = 0) the block is 0.
template <int EPB, class T>
__device__ __forceinline__ uint32_t state_off(const View<T> &v, int64_t b, int64_t e, int L)
{
    const uint32_t q = v.bb ? (uint32_t)v.bb / (uint32_t)EPB : 0xffffffffu;
    const uint32_t blk = (uint32_t)b / q;
    const uint32_t eb = (uint32_t)e - blk * (uint32_t)v.bb;
    return (blk * (uint32_t)v.bs + eb * (uint32_t)v.es + (uint32_t)L * (uint32_t)v.ls) *
           (uint32_t)sizeof(T);
}

template <class TC> __device__ __forceinline__ TC hinv_of(TC H)
{
    // PrimitiveState::update_derived, primitive_equations.cpp:23
    return (H > (TC)1e-10) ? (TC)1 / H : (TC)0;
}

// y = M x along one line (n taps), M row-major.
template <int n, class TC>
__device__ __forceinline__ void dline(const TC *__restrict__ M, const TC (&x)[n], TC (&y)[n])
{
#pragma unroll
    for (int i = 0; i < n; ++i) {
        TC s = M[i * n] * x[0];
#pragma unroll
        for (int m = 1; m < n; ++m)
            s += M[i * n + m] * x[m];
        y[i] = s;
    }
}

// Second derivative along one line.  FP64: D (D x), two contractions as the
// reference applies its gradient twice, with only D in SGPRs.  FP32: D^2
// formed once on the host (one contraction; two float matrices fit the SGPR
// file).
template <int n, class TC>
__device__ __forceinline__ void d2line(const TC *__restrict__ D, const TC *__restrict__ D2,
                                       const TC (&x)[n], TC (&y)[n])
{
    if constexpr (sizeof(TC) == 8) {
        TC t[n];
        dline<n>(D, x, t);
        dline<n>(D, t, y);
    } else {
        dline<n>(D2, x, y);
    }
}

// The state lines a thread needs for phase P1, with the Coriolis parameter
// along the line (a field, or the constant f0).
template <int n, class TC> struct Lines {
    TC q[5][n]; // Hu, Hv, eta, HT, HS
    TC hb[n], fc[n];
};

template <int n, class TS, class TC>
__device__ __forceinline__ void load_h(Lines<n, TC> &L, const VolGeom<TS> &geo, int64_t e, int line)
{
    const uint32_t ho = flat_off(geo.h, e, line);
#pragma unroll
    for (int i = 0; i < n; ++i)
        L.hb[i] = ldo<TS, TC>(geo.h.p + i * geo.h.is, ho);
}
template <int n, class TS, class TC>
__device__ __forceinline__ void load_f(Lines<n, TC> &L, const VolGeom<TS> &geo, int64_t e, int line)
{
    if (geo.f.p) {
        const uint32_t fo = flat_off(geo.f, e, line);
#pragma unroll
        for (int i = 0; i < n; ++i)
            L.fc[i] = ldo<TS, TC>(geo.f.p + i * geo.f.is, fo);
    } else {
#pragma unroll
        for (int i = 0; i < n; ++i)
            L.fc[i] = (TC)geo.f0;
    }
}

// Fields [F0, F0 + NFD) of the xi-line at offset so into u[0..], node by node
// or (BY_FIELD) field by field
template <int n, int F0, int NFD, bool ADJ, bool BY_FIELD = false, class TS, class TC, int NU>
__device__ __forceinline__ void load_fields(const View<const TS> &U, uint32_t so, TC (&u)[NU][n])
{
    if constexpr (ADJ) {
#pragma unroll
        for (int f = 0; f < NFD; ++f)
            ld_run<n, TS, TC>(U.p + (F0 + f) * U.fs, so, u[f]);
    } else if constexpr (BY_FIELD) {
#pragma unroll
        for (int f = 0; f < NFD; ++f)
#pragma unroll
            for (int i = 0; i < n; ++i)
                u[f][i] = ldo<TS, TC>(U.p + (F0 + f) * U.fs + i * U.is, so);
    } else {
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                u[f][i] = ldo<TS, TC>(U.p + (F0 + f) * U.fs + i * U.is, so);
    }
}

// Plain right-hand sides whose lines fill the registers (FP64 from N = 5, FP32
// at N = 8) load a node's bathymetry with its fields and take the LDS places of
// their lines from outside the phases: 4 M nodes, FP64 N = 6 133.4 -> 130.6, N =
// 7 118.0 -> 115.3, mixed N = 8 93.4 -> 90.2 us.  The others were the same or
// slower (mixed N = 6 56.8 -> 57.6, FP64 N = 4 83.7 -> 84.0 us).
template <int n, class TC> constexpr bool wide_line() { return sizeof(TC) == 8 ? n >= 6 : n == 9; }

// All of P1's global loads are issued here, so that P1 itself waits only for
// them: a load issued inside P1 would make the wave wait for every store of
// the previous batch as well (gfx9 counts loads and stores in one in-order
// counter).
template <int n, int EPB, int NF, bool WITH_F, bool ADJ, class TS, class TC>
__device__ __forceinline__ void load_lines(Lines<n, TC> &L, const View<const TS> &U,
                                           const VolGeom<TS> &geo, int64_t b, int64_t e, int line)
{
    const uint32_t uo = state_off<EPB>(U, b, e, line);
    if constexpr (WITH_F && !ADJ && wide_line<n, TC>()) {
        // a node's bathymetry with its fields, as P1 takes both node by node:
        // with h last P1 waited for the whole line
        const uint32_t ho = flat_off(geo.h, e, line);
#pragma unroll
        for (int i = 0; i < n; ++i) {
#pragma unroll
            for (int f = 0; f < NF; ++f)
                L.q[f][i] = ldo<TS, TC>(U.p + f * U.fs + i * U.is, uo);
            L.hb[i] = ldo<TS, TC>(geo.h.p + i * geo.h.is, ho);
        }
    } else {
        load_fields<n, 0, NF, ADJ>(U, uo, L.q);
        load_h<n, TS, TC>(L, geo, e, line);
    }
    if (WITH_F)
        load_f<n, TS, TC>(L, geo, e, line);
}

constexpr int kXcds = 8; // MI355X: 8 XCDs of 32 CUs

// Writes fields [F0, F0 + NFD) of the thread's xi-line.  so: the line's byte
// offset in the state views (state_off).
template <int n, int F0, int NFD, bool ADJ, bool NT, class TS, class TC>
__device__ __forceinline__ void write_fields(const View<TS> &R, uint32_t so,
                                             const TC (&kv)[NFD][n])
{
#pragma unroll
    for (int f = 0; f < NFD; ++f)
        if constexpr (ADJ) {
            st_run<n, TS, TC>(R.p + (F0 + f) * R.fs, so, kv[f]);
        } else {
#pragma unroll
            for (int i = 0; i < n; ++i)
                sto<TS, NT>(R.p + (F0 + f) * R.fs + i * R.is, so, (TS)kv[f][i]);
        }
}

// What the schemes read of the thread's xi-line besides the tendency: the
// step's initial state, which is U until the step's own stores and is read
// again (from the L2) a phase before each use, and an accumulator, which stays
// in registers.  (With the initial state in registers too, FP64 at N = 4
// spilled 48 VGPRs per lane.)
constexpr bool step_reads_u0(int epi) { return epi != EPI_RHS && epi != EPI_LSRK; }
constexpr bool step_has_acc(int epi) { return epi == EPI_RK4 || epi == EPI_LSRK; }

// The coefficients of one stage (EpiMode), the dt-proportional one formed from
// the device dt in adaptive steps.
template <class TC> struct StageCoefs {
    TC c1, c2, c3;
    bool first, last;
};
template <class TS, class TC>
__device__ __forceinline__ StageCoefs<TC> stage_coefs(const Epi<TS> &epi, int st)
{
    double d = epi.c1[st];
    if (epi.dtp)
        d = (d * *epi.dtp) / epi.q[st];
    return {(TC)d, (TC)epi.c2[st], (TC)epi.c3[st], st == 0, st == epi.nst - 1};
}

// Fields [F0, F0 + NFD) of the stage state y after a stage with tendency k
// and initial state u0, with the association of the reference's stage sums.
// acc is 0 before the first stage.  First and last stages differ by selects:
// branches on them, one per value, cost registers and time.
template <int n, int F0, int NFD, int EPI, int NA, class TC>
__device__ __forceinline__ void stage_update(const StageCoefs<TC> &c, const TC (&k)[NFD][n],
                                             const TC (&u0)[NFD][n], TC (&y)[5][n],
                                             TC (&acc)[NA][n])
{
#pragma unroll
    for (int f = 0; f < NFD; ++f)
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const TC ki = k[f][i];
            TC &yi = y[F0 + f][i];
            if constexpr (EPI == EPI_STAGE) {
                yi = u0[f][i] + c.c1 * ki;
            } else if constexpr (EPI == EPI_SSP3) {
                const TC t = yi + c.c1 * ki; // y is u0 in the first stage
                const TC r = c.c2 * u0[f][i] + c.c3 * t;
                yi = c.first ? t : r;
            } else if constexpr (EPI == EPI_RK4) {
                TC &a = acc[F0 + f][i]; // c2 = 1, 2, 2, 1
                a = a + c.c2 * ki;
                yi = u0[f][i] + c.c1 * (c.last ? a : ki);
            } else if constexpr (EPI == EPI_LSRK) {
                TC &a = acc[F0 + f][i]; // c2 = 0 first
                a = c.c2 * a + c.c1 * ki;
                yi = yi + c.c3 * a;
            }
        }
}

// The conforming face term in the plain right-hand side: none, or with one of
// the scalar fluxes (a template argument: a branch between the two fluxes
// around the neighbours' nodes spilled them).
enum : int { FACES_NONE = 0, FACES_LF = 1, FACES_UPWIND = 2 };

// One face of the conforming face term seen from one of its elements, for
// nodes with the value own here and other across: what face_elem_kernel
// (faces.hip) adds, bit for bit on finite values.  With the interface's normal
// n = +-e_axis and F its flux in left/right order, the contribution is +wq F
// on the left and -wq F on the right; both equal wq times the flux formed with
// this element's outward normal, since every term only changes sign and sums
// commute.  (UPWIND at vn = 0 takes the left value.)
//   LF_ADV  0.5 (vn own + vn other) - 0.5 lambda (other - own), and the
//           normal's zero components make it NaN where a value is not finite
//   UPWIND  vn (own or other)
template <class T, bool LF> struct FaceFlux {
    T vn, hl;
    bool take_own;
    __device__ __forceinline__ FaceFlux(const VolFaces<T> &fc, int axis, bool upper, uint32_t entry)
    {
        vn = upper ? fc.p[axis] : -fc.p[axis];
        hl = T(0.5) * fc.p[3];
        take_own = (entry & 1u) ? !(vn <= T(0)) : vn >= T(0);
    }
    __device__ __forceinline__ T operator()(T own, T other, T wq) const
    {
#pragma clang fp contract(off)
        if constexpr (LF) {
            const T d = other - own;
            const T F = T(0.5) * (vn * own + vn * other) - hl * d;
            return wq * __builtin_elementwise_fma(d, T(0), F);
        }
        return wq * (vn * (take_own ? own : other));
    }
};

// The faces xi-line L lies on: both x-faces at its ends, a y-face when j is 0
// or N, a z-face when k is 0 or N, as entries of the plan's element table
// (kNoFace elsewhere).  Of a y- or z-face only the lines with points of the
// N-point face rule (DOFs it + n jt < nq) are kept.
constexpr uint32_t kNoFace = 0xffffffffu;
template <int n> struct FaceLine {
    static constexpr int nq1 = n <= 2 ? 2 : n - 1, nq = nq1 * nq1;
    uint32_t x0, x1, y, z;
    __device__ __forceinline__ void load(const uint32_t *__restrict__ eface, int64_t e, int L)
    {
        const int j = L % n, k = L / n;
        const uint32_t *t = eface + 6 * e;
        const bool x = L < nq, yb = (j == 0 || j == n - 1) && n * k < nq,
                   zb = (k == 0 || k == n - 1) && n * j < nq;
        x0 = x ? t[0] : kNoFace;
        x1 = x ? t[1] : kNoFace;
        y = yb ? t[j == 0 ? 2 : 3] : kNoFace;
        z = zb ? t[k == 0 ? 4 : 5] : kNoFace;
    }
};

// Byte offset of line L of the neighbour of a table entry (neighbour << 1 | side)
template <int N, class T>
__device__ __forceinline__ uint32_t nb_off(const View<T> &v, uint32_t entry, int L)
{
    constexpr uint32_t B = (uint32_t)vol_batch_elements(N, N <= 4 ? 512 : 128);
    const uint32_t e = entry >> 1;
    uint32_t base = e * (uint32_t)v.es;
    if (v.bb) // the blocked layout's block is B elements (layout_strides)
        base = e / B * (uint32_t)v.bs + e % B * (uint32_t)v.es;
    return (base + (uint32_t)L * (uint32_t)v.ls) * (uint32_t)sizeof(T);
}

// The neighbours' nodes of fields [F0, F0 + NFD) across the line's faces
template <int n, int NFD, class T> struct FaceNodes {
    T x0[NFD], x1[NFD], y[NFD][n], z[NFD][n];
    template <int F0>
    __device__ __forceinline__ void load(const FaceLine<n> &fl, const View<const T> &U, int L)
    {
        constexpr int nq = FaceLine<n>::nq;
        const int j = L % n, k = L / n;
        auto at = [&](int f, int i, uint32_t off) { return ldo<T, T>(U.p + f * U.fs + i * U.is, off); };
        if (fl.x0 != kNoFace) {
            const uint32_t o = nb_off<n - 1>(U, fl.x0, L);
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                x0[f] = at(F0 + f, n - 1, o);
        }
        if (fl.x1 != kNoFace) {
            const uint32_t o = nb_off<n - 1>(U, fl.x1, L);
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                x1[f] = at(F0 + f, 0, o);
        }
        if (fl.y != kNoFace) {
            const uint32_t o = nb_off<n - 1>(U, fl.y, (n - 1 - j) + n * k);
#pragma unroll
            for (int f = 0; f < NFD; ++f)
#pragma unroll
                for (int i = 0; i < n; ++i)
                    if (i + n * k < nq)
                        y[f][i] = at(F0 + f, i, o);
        }
        if (fl.z != kNoFace) {
            const uint32_t o = nb_off<n - 1>(U, fl.z, j + n * (n - 1 - k));
#pragma unroll
            for (int f = 0; f < NFD; ++f)
#pragma unroll
                for (int i = 0; i < n; ++i)
                    if (i + n * j < nq)
                        z[f][i] = at(F0 + f, i, o);
        }
    }
    // out[F0 + f] = M^-1 (x, y and z contributions, summed in that order) of
    // the own nodes q[F0 + f].  A node that was not loaded is not read.
    template <int F0, bool LF>
    __device__ __forceinline__ void contrib(const FaceLine<n> &fl, const VolFaces<T> &fc,
                                            const T (&q)[5][n], int L, const T *sWq,
                                            const T *sMinv, T (&out)[5][n]) const
    {
#pragma clang fp contract(off)
        constexpr int nq = FaceLine<n>::nq;
        const int j = L % n, k = L / n;
#pragma unroll
        for (int f = 0; f < NFD; ++f)
#pragma unroll
            for (int i = 0; i < n; ++i)
                out[F0 + f][i] = T(0);
        if (fl.x0 != kNoFace) {
            const FaceFlux<T, LF> F(fc, 0, false, fl.x0);
            const T w = sWq[L];
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                out[F0 + f][0] += F(q[F0 + f][0], x0[f], w);
        }
        if (fl.x1 != kNoFace) {
            const FaceFlux<T, LF> F(fc, 0, true, fl.x1);
            const T w = sWq[L];
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                out[F0 + f][n - 1] += F(q[F0 + f][n - 1], x1[f], w);
        }
        if (fl.y != kNoFace) {
            const FaceFlux<T, LF> F(fc, 1, j != 0, fl.y);
#pragma unroll
            for (int i = 0; i < n; ++i)
                if (i + n * k < nq) {
                    const T w = sWq[i + n * k];
#pragma unroll
                    for (int f = 0; f < NFD; ++f)
                        out[F0 + f][i] += F(q[F0 + f][i], y[f][i], w);
                }
        }
        if (fl.z != kNoFace) {
            const FaceFlux<T, LF> F(fc, 2, k != 0, fl.z);
#pragma unroll
            for (int i = 0; i < n; ++i)
                if (i + n * j < nq) {
                    const T w = sWq[i + n * j];
#pragma unroll
                    for (int f = 0; f < NFD; ++f)
                        out[F0 + f][i] += F(q[F0 + f][i], z[f][i], w);
                }
        }
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const T m = sMinv[i + n * L];
#pragma unroll
            for (int f = 0; f < NFD; ++f)
                out[F0 + f][i] = m * out[F0 + f][i];
        }
    }
};

// Fields whose neighbour nodes are in flight at once: all where the registers
// allow it, else one chunk while the next one loads.  Coastline octree, 39,280
// elements, line layout, LF / UPWIND, in us, and the VGPRs spilled at N = 4:
//              all at once      in twos          one by one
//   FP64 N = 1  26.0 /  25.9    25.7 /  25.7     26.1 /  26.0
//   FP64 N = 2  49.2 /  48.1    48.6 /  47.8     50.8 /  51.4
//   FP64 N = 3  96.4 /  95.7    96.4 /  96.3    100.8 / 100.0
//   FP64 N = 4   293 /   287 (53)  219 / 249 (28)  212 / 207 (5)
//   FP32 N = 1  21.8 /  21.7    21.0 /  21.0     21.3 /  21.3
//   FP32 N = 2  32.8 /  32.4    33.0 /  33.6     35.4 /  35.8
//   FP32 N = 3  53.4 /  53.2    56.8 /  56.4     61.0 /  62.0
//   FP32 N = 4   122 /   122 (15)  109 / 118 (10)  112 / 113 (0)
// The packed and structure-of-arrays layouts (ADJ) agree, but for FP32: UPWIND at
// N = 4 takes 118.0 in twos and 118.6 one by one, LF at N = 2 32.0 all at once and
// 31.2 in twos (UPWIND 30.9 and 31.6).
template <int N, class T, int FACES, bool ADJ> constexpr int face_chunk()
{
    if (N <= 3)
        return 5;
    return sizeof(T) == 8 || (FACES == FACES_UPWIND && !ADJ) ? 1 : 2;
}
template <int n, int CH, int F0, bool LF, int NFD, class T>
__device__ __forceinline__ void face_fields(const FaceNodes<n, NFD, T> &fn, const FaceLine<n> &fl,
                                            const VolFaces<T> &fc, const View<const T> &U,
                                            const T (&q)[5][n], int L, const T *sWq,
                                            const T *sMinv, T (&out)[5][n])
{
    constexpr int F1 = F0 + NFD;
    if constexpr (F1 < 5) {
        FaceNodes<n, (F1 + CH <= 5 ? CH : 5 - F1), T> next;
        next.template load<F1>(fl, U, L);
        fn.template contrib<F0, LF>(fl, fc, q, L, sWq, sMinv, out);
        face_fields<n, CH, F1, LF>(next, fl, fc, U, q, L, sWq, sMinv, out);
    } else {
        fn.template contrib<F0, LF>(fl, fc, q, L, sWq, sMinv, out);
    }
}

template <int n, int F0, int NFD, class T>
__device__ __forceinline__ void add_faces(T (&k)[NFD][n], const T (&fa)[5][n])
{
#pragma unroll
    for (int f = 0; f < NFD; ++f)
#pragma unroll
        for (int i = 0; i < n; ++i)
            k[f][i] = k[f][i] + fa[F0 + f][i];
}

// The kernel.  Seven LDS slots per element node, six of them reused in two
// rounds (momentum, then tracers), so a workgroup of 5 N=4 elements needs
// 35 KB of staging plus 4 KB of column integrals, and the CU's occupancy is
// set by registers (4 workgroups at N=4 FP64) rather than by LDS.
//
// With EPI a step's scheme, the phases below run once per stage on a batch
// whose state never leaves the registers: memory sees the state read and
// written once per step and, each stage, the batch's own lines of U and h
// again, which the L2 still holds (about 100 KB per CU).  One launch per
// stage, each streaming the state and its operands, was bound by HBM at
// 10 GB per RK4 step of 262,144 FP32 N=4 elements; here the bound is the
// VALU and the LDS.  RK4, N=4: FP64 32,768 elements 640 -> 196 us, FP32
// 262,144 elements 2,950 -> 750 us; SSP-RK3, FP64, N=3, 4,096 elements
// 35.8 -> 20 us (one launch in place of three).
//
//   P1  xi-owner   xi-derivatives of the momentum terms (registers), column
//                  integrals (FP64), stages A=Hu v, B=Hv v, C=eta, D=u, E=v, F=H,
//                  G=1/H (the dry-node guard of update_derived applied once)
//   P2a eta-owner  eta-derivatives of the momentum terms -> A, B
//   P3a zeta-owner vertical diffusion of u, v             -> A, B +=
//   P4a xi-owner   dHu, dHv complete (written out); xi-derivatives of the
//                  tracer terms; restages A=v HT, B=v HS, C=T, D=S (F, G kept)
//   P23b eta-owner eta-derivatives of the tracer fluxes    -> A, B
//        zeta-owner vertical diffusion of T, S (same phase) -> C, D
//   P4b xi-owner   dHT, dHS and d eta complete (written out)
//   FACES: after P1's barrier the xi-owner, its state line still in registers,
//        forms its line's face term, which P4a and P4b add
template <int N, class TS, class TC, int EPI, int LW, int FACES, bool ADJ>
__global__ void __launch_bounds__((Cfg<N, LW>::BLOCK)) __attribute__((amdgpu_waves_per_eu(Cfg<N, LW>::template wpe<TS, EPI>())))
    volume_kernel(const VolGeom<TS> geo, const KOps<N + 1, TC> ops, const Phys ph,
                  const View<const TS> U, const Epi<TS> epi, const int64_t nbatch)
{
    using C = Cfg<N, LW>;
    // The right-hand side prefetches the next batch's lines.  A Runge-Kutta
    // step keeps its stage state, initial state and accumulator in those
    // registers instead, and runs every stage of one batch before the next.
    constexpr int n = C::n;
    constexpr bool STEP = EPI != EPI_RHS;
    constexpr bool PREFETCH = !STEP;
    // With faces FP64 at N = 4 has no registers to prefetch the tracers, which
    // are first needed after P1: they are loaded with the neighbours' nodes
    // (prefetched, 37 VGPRs spilled).
    // With faces the tendencies stream past the L2, which the neighbours' reads
    // need, except where a lane's nodes are adjacent and accesses share lines
    // (FP64 N = 3 246 -> 401 us).  Coastline octree, kept and streamed: FP64 N =
    // 2 50.2 and 49.3, N = 3 101.2 and 96.4, N = 4 219.9 and 212.5 us; FP32 N = 3
    // 55.5 and 53.4, N = 4 114.0 and 108.9 us; the same at N = 1, and FP32 N = 2
    // 32.4 and 32.8 us.
    constexpr bool NTS = FACES != FACES_NONE && !ADJ;
    constexpr int NPRE = FACES && sizeof(TC) == 8 && N == 4 ? 3 : 5;
    // FP64 from N = 6 has no registers to load a step's initial state a phase
    // early (SSP-RK3 at N = 8: 555 us early, 544 us at the use)
    constexpr bool LATE = sizeof(TC) == 8 && N >= 6;
    // ... and then field by field where that was the faster order: 4 M nodes,
    // node by node and field by field, Euler N = 6 148.7 and 147.2, N = 8 219.8
    // and 213.5 us, RK4 N = 6 426 and 400, N = 8 675 and 666 us, SSP-RK3 N = 8
    // 542 and 523 us, but N = 7 301 and 306 us.
    constexpr bool BY_FIELD = LATE && N != 7;
    constexpr bool PLACES_OUTSIDE = !STEP && FACES == FACES_NONE && wide_line<n, TC>();
    // The plain right-hand side's phases stand in a loop of one trip where the
    // compiler then keeps fewer bases and operators live across them (4 M nodes,
    // straight and in the loop: FP64 N = 6 133 and 113 us; FP32 N = 2 48.2 and
    // 44.2, N = 3 42.4 and 41.0 us); every other order was the same or slower
    // (FP64 N = 5 85 and 93, FP32 N = 4 46.5 and 50.3, N = 7 56 and 79 us).
    constexpr bool ONE_TRIP = !STEP && FACES == FACES_NONE &&
                              (sizeof(TC) == 8 ? N == 6 : N == 2 || N == 3);
    constexpr int n2 = C::n2, n3 = C::n3, EPB = C::EPB;
    using P = Place<n, (int)sizeof(TC)>;
    __shared__ TC sm[EPB * P::ES];
    // column integrals, double-buffered by batch parity: the last phase of
    // one batch reads them while the first phase of the next writes
    __shared__ double bar[2][EPB][2][n2];
    // the FP64 D of the column integrals, indexed per lane in P4b (from the
    // kernel arguments such an index compiles to a global load, and its wait
    // would drain the next batch's prefetch and this batch's stores)
    __shared__ double sDc[n * n];
    // FACES: face-rule weight by face DOF and M^-1 by node
    __shared__ TS sWq[FACES ? n2 : 1], sMinv[FACES ? n3 : 1];

    // Every lane runs through every phase, so that no phase sits behind an
    // exec-mask branch: lanes past the tile repeat the last line of the last
    // element (in the same wavefront, in lockstep), and elements past the end
    // of the mesh repeat element E - 1 in their own LDS slots.  Their stores
    // of the right-hand side write the values the owners write.  With the
    // stores on every path, P1 waits only for the prefetched lines and not
    // for the previous batch's stores to drain.  A step, which rewrites its
    // input in place, stores from the owners only (what the other lanes read
    // may already be the new state; nothing of theirs is kept).
    const int tid = threadIdx.x;
    const int tq = tid >= C::NT ? C::NT - 1 : tid;
    const int le = tq / n2;
    const int L0 = tq - le * n2;
    // first nodes of this lane's eta- and zeta-line
    const uint32_t lines = LineTable<n, EPB, (int)sizeof(TC)>::order.v[tq];
    const int64_t elast = geo.E - 1;
    auto elem = [&](int64_t bb) {
        const int64_t x = bb * EPB + le;
        return x > elast ? elast : x;
    };

    const TC g = (TC)ph.g, nu_h = (TC)ph.nu_h, nu_v = (TC)ph.nu_v, kT = (TC)ph.kT, kS = (TC)ph.kS;
    const TC *__restrict__ D = ops.D;
    const TC *__restrict__ D2 = ops.D2;
    // the FP64 D of the column integrals is D itself when TC is double:
    // reading it from D keeps one operator fewer in SGPRs
    const double *__restrict__ Dc =
        std::is_same<TC, double>::value ? (const double *)ops.D : ops.Dc;

    // XCD-aware batch order.  Workgroups are dealt round-robin to the 8 XCDs
    // (blockIdx % 8), each with its own L2.  Renumbering them so that
    // consecutive logical workgroups sit on one XCD puts neighbouring
    // batches -- whose line spans share a 128-byte cache line, the spans not
    // being line-aligned -- behind the same L2, while the grid as a whole
    // still sweeps memory in one contiguous window per round.
    const int64_t G = gridDim.x;
    const int64_t lw = (geo.xcd_remap && G % kXcds == 0)
                           ? (blockIdx.x % kXcds) * (G / kXcds) + blockIdx.x / kXcds
                           : (int64_t)blockIdx.x;
    int64_t b = lw, bend = nbatch, bstep = G;
    if (FACES && geo.xcd_remap && G % kXcds == 0) {
        // neighbours are read too: each XCD sweeps an eighth of the mesh of its
        // own, so that they come through its L2
        const int64_t x = blockIdx.x % kXcds;
        bstep = G / kXcds;
        b = nbatch * x / kXcds + blockIdx.x / kXcds;
        bend = nbatch * (x + 1) / kXcds;
    }
    if (tid < n * n)
        sDc[tid] = Dc[tid]; // first read in P4b, after P1's barrier
    if constexpr (FACES) {
        for (int q = tid; q < n2; q += blockDim.x)
            sWq[q] = geo.faces.wq[q];
        for (int d = tid; d < n3; d += blockDim.x) {
            // 1 / (w_i w_j w_k), w = 2 sw exactly, rounded to the state type
            const TS wi = (TS)(2.0 * ops.sw[d % n]), wj = (TS)(2.0 * ops.sw[(d / n) % n]),
                     wk = (TS)(2.0 * ops.sw[d / n2]);
            const TS w = wi * wj * wk;
            sMinv[d] = TS(1) / w;
        }
    }
    Lines<n, TC> nxt;
    FaceLine<n> fl;
    if (PREFETCH) {
        const int64_t e0 = elem(b);
        if (b < bend && e0 < geo.E) {
            load_lines<n, EPB, NPRE, PREFETCH && !FACES, ADJ, TS, TC>(nxt, U, geo, b, e0, L0);
            if constexpr (FACES)
                fl.load(geo.faces.eface, e0, L0);
        }
    }

    int par = 0;
    for (; b < bend; b += bstep) {
        const int64_t e = elem(b);
        // P1 reads the prefetched lines in place (the next batch's loads
        // overwrite them only after P1's barrier), so the loop carries no
        // register copies that would wait for those loads.  In a step, nxt
        // is the stage state.
        if (STEP)
            load_lines<n, EPB, 5, false, ADJ, TS, TC>(nxt, U, geo, b, e, L0);
        Lines<n, TC> &cur = nxt;
        TC acc[step_has_acc(EPI) ? 5 : 1][n];
        if constexpr (step_has_acc(EPI)) {
#pragma unroll
            for (int f = 0; f < 5; ++f)
#pragma unroll
                for (int i = 0; i < n; ++i)
                    acc[f][i] = (TC)0;
        }
        // nodes of the xi-, eta- and zeta-line in slot 0
        TC *rx = nullptr, *ry = nullptr, *rz = nullptr;
        if constexpr (PLACES_OUTSIDE) {
            rx = sm + le * P::ES + (L0 % n) * P::SJ + (L0 / n) * P::SK;
            ry = sm + (lines & 0xffffu);
            rz = sm + (lines >> 16);
        }
        // One evaluation of the right-hand side of cur.
        auto evaluate = [&](int st) __attribute__((always_inline)) {
        // In a step the line is opaque to the compiler, so that it hoists no
        // load or address out of the stages into registers they do not have.
        int L = L0;
        if constexpr (STEP)
            asm volatile("" : "+v"(L));
        TC *sx = PLACES_OUTSIDE ? rx : sm + le * P::ES + (L % n) * P::SJ + (L / n) * P::SK;
        TC *sy = PLACES_OUTSIDE ? ry : sm + (lines & 0xffffu),
           *sz = PLACES_OUTSIDE ? rz : sm + (lines >> 16);
        const StageCoefs<TC> sc = stage_coefs<TS, TC>(epi, st);

        // Register state carried by the xi-owner: the momentum partials
        // (P1 -> P4a), HT and HS (P1 -> P4a), the tracer partials (P4a -> P4b).
        TC pHu[n], pHv[n], ht[n], hs[n];

        // ---------------- P1: xi-line (j, k) = (L % n, L / n) ----------------
        if constexpr (STEP || FACES)
            load_f<n, TS, TC>(nxt, geo, e, L);
        if constexpr (NPRE == 3) {
            const uint32_t uo = state_off<EPB>(U, b, e, L);
#pragma unroll
            for (int f = 3; f < 5; ++f)
                if constexpr (ADJ) {
                    ld_run<n, TS, TC>(U.p + f * U.fs, uo, nxt.q[f]);
                } else {
#pragma unroll
                    for (int i = 0; i < n; ++i)
                        nxt.q[f][i] = ldo<TS, TC>(U.p + f * U.fs + i * U.is, uo);
                }
        }
        {
            TC H[n], u[n], v[n], hinv[n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                H[i] = cur.q[2][i] + cur.hb[i];
                hinv[i] = hinv_of(H[i]);
                const TC hi = hinv[i];
                u[i] = cur.q[0][i] * hi;
                v[i] = cur.q[1][i] * hi;
                ht[i] = cur.q[3][i];
                hs[i] = cur.q[4][i];
            }
            // xi-derivatives (momentum_advection :275-305,
            // barotropic_pressure_gradient :322-337, horizontal_diffusion
            // :339-355) and Coriolis (:307-320)
            TC x[n], d[n];
#pragma unroll
            for (int i = 0; i < n; ++i)
                x[i] = cur.q[0][i] * u[i];
            dline<n>(D, x, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHu[i] = -d[i] + cur.fc[i] * cur.q[1][i];
#pragma unroll
            for (int i = 0; i < n; ++i)
                x[i] = cur.q[1][i] * u[i];
            dline<n>(D, x, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHv[i] = -d[i] + (-cur.fc[i]) * cur.q[0][i];
            dline<n>(D, cur.q[2], d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHu[i] += (-g * H[i]) * d[i];
            d2line<n>(D, D2, u, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHu[i] += H[i] * (nu_h * d[i]);
            d2line<n>(D, D2, v, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHv[i] += H[i] * (nu_h * d[i]);
#pragma unroll
            for (int i = 0; i < n; ++i) {
                sx[S_A * P::SS + i] = cur.q[0][i] * v[i];
                sx[S_B * P::SS + i] = cur.q[1][i] * v[i];
                sx[S_C * P::SS + i] = cur.q[2][i];
                sx[S_D * P::SS + i] = u[i];
                sx[S_E * P::SS + i] = v[i];
                sx[S_F * P::SS + i] = H[i];
                sx[S_G * P::SS + i] = hinv[i];
            }
            // Column integrals of compute_eta_rhs (:244-254): over the xi index,
            // summed in node order from 0, in FP64 at every precision.
            double su = 0.0, sv = 0.0;
#pragma unroll
            for (int i = 0; i < n; ++i) {
                su += ops.sw[i] * (double)cur.q[0][i];
                sv += ops.sw[i] * (double)cur.q[1][i];
            }
            bar[par][le][0][L] = su;
            bar[par][le][1][L] = sv;
        }
        TC fa[FACES ? 5 : 1][n];
        if constexpr (FACES) {
            constexpr int CH = face_chunk<N, TC, FACES, ADJ>();
            FaceNodes<n, CH, TC> fn;
            fn.template load<0>(fl, U, L);
            __syncthreads();
            face_fields<n, CH, 0, FACES == FACES_LF>(fn, fl, geo.faces, U, cur.q, L, sWq, sMinv, fa);
        } else {
            __syncthreads();
        }

        if (PREFETCH) {
            // Next batch of this workgroup, in flight during the other phases.
            const int64_t bn = b + bstep;
            const int64_t en = elem(bn);
            // issued at raised wave priority, so that the SIMD's other wave
            // does not interleave its arithmetic with these loads (6 (N + 1)
            // per lane; 1 % on the FP64 and mixed RHS at 128x128x16, N = 4)
            __builtin_amdgcn_s_setprio(2);
            if (bn < bend && en < geo.E) {
                load_lines<n, EPB, NPRE, PREFETCH && !FACES, ADJ, TS, TC>(nxt, U, geo, bn, en, L);
                if constexpr (FACES)
                    fl.load(geo.faces.eface, en, L);
            }
            __builtin_amdgcn_s_setprio(0);
        }

        // ---------------- P2a: eta-line (i, k) = (L % n, L / n) ----------------
        {
            TC fuv[n], fvv[n], et[n], u[n], v[n], H[n];
#pragma unroll
            for (int j = 0; j < n; ++j) {
                fuv[j] = sy[S_A * P::SS + j * P::SJ];
                fvv[j] = sy[S_B * P::SS + j * P::SJ];
                et[j] = sy[S_C * P::SS + j * P::SJ];
                u[j] = sy[S_D * P::SS + j * P::SJ];
                v[j] = sy[S_E * P::SS + j * P::SJ];
                H[j] = sy[S_F * P::SS + j * P::SJ];
            }
            TC d[n], aHu[n], aHv[n];
            dline<n>(D, fuv, d);
#pragma unroll
            for (int j = 0; j < n; ++j)
                aHu[j] = -d[j];
            d2line<n>(D, D2, u, d);
#pragma unroll
            for (int j = 0; j < n; ++j)
                aHu[j] += H[j] * (nu_h * d[j]);
            dline<n>(D, fvv, d);
#pragma unroll
            for (int j = 0; j < n; ++j)
                aHv[j] = -d[j];
            dline<n>(D, et, d);
#pragma unroll
            for (int j = 0; j < n; ++j)
                aHv[j] += (-g * H[j]) * d[j];
            d2line<n>(D, D2, v, d);
#pragma unroll
            for (int j = 0; j < n; ++j)
                aHv[j] += H[j] * (nu_h * d[j]);
#pragma unroll
            for (int j = 0; j < n; ++j) {
                sy[S_A * P::SS + j * P::SJ] = aHu[j];
                sy[S_B * P::SS + j * P::SJ] = aHv[j];
            }
        }
        __syncthreads();

        // ---------------- P3a: zeta-line (i, j) = L, momentum ----------------
        TC um[2][n]; // initial Hu, Hv for P4a
        if constexpr (step_reads_u0(EPI) && !LATE)
            load_fields<n, 0, 2, ADJ>(U, state_off<EPB>(U, b, e, L), um);
        {
            TC u[n], v[n], hi[n];
#pragma unroll
            for (int k = 0; k < n; ++k) {
                u[k] = sz[S_D * P::SS + k * P::SK];
                v[k] = sz[S_E * P::SS + k * P::SK];
                hi[k] = sz[S_G * P::SS + k * P::SK];
            }
            // vertical_diffusion :357-375: nu_v * d2/dzeta2 * Hinv
            TC d[n];
            d2line<n>(D, D2, u, d);
#pragma unroll
            for (int k = 0; k < n; ++k)
                sz[S_A * P::SS + k * P::SK] += nu_v * d[k] * hi[k];
            d2line<n>(D, D2, v, d);
#pragma unroll
            for (int k = 0; k < n; ++k)
                sz[S_B * P::SS + k * P::SK] += nu_v * d[k] * hi[k];
        }
        __syncthreads();

        // ---------------- P4a: xi-line again: momentum done, tracers staged ----------------
        TC pHT[n], pHS[n];
        {
            TC kv[2][n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                kv[0][i] = pHu[i] + sx[S_A * P::SS + i];
                kv[1][i] = pHv[i] + sx[S_B * P::SS + i];
            }
            if constexpr (step_reads_u0(EPI) && LATE)
                load_fields<n, 0, 2, ADJ, BY_FIELD>(U, state_off<EPB>(U, b, e, L), um);
            if constexpr (STEP)
                stage_update<n, 0, 2, EPI>(sc, kv, um, cur.q, acc);
            else
            {
                if constexpr (FACES)
                    add_faces<n, 0, 2>(kv, fa);
                write_fields<n, 0, 2, ADJ, NTS>(epi.R, state_off<EPB>(U, b, e, L), kv);
            }
            TC u[n], v[n], hi[n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                u[i] = sx[S_D * P::SS + i];
                v[i] = sx[S_E * P::SS + i];
                hi[i] = sx[S_G * P::SS + i];
            }
            // tracer_advection :377-393 along xi
            TC x[n], d[n];
#pragma unroll
            for (int i = 0; i < n; ++i)
                x[i] = u[i] * ht[i];
            dline<n>(D, x, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHT[i] = -d[i];
#pragma unroll
            for (int i = 0; i < n; ++i)
                x[i] = u[i] * hs[i];
            dline<n>(D, x, d);
#pragma unroll
            for (int i = 0; i < n; ++i)
                pHS[i] = -d[i];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                sx[S_A * P::SS + i] = v[i] * ht[i];
                sx[S_B * P::SS + i] = v[i] * hs[i];
                sx[S_C * P::SS + i] = ht[i] * hi[i];
                sx[S_D * P::SS + i] = hs[i] * hi[i];
            }
        }
        __syncthreads();

        // ---------------- P23b: eta-line and zeta-line, tracers ----------------
        // Both roles in one phase: the eta-owner reads and rewrites A, B along
        // its eta-line, the zeta-owner C, D along its zeta-line, so no two
        // threads touch the same node of the same slot.
        TC ut[3][n]; // initial eta, HT, HS for P4b
        if constexpr (step_reads_u0(EPI) && !LATE)
            load_fields<n, 2, 3, ADJ>(U, state_off<EPB>(U, b, e, L), ut);
        {
            TC ftv[n], fsv[n];
#pragma unroll
            for (int j = 0; j < n; ++j) {
                ftv[j] = sy[S_A * P::SS + j * P::SJ];
                fsv[j] = sy[S_B * P::SS + j * P::SJ];
            }
            TC dT[n], dS[n];
            dline<n>(D, ftv, dT);
            dline<n>(D, fsv, dS);
#pragma unroll
            for (int j = 0; j < n; ++j) {
                sy[S_A * P::SS + j * P::SJ] = -dT[j];
                sy[S_B * P::SS + j * P::SJ] = -dS[j];
            }
            TC T[n], S[n], hi[n];
#pragma unroll
            for (int k = 0; k < n; ++k) {
                T[k] = sz[S_C * P::SS + k * P::SK];
                S[k] = sz[S_D * P::SS + k * P::SK];
                hi[k] = sz[S_G * P::SS + k * P::SK];
            }
            TC d[n];
            d2line<n>(D, D2, T, d);
#pragma unroll
            for (int k = 0; k < n; ++k)
                sz[S_C * P::SS + k * P::SK] = kT * d[k] * hi[k];
            d2line<n>(D, D2, S, d);
#pragma unroll
            for (int k = 0; k < n; ++k)
                sz[S_D * P::SS + k * P::SK] = kS * d[k] * hi[k];
        }
        __syncthreads();

        // ---------------- P4b: xi-line: free surface and tracers done ----------------
        if constexpr (STEP)
            // for the next stage's P1, after the last one too: a branch here
            // keeps the old line alive (RK4, FP64, N = 4: 196 -> 381 us)
            load_h<n, TS, TC>(nxt, geo, e, L);
        {
            const int j0 = L % n, k0 = L / n;
            // eta tendency (:256-272): -(D_x2d HU_bar + D_y2d HV_bar), where the
            // 2D "x" index is j and the 2D "y" index is k.
            double s1 = 0.0, s2 = 0.0;
#pragma unroll
            for (int m = 0; m < n; ++m) {
                s1 += sDc[j0 * n + m] * bar[par][le][0][m + n * k0];
                s2 += sDc[k0 * n + m] * bar[par][le][1][j0 + n * m];
            }
            const TC deta = (TC)(-(s1 + s2));
            TC kv[3][n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                kv[0][i] = deta;
                kv[1][i] = (pHT[i] + sx[S_A * P::SS + i]) + sx[S_C * P::SS + i];
                kv[2][i] = (pHS[i] + sx[S_B * P::SS + i]) + sx[S_D * P::SS + i];
            }
            if constexpr (step_reads_u0(EPI) && LATE)
                load_fields<n, 2, 3, ADJ, BY_FIELD>(U, state_off<EPB>(U, b, e, L), ut);
            if constexpr (STEP)
                stage_update<n, 2, 3, EPI>(sc, kv, ut, cur.q, acc);
            else
            {
                if constexpr (FACES)
                    add_faces<n, 2, 3>(kv, fa);
                write_fields<n, 2, 3, ADJ, NTS>(epi.R, state_off<EPB>(U, b, e, L), kv);
            }
        }
        // No barrier here: this phase reads only its own line's slots and the
        // column integrals of this parity; the next P1 (of the next stage or
        // batch) writes its own line's slots and the other parity.
        par ^= 1;
        };
        if constexpr (STEP) {
#pragma unroll 1
            for (int st = 0; st < epi.nst; ++st)
                evaluate(st);
        } else if constexpr (ONE_TRIP) {
#pragma unroll 1
            for (int st = 0; st < 1; ++st)
                evaluate(st);
        } else {
            evaluate(0);
        }
        if constexpr (STEP)
            if (tid < C::NT && b * EPB + le < geo.E)
                write_fields<n, 0, 5, ADJ, false>(epi.R, state_off<EPB>(U, b, e, L0), cur.q);
    }
}

template <int n, class TC> KOps<n, TC> make_ops(const Ops &o)
{
    KOps<n, TC> r{};
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) {
            double s = 0.0;
            for (int m = 0; m < n; ++m)
                s += o.D[i * n + m] * o.D[m * n + j];
            r.D[i * n + j] = (TC)o.D[i * n + j];
            r.D2[i * n + j] = (TC)s;
            r.Dc[i * n + j] = o.D[i * n + j];
        }
    for (int i = 0; i < n; ++i)
        r.sw[i] = o.sw[i];
    return r;
}

inline int num_cus()
{
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess)
            cus = p.multiProcessorCount;
        if (cus <= 0)
            cus = 256;
    }
    return cus;
}

template <int N, class TS, class TC, int EPI, int LW, int FACES, bool ADJ>
hipError_t launch_ne(const VolGeom<TS> &geo, const Ops &ops, const Phys &ph, View<const TS> U,
                     const Epi<TS> &epi, hipStream_t s)
{
    using C = Cfg<N, LW>;
    if (geo.E <= 0)
        return hipSuccess;
    // blocked states: whole batches per block
    if (U.bb && U.bb % C::EPB != 0)
        return hipErrorInvalidValue;
    const int64_t nbatch = (geo.E + C::EPB - 1) / C::EPB;
    auto kern = volume_kernel<N, TS, TC, EPI, LW, FACES, ADJ>;
    // resident workgroups per CU (queried once per instantiation: the launch
    // path stays free of runtime queries)
    static const int per_cu = [&] {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, kern, C::BLOCK, 0) != hipSuccess ||
            v < 1)
            v = 1;
        return v;
    }();
    int64_t grid = nbatch;
    if (EPI == EPI_RHS) {
        // persistent workgroups: a few rounds per workgroup so the next batch's
        // loads overlap the current batch's arithmetic
        const int wpc = (geo.wg_per_cu > 0 && geo.wg_per_cu < per_cu) ? geo.wg_per_cu : per_cu;
        // what a requested shape amounts to, for the autotuner's report
        g_rhs_per_cu[sizeof(TS) == 8 ? 0 : 1][LW == 128 ? 0 : LW == 256 ? 1 : 2][N][FACES != FACES_NONE] =
            per_cu;
        grid = (int64_t)num_cus() * wpc;
        if (grid > nbatch)
            grid = nbatch;
    } else {
        // A step has nothing to prefetch: one batch per workgroup, so that the
        // hardware balances the last round, in whole rounds of the XCDs for the
        // batch order (against resident workgroups that loop: RK4 with 4 M
        // nodes, N = 4, FP64 196 and 219 us, FP32 100 and 114 us).  In FP64
        // from N = 6 the operators no longer fit the SGPRs and a workgroup's
        // start, which spills them, costs more than the imbalance: N = 6 424
        // one batch each, 400 us resident, N = 8 695 and 667 us.
        grid = (nbatch + kXcds - 1) / kXcds * kXcds;
        const int64_t resident = (int64_t)num_cus() * per_cu;
        if (sizeof(TS) == 8 && N >= 6 && grid > resident)
            grid = resident;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(C::BLOCK), 0, s, geo,
                       make_ops<N + 1, TC>(ops), ph, U, epi, nbatch);
    return hipGetLastError();
}

template <int N, class TS, class TC, int EPI, int LW, int FACES>
hipError_t launch_nl(const VolGeom<TS> &geo, const Ops &ops, const Phys &ph, View<const TS> U,
                     const Epi<TS> &epi, hipStream_t s)
{
    if (U.is == 1)
        return launch_ne<N, TS, TC, EPI, LW, FACES, true>(geo, ops, ph, U, epi, s);
    return launch_ne<N, TS, TC, EPI, LW, FACES, false>(geo, ops, ph, U, epi, s);
}

template <int N, class TS, class TC, int LW>
hipError_t launch_n(const VolGeom<TS> &geo, const Ops &ops, const Phys &ph, View<const TS> U,
                    const Epi<TS> &epi, hipStream_t s)
{
    if constexpr (N <= 4) // face plans are built for orders 1-4
        if (epi.mode == EPI_RHS && geo.faces.eface) {
            if (geo.faces.kind == DRF_FLUX_UPWIND)
                return launch_nl<N, TS, TC, EPI_RHS, LW, FACES_UPWIND>(geo, ops, ph, U, epi, s);
            return launch_nl<N, TS, TC, EPI_RHS, LW, FACES_LF>(geo, ops, ph, U, epi, s);
        }
    if (epi.mode == EPI_RHS)
        return launch_nl<N, TS, TC, EPI_RHS, LW, FACES_NONE>(geo, ops, ph, U, epi, s);
    if constexpr (LW == 128) // whole steps
        switch (epi.mode) {
        case EPI_STAGE: return launch_nl<N, TS, TC, EPI_STAGE, LW, FACES_NONE>(geo, ops, ph, U, epi, s);
        case EPI_SSP3: return launch_nl<N, TS, TC, EPI_SSP3, LW, FACES_NONE>(geo, ops, ph, U, epi, s);
        case EPI_RK4: return launch_nl<N, TS, TC, EPI_RK4, LW, FACES_NONE>(geo, ops, ph, U, epi, s);
        case EPI_LSRK: return launch_nl<N, TS, TC, EPI_LSRK, LW, FACES_NONE>(geo, ops, ph, U, epi, s);
        default: break;
        }
    return hipErrorInvalidValue;
}

// Orders above 4 run at 128 lines per workgroup only: their registers exceed
// what wider workgroups allow (256 VGPRs at two waves per SIMD).
template <class TS, class TC, int LW>
hipError_t dispatch(int order, const VolGeom<TS> &geo, const Ops &ops, const Phys &ph,
                    View<const TS> U, const Epi<TS> &epi, hipStream_t s)
{
    switch (order) {
    case 1: return launch_n<1, TS, TC, LW>(geo, ops, ph, U, epi, s);
    case 2: return launch_n<2, TS, TC, LW>(geo, ops, ph, U, epi, s);
    case 3: return launch_n<3, TS, TC, LW>(geo, ops, ph, U, epi, s);
    case 4: return launch_n<4, TS, TC, LW>(geo, ops, ph, U, epi, s);
    default: break;
    }
    if constexpr (LW == 128) {
        switch (order) {
        case 5: return launch_n<5, TS, TC, LW>(geo, ops, ph, U, epi, s);
        case 6: return launch_n<6, TS, TC, LW>(geo, ops, ph, U, epi, s);
        case 7: return launch_n<7, TS, TC, LW>(geo, ops, ph, U, epi, s);
        case 8: return launch_n<8, TS, TC, LW>(geo, ops, ph, U, epi, s);
        default: break;
        }
    }
    return hipErrorInvalidValue;
}

} // namespace vol
} // namespace drf
