// libedus_hip.so -- the MI355X engine of the EDUS time-stepping path.
//
// Device layout (all FP64):
//   * The density matrix is exactly Hermitian with a real diagonal at every step
//     of the reference's three steppers (the right-hand side is hermitised,
//     RungeKutta.h:283-294, and every update is a real-linear combination), so a
//     k point is stored packed: nb real diagonal entries, then (re, im) of the
//     strict upper triangle in row-major pair order -> nb*nb doubles.  This is
//     lossless and halves the HBM traffic of the reference's full complex arrays.
//   * nb <= 4: "SoA" -- element e of k at e*nkp + k (a lane per k and term, coalesced).
//     nb >= 5: "AoS" -- k-major, nb*nb contiguous doubles (32, 64 or 256 threads per k).
//   * H is packed like the state (upper triangle, as the RHS reads it);
//     D components are packed by their upper triangle, the lower one being D_ij
//     (symmetric tables) or conj(D_ij) (Hermitian tables); U is full complex.
//
// Kernels: fused RHS + stage update per RK4 stage / Adams-Bashforth step /
// Taylor step (RungeKutta.h:7-355, RungeKutta.cpp, Linear_Multistep_ODE_solvers.cpp,
// Taylor_DE_solver_deriv_Polynom.cpp), observables in one launch with
// error-compensated sums over the grid (Observables_MPI.h:217-775) and the Wannier phase
// contraction (Wannier.h:278-471).
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <complex>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../../include/edus.h"
#include "offsets.hpp"

namespace {

thread_local std::string g_err;

int set_err(int code, const std::string &m) {
    g_err = m;
    return code;
}

#define HIP_TRY(expr)                                                                                 \
    do {                                                                                              \
        hipError_t e_ = (expr);                                                                       \
        if (e_ != hipSuccess)                                                                         \
            return set_err(e_ == hipErrorOutOfMemory ? EDUS_ERR_NOMEM : EDUS_ERR_HIP,                \
                           std::string(#expr) + ": " + hipGetErrorString(e_));                       \
    } while (0)

enum Mode { RK1 = 0, RK2 = 1, RK3 = 2, RK4S = 3, ABM = 4, TAY = 5, RHSO = 6 };

constexpr int kMaxNbr = 64;
constexpr int kMaxTinv = (EDUS_MAX_ORDER - 1) * (EDUS_MAX_ORDER - 1);

// Per-context constants of the right-hand side.
struct ConstArgs {
    const double *H;     // packed (layout of the state)
    const double *D;     // 3 packed components (upper triangle; lower = D_ij or conj(D_ij), see dherm)
    const double *U;     // full complex AoS [k][nb][nb] (dissipation)
    const double *T;     // [nb][nb]
    const float *Hf, *Df, *Uf;  // mixed precision: H, D, U in FP32 (same layouts)
    const int *nbr;      // [n_nbr][nkp]
    const int *eidx;     // packed element e -> i | j << 8 | comp << 16 (wave layout)
    int nk, nkp, nb, nch, ncc, n_nbr, diss, dherm;  // dherm: D_ji = conj(D_ij) (else D_ji = D_ij)
    int hole;            // some filled band has T_vv != 0 (else the hole source is an exact zero and is not formed)
    int sw, scol;        // wave kernels: strip width and row length of the workgroup order (sw = 0: k order)
    // Wave kernels of one k per workgroup: pair = 1 when every pair of k (2q, 2q+1)
    // has the same stencil overlap (a uniform grid of even length along the
    // fastest axis); a workgroup then serves both and loads each shared
    // neighbour once.  pat[n] (n < n_nbr): the slot of 2q+1's stencil that is
    // 2q's slot n, or -1; pat[kMaxNbr + t] (t < npnew): 2q+1's slots found in
    // neither 2q's stencil nor 2q itself; pself: 2q+1's slot holding 2q, or -1.
    int pair, pself, npnew;
    const int *pat;
    double wx2;
};

// Per-launch stage data.  `tab` points at the stage's row of the field table:
// [0..2] pump sum, [3..5] half probe, [6..6+n_nbr) gradient coefficients
// c_n = sum_x E_pump[x] * w_shell b_n[x], [6+n_nbr] gradient flag.
struct StageArgs {
    const int *ctr;      // device step counter (field table path), or null: the row is `tab` itself
    long long ctr_stride;  // doubles per counted step of the field table
    const double *Y;     // stage input (neighbours gathered from it)
    const double *P0;    // RK: state at t_n
    double *ACC;         // RK: accumulator
    double *OUT;         // stage output
    double *HIST;        // AB/Taylor history slots
    const double *tab;
    int slot_out, order;
    int dmask;           // bit x: some field of the call has a nonzero x component (else D_x is not read)
    int pad1;
    int slots[EDUS_MAX_ORDER];
    double coef[EDUS_MAX_ORDER];
    double tinv[kMaxTinv];
    double dtp[EDUS_MAX_ORDER];
    double ca, cb, dt;
};

// The field-table row of a stage: `tab`, advanced by the device step counter when
// the launch belongs to a captured step (its arguments are fixed at capture, the
// counter moves on between replays).
// Read-only while any launch that reads it runs, so its (uniform) loads are scalar.
typedef const __attribute__((address_space(4))) double *TabRow;
__device__ __forceinline__ TabRow stage_row(const StageArgs &a) {
    return (TabRow)(a.ctr ? a.tab + (size_t)(*a.ctr) * (size_t)a.ctr_stride : a.tab);
}

// Pointers into device memory.  Those of a batch come from a table in memory, and
// the compiler would have to access through them with flat instructions, which
// also count as LDS traffic (8 bands, batch: every stage access).
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T *gm(const T *p) {
    return (const __attribute__((address_space(1))) T *)p;
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gm(T *p) {
    return (__attribute__((address_space(1))) T *)p;
}

// ---------------------------------------------------------------- complex helpers
struct cd {
    double x, y;
};
__device__ __forceinline__ cd mk(double a, double b) { return cd{a, b}; }
__device__ __forceinline__ cd cmul(cd a, cd b) { return cd{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ __forceinline__ cd cadd(cd a, cd b) { return cd{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ cd csub(cd a, cd b) { return cd{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ cd cconj(cd a) { return cd{a.x, -a.y}; }
__device__ __forceinline__ cd cscale(cd a, double s) { return cd{a.x * s, a.y * s}; }

// A double of another lane by data-parallel primitives: quad_perm, row mirrors.
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Halves (ROWS = 32) or odd and even 16-lane rows (16) of a wave added, in every lane
// as (lower + upper).
template <int ROWS>
__device__ __forceinline__ double swap_add(double v) {
    const unsigned long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    const auto l = ROWS == 32 ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false) : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = ROWS == 32 ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false) : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __longlong_as_double(((unsigned long long)h[0] << 32) | l[0]) + __longlong_as_double(((unsigned long long)h[1] << 32) | l[1]);
}

// Reductions over the 64 lanes of a wave (every lane gets the result; the order of
// the additions is fixed).  The sum runs on register moves inside rows of 16 lanes
// and on row swaps: six rounds of LDS permutes per value cost the observables of a
// small grid about 2 us.
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp64<0xB1>(v);   // lanes i, i ^ 1
    v += dpp64<0x4E>(v);   // i ^ 2
    v += dpp64<0x141>(v);  // the other four of eight lanes (half-row mirror: each four agree by now)
    v += dpp64<0x140>(v);  // the other eight of sixteen (row mirror)
    return swap_add<32>(swap_add<16>(v));
}
__device__ __forceinline__ double wave_min(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

// Single-precision complex for the mixed-precision stage (operators and LDS products).
struct cf {
    float x, y;
};
template <typename R> struct CplxOf;
template <> struct CplxOf<double> { using T = cd; };
template <> struct CplxOf<float> { using T = cf; };

// Block index remapped so that each of the 8 XCDs (which receive workgroups
// round-robin) works on one contiguous range of k: the 12-point gradient stencil
// then finds its neighbours in the XCD's own L2.
__device__ __forceinline__ int xcd_block() {
    const int G = gridDim.x, b = blockIdx.x;
    const int x = b & 7, idx = b >> 3, per = G >> 3, rem = G & 7;
    return x * per + min(x, rem) + idx;
}

// k of the wave kernels' workgroup L when the grid is walked in strips: the
// nk / scol rows of scol points (k = row * scol + col) are cut into strips of
// sw columns (the last one narrower if sw does not divide scol), and each strip
// is walked row by row.  A strip's rows then meet their stencil neighbours on
// the rows above and below while those are still in L2, where whole rows of
// large matrices would not fit.  A bijection of [0, nk); sw = 0 keeps k = L.
constexpr long long kStripL2Bytes = 1 << 20;

// 1..4 bands: above so many bytes of a stage (its neighbour table and kStageArrays states'
// worth of state, accumulator, base state, output, H and one component of D) the Infinity
// Cache (256 MB) no longer keeps them from one stage to the next, and the operators,
// accumulator and histories are read as non-temporal streams.
// RK4 step, plain and so: 4 bands 600 x 600 k (294 MB) 303 and 345 us, 3 bands 800 x 800
// (307 MB) 293 and 324, 1 band 2000 x 2000 (384 MB) 329 and 289, 3 bands 1000 x 1000 (480
// MB) 513 and 489.
constexpr int kStageArrays = 6;
constexpr double kStageCacheBytes = 340e6;

__device__ __forceinline__ int strip_k(int L, int nk, int sw, int scol) {
    if (sw == 0) return L;
    const int nrow = nk / scol, nfull = scol / sw, per = nrow * sw, s = L / per;
    if (s < nfull) {
        const int u = L - s * per;
        return (u / sw) * scol + s * sw + u % sw;
    }
    const int wr = scol - nfull * sw, u = L - nfull * per;
    return (u / wr) * scol + nfull * sw + u % wr;
}

// Pair index of (i<j) in row-major upper-triangle order.
__host__ __device__ __forceinline__ int pair_index(int i, int j, int nb) { return i * nb - i * (i + 1) / 2 + (j - i - 1); }

// Streaming accesses: operators, accumulators, histories and stage outputs are
// touched once per launch, so they bypass the caches' normal retention and leave
// L2 to the stage input, whose 12 stencil neighbours are re-read from it.  From 9
// bands on (plain ones: 16 bands 200 x 200 117 -> 127 us per stage, 32 bands 128 x
// 128 214 -> 228); below, a grid's arrays fit in the Infinity Cache, which
// non-temporal accesses pass by (8 bands 200 x 200, plain: 39.1 -> 35.1 us).
__device__ __forceinline__ double ldnt(const double *p) { return __builtin_nontemporal_load(gm(p)); }
__device__ __forceinline__ float ldnt(const float *p) { return __builtin_nontemporal_load(gm(p)); }
__device__ __forceinline__ void stnt(double *p, double v) { __builtin_nontemporal_store(v, gm(p)); }
__device__ __forceinline__ void stnt(float *p, float v) { __builtin_nontemporal_store(v, gm(p)); }

// Two adjacent packed elements in one access (16 bytes in FP64, 8 in FP32, at any
// element's alignment).  Halves the vector memory instructions of the wave kernels,
// whose address unit is their busiest memory stage.
// The pointers are cast to the pair type in one go: a template that deduces it (gm)
// would drop its alignment and promise 16 bytes.
template <typename T> struct Pair;
template <> struct Pair<double> { typedef double V __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct Pair<float> { typedef float V __attribute__((ext_vector_type(2), aligned(4))); };
template <bool NT, typename T>
__device__ __forceinline__ void ld2(const T *p, size_t o, T &a, T &b) {
    const auto *q = (const __attribute__((address_space(1))) typename Pair<T>::V *)(p + o);
    const typename Pair<T>::V v = NT ? __builtin_nontemporal_load(q) : *q;
    a = v.x;
    b = v.y;
}
template <bool NT, typename T>
__device__ __forceinline__ void st2(T *p, size_t o, T a, T b) {
    typename Pair<T>::V v;
    v.x = a;
    v.y = b;
    auto *q = (__attribute__((address_space(1))) typename Pair<T>::V *)(p + o);
    if (NT) __builtin_nontemporal_store(v, q);
    else *q = v;
}
// The elements at o0 and o1, in one access where they are neighbours (`vec`).
template <bool NT, typename T>
__device__ __forceinline__ void ld2_or_two(const T *p, size_t o0, size_t o1, bool vec, T &a, T &b) {
    if (vec) {
        ld2<NT>(p, o0, a, b);
    } else {
        a = NT ? ldnt(p + o0) : *gm(p + o0);
        b = NT ? ldnt(p + o1) : *gm(p + o1);
    }
}

// ---------------------------------------------------------------- stage update (nb >= 5)
// The Adams-Bashforth tail for the packed elements o0 and o0 + 1,
// history and state accessed as pairs; the order-1 history loads are issued
// together before the sum, which keeps the order of the coefficients.  h: stride
// between history slots.  S: storage type of the history (double, or float in the
// mixed form with FP32 stage storage); the state and its update stay FP64.
template <bool NT, typename S>
__device__ __forceinline__ void stage_update2_abm(const StageArgs &a, size_t o0, size_t h, double kv0,
                                                  double kv1, double y0, double y1) {
    S *const hist = reinterpret_cast<S *>(a.HIST);
    const size_t so = (size_t)a.slot_out * h;
    st2<NT>(hist, so + o0, (S)kv0, (S)kv1);
    double h0[5], h1[5];
#pragma unroll
    for (int s = 1; s < 5; s++) {
        h0[s] = h1[s] = 0.0;
        if (s < a.order) {
            const size_t sl = (size_t)a.slots[s] * h;
            S u0, u1;
            ld2<NT>(hist, sl + o0, u0, u1);
            h0[s] = (double)u0;
            h1[s] = (double)u1;
        }
    }
    double d0 = a.coef[0] * kv0, d1 = a.coef[0] * kv1;
#pragma unroll
    for (int s = 1; s < 5; s++)
        if (s < a.order) {
            d0 += a.coef[s] * h0[s];
            d1 += a.coef[s] * h1[s];
        }
    st2<NT>(a.OUT, o0, y0 + a.dt * d0, y1 + a.dt * d1);
}

// The Taylor tail for two adjacent packed elements: the history is read as
// pairs, then each element's update is formed on its own (one set of
// differences live at a time).
template <bool NT, typename S>
__device__ __forceinline__ void stage_update2_tay(const StageArgs &a, size_t o0, size_t h, double kv0,
                                                  double kv1, double y0, double y1) {
    S *const hist = reinterpret_cast<S *>(a.HIST);
    const size_t so = (size_t)a.slot_out * h;
    st2<NT>(hist, so + o0, (S)kv0, (S)kv1);
    const int n = a.order - 1;
    S u0[EDUS_MAX_ORDER - 1], u1[EDUS_MAX_ORDER - 1];
#pragma unroll
    for (int i = 0; i < EDUS_MAX_ORDER - 1; i++) {
        u0[i] = u1[i] = (S)0;
        if (i < n) {
            const size_t sl = (size_t)a.slots[i + 1] * h;
            ld2<NT>(hist, sl + o0, u0[i], u1[i]);
        }
    }
    double out[2];
#pragma unroll
    for (int w = 0; w < 2; w++) {
        const double kv = w ? kv1 : kv0;
        double dp[EDUS_MAX_ORDER];
#pragma unroll
        for (int i = 0; i < EDUS_MAX_ORDER - 1; i++) dp[i] = (i < n) ? kv - (double)(w ? u1[i] : u0[i]) : 0.0;
        double delta = kv * a.dt;
        for (int i = 1; i <= n; i++) {
            double al = 0.0;
            for (int q = 0; q < n; q++) al += a.tinv[(i - 1) * n + q] * dp[q];
            delta += (a.dtp[i] * al) / (double)(i + 1);
        }
        out[w] = (w ? y1 : y0) + delta;
    }
    st2<NT>(a.OUT, o0, out[0], out[1]);
}

// ================================================================ nb <= 4: a lane per k and term
// The right-hand side of a k is a sum of terms that only meet at the end: the
// commutator, the dephasing sandwich and the field drift.
// Each term of 64 k has a wave of its own (threadIdx.y: 0 the commutator, then the
// dephasing if the context has it, then the drift); the terms meet in LDS, and the
// waves share out the packed elements of the stage update, whose reads (accumulator,
// base state, histories) are requested with everything else at the start.
//
// What bounds it: on small grids one wave's own instruction stream and the latency
// of its dependent loads (a wave issues an FP64 instruction every 4 cycles, and 60 x
// 60 k are 57 waves on 1024 SIMDs), on large ones the loads in flight.  Two or three
// shorter streams side by side shorten both, and every term's registers leave room
// for more of them.  RK4 stage, one lane doing all of a k's terms -> this form: 3 bands
// 60 x 60 with dephasing 8.1 -> 4.8 us, 4 bands 251 x 307 34.2 -> 21.9; AB4 with the
// mean field 300 x 300 23.4 -> 19.3.  Loads are plain, but for U, while a stage's arrays
// stay in the Infinity Cache: as non-temporal ones they took the 4-band stage to 27.1 us.
// Six stencil rows in flight per wave instead of three took it to 25.9.
//
// DISS: the context has dephasing terms (c.diss).  NT: the arrays of a stage exceed the
// caches (kStageCacheBytes).
template <int NB, bool DISS>
struct SmallGeom {
    static constexpr int NP = NB * NB;
    static constexpr int GW = NB <= 2 ? 1 : 2;       // waves of the drift, a part of the stencil each
    static constexpr int R = 1 + (DISS ? 1 : 0) + GW;  // waves per 64 k
    static constexpr int EPR = (NP + R - 1) / R;     // packed elements of the update per wave
    static constexpr int GB = NB <= 2 ? 6 : 3;       // stencil rows in flight together
};
constexpr int kSmallMaxThreads = 512;
// waves per SIMD that the registers have to allow
template <int NB, int MODE, bool DISS>
constexpr int small_wpe() {
    if (MODE == TAY && NB == 2) return 4;  // up to seven histories per element
    return (NB <= 2 ? 5 : NB == 3 ? 4 : 3) - (DISS && NB > 2 ? 1 : 0);
}

// An element row of a SoA array at the lane's byte offset (SmallOff): the row address
// is uniform, so a 32-bit offset needs no address arithmetic in vector registers.
template <bool NT = false, typename O>
__device__ __forceinline__ double ldrow(const double *row, O off) {
    const double *p = reinterpret_cast<const double *>(reinterpret_cast<const char *>(row) + off);
    return NT ? ldnt(p) : *gm(p);
}
template <typename O>
__device__ __forceinline__ void strow_nt(double *row, O off, double v) {
    stnt(reinterpret_cast<double *>(reinterpret_cast<char *>(row) + off), v);
}

// Neighbour n of the lane's k.
template <typename O>
__device__ __forceinline__ int small_index(const ConstArgs &c, int n, O ko) {
    return *gm(reinterpret_cast<const int *>(reinterpret_cast<const char *>(c.nbr + (size_t)n * c.nkp) + ko / 2));
}

// Full P from its packed rows.
template <int NB>
__device__ __forceinline__ void small_state(const double *Y, size_t nkp, SmallOff<NB> ko, cd (&P)[NB][NB]) {
#pragma unroll
    for (int i = 0; i < NB; i++) {
        P[i][i] = mk(ldrow(Y + i * nkp, ko), 0.0);
#pragma unroll
        for (int j = i + 1; j < NB; j++) {
            const int p = NB + 2 * pair_index(i, j, NB);
            P[i][j] = mk(ldrow(Y + p * nkp, ko), ldrow(Y + (p + 1) * nkp, ko));
            P[j][i] = cconj(P[i][j]);
        }
    }
}

// -i[M, rho] in the transposed storage with M = H + E.D, the probe on core<->non-core
// elements, and the RWA term (RungeKutta.h:158-212), packed.
template <int NB, bool NT>
__device__ __forceinline__ void small_commutator(const ConstArgs &c, const StageArgs &a, TabRow tab, SmallOff<NB> ko,
                                                 double (&pv)[NB * NB]) {
    constexpr int NP = NB * NB;
    const size_t nkp = c.nkp;
    const double Ep[3] = {tab[0], tab[1], tab[2]}, Eq[3] = {tab[3], tab[4], tab[5]};
    cd P[NB][NB], M[NB][NB];
    small_state<NB>(a.Y, nkp, ko, P);
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = i; j < NB; j++) {
            const int p = i == j ? i : NB + 2 * pair_index(i, j, NB);
            M[i][j] = mk(ldrow<NT>(c.H + p * nkp, ko), i == j ? 0.0 : ldrow<NT>(c.H + (p + 1) * nkp, ko));
            if (i != j) M[j][i] = cconj(M[i][j]);
        }
#pragma unroll
    for (int x = 0; x < 3; x++)
        if (a.dmask >> x & 1) {
#pragma unroll
            for (int i = 0; i < NB; i++)
#pragma unroll
                for (int j = i; j < NB; j++) {
                    const bool w = (i >= c.nch && j < c.nch) || (i < c.nch && j >= c.nch);
                    const double E = w ? Eq[x] : Ep[x];
                    const int p = i == j ? i : NB + 2 * pair_index(i, j, NB);
                    const double *row = c.D + (size_t)(x * NP + p) * nkp;
                    const cd d = mk(ldrow<NT>(row, ko), i == j ? 0.0 : ldrow<NT>(row + nkp, ko));
                    M[i][j] = cadd(M[i][j], cscale(d, E));
                    if (i != j) M[j][i] = cadd(M[j][i], cscale(c.dherm ? cconj(d) : d, E));
                }
        }
#pragma unroll
    for (int i = 0; i < NB; i++) {
        cd beta = mk(0.0, 0.0);
#pragma unroll
        for (int j = 0; j < NB; j++) beta = cadd(beta, cmul(M[i][j], P[i][j]));
        pv[i] = 2. * beta.y;
    }
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = i + 1; j < NB; j++) {
            cd beta = mk(0.0, 0.0);
#pragma unroll
            for (int l = 0; l < NB; l++) beta = cadd(beta, csub(cmul(M[j][l], P[i][l]), cconj(cmul(M[i][l], P[j][l]))));
            cd v = mk(beta.y, -beta.x);                      // -i * beta
            if (i < c.nch && j >= c.nch) v = cadd(v, mk(-c.wx2 * P[i][j].y, c.wx2 * P[i][j].x));  // RWA term
            const int p = pair_index(i, j, NB);
            pv[NB + 2 * p] = v.x;
            pv[NB + 2 * p + 1] = v.y;
        }
}

// Dephasing in the eigenbasis (RungeKutta.h:219-254): the hole source minus
// conj(U) (T o (conj(U) P U^T)) conj(U), packed.
template <int NB>
__device__ __forceinline__ void small_dephasing(const ConstArgs &c, const double *Y, SmallOff<NB> ko, double (&pv)[NB * NB]) {
    cd P[NB][NB], U[NB][NB];
    const double *u = c.U + (size_t)(ko / 8) * NB * NB * 2;
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {  // one 16-byte load per complex entry (the k's U is 16-byte aligned)
            double re, im;
            ld2<true>(u, (i * NB + j) * 2, re, im);
            U[i][j] = mk(re, im);
        }
    small_state<NB>(Y, c.nkp, ko, P);
    cd G[NB][NB];
#pragma unroll
    for (int ib = 0; ib < NB; ib++) {
        cd t[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            t[i] = mk(0.0, 0.0);
#pragma unroll
            for (int j = 0; j < NB; j++) t[i] = cadd(t[i], cmul(U[ib][j], P[i][j]));
        }
#pragma unroll
        for (int ia = 0; ia < NB; ia++) {
            cd g = mk(0.0, 0.0);
#pragma unroll
            for (int i = 0; i < NB; i++) g = cadd(g, cmul(cconj(U[ia][i]), t[i]));
            G[ia][ib] = cscale(g, *gm(c.T + ia * NB + ib));
        }
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
        cd t[NB];
#pragma unroll
        for (int ia = 0; ia < NB; ia++) {
            t[ia] = mk(0.0, 0.0);
#pragma unroll
            for (int ib = 0; ib < NB; ib++) t[ia] = cadd(t[ia], cmul(G[ia][ib], cconj(U[ib][j])));
        }
#pragma unroll
        for (int i = 0; i <= j; i++) {
            cd w = mk(0.0, 0.0);
#pragma unroll
            for (int ia = 0; ia < NB; ia++) w = cadd(w, cmul(cconj(U[i][ia]), t[ia]));
            cd hole = mk(0.0, 0.0);
#pragma unroll
            for (int v = 0; v < NB; v++)  // static indices keep U in registers
                if (c.hole && v < c.ncc) hole = cadd(hole, cscale(cmul(cconj(U[v][j]), U[v][i]), *gm(c.T + v * NB + v)));
            if (i == j) {
                pv[i] = hole.x - w.x;
            } else {
                const int p = pair_index(i, j, NB);
                pv[NB + 2 * p] = hole.x - w.x;
                pv[NB + 2 * p + 1] = hole.y - w.y;
            }
        }
    }
}

// Field drift E.grad_k rho on the shell stencil (RungeKutta.h:258-276): the rows of
// neighbours n0..n1-1, GB at a time, all in flight; the sum keeps the stencil order.
// The first NPRE indices (`pre`) are requested by the caller.
template <int NB, int GB, int NPRE>
__device__ __forceinline__ void small_drift(const ConstArgs &c, const double *Y, TabRow tab, SmallOff<NB> ko, int n0, int n1,
                                            const int (&pre)[NPRE], double (&g)[NB * NB]) {
    constexpr int NP = NB * NB;
    static_assert(NPRE % GB == 0, "whole batches of requested indices");
    const size_t nkp = c.nkp;
    auto batch = [&](int n, const SmallOff<NB> (&off)[GB]) {
        double v[GB][NP];
#pragma unroll
        for (int j = 0; j < GB; j++)
#pragma unroll
            for (int e = 0; e < NP; e++) v[j][e] = ldrow(Y + e * nkp, off[j]);
#pragma unroll
        for (int j = 0; j < GB; j++)
            if (n + j < n1) {
                const double cn = tab[6 + n + j];
#pragma unroll
                for (int e = 0; e < NP; e++) g[e] += cn * v[j][e];
            }
    };
#pragma unroll
    for (int e = 0; e < NP; e++) g[e] = 0.0;
#pragma unroll
    for (int q = 0; q < NPRE; q += GB) {
        if (n0 + q >= n1) break;
        SmallOff<NB> off[GB];
#pragma unroll
        for (int j = 0; j < GB; j++) off[j] = small_offset<NB>(pre[q + j]);
        batch(n0 + q, off);
    }
    for (int n = n0 + NPRE; n < n1; n += GB) {
        SmallOff<NB> off[GB];
#pragma unroll
        for (int j = 0; j < GB; j++) off[j] = small_offset<NB>(small_index(c, min(n + j, n1 - 1), ko));
        batch(n, off);
    }
}

// What the update of a packed element reads besides the right-hand side.
template <int MODE>
struct SmallTail {
    static constexpr int NH = MODE == ABM ? 4 : MODE == TAY ? EDUS_MAX_ORDER - 1 : 0;
    double y, p0, p1, h[NH > 0 ? NH : 1];
};

template <int MODE, bool NT, typename O>
__device__ __forceinline__ void small_tail_load(const StageArgs &a, size_t row, size_t hstride, O ko, SmallTail<MODE> &t) {
    t.y = t.p0 = t.p1 = 0.0;
    if constexpr (MODE == RK1 || MODE == ABM || MODE == TAY) t.y = ldrow(a.Y + row, ko);
    if constexpr (MODE == RK2 || MODE == RK3 || MODE == RK4S) t.p0 = ldrow<NT>(a.ACC + row, ko);
    if constexpr (MODE == RK2 || MODE == RK3) t.p1 = ldrow<NT>(a.P0 + row, ko);
#pragma unroll
    for (int s = 0; s < SmallTail<MODE>::NH; s++)
        t.h[s] = s + 1 < a.order ? ldrow<NT>(a.HIST + (size_t)a.slots[s + 1] * hstride + row, ko) : 0.0;
}

template <int MODE, typename O>
__device__ __forceinline__ void small_tail_store(const StageArgs &a, size_t row, size_t hstride, O ko, double kv, const SmallTail<MODE> &t) {
    if constexpr (MODE == RK1) {
        strow_nt(a.ACC + row, ko, t.y + kv * a.ca);
        strow_nt(a.OUT + row, ko, t.y + kv * a.cb);
    } else if constexpr (MODE == RK2 || MODE == RK3) {
        strow_nt(a.ACC + row, ko, t.p0 + kv * a.ca);
        strow_nt(a.OUT + row, ko, t.p1 + kv * a.cb);
    } else if constexpr (MODE == RK4S) {
        strow_nt(a.OUT + row, ko, t.p0 + kv * a.ca);
    } else if constexpr (MODE == ABM) {
        strow_nt(a.HIST + (size_t)a.slot_out * hstride + row, ko, kv);
        double delta = a.coef[0] * kv;
#pragma unroll
        for (int s = 1; s < 5; s++)
            if (s < a.order) delta += a.coef[s] * t.h[s - 1];
        strow_nt(a.OUT + row, ko, t.y + a.dt * delta);
    } else if constexpr (MODE == TAY) {
        strow_nt(a.HIST + (size_t)a.slot_out * hstride + row, ko, kv);
        const int n = a.order - 1;
        double dp[EDUS_MAX_ORDER];
#pragma unroll
        for (int i = 0; i < EDUS_MAX_ORDER - 1; i++) dp[i] = (i < n) ? kv - t.h[i] : 0.0;
        double delta = kv * a.dt;
        for (int i = 1; i <= n; i++) {
            double al = 0.0;
#pragma unroll
            for (int p = 0; p < EDUS_MAX_ORDER - 1; p++)
                if (p < n) al += a.tinv[(i - 1) * n + p] * dp[p];
            delta += (a.dtp[i] * al) / (double)(i + 1);
        }
        strow_nt(a.OUT + row, ko, t.y + delta);
    } else {
        strow_nt(a.OUT + row, ko, kv);
    }
}

// kk: the lane's k (past the grid: clamped, nothing stored); lk, tk: its place among
// the workgroup's tk k; term: threadIdx.y, uniform in a wave; lds: [R][NP][tk].
template <int NB, int MODE, bool DISS, bool NT>
__device__ __forceinline__ void stage_small(const ConstArgs &c, const StageArgs &a, TabRow tab, const int kk, const int lk, const int tk, const int term,
                                            double *lds) {
    using G = SmallGeom<NB, DISS>;
    constexpr int NP = G::NP, R = G::R, EPR = G::EPR;
    const bool store = kk < c.nk;
    const SmallOff<NB> ko = small_offset<NB>(min(kk, c.nk - 1));
    const size_t nkp = c.nkp;
    const int nn = c.n_nbr;
    SmallTail<MODE> tail[EPR];
    auto load_tail = [&] {
#pragma unroll
        for (int m = 0; m < EPR; m++)
            if (term + R * m < NP) small_tail_load<MODE, NT>(a, (size_t)(term + R * m) * nkp, NP * nkp, ko, tail[m]);
    };
    // At 4 bands the Taylor step's histories do not fit beside the terms' registers:
    // they are requested behind them (600 x 600 k, without dephasing: 187 us spilling,
    // 110 so, 169 with one lane doing all of a k's terms).
    constexpr bool kLateTail = MODE == TAY && NB == 4;
    if constexpr (!kLateTail) load_tail();
    double pv[NP];
    if (term == 0) small_commutator<NB, NT>(c, a, tab, ko, pv);
    else if (DISS && term == 1) small_dephasing<NB>(c, a.Y, ko, pv);
    else if (nn > 0) {
        // this wave's part of the stencil; its indices come with the field row, not
        // after the row has told whether the drift is on
        constexpr int NPRE = 12 / G::GW;
        const int q = term - (R - G::GW), n0 = nn * q / G::GW, n1 = nn * (q + 1) / G::GW;
        int pre[NPRE];
#pragma unroll
        for (int n = 0; n < NPRE; n++) pre[n] = small_index(c, min(n0 + n, nn - 1), ko);
        if (tab[6 + nn] != 0.0) {
            small_drift<NB, G::GB, NPRE>(c, a.Y, tab, ko, n0, n1, pre, pv);
        } else {
#pragma unroll
            for (int e = 0; e < NP; e++) pv[e] = 0.0;
        }
    } else {
#pragma unroll
        for (int e = 0; e < NP; e++) pv[e] = 0.0;
    }
#pragma unroll
    for (int e = 0; e < NP; e++) lds[(term * NP + e) * tk + lk] = pv[e];
    if constexpr (kLateTail) load_tail();
    __syncthreads();
    if (!store) return;
#pragma unroll
    for (int m = 0; m < EPR; m++) {
        const int e = term + R * m;
        if (e < NP) {
            double kv = lds[e * tk + lk], g = lds[((R - G::GW) * NP + e) * tk + lk];
            if constexpr (DISS) kv += lds[(NP + e) * tk + lk];
            if constexpr (G::GW == 2) g += lds[((R - 1) * NP + e) * tk + lk];
            kv += g;
            small_tail_store<MODE>(a, (size_t)e * nkp, NP * nkp, ko, kv, tail[m]);
        }
    }
}

// blockDim = (k per workgroup, SmallGeom::R)
template <int NB, int MODE, bool DISS, bool NT>
__global__ __launch_bounds__(kSmallMaxThreads, (small_wpe<NB, MODE, DISS>())) void k_stage_small(ConstArgs c, StageArgs a) {
    extern __shared__ __align__(16) double smem_d[];
    const int term = __builtin_amdgcn_readfirstlane(threadIdx.y);
    stage_small<NB, MODE, DISS, NT>(c, a, stage_row(a), xcd_block() * blockDim.x + threadIdx.x, threadIdx.x, blockDim.x, term, smem_d);
}

// ================================================================ Coulomb mean field
// P in the eigenbasis for the Coulomb_diag_basis form (get_P_in_dia_vect,
// InitParameters.h:264-335): PD = conj(U) P U^T per k in the transposed storage,
// diagonal real, packed like the state (thread per k, nb <= 4).
template <int NB>
__global__ __launch_bounds__(256) void k_coul_pdiag(const double *__restrict__ Y, const double *__restrict__ Uall, int nk, int nkp,
                                                    double *__restrict__ PD) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nk) return;
    cd P[NB][NB], U[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        P[i][i] = mk(Y[(size_t)i * nkp + k], 0.0);
#pragma unroll
        for (int j = i + 1; j < NB; j++) {
            const int p = pair_index(i, j, NB);
            P[i][j] = mk(Y[(size_t)(NB + 2 * p) * nkp + k], Y[(size_t)(NB + 2 * p + 1) * nkp + k]);
            P[j][i] = cconj(P[i][j]);
        }
    }
    const double *uk = Uall + (size_t)k * NB * NB * 2;
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) U[i][j] = mk(uk[(i * NB + j) * 2], uk[(i * NB + j) * 2 + 1]);
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int b = a; b < NB; b++) {
            cd acc = mk(0.0, 0.0);
#pragma unroll
            for (int i = 0; i < NB; i++) {
                cd t = mk(0.0, 0.0);
#pragma unroll
                for (int j = 0; j < NB; j++) t = cadd(t, cmul(P[i][j], U[b][j]));
                acc = cadd(acc, cmul(cconj(U[a][i]), t));
            }
            if (a == b) {
                PD[(size_t)a * nkp + k] = acc.x;
            } else {
                const int p = pair_index(a, b, NB);
                PD[(size_t)(NB + 2 * p) * nkp + k] = acc.x;
                PD[(size_t)(NB + 2 * p + 1) * nkp + k] = acc.y;
            }
        }
}

// Separable partial 2D Fourier sums of the packed state over the grid
// k = (i1, i2) (Coulomb.h:273-350):
//   S_y[i1][n][e] = sum_i2 y_n(i2) P_e(i1, i2)                     (y = cos, sin)
//   F_xy[mm][e]   = w (1 + corr_mn) sum_i1 x_m(i1) S_y[i1][n][e]    (4 combinations)
// then X_mn from A..D minus the equilibrium (Coulomb.h:413-470), the column sums of
// the reconstruction and its row sum with the renormalised H (Coulomb.h:510-541).
struct CoulArgs {
    const double *Y;
    int nk, nkp, nb, NP, N1, N2, ncut, nu;
    double w;
    const double *cxm, *sxm, *cyn, *syn;
    double *S;
    double *X;                 // [4][ncut^2][nb][nb] complex
    const double *X0;
    const double *A, *B, *C, *D, *vh;  // complex
    double *EH;
    const double *EH0;
    double *Tt;                // [2][ncut][nu][N2] complex
    double *Xw;                // [2 nu][nkp]: mean-field matrix per k (upper elements, re/im; diagonal basis)
};
// The peak correction is on once a band holds carriers (RungeKutta.h:69-138).
__host__ __device__ __forceinline__ bool mean_field_gate(double n_cond) { return n_cond > 1e-20; }
// What the renormalised H takes besides: bare H, U, the equilibrium state, the peak
// correction and its gate.
struct CoulHArgs {
    const double *H, *U, *PW0, *screen;
    double *Hr;
    double n_cond;
};

constexpr int kCoulThreads = 256;

// S_y[i1][n][e] = sum_i2 y_n(i2) P_e(i1, i2) as one product on the FP64 matrix
// cores (a thread per output with a sequential sum took 28 us at 300 x 300,
// bound by the address throughput of its uncoalesced loads): rows r = e N1 + i1
// (the state row Y[e][i1 N2 + i2], contiguous in i2), columns c = q ncut + n
// (q = 0: cos, 1: sin), K = N2.  One workgroup per 16 x 16 tile; its four waves take
// a quarter of K each and are added in wave order.  A wave walks its quarter four k at
// a time with v_mfma_f64_16x16x4f64 (lane l feeds A[row l%16][k l/16] and
// B[k l/16][col l%16] and ends with C[l/16 + 4 i][l%16]); out-of-range rows,
// columns and k are fed zeros.  The pass waits for its loads: one wave per tile with 16
// of them in flight took 13.8 us at 300 x 300, this form 11.1.
__global__ __launch_bounds__(256) void k_coul_s1_mfma(CoulArgs a) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    constexpr int KB = 12;  // k slices of four whose loads are in flight together
    __shared__ double red[3][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r0 = blockIdx.x * 16, c0 = blockIdx.y * 16;
    const int nrow = a.NP * a.N1, ncol = 2 * a.ncut;
    const int ra = r0 + (lane & 15), cb = c0 + (lane & 15), kq = lane >> 4;
    const bool rok = ra < nrow, cok = cb < ncol;
    const double *yrow = a.Y + (rok ? (size_t)(ra / a.N1) * a.nkp + (size_t)(ra % a.N1) * a.N2 : 0);
    const int q = cok ? cb / a.ncut : 0, n = cok ? cb % a.ncut : 0;
    const double *trig = (q ? a.syn : a.cyn) + (size_t)n * a.N2;
    const int per = ((a.N2 + 15) / 16) * 4, kbeg = wave * per, kend = min(a.N2, kbeg + per);
    v4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = kbeg; k0 < kend; k0 += 4 * KB) {
        double yv[KB], tv[KB];
#pragma unroll
        for (int u = 0; u < KB; u++) {
            const int kc = min(k0 + 4 * u + kq, a.N2 - 1);
            yv[u] = yrow[kc];
            tv[u] = trig[kc];
        }
#pragma unroll
        for (int u = 0; u < KB; u++) {
            const bool kok = k0 + 4 * u + kq < kend;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((rok && kok) ? yv[u] : 0.0, (cok && kok) ? tv[u] : 0.0, acc, 0, 0, 0);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) red[wave - 1][i][lane] = acc[i];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = r0 + (lane >> 4) + 4 * i, c = c0 + (lane & 15);
        if (r < nrow && c < ncol) {
            const int e = r / a.N1, i1 = r % a.N1, qq = c / a.ncut, nn = c % a.ncut;
            a.S[(((size_t)qq * a.N1 + i1) * a.ncut + nn) * a.NP + e] = ((acc[i] + red[0][i][lane]) + red[1][i][lane]) + red[2][i][lane];
        }
    }
}

// F_xy[mm][e] = w (1 + corr_mn) sum_i1 x_m(i1) S_y[i1][n][e]: one workgroup per
// mm; thread t takes element e = t % NP and every (256/NP)-th term of the sum,
// and the parts are added in a fixed tree per element (10.0 -> 8.6 us at 300 x 300).
// The same workgroup then forms X_mn from its F (coul_x_elem) and, for mm = 0, the Hartree shift: X_mn
// needs no other mode's F, so no launch of its own.
constexpr int kCoulMaxNP = 16;  // the mean field runs at nb <= 4

__device__ __forceinline__ void coul_x_elem(const CoulArgs &a, const double (*Fs)[kCoulMaxNP], int mm, int u);

__global__ __launch_bounds__(kCoulThreads) void k_coul_s2(CoulArgs a) {
    __shared__ double red[4][kCoulThreads];
    __shared__ double Fs[4][kCoulMaxNP];
    const int mm = blockIdx.x, m = mm / a.ncut, n = mm % a.ncut, t = threadIdx.x;
    const int NP = a.NP, nparts = kCoulThreads / NP, e = t % NP, part = t / NP;
    double cc = 0, cs = 0, sc = 0, ss = 0;
    if (part < nparts) {
#pragma unroll 4
        for (int i1 = part; i1 < a.N1; i1 += nparts) {
            const double xc = a.cxm[m * a.N1 + i1], xs = a.sxm[m * a.N1 + i1];
            const double yc = a.S[(((size_t)0 * a.N1 + i1) * a.ncut + n) * NP + e];
            const double ys = a.S[(((size_t)1 * a.N1 + i1) * a.ncut + n) * NP + e];
            cc += xc * yc;
            cs += xc * ys;
            sc += xs * yc;
            ss += xs * ys;
        }
    }
    red[0][t] = cc;
    red[1][t] = cs;
    red[2][t] = sc;
    red[3][t] = ss;
    // the parts in a fixed tree (one after the other they took half of the pass)
    int h = 1;
    while (h < nparts) h *= 2;
    for (h /= 2; h > 0; h /= 2) {
        __syncthreads();
        if (part < h && part + h < nparts) {
#pragma unroll
            for (int qd = 0; qd < 4; qd++) red[qd][t] += red[qd][t + h * NP];
        }
    }
    __syncthreads();
    if (t < 4 * NP) {
        const double corr = -4 * M_PI * M_PI * (m * m + n * n) / ((double)a.nk * 27);
        const double f = a.w * (1. + corr);
        const int qd = t / NP, el = t % NP;
        Fs[qd][el] = red[qd][el] * f;
    }
    __syncthreads();
    if (mm == 0 && t < a.nb) {  // Hartree shift from mode 0 (Coulomb.h:385-410)
        double e = 0.;
        for (int jc = 0; jc < a.nb; jc++) e += Fs[0][jc] * a.vh[2 * (t * a.nb + jc)];
        a.EH[t] = e - a.EH0[t];
    }
    if (t < a.nu) coul_x_elem(a, Fs, mm, t);
}

// X_mn for upper element u of mode mm from the mode's F (Coulomb.h:413-470).
__device__ __forceinline__ void coul_x_elem(const CoulArgs &a, const double (*Fs)[kCoulMaxNP], int mm, int u) {
    const int nb = a.nb, nmm = a.ncut * a.ncut, nb2 = nb * nb;
    int i = 0, j = 0;
    for (int q = u, r = 0; ; r++) {
        if (q < nb - r) { i = r; j = r + q; break; }
        q -= nb - r;
    }
    auto fget = [&](int qd) -> cd {
        const double *F = Fs[qd];
        if (i == j) return mk(F[i], 0.0);
        const int p = pair_index(i, j, nb);
        return mk(F[nb + 2 * p], F[nb + 2 * p + 1]);
    };
    const cd fcc = fget(0), fcs = fget(1), fsc = fget(2), fss = fget(3);
    const int d = i * nb + j, od = j * nb + i;
    const size_t base = (size_t)mm * nb2;
    const cd *A = reinterpret_cast<const cd *>(a.A), *B = reinterpret_cast<const cd *>(a.B);
    const cd *C = reinterpret_cast<const cd *>(a.C), *D = reinterpret_cast<const cd *>(a.D);
    const cd *X0 = reinterpret_cast<const cd *>(a.X0);
    cd *X = reinterpret_cast<cd *>(a.X);
    const cd Amn = A[base + (i == j ? 0 : d)], Dmn = D[base + (i == j ? 0 : d)];
    cd xcc = csub(cadd(cmul(Amn, fcc), cmul(Dmn, fss)), X0[0 * (size_t)nmm * nb2 + base + d]);
    cd xcs = csub(csub(cmul(Amn, fcs), cmul(Dmn, fsc)), X0[1 * (size_t)nmm * nb2 + base + d]);
    cd xsc = csub(csub(cmul(Amn, fsc), cmul(Dmn, fcs)), X0[2 * (size_t)nmm * nb2 + base + d]);
    cd xss = csub(cadd(cmul(Amn, fss), cmul(Dmn, fcc)), X0[3 * (size_t)nmm * nb2 + base + d]);
    if (i != j) {
        const cd Bmn = B[base + d], Cmn = C[base + d];
        xcc = cadd(xcc, cadd(cmul(Bmn, fcs), cmul(Cmn, fsc)));
        xcs = cadd(xcs, csub(cmul(Cmn, fss), cmul(Bmn, fcc)));
        xsc = cadd(xsc, csub(cmul(Bmn, fss), cmul(Cmn, fcc)));
        xss = csub(xss, cadd(cmul(Bmn, fsc), cmul(Cmn, fcs)));
        X[0 * (size_t)nmm * nb2 + base + od] = cconj(xcc);
        X[1 * (size_t)nmm * nb2 + base + od] = cconj(xcs);
        X[2 * (size_t)nmm * nb2 + base + od] = cconj(xsc);
        X[3 * (size_t)nmm * nb2 + base + od] = cconj(xss);
    }
    X[0 * (size_t)nmm * nb2 + base + d] = xcc;
    X[1 * (size_t)nmm * nb2 + base + d] = xcs;
    X[2 * (size_t)nmm * nb2 + base + d] = xsc;
    X[3 * (size_t)nmm * nb2 + base + d] = xss;
}

// Column sums of the reconstruction for upper element u = (i <= j), which reads
// (X_mn)_{ji} because the reference stores X_{jc,ic} (Coulomb.h:537).
__global__ __launch_bounds__(64) void k_coul_s3(CoulArgs a) {
    const int nb = a.nb, nmm = a.ncut * a.ncut, nb2 = nb * nb;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.N2 * a.ncut * a.nu) return;
    const int i2 = t % a.N2, u = (t / a.N2) % a.nu, m = t / (a.N2 * a.nu);
    int i = 0, j = 0;
    for (int q = u, r = 0; ; r++) {
        if (q < nb - r) { i = r; j = r + q; break; }
        q -= nb - r;
    }
    const cd *X = reinterpret_cast<const cd *>(a.X);
    cd tc = mk(0, 0), ts = mk(0, 0);
    constexpr int NBLK = 10;  // of 4: 6.6 us at 300 x 300, of 10 5.7
    // n in blocks of NBLK: the block's loads (at a clamped n) are issued together,
    // the sums keep the order of n.
    for (int n0 = 0; n0 < a.ncut; n0 += NBLK) {
        cd xv[NBLK][4];
        double ycv[NBLK], ysv[NBLK];
#pragma unroll
        for (int b = 0; b < NBLK; b++) {
            const int n = min(n0 + b, a.ncut - 1);
            const size_t d = (size_t)(m * a.ncut + n) * nb2 + j * nb + i;
#pragma unroll
            for (int qd = 0; qd < 4; qd++) xv[b][qd] = X[qd * (size_t)nmm * nb2 + d];
            ycv[b] = a.cyn[n * a.N2 + i2];
            ysv[b] = a.syn[n * a.N2 + i2];
        }
#pragma unroll
        for (int b = 0; b < NBLK; b++)
            if (n0 + b < a.ncut) {
                tc = cadd(tc, cadd(cscale(xv[b][0], ycv[b]), cscale(xv[b][1], ysv[b])));
                ts = cadd(ts, cadd(cscale(xv[b][2], ycv[b]), cscale(xv[b][3], ysv[b])));
            }
    }
    cd *T = reinterpret_cast<cd *>(a.Tt);
    T[(((size_t)0 * a.ncut + m) * a.nu + u) * a.N2 + i2] = tc;
    T[(((size_t)1 * a.ncut + m) * a.nu + u) * a.N2 + i2] = ts;
}

// Renormalised H of every k from the column sums (Coulomb.h:510-541, RungeKutta.h:69-138):
// X_W(i1, i2)_u = -sum_m [cos_m(i1) Tc(m, u, i2) + sin_m(i1) Ts(m, u, i2)] formed as
// products on the FP64 matrix cores, A[i1][kk] = [cos_m(i1) | sin_m(i1)] and
// B[kk][c] = [Tc(m, u, i2) ; Ts(m, u, i2)] (K = 2 Ncut), rows i1, one wave per 16 x
// 16 tile, its K loads issued before the products (lane l feeds A[row l%16][kk l/16]
// and B[kk l/16][col l%16] and ends with C[l/16 + 4 i][l%16]).
// Wannier basis (FULL): columns c = e N2 + i2 over the packed elements e, and the
// tile's lanes go on to Hr = H + X_W, minus Screen_const * (P - P0)_{ji} when n_cond >
// 1e-20, real diagonal, plus the Hartree shift: the stage kernel then reads Hr like
// any H.  (Storing X_W and forming Hr in the stage kernel moved 42 instead of 36
// doubles per k at 3 bands and cost the stage its registers: 300 x 300 AB4, stage
// 29.7 + this pass 10.0 us -> 23.4 + 12.3.)
// Diagonal basis: columns c = (2u + re/im) N2 + i2, stored as Xw[2u + re/im][k].
template <bool FULL>
__global__ __launch_bounds__(64) void k_coul_w_mfma(CoulArgs a, CoulHArgs h) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    constexpr int KB = 40;  // K terms loaded per block (2 Ncut <= 64)
    const int lane = threadIdx.x, r0 = blockIdx.x * 16, c0 = blockIdx.y * 16, nb = a.nb;
    const int ncut = a.ncut, K = 2 * ncut, ncol = (FULL ? a.NP : 2 * a.nu) * a.N2, N1 = a.N1;
    const int ra = r0 + (lane & 15), cb = c0 + (lane & 15), kq = lane >> 4;
    const bool rok = ra < N1, cok = cb < ncol;
    const int i1 = rok ? ra : 0, uc = cok ? cb / a.N2 : 0, i2 = cok ? cb % a.N2 : 0;
    // column -> upper element (bi <= bj) and component
    int bi = 0, bj = 0, ri = 0, u = 0;
    if (FULL && uc < nb) {
        bi = bj = uc;
    } else {
        ri = FULL ? (uc - nb) & 1 : uc & 1;
        int q = FULL ? (uc - nb) >> 1 : uc >> 1;
        const int d = FULL ? 1 : 0;  // pairs i < j, or i <= j
        while (q >= nb - bi - d) q -= nb - bi++ - d;
        bj = bi + d + q;
    }
    u = bi * nb - bi * (bi - 1) / 2 + bj - bi;
    // the tile's own operands are in flight during the products
    const bool diag = bi == bj, scr = FULL && mean_field_gate(h.n_cond);
    double hv[4], pr[4], pi[4];
    if constexpr (FULL) {
        const int p = diag ? bi : nb + 2 * pair_index(bi, bj, nb);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t k = (size_t)min(r0 + (lane >> 4) + 4 * i, N1 - 1) * a.N2 + i2;
            hv[i] = h.H[(size_t)uc * a.nkp + k];
            pr[i] = pi[i] = 0.0;
            if (scr) {
                const size_t o = (size_t)p * a.nkp + k, o1 = diag ? o : o + a.nkp;
                pr[i] = a.Y[o] - h.PW0[o];
                pi[i] = diag ? 0.0 : a.Y[o1] - h.PW0[o1];
            }
        }
    }
    v4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < K; k0 += KB) {
        double av[KB / 4], bv[KB / 4];
#pragma unroll
        for (int b = 0; b < KB / 4; b++) {
            const int kk = min(k0 + 4 * b + kq, K - 1), q = kk >= ncut, m = kk - q * ncut;
            av[b] = (q ? a.sxm : a.cxm)[m * N1 + i1];
            bv[b] = a.Tt[((((size_t)q * ncut + m) * a.nu + u) * a.N2 + i2) * 2 + ri];
        }
#pragma unroll
        for (int b = 0; b < KB / 4; b++) {
            const bool kok = k0 + 4 * b + kq < K;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((rok && kok) ? av[b] : 0.0, (cok && kok) ? bv[b] : 0.0, acc, 0, 0, 0);
        }
    }
    if (!cok) return;
    if constexpr (!FULL) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = r0 + (lane >> 4) + 4 * i;
            if (r < N1) a.Xw[(size_t)uc * a.nkp + (size_t)r * a.N2 + i2] = -acc[i];
        }
    } else {
        const int idx = diag ? 0 : bi * nb + bj;
        const cd s = mk(h.screen[2 * idx], -h.screen[2 * idx + 1]);  // conj(Screen_const)
        const double eh = diag ? a.EH[bi] : 0.0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = r0 + (lane >> 4) + 4 * i;
            if (r >= N1) continue;
            // (P - P0)_{ji} = conj((P - P0)_{ij})
            const cd x = cmul(s, mk(pr[i], -pi[i]));
            h.Hr[(size_t)uc * a.nkp + (size_t)r * a.N2 + i2] = hv[i] + (-acc[i] - (ri ? x.y : x.x)) + eh;
        }
    }
}

// Diagonal basis (RungeKutta.h:97-124): X_d from the sums over PD, minus
// Screen_const[0][0] (PD - P_Bloch_0) on the diagonal (P_Bloch_0: the filled bands)
// and conj(Screen_const[0][1]) PD_ji off it; back to the orbital basis as U^+ X_d U
// (InitParameters.h:340-370), real diagonal plus the Hartree shift.  Thread per k.
template <int NB>
__global__ __launch_bounds__(256) void k_coul_hdiag(CoulArgs a, CoulHArgs h, int ncc) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nk) return;
    const size_t nkp = a.nkp;
    const double *PD = a.Y;
    cd Xd[NB][NB], U[NB][NB];
    const double *uk = h.U + (size_t)k * NB * NB * 2;
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            double re, im;
            ld2<false>(uk, (i * NB + j) * 2, re, im);
            U[i][j] = mk(re, im);
        }
    const cd scr0 = mk(h.screen[0], h.screen[1]), scr1c = mk(h.screen[2], -h.screen[3]);
    int u = 0;
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = i; j < NB; j++, u++) {
            cd xk = mk(a.Xw[(size_t)(2 * u) * nkp + k], a.Xw[(size_t)(2 * u + 1) * nkp + k]);
            if (i == j) {
                Xd[i][i] = csub(xk, cscale(scr0, PD[i * nkp + k] - (i < ncc ? 1.0 : 0.0)));
            } else {
                const int p = pair_index(i, j, NB);
                // PD_ji = conj(PD_ij)
                const cd pdji = mk(PD[(NB + 2 * p) * nkp + k], -PD[(NB + 2 * p + 1) * nkp + k]);
                xk = csub(xk, cmul(scr1c, pdji));
                Xd[i][j] = xk;
                Xd[j][i] = cconj(xk);
            }
        }
    cd T1[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            cd t = mk(0.0, 0.0);
#pragma unroll
            for (int l = 0; l < NB; l++) t = cadd(t, cmul(Xd[i][l], U[l][j]));
            T1[i][j] = t;
        }
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = i; j < NB; j++) {
            cd xw = mk(0.0, 0.0);
#pragma unroll
            for (int l = 0; l < NB; l++) xw = cadd(xw, cmul(cconj(U[l][i]), T1[l][j]));
            if (i == j) {
                h.Hr[i * nkp + k] = h.H[i * nkp + k] + xw.x + a.EH[i];
            } else {
                const int p = pair_index(i, j, NB);
                h.Hr[(NB + 2 * p) * nkp + k] = h.H[(NB + 2 * p) * nkp + k] + xw.x;
                h.Hr[(NB + 2 * p + 1) * nkp + k] = h.H[(NB + 2 * p + 1) * nkp + k] + xw.y;
            }
        }
}

// ================================================================ nb in 5..32: one workgroup per k
// Threads per k: 32 for nb <= 8 (eight k per workgroup), one wavefront for
// nb <= 16, four for nb <= 32.  The LDS GEMM of the VALU form (nb <= 8) runs on a
// GR x GC thread grid, each thread owning an RBR x RBC block of the NBT x NBT
// result.  OPA: conj(A) if 1.  OPB: 0 -> B[j][l] (result A B^T), 1 -> B[l][j],
// 2 -> conj(B[l][j]).
template <int NBT>
struct WaveGeom {
    // threads per k: 256 at 32 bands, 64 at 16, 32 at 8 (two packed elements
    // each, moved as one 16-byte pair)
    static constexpr int TPK = NBT >= 32 ? 256 : NBT >= 16 ? 64 : 32;
    // VALU product lane grid GR x GC, each thread an RBR x RBC block (interleaved)
    static constexpr int GR = TPK == 256 ? 16 : TPK == 64 ? 8 : 4;
    static constexpr int GC = TPK == 256 ? 16 : 8;
    static constexpr int RBR = NBT / GR, RBC = NBT / GC;
    static constexpr int PER = (NBT * NBT + TPK - 1) / TPK;  // packed doubles per thread
    static constexpr int LD = NBT + 1;  // LDS row length in complex elements (one pad)
    // k per workgroup: at nb <= 8 one k is little work, so eight k (256 threads)
    // share a workgroup and the dispatcher handles an eighth as many
    static constexpr int KPB = NBT == 8 ? 8 : 1;
    static constexpr int GATHER = NBT <= 8 ? 12 : NBT <= 16 ? 6 : 4;  // stencil neighbours per load batch
};

// The matrices are zero beyond nb (filled before use, and every product of
// zero-padded operands is zero there), so the inner loop has the compile-time
// trip count NBT; unrolled by 4 (a full unroll hoists every LDS read and
// costs twice the registers).
template <int NBT, int OPA, int OPB, typename T>
__device__ __forceinline__ void gemm_lds(const T *A, const T *B, int t,
                                         T (&acc)[WaveGeom<NBT>::RBR][WaveGeom<NBT>::RBC]) {
    constexpr int RBR = WaveGeom<NBT>::RBR, RBC = WaveGeom<NBT>::RBC, GR = WaveGeom<NBT>::GR, GC = WaveGeom<NBT>::GC;
    constexpr int LD = WaveGeom<NBT>::LD;
    // Lane (r0, c0) owns rows r0 + i GR and columns c0 + j GC (interleaved, not
    // blocked): the rows one LDS read instruction touches are then consecutive,
    // and rows NBT+1 complex apart start 4 banks apart, so the reads are free of
    // bank conflicts.
    const int r0 = t / GC, c0 = t % GC;
#pragma unroll
    for (int i = 0; i < RBR; i++)
#pragma unroll
        for (int j = 0; j < RBC; j++) acc[i][j] = T{0, 0};
#pragma unroll 4
    for (int l = 0; l < NBT; l++) {
        T av[RBR], bv[RBC];
#pragma unroll
        for (int i = 0; i < RBR; i++) {
            T v = A[(r0 + i * GR) * LD + l];
            av[i] = OPA ? T{v.x, -v.y} : v;
        }
#pragma unroll
        for (int j = 0; j < RBC; j++) {
            T v = (OPB == 0) ? B[(c0 + j * GC) * LD + l] : B[l * LD + c0 + j * GC];
            bv[j] = (OPB == 2) ? T{v.x, -v.y} : v;
        }
#pragma unroll
        for (int i = 0; i < RBR; i++)
#pragma unroll
            for (int j = 0; j < RBC; j++) {
                acc[i][j].x += av[i].x * bv[j].x - av[i].y * bv[j].y;
                acc[i][j].y += av[i].x * bv[j].y + av[i].y * bv[j].x;
            }
    }
}

template <int NBT, typename T>
__device__ __forceinline__ void store_block(T *C, int t, const T (&acc)[WaveGeom<NBT>::RBR][WaveGeom<NBT>::RBC]) {
    constexpr int RBR = WaveGeom<NBT>::RBR, RBC = WaveGeom<NBT>::RBC, GR = WaveGeom<NBT>::GR, GC = WaveGeom<NBT>::GC;
    constexpr int LD = WaveGeom<NBT>::LD;
    const int r0 = t / GC, c0 = t % GC;  // rows r0 + i GR, columns c0 + j GC
#pragma unroll
    for (int i = 0; i < RBR; i++)
#pragma unroll
        for (int j = 0; j < RBC; j++) C[(r0 + i * GR) * LD + c0 + j * GC] = acc[i][j];
}

// The same products on the matrix cores (NBT = 16: the k's one wave computes the
// 16x16 result; NBT = 32: wave w of the k's four computes tile (w / 2, w % 2)).
// A complex product is four real 16x16x4 MFMA chains per 4-wide slice of l:
// Re += Ar Br - Ai Bi, Im += Ar Bi + Ai Br.  Lane l feeds op(A)[row l%16][l/16]
// and op(B)[l/16][col l%16]; accumulator element i of lane l is C[row][l%16] with
// row = l/16 + 4 i for the FP64 instruction and 4 (l/16) + i for the FP32 one.
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
template <typename R> struct MfmaAcc;
template <> struct MfmaAcc<double> { using T = v4d; };
template <> struct MfmaAcc<float> { using T = v4f; };
__device__ __forceinline__ v4d mfma16(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4f mfma16(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <typename R>
__device__ __forceinline__ int mfma_row(int lane, int i) {
    return std::is_same<R, double>::value ? (lane >> 4) + 4 * i : 4 * (lane >> 4) + i;
}

template <int NBT>
__device__ __forceinline__ void mfma_tile(int t, int &r0, int &c0) {
    const int w = t >> 6;
    r0 = NBT == 32 ? (w >> 1) * 16 : 0;
    c0 = NBT == 32 ? (w & 1) * 16 : 0;
}

// LDS complex element access: an FP64 complex moves as one 16-byte access
// (ds_read_b128 / ds_write_b128; the LDS arrays are declared 16-byte aligned and every
// element is 16 bytes) rather than two 8-byte halves, whose 32-lane passes put
// rows r and r + 1 of neighbouring K slices on one bank.
template <typename T>
__device__ __forceinline__ T lds_get(const T *p) { return *p; }
template <typename T>
__device__ __forceinline__ void lds_put(T *p, T v) { *p = v; }
template <>
__device__ __forceinline__ cd lds_get<cd>(const cd *p) {
    const v2d v = *reinterpret_cast<const v2d *>(p);
    return cd{v.x, v.y};
}
template <>
__device__ __forceinline__ void lds_put<cd>(cd *p, cd v) {
    *reinterpret_cast<v2d *>(p) = v2d{v.x, v.y};
}

template <int NBT, int OPA, int OPB, typename R, typename T = typename CplxOf<R>::T, typename V = typename MfmaAcc<R>::T>
__device__ __forceinline__ void gemm_mfma(const T *A, const T *B, int t, V &cre, V &cim) {
    constexpr int LD = WaveGeom<NBT>::LD;
    int r0, c0;
    mfma_tile<NBT>(t, r0, c0);
    const int lane = t & 63, ra = r0 + (lane & 15), cb = c0 + (lane & 15), kq = lane >> 4;
    cre = V{0, 0, 0, 0};
    cim = V{0, 0, 0, 0};
#pragma unroll
    for (int k0 = 0; k0 < NBT; k0 += 4) {
        const int l = k0 + kq;
        T a = lds_get(A + ra * LD + l);
        if (OPA) a.y = -a.y;
        T b = lds_get(B + ((OPB == 0) ? cb * LD + l : l * LD + cb));
        if (OPB == 2) b.y = -b.y;
        cre = mfma16(a.x, b.x, cre);
        cre = mfma16(-a.y, b.y, cre);
        cim = mfma16(a.x, b.y, cim);
        cim = mfma16(a.y, b.x, cim);
    }
}

template <int NBT, typename R, typename T = typename CplxOf<R>::T, typename V = typename MfmaAcc<R>::T>
__device__ __forceinline__ void store_mfma(T *C, int t, const V &cre, const V &cim) {
    constexpr int LD = WaveGeom<NBT>::LD;
    int r0, c0;
    mfma_tile<NBT>(t, r0, c0);
    const int lane = t & 63;
#pragma unroll
    for (int i = 0; i < 4; i++) lds_put(C + (r0 + mfma_row<R>(lane, i)) * LD + c0 + (lane & 15), T{cre[i], cim[i]});
}

// BF16x3 split products on the bf16 matrix cores: each FP32 operand x is split
// into hi = bf16(x) and lo = bf16(x - hi) and every real product is taken as
// lo*hi + hi*lo + hi*hi with FP32 accumulation (v_mfma_f32_16x16x32_bf16: lane l
// feeds op(A)[row l%16][8 (l/16) + q] and op(B)[8 (l/16) + q][col l%16], q < 8;
// the accumulator layout is the FP32 16x16x4 one).  The same operands, result
// and tile assignment as gemm_mfma<..., float>; K runs in slices of 32 (zero
// beyond NBT).
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void bf16_split(float x, __bf16 &hi, __bf16 &lo) {
    hi = (__bf16)x;
    lo = (__bf16)(x - (float)hi);
}

__device__ __forceinline__ v4f prod3(const v8bf &xh, const v8bf &xl, const v8bf &yh, const v8bf &yl, v4f acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, yh, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yl, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yh, acc, 0, 0, 0);
}

template <int NBT, int OPA, int OPB>
__device__ __forceinline__ void gemm_bf16x3(const cf *A, const cf *B, int t, v4f &cre, v4f &cim) {
    constexpr int LD = WaveGeom<NBT>::LD;
    int r0, c0;
    mfma_tile<NBT>(t, r0, c0);
    const int lane = t & 63, ra = r0 + (lane & 15), cb = c0 + (lane & 15), kq = 8 * (lane >> 4);
    cre = v4f{0.f, 0.f, 0.f, 0.f};
    cim = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < NBT; k0 += 32) {
        v8bf arh, arl, aih, ail, anh, anl, brh, brl, bih, bil;
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int l = k0 + kq + q;
            cf a = cf{0.f, 0.f}, b = cf{0.f, 0.f};
            if (l < NBT) {
                a = A[ra * LD + l];
                b = (OPB == 0) ? B[cb * LD + l] : B[l * LD + cb];
            }
            if (OPA) a.y = -a.y;
            if (OPB == 2) b.y = -b.y;
            __bf16 h, lo;
            bf16_split(a.x, h, lo); arh[q] = h; arl[q] = lo;
            bf16_split(a.y, h, lo); aih[q] = h; ail[q] = lo;
            bf16_split(-a.y, h, lo); anh[q] = h; anl[q] = lo;
            bf16_split(b.x, h, lo); brh[q] = h; brl[q] = lo;
            bf16_split(b.y, h, lo); bih[q] = h; bil[q] = lo;
        }
        // Re += Ar Br - Ai Bi, Im += Ar Bi + Ai Br
        cre = prod3(arh, arl, brh, brl, cre);
        cre = prod3(anh, anl, bih, bil, cre);
        cim = prod3(arh, arl, bih, bil, cim);
        cim = prod3(aih, ail, brh, brl, cim);
    }
}

// The stage kernels' products: native MFMA of R, or BF16x3 (B3, R = float).
template <int NBT, int OPA, int OPB, typename R, bool B3>
__device__ __forceinline__ void gemm_prod(const typename CplxOf<R>::T *A, const typename CplxOf<R>::T *B, int t,
                                          typename MfmaAcc<R>::T &cre, typename MfmaAcc<R>::T &cim) {
    if constexpr (B3) {
        static_assert(std::is_same<R, float>::value, "BF16x3 products take FP32 operands");
        gemm_bf16x3<NBT, OPA, OPB>(A, B, t, cre, cim);
    } else {
        gemm_mfma<NBT, OPA, OPB, R>(A, B, t, cre, cim);
    }
}

// Row and column of accumulator element i of thread t (for the dephasing rates).
template <int NBT, typename R>
__device__ __forceinline__ void mfma_elem(int t, int i, int &row, int &col) {
    int r0, c0;
    mfma_tile<NBT>(t, r0, c0);
    row = r0 + mfma_row<R>(t & 63, i);
    col = c0 + (t & 15);
}

// Number of LDS matrices of one wave: P, M (the product X = P M^T overwrites M)
// and, with dephasing, U.
__host__ __device__ constexpr int wave_mats(int diss) { return diss ? 3 : 2; }

// One k per workgroup.  Every global operand of the stage (own state, H, D, the
// stage's accumulator and base state, the 12 stencil neighbours) is requested at
// the start, so their latencies overlap each other and the LDS work; with one
// k per workgroup the barriers only order that k's own LDS traffic.
// R is the precision of the operators and of the LDS products: double for the
// drop-in, float for the mixed-precision mode (state, stencil and increments stay
// FP64 in both).
// LDS of one k of the wave kernel, in doubles.
template <int NBT, typename R>
__host__ __device__ constexpr int wave_lds_doubles(int diss) {
    return wave_mats(diss) * NBT * WaveGeom<NBT>::LD * (int)sizeof(typename CplxOf<R>::T) / 8;
}

// k: the k this group of TPK threads serves (a valid index); lane: thread within
// the group; smem: the group's LDS; store: false for a group past the end of the
// grid, which computes its clamped k again but writes nothing (some stage modes
// update their accumulator in place).
// ROLE 0: k alone.  A stencil pair (k, kb = k + 1, see ConstArgs::pair) is served
// by two calls: ROLE 1 steps k and forms kb's stencil sum in gb, ROLE 2 steps kb
// with that sum.  The sum of k runs in its own slot order (as alone); the one of
// kb adds the neighbours it shares with k in k's slot order, then k itself, then
// its other neighbours in its own slot order.
// S: storage type of the RK stage inputs/outputs (YA, YB) and of the multistep
// histories: double, or float in the mixed form with FP32 stage storage, where
// the state at t_n (P0), the RK accumulator and every update stay FP64.
template <int NBT, int MODE, typename R, typename S = double, bool B3 = false, int ROLE = 0>
__device__ __forceinline__ void stage_wave(const ConstArgs &c, const StageArgs &a, TabRow tab, const int k, const int kb, const int lane,
                                           double *smem, const bool store, double (&gb)[WaveGeom<NBT>::PER]) {
    using CT = typename CplxOf<R>::T;
    // stage input in S for the RK stages 2-4 (they read YA / YB); the FP64 state otherwise
    constexpr bool kInS = std::is_same<S, float>::value && (MODE == RK2 || MODE == RK3 || MODE == RK4S);
    using YT = typename std::conditional<kInS, S, double>::type;
    const YT *const Yin = reinterpret_cast<const YT *>(a.Y);
    constexpr int TPK = WaveGeom<NBT>::TPK, RBR = WaveGeom<NBT>::RBR, RBC = WaveGeom<NBT>::RBC, PER = WaveGeom<NBT>::PER;
    constexpr int LD = WaveGeom<NBT>::LD, MAT = NBT * LD;
    const int nb = c.nb, NP = nb * nb, nmat = wave_mats(c.diss);
    // non-temporal streams: see ldnt
    constexpr bool kNT = NBT >= 16;
    constexpr bool kMfma = NBT >= 16;  // 16x16 matrix-core tiles; NBT = 8 stays on the VALU
    CT *A = reinterpret_cast<CT *>(smem), *B = A + MAT, *C = c.diss ? B + MAT : B;
    const R *Hop = reinterpret_cast<const R *>(sizeof(R) == 8 ? (const void *)c.H : (const void *)c.Hf);
    const R *Dop = reinterpret_cast<const R *>(sizeof(R) == 8 ? (const void *)c.D : (const void *)c.Df);
    const R *Uop = reinterpret_cast<const R *>(sizeof(R) == 8 ? (const void *)c.U : (const void *)c.Uf);
    const R Ep[3] = {(R)tab[0], (R)tab[1], (R)tab[2]}, Eq[3] = {(R)tab[3], (R)tab[4], (R)tab[5]};
    const int nn = c.n_nbr;
    const bool grad = tab[6 + nn] != 0.0;

    // With an even number of doubles per thread, a lane owns adjacent pairs of
    // elements (2q, 2q+1), q = lane + TPK m', always read and written 16 bytes at a
    // time (8 in FP32): the memory unit takes any element's alignment, so odd band
    // counts, whose k start at odd offsets, need no second form.  Lanes past the last
    // pair repeat it, and the last lane of an odd count takes (NP-2, NP-1): every
    // load stays in bounds without a branch, and repeated LDS and global stores write
    // the same value to the same address.  A choice between one wide and two single
    // accesses in front of each load and store took registers and instructions even
    // where it always fell the same way: RK4 stage of 8 bands, 200 x 200 k, 33.7 us
    // -> 29.2, of 16 119 -> 112, of 32 bands, 128 x 128, 216 -> 203; AB4 step of 13
    // bands with dephasing, 61 x 85, 42.1 -> 38.7; Taylor step of 24 bands, 96 x 100,
    // FP32 operators 131 -> 110.
    static_assert(PER % 2 == 0, "a lane owns pairs of packed elements");
    // A stencil pair's calls load the RK2/RK3 accumulator and state at t_n after
    // the products, not with the other inputs: the registers then hold kb's
    // stencil sum instead through the gather and the products.
    constexpr bool kLatePre = ROLE != 0;
    const bool cp = NP % 2 == 0;  // each pair is (re, im) of one upper element or two diagonal ones
    int eo[PER], ei[PER], ej[PER], ec[PER];
    double y[PER], pv[PER], g[PER], pre0[PER], pre1[PER];
    R hv[PER], dv[PER][3];
    const size_t base = (size_t)k * NP;
#pragma unroll
    for (int m = 0; m < PER; m++) {
        const int e = min(2 * (lane + TPK * (m >> 1)), NP - 2) + (m & 1);
        eo[m] = e;
        const int code = *gm(c.eidx + e);
        ei[m] = code & 255;
        ej[m] = (code >> 8) & 255;
        ec[m] = code >> 16;
        g[m] = pre0[m] = pre1[m] = 0.0;
        if constexpr (ROLE == 1) gb[m] = 0.0;
    }
    // Neighbour data of the stage input, GB neighbours per call, their loads all
    // issued before any is used (k's or kb's stencil slots, by `slot`).
    constexpr int GB = WaveGeom<NBT>::GATHER;
    auto fetch = [&](const auto &row, auto &v) {
        constexpr int NV = std::extent<std::remove_reference_t<decltype(v)>>::value;
        size_t kn[NV];
#pragma unroll
        for (int j = 0; j < NV; j++) kn[j] = (size_t)row[j] * NP;
#pragma unroll
        for (int j = 0; j < NV; j++) {
#pragma unroll
            for (int h = 0; h < PER / 2; h++) {
                YT v0, v1;
                ld2<false>(Yin, kn[j] + eo[2 * h], v0, v1);
                v[j][2 * h] = (double)v0;
                v[j][2 * h + 1] = (double)v1;
            }
        }
    };
    auto gather = [&](const int kk, auto slot, const int cnt, auto &v) {
        constexpr int NV = std::extent<std::remove_reference_t<decltype(v)>>::value;
        int row[NV];
#pragma unroll
        for (int j = 0; j < NV; j++) row[j] = *gm(c.nbr + (size_t)slot(min(j, cnt - 1)) * c.nkp + kk);
        fetch(row, v);
    };
    // Up to 8 bands a wave serves two k and its stencil rows are vector loads, which
    // return in the order of their requests: the first batch's are requested in front
    // of the stage's operands, not behind them (8 bands, 200 x 200 k, RK4 stage 36 us
    // -> 33.7; 29.2 with the accesses above).
    constexpr bool kRowsFirst = WaveGeom<NBT>::KPB > 1;
    int row0[kRowsFirst ? GB : 1];
    if constexpr (kRowsFirst) {
#pragma unroll
        for (int j = 0; j < GB; j++) row0[j] = *gm(c.nbr + (size_t)max(min(j, nn - 1), 0) * c.nkp + k);
    }
#pragma unroll
    for (int h = 0; h < PER / 2; h++) {
        const int m = 2 * h;
        const size_t o0 = base + eo[m];
        YT y0, y1;
        ld2<false>(Yin, o0, y0, y1);
        y[m] = (double)y0;
        y[m + 1] = (double)y1;
        ld2<kNT>(Hop, o0, hv[m], hv[m + 1]);
#pragma unroll
        for (int x = 0; x < 3; x++) {
            if (a.dmask >> x & 1) ld2<kNT>(Dop + (size_t)x * c.nk * NP, o0, dv[m][x], dv[m + 1][x]);
            else dv[m][x] = dv[m + 1][x] = (R)0;
        }
        if constexpr ((MODE == RK2 || MODE == RK3) && !kLatePre) {
            ld2<kNT>(a.ACC, o0, pre0[m], pre0[m + 1]);
            ld2<kNT>(a.P0, o0, pre1[m], pre1[m + 1]);
        } else if constexpr (MODE == RK4S) {
            ld2<kNT>(a.ACC, o0, pre0[m], pre0[m + 1]);
        }
    }
    // The dephasing's U and rates, requested before the drift and the products that
    // come first (loaded where they are used, each k waited for them: AB4 step of 13
    // bands on 61 x 85 k 50.4 us -> 41.9).
    constexpr bool kPreDiss = NBT == 16 && ROLE == 0;  // elsewhere the registers are taken
    R ur[kPreDiss ? PER : 1], ui[kPreDiss ? PER : 1], tr[4];
    if constexpr (kPreDiss) {
        if (c.diss) {
            const R *u = Uop + (size_t)k * nb * nb * 2;
#pragma unroll
            for (int m = 0; m < PER; m++) {
                const int t = min(lane + TPK * m, nb * nb - 1);
                ld2<true>(u, 2 * t, ur[m], ui[m]);
            }
            if constexpr (kMfma) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    int ia, ib;
                    mfma_elem<NBT, R>(lane, i, ia, ib);
                    tr[i] = (ia < nb && ib < nb) ? (R)*gm(c.T + ia * nb + ib) : (R)0;
                }
            }
        }
    }
    // Field drift E.grad_k rho on the shell stencil (RungeKutta.h:258-276).  The
    // neighbours are fetched GB at a time: their index and data loads are all in
    // flight together, and the sum keeps the stencil order.  First of a pair
    // (ROLE 1): every neighbour of k that is also one of kb's adds to kb's sum gb
    // as well, and kb's remaining neighbours are fetched after k's.  Second of a
    // pair (ROLE 2): the sum is gb.
    if constexpr (ROLE == 2) {
#pragma unroll
        for (int m = 0; m < PER; m++) g[m] = gb[m];
    } else if (grad) {
        for (int n0 = 0; n0 < nn; n0 += GB) {
            double v[GB][PER];
            if constexpr (kRowsFirst) {
                fetch(row0, v);
                if (n0 + GB < nn) {
#pragma unroll
                    for (int j = 0; j < GB; j++) row0[j] = *gm(c.nbr + (size_t)min(n0 + GB + j, nn - 1) * c.nkp + k);
                }
            } else {
                gather(k, [&](int j) { return n0 + j; }, nn - n0, v);
            }
#pragma unroll
            for (int j = 0; j < GB; j++)
                if (n0 + j < nn) {
                    const double cn = tab[6 + n0 + j];
#pragma unroll
                    for (int m = 0; m < PER; m++) g[m] += cn * v[j][m];
                    if constexpr (ROLE == 1) {
                        const int pj = gm(c.pat)[n0 + j];
                        if (pj >= 0) {
                            const double cb = tab[6 + pj];
#pragma unroll
                            for (int m = 0; m < PER; m++) gb[m] += cb * v[j][m];
                        }
                    }
                }
        }
        if constexpr (ROLE == 1) {
            if (c.pself >= 0) {
                const double cb = tab[6 + c.pself];
#pragma unroll
                for (int m = 0; m < PER; m++) gb[m] += cb * y[m];
            }
            // kb's own rows (5 on the hexagonal two-shell stencil) in one batch
            constexpr int GBN = GB < 5 ? 5 : GB;
            for (int t0 = 0; t0 < c.npnew; t0 += GBN) {
                double v[GBN][PER];
                gather(kb, [&](int j) { return gm(c.pat)[kMaxNbr + t0 + j]; }, c.npnew - t0, v);
#pragma unroll
                for (int j = 0; j < GBN; j++)
                    if (t0 + j < c.npnew) {
                        const double cb = tab[6 + gm(c.pat)[kMaxNbr + t0 + j]];
#pragma unroll
                        for (int m = 0; m < PER; m++) gb[m] += cb * v[j][m];
                    }
            }
        }
    }
    if (nb < NBT)
        for (int t = lane; t < nmat * MAT; t += TPK) A[t] = CT{0, 0};
    __syncthreads();
    // A <- P (full Hermitian), B <- M = H + E.D.  Element (i, j, comp) writes its
    // upper value and its mirror; a diagonal element writes (y, 0).  A lane's pair
    // (re, im) of one upper element writes both as one complex, upper and mirror.
    {
        R *Ad = reinterpret_cast<R *>(A), *Bd = reinterpret_cast<R *>(B);
#pragma unroll
        for (int m = 0; m < PER; m++) {
            if ((m & 1) == 0 && cp && eo[m] >= nb) {
                const int i = ei[m], j = ej[m];
                const bool w = (i >= c.nch && j < c.nch) || (i < c.nch && j >= c.nch);
                const R E[3] = {w ? Eq[0] : Ep[0], w ? Eq[1] : Ep[1], w ? Eq[2] : Ep[2]};
                R dr = hv[m], di = hv[m + 1], ddi = 0;
#pragma unroll
                for (int x = 0; x < 3; x++) {
                    dr += E[x] * dv[m][x];
                    di += E[x] * dv[m + 1][x];
                    ddi += E[x] * dv[m + 1][x];
                }
                const R yr = (R)y[m], yi = (R)y[m + 1];
                lds_put(A + i * LD + j, CT{yr, yi});
                lds_put(A + j * LD + i, CT{yr, -yi});
                lds_put(B + i * LD + j, CT{dr, di});
                lds_put(B + j * LD + i, CT{dr, c.dherm ? -di : -hv[m + 1] + ddi});
                continue;
            }
            if ((m & 1) == 1 && cp && eo[m - 1] >= nb) continue;  // written with m - 1
            const int i = ei[m], j = ej[m], comp = ec[m];
            const bool w = (i >= c.nch && j < c.nch) || (i < c.nch && j >= c.nch);
            const R E[3] = {w ? Eq[0] : Ep[0], w ? Eq[1] : Ep[1], w ? Eq[2] : Ep[2]};  // selects, no pointer
            R dsum = hv[m], dd = 0;
#pragma unroll
            for (int x = 0; x < 3; x++) {
                dsum += E[x] * dv[m][x];
                dd += E[x] * dv[m][x];
            }
            const bool diag = i == j;
            const R yr = (R)y[m];
            const int up = 2 * (i * LD + j) + comp;
            const int lo = diag ? up + 1 : 2 * (j * LD + i) + comp;
            const R mlo = comp ? (c.dherm ? -dsum : -hv[m] + dd) : dsum;
            Ad[up] = yr;
            Ad[lo] = diag ? (R)0 : (comp ? -yr : yr);
            Bd[up] = dsum;
            Bd[lo] = diag ? (R)0 : mlo;
        }
    }
    __syncthreads();
    // X = P M^T; -i[M,rho] (transposed storage) = -i (X - X^+)
    if constexpr (kMfma) {
        typename MfmaAcc<R>::T cre, cim;
        gemm_prod<NBT, 0, 0, R, B3>(A, B, lane, cre, cim);
        if (C == B) __syncthreads();  // every lane has finished reading M
        store_mfma<NBT, R>(C, lane, cre, cim);
    } else {
        CT acc[RBR][RBC];
        gemm_lds<NBT, 0, 0>(A, B, lane, acc);
        if (C == B) __syncthreads();  // every lane has finished reading M
        store_block<NBT>(C, lane, acc);
    }
    __syncthreads();
    if constexpr (kLatePre && (MODE == RK2 || MODE == RK3)) {
#pragma unroll
        for (int h = 0; h < PER / 2; h++) {
            const int m = 2 * h;
            const size_t o0 = base + eo[m];
            ld2<kNT>(a.ACC, o0, pre0[m], pre0[m + 1]);
            ld2<kNT>(a.P0, o0, pre1[m], pre1[m + 1]);
        }
    }
    // pv = -i (X_ij - conj(X_ji)) plus the RWA term on core -> non-core pairs; on
    // the diagonal this is 2 Im X_ii.
#pragma unroll
    for (int m = 0; m < PER; m++) {
        if ((m & 1) == 1 && cp && eo[m - 1] >= nb) continue;  // formed with m - 1
        const int i = ei[m], j = ej[m];
        const CT xij = lds_get(C + i * LD + j), xji = lds_get(C + j * LD + i), pij = lds_get(A + i * LD + j);
        const double bre = (double)xij.x - (double)xji.x, bim = (double)xij.y + (double)xji.y;
        const double wr = (i < c.nch && j >= c.nch) ? c.wx2 : 0.0;
        const double vr = bim + -wr * (double)pij.y, vi = -bre + wr * (double)pij.x;
        if ((m & 1) == 0 && cp && eo[m] >= nb) {
            pv[m] = vr;
            pv[m + 1] = vi;
        } else {
            pv[m] = ec[m] ? vi : vr;
        }
    }
    if (c.diss) {
        __syncthreads();
        // C <- U
        if constexpr (kPreDiss) {
#pragma unroll
            for (int m = 0; m < PER; m++) {
                const int t = min(lane + TPK * m, nb * nb - 1);
                lds_put(C + (t / nb) * LD + (t % nb), CT{ur[m], ui[m]});
            }
        } else {
            const R *u = Uop + (size_t)k * nb * nb * 2;
            for (int t = lane; t < nb * nb; t += TPK) {
                R re, im;
                ld2<true>(u, 2 * t, re, im);
                lds_put(C + (t / nb) * LD + (t % nb), CT{re, im});
            }
        }
        __syncthreads();
        if constexpr (kMfma) {
            typename MfmaAcc<R>::T cre, cim;
            gemm_prod<NBT, 0, 0, R, B3>(A, C, lane, cre, cim);     // T1 = P U^T
            __syncthreads();
            store_mfma<NBT, R>(B, lane, cre, cim);
            __syncthreads();
            gemm_prod<NBT, 1, 1, R, B3>(C, B, lane, cre, cim);     // G = conj(U) T1
#pragma unroll
            for (int i = 0; i < 4; i++) {
                int ia, ib;
                mfma_elem<NBT, R>(lane, i, ia, ib);
                const R t = kPreDiss ? tr[i] : (ia < nb && ib < nb) ? (R)*gm(c.T + ia * nb + ib) : (R)0;
                cre[i] *= t;
                cim[i] *= t;
            }
            __syncthreads();
            store_mfma<NBT, R>(A, lane, cre, cim);               // A <- K = T o G
            __syncthreads();
            gemm_prod<NBT, 0, 2, R, B3>(A, C, lane, cre, cim);     // T2 = K conj(U)
            __syncthreads();
            store_mfma<NBT, R>(B, lane, cre, cim);
            __syncthreads();
            gemm_prod<NBT, 1, 1, R, B3>(C, B, lane, cre, cim);     // W = conj(U) T2
            __syncthreads();
            store_mfma<NBT, R>(A, lane, cre, cim);
            __syncthreads();
        } else {
            CT acc[RBR][RBC];
            gemm_lds<NBT, 0, 0>(A, C, lane, acc);     // T1 = P U^T
            __syncthreads();
            store_block<NBT>(B, lane, acc);
            __syncthreads();
            gemm_lds<NBT, 1, 1>(C, B, lane, acc);     // G = conj(U) T1
            {
                constexpr int GR = WaveGeom<NBT>::GR, GC = WaveGeom<NBT>::GC;
                const int r0 = lane / GC, c0 = lane % GC;
    #pragma unroll
                for (int i = 0; i < RBR; i++)
    #pragma unroll
                    for (int j = 0; j < RBC; j++) {
                        const int ia = r0 + i * GR, ib = c0 + j * GC;
                        const R t = (ia < nb && ib < nb) ? (R)*gm(c.T + ia * nb + ib) : (R)0;
                        acc[i][j] = CT{acc[i][j].x * t, acc[i][j].y * t};
                    }
            }
            __syncthreads();
            store_block<NBT>(A, lane, acc);               // A <- K = T o G
            __syncthreads();
            gemm_lds<NBT, 0, 2>(A, C, lane, acc);     // T2 = K conj(U)
            __syncthreads();
            store_block<NBT>(B, lane, acc);
            __syncthreads();
            gemm_lds<NBT, 1, 1>(C, B, lane, acc);     // W = conj(U) T2
            __syncthreads();
            store_block<NBT>(A, lane, acc);
            __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < PER; m++) {
            if ((m & 1) == 1 && cp && eo[m - 1] >= nb) continue;  // formed with m - 1
            const int i = ei[m], j = ej[m];
            const CT w = A[i * LD + j];
            CT hole = CT{0, 0};
            for (int v = 0; v < (c.hole ? c.ncc : 0); v++) {
                const CT uj = C[v * LD + j], ui = C[v * LD + i];
                const R tv = (R)*gm(c.T + v * nb + v);
                // conj(U[v][j]) U[v][i] T[v][v]
                hole.x += (uj.x * ui.x + uj.y * ui.y) * tv;
                hole.y += (uj.x * ui.y - uj.y * ui.x) * tv;
            }
            if ((m & 1) == 0 && cp && eo[m] >= nb) {
                pv[m] = pv[m] - (double)w.x + (double)hole.x;
                pv[m + 1] = pv[m + 1] - (double)w.y + (double)hole.y;
            } else {
                pv[m] = ec[m] ? pv[m] - (double)w.y + (double)hole.y : pv[m] - (double)w.x + (double)hole.x;
            }
        }
    }
    if (!store) return;  // after the last barrier (a group past the grid serves no pair)
    S *const outs = reinterpret_cast<S *>(a.OUT);  // RK stages 1-3 write the next stage input
#pragma unroll
    for (int h = 0; h < PER / 2; h++) {
        const int m = 2 * h;
        // A lane that repeats an element of another wave leaves its result to that
        // one: with kLatePre it may have read the accumulator after the update.  The
        // two lanes that share element NP-2 of an odd count are of one wave
        // (odd_tail_in_one_wave), whose reads all precede its stores.
        if (TPK > 64 && 2 * (lane + TPK * h) >= NP) break;
        const double k0 = pv[m] + g[m], k1 = pv[m + 1] + g[m + 1];
        const size_t o0 = base + eo[m];
        if constexpr (MODE == ABM) {
            stage_update2_abm<kNT, S>(a, o0, (size_t)c.nk * NP, k0, k1, y[m], y[m + 1]);
        } else if constexpr (MODE == TAY) {
            stage_update2_tay<kNT, S>(a, o0, (size_t)c.nk * NP, k0, k1, y[m], y[m + 1]);
        } else if constexpr (MODE == RK1) {
            st2<kNT>(a.ACC, o0, y[m] + k0 * a.ca, y[m + 1] + k1 * a.ca);
            st2<kNT>(outs, o0, (S)(y[m] + k0 * a.cb), (S)(y[m + 1] + k1 * a.cb));
        } else if constexpr (MODE == RK2 || MODE == RK3) {
            st2<kNT>(a.ACC, o0, pre0[m] + k0 * a.ca, pre0[m + 1] + k1 * a.ca);
            st2<kNT>(outs, o0, (S)(pre1[m] + k0 * a.cb), (S)(pre1[m + 1] + k1 * a.cb));
        } else if constexpr (MODE == RK4S) {
            st2<kNT>(a.OUT, o0, pre0[m] + k0 * a.ca, pre0[m + 1] + k1 * a.ca);
        } else {
            st2<kNT>(a.OUT, o0, k0, k1);
        }
    }
}

// Waves per SIMD that the registers are to allow: some modes otherwise end a few
// registers above the limit.
constexpr int wave_occupancy(int nbt, bool pair) { return nbt == 8 ? 4 : nbt == 16 && !pair ? 3 : 1; }

// Odd band counts of a tile whose k spans several waves: the last lane, (NP - 1) / 2 in
// the order of pairs, takes elements (NP-2, NP-1), and the lane before it owns NP-2.
constexpr bool odd_tail_in_one_wave(int lo, int hi) {
    for (int nb = lo | 1; nb <= hi; nb += 2)
        if ((nb * nb - 1) / 2 % 64 == 0) return false;
    return true;
}
static_assert(WaveGeom<16>::TPK == 64 && odd_tail_in_one_wave(17, 32), "element NP-2 needs one owner");

// One k per workgroup, or with PAIR (ConstArgs::pair, one k per workgroup only)
// the stencil pair (2q, 2q + 1).
template <int NBT, int MODE, typename R, typename S = double, bool B3 = false, bool PAIR = false>
__global__ __launch_bounds__(WaveGeom<NBT>::TPK * WaveGeom<NBT>::KPB, wave_occupancy(NBT, PAIR)) void k_stage_wave(ConstArgs c, StageArgs a) {
    extern __shared__ __align__(16) double smem_d[];
    constexpr int TPK = WaveGeom<NBT>::TPK;
    double gb[WaveGeom<NBT>::PER];
    if constexpr (PAIR) {
        static_assert(WaveGeom<NBT>::KPB == 1, "stencil pairs: one k per workgroup");
        // xcd_block and strip_k: bijections of the nk / 2 pairs (the pair grid has
        // half as many columns: strips of sw / 2 pairs)
        const int k = 2 * strip_k(xcd_block(), c.nk >> 1, c.sw >> 1, c.scol >> 1);
        stage_wave<NBT, MODE, R, S, B3, 1>(c, a, stage_row(a), k, k + 1, threadIdx.x, smem_d, true, gb);
        __syncthreads();  // every lane is done with k's matrices
        // the second call forms its lane-derived indices and addresses anew
        // rather than keeping the first call's live across both
        int lane2 = threadIdx.x;
        asm volatile("" : "+v"(lane2));
        stage_wave<NBT, MODE, R, S, B3, 2>(c, a, stage_row(a), k + 1, -1, lane2, smem_d, true, gb);
    } else if constexpr (WaveGeom<NBT>::KPB == 1) {
        // xcd_block and strip_k: bijections of [0, nk)
        stage_wave<NBT, MODE, R, S, B3>(c, a, stage_row(a), strip_k(xcd_block(), c.nk, c.sw, c.scol), -1, threadIdx.x, smem_d, true, gb);
    } else {
        const int sub = threadIdx.x / TPK;
        const int kk = xcd_block() * WaveGeom<NBT>::KPB + sub;
        stage_wave<NBT, MODE, R, S, B3>(c, a, stage_row(a), strip_k(min(kk, c.nk - 1), c.nk, c.sw, c.scol), -1, threadIdx.x % TPK,
                                 smem_d + sub * wave_lds_doubles<NBT, R>(c.diss), kk < c.nk, gb);
    }
}

// ---------------------------------------------------------------- batched instances
// One launch per RK4 stage and kernel class advances several independent
// problems: workgroup b serves (instance, block of that instance) from a device
// table, and every instance's arguments sit in a device array.  The stage body
// is the single-problem kernel's, so a batched step is bit-identical to
// stepping each problem on its own.
// k per workgroup of the batched small kernel: an instance of a few thousand k
// then spreads over more CUs.
constexpr int kSmallBatchThreads = 64;

struct BatchEntry {
    ConstArgs c;
    StageArgs a[4];  // RK4 stages; tab is the instance's row of the call's first step
};

template <int MODE>
__host__ __device__ constexpr int rk4_stage_of() { return MODE == RK1 ? 0 : MODE == RK2 ? 1 : MODE == RK3 ? 2 : 3; }

template <int NB, int MODE, bool DISS>
__global__ __launch_bounds__(kSmallBatchThreads * 4, (small_wpe<NB, MODE, DISS>())) void k_stage_small_batch(const BatchEntry *E, const int2 *blk, const int *dmask, size_t tab_step) {
    extern __shared__ __align__(16) double smem_d[];
    const int term = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int2 w = blk[xcd_block()];
    const BatchEntry &be = E[w.x];
    StageArgs a = be.a[rk4_stage_of<MODE>()];
    a.tab += tab_step;
    a.dmask = dmask[w.x];
    stage_small<NB, MODE, DISS, false>(be.c, a, (TabRow)a.tab, w.y * kSmallBatchThreads + threadIdx.x, threadIdx.x, kSmallBatchThreads, term, smem_d);
}

template <int NBT, int MODE, typename R, bool PAIR = false>
__global__ __launch_bounds__(WaveGeom<NBT>::TPK * WaveGeom<NBT>::KPB, wave_occupancy(NBT, PAIR)) void k_stage_wave_batch(
    const BatchEntry *E, const int2 *blk, const int *dmask, size_t tab_step) {
    extern __shared__ __align__(16) double smem_d[];
    constexpr int TPK = WaveGeom<NBT>::TPK;
    const int2 w = blk[xcd_block()];
    const BatchEntry &be = E[w.x];
    StageArgs a = be.a[rk4_stage_of<MODE>()];
    a.tab += tab_step;
    a.dmask = dmask[w.x];
    double gb[WaveGeom<NBT>::PER];
    if constexpr (PAIR) {  // every instance of the class is paired: block w.y serves pair w.y
        static_assert(WaveGeom<NBT>::KPB == 1, "stencil pairs: one k per workgroup");
        stage_wave<NBT, MODE, R, double, false, 1>(be.c, a, (TabRow)a.tab, 2 * w.y, 2 * w.y + 1, threadIdx.x, smem_d, true, gb);
        __syncthreads();  // every lane is done with the first k's matrices
        stage_wave<NBT, MODE, R, double, false, 2>(be.c, a, (TabRow)a.tab, 2 * w.y + 1, -1, threadIdx.x, smem_d, true, gb);
    } else if constexpr (WaveGeom<NBT>::KPB == 1) {
        stage_wave<NBT, MODE, R>(be.c, a, (TabRow)a.tab, w.y, -1, threadIdx.x, smem_d, true, gb);
    } else {
        const int sub = threadIdx.x / TPK, kk = w.y * WaveGeom<NBT>::KPB + sub;
        stage_wave<NBT, MODE, R>(be.c, a, (TabRow)a.tab, min(kk, be.c.nk - 1), -1, threadIdx.x % TPK,
                                 smem_d + sub * wave_lds_doubles<NBT, R>(be.c.diss), kk < be.c.nk, gb);
    }
}

// ================================================================ observables
// Values per partial: pop[nb], J1 re x3, J2 (re,im) x3, TAbs (re,im) x3 -> nb + 15,
// plus min and max of the population diagnostics.  J2_x = sum_ij P_ij (H D_x^+)_ij
// is taken as sum_jc conj(D_x,jc) W_jc with W = conj(P) H (P is Hermitian), so the
// packed operators are read instead of a table of products: 80 nb^2 bytes per k
// (P, H, U, three components of D and of the gradient of H).
constexpr int kObsSums = 15;         // J1, J2, TAbs
constexpr int kObsThreads = 256;
constexpr int kObsMaxBlocks = 1024;  // wave kernels: a block walks its share of the grid

struct ObsArgs {
    const double *P;     // state, packed
    const double *U;     // full complex AoS (not read with the mean field)
    const double *GE;    // packed Hermitian gradient of H, components x stride dxs (may be null: J1 = 0)
    const double *H;     // packed H, or the renormalised H of the mean field
    const double *D;     // packed dipole, components x stride dxs
    const int *eidx;     // packed element -> (i, j, comp) (wave layout)
    double *part;        // [2 nv + 2][gridDim.x] block partials (obs_put)
    unsigned *count;     // finished blocks (0 between launches)
    double *out;         // [nv + 2] results, host memory mapped to the device
    int nk, nkp, nb, nch, ncc, dherm;
    size_t dxs;
    // mean field: stencil of the gradient of the renormalised H; its eigenvalues [nk][nb]
    const int *nbr;
    const double *wb;
    int n_nbr;
    double *Ek;
};

// A running sum and the rounding errors of its additions (error-free two-sum): s + e is
// the sum as if formed in twice the precision and rounded at the end.
struct Sum2 {
    double s = 0.0, e = 0.0;
    __device__ __forceinline__ void add(double v) {
        const double t = s + v, b = t - s;
        e += (s - (t - b)) + (v - b);
        s = t;
    }
};
// The sums of lane groups OFF apart, in all their lanes (operands in lane order, so that
// all form the same sum); the groups of OFF lanes hold one sum each.
template <int OFF>
__device__ __forceinline__ double lane_xor(double v) {
    if constexpr (OFF == 1) return dpp64<0xB1>(v);
    else if constexpr (OFF == 2) return dpp64<0x4E>(v);
    else if constexpr (OFF == 4) return dpp64<0x141>(v);  // half-row mirror
    else if constexpr (OFF == 8) return dpp64<0x140>(v);  // row mirror
    else return __shfl_xor(v, OFF, 64);
}
template <int OFF>
__device__ __forceinline__ void sum2_xor(Sum2 &a) {
    const double s2 = lane_xor<OFF>(a.s), e2 = lane_xor<OFF>(a.e);
    const bool first = (threadIdx.x & OFF) == 0;
    Sum2 r;
    r.s = first ? a.s : s2;
    r.e = first ? a.e : e2;
    r.add(first ? s2 : a.s);
    r.e += first ? e2 : a.e;
    a = r;
}

// Accesses of the block partials at device scope, one by one: a device-scope fence
// per block instead writes back and invalidates the XCD's whole L2 each time
// (8 bands, 200 x 200, 1024 blocks: 203 us with the fence).
__device__ __forceinline__ void put_agent(double *p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ double get_agent(const double *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Partials of a block: value c < nb + kObsSums as (sum, error) at rows 2c and 2c + 1 of
// `part`, then min and max, a column per block.
__device__ __forceinline__ void obs_put(const ObsArgs &o, int c, const Sum2 &v) {
    double *p = o.part + (size_t)(2 * c) * gridDim.x + blockIdx.x;
    put_agent(p, v.s);
    put_agent(p + gridDim.x, v.e);
}

// Sums of N values over the block's threads (thread t: s[x] + e[x]; HAS_E = false: e is
// zero) as the partials c0, c0 + 1, ..., V of them at a time through `buf` in LDS
// (obs_buf doubles): eight lanes per value take 32 threads' terms each.  Every addition
// keeps its error: J1, J2 and TAbs cancel over the grid.  Six rounds of lane exchanges
// per value instead, with the errors, are 3.5 times the instructions.
constexpr int kObsRow = kObsThreads + 8;  // eight values' rows start in different LDS banks
template <int V, bool HAS_E>
constexpr int obs_buf() { return V * (HAS_E ? 2 : 1) * kObsRow; }

template <int V, bool HAS_E, int N>
__device__ __forceinline__ void obs_block_sums(const ObsArgs &o, int c0, const double (&s)[N], const double (&e)[N], double *buf) {
    const int t = threadIdx.x, x = t >> 3;
    static_assert(V * 8 <= kObsThreads, "eight lanes per value");
#pragma unroll
    for (int r = 0; r < N; r += V) {
        __syncthreads();  // the buffer's last use is over
#pragma unroll
        for (int v = 0; v < V; v++)
            if (r + v < N) {
                buf[v * kObsRow + t] = s[r + v < N ? r + v : 0];
                if (HAS_E) buf[(V + v) * kObsRow + t] = e[r + v < N ? r + v : 0];
            }
        __syncthreads();
        Sum2 a;
        const bool mine = x < V && r + x < N;
        if (mine) {
#pragma unroll 8
            for (int i = t & 7; i < kObsThreads; i += 8) {
                a.add(buf[x * kObsRow + i]);
                if (HAS_E) a.e += buf[(V + x) * kObsRow + i];
            }
        }
        sum2_xor<1>(a);
        sum2_xor<2>(a);
        sum2_xor<4>(a);
        if (mine && (t & 7) == 0) obs_put(o, c0 + r + x, a);
    }
}

// After the block's sums: `pmin`, `pmax` to its partials, and, in the block that
// finishes last, the partials of the first nsum values to the results (the rest are
// zero): one wave per value, each lane a strided subset, errors kept, the additions in a
// fixed order.  One launch instead of a reduction kernel and a copy to the host after
// it: a 70 x 70 grid of 3 bands spent 10 us on the second kernel and 4 us on the copy.
__device__ __forceinline__ void obs_finish(const ObsArgs &o, int nsum, double pmin, double pmax) {
    constexpr int NW = kObsThreads / 64;
    __shared__ double red[NW][2];
    __shared__ int last;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nv = o.nb + kObsSums, G = gridDim.x;
    const double mn = wave_min(pmin), mx = wave_max(pmax);
    if (lane == 0) {
        red[wave][0] = mn;
        red[wave][1] = mx;
    }
    __syncthreads();
    if (t < 2) {
        double v = red[0][t];
        for (int w = 1; w < NW; w++) v = t == 0 ? fmin(v, red[w][0]) : fmax(v, red[w][1]);
        put_agent(o.part + (size_t)(2 * nv + t) * G + blockIdx.x, v);
    }
    // the block's partials have reached the device's coherence point (every wave
    // waits for its own agent-scope stores) before its arrival is counted
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) last = atomicAdd(o.count, 1u) == (unsigned)(G - 1);
    __syncthreads();
    if (!last) return;
    for (int c = wave; c < nv + 2; c += NW) {
        if (c < nv) {
            const double *p = o.part + (size_t)(2 * c) * G;
            Sum2 a;
            if (c < nsum) {
#pragma unroll 4
                for (int b = lane; b < G; b += 64) {
                    a.add(get_agent(p + b));
                    a.e += get_agent(p + G + b);
                }
                sum2_xor<1>(a);
                sum2_xor<2>(a);
                sum2_xor<4>(a);
                sum2_xor<8>(a);
                sum2_xor<16>(a);
                sum2_xor<32>(a);
            }
            if (lane == 0) o.out[c] = a.s + a.e;
        } else {
            const double *p = o.part + (size_t)(nv + c) * G;
            double v = c == nv ? 1.0 : 0.0;
            for (int b = lane; b < G; b += 64) v = c == nv ? fmin(v, get_agent(p + b)) : fmax(v, get_agent(p + b));
            v = c == nv ? wave_min(v) : wave_max(v);
            if (lane == 0) o.out[c] = v;
        }
    }
    if (t == 0) *o.count = 0;
}

// Eigenvalues (ascending) and eigenvectors (columns of V) of a Hermitian matrix by
// cyclic Jacobi; every index is a compile-time constant, so A and V stay in
// registers (a run-time column order put them in scratch memory).
template <int NB>
__device__ __forceinline__ void jacobi_small(cd (&A)[NB][NB], cd (&V)[NB][NB], double (&w)[NB]) {
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) V[i][j] = mk(i == j ? 1.0 : 0.0, 0.0);
    for (int sweep = 0; sweep < 20; sweep++) {
        double off = 0, tot = 0;
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const double v = A[i][j].x * A[i][j].x + A[i][j].y * A[i][j].y;
                tot += v;
                if (i != j) off += v;
            }
        if (off <= 1e-30 * tot) break;
#pragma unroll
        for (int p = 0; p < NB; p++)
#pragma unroll
            for (int q = p + 1; q < NB; q++) {
                const double mag = sqrt(A[p][q].x * A[p][q].x + A[p][q].y * A[p][q].y);
                if (mag == 0.0) continue;
                const cd e = mk(A[p][q].x / mag, A[p][q].y / mag);
                const double th = 0.5 * (A[q][q].x - A[p][p].x) / mag;
                const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
                const double cs = 1.0 / sqrt(t * t + 1.0), sn = t * cs;
#pragma unroll
                for (int r = 0; r < NB; r++) {
                    cd x = A[r][p], y = A[r][q];
                    A[r][p] = csub(cscale(x, cs), cscale(cmul(cconj(e), y), sn));
                    A[r][q] = cadd(cscale(cmul(e, x), sn), cscale(y, cs));
                    x = V[r][p]; y = V[r][q];
                    V[r][p] = csub(cscale(x, cs), cscale(cmul(cconj(e), y), sn));
                    V[r][q] = cadd(cscale(cmul(e, x), sn), cscale(y, cs));
                }
#pragma unroll
                for (int r = 0; r < NB; r++) {
                    cd x = A[p][r], y = A[q][r];
                    A[p][r] = csub(cscale(x, cs), cscale(cmul(e, y), sn));
                    A[q][r] = cadd(cscale(cmul(cconj(e), x), sn), cscale(y, cs));
                }
            }
    }
#pragma unroll
    for (int i = 0; i < NB; i++) w[i] = A[i][i].x;
    // exchange sort of (w, column): the same exchanges as sorting an index list
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = i + 1; j < NB; j++) {
            const bool sw = w[j] < w[i];
            const double wi = w[i];
            w[i] = sw ? w[j] : wi;
            w[j] = sw ? wi : w[j];
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const cd x = V[r][i], y = V[r][j];
                V[r][i] = mk(sw ? y.x : x.x, sw ? y.y : x.y);
                V[r][j] = mk(sw ? x.x : y.x, sw ? x.y : y.y);
            }
        }
}

// nb <= 4: a thread per k, all matrices in registers; the SoA tables are read
// coalesced.  COUL: populations in the eigenbasis of the renormalised H and the
// currents of that H (Observables_MPI.h:286-304, if_resolution.cpp:125-192), its
// shell gradient contracted with P neighbour by neighbour; the eigenvalues are
// kept for edus_renorm_energies.  Bound by the latency of its loads and of the
// final sums: 60 x 60 k of 3 bands 23 us (two kernels of a wave per k) -> 13;
// with the mean field, 300 x 300, 345 us (tables written, then read) -> 43.
// Waves per SIMD: at 3 and 4 bands the compiler would give up loads in flight for one
// more (4 bands 1000 x 1000 k, whole call: 373 us, 318 with two; 3 bands 300 x 300 44.8,
// 42.5 with three).
constexpr int obs_wpe(int nb, int other) { return nb == 4 ? 2 : nb == 3 ? 3 : other; }
template <int NB, bool COUL>
__global__ __launch_bounds__(kObsThreads) __attribute__((amdgpu_waves_per_eu(obs_wpe(NB, 1), obs_wpe(NB, 8)))) void k_obs_small(ObsArgs o) {
    constexpr int NP = NB * NB;
    constexpr int V = NB + kObsSums;  // up to 40 KB of LDS, and four blocks per CU
    __shared__ double buf[obs_buf<V, false>()];
    const size_t nkp = o.nkp;
    double val[NB + kObsSums], pmin = 1.0, pmax = 0.0;  // populations, J1, J2, TAbs
    double *const acc = val + NB;
#pragma unroll
    for (int x = 0; x < NB + kObsSums; x++) val[x] = 0.0;
    const int k = blockIdx.x * kObsThreads + threadIdx.x;
    if (k < o.nk) {
        double y[NP], h[NP];
#pragma unroll
        for (int e = 0; e < NP; e++) {
            y[e] = o.P[e * nkp + k];
            h[e] = o.H[e * nkp + k];
        }
        cd U[NB][NB];
        if constexpr (COUL) {
            cd A[NB][NB], V[NB][NB];
            double w[NB];
#pragma unroll
            for (int i = 0; i < NB; i++) {
                A[i][i] = mk(h[i], 0.0);
#pragma unroll
                for (int j = i + 1; j < NB; j++) {
                    const int p = pair_index(i, j, NB);
                    A[i][j] = mk(h[NB + 2 * p], h[NB + 2 * p + 1]);
                    A[j][i] = cconj(A[i][j]);
                }
            }
            jacobi_small<NB>(A, V, w);
#pragma unroll
            for (int a = 0; a < NB; a++) {
                o.Ek[(size_t)k * NB + a] = w[a];
#pragma unroll
                for (int b = 0; b < NB; b++) U[a][b] = cconj(V[b][a]);
            }
        } else {
            const double *u = o.U + (size_t)k * NP * 2;
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    double re, im;
                    ld2<false>(u, (a * NB + b) * 2, re, im);
                    U[a][b] = mk(re, im);
                }
        }
        cd P[NB][NB], H[NB][NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            P[i][i] = mk(y[i], 0.0);
            H[i][i] = mk(h[i], 0.0);
#pragma unroll
            for (int j = i + 1; j < NB; j++) {
                const int p = pair_index(i, j, NB);
                P[i][j] = mk(y[NB + 2 * p], y[NB + 2 * p + 1]);
                P[j][i] = cconj(P[i][j]);
                H[i][j] = mk(h[NB + 2 * p], h[NB + 2 * p + 1]);
                H[j][i] = cconj(H[i][j]);
            }
        }
        // population of band c = Re (conj(U) P U^T)_cc (InitParameters.h:264-335)
#pragma unroll
        for (int c = 0; c < NB; c++) {
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < NB; i++) {
                cd t = mk(0.0, 0.0);
#pragma unroll
                for (int j = 0; j < NB; j++) t = cadd(t, cmul(P[i][j], U[c][j]));
                s += U[c][i].x * t.x + U[c][i].y * t.y;
            }
            val[c] = s;
            const double hv = (c < o.ncc) ? 1. - s : s;
            pmax = fmax(pmax, fabs(hv));
            pmin = fmin(pmin, hv);
        }
        // Current1: sum_ij P_ij gradH_ij (real: both Hermitian; a pair counts twice)
        if (o.GE) {
            if constexpr (COUL) {
                double j1[3] = {0.0, 0.0, 0.0};
                for (int n = 0; n < o.n_nbr; n++) {
                    const int kn = o.nbr[(size_t)n * nkp + k];
                    double s = 0.0;
#pragma unroll
                    for (int e = 0; e < NP; e++) {
                        const double f = e < NB ? y[e] : ((e - NB) & 1) ? -2. * y[e] : 2. * y[e];
                        s += f * (o.H[e * nkp + kn] - h[e]);
                    }
#pragma unroll
                    for (int x = 0; x < 3; x++) j1[x] += o.wb[n * 3 + x] * s;
                }
#pragma unroll
                for (int x = 0; x < 3; x++) acc[x] = j1[x];
            } else {
#pragma unroll
                for (int x = 0; x < 3; x++) {
                    double s = 0.0;
#pragma unroll
                    for (int e = 0; e < NP; e++) {
                        const double f = e < NB ? y[e] : ((e - NB) & 1) ? -2. * y[e] : 2. * y[e];
                        s += f * o.GE[x * o.dxs + e * nkp + k];
                    }
                    acc[x] = s;
                }
            }
        }
        // W = conj(P) H; Current2 = sum_jc conj(D_jc) W_jc and the transient
        // absorption -2 sum_{i<nch<=j} D_ij P_ij (Observables_MPI.h:559-569, 726-775)
        cd W[NB][NB];
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int c = 0; c < NB; c++) {
                cd s = mk(0.0, 0.0);
#pragma unroll
                for (int i = 0; i < NB; i++) s = cadd(s, cmul(P[i][j], H[i][c]));
                W[j][c] = s;
            }
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const double *d = o.D + x * o.dxs + k;
            cd s = mk(0.0, 0.0), ta = mk(0.0, 0.0);
#pragma unroll
            for (int j = 0; j < NB; j++) {
                s = cadd(s, cscale(W[j][j], d[j * nkp]));
#pragma unroll
                for (int c = j + 1; c < NB; c++) {
                    const int p = pair_index(j, c, NB);
                    const cd v = mk(d[(NB + 2 * p) * nkp], d[(NB + 2 * p + 1) * nkp]);
                    s = cadd(s, cadd(cmul(cconj(v), W[j][c]), cmul(o.dherm ? v : cconj(v), W[c][j])));
                    if (j < o.nch && c >= o.nch) ta = cadd(ta, cmul(v, P[j][c]));
                }
            }
            acc[3 + 2 * x] = s.x;
            acc[4 + 2 * x] = s.y;
            acc[9 + 2 * x] = -2. * ta.x;
            acc[10 + 2 * x] = -2. * ta.y;
        }
    }
    obs_block_sums<V, false>(o, 0, val, val, buf);
    obs_finish(o, NB + kObsSums, pmin, pmax);
}

// nb 5..32: the stage kernels' thread groups (TPK threads per k), P, U and H of
// the k in LDS, T = P U^T and W = conj(P) H on the stage kernels' product tiles.
// All operands of a k are requested together; a lane multiplies its packed
// elements of D and of the gradient by what it finds in LDS.  Memory-bound at 32
// bands (80 KB per k): 128 x 128 k take 297 us (4.5 TB/s), where the form that took
// the population with nb LDS reads per term and read a table of H D^+ took 1168; 16
// bands 200 x 200 534 -> 167 us, 8 bands 99 -> 60.  With the matrices 8 bytes off the
// boundary of their 16-byte LDS accesses a whole call takes 461 us at 32 bands, not 313,
// and 212 at 16, not 178.  Registers decide how many
// blocks a CU holds: without TAbs (no core bands) its six sums are compiled out.
constexpr int kObsWaveV = 9;  // sums per round of obs_block_sums, in the matrices' LDS
template <int NBT>
__host__ __device__ constexpr int obs_mat_doubles() {
    constexpr int mats = (kObsThreads / WaveGeom<NBT>::TPK) * 3 * NBT * WaveGeom<NBT>::LD * 2, sums = obs_buf<kObsWaveV, true>();
    return mats > sums ? mats : sums;
}
template <int NBT>
__host__ __device__ constexpr int obs_lds_doubles() {
    return obs_mat_doubles<NBT>() + (kObsThreads / WaveGeom<NBT>::TPK) * 2 * NBT + (NBT == 32 ? 64 : 0);
}

template <int NBT, bool TA>
__global__ __launch_bounds__(kObsThreads, TA ? 2 : NBT == 8 ? 4 : 3) void k_obs_wave(ObsArgs o) {
    extern __shared__ __align__(16) double smem_d[];
    constexpr int TPK = WaveGeom<NBT>::TPK, KPB = kObsThreads / TPK, PER = WaveGeom<NBT>::PER, LD = WaveGeom<NBT>::LD, MAT = NBT * LD;
    constexpr int RBR = WaveGeom<NBT>::RBR, RBC = WaveGeom<NBT>::RBC;
    static_assert(PER % 2 == 0, "a thread owns pairs of packed elements");
    const int grp = threadIdx.x / TPK, lane = threadIdx.x % TPK;
    const int nb = o.nb, NP = nb * nb, nch = o.nch;
    cd *A = reinterpret_cast<cd *>(smem_d) + (size_t)grp * 3 * MAT, *B = A + MAT, *C = B + MAT;
    Sum2 *pops = reinterpret_cast<Sum2 *>(smem_d + obs_mat_doubles<NBT>());  // [KPB][NBT], written at the end
    double *popw = reinterpret_cast<double *>(pops + KPB * NBT);                // NBT = 32: [2][32] per-k halves of the population
    for (int t = lane; t < 3 * MAT; t += TPK) A[t] = mk(0.0, 0.0);
    auto elem = [&](int m) { return 2 * (lane + TPK * (m >> 1)) + (m & 1); };
    int code0[PER];
#pragma unroll
    for (int m = 0; m < PER; m++) code0[m] = o.eidx[min(elem(m), NP - 1)];
    constexpr int NS = TA ? kObsSums : 9;
    Sum2 pop, acc[NS];
    double pmin = 1.0, pmax = 0.0;
    auto band = [&](int c, double sre) {
        pop.add(sre);
        const double hv = (c < o.ncc) ? 1. - sre : sre;
        pmax = fmax(pmax, fabs(hv));
        pmin = fmin(pmin, hv);
    };
    for (int k0 = blockIdx.x * KPB; k0 < o.nk; k0 += gridDim.x * KPB) {
        const bool live = k0 + grp < o.nk;
        const int k = min(k0 + grp, o.nk - 1);
        const size_t base = (size_t)k * NP;
        // the lane's elements, decoded anew for each k: their LDS addresses kept live
        // over the loop took the registers of a third block per CU
        int code[PER], eo[PER];
        bool v2[PER / 2];
#pragma unroll
        for (int m = 0; m < PER; m++) {
            code[m] = code0[m];
            asm volatile("" : "+v"(code[m]));
            eo[m] = min(elem(m), NP - 1);
        }
#pragma unroll
        for (int q = 0; q < PER / 2; q++) v2[q] = NP % 2 == 0 && elem(2 * q + 1) < NP;
        auto row = [&](int m) { return code[m] & 255; };
        auto col = [&](int m) { return (code[m] >> 8) & 255; };
        auto imag = [&](int m) { return (code[m] >> 16) != 0; };
        double y[PER], h[PER], ur[PER], ui[PER];
#pragma unroll
        for (int q = 0; q < PER / 2; q++) {
            const int m = 2 * q;
            const size_t o0 = base + eo[m], o1 = base + eo[m + 1];
            ld2_or_two<false>(o.P, o0, o1, v2[q], y[m], y[m + 1]);
            ld2_or_two<true>(o.H, o0, o1, v2[q], h[m], h[m + 1]);
        }
#pragma unroll
        for (int m = 0; m < PER; m++) {
            const size_t t = base + min(lane + TPK * m, NP - 1);
            ld2<true>(o.U, 2 * t, ur[m], ui[m]);
        }
        if (o.GE) {  // J1: sum_ij P_ij gradH_ij (real: both Hermitian; a pair counts twice)
            const double *ge = o.GE + (size_t)k * 3 * NP;
            double g[PER][3];
#pragma unroll
            for (int q = 0; q < PER / 2; q++)
#pragma unroll
                for (int x = 0; x < 3; x++)
                    ld2_or_two<true>(ge + (size_t)x * NP, eo[2 * q], eo[2 * q + 1], v2[q], g[2 * q][x], g[2 * q + 1][x]);
#pragma unroll
            for (int m = 0; m < PER; m++) {
                if (!live || elem(m) >= NP) continue;
                const double f = row(m) == col(m) ? y[m] : imag(m) ? -2. * y[m] : 2. * y[m];
#pragma unroll
                for (int x = 0; x < 3; x++) acc[x].add(f * g[m][x]);
            }
        }
        __syncthreads();  // the previous k's LDS reads are done
#pragma unroll
        for (int m = 0; m < PER; m++) {
            const int i = row(m), j = col(m), c = imag(m);
            double *Ad = reinterpret_cast<double *>(A), *Cd = reinterpret_cast<double *>(C);
            const int up = 2 * (i * LD + j) + c, lo = 2 * (j * LD + i) + c;
            Ad[up] = y[m];
            Cd[up] = h[m];
            if (i != j) {
                Ad[lo] = c ? -y[m] : y[m];
                Cd[lo] = c ? -h[m] : h[m];
            } else {  // W has replaced P here: the diagonal's imaginary part is zero again
                Ad[up + 1] = 0.0;
            }
            const int t = min(lane + TPK * m, NP - 1);
            lds_put(B + (t / nb) * LD + t % nb, mk(ur[m], ui[m]));
        }
        __syncthreads();
        // population of band c = Re (conj(U) P U^T)_cc = Re sum_i conj(U_ci) T_ic
        cd pij[PER];
        if constexpr (TA) {
#pragma unroll
            for (int m = 0; m < PER; m++) pij[m] = lds_get(A + row(m) * LD + col(m));
        }
        double d[PER][3];  // in flight during the products
#pragma unroll
        for (int q = 0; q < PER / 2; q++)
#pragma unroll
            for (int x = 0; x < 3; x++)
                ld2_or_two<true>(o.D + x * o.dxs, base + eo[2 * q], base + eo[2 * q + 1], v2[q], d[2 * q][x], d[2 * q + 1][x]);
        if constexpr (NBT >= 16) {
            int r0, c0;
            mfma_tile<NBT>(lane, r0, c0);
            v4d cre, cim;
            gemm_mfma<NBT, 0, 0, double>(A, B, lane, cre, cim);
            const int cb = c0 + (lane & 15);
            double ps = 0.0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const cd u = lds_get(B + cb * LD + r0 + mfma_row<double>(lane & 63, i));
                ps += u.x * cre[i] + u.y * cim[i];
            }
            ps += __shfl_xor(ps, 16, 64);
            ps += __shfl_xor(ps, 32, 64);
            if constexpr (NBT == 32) {
                if ((lane & 63) < 16) popw[(r0 >> 4) * 32 + cb] = ps;
            } else if (live && lane < nb) {
                band(lane, ps);
            }
            gemm_mfma<NBT, 1, 1, double>(A, C, lane, cre, cim);  // W = conj(P) H
            __syncthreads();
            store_mfma<NBT, double>(A, lane, cre, cim);
        } else {
            cd r[RBR][RBC];
            gemm_lds<NBT, 0, 0>(A, B, lane, r);
            constexpr int GR = WaveGeom<NBT>::GR, GC = WaveGeom<NBT>::GC;
            static_assert(RBC == 1, "one column per lane");
            const int rr = lane / GC, c = lane % GC;
            double ps = 0.0;
#pragma unroll
            for (int i = 0; i < RBR; i++) {
                const cd u = lds_get(B + c * LD + rr + i * GR);
                ps += u.x * r[i][0].x + u.y * r[i][0].y;
            }
#pragma unroll
            for (int off = GC; off < TPK; off <<= 1) ps += __shfl_xor(ps, off, 64);
            if (live && lane < nb) band(lane, ps);
            gemm_lds<NBT, 1, 1>(A, C, lane, r);
            __syncthreads();
            store_block<NBT>(A, lane, r);
        }
        __syncthreads();
        if constexpr (NBT == 32) {
            if (live && lane < nb) band(lane, popw[lane] + popw[32 + lane]);
        }
        // J2: conj(D_jc) W_jc + conj(D_cj) W_cj per element of the upper triangle, the
        // lower one being D_jc or its conjugate; TAbs
#pragma unroll
        for (int m = 0; m < PER; m++) {
            if (!live || elem(m) >= NP) continue;
            const int i = row(m), j = col(m);
            const bool im = imag(m);
            const cd wu = lds_get(A + i * LD + j), wl = lds_get(A + j * LD + i);
            cd w;
            if (i == j) w = wu;
            else if (!im) w = cadd(wu, wl);
            else if (o.dherm) w = mk(wu.y - wl.y, wl.x - wu.x);
            else w = mk(wu.y + wl.y, -(wu.x + wl.x));
#pragma unroll
            for (int x = 0; x < 3; x++) {
                acc[3 + 2 * x].add(d[m][x] * w.x);
                acc[4 + 2 * x].add(d[m][x] * w.y);
            }
            if (TA && i < nch && j >= nch) {
                const cd p = im ? mk(-pij[m].y, pij[m].x) : pij[m];
#pragma unroll
                for (int x = 0; x < 3; x++) {
                    acc[TA ? 9 + 2 * x : 0].add(-2. * d[m][x] * p.x);
                    acc[TA ? 10 + 2 * x : 0].add(-2. * d[m][x] * p.y);
                }
            }
        }
    }
    if (lane < nb) pops[grp * NBT + lane] = pop;
    double s[NS], e[NS];
#pragma unroll
    for (int x = 0; x < NS; x++) {
        s[x] = acc[x].s;
        e[x] = acc[x].e;
    }
    obs_block_sums<kObsWaveV, true>(o, nb, s, e, smem_d);
    if (threadIdx.x < nb) {
        Sum2 a;
        for (int g = 0; g < KPB; g++) {
            const Sum2 v = pops[g * NBT + threadIdx.x];
            a.add(v.s);
            a.e += v.e;
        }
        obs_put(o, threadIdx.x, a);
    }
    obs_finish(o, nb + NS, pmin, pmax);
}

// ================================================================ setup helpers
// FP32 copy of an operator table (mixed-precision mode), grid-stride.
__global__ __launch_bounds__(256) void k_to_float(const double *src, float *dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = (float)src[i];
}

// Engine creation packs the host's reference-layout tables on the device: a
// chunk of kc k is copied as is, then one thread per (k, i, j) writes the upper
// triangle of component x (complex stride cs per element) to dst[k sk + e se]
// (e = i on the diagonal, real part only; nb + 2 pair(i, j) and + 1 above it).
__global__ void k_pack(const double *__restrict__ src, long long n, int nb, int cs, int x, size_t sk, size_t se,
                       double *__restrict__ dst) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int nb2 = nb * nb, ij = (int)(t % nb2), i = ij / nb, j = ij % nb;
    if (j < i) return;
    const size_t k = (size_t)(t / nb2);
    const double re = src[((size_t)t * cs + x) * 2], im = src[((size_t)t * cs + x) * 2 + 1];
    if (i == j) {
        dst[k * sk + (size_t)i * se] = re;
    } else {
        const size_t e = nb + 2 * (size_t)pair_index(i, j, nb);
        dst[k * sk + e * se] = re;
        dst[k * sk + (e + 1) * se] = im;
    }
}

// ================================================================ captured steps
// The step counter of the field-table path: set by the host's table upload (in
// stream order) and advanced by one at the end of every captured step.
__global__ void k_counter_set(int *ctr, int v) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *ctr = v;
}
__global__ void k_counter_step(int *ctr) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *ctr += 1;
}

// Packed matrices of k0 .. k0 + n/nb^2 - 1 to the full reference layout [k][i][j], one
// thread per element (k at k sk + e se in the packed array).
__global__ __launch_bounds__(256) void k_unpack(const double *__restrict__ Y, long long n, int nb, size_t sk, size_t se, int k0,
                                                cd *__restrict__ out) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const int nb2 = nb * nb, ij = (int)(t % nb2), i = ij / nb, j = ij % nb;
    const double *y = Y + (size_t)(k0 + t / nb2) * sk;
    if (i == j) {
        out[t] = mk(y[i * se], 0.0);
    } else {
        const size_t e = nb + 2 * (size_t)pair_index(min(i, j), max(i, j), nb);
        const double re = y[e * se], im = y[(e + 1) * se];
        out[t] = mk(re, i < j ? im : -im);
    }
}

// ================================================================ adaptive dt
// Diagonal of the state before a step (P_W_prev, RungeKutta.cpp:1-9,139-147 and
// Taylor_DE_solver_deriv_Polynom.cpp:75-84).  Element e of k sits at k*sk + e*se.
__global__ void k_diag_save(const double *Y, double *DG, int nk, int nb, size_t sk, size_t se) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nk) return;
    for (int i = 0; i < nb; i++) DG[(size_t)i * nk + k] = Y[k * sk + i * se];
}

// Block maxima of the step-size measure of dyn_dt_evolution.cpp:74-87:
// 2 |P_ii(before) - P_ii(after)| / (cond + |P_ii(after)| + 1e-7), cond = P_cond_max + n_cond.
__global__ __launch_bounds__(256) void k_diag_dp(const double *Y, const double *DG, int nk, int nb, size_t sk, size_t se,
                                                 double cond, double *part) {
    __shared__ double red[4];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (k < nk)
        for (int i = 0; i < nb; i++) {
            const double y = Y[k * sk + i * se];
            m = fmax(m, 2. * fabs(DG[(size_t)i * nk + k] - y) / (cond + fabs(y) + 1.0e-7));
        }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// ================================================================ k-resolved snapshots
// Element (ic, jc) of conj(U) P_sym U^T per k, P_sym from the stored upper
// triangle, diagonal forced real (get_P_in_dia_vect, InitParameters.h:264-335).
// L lanes per k: each takes every L-th packed element and forms what it and its
// mirror contribute, conj(U_ic,i) P_ij U_jc,j + conj(U_ic,j) conj(P_ij) U_jc,i; the
// two rows of U sit in LDS.  L = 1 for the SoA layout (nb <= 4), whose loads are
// coalesced over k; a thread per k in the k-major layout read 8 nb^2 bytes with a
// stride of 8 nb^2 (32 bands, 128 x 128: 619 us -> 27, 5.6 TB/s of 150 MB).
constexpr int kElemThreads = 256;

template <int L>
__global__ __launch_bounds__(kElemThreads) void k_eigen_element(const double *__restrict__ Y, const double *__restrict__ U,
                                                                const int *__restrict__ eidx, int nk, int nb, size_t sk, size_t se,
                                                                int ic, int jc, double *__restrict__ out) {
    constexpr int KPB = kElemThreads / L;
    __shared__ cd rows[L > 1 ? KPB : 1][2][L > 1 ? EDUS_MAX_NB + 1 : 1];
    const int g = threadIdx.x / L, l = threadIdx.x % L, NP = nb * nb;
    const int kk = blockIdx.x * KPB + g, k = min(kk, nk - 1);
    const double *u = U + (size_t)k * nb * nb * 2;
    cd acc = mk(0.0, 0.0);
    if constexpr (L == 1) {
        auto pel = [&](int i, int j) -> cd {
            if (i == j) return mk(Y[k * sk + i * se], 0.0);
            const int a = min(i, j), b = max(i, j), p = pair_index(a, b, nb);
            const cd v = mk(Y[k * sk + (nb + 2 * p) * se], Y[k * sk + (nb + 2 * p + 1) * se]);
            return (i < j) ? v : cconj(v);
        };
        for (int ii = 0; ii < nb; ii++) {
            cd m = mk(0.0, 0.0);
            for (int jj = 0; jj < nb; jj++) m = cadd(m, cmul(pel(ii, jj), mk(u[(jc * nb + jj) * 2], u[(jc * nb + jj) * 2 + 1])));
            acc = cadd(acc, cmul(mk(u[(ic * nb + ii) * 2], -u[(ic * nb + ii) * 2 + 1]), m));
        }
    } else {
        for (int t = l; t < 2 * nb; t += L) {
            const int r = t >= nb, i = t - r * nb;
            const double *q = u + ((size_t)(r ? jc : ic) * nb + i) * 2;
            rows[g][r][i] = mk(q[0], q[1]);
        }
        __syncthreads();
        const cd *a = rows[g][0], *b = rows[g][1];
        const double *yk = Y + (size_t)k * NP;
#pragma unroll 4
        for (int e = l; e < NP; e += L) {
            const int code = eidx[e], i = code & 255, j = (code >> 8) & 255;
            const double v = yk[e];
            const cd w = cmul(cconj(a[i]), b[j]), x = cmul(cconj(a[j]), b[i]);
            if (i == j) acc = cadd(acc, cscale(w, v));
            else if (code >> 16) acc = cadd(acc, mk(v * (x.y - w.y), v * (w.x - x.x)));
            else acc = cadd(acc, cscale(cadd(w, x), v));
        }
#pragma unroll
        for (int off = L / 2; off > 0; off >>= 1) {
            acc.x += __shfl_xor(acc.x, off, 64);
            acc.y += __shfl_xor(acc.y, off, 64);
        }
    }
    if (kk >= nk || l != 0) return;
    if (ic == jc) acc.y = 0.0;
    out[2 * (size_t)k] = acc.x;
    out[2 * (size_t)k + 1] = acc.y;
}

// ================================================================ Wannier contraction
// Out[k][c] = sum_R phase(k,R) Val[R][c], the columns c being the nw^2 elements of H
// and the three components of the upper triangle (i <= j, component fastest) of
// (r + r^T)/2: D = (r + r^T)/2 (Wannier.h:577-578, save_HUD.cpp:187-191) is linear in
// r(R), so it is taken before the sum, which then has nw^2 + 3 nw (nw+1)/2 columns
// instead of 4 nw^2, and a product tile goes straight to the caller's layouts.
// phase(k,R) = prod_l (-1)^{R_l} w_l[(i_l R_l) mod N_l] for N_l > 1 (k_l = -1/2 + i_l/N_l).
__host__ __device__ inline long long wannier_cols(long long nw) { return nw * nw + 3 * (nw * (nw + 1) / 2); }

// Val[r0 + r][.] of n lattice vectors from the caller's H(R) [n][nw][nw] and r(R)
// [n][nw][nw][3], and (r0 = 0) the column table: element ij = i nw + j of H as (ij, 1 on
// the diagonal, else 0), pair i <= j of D as (i nw + j, j nw + i).
// PLAIN: Val[r] = [H | r_x | r_y | r_z] as the FP32 and BF16x3 forms take it (no Col).
template <bool PLAIN>
__global__ __launch_bounds__(256) void k_wannier_val(const cd *__restrict__ HR, const cd *__restrict__ rR, int r0, int n, int nw, int ncol,
                                                     cd *__restrict__ Val, int2 *__restrict__ Col) {
    const int nw2 = nw * nw;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)n * nw2) return;
    const int r = (int)(t / nw2), ij = (int)(t % nw2), i = ij / nw, j = ij % nw;
    cd *v = Val + (size_t)(r0 + r) * ncol;
    v[ij] = HR[t];
    if constexpr (PLAIN) {
        for (int x = 0; x < 3; x++) v[(x + 1) * nw2 + ij] = rR[3 * t + x];
        return;
    }
    const int ji = j * nw + i, c = nw2 + 3 * (i * nw - i * (i - 1) / 2 + j - i);
    if (i <= j) {
        const cd *a = rR + 3 * t, *b = rR + 3 * ((long long)r * nw2 + ji);
        for (int x = 0; x < 3; x++) v[c + x] = mk(0.5 * (a[x].x + b[x].x), 0.5 * (a[x].y + b[x].y));
    }
    if (r0 == 0 && r == 0) {
        Col[ij] = make_int2(ij, i == j ? 1 : 0);
        if (i <= j)
            for (int x = 0; x < 3; x++) Col[c + x] = make_int2(ij, ji);
    }
}

// Column c of k row kk of the caller's H [k][i][j] (zero diagonal imaginary parts,
// Wannier.h:489-492) or D [k][i][j][x] (likewise, both mirrored elements); Dd may be null.
__device__ __forceinline__ void wannier_store(int kk, int c, int nw2, int2 col, double re, double im, cd *Hd, cd *Dd) {
    if (c < nw2) {
        Hd[(size_t)kk * nw2 + c] = mk(re, col.y ? 0.0 : im);
    } else if (Dd) {
        const int x = (c - nw2) % 3;
        const cd v = mk(re, col.x == col.y ? 0.0 : im);
        Dd[((size_t)kk * nw2 + col.x) * 3 + x] = v;
        if (col.x != col.y) Dd[((size_t)kk * nw2 + col.y) * 3 + x] = v;
    }
}

// Per-direction phase tables of the contraction, built once per call:
// PT[Off_l + r N_l + i] = tw[Off'_l + (i R_l mod N_l)] (-1)^{R_l}, the factor of
// direction l in e^{2 pi i k.R} for grid index i (exact integer reduction; the
// sign flip for odd R_l is the shift of the grid to k = -0.5 + i/N); 1 for a
// direction with a single k point.
__global__ void k_wannier_ptab(const int *R, const cd *tw, int nR, int N0, int N1, int N2, int toff1, int toff2, cd *PT) {
    const int Nn[3] = {N0, N1, N2}, Toff[3] = {0, toff1, toff2};
    const long long o1 = (long long)nR * N0, o2 = o1 + (long long)nR * N1, tot = o2 + (long long)nR * N2;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < tot; t += (long long)gridDim.x * blockDim.x) {
        const int l = t < o1 ? 0 : t < o2 ? 1 : 2;
        const long long u = t - (l == 0 ? 0 : l == 1 ? o1 : o2);
        const int r = (int)(u / Nn[l]), i = (int)(u % Nn[l]);
        const long long Rl = R[r * 3 + l];
        long long q = ((long long)i * Rl) % Nn[l];
        if (q < 0) q += Nn[l];
        cd w = tw[Toff[l] + q];
        if (Rl & 1) w = mk(-w.x, -w.y);
        PT[t] = Nn[l] == 1 ? mk(1.0, 0.0) : w;  // a direction without k points contributes no phase
    }
}

// Phase of grid point ka and lattice vector r from the tables above.
__device__ __forceinline__ cd wannier_phase(const cd *PT, int nR, int ka, int r, int N0, int N1, int N2) {
    const int i0 = ka / (N1 * N2), i1 = (ka / N2) % N1, i2 = ka % N2;
    const size_t o1 = (size_t)nR * N0, o2 = o1 + (size_t)nR * N1;
    cd ph = PT[(size_t)r * N0 + i0];
    ph = cmul(ph, PT[o1 + (size_t)r * N1 + i1]);
    return cmul(ph, PT[o2 + (size_t)r * N2 + i2]);
}

// The contraction on the FP64 matrix cores: Out = Ph Val as four real products
// (Re = PhR ValR - PhI ValI, Im = PhR ValI + PhI ValR) of 16x16x4 v_mfma_f64 tiles.
// A workgroup of 4 waves owns 64 k x 64 columns (each wave 16 k: four 16x16 tiles with
// real and imaginary accumulators), so a phase formed in LDS serves 64 columns and one
// read of it four tiles (32 columns and two tiles: every phase formed twice as often);
// R is consumed 16 at a time.  Lane l feeds A[row l%16][kk l/16] and B[kk l/16][col
// l%16] and holds D[l/16 + 4 i][l%16], i = 0..3 (the layout of the gfx950 instruction,
// checked against a host product).  16 bands, 441 R, 96 x 96 k: 1004 us
// (with the pass to the caller's layouts that this form has no need of) -> 630, 34 TF/s
// of useful product.
constexpr int WMK = 64, WMN = 32, WMR = 16;

__global__ __launch_bounds__(256) void k_wannier_mfma(const cd *__restrict__ PT, const cd *__restrict__ Val, const int2 *__restrict__ Col,
                                                      int N0, int N1, int N2, int nR, int nw2, int nm, int ncol, int nk, int kbase,
                                                      cd *__restrict__ Hd, cd *__restrict__ Dd) {
    constexpr int NT = 4;
    __shared__ __align__(16) cd Ph[WMK][WMR + 1];
    __shared__ __align__(16) cd Vs[WMR][16 * NT + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k0 = blockIdx.y * WMK, m0 = blockIdx.x * 16 * NT;
    v4d are[NT], aim[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) are[t] = aim[t] = v4d{0.0, 0.0, 0.0, 0.0};
    for (int r0 = 0; r0 < nR; r0 += WMR) {
        for (int t = threadIdx.x; t < WMK * WMR; t += 256) {
            const int kk = t / WMR, rr = t % WMR, k = k0 + kk, r = r0 + rr;
            Ph[kk][rr] = (k < nk && r < nR) ? wannier_phase(PT, nR, kbase + k, r, N0, N1, N2) : mk(0.0, 0.0);
        }
        for (int t = threadIdx.x; t < WMR * 16 * NT; t += 256) {
            const int rr = t / (16 * NT), mm = t % (16 * NT), r = r0 + rr, m = m0 + mm;
            Vs[rr][mm] = (r < nR && m < nm) ? Val[(size_t)r * ncol + m] : mk(0.0, 0.0);
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < WMR / 4; ks++) {
            const cd a = lds_get(&Ph[wave * 16 + (lane & 15)][ks * 4 + (lane >> 4)]);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const cd b = lds_get(&Vs[ks * 4 + (lane >> 4)][t * 16 + (lane & 15)]);
                are[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, are[t], 0, 0, 0);
                aim[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, aim[t], 0, 0, 0);
                are[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, are[t], 0, 0, 0);
                aim[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, aim[t], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int m = m0 + t * 16 + (lane & 15);
        if (m >= nm) continue;
        const int2 col = Col[m];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = k0 + wave * 16 + (lane >> 4) + 4 * i;
            if (k < nk) wannier_store(k, m, nw2, col, are[t][i], aim[t][i], Hd, Dd);
        }
    }
}

// The contraction in FP32 on the matrix cores (v_mfma_f32_16x16x4f32, FP32
// accumulation): the phases are formed in FP64 from the exact per-direction
// tables and rounded once into LDS, H(R) and r(R) likewise; the sums are widened
// to FP64 on the way out.  A workgroup owns 64 k x 32 columns of
// Val = [H | r_x | r_y | r_z]; each sum is rounded to FP32 before D = (r + r^T)/2 is
// taken from it.  The FP32 instruction holds D[4 (l/16) + i][l%16] in lane l.
__global__ __launch_bounds__(256) void k_wannier_mfma32(const cd *__restrict__ PT, const cd *__restrict__ Val, int N0, int N1, int N2,
                                                        int nR, int nm, int nk, int kbase, cd *__restrict__ Out) {
    __shared__ cf Ph[WMK][WMR + 1];
    __shared__ cf Vs[WMR][WMN + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k0 = blockIdx.y * WMK, m0 = blockIdx.x * WMN;
    v4f are[2], aim[2];
#pragma unroll
    for (int t = 0; t < 2; t++) are[t] = aim[t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < nR; r0 += WMR) {
        for (int t = threadIdx.x; t < WMK * WMR; t += 256) {
            const int kk = t / WMR, rr = t % WMR, k = k0 + kk, r = r0 + rr;
            const cd ph = (k < nk && r < nR) ? wannier_phase(PT, nR, kbase + k, r, N0, N1, N2) : mk(0.0, 0.0);
            Ph[kk][rr] = cf{(float)ph.x, (float)ph.y};
        }
        for (int t = threadIdx.x; t < WMR * WMN; t += 256) {
            const int rr = t / WMN, mm = t % WMN, r = r0 + rr, m = m0 + mm;
            const cd v = (r < nR && m < nm) ? Val[(size_t)r * nm + m] : mk(0.0, 0.0);
            Vs[rr][mm] = cf{(float)v.x, (float)v.y};
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < WMR / 4; ks++) {
            const cf a = Ph[wave * 16 + (lane & 15)][ks * 4 + (lane >> 4)];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const cf b = Vs[ks * 4 + (lane >> 4)][t * 16 + (lane & 15)];
                are[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, are[t], 0, 0, 0);
                are[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(-a.y, b.y, are[t], 0, 0, 0);
                aim[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.y, aim[t], 0, 0, 0);
                aim[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.x, aim[t], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = k0 + wave * 16 + 4 * (lane >> 4) + i, m = m0 + t * 16 + (lane & 15);
            if (k < nk && m < nm) Out[(size_t)k * nm + m] = mk((double)are[t][i], (double)aim[t][i]);
        }
}

// The contraction as BF16x3 split products on the bf16 matrix cores
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation): every FP32 operand x is split
// into hi = bf16(x) and lo = bf16(x - hi), and each real product a b is taken as
// a_hi b_hi + a_hi b_lo + a_lo b_hi (the lo lo term, ~2^-16 |a b|, dropped).
// Phases and H(R), r(R) are formed in FP64 and rounded once to FP32.  Tiling as
// k_wannier_mfma32 with R consumed 32 at a time (one K slice of the
// instruction); lane l supplies A[row l%16][8 (l/16) .. +7] and B[same k][col l%16]
// and holds D[4 (l/16) + i][l%16].
constexpr int WBR = 32;

__global__ __launch_bounds__(256) void k_wannier_mfma_bf16x3(const cd *__restrict__ PT, const cd *__restrict__ Val, int N0, int N1,
                                                             int N2, int nR, int nm, int nk, int kbase, cd *__restrict__ Out) {
    // [hi, lo] planes of the real and imaginary parts, K (R) innermost with one pad
    __shared__ __bf16 Ph[2][2][WMK][WBR + 8];
    __shared__ __bf16 Vs[2][2][WMN][WBR + 8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k0 = blockIdx.y * WMK, m0 = blockIdx.x * WMN;
    v4f are[2], aim[2];
#pragma unroll
    for (int t = 0; t < 2; t++) are[t] = aim[t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < nR; r0 += WBR) {
        for (int t = threadIdx.x; t < WMK * WBR; t += 256) {
            const int kk = t / WBR, rr = t % WBR, k = k0 + kk, r = r0 + rr;
            const cd ph = (k < nk && r < nR) ? wannier_phase(PT, nR, kbase + k, r, N0, N1, N2) : mk(0.0, 0.0);
            bf16_split((float)ph.x, Ph[0][0][kk][rr], Ph[0][1][kk][rr]);
            bf16_split((float)ph.y, Ph[1][0][kk][rr], Ph[1][1][kk][rr]);
        }
        for (int t = threadIdx.x; t < WBR * WMN; t += 256) {
            const int rr = t / WMN, mm = t % WMN, r = r0 + rr, m = m0 + mm;
            const cd v = (r < nR && m < nm) ? Val[(size_t)r * nm + m] : mk(0.0, 0.0);
            bf16_split((float)v.x, Vs[0][0][mm][rr], Vs[0][1][mm][rr]);
            bf16_split((float)v.y, Vs[1][0][mm][rr], Vs[1][1][mm][rr]);
        }
        __syncthreads();
        const int ka = 8 * (lane >> 4);
        v8bf a[2][2], an[2];  // [re/im][hi/lo]; an: -Im (hi, lo)
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int q = 0; q < 8; q++) a[c][h][q] = Ph[c][h][wave * 16 + (lane & 15)][ka + q];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int q = 0; q < 8; q++) an[h][q] = (__bf16)(-(float)a[1][h][q]);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            v8bf b[2][2];
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int q = 0; q < 8; q++) b[c][h][q] = Vs[c][h][t * 16 + (lane & 15)][ka + q];
            // Re += PhR VR - PhI VI, Im += PhR VI + PhI VR, each as hi hi + hi lo + lo hi
            auto prod3 = [&](const v8bf &xh, const v8bf &xl, const v8bf &yh, const v8bf &yl, v4f acc) {
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, yh, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yl, acc, 0, 0, 0);
                return __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yh, acc, 0, 0, 0);
            };
            are[t] = prod3(a[0][0], a[0][1], b[0][0], b[0][1], are[t]);
            are[t] = prod3(an[0], an[1], b[1][0], b[1][1], are[t]);
            aim[t] = prod3(a[0][0], a[0][1], b[1][0], b[1][1], aim[t]);
            aim[t] = prod3(a[1][0], a[1][1], b[0][0], b[0][1], aim[t]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int k = k0 + wave * 16 + 4 * (lane >> 4) + i, m = m0 + t * 16 + (lane & 15);
            if (k < nk && m < nm) Out[(size_t)k * nm + m] = mk((double)are[t][i], (double)aim[t][i]);
        }
}

// Output [k][c][i][j] (c = 0 H, 1..3 r) of the FP32 and BF16x3 forms to the caller's layouts,
// one thread per (k, i, j): H with zero diagonal imaginary parts
// (Wannier.h:489-492) and D = (r + r^T)/2 with zero diagonal imaginary parts
// (Wannier.h:577-578, save_HUD.cpp:187-191), [k][i][j][x].
__global__ void k_wannier_finish(const cd *__restrict__ Out, int kc, int nw, double *__restrict__ Hd, double *__restrict__ Dd) {
    const int nw2 = nw * nw;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)kc * nw2) return;
    const int kk = (int)(t / nw2), ij = (int)(t % nw2), i = ij / nw, j = ij % nw;
    const cd *src = Out + (size_t)kk * 4 * nw2;
    const cd h = src[ij];
    Hd[2 * t] = h.x;
    Hd[2 * t + 1] = (i == j) ? 0.0 : h.y;
    if (!Dd) return;
#pragma unroll
    for (int x = 0; x < 3; x++) {
        const cd a = src[(x + 1) * nw2 + i * nw + j];
        const cd b = src[(x + 1) * nw2 + j * nw + i];
        const double ai = (i == j) ? 0.0 : a.y, bi = (i == j) ? 0.0 : b.y;
        Dd[(3 * t + x) * 2] = 0.5 * (a.x + b.x);
        Dd[(3 * t + x) * 2 + 1] = 0.5 * (ai + bi);
    }
}

// ================================================================ Coulomb coefficient generator
// W(q) = sum_G V(|q+G|) e^{i (q+G).(d_i - d_j)} on a grid of q (Create_Wq_with_G_sum,
// Coulomb.h:87-175): an all-pairs sum, every q meets every G.  The phase is split as
// e^{i q.beta} e^{i G.beta} with beta_p = b.(d_i - d_j) per band pair p; the q factor
// leaves the sum.  FP64-bound: per (q, G) the potential and two FMAs per pair.
//   * q + G in two orthonormal components (the lattice's Cholesky frame), the G part
//     from the table: two additions.
//   * V = 2 pi / (eps sqrt(Q2 + qTF2) (sqrt(Q2) r0 + 1)) as one square root and one
//     reciprocal square root, each a hardware estimate and one third-order step,
//     instead of two square roots and a division.
//   * Two q per thread share the reads of the G table (LDS, one address per wave).
//   * A list of G closed under G -> -G gives W(-q) = conj W(q): the second half of a
//     symmetric set of q is the first one reversed and conjugated.
//   * Few q: the G list is split over blockIdx.y and the parts added afterwards.
// 999^2 q, 2849 G, 3 bands, with the correction around q = 0: 13.2 ms -> 2.0 ms.
constexpr int kCgTile = 128;
constexpr int kCgMaxPair = 6;  // nb <= 4
constexpr int kCgQ = 2;        // q per thread
constexpr int kCgThreads = 256;

struct CGenArgs {
    int npair, n_g, N, mode;    // mode 0: grid q = -0.5 + i h (N per direction); 1: list of (ix, iy) on that grid
    int gper;                   // G per blockIdx.y
    double qtf2, r0;
    // 2 pi / eps, and q = (qx, qy) -> (l11 qx + l21 qy, l22 qy), as [value, rest]: their
    // rounding would shift every term alike (1e-15 of the coefficients)
    double scale[2], l11[2], l21[2], l22[2];
    double beta1[kCgMaxPair], beta2[kCgMaxPair];
    const double *g;            // [n_g][2 + 2 npair]: components of G, e^{i G.beta_p}
    const int *qlist;           // mode 1: [nq][2]
};

__device__ __forceinline__ void cgen_q(const CGenArgs &a, long long iq, double &qx, double &qy) {
    int ix, iy;
    if (a.mode == 0) {
        ix = (int)(iq / a.N);
        iy = (int)(iq % a.N);
    } else {
        ix = a.qlist[2 * iq];
        iy = a.qlist[2 * iq + 1];
    }
    // Grid_and_Simpson (integrationWeight.h:5-8): q_i = -0.5 + i / (N - 1), formed so
    // that q_{N-1-i} = -q_i exactly: with i h the rounding of h shifts all q alike, and
    // a W taken from the mirrored q would see the shift with the wrong sign (1e-14 of
    // the q ~ 0 correction)
    qx = (double)(2 * ix - (a.N - 1)) / (double)(2 * (a.N - 1));
    qy = (double)(2 * iy - (a.N - 1)) / (double)(2 * (a.N - 1));
}

// 1 / sqrt(x) for a normal x > 0: the hardware's estimate y, then the series
// y (1 - e)^(-1/2) = y (1 + e/2 + 3 e^2/8 + ...) with e = 1 - x y^2 (the cubic term
// changed no digit).
__device__ __forceinline__ double rsqrt_step(double x, double &m, double &ep) {
    const double y = __builtin_amdgcn_rsq(x);
    m = x * y;  // ~ sqrt(x)
    const double e = __builtin_fma(-m, y, 1.0);
    ep = e * __builtin_fma(0.375, e, 0.5);
    return y;
}

// V(|q + G|) without the scale, Q2 = |q + G|^2 (Coloumb_THh_F, Coulomb.h:60-84).  The
// fast forms take (q^2 + qTF^2) (|q| r0 + 1)^2 as a whole, which has to be a normal
// number with |q| r0 + 1 > 0 (edus_coulomb_coefficients looks the parameters over); the
// general one is the formula as it stands.
enum CgForm { CG_PLAIN, CG_RYTOVA, CG_GENERAL };
template <int FORM>
__device__ __forceinline__ double cgen_v(double q2, double qtf2, double r0) {
    double u = q2 + qtf2, m, ep;
    if constexpr (FORM == CG_GENERAL) return 1.0 / (sqrt(u) * (r0 != 0.0 ? sqrt(q2) * r0 + 1.0 : 1.0));
    if constexpr (FORM == CG_RYTOVA) {
        rsqrt_step(fmax(q2, 1e-290), m, ep);   // q = 0 and G = 0: sqrt is 0 to within 1e-145
        const double t = __builtin_fma(__builtin_fma(m, ep, m), r0, 1.0);
        u = u * t * t;
    }
    const double y = rsqrt_step(u, m, ep), v = __builtin_fma(y, ep, y);
    return u == 0.0 ? __builtin_inf() : v;  // q = 0 without screening
}

// part[y][t][1 + 2 npair]: sums of q number iq0 + t over the G of blockIdx.y.
template <int NPAIR, int FORM>
__global__ __launch_bounds__(kCgThreads) void k_cgen_w(CGenArgs a, long long iq0, int nq, double *part) {
    constexpr int ROW = 2 + 2 * NPAIR, NW = 1 + 2 * NPAIR;
    __shared__ double sg[kCgTile * ROW];
    const int t0 = blockIdx.x * kCgThreads * kCgQ + threadIdx.x;
    double x[kCgQ], y[kCgQ], w[kCgQ][NW];
#pragma unroll
    for (int j = 0; j < kCgQ; j++) {
        double qx, qy;
        cgen_q(a, iq0 + min(t0 + j * kCgThreads, nq - 1), qx, qy);
        x[j] = __builtin_fma(a.l11[0], qx, __builtin_fma(a.l21[0], qy, __builtin_fma(a.l11[1], qx, a.l21[1] * qy)));
        y[j] = __builtin_fma(a.l22[0], qy, a.l22[1] * qy);
#pragma unroll
        for (int c = 0; c < NW; c++) w[j][c] = 0.0;
    }
    const int gend = min(a.n_g, (int)(blockIdx.y + 1) * a.gper);
    for (int g0 = blockIdx.y * a.gper; g0 < gend; g0 += kCgTile) {
        const int nt = min(kCgTile, gend - g0);
        __syncthreads();
        for (int i = threadIdx.x; i < nt * ROW; i += kCgThreads) sg[i] = a.g[(size_t)g0 * ROW + i];
        __syncthreads();
#pragma unroll 2
        for (int j = 0; j < nt; j++) {
            const double *s = sg + j * ROW;
#pragma unroll
            for (int q = 0; q < kCgQ; q++) {
                const double cx = x[q] + s[0], cy = y[q] + s[1];
                const double v = cgen_v<FORM>(__builtin_fma(cx, cx, cy * cy), a.qtf2, a.r0);
                w[q][0] += v;
#pragma unroll
                for (int p = 0; p < 2 * NPAIR; p++) w[q][1 + p] = __builtin_fma(v, s[2 + p], w[q][1 + p]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kCgQ; j++) {
        const int t = t0 + j * kCgThreads;
        if (t >= nq) continue;
        double *o = part + ((size_t)blockIdx.y * nq + t) * NW;
#pragma unroll
        for (int c = 0; c < NW; c++) o[c] = w[j][c];
    }
}

// W of q number iq0 + t from the ny parts, times e^{i q.beta} and the scale; mirror:
// its conjugate also goes to the q of the same place from the end of the ntot.
__global__ __launch_bounds__(256) void k_cgen_finish(CGenArgs a, long long iq0, int nq, int ny, long long ntot, int mirror,
                                                     const double *part, double *W) {
    const int t = blockIdx.x * 256 + threadIdx.x, nw = 1 + 2 * a.npair;
    if (t >= nq) return;
    double qx, qy;
    cgen_q(a, iq0 + t, qx, qy);
    auto sum = [&](int c) {
        double s = 0.0;
        for (int b = 0; b < ny; b++) s += part[((size_t)b * nq + t) * nw + c];
        return __builtin_isinf(s) ? s * a.scale[0] : __builtin_fma(s, a.scale[0], s * a.scale[1]);
    };
    double *o = W + (size_t)(iq0 + t) * nw, *m = W + (size_t)(ntot - 1 - iq0 - t) * nw;
    const bool both = mirror && m != o;
    o[0] = sum(0);
    if (both) m[0] = o[0];
    for (int p = 0; p < a.npair; p++) {
        double s, c;
        sincos(qx * a.beta1[p] + qy * a.beta2[p], &s, &c);
        const cd w = cmul(mk(c, s), mk(sum(1 + 2 * p), sum(2 + 2 * p)));
        o[1 + 2 * p] = w.x;
        o[2 + 2 * p] = w.y;
        if (both) {
            m[1 + 2 * p] = w.x;
            m[2 + 2 * p] = -w.y;
        }
    }
}

// T[t][j] = sum_ix wt[ix][t] W[ix][j], j = (iy, c) (first pass of the separable Simpson
// integral, Fourier_Coulomb.cpp:230-265 with Coulomb.h:182-232): trig_t = cos(2 pi m q),
// t < ncut, sin(2 pi (t - ncut) q) otherwise, with the weights in wt (rows padded with
// zeros to ldt, a multiple of 16 TT).  On the FP64 matrix cores: a workgroup owns 16 j
// and 16 TT trig rows, its four waves every fourth slice of four ix, added in wave
// order.  W is read once per 16 TT rows instead of once per row.
constexpr int kCgTT = 3;
__global__ __launch_bounds__(256) void k_cgen_pass1(const double *__restrict__ W, const double *__restrict__ wt, int N, int ldt, int ntrig,
                                                    int J, double *__restrict__ T) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    __shared__ double red[3][kCgTT][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * kCgTT;
    const int l = lane & 15, kq = lane >> 4, jc = min(j0 + l, J - 1);
    v4 acc[kCgTT];
#pragma unroll
    for (int u = 0; u < kCgTT; u++) acc[u] = v4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int s = wave * 4; s < N; s += 16) {
        const int ix = s + kq, ic = min(ix, N - 1);
        double b = W[(size_t)ic * J + jc], av[kCgTT];
#pragma unroll
        for (int u = 0; u < kCgTT; u++) av[u] = wt[(size_t)ic * ldt + t0 + 16 * u + l];
        if (ix >= N) b = 0.0;
#pragma unroll
        for (int u = 0; u < kCgTT; u++) acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ix < N ? av[u] : 0.0, b, acc[u], 0, 0, 0);
    }
    if (wave > 0) {
#pragma unroll
        for (int u = 0; u < kCgTT; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) red[wave - 1][u][i][lane] = acc[u][i];
    }
    __syncthreads();
    if (wave > 0 || j0 + l >= J) return;
#pragma unroll
    for (int u = 0; u < kCgTT; u++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = t0 + 16 * u + kq + 4 * i;
            if (t < ntrig) T[(size_t)t * J + j0 + l] = ((acc[u][i] + red[0][u][i][lane]) + red[1][u][i][lane]) + red[2][u][i][lane];
        }
}

// S[t1][t2][c] = sum_iy wtrig[t2][iy] T[t1][iy][c]: a wave per (t1, t2), lanes over iy.
__global__ __launch_bounds__(256) void k_cgen_pass2(const double *T, const double *wtrig, int N, int ntrig, int nw, double *S) {
    constexpr int NWMAX = 1 + 2 * kCgMaxPair;
    const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (id >= ntrig * ntrig) return;
    const int t1 = id / ntrig, t2 = id % ntrig;
    double s[NWMAX];
#pragma unroll
    for (int c = 0; c < NWMAX; c++) s[c] = 0.0;
    for (int iy = lane; iy < N; iy += 64) {
        const double w = wtrig[(size_t)t2 * N + iy];
        const double *p = T + ((size_t)t1 * N + iy) * nw;
#pragma unroll
        for (int c = 0; c < NWMAX; c++)
            if (c < nw) s[c] += w * p[c];
    }
#pragma unroll
    for (int c = 0; c < NWMAX; c++)
        if (c < nw) {
            const double v = wave_sum(s[c]);
            if (lane == 0) S[(size_t)id * nw + c] = v;
        }
}

// Correction around q = 0 (Fourier_Coulomb.cpp:375-456): per listed point,
// (W0 - Fourier series) * dk2 for the entries ic <= jc, block partial sums.  A thread's
// cos and sin of 2 pi n qy wait in LDS, NC of them at a time, and all entries are
// summed in one walk over (m, n) (each entry of each n formed its own before:
// 1.01 -> 0.43 ms at 9999^2 points of the q grid).
constexpr int kCgPeakThreads = 128, kCgPeakNC = 16;
template <int NB>
__global__ __launch_bounds__(kCgPeakThreads) void k_cgen_peak(const double *W0, const int *qlist, int np, int ncut, int Np, double dk2,
                                                              const double *A, const double *B, const double *C, const double *D,
                                                              double *part) {
    constexpr int NB2 = NB * NB, NE = NB * (NB + 1) / 2, NW = 1 + NB * (NB - 1), NWV = kCgPeakThreads / 64;
    __shared__ double tc[kCgPeakNC][kCgPeakThreads], ts[kCgPeakNC][kCgPeakThreads];
    __shared__ double red[NWV][2 * NE];
    const int th = threadIdx.x, t = blockIdx.x * kCgPeakThreads + th, tt = min(t, np - 1);
    const double qx = (double)(2 * qlist[2 * tt] - (Np - 1)) / (2 * (Np - 1)), qy = (double)(2 * qlist[2 * tt + 1] - (Np - 1)) / (2 * (Np - 1));
    double vr[NE], vi[NE];
#pragma unroll
    for (int e = 0; e < NE; e++) vr[e] = vi[e] = 0.0;
    // Fourier_series_Coloumb (Coulomb.h:235-267)
    for (int n0 = 0; n0 < ncut; n0 += kCgPeakNC) {
        const int nn = min(kCgPeakNC, ncut - n0);
        for (int n = 0; n < nn; n++) sincos(2 * M_PI * (n0 + n) * qy, &ts[n][th], &tc[n][th]);
        for (int m = 0; m < ncut; m++) {
            double sm, cm;
            sincos(2 * M_PI * m * qx, &sm, &cm);
            for (int n = 0; n < nn; n++) {
                const double cn = tc[n][th], sn = ts[n][th], f0 = cm * cn, f1 = cm * sn, f2 = sm * cn, f3 = sm * sn;
                const size_t r0 = (size_t)(n0 + n + ncut * m) * NB2 * 2;
                int e = 0;
#pragma unroll
                for (int ic = 0; ic < NB; ic++)
#pragma unroll
                    for (int jc = ic; jc < NB; jc++, e++) {
                        const size_t r = r0 + 2 * (ic * NB + jc);
                        vr[e] += A[r] * f0 + B[r] * f1 + C[r] * f2 + D[r] * f3;
                        vi[e] += A[r + 1] * f0 + B[r + 1] * f1 + C[r + 1] * f2 + D[r + 1] * f3;
                    }
            }
        }
    }
    const double *w = W0 + (size_t)tt * NW;
    int e = 0, p = 0;
#pragma unroll
    for (int ic = 0; ic < NB; ic++)
#pragma unroll
        for (int jc = ic; jc < NB; jc++, e++) {
            const double wr = jc == ic ? w[0] : w[1 + 2 * p], wi = jc == ic ? 0.0 : w[2 + 2 * p];
            if (jc != ic) p++;
            const double r = wave_sum(t < np ? (wr - vr[e]) * dk2 : 0.0), i = wave_sum(t < np ? (wi - vi[e]) * dk2 : 0.0);
            if ((th & 63) == 0) {
                red[th >> 6][2 * e] = r;
                red[th >> 6][2 * e + 1] = i;
            }
        }
    __syncthreads();
    if (th < 2 * NE) {
        double v = 0.0;
        for (int b = 0; b < NWV; b++) v += red[b][th];
        int ic = 0, q = th >> 1;
        while (q >= NB - ic) q -= NB - ic++;
        part[((size_t)blockIdx.x * NB2 + ic * NB + ic + q) * 2 + (th & 1)] = v;
    }
}

// Copies of large results to the caller's ordinary memory.  hipMemcpy locks that
// memory page by page in front of the copy engine (9.3 GB/s into fresh pages, 17 into
// touched ones, where pinned memory takes 56); here pieces go through a ring of pinned
// memory, and each of a few threads copies its own piece on to the caller's pages
// while the next pieces are under way (151 MB: 15 -> 4.5 ms).  The ring (12 MB) belongs
// to the object, made by its first copy of kRingFrom bytes (16.8 MB: 1.24 -> 1.07 ms, 33
// MB 2.5 -> 1.6; 8 MB even).  An object of one call frees it again, which takes 1 to 2 ms
// with the call's other buffers: for_call (a Wannier call with 28 MB of results 2.4 ms
// without, 3.4 with; 44 MB even; 56 MB 6.3 and 3.2).
class Downloader {
    static constexpr size_t kPiece = 2 << 20;
    static constexpr int kWorkers = 6;
    const size_t from;
    char *ring = nullptr;
    hipEvent_t ev[kWorkers] = {};
    int dev = 0;

    bool ready() {
        if (ring) return true;
        if (hipGetDevice(&dev) != hipSuccess) return false;
        for (hipEvent_t &e : ev)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
        void *p = nullptr;
        if (hipHostMalloc(&p, kWorkers * kPiece, hipHostMallocDefault) != hipSuccess) return false;
        ring = static_cast<char *>(p);
        return true;
    }

public:
    static constexpr size_t kRingFrom = 16 << 20;
    explicit Downloader(size_t ring_from = kRingFrom) : from(ring_from) {}
    // the least copy that takes the ring, in a call with so many bytes of results
    static size_t for_call(size_t total) { return total >= (48u << 20) ? kRingFrom : (size_t)-1; }
    Downloader(const Downloader &) = delete;
    Downloader &operator=(const Downloader &) = delete;
    ~Downloader() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (ring) (void)hipHostFree(ring);
    }
    // n bytes of device memory, in the stream's order; returns when dst holds them.
    hipError_t copy(void *dst, const void *src, size_t n, hipStream_t st) {
        const bool large = n >= from;
        if (!large || !ready()) {
            if (large) (void)hipGetLastError();  // the ring's: this copy does without it
            const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st);
            return e == hipSuccess ? hipStreamSynchronize(st) : e;
        }
        std::mutex mu;
        size_t next = 0;
        hipError_t err = hipSuccess;
        auto work = [&](int w) {
            char *slot = ring + w * kPiece;
            hipError_t e = hipSetDevice(dev);
            for (;;) {
                size_t o, len;
                {
                    std::lock_guard<std::mutex> lock(mu);
                    if (e != hipSuccess) err = e;
                    if (err != hipSuccess || next >= n) return;
                    o = next;
                    len = std::min(kPiece, n - o);
                    next += len;
                    e = hipMemcpyAsync(slot, static_cast<const char *>(src) + o, len, hipMemcpyDeviceToHost, st);
                    if (e == hipSuccess) e = hipEventRecord(ev[w], st);
                }
                if (e == hipSuccess) e = hipEventSynchronize(ev[w]);
                if (e == hipSuccess) std::memcpy(static_cast<char *>(dst) + o, slot, len);
            }
        };
        std::thread th[kWorkers - 1];
        try {
            for (int w = 1; w < kWorkers; w++) th[w - 1] = std::thread(work, w);
        } catch (...) {
            // fewer workers: the others, this thread at least, take their pieces
        }
        work(0);
        for (std::thread &t : th)
            if (t.joinable()) t.join();
        return err;
    }
};

}  // namespace

// ==================================================================== context
struct edus_ctx {
    int dev = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int nk = 0, nkp = 0, nb = 0, np = 0, nch = 0, ncc = 0, n_nbr = 0, stepper = 0, order = 1, diss = 0, dherm = 0, hole = 0;
    int sw = 0, scol = 0;  // strip order of the wave kernels (strip_k)
    int pair = 0, pself = -1, npnew = 0;  // stencil pairs of the wave kernels (ConstArgs::pair)
    bool streamed = false; // nb <= 4: a stage's arrays exceed the caches (kStageCacheBytes)
    int tpb = 0;           // k per workgroup of the nb <= 4 kernel (0: small_group's choice)
    int precision = EDUS_PRECISION_FP64;
    float *Hf = nullptr, *Df = nullptr, *Uf = nullptr;  // FP32 operator copies (mixed precision)
    int *eidx = nullptr;  // packed element -> (i, j, comp) of the wave layout
    int dmask = 7;        // D components some field of the current call needs (see upload_table)
    bool soa = true;
    bool own_stream = true;  // false when the stream belongs to a batch
    double dt = 0, wx2 = 0, j_norm = 0, tabs_norm = 0, nktot = 0;
    std::vector<double> tinv, coef;
    std::vector<double> wb;  // [n_nbr][3]
    // device buffers
    double *P0 = nullptr, *ACC = nullptr, *YA = nullptr, *YB = nullptr, *HIST = nullptr;
    double *H = nullptr, *D = nullptr, *U = nullptr, *T = nullptr, *GE = nullptr;
    int *nbr = nullptr;
    double *tab = nullptr;
    size_t tab_cap = 0;
    Downloader down;                  // large results to the host
    double *part = nullptr;           // observables: block partials, finished-block count, results (host memory)
    unsigned *obs_count = nullptr;
    double *obs = nullptr;
    int obs_blocks = 0;
    int cur = 0;          // AB/Taylor: state in P0 (0) or YA (1)
    long long nstep = 0;  // steps done (history ring position)
    float last_ms = 0;
    int last_launches = 0;
    std::vector<void *> allocs;
    // Coulomb mean field
    int coul = 0, coul_diag = 0, N1 = 0, N2 = 0, ncut = 0, nu = 0;
    double *cPD = nullptr;  // diagonal basis: packed state in the eigenbasis
    double n_cond = 0.0;
    double *cxm = nullptr, *sxm = nullptr, *cyn = nullptr, *syn = nullptr, *cS = nullptr;
    double *cX = nullptr, *cX0 = nullptr, *cA = nullptr, *cB = nullptr, *cC = nullptr, *cD = nullptr, *cvh = nullptr;
    double *cEH = nullptr, *cEH0 = nullptr, *cT = nullptr, *cPW0 = nullptr, *cHr = nullptr, *cscreen = nullptr, *cXw = nullptr;
    double *dwb = nullptr, *cEk = nullptr;
    bool cEk_valid = false;
    double *snap = nullptr;  // [nk] complex, k-resolved snapshot element
    // adaptive dt: diagonal before the step, block maxima
    double *DG = nullptr, *dpart = nullptr;
    // device-resident field table of a run and the captured RK4 step reading it
    double *gtab = nullptr;
    size_t gtab_cap = 0;
    int *gctr = nullptr;          // rows consumed, in steps (advanced by the captured step)
    long long gtab_steps = 0, gpos = 0;
    int gdmask = 7;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
};

namespace {

template <class T>
int dalloc(edus_ctx *c, T **p, size_t n) {
    void *q = nullptr;
    HIP_TRY(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
    c->allocs.push_back(q);
    *p = static_cast<T *>(q);
    return 0;
}

// Packs reference [k][nb][nb] complex (upper triangle) into the state layout.
void pack_state(const edus_ctx *c, const double *full, std::vector<double> &out) {
    const int nb = c->nb, np = c->np;
    out.assign(c->soa ? (size_t)np * c->nkp : (size_t)np * c->nk, 0.0);
    for (int k = 0; k < c->nk; k++) {
        const double *m = full + (size_t)k * nb * nb * 2;
        for (int i = 0; i < nb; i++) {
            const size_t e = i;
            out[c->soa ? e * c->nkp + k : (size_t)k * np + e] = m[(i * nb + i) * 2];
            for (int j = i + 1; j < nb; j++) {
                const int p = pair_index(i, j, nb);
                const size_t er = nb + 2 * p;
                out[c->soa ? er * c->nkp + k : (size_t)k * np + er] = m[(i * nb + j) * 2];
                out[c->soa ? (er + 1) * c->nkp + k : (size_t)k * np + er + 1] = m[(i * nb + j) * 2 + 1];
            }
        }
    }
}

void unpack_state(const edus_ctx *c, const std::vector<double> &in, double *full) {
    const int nb = c->nb, np = c->np;
    for (int k = 0; k < c->nk; k++) {
        double *m = full + (size_t)k * nb * nb * 2;
        auto at = [&](size_t e) { return in[c->soa ? e * c->nkp + k : (size_t)k * np + e]; };
        for (int i = 0; i < nb; i++) {
            m[(i * nb + i) * 2] = at(i);
            m[(i * nb + i) * 2 + 1] = 0.0;
            for (int j = i + 1; j < nb; j++) {
                const int p = pair_index(i, j, nb);
                const double re = at(nb + 2 * p), im = at(nb + 2 * p + 1);
                m[(i * nb + j) * 2] = re;
                m[(i * nb + j) * 2 + 1] = im;
                m[(j * nb + i) * 2] = re;
                m[(j * nb + i) * 2 + 1] = -im;
            }
        }
    }
}

// A host table of nk rows (each nb x nb elements of cs complex values, the
// reference layout) copied in chunks of stage_k rows through the device buffer
// `stage`; pack(k0, kc) launches the packing of each chunk, in stream order.
template <class F>
int upload_packed(edus_ctx *c, const double *src, int cs, double *stage, int stage_k, F pack) {
    const size_t per = (size_t)c->nb * c->nb * cs * 2;
    for (int k0 = 0; k0 < c->nk; k0 += stage_k) {
        const int kc = std::min(stage_k, c->nk - k0);
        HIP_TRY(hipMemcpyAsync(stage, src + (size_t)k0 * per, (size_t)kc * per * sizeof(double), hipMemcpyHostToDevice, c->stream));
        pack(k0, kc);
        HIP_TRY(hipGetLastError());
    }
    return 0;
}

void launch_pack(const edus_ctx *c, const double *stage, int kc, int cs, int x, size_t sk, size_t se, double *dst) {
    const long long n = (long long)kc * c->nb * c->nb;
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, stage, n, c->nb, cs, x, sk, se, dst);
}

// Pinned host memory that the observables kernels write their results to: slots of
// one context each in slabs of 64 (an allocation of its own took each context 1 to
// 2 ms).  A slab whose slots are all back is freed, except the last one, which
// stays (32 KB); thread-safe.
class ResultSlots {
    static constexpr int kSlot = EDUS_MAX_NB + kObsSums + 17, kSlots = 64;  // doubles per slot (512 bytes)
    struct Slab {
        double *base;
        uint64_t used;
    };
    std::mutex mu;
    std::vector<Slab> slabs;

public:
    double *take() {
        std::lock_guard<std::mutex> lock(mu);
        for (Slab &s : slabs)
            if (~s.used) {
                const int i = __builtin_ctzll(~s.used);
                s.used |= 1ull << i;
                return s.base + (size_t)i * kSlot;
            }
        void *p = nullptr;
        if (hipHostMalloc(&p, (size_t)kSlots * kSlot * sizeof(double), hipHostMallocPortable) != hipSuccess) return nullptr;
        slabs.push_back({static_cast<double *>(p), 1});
        return slabs.back().base;
    }
    void give(double *p) {
        if (!p) return;
        std::lock_guard<std::mutex> lock(mu);
        for (size_t i = 0; i < slabs.size(); i++) {
            const ptrdiff_t d = p - slabs[i].base;
            if (d < 0 || d >= (ptrdiff_t)kSlots * kSlot) continue;
            slabs[i].used &= ~(1ull << (d / kSlot));
            if (!slabs[i].used && slabs.size() > 1) {
                (void)hipHostFree(slabs[i].base);
                slabs.erase(slabs.begin() + i);
            }
            return;
        }
    }
};
ResultSlots g_results;

struct DeviceFree {
    void operator()(double *p) const { (void)hipFree(p); }
};

int upload(edus_ctx *c, double *dst, const std::vector<double> &v) {
    HIP_TRY(hipMemcpyAsync(dst, v.data(), v.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
    return 0;
}

int state_elems(const edus_ctx *c) { return c->soa ? c->np * c->nkp : c->np * c->nk; }

// ---------------------------------------------------------------- launches
CoulArgs coul_args(edus_ctx *c, const double *Y) {
    CoulArgs a;
    a.Y = Y; a.nk = c->nk; a.nkp = c->nkp; a.nb = c->nb; a.NP = c->np; a.N1 = c->N1; a.N2 = c->N2; a.ncut = c->ncut; a.nu = c->nu;
    a.w = 1.0 / (double)c->nk;
    a.cxm = c->cxm; a.sxm = c->sxm; a.cyn = c->cyn; a.syn = c->syn; a.S = c->cS; a.X = c->cX; a.X0 = c->cX0;
    a.A = c->cA; a.B = c->cB; a.C = c->cC; a.D = c->cD; a.vh = c->cvh; a.EH = c->cEH; a.EH0 = c->cEH0; a.Tt = c->cT;
    a.Xw = c->cXw;
    return a;
}

// Mean-field coefficients of state Y: reduction, X_mn, column sums (3 launches).
int launch_coulomb(edus_ctx *c, const double *Y) {
    CoulArgs a = coul_args(c, Y);
    const int t3 = c->N2 * c->ncut * c->nu;
    // Pass 1: a workgroup of four waves per 16 x 16 tile; pass 3: 64-thread workgroups,
    // which spread its few 10^4 outputs over all CUs.
    hipLaunchKernelGGL(k_coul_s1_mfma, dim3((c->np * c->N1 + 15) / 16, (2 * c->ncut + 15) / 16), dim3(256), 0, c->stream, a);
    hipLaunchKernelGGL(k_coul_s2, dim3(c->ncut * c->ncut), dim3(kCoulThreads), 0, c->stream, a);
    hipLaunchKernelGGL(k_coul_s3, dim3((t3 + 63) / 64), dim3(64), 0, c->stream, a);
    HIP_TRY(hipGetLastError());
    return 0;
}

// The renormalised H of the stage input Y into c->cHr: the sums over Y itself
// (Wannier basis) or over Y in the eigenbasis (Coulomb_diag_basis, RungeKutta.h:41-55).
int launch_mean_field(edus_ctx *c, const double *Y) {
    CoulHArgs h;
    h.H = c->H; h.U = c->U; h.PW0 = c->cPW0; h.screen = c->cscreen; h.Hr = c->cHr; h.n_cond = c->n_cond;
    const int rt = (c->N1 + 15) / 16;
    int rc;
    if (!c->coul_diag) {
        if ((rc = launch_coulomb(c, Y))) return rc;
        hipLaunchKernelGGL(k_coul_w_mfma<true>, dim3(rt, (c->np * c->N2 + 15) / 16), dim3(64), 0, c->stream, coul_args(c, Y), h);
        HIP_TRY(hipGetLastError());
        return 0;
    }
    const dim3 grid((c->nk + 255) / 256), block(256);
    auto go = [&](auto tag) -> int {
        constexpr int NB = decltype(tag)::value;
        hipLaunchKernelGGL(k_coul_pdiag<NB>, grid, block, 0, c->stream, Y, (const double *)c->U, c->nk, c->nkp, c->cPD);
        HIP_TRY(hipGetLastError());
        if ((rc = launch_coulomb(c, c->cPD))) return rc;
        const CoulArgs a = coul_args(c, c->cPD);
        hipLaunchKernelGGL(k_coul_w_mfma<false>, dim3(rt, (2 * c->nu * c->N2 + 15) / 16), dim3(64), 0, c->stream, a, h);
        hipLaunchKernelGGL(k_coul_hdiag<NB>, grid, block, 0, c->stream, a, h, c->ncc);
        HIP_TRY(hipGetLastError());
        return 0;
    };
    switch (c->nb) {
        case 1: return go(std::integral_constant<int, 1>{});
        case 2: return go(std::integral_constant<int, 2>{});
        case 3: return go(std::integral_constant<int, 3>{});
        default: return go(std::integral_constant<int, 4>{});
    }
}

ConstArgs const_args(const edus_ctx *c) {
    ConstArgs ca;
    std::memset(&ca, 0, sizeof ca);
    ca.H = c->coul ? c->cHr : c->H; ca.D = c->D; ca.U = c->U; ca.T = c->T; ca.nbr = c->nbr;
    ca.Hf = c->Hf; ca.Df = c->Df; ca.Uf = c->Uf; ca.eidx = c->eidx;
    ca.nk = c->nk; ca.nkp = c->nkp; ca.nb = c->nb; ca.nch = c->nch; ca.ncc = c->ncc; ca.n_nbr = c->n_nbr;
    ca.diss = c->diss; ca.hole = c->hole; ca.dherm = c->dherm; ca.wx2 = c->wx2; ca.sw = c->sw; ca.scol = c->scol;
    ca.pair = c->pair; ca.pself = c->pself; ca.npnew = c->npnew; ca.pat = c->nbr + (size_t)std::max(c->n_nbr, 1) * c->nkp;
    return ca;
}

// Whether the stage kernels of a context serve stencil pairs (nb > 8; see
// stencil_pairs): not in the BF16x3 form, whose split products leave no registers for
// the second k's stencil sum, and not at 9..16 bands with dephasing, where the
// dephasing's own operands are worth them more.  16 bands, paired and one k per
// workgroup, per step: RK4 60 x 60 k 104 and 107 us, 200 x 200 844 and 743, 320 x 320
// 2077 and 1894 (MIXED 586 and 556 at 200 x 200, MIXED32 542 and 510), AB4 238 and 221
// at 200 x 200; 12 bands 802 and 739 (RK4), MIXED and MIXED32 even.
bool runs_paired(const edus_ctx *c) {
    return c->pair && c->precision != EDUS_PRECISION_BF16X3 && !(c->diss && c->nb <= 16);
}

// k per workgroup of the nb <= 4 kernel: 64 unless edus_autotune picked another.
int small_group(const edus_ctx *c) { return c->tpb ? c->tpb : 64; }

template <int MODE>
int launch_stage(edus_ctx *c, StageArgs a) {
    a.dmask = c->dmask;
    const ConstArgs ca = const_args(c);
    if (c->coul) {
        int rc = launch_mean_field(c, a.Y);
        if (rc) return rc;
    }
    if (c->soa) {
        const int tpb = small_group(c), blocks = (c->nk + tpb - 1) / tpb;
        auto go = [&](auto dtag) {
            constexpr bool DISS = decltype(dtag)::value;
            auto nbgo = [&](auto ntag) {
                constexpr int NB = decltype(ntag)::value, R = SmallGeom<NB, DISS>::R;
                const size_t lds = (size_t)R * NB * NB * tpb * sizeof(double);
                if (c->streamed) hipLaunchKernelGGL((k_stage_small<NB, MODE, DISS, true>), dim3(blocks), dim3(tpb, R), lds, c->stream, ca, a);
                else hipLaunchKernelGGL((k_stage_small<NB, MODE, DISS, false>), dim3(blocks), dim3(tpb, R), lds, c->stream, ca, a);
            };
            switch (c->nb) {
                case 1: nbgo(std::integral_constant<int, 1>{}); break;
                case 2: nbgo(std::integral_constant<int, 2>{}); break;
                case 3: nbgo(std::integral_constant<int, 3>{}); break;
                default: nbgo(std::integral_constant<int, 4>{}); break;
            }
        };
        if (c->nb < 1 || c->nb > 4) return set_err(EDUS_ERR_UNSUPPORTED, "no small kernel for this band count");
        if (c->diss) go(std::true_type{});
        else go(std::false_type{});
    } else {
        auto go = [&](auto tag, auto ptag) {
            constexpr int NBT = decltype(tag)::value, KPB = WaveGeom<NBT>::KPB;
            constexpr bool PAIR = decltype(ptag)::value;
            const dim3 grid(PAIR ? c->nk / 2 : (c->nk + KPB - 1) / KPB), block(WaveGeom<NBT>::TPK * KPB);
            const size_t lds_f = (size_t)KPB * wave_lds_doubles<NBT, float>(c->diss) * 8;
            const size_t lds_d = (size_t)KPB * wave_lds_doubles<NBT, double>(c->diss) * 8;
            if constexpr (NBT >= 16 && !PAIR) {
                if (c->precision == EDUS_PRECISION_BF16X3) {
                    hipLaunchKernelGGL((k_stage_wave<NBT, MODE, float, double, true>), grid, block, lds_f, c->stream, ca, a);
                    return;
                }
            }
            if (c->precision == EDUS_PRECISION_MIXED32)
                hipLaunchKernelGGL((k_stage_wave<NBT, MODE, float, float, false, PAIR>), grid, block, lds_f, c->stream, ca, a);
            else if (c->precision == EDUS_PRECISION_MIXED)
                hipLaunchKernelGGL((k_stage_wave<NBT, MODE, float, double, false, PAIR>), grid, block, lds_f, c->stream, ca, a);
            else
                hipLaunchKernelGGL((k_stage_wave<NBT, MODE, double, double, false, PAIR>), grid, block, lds_d, c->stream, ca, a);
        };
        // stencil pairs where a workgroup serves one k and where they measured
        // faster (runs_paired), and not in the 32-band Taylor step with FP32 storage
        // (3.73 ms paired, 3.53 one k per workgroup; its RK4 stages gain: 2.21
        // against 2.26 ms)
        const bool pair = runs_paired(c) && !(MODE == TAY && c->nb > 16 && c->precision == EDUS_PRECISION_MIXED32);
        if (c->nb <= 8) go(std::integral_constant<int, 8>{}, std::false_type{});
        else if (c->nb <= 16 && pair) go(std::integral_constant<int, 16>{}, std::true_type{});
        else if (c->nb <= 16) go(std::integral_constant<int, 16>{}, std::false_type{});
        else if (pair) go(std::integral_constant<int, 32>{}, std::true_type{});
        else go(std::integral_constant<int, 32>{}, std::false_type{});
    }
    HIP_TRY(hipGetLastError());
    return 0;
}

// Field table rows for n stages: E (6), gradient coefficients (n_nbr), flag.
// A field component that is zero in every row of the call multiplies its
// dipole component by an exact zero, so the stage kernels skip loading it (the
// sums are bit-identical).  Rows are [E_pump(3), E_probe/2(3), ...] of length rs.
int upload_table(edus_ctx *c, const std::vector<double> &rows) {
    const size_t rs = 7 + (size_t)c->n_nbr;
    int mask = 0;
    for (size_t r = 0; r + rs <= rows.size(); r += rs)
        for (int x = 0; x < 3; x++)
            if (rows[r + x] != 0.0 || rows[r + 3 + x] != 0.0) mask |= 1 << x;
    c->dmask = mask;
    if (rows.size() > c->tab_cap) {
        if (c->tab) {
            HIP_TRY(hipStreamSynchronize(c->stream));
            HIP_TRY(hipFree(c->tab));
            c->tab = nullptr;
        }
        size_t cap = std::max<size_t>(rows.size(), 4096);
        HIP_TRY(hipMalloc(&c->tab, cap * sizeof(double)));
        c->tab_cap = cap;
    }
    HIP_TRY(hipMemcpyAsync(c->tab, rows.data(), rows.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
    return 0;
}

void table_row(const edus_ctx *c, const double *E, uint8_t on, double *row) {
    for (int i = 0; i < 6; i++) row[i] = E[i];
    for (int n = 0; n < c->n_nbr; n++)
        row[6 + n] = E[0] * c->wb[n * 3] + E[1] * c->wb[n * 3 + 1] + E[2] * c->wb[n * 3 + 2];
    row[6 + c->n_nbr] = on ? 1.0 : 0.0;
}

int check_ctx(edus_ctx *c) {
    if (!c) return set_err(EDUS_ERR_INVALID, "null context");
    hipError_t e = hipSetDevice(c->dev);
    if (e != hipSuccess) return set_err(EDUS_ERR_HIP, std::string("hipSetDevice: ") + hipGetErrorString(e));
    return 0;
}

// Stencil overlap of the pairs (ka, kb) = (2q, 2q + 1) of a neighbour table
// nbr[k][nn]: each slot j of kb's stencil is matched to the first unmatched slot
// of ka's holding the same point (pat[i] = j for ka's slot i), else to ka itself
// (pself = j), else listed as new (pat[kMaxNbr + t] = j, t < npnew).  True when
// every pair has the same pattern, as on a uniform grid of even length along the
// fastest axis; the wave kernels then serve a pair per workgroup.
bool stencil_pairs(const int32_t *nbr, int nk, int nn, int *pat, int &pself, int &npnew) {
    if (nn > kMaxNbr || nk < 2 || nk % 2) return false;
    struct Pattern {
        int pm[kMaxNbr], pn[kMaxNbr], self, cnt;
    };
    auto pattern = [&](int q, Pattern &P) {
        const int32_t *A = nbr + (size_t)(2 * q) * nn, *B = A + nn;
        uint64_t used = 0;
        P.self = -1;
        P.cnt = 0;
        for (int i = 0; i < nn; i++) P.pm[i] = -1;
        for (int j = 0; j < nn; j++) {
            int hit = -1;
            for (int i = 0; i < nn && hit < 0; i++)
                if (!(used >> i & 1) && A[i] == B[j]) hit = i;
            if (hit >= 0) {
                P.pm[hit] = j;
                used |= 1ull << hit;
            } else if (B[j] == 2 * q && P.self < 0) {
                P.self = j;
            } else {
                P.pn[P.cnt++] = j;
            }
        }
    };
    Pattern P0, P;
    pattern(0, P0);
    for (int q = 1; q < nk / 2; q++) {
        pattern(q, P);
        if (P.self != P0.self || P.cnt != P0.cnt || std::memcmp(P.pm, P0.pm, nn * sizeof(int)) ||
            std::memcmp(P.pn, P0.pn, P.cnt * sizeof(int)))
            return false;
    }
    for (int i = 0; i < nn; i++) pat[i] = P0.pm[i];
    for (int t = 0; t < P0.cnt; t++) pat[kMaxNbr + t] = P0.pn[t];
    pself = P0.self;
    npnew = P0.cnt;
    return true;
}

}  // namespace

// ==================================================================== fixed scratch
// Device buffers of edus_wannier_hk_noalloc: one copy of this array per device,
// held from the library's load until the process ends.  Host code never uses
// the name itself as an address (on the host it is only a stand-in): the
// device address comes from hipGetSymbolAddress, per device (noalloc_scratch).
static __device__ __align__(256) unsigned char scratch[EDUS_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up on the first
// call with that device current and kept.
int noalloc_scratch(void **out) {
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return set_err(EDUS_ERR_UNSUPPORTED, "device index above 63");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return 0;
}

}  // namespace

// ==================================================================== C-ABI
extern "C" {

const char *edus_last_error(void) { return g_err.c_str(); }

int edus_create(const edus_problem *p, edus_ctx **out) {
    if (!p || !out) return set_err(EDUS_ERR_INVALID, "null argument");
    *out = nullptr;
    const int nb = p->nb;
    if (p->nk < 1 || nb < 1 || nb > EDUS_MAX_NB) return set_err(EDUS_ERR_INVALID, "nk/nb out of range");
    const long long padded = nb <= 4 ? ((long long)p->nk + 255) / 256 * 256 : (long long)p->nk;
    if (padded * nb * nb > kMaxStateElems) return set_err(EDUS_ERR_UNSUPPORTED, "grid too large: nk nb^2 must stay below 2^31");
    if (p->nch < 0 || p->nch > nb || p->ncc < p->nch || p->ncc > nb) return set_err(EDUS_ERR_INVALID, "core/filled band counts out of range");
    if (p->n_nbr < 0 || p->n_nbr > kMaxNbr) return set_err(EDUS_ERR_INVALID, "neighbour count out of range (0..64)");
    if (!p->H || !p->D || !p->U || !p->T || !p->rho0 || (p->n_nbr > 0 && (!p->nbr || !p->nbr_wb)))
        return set_err(EDUS_ERR_INVALID, "missing table");
    if (p->stepper < 0 || p->stepper > 2) return set_err(EDUS_ERR_INVALID, "unknown stepper");
    if (p->stepper != EDUS_STEPPER_RK4 && (p->order < 1 || p->order > EDUS_MAX_ORDER))
        return set_err(EDUS_ERR_INVALID, "order out of range");
    if (p->stepper == EDUS_STEPPER_TAYLOR && (p->order < 2 || !p->taylor_tau_inv))
        return set_err(EDUS_ERR_INVALID, "Taylor needs order >= 2 and tau^-1");
    // Neighbour indices must address the grid: the gradient gather trusts them.
    for (size_t i = 0; i < (size_t)p->nk * p->n_nbr; i++)
        if (p->nbr[i] < 0 || p->nbr[i] >= p->nk) return set_err(EDUS_ERR_INVALID, "neighbour index outside the grid");
    // The packed operator layout needs D symmetric (tight binding, the Wannier
    // (D + D^T)/2) or Hermitian (the crystal interface), with a real diagonal.
    bool dsym = true, dhermit = true;
    for (int k = 0; k < p->nk; k++)
        for (int x = 0; x < 3; x++)
            for (int i = 0; i < nb; i++) {
                const double *dii = p->D + (((size_t)k * nb + i) * nb + i) * 6 + 2 * x;
                if (dii[1] != 0.0) return set_err(EDUS_ERR_UNSUPPORTED, "dipole diagonal must be real");
                for (int j = i + 1; j < nb; j++) {
                    const double *a = p->D + (((size_t)k * nb + i) * nb + j) * 6 + 2 * x;
                    const double *b = p->D + (((size_t)k * nb + j) * nb + i) * 6 + 2 * x;
                    if (a[0] != b[0] || a[1] != b[1]) dsym = false;
                    if (a[0] != b[0] || a[1] != -b[1]) dhermit = false;
                }
            }
    if (!dsym && !dhermit) return set_err(EDUS_ERR_UNSUPPORTED, "dipole table must be symmetric or Hermitian");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(EDUS_ERR_NODEVICE, "no HIP device visible");

    auto *c = new edus_ctx();
    c->dherm = (!dsym && dhermit) ? 1 : 0;
    auto fail = [&](int rc) { edus_destroy(c); return rc; };
    if (hipGetDevice(&c->dev) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "hipGetDevice failed"));
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "stream create failed"));
    if (hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "event create failed"));
    c->nk = p->nk; c->nb = nb; c->np = nb * nb; c->nch = p->nch; c->ncc = p->ncc; c->n_nbr = p->n_nbr;
    c->stepper = p->stepper; c->order = (p->stepper == EDUS_STEPPER_RK4) ? 4 : p->order;
    c->soa = nb <= 4;
    c->precision = p->precision;
    if (c->precision != EDUS_PRECISION_FP64 && c->precision != EDUS_PRECISION_MIXED && c->precision != EDUS_PRECISION_MIXED32 &&
        c->precision != EDUS_PRECISION_BF16X3)
        return fail(set_err(EDUS_ERR_INVALID, "precision must be EDUS_PRECISION_FP64, _MIXED, _MIXED32 or _BF16X3"));
    if (c->precision != EDUS_PRECISION_FP64 && c->soa)
        return fail(set_err(EDUS_ERR_UNSUPPORTED, "mixed precision is implemented for nb >= 5"));
    if (c->precision == EDUS_PRECISION_BF16X3 && nb <= 8)
        return fail(set_err(EDUS_ERR_UNSUPPORTED, "EDUS_PRECISION_BF16X3 runs on the matrix-core tiles of nb >= 9"));
    c->nkp = (int)padded;
    c->streamed = c->soa && (double)c->nkp * (4. * p->n_nbr + 8. * c->np * kStageArrays) > kStageCacheBytes;
    // Wave kernels: walk the grid in strips (strip_k) when a strip's two previous
    // rows of packed state, the stencil's reach, fit in kStripL2Bytes while whole
    // rows would not (512 x 512 k at 32 bands: 64-column strips).
    if (!c->soa) {
        const long long n0 = p->nk_dims[0], n1 = p->nk_dims[1], n2 = p->nk_dims[2];
        if (n0 > 0 && n1 > 0 && n2 > 0 && n0 * n1 * n2 == p->nk) {
            const long long row_k = 2LL * 8 * nb * nb;  // two rows' bytes per column
            long long sw = 16;
            while (2 * sw * row_k <= kStripL2Bytes) sw *= 2;
            if (sw < n2) {
                c->sw = (int)sw;
                c->scol = (int)n2;
            }
        }
    }
    c->dt = p->dt; c->wx2 = p->wx2; c->j_norm = p->j_norm; c->tabs_norm = p->tabs_norm; c->nktot = p->nktot;
    c->wb.assign(p->nbr_wb, p->nbr_wb + (size_t)p->n_nbr * 3);
    for (int i = 0; i < nb * nb; i++)
        if (std::fabs(p->T[i]) > 1e-24) c->diss = 1;
    for (int v = 0; v < c->ncc; v++)
        if (p->T[v * nb + v] != 0.0) c->hole = 1;
    if (p->stepper == EDUS_STEPPER_TAYLOR) c->tinv.assign(p->taylor_tau_inv, p->taylor_tau_inv + (size_t)(p->order - 1) * (p->order - 1));
    // Adams-Bashforth coefficients (ODE_solver.h:152-179).
    if (p->stepper == EDUS_STEPPER_AB) {
        static const double ab[5][5] = {{1., 0, 0, 0, 0},
                                        {3.0 / 2.0, -1.0 / 2.0, 0, 0, 0},
                                        {23.0 / 12.0, -16.0 / 12.0, 5.0 / 12.0, 0, 0},
                                        {55.0 / 24.0, -59.0 / 24.0, 37.0 / 24.0, -9.0 / 24.0, 0},
                                        {1901.0 / 720.0, -2774.0 / 720.0, 2616.0 / 720.0, -1274.0 / 720.0, 251.0 / 720.0}};
        if (p->order > 5) return fail(set_err(EDUS_ERR_UNSUPPORTED, "Adams-Bashforth order > 5"));
        c->coef.assign(ab[p->order - 1], ab[p->order - 1] + p->order);
    }

    const size_t se = state_elems(c);
    int rc = 0;
    if ((rc = dalloc(c, &c->P0, se)) || (rc = dalloc(c, &c->ACC, se)) || (rc = dalloc(c, &c->YA, se)) || (rc = dalloc(c, &c->YB, se)))
        return fail(rc);
    if (c->stepper != EDUS_STEPPER_RK4) {
        if ((rc = dalloc(c, &c->HIST, se * c->order))) return fail(rc);
        if (hipMemsetAsync(c->HIST, 0, se * c->order * sizeof(double), c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "memset history"));
    }
    if (!c->soa) {
        std::vector<int> ex(c->np);
        for (int i = 0; i < nb; i++) ex[i] = i | (i << 8);
        for (int i = 0; i < nb; i++)
            for (int j = i + 1; j < nb; j++) {
                const int pp = pair_index(i, j, nb);
                ex[nb + 2 * pp] = i | (j << 8);
                ex[nb + 2 * pp + 1] = i | (j << 8) | (1 << 16);
            }
        if ((rc = dalloc(c, &c->eidx, ex.size())) ||
            hipMemcpyAsync(c->eidx, ex.data(), ex.size() * sizeof(int), hipMemcpyHostToDevice, c->stream) != hipSuccess ||
            hipStreamSynchronize(c->stream) != hipSuccess)
            return fail(rc ? rc : set_err(EDUS_ERR_HIP, "element table upload"));
    }
    // Operators in the state layout, packed on the device from chunks of the
    // host tables (sk, sek: k and element strides of the state layout).
    const size_t sk = c->soa ? 1 : (size_t)c->np, sek = c->soa ? (size_t)c->nkp : 1;
    const int stage_k = (int)std::max<long long>(1, std::min<long long>(p->nk, (1LL << 25) / ((long long)nb * nb * 6)));
    std::unique_ptr<double, DeviceFree> stage;
    {
        double *q = nullptr;
        if (hipMalloc(&q, (size_t)stage_k * nb * nb * 6 * sizeof(double)) != hipSuccess)
            return fail(set_err(EDUS_ERR_NOMEM, "staging buffer"));
        stage.reset(q);
    }
    double *st = stage.get();
    if ((rc = dalloc(c, &c->H, se)) || (rc = dalloc(c, &c->D, 3 * se))) return fail(rc);
    if (c->soa && (hipMemsetAsync(c->H, 0, se * sizeof(double), c->stream) != hipSuccess ||
                   hipMemsetAsync(c->D, 0, 3 * se * sizeof(double), c->stream) != hipSuccess))
        return fail(set_err(EDUS_ERR_HIP, "memset operators"));  // padding columns of the SoA layout
    if ((rc = upload_packed(c, p->H, 1, st, stage_k, [&](int k0, int kc) { launch_pack(c, st, kc, 1, 0, sk, sek, c->H + k0 * sk); })))
        return fail(rc);
    // D: three packed components [x][state]
    rc = upload_packed(c, p->D, 3, st, stage_k, [&](int k0, int kc) {
        for (int x = 0; x < 3; x++) launch_pack(c, st, kc, 3, x, sk, sek, c->D + x * se + k0 * sk);
    });
    if (rc) return fail(rc);
    {
        const size_t nu = (size_t)p->nk * nb * nb * 2;
        if ((rc = dalloc(c, &c->U, nu)) || (rc = dalloc(c, &c->T, (size_t)nb * nb))) return fail(rc);
        if (hipMemcpyAsync(c->U, p->U, nu * sizeof(double), hipMemcpyHostToDevice, c->stream) != hipSuccess ||
            hipMemcpyAsync(c->T, p->T, (size_t)nb * nb * sizeof(double), hipMemcpyHostToDevice, c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "upload U, T"));
    }
    if (c->precision != EDUS_PRECISION_FP64) {
        const size_t nh = se, nd = 3 * se, nu = (size_t)p->nk * nb * nb * 2;
        if ((rc = dalloc(c, &c->Hf, nh)) || (rc = dalloc(c, &c->Df, nd)) || (rc = dalloc(c, &c->Uf, nu))) return fail(rc);
        const double *src[3] = {c->H, c->D, c->U};
        float *dst[3] = {c->Hf, c->Df, c->Uf};
        const size_t n[3] = {nh, nd, nu};
        for (int q = 0; q < 3; q++)
            hipLaunchKernelGGL(k_to_float, dim3((unsigned)std::min<size_t>((n[q] + 255) / 256, 65536)), dim3(256), 0, c->stream, src[q], dst[q], n[q]);
        if (hipGetLastError() != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "k_to_float launch"));
    }
    if (p->gradH) {
        // packed Hermitian gradient of H: like D for the SoA layout, [k][3][NP] k-major
        const size_t np3 = (size_t)3 * c->np;
        if ((rc = dalloc(c, &c->GE, c->soa ? 3 * se : (size_t)p->nk * np3))) return fail(rc);
        rc = upload_packed(c, p->gradH, 3, st, stage_k, [&](int k0, int kc) {
            for (int x = 0; x < 3; x++)
                if (c->soa) launch_pack(c, st, kc, 3, x, sk, sek, c->GE + x * se + k0 * sk);
                else launch_pack(c, st, kc, 3, x, np3, 1, c->GE + (size_t)k0 * np3 + (size_t)x * c->np);
        });
        if (rc) return fail(rc);
    }
    {
        // [n_nbr][nkp] table, then the stencil-pair pattern (2 kMaxNbr ints)
        const size_t ntab = (size_t)std::max(p->n_nbr, 1) * c->nkp;
        std::vector<int> nbr(ntab + 2 * kMaxNbr, -1);
        for (int k = 0; k < p->nk; k++)
            for (int n = 0; n < p->n_nbr; n++) nbr[(size_t)n * c->nkp + k] = p->nbr[(size_t)k * p->n_nbr + n];
        if (!c->soa && nb > 8 && p->n_nbr > 0 && p->nk % 2 == 0 && c->scol % 2 == 0 &&
            stencil_pairs(p->nbr, p->nk, p->n_nbr, nbr.data() + ntab, c->pself, c->npnew))
            c->pair = 1;
        if ((rc = dalloc(c, &c->nbr, nbr.size()))) return fail(rc);
        if (hipMemcpyAsync(c->nbr, nbr.data(), nbr.size() * sizeof(int), hipMemcpyHostToDevice, c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "upload nbr"));
    }
    {
        // nb <= 4: a thread per k.  Above, blocks that stay resident (from 9 bands
        // LDS and registers hold three per CU) walk the grid.
        const int kpb = c->soa ? kObsThreads : kObsThreads / (nb <= 8 ? WaveGeom<8>::TPK : nb <= 16 ? WaveGeom<16>::TPK : WaveGeom<32>::TPK);
        const int nblk = (p->nk + kpb - 1) / kpb;
        c->obs_blocks = c->soa ? nblk : std::min(nb <= 8 ? kObsMaxBlocks : 3 * kObsMaxBlocks / 4, nblk);
        if ((rc = dalloc(c, &c->part, (size_t)c->obs_blocks * 2 * (nb + kObsSums + 1))) || (rc = dalloc(c, &c->obs_count, 1))) return fail(rc);
        if (!(c->obs = g_results.take())) return fail(set_err(EDUS_ERR_NOMEM, "observables result buffer"));
        if (hipMemsetAsync(c->obs_count, 0, sizeof(unsigned), c->stream) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "memset count"));
    }
    {
        if (c->soa && hipMemsetAsync(c->P0, 0, se * sizeof(double), c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "memset state"));
        if ((rc = upload_packed(c, p->rho0, 1, st, stage_k, [&](int k0, int kc) { launch_pack(c, st, kc, 1, 0, sk, sek, c->P0 + k0 * sk); })))
            return fail(rc);
        if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "table packing"));
        stage.reset();
        if (c->soa) {  // padding columns stay zero in every state buffer
            if (hipMemsetAsync(c->ACC, 0, se * sizeof(double), c->stream) != hipSuccess ||
                hipMemsetAsync(c->YA, 0, se * sizeof(double), c->stream) != hipSuccess ||
                hipMemsetAsync(c->YB, 0, se * sizeof(double), c->stream) != hipSuccess)
                return fail(set_err(EDUS_ERR_HIP, "memset state"));
        }
    }
    if (p->coulomb) {
        const edus_coulomb *q = p->coulomb;
        if (!c->soa) return fail(set_err(EDUS_ERR_UNSUPPORTED, "the Coulomb term is implemented for nb <= 4"));
        if (p->nk_dims[0] != 1 || p->nk_dims[1] * p->nk_dims[2] != p->nk)
            return fail(set_err(EDUS_ERR_UNSUPPORTED, "the Coulomb term needs a 1 x n1 x n2 grid (sample in yz)"));
        if (q->ncut < 1 || !q->A || !q->B || !q->C || !q->D || !q->screen || !q->v_hartree)
            return fail(set_err(EDUS_ERR_INVALID, "incomplete Coulomb tables"));
        if (q->ncut > 32) return fail(set_err(EDUS_ERR_UNSUPPORTED, "Ncut above 32"));
        c->coul = 1; c->N1 = p->nk_dims[1]; c->N2 = p->nk_dims[2]; c->ncut = q->ncut; c->nu = nb * (nb + 1) / 2;
        const int nmm = c->ncut * c->ncut, nb2 = nb * nb;
        // trig tables cos/sin(2 pi m k) with k = -0.5 + i/N (integrationWeight.h:139-175)
        std::vector<double> cx((size_t)c->ncut * c->N1), sx(cx.size()), cy((size_t)c->ncut * c->N2), sy(cy.size());
        for (int m = 0; m < c->ncut; m++) {
            for (int i = 0; i < c->N1; i++) {
                const double kk = (1. / c->N1 != 1.) ? -0.5 + (1. / c->N1) * i : 0.;
                const double arg = 2 * M_PI * m * (kk);
                cx[(size_t)m * c->N1 + i] = cos(arg);
                sx[(size_t)m * c->N1 + i] = sin(arg);
            }
            for (int i = 0; i < c->N2; i++) {
                const double kk = (1. / c->N2 != 1.) ? -0.5 + (1. / c->N2) * i : 0.;
                const double arg = 2 * M_PI * m * (kk);
                cy[(size_t)m * c->N2 + i] = cos(arg);
                sy[(size_t)m * c->N2 + i] = sin(arg);
            }
        }
        auto up = [&](double **dst, const std::vector<double> &v) -> int {
            int r = dalloc(c, dst, v.size());
            return r ? r : upload(c, *dst, v);
        };
        auto upc = [&](double **dst, const double *src, size_t n) -> int { return up(dst, std::vector<double>(src, src + n)); };
        if ((rc = up(&c->cxm, cx)) || (rc = up(&c->sxm, sx)) || (rc = up(&c->cyn, cy)) || (rc = up(&c->syn, sy))) return fail(rc);
        if ((rc = upc(&c->cA, q->A, (size_t)nmm * nb2 * 2)) || (rc = upc(&c->cB, q->B, (size_t)nmm * nb2 * 2)) ||
            (rc = upc(&c->cC, q->C, (size_t)nmm * nb2 * 2)) || (rc = upc(&c->cD, q->D, (size_t)nmm * nb2 * 2)) ||
            (rc = upc(&c->cscreen, q->screen, (size_t)nb2 * 2)) || (rc = upc(&c->cvh, q->v_hartree, (size_t)nb2 * 2)))
            return fail(rc);
        if ((rc = dalloc(c, &c->cS, (size_t)2 * c->N1 * c->ncut * c->np)) ||
            (rc = dalloc(c, &c->cX, (size_t)4 * nmm * nb2 * 2)) || (rc = dalloc(c, &c->cT, (size_t)2 * c->N2 * c->ncut * c->nu * 2)) ||
            (rc = dalloc(c, &c->cEH, nb)) || (rc = dalloc(c, &c->cPW0, se)) || (rc = dalloc(c, &c->cHr, se)) ||
            (rc = dalloc(c, &c->cEk, (size_t)p->nk * nb)) ||
            (q->diag_basis && (rc = dalloc(c, &c->cXw, (size_t)2 * c->nu * c->nkp))))
            return fail(rc);
        if ((rc = up(&c->cX0, std::vector<double>((size_t)4 * nmm * nb2 * 2, 0.0))) || (rc = up(&c->cEH0, std::vector<double>(nb, 0.0))) ||
            (rc = upc(&c->dwb, p->nbr_wb, (size_t)std::max(p->n_nbr, 1) * 3)))
            return fail(rc);
        // P_Wannier_0 = P0, renormalised H starts as H (main_MPI.cpp:214, 330)
        if (hipMemcpyAsync(c->cPW0, c->P0, se * sizeof(double), hipMemcpyDeviceToDevice, c->stream) != hipSuccess ||
            hipMemcpyAsync(c->cHr, c->H, se * sizeof(double), hipMemcpyDeviceToDevice, c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "copy P0/H"));
        // equilibrium: X0 and the Hartree shift of P0 (main_MPI.cpp:276-321); in the
        // diagonal basis of the filled bands, occupation 1 (main_MPI.cpp:291-303)
        if (q->diag_basis) {
            c->coul_diag = 1;
            if ((rc = dalloc(c, &c->cPD, se))) return fail(rc);
            std::vector<double> peq(se, 0.0);
            for (int i = 0; i < c->ncc; i++)
                for (int k = 0; k < p->nk; k++) peq[(size_t)i * c->nkp + k] = 1.0;
            if ((rc = upload(c, c->cPD, peq))) return fail(rc);
            if ((rc = launch_coulomb(c, c->cPD))) return fail(rc);
            if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "diagonal-basis equilibrium"));
        } else if ((rc = launch_coulomb(c, c->P0))) {
            return fail(rc);
        }
        if (hipMemcpyAsync(c->cX0, c->cX, (size_t)4 * nmm * nb2 * 2 * sizeof(double), hipMemcpyDeviceToDevice, c->stream) != hipSuccess ||
            hipMemcpyAsync(c->cEH0, c->cEH, nb * sizeof(double), hipMemcpyDeviceToDevice, c->stream) != hipSuccess)
            return fail(set_err(EDUS_ERR_HIP, "copy equilibrium"));
        c->n_cond = 0.0;
    }
    if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "sync after upload"));
    *out = c;
    g_err.clear();
    return 0;
}

int edus_destroy(edus_ctx *c) {
    if (!c) return 0;
    (void)hipSetDevice(c->dev);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
    if (c->graph) (void)hipGraphDestroy(c->graph);
    if (c->gtab) (void)hipFree(c->gtab);
    for (void *p : c->allocs) (void)hipFree(p);
    if (c->tab) (void)hipFree(c->tab);
    g_results.give(c->obs);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->stream && c->own_stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return 0;
}

static int finish_step(edus_ctx *c, int launches) {
    HIP_TRY(hipEventRecord(c->ev1, c->stream));
    HIP_TRY(hipEventSynchronize(c->ev1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = launches;
    return 0;
}

// Arguments of RK4 stage st (0..3) of size dt reading the field row `row`
// (RungeKutta.cpp:11-150): y_n in P0, stages through YA/YB, k-sum in ACC.
static StageArgs rk4_stage_args(const edus_ctx *c, int st, const double *row, double dt) {
    StageArgs a;
    std::memset(&a, 0, sizeof a);
    a.dt = dt;
    a.tab = row;
    a.dmask = c->dmask;
    a.P0 = c->P0; a.ACC = c->ACC;
    const double dt6 = dt / 6.0, dt3 = dt / 3.0, dt2 = dt / 2.0;
    switch (st) {
        case 0: a.Y = c->P0; a.OUT = c->YA; a.ca = dt6; a.cb = dt2; break;
        case 1: a.Y = c->YA; a.OUT = c->YB; a.ca = dt3; a.cb = dt2; break;
        case 2: a.Y = c->YB; a.OUT = c->YA; a.ca = dt3; a.cb = dt; break;
        default: a.Y = c->YA; a.OUT = c->P0; a.ca = dt6; break;
    }
    return a;
}

// One RK4 step of size dt from the four table rows at `tab`.
static int rk4_step(edus_ctx *c, const double *tab, int rs, double dt) {
    int rc;
    if ((rc = launch_stage<RK1>(c, rk4_stage_args(c, 0, tab, dt)))) return rc;
    if ((rc = launch_stage<RK2>(c, rk4_stage_args(c, 1, tab + rs, dt)))) return rc;
    if ((rc = launch_stage<RK3>(c, rk4_stage_args(c, 2, tab + 2 * rs, dt)))) return rc;
    return launch_stage<RK4S>(c, rk4_stage_args(c, 3, tab + 3 * rs, dt));
}

// Fields [nsteps][3][6] -> table rows [nsteps][4] (stage 3 reuses the midpoint field).
static void rk4_rows(const edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on, std::vector<double> &rows) {
    const int rs = 7 + c->n_nbr;
    rows.assign((size_t)nsteps * 4 * rs, 0.0);
    static const int evalof[4] = {0, 1, 1, 2};
    for (int s = 0; s < nsteps; s++)
        for (int st = 0; st < 4; st++)
            table_row(c, fields + ((size_t)s * 3 + evalof[st]) * 6, grad_on[s], &rows[((size_t)s * 4 + st) * rs]);
}

int edus_step_rk4(edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (c->stepper != EDUS_STEPPER_RK4) return set_err(EDUS_ERR_INVALID, "context was created for another stepper");
    if (nsteps < 0 || (nsteps > 0 && (!fields || !grad_on))) return set_err(EDUS_ERR_INVALID, "bad step arguments");
    const int rs = 7 + c->n_nbr;
    std::vector<double> rows;
    rk4_rows(c, nsteps, fields, grad_on, rows);
    if ((rc = upload_table(c, rows))) return rc;
    HIP_TRY(hipEventRecord(c->ev0, c->stream));
    for (int s = 0; s < nsteps; s++)
        if ((rc = rk4_step(c, c->tab + (size_t)s * 4 * rs, rs, c->dt))) return rc;
    c->nstep += nsteps;
    return finish_step(c, 4 * nsteps);
}

static void drop_graph(edus_ctx *c) {
    if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
    if (c->graph) (void)hipGraphDestroy(c->graph);
    c->gexec = nullptr;
    c->graph = nullptr;
}

int edus_set_field_table(edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (c->stepper != EDUS_STEPPER_RK4) return set_err(EDUS_ERR_UNSUPPORTED, "the field-table path runs RK4 contexts");
    if (nsteps < 1 || !fields || !grad_on) return set_err(EDUS_ERR_INVALID, "bad field table");
    std::vector<double> rows;
    rk4_rows(c, nsteps, fields, grad_on, rows);
    const size_t rs = 7 + (size_t)c->n_nbr;
    int mask = 0;
    for (size_t r = 0; r + rs <= rows.size(); r += rs)
        for (int x = 0; x < 3; x++)
            if (rows[r + x] != 0.0 || rows[r + 3 + x] != 0.0) mask |= 1 << x;
    if (rows.size() > c->gtab_cap || mask != c->gdmask) drop_graph(c);  // the graph holds the table address and the mask
    if (rows.size() > c->gtab_cap) {
        HIP_TRY(hipStreamSynchronize(c->stream));
        if (c->gtab) HIP_TRY(hipFree(c->gtab));
        c->gtab = nullptr;
        c->gtab_cap = 0;
        HIP_TRY(hipMalloc(&c->gtab, rows.size() * sizeof(double)));
        c->gtab_cap = rows.size();
    }
    if (!c->gctr) {
        int *q = nullptr;
        HIP_TRY(hipMalloc(&q, sizeof(int)));
        c->allocs.push_back(q);
        c->gctr = q;
    }
    c->gdmask = mask;
    HIP_TRY(hipMemcpyAsync(c->gtab, rows.data(), rows.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(k_counter_set, dim3(1), dim3(1), 0, c->stream, c->gctr, 0);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));  // the host rows are released on return
    c->gtab_steps = nsteps;
    c->gpos = 0;
    return 0;
}

// One RK4 step whose stage rows come from the field table at the device step
// counter, captured once into a graph (four stage launches and the counter
// advance; Coulomb passes included) and replayed for every step.
static int build_step_graph(edus_ctx *c) {
    const int rs = 7 + c->n_nbr;
    const int saved = c->dmask;
    c->dmask = c->gdmask;
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    int rc = 0;
    for (int st = 0; st < 4 && rc == 0; st++) {
        StageArgs a = rk4_stage_args(c, st, c->gtab + (size_t)st * rs, c->dt);
        a.ctr = c->gctr;
        a.ctr_stride = 4LL * rs;
        rc = st == 0 ? launch_stage<RK1>(c, a) : st == 1 ? launch_stage<RK2>(c, a) : st == 2 ? launch_stage<RK3>(c, a) : launch_stage<RK4S>(c, a);
    }
    if (rc == 0) hipLaunchKernelGGL(k_counter_step, dim3(1), dim3(1), 0, c->stream, c->gctr);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(c->stream, &g);
    c->dmask = saved;
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return set_err(EDUS_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    c->graph = g;
    HIP_TRY(hipGraphInstantiate(&c->gexec, c->graph, nullptr, nullptr, 0));
    return 0;
}

int edus_step_rk4_graph(edus_ctx *c, int32_t nsteps) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (c->stepper != EDUS_STEPPER_RK4) return set_err(EDUS_ERR_UNSUPPORTED, "the field-table path runs RK4 contexts");
    if (!c->gtab) return set_err(EDUS_ERR_INVALID, "no field table: call edus_set_field_table first");
    if (nsteps < 0 || c->gpos + nsteps > c->gtab_steps) return set_err(EDUS_ERR_INVALID, "steps beyond the end of the field table");
    if (!c->gexec && (rc = build_step_graph(c))) return rc;
    HIP_TRY(hipEventRecord(c->ev0, c->stream));
    for (int s = 0; s < nsteps; s++) HIP_TRY(hipGraphLaunch(c->gexec, c->stream));
    c->gpos += nsteps;
    c->nstep += nsteps;
    return finish_step(c, 4 * nsteps);
}

// One AB or Taylor step of size dt from the table row at `tab`
// (Linear_Multistep_ODE_solvers.cpp:1-93, Taylor_DE_solver_deriv_Polynom.cpp:1-177).
static int multistep_one(edus_ctx *c, const double *tab, bool taylor, double dt, const double *tinv) {
    const int o = c->order;
    StageArgs a;
    std::memset(&a, 0, sizeof a);
    a.dt = dt;
    a.order = o;
    a.tab = tab;
    a.HIST = c->HIST;
    // The derivative of step n lives in slot (-n-1) mod order (ODE_solver.h:66-75
    // shifts the ring before each step); slots[s] holds f_{n-s}.
    const long long n = c->nstep;
    for (int q = 0; q < o; q++) a.slots[q] = (int)((((q - n - 1) % o) + o) % o);
    a.slot_out = a.slots[0];
    if (taylor) {
        std::copy(tinv, tinv + (size_t)(o - 1) * (o - 1), a.tinv);
        for (int i = 0; i < o; i++) a.dtp[i] = std::pow(dt, i + 1);
    } else {
        std::copy(c->coef.begin(), c->coef.end(), a.coef);
    }
    double *in = c->cur ? c->YA : c->P0, *out = c->cur ? c->P0 : c->YA;
    a.Y = in; a.P0 = in; a.OUT = out;
    const int rc = taylor ? launch_stage<TAY>(c, a) : launch_stage<ABM>(c, a);
    if (rc) return rc;
    c->cur ^= 1;
    c->nstep++;
    return 0;
}

static int step_multistep(edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on, bool taylor) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (c->stepper != (taylor ? EDUS_STEPPER_TAYLOR : EDUS_STEPPER_AB)) return set_err(EDUS_ERR_INVALID, "context was created for another stepper");
    if (nsteps < 0 || (nsteps > 0 && (!fields || !grad_on))) return set_err(EDUS_ERR_INVALID, "bad step arguments");
    const int rs = 7 + c->n_nbr;
    std::vector<double> rows((size_t)nsteps * rs);
    for (int s = 0; s < nsteps; s++) table_row(c, fields + (size_t)s * 6, grad_on[s], &rows[(size_t)s * rs]);
    if ((rc = upload_table(c, rows))) return rc;
    HIP_TRY(hipEventRecord(c->ev0, c->stream));
    for (int s = 0; s < nsteps; s++)
        if ((rc = multistep_one(c, c->tab + (size_t)s * rs, taylor, c->dt, c->tinv.data()))) return rc;
    return finish_step(c, nsteps);
}

int edus_step_ab(edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on) {
    return step_multistep(c, nsteps, fields, grad_on, false);
}

int edus_step_taylor(edus_ctx *c, int32_t nsteps, const double *fields, const uint8_t *grad_on) {
    return step_multistep(c, nsteps, fields, grad_on, true);
}

namespace {
// Packed array Y of the context (complete in stream order) to the caller's full
// matrices.  From 16 MB of them on they are unpacked on the device, up to 64 MB at a
// time, into the accumulator (scratch between steps for every stepper).  Nothing is
// allocated or freed on the device: that waits for every stream of it (an 82 MB state
// beside another context's steps: 259 ms with a buffer of the call's own, 4 as now).
// Below, the host unpacks.
int download_full(edus_ctx *c, const double *Y, double *out) {
    const size_t per = (size_t)c->np * 16;
    if (c->nk * per < ((size_t)16 << 20)) {
        std::vector<double> st(state_elems(c));
        HIP_TRY(hipMemcpyAsync(st.data(), Y, st.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        unpack_state(c, st, out);
        return 0;
    }
    const int chunk = (int)std::min<size_t>(state_elems(c) / (2 * (size_t)c->np), ((size_t)64 << 20) / per);
    double *buf = c->ACC;
    const size_t sk = c->soa ? 1 : (size_t)c->np, se = c->soa ? (size_t)c->nkp : 1;
    for (int k0 = 0; k0 < c->nk; k0 += chunk) {
        const int kc = std::min(chunk, c->nk - k0);
        const long long n = (long long)kc * c->np;
        hipLaunchKernelGGL(k_unpack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, Y, n, c->nb, sk, se, k0,
                           reinterpret_cast<cd *>(buf));
        HIP_TRY(hipGetLastError());
        HIP_TRY(c->down.copy(out + (size_t)k0 * c->np * 2, buf, kc * per, c->stream));
    }
    return 0;
}
}  // namespace

static const double *current_state(const edus_ctx *c) {
    if (c->stepper == EDUS_STEPPER_RK4) return c->P0;
    return c->cur ? c->YA : c->P0;
}

int edus_step_dyn(edus_ctx *c, double dt, const double *fields, uint8_t grad_on, const double *taylor_tau_inv, double cond,
                  double *max_dp) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!(dt > 0) || !fields || !max_dp) return set_err(EDUS_ERR_INVALID, "bad adaptive step arguments");
    const bool taylor = c->stepper == EDUS_STEPPER_TAYLOR;
    if (!taylor && c->stepper != EDUS_STEPPER_RK4)
        return set_err(EDUS_ERR_UNSUPPORTED, "adaptive steps run RK4 or Taylor contexts");
    if (taylor && !taylor_tau_inv) return set_err(EDUS_ERR_INVALID, "Taylor adaptive step needs tau^-1");
    const int nblk = (c->nk + 255) / 256;
    if (!c->DG) {
        if ((rc = dalloc(c, &c->DG, (size_t)c->nb * c->nk)) || (rc = dalloc(c, &c->dpart, (size_t)nblk))) return rc;
    }
    const int rs = 7 + c->n_nbr;
    std::vector<double> rows;
    if (taylor) {
        rows.resize(rs);
        table_row(c, fields, grad_on, rows.data());
    } else {
        rk4_rows(c, 1, fields, &grad_on, rows);
    }
    if ((rc = upload_table(c, rows))) return rc;
    const size_t sk = c->soa ? 1 : (size_t)c->np, se = c->soa ? (size_t)c->nkp : 1;
    HIP_TRY(hipEventRecord(c->ev0, c->stream));
    hipLaunchKernelGGL(k_diag_save, dim3(nblk), dim3(256), 0, c->stream, current_state(c), c->DG, c->nk, c->nb, sk, se);
    HIP_TRY(hipGetLastError());
    if (taylor) rc = multistep_one(c, c->tab, true, dt, taylor_tau_inv);
    else {
        rc = rk4_step(c, c->tab, rs, dt);
        c->nstep++;
    }
    if (rc) return rc;
    hipLaunchKernelGGL(k_diag_dp, dim3(nblk), dim3(256), 0, c->stream, current_state(c), (const double *)c->DG, c->nk, c->nb, sk, se,
                       cond, c->dpart);
    HIP_TRY(hipGetLastError());
    std::vector<double> part(nblk);
    HIP_TRY(hipMemcpyAsync(part.data(), c->dpart, nblk * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    if ((rc = finish_step(c, taylor ? 1 : 4))) return rc;
    double m = 0.0;
    for (double v : part) m = std::max(m, v);
    *max_dp = m;
    return 0;
}

int edus_eigen_element(edus_ctx *c, int32_t ic, int32_t jc, double *out) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!out || ic < 0 || jc < 0 || ic >= c->nb || jc >= c->nb) return set_err(EDUS_ERR_INVALID, "bad snapshot element");
    if (!c->snap && (rc = dalloc(c, &c->snap, (size_t)2 * c->nk))) return rc;
    const size_t sk = c->soa ? 1 : (size_t)c->np, se = c->soa ? (size_t)c->nkp : 1;
    auto go = [&](auto tag) {
        constexpr int L = decltype(tag)::value, KPB = kElemThreads / L;
        hipLaunchKernelGGL(k_eigen_element<L>, dim3((c->nk + KPB - 1) / KPB), dim3(kElemThreads), 0, c->stream, current_state(c),
                           (const double *)c->U, (const int *)c->eidx, c->nk, c->nb, sk, se, ic, jc, c->snap);
    };
    if (c->soa) go(std::integral_constant<int, 1>{});
    else if (c->nb <= 8) go(std::integral_constant<int, 16>{});
    else go(std::integral_constant<int, 64>{});
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(out, c->snap, (size_t)2 * c->nk * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return 0;
}

int edus_renorm_energies(edus_ctx *c, double *out) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!out) return set_err(EDUS_ERR_INVALID, "null output");
    if (!c->coul) return set_err(EDUS_ERR_INVALID, "no Coulomb term in this context");
    if (!c->cEk_valid) return set_err(EDUS_ERR_INVALID, "call edus_observables first");
    HIP_TRY(hipMemcpyAsync(out, c->cEk, (size_t)c->nk * c->nb * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return 0;
}

int edus_observables(edus_ctx *c, double *pop, double *j1, double *j2, double *tabs, double *pminmax) {
    int rc = check_ctx(c);
    if (rc) return rc;
    ObsArgs o;
    std::memset(&o, 0, sizeof o);
    o.P = current_state(c); o.U = c->U; o.GE = c->GE; o.H = c->coul ? c->cHr : c->H; o.D = c->D; o.eidx = c->eidx;
    o.part = c->part; o.count = c->obs_count; o.out = c->obs;
    o.nk = c->nk; o.nkp = c->nkp; o.nb = c->nb; o.nch = c->nch; o.ncc = c->ncc; o.dherm = c->dherm; o.dxs = (size_t)state_elems(c);
    o.nbr = c->nbr; o.wb = c->dwb; o.n_nbr = c->n_nbr; o.Ek = c->cEk;
    const dim3 grid(c->obs_blocks), block(kObsThreads);
    auto wave = [&](auto tag) {
        constexpr int NBT = decltype(tag)::value;
        const size_t lds = obs_lds_doubles<NBT>() * sizeof(double);
        if (c->nch > 0) hipLaunchKernelGGL((k_obs_wave<NBT, true>), grid, block, lds, c->stream, o);
        else hipLaunchKernelGGL((k_obs_wave<NBT, false>), grid, block, lds, c->stream, o);
    };
    auto small = [&](auto ctag) {
        constexpr bool COUL = decltype(ctag)::value;
        switch (c->nb) {
            case 1: hipLaunchKernelGGL((k_obs_small<1, COUL>), grid, block, 0, c->stream, o); break;
            case 2: hipLaunchKernelGGL((k_obs_small<2, COUL>), grid, block, 0, c->stream, o); break;
            case 3: hipLaunchKernelGGL((k_obs_small<3, COUL>), grid, block, 0, c->stream, o); break;
            default: hipLaunchKernelGGL((k_obs_small<4, COUL>), grid, block, 0, c->stream, o); break;
        }
    };
    if (c->coul) small(std::true_type{});
    else if (c->soa) small(std::false_type{});
    else if (c->nb <= 8) wave(std::integral_constant<int, 8>{});
    else if (c->nb <= 16) wave(std::integral_constant<int, 16>{});
    else wave(std::integral_constant<int, 32>{});
    HIP_TRY(hipGetLastError());
    c->cEk_valid = c->coul != 0;
    HIP_TRY(hipStreamSynchronize(c->stream));
    const double *h = c->obs;
    const int nv = c->nb + kObsSums;
    const int nb = c->nb;
    const double inv = 1. / c->nktot;
    if (pop)
        for (int i = 0; i < nb; i++) pop[i] = h[i] * inv;
    if (j1)
        for (int x = 0; x < 3; x++) { j1[2 * x] = h[nb + x] * c->j_norm; j1[2 * x + 1] = 0.0; }
    if (j2)
        for (int x = 0; x < 3; x++) { j2[2 * x] = h[nb + 3 + 2 * x] * c->j_norm; j2[2 * x + 1] = h[nb + 4 + 2 * x] * c->j_norm; }
    if (tabs)
        for (int x = 0; x < 3; x++) { tabs[2 * x] = h[nb + 9 + 2 * x] * c->tabs_norm; tabs[2 * x + 1] = h[nb + 10 + 2 * x] * c->tabs_norm; }
    if (pminmax) { pminmax[0] = h[nv]; pminmax[1] = h[nv + 1]; }
    if (c->coul) {  // n_cond: largest printed population (Observables_MPI.h:413-426)
        double nc = 0;
        for (int i = 0; i < nb; i++) {
            const double v = (i < c->ncc) ? 1.0 - h[i] * inv : h[i] * inv;
            if (v > nc) nc = v;
        }
        if (mean_field_gate(nc) != mean_field_gate(c->n_cond)) drop_graph(c);  // a captured step holds the gate
        c->n_cond = nc;
    }
    return 0;
}

int edus_rhs(edus_ctx *c, const double *field6, uint8_t grad_on, double *pv) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!field6 || !pv) return set_err(EDUS_ERR_INVALID, "null argument");
    std::vector<double> row(7 + c->n_nbr);
    table_row(c, field6, grad_on, row.data());
    if ((rc = upload_table(c, row))) return rc;
    StageArgs a;
    std::memset(&a, 0, sizeof a);
    a.tab = c->tab;
    a.Y = current_state(c);
    a.OUT = c->YB;
    if ((rc = launch_stage<RHSO>(c, a))) return rc;
    return download_full(c, c->YB, pv);
}

int edus_get_state(edus_ctx *c, double *rho) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!rho) return set_err(EDUS_ERR_INVALID, "null output");
    return download_full(c, current_state(c), rho);
}

int edus_set_state(edus_ctx *c, const double *rho) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!rho) return set_err(EDUS_ERR_INVALID, "null input");
    std::vector<double> st;
    pack_state(c, rho, st);
    HIP_TRY(hipMemcpyAsync(const_cast<double *>(current_state(c)), st.data(), st.size() * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return 0;
}

// Schedule of the stage kernels picked by timing the context's own right-hand
// side: every candidate gives the same sums for every k (only the order of the
// workgroups or their size changes), so the choice cannot change a result.
int edus_autotune(edus_ctx *c, const double *field6, uint8_t grad_on, int32_t reps, int32_t *chosen) {
    int rc = check_ctx(c);
    if (rc) return rc;
    if (!field6 || reps < 1 || reps > 1000) return set_err(EDUS_ERR_INVALID, "bad autotune arguments");
    std::vector<double> row(7 + c->n_nbr);
    table_row(c, field6, grad_on, row.data());
    if ((rc = upload_table(c, row))) return rc;
    StageArgs a;
    std::memset(&a, 0, sizeof a);
    a.tab = c->tab;
    a.Y = current_state(c);
    a.OUT = c->YB;  // scratch between steps: the state is not touched
    std::vector<int> cand;
    if (c->soa) {
        cand = {64, 128};
        if (c->nb <= 2 && !c->diss) cand.push_back(256);  // with more terms 128 k fill kSmallMaxThreads
    } else {
        cand.push_back(0);
        if (c->scol > 0)
            for (int w : {16, 32, 64, 128, 256})
                if (w < c->scol) cand.push_back(w);
    }
    // 1..4 bands: the right-hand sides of 64 and 128 k per workgroup are even, and a
    // choice by their noise can cost the step, whose kernel holds more (4 bands 1000 x
    // 1000, AB4 step 290 and 372 us; 3 bands, Taylor 159 and 180): a larger one has to
    // gain 3 %.
    const float gain = c->soa ? 0.97f : 1.f;
    int &knob = c->soa ? c->tpb : c->sw;
    const int before = knob;
    int best = cand[0];
    float best_ms = 0.f;
    for (size_t i = 0; i < cand.size(); i++) {
        knob = cand[i];
        if ((rc = launch_stage<RHSO>(c, a))) { knob = before; return rc; }  // untimed
        HIP_TRY(hipEventRecord(c->ev0, c->stream));
        for (int r = 0; r < reps; r++)
            if ((rc = launch_stage<RHSO>(c, a))) { knob = before; return rc; }
        HIP_TRY(hipEventRecord(c->ev1, c->stream));
        HIP_TRY(hipEventSynchronize(c->ev1));
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, c->ev0, c->ev1));
        if (i == 0 || ms < gain * best_ms) { best_ms = ms; best = cand[i]; }
    }
    knob = best;
    if (best != before) drop_graph(c);  // a captured step holds the old launch shape
    if (chosen) *chosen = best;
    return 0;
}

int edus_last_step_time(edus_ctx *c, double *ms, int32_t *nlaunch) {
    if (!c) return set_err(EDUS_ERR_INVALID, "null context");
    if (ms) *ms = c->last_ms;
    if (nlaunch) *nlaunch = c->last_launches;
    return 0;
}

int edus_launch_schedule(edus_ctx *c, int32_t *out) {
    if (!c || !out) return set_err(EDUS_ERR_INVALID, "null argument");
    out[0] = c->soa ? 0 : (c->nb <= 8 ? 8 : c->nb <= 16 ? 16 : 32);
    out[1] = c->sw;
    out[2] = c->pair;
    out[3] = c->pair ? c->npnew : 0;
    out[4] = c->soa ? small_group(c) : 0;
    return 0;
}

// ---------------------------------------------------------------- batched instances
struct edus_batch {
    int dev = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<edus_ctx *> inst;
    struct Cls {
        bool soa = true;
        int nb_small = 0, nbt = 0, precision = EDUS_PRECISION_FP64, diss = 0, pair = 0;
        std::vector<int> members;
        int2 *blk = nullptr;
        int nblocks = 0;
    };
    std::vector<Cls> cls;
    BatchEntry *entries = nullptr;
    int *masks = nullptr;   // [n] dipole components the call's fields need, per member
    double *tab = nullptr;  // [step][stage][R_tot]; instance i's row at roff[i]
    size_t tab_steps = 0;
    int R_tot = 0;
    std::vector<int> roff;
    std::vector<void *> allocs;
    double last_ms = 0.0;
    int last_launches = 0;
};

extern "C++" {
namespace {

int batch_write_entries(edus_batch *b) {
    std::vector<BatchEntry> e(b->inst.size());
    for (size_t i = 0; i < b->inst.size(); i++) {
        const edus_ctx *c = b->inst[i];
        e[i].c = const_args(c);
        for (int st = 0; st < 4; st++) {
            e[i].a[st] = rk4_stage_args(c, st, b->tab + (size_t)st * b->R_tot + b->roff[i], c->dt);
            e[i].a[st].dmask = 7;  // replaced per call by the member's mask (b->masks)
        }
    }
    HIP_TRY(hipMemcpyAsync(b->entries, e.data(), e.size() * sizeof(BatchEntry), hipMemcpyHostToDevice, b->stream));
    HIP_TRY(hipStreamSynchronize(b->stream));
    return 0;
}

int batch_table_capacity(edus_batch *b, size_t nsteps) {
    if (nsteps <= b->tab_steps) return 0;
    HIP_TRY(hipStreamSynchronize(b->stream));
    if (b->tab) HIP_TRY(hipFree(b->tab));
    b->tab = nullptr;
    const size_t cap = std::max<size_t>(nsteps, 16);
    HIP_TRY(hipMalloc(&b->tab, cap * 4 * (size_t)b->R_tot * sizeof(double)));
    b->tab_steps = cap;
    return batch_write_entries(b);
}

template <int MODE>
int batch_launch(edus_batch *b, const edus_batch::Cls &k, size_t tab_step) {
    const dim3 grid(k.nblocks);
    if (k.soa) {
        auto go = [&](auto dtag) {
            constexpr bool DISS = decltype(dtag)::value;
            auto nbgo = [&](auto ntag) {
                constexpr int NB = decltype(ntag)::value, R = SmallGeom<NB, DISS>::R;
                hipLaunchKernelGGL((k_stage_small_batch<NB, MODE, DISS>), grid, dim3(kSmallBatchThreads, R),
                                   (size_t)R * NB * NB * kSmallBatchThreads * sizeof(double), b->stream, b->entries, k.blk, b->masks, tab_step);
            };
            switch (k.nb_small) {
                case 1: nbgo(std::integral_constant<int, 1>{}); break;
                case 2: nbgo(std::integral_constant<int, 2>{}); break;
                case 3: nbgo(std::integral_constant<int, 3>{}); break;
                default: nbgo(std::integral_constant<int, 4>{}); break;
            }
        };
        if (k.diss) go(std::true_type{});
        else go(std::false_type{});
    } else {
        auto go = [&](auto tag, auto ptag) {
            constexpr int NBT = decltype(tag)::value, KPB = WaveGeom<NBT>::KPB;
            constexpr bool PAIR = decltype(ptag)::value;
            const dim3 block(WaveGeom<NBT>::TPK * KPB);
            const size_t lds_f = (size_t)KPB * wave_lds_doubles<NBT, float>(k.diss) * 8;
            const size_t lds_d = (size_t)KPB * wave_lds_doubles<NBT, double>(k.diss) * 8;
            if (k.precision == EDUS_PRECISION_MIXED)
                hipLaunchKernelGGL((k_stage_wave_batch<NBT, MODE, float, PAIR>), grid, block, lds_f, b->stream, b->entries, k.blk, b->masks, tab_step);
            else
                hipLaunchKernelGGL((k_stage_wave_batch<NBT, MODE, double, PAIR>), grid, block, lds_d, b->stream, b->entries, k.blk, b->masks, tab_step);
        };
        if (k.nbt == 8) go(std::integral_constant<int, 8>{}, std::false_type{});
        else if (k.nbt == 16 && k.pair) go(std::integral_constant<int, 16>{}, std::true_type{});
        else if (k.nbt == 16) go(std::integral_constant<int, 16>{}, std::false_type{});
        else if (k.pair) go(std::integral_constant<int, 32>{}, std::true_type{});
        else go(std::integral_constant<int, 32>{}, std::false_type{});
    }
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace
}  // extern "C++"

int edus_batch_destroy(edus_batch *b) {
    if (!b) return 0;
    (void)hipSetDevice(b->dev);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (edus_ctx *c : b->inst) edus_destroy(c);
    for (auto &k : b->cls)
        if (k.blk) (void)hipFree(k.blk);
    for (void *p : b->allocs) (void)hipFree(p);
    if (b->tab) (void)hipFree(b->tab);
    if (b->ev0) (void)hipEventDestroy(b->ev0);
    if (b->ev1) (void)hipEventDestroy(b->ev1);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return 0;
}

int edus_batch_create(const edus_problem *const *problems, int32_t n, edus_batch **out) {
    if (!problems || !out || n < 1) return set_err(EDUS_ERR_INVALID, "null argument or empty batch");
    *out = nullptr;
    for (int i = 0; i < n; i++) {
        if (!problems[i]) return set_err(EDUS_ERR_INVALID, "null problem in batch");
        if (problems[i]->stepper != EDUS_STEPPER_RK4) return set_err(EDUS_ERR_UNSUPPORTED, "batches run RK4 problems");
        if (problems[i]->coulomb) return set_err(EDUS_ERR_UNSUPPORTED, "batches do not carry the Coulomb term");
        if (problems[i]->precision == EDUS_PRECISION_MIXED32 || problems[i]->precision == EDUS_PRECISION_BF16X3)
            return set_err(EDUS_ERR_UNSUPPORTED, "batches run FP64 or EDUS_PRECISION_MIXED members");
    }
    auto *b = new edus_batch();
    auto fail = [&](int rc) { edus_batch_destroy(b); return rc; };
    if (hipGetDevice(&b->dev) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "hipGetDevice failed"));
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "stream create failed"));
    if (hipEventCreate(&b->ev0) != hipSuccess || hipEventCreate(&b->ev1) != hipSuccess) return fail(set_err(EDUS_ERR_HIP, "event create failed"));
    for (int i = 0; i < n; i++) {
        edus_ctx *c = nullptr;
        const int rc = edus_create(problems[i], &c);
        if (rc) return fail(rc);
        // every instance works on the batch's stream
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamDestroy(c->stream);
        c->stream = b->stream;
        c->own_stream = false;
        b->inst.push_back(c);
        b->roff.push_back(b->R_tot);
        b->R_tot += 7 + c->n_nbr;
    }
    // kernel classes: small kernels by band count, wave kernels by tile and
    // precision, each split by the presence of dephasing and by stencil pairing
    for (int i = 0; i < n; i++) {
        const edus_ctx *c = b->inst[i];
        const int nbt = c->soa ? 0 : (c->nb <= 8 ? 8 : c->nb <= 16 ? 16 : 32);
        edus_batch::Cls *hit = nullptr;
        for (auto &k : b->cls)
            if (k.soa == c->soa && k.nb_small == (c->soa ? c->nb : 0) && k.nbt == nbt && k.precision == c->precision &&
                k.diss == c->diss && k.pair == (int)runs_paired(c))
                hit = &k;
        if (!hit) {
            b->cls.emplace_back();
            hit = &b->cls.back();
            hit->soa = c->soa; hit->nb_small = c->soa ? c->nb : 0; hit->nbt = nbt; hit->precision = c->precision;
            hit->diss = c->diss; hit->pair = runs_paired(c);
        }
        hit->members.push_back(i);
    }
    for (auto &k : b->cls) {
        std::vector<int2> map;
        for (int i : k.members) {
            const edus_ctx *c = b->inst[i];
            const int kpb = c->nb <= 8 ? WaveGeom<8>::KPB : c->nb <= 16 ? WaveGeom<16>::KPB : WaveGeom<32>::KPB;
            const int nblk = c->soa    ? (c->nk + kSmallBatchThreads - 1) / kSmallBatchThreads
                             : runs_paired(c) ? c->nk / 2
                                       : (c->nk + kpb - 1) / kpb;
            for (int q = 0; q < nblk; q++) map.push_back(make_int2(i, q));
        }
        k.nblocks = (int)map.size();
        if (hipMalloc(&k.blk, map.size() * sizeof(int2)) != hipSuccess ||
            hipMemcpy(k.blk, map.data(), map.size() * sizeof(int2), hipMemcpyHostToDevice) != hipSuccess)
            return fail(set_err(EDUS_ERR_NOMEM, "batch block table"));
    }
    void *ent = nullptr;
    if (hipMalloc(&ent, (size_t)n * sizeof(BatchEntry)) != hipSuccess) return fail(set_err(EDUS_ERR_NOMEM, "batch entries"));
    b->allocs.push_back(ent);
    b->entries = static_cast<BatchEntry *>(ent);
    void *msk = nullptr;
    if (hipMalloc(&msk, (size_t)n * sizeof(int)) != hipSuccess) return fail(set_err(EDUS_ERR_NOMEM, "batch masks"));
    b->allocs.push_back(msk);
    b->masks = static_cast<int *>(msk);
    int rc = batch_table_capacity(b, 16);
    if (rc) return fail(rc);
    *out = b;
    g_err.clear();
    return 0;
}

// ---------------------------------------------------------------- setup: batched eigensolve
// Rows a of U are conj(v_a), the eigenvectors of H in ascending eigenvalue order
// (Wannier.h:496-542).  rocSOLVER's batched Jacobi solver reads our row-major
// H as its column-major transpose conj(H) (its lower triangle is our upper
// one, the triangle the engine packs), whose eigenvectors conj(v_a) it
// returns as columns, i.e. as our rows: the memory is U up to the phases,
// which k_eig_phase then fixes (largest-modulus component real positive, the
// first of equal moduli within 1e-12 -- the host Jacobi's convention).
__global__ void k_eig_phase(cd *U, int nmat, int nb) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= (long long)nmat * nb) return;
    cd *row = U + r * nb;
    int best = 0;
    double bm = -1.0;
    for (int i = 0; i < nb; i++) {
        const double m = sqrt(row[i].x * row[i].x + row[i].y * row[i].y);
        if (m > bm + 1e-12) { bm = m; best = i; }
    }
    const cd ub = row[best];
    const double mag = sqrt(ub.x * ub.x + ub.y * ub.y);
    if (mag == 0.0) return;
    const cd ph = mk(ub.x / mag, -ub.y / mag);  // conj(u_best) / |u_best|
    for (int i = 0; i < nb; i++) row[i] = cmul(row[i], ph);
}

int edus_eigh_batched(int32_t nmat, int32_t nb, const double *H, double *w, double *U) {
    if (nmat < 0 || nb < 1 || nb > EDUS_MAX_NB || (nmat > 0 && (!H || !w || !U))) return set_err(EDUS_ERR_INVALID, "bad eigensolve arguments");
    if (nmat == 0) return 0;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(EDUS_ERR_NODEVICE, "no HIP device visible");
    const size_t nn = (size_t)nb * nb, chunk = std::min<size_t>((size_t)nmat, 32768);
    rocblas_handle hd = nullptr;
    if (rocblas_create_handle(&hd) != rocblas_status_success) return set_err(EDUS_ERR_HIP, "rocblas_create_handle failed");
    hipStream_t st = nullptr;
    void *dA = nullptr, *dW = nullptr, *dres = nullptr, *dinfo = nullptr, *dsw = nullptr;
    int rc = 0;
    auto done = [&](int r) {
        if (st) (void)hipStreamSynchronize(st);
        (void)hipFree(dA); (void)hipFree(dW); (void)hipFree(dres); (void)hipFree(dinfo); (void)hipFree(dsw);
        if (st) (void)hipStreamDestroy(st);
        rocblas_destroy_handle(hd);
        return r;
    };
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess || rocblas_set_stream(hd, st) != rocblas_status_success)
        return done(set_err(EDUS_ERR_HIP, "eigensolve stream"));
    if (hipMalloc(&dA, chunk * nn * 16) != hipSuccess || hipMalloc(&dW, chunk * nb * 8) != hipSuccess ||
        hipMalloc(&dres, chunk * 8) != hipSuccess || hipMalloc(&dinfo, chunk * 4) != hipSuccess || hipMalloc(&dsw, chunk * 4) != hipSuccess)
        return done(set_err(EDUS_ERR_NOMEM, "eigensolve buffers"));
    std::vector<int> info(chunk);
    for (size_t m0 = 0; m0 < (size_t)nmat; m0 += chunk) {
        const size_t m = std::min(chunk, (size_t)nmat - m0);
        if (hipMemcpyAsync(dA, H + m0 * nn * 2, m * nn * 16, hipMemcpyHostToDevice, st) != hipSuccess)
            return done(set_err(EDUS_ERR_HIP, "eigensolve upload"));
        const rocblas_status s1 = rocsolver_zheevj_strided_batched(
            hd, rocblas_esort_ascending, rocblas_evect_original, rocblas_fill_lower, nb, static_cast<rocblas_double_complex *>(dA), nb,
            (rocblas_stride)nn, 0.0, static_cast<double *>(dres), 100, static_cast<rocblas_int *>(dsw), static_cast<double *>(dW), nb,
            static_cast<rocblas_int *>(dinfo), (rocblas_int)m);
        if (s1 != rocblas_status_success) return done(set_err(EDUS_ERR_HIP, "rocsolver_zheevj_strided_batched failed"));
        const long long rows = (long long)m * nb;
        hipLaunchKernelGGL(k_eig_phase, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, st, static_cast<cd *>(dA), (int)m, nb);
        if (hipGetLastError() != hipSuccess) return done(set_err(EDUS_ERR_HIP, "k_eig_phase launch"));
        if (hipMemcpyAsync(U + m0 * nn * 2, dA, m * nn * 16, hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipMemcpyAsync(w + m0 * nb, dW, m * nb * 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipMemcpyAsync(info.data(), dinfo, m * 4, hipMemcpyDeviceToHost, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
            return done(set_err(EDUS_ERR_HIP, "eigensolve download"));
        for (size_t i = 0; i < m; i++)
            if (info[i] != 0) return done(set_err(EDUS_ERR_HIP, "Jacobi eigensolver did not converge for matrix " + std::to_string(m0 + i)));
    }
    g_err.clear();
    return done(rc);
}

int edus_batch_size(const edus_batch *b) { return b ? (int)b->inst.size() : 0; }

int edus_batch_step_rk4(edus_batch *b, int32_t nsteps, const double *const *fields, const uint8_t *const *grad_on) {
    if (!b) return set_err(EDUS_ERR_INVALID, "null batch");
    HIP_TRY(hipSetDevice(b->dev));
    const int n = (int)b->inst.size();
    if (nsteps < 0 || (nsteps > 0 && (!fields || !grad_on))) return set_err(EDUS_ERR_INVALID, "bad step arguments");
    if (nsteps == 0) return 0;
    for (int i = 0; i < n; i++)
        if (!fields[i] || !grad_on[i]) return set_err(EDUS_ERR_INVALID, "null fields of a batch member");
    int rc = batch_table_capacity(b, (size_t)nsteps);
    if (rc) return rc;
    std::vector<double> rows((size_t)nsteps * 4 * b->R_tot), one;
    std::vector<int> masks(n, 0);
    for (int i = 0; i < n; i++) {
        const edus_ctx *c = b->inst[i];
        const int rs = 7 + c->n_nbr;
        rk4_rows(c, nsteps, fields[i], grad_on[i], one);
        for (size_t r = 0; r < (size_t)nsteps * 4; r++) {
            std::copy(one.begin() + r * rs, one.begin() + (r + 1) * rs, rows.begin() + r * b->R_tot + b->roff[i]);
            for (int x = 0; x < 3; x++)
                if (one[r * rs + x] != 0.0 || one[r * rs + 3 + x] != 0.0) masks[i] |= 1 << x;
        }
    }
    HIP_TRY(hipMemcpyAsync(b->tab, rows.data(), rows.size() * sizeof(double), hipMemcpyHostToDevice, b->stream));
    HIP_TRY(hipMemcpyAsync(b->masks, masks.data(), n * sizeof(int), hipMemcpyHostToDevice, b->stream));
    HIP_TRY(hipEventRecord(b->ev0, b->stream));
    int launches = 0;
    for (int s = 0; s < nsteps; s++) {
        const size_t ts = (size_t)s * 4 * b->R_tot;
        for (const auto &k : b->cls) if ((rc = batch_launch<RK1>(b, k, ts))) return rc;
        for (const auto &k : b->cls) if ((rc = batch_launch<RK2>(b, k, ts))) return rc;
        for (const auto &k : b->cls) if ((rc = batch_launch<RK3>(b, k, ts))) return rc;
        for (const auto &k : b->cls) if ((rc = batch_launch<RK4S>(b, k, ts))) return rc;
        launches += 4 * (int)b->cls.size();
    }
    HIP_TRY(hipEventRecord(b->ev1, b->stream));
    HIP_TRY(hipEventSynchronize(b->ev1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, b->ev0, b->ev1));
    b->last_ms = ms;
    b->last_launches = launches;
    for (edus_ctx *c : b->inst) c->nstep += nsteps;
    return 0;
}

int edus_batch_last_step_time(const edus_batch *b, double *ms, int32_t *nlaunch) {
    if (!b) return set_err(EDUS_ERR_INVALID, "null batch");
    if (ms) *ms = b->last_ms;
    if (nlaunch) *nlaunch = b->last_launches;
    return 0;
}

edus_ctx *edus_batch_member(edus_batch *b, int32_t i) {
    if (!b || i < 0 || i >= (int)b->inst.size()) {
        set_err(EDUS_ERR_INVALID, "batch member index out of range");
        return nullptr;
    }
    return b->inst[i];
}

int edus_coulomb_coefficients(const edus_coulomb_gen *g, double *Ao, double *Bo, double *Co, double *Do, double *screen, double *vh) {
    if (!g || !Ao || !Bo || !Co || !Do || !screen || !vh || !g->g || !g->disp) return set_err(EDUS_ERR_INVALID, "null argument");
    const int nb = g->nb, nc = g->ncut, N = g->n_sum, Np = g->n_peak;
    if (nb < 1 || nb > 4) return set_err(EDUS_ERR_UNSUPPORTED, "the coefficient generator supports 1..4 bands");
    if (nc < 1 || N < 3 || Np < 3 || g->n_g < 1) return set_err(EDUS_ERR_INVALID, "ncut, n_sum, n_peak, n_g out of range");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(EDUS_ERR_NODEVICE, "no HIP device visible");
    const int nb2 = nb * nb, npair = nb * (nb - 1) / 2, nw = 1 + 2 * npair, nmm = nc * nc, ntrig = 2 * nc;
    const double twopi = 2 * M_PI;
    auto vq = [&](double q2, double qtf) {
        return (g->rytova_keldysh ? g->eps_area * std::sqrt(q2 + qtf * qtf) * (std::sqrt(q2) * g->r0 + 1.0)
                                  : g->eps_area * std::sqrt(q2 + qtf * qtf));
    };
    // band pairs ic < jc and their beta = b.(d_ic - d_jc)
    std::vector<int> pic, pjc;
    CGenArgs a;
    std::memset(&a, 0, sizeof a);
    for (int ic = 0; ic < nb; ic++)
        for (int jc = ic + 1; jc < nb; jc++) {
            const int p = (int)pic.size();
            pic.push_back(ic);
            pjc.push_back(jc);
            double b1d = 0, b2d = 0;
            for (int x = 0; x < 3; x++) {
                const double dd = g->disp[ic * 3 + x] - g->disp[jc * 3 + x];
                b1d += g->b1[x] * dd;
                b2d += g->b2[x] * dd;
            }
            a.beta1[p] = b1d;
            a.beta2[p] = b2d;
        }
    // Hartree term at q = 0 on the host (Fourier_Coulomb.cpp:173-193): V = 0 where
    // the G offsets sum to <= 0, as written there.
    {
        double w00 = 0;
        std::vector<std::complex<double>> wp(npair, 0.0);
        for (int ig = 0; ig < g->n_g; ig++) {
            const double gx = g->g[2 * ig], gy = g->g[2 * ig + 1];
            double cart[3];
            for (int x = 0; x < 3; x++) cart[x] = g->b1[x] * gx + g->b2[x] * gy;
            const double q2 = cart[0] * cart[0] + cart[1] * cart[1] + cart[2] * cart[2];
            const double V = ((gx + gy) < 1e-16) ? 0.0 : twopi / vq(q2, g->qtf);
            w00 += V;
            for (int p = 0; p < npair; p++) {
                double phi = 0;
                for (int x = 0; x < 3; x++) phi += cart[x] * (g->disp[pic[p] * 3 + x] - g->disp[pjc[p] * 3 + x]);
                wp[p] += V * std::exp(std::complex<double>(0.0, phi));
            }
        }
        for (int i = 0; i < nb2 * 2; i++) vh[i] = 0.0;
        for (int ic = 0; ic < nb; ic++) vh[(ic * nb + ic) * 2] = w00;
        for (int p = 0; p < npair; p++) {
            const double r = wp[p].real();
            vh[(pic[p] * nb + pjc[p]) * 2] = r;
            vh[(pjc[p] * nb + pic[p]) * 2] = r;
        }
    }
    // The lattice's Cholesky frame: q b1 + q' b2 = (l11 q + l21 q', l22 q') in
    // orthonormal components of the plane.
    auto two = [](long double v, double (&o)[2]) {
        o[0] = (double)v;
        o[1] = (double)(v - (long double)o[0]);
    };
    long double l11, l21, l22;
    {
        long double g11 = 0, g12 = 0, g22 = 0, c2 = 0;
        for (int x = 0; x < 3; x++) {
            const long double u = g->b1[(x + 1) % 3], v = g->b1[(x + 2) % 3], p = g->b2[(x + 1) % 3], r = g->b2[(x + 2) % 3];
            g11 += (long double)g->b1[x] * g->b1[x];
            g12 += (long double)g->b1[x] * g->b2[x];
            g22 += (long double)g->b2[x] * g->b2[x];
            c2 += (u * r - v * p) * (u * r - v * p);
        }
        l11 = sqrtl(g11);
        l21 = g11 > 0 ? g12 / l11 : 0.0L;
        l22 = g11 > 0 ? sqrtl(c2) / l11 : sqrtl(g22);
    }
    two(l11, a.l11);
    two(l21, a.l21);
    two(l22, a.l22);
    two((long double)twopi / g->eps_area, a.scale);
    // per-G data: components and e^{i G.beta_p}
    const int grow = 2 + 2 * npair;
    std::vector<double> gd((size_t)g->n_g * grow);
    for (int ig = 0; ig < g->n_g; ig++) {
        const double gx = g->g[2 * ig], gy = g->g[2 * ig + 1];
        double *r = &gd[(size_t)ig * grow];
        r[0] = (double)(l11 * gx + l21 * gy);
        r[1] = (double)(l22 * gy);
        for (int p = 0; p < npair; p++) {
            const double ph = gx * a.beta1[p] + gy * a.beta2[p];
            r[2 + 2 * p] = std::cos(ph);
            r[3 + 2 * p] = std::sin(ph);
        }
    }
    // Is the list of G closed under G -> -G (as every shell |G| < R is)?
    bool gsym;
    {
        std::vector<std::pair<int, int>> l(g->n_g), m(g->n_g);
        for (int ig = 0; ig < g->n_g; ig++) {
            l[ig] = {g->g[2 * ig], g->g[2 * ig + 1]};
            m[ig] = {-g->g[2 * ig], -g->g[2 * ig + 1]};
        }
        std::sort(l.begin(), l.end());
        std::sort(m.begin(), m.end());
        gsym = l == m;
    }
    // Simpson weights and trig tables (integrationWeight.h:5-18)
    auto simpson = [](int n, std::vector<double> &q, std::vector<double> &w) {
        q.resize(n);
        w.resize(n);
        const double hs = 3 * (n - 1);
        for (int i = 0; i < n; i++) q[i] = (double)(2 * i - (n - 1)) / (double)(2 * (n - 1));  // as cgen_q
        w[0] = 1 / hs;
        for (int i = 1; i < n; i += 2) w[i] = 4.0 / hs;
        for (int i = 2; i < n; i += 2) w[i] = 2.0 / hs;
        w[n - 1] = 1 / hs;
    };
    std::vector<double> q, w;
    simpson(N, q, w);
    const int ldt = (ntrig + 16 * kCgTT - 1) / (16 * kCgTT) * (16 * kCgTT);
    std::vector<double> wtrig((size_t)ntrig * N), wt((size_t)N * ldt, 0.0);  // [t][i], and [i][t] padded with zeros
    for (int t = 0; t < ntrig; t++)
        for (int i = 0; i < N; i++) {
            const int m = t < nc ? t : t - nc;
            const double arg = 2 * M_PI * m * q[i];
            wt[(size_t)i * ldt + t] = wtrig[(size_t)t * N + i] = w[i] * (t < nc ? std::cos(arg) : std::sin(arg));
        }
    const size_t nq = (size_t)N * N;
    double *dG = nullptr, *dW = nullptr, *dTr = nullptr, *dWt = nullptr, *dT = nullptr, *dS = nullptr, *dCoef = nullptr, *dW0 = nullptr,
           *dPart = nullptr, *dSum = nullptr;
    int *dQl = nullptr;
    auto cleanup = [&]() {
        for (void *p : {(void *)dG, (void *)dW, (void *)dTr, (void *)dWt, (void *)dT, (void *)dS, (void *)dCoef, (void *)dW0, (void *)dPart,
                        (void *)dSum, (void *)dQl})
            (void)hipFree(p);
    };
    auto fail = [&](int code, const std::string &m) {
        cleanup();
        return set_err(code, m);
    };
    // A set of n q: chunks of blocks of q, the G list in gs parts when the chunk alone
    // would leave the chip idle (four waves per SIMD: 1024 blocks).
    const long long chunk = 1LL << 21;
    auto blocks_of = [](long long n) { return (int)((n + kCgThreads * kCgQ - 1) / (kCgThreads * kCgQ)); };
    auto split_of = [&](long long n) { return (int)std::max<long long>(1, std::min<long long>({16, 1024 / blocks_of(n), g->n_g / kCgTile})); };
    auto sums_of = [&](long long n) { return (size_t)std::min(n, chunk) * split_of(std::min(n, chunk)) * nw * 8; };
    const long long half = gsym ? (long long)(nq + 1) / 2 : (long long)nq;
    if (hipMalloc(&dG, gd.size() * 8) != hipSuccess || hipMalloc(&dW, nq * nw * 8) != hipSuccess ||
        hipMalloc(&dTr, wtrig.size() * 8) != hipSuccess || hipMalloc(&dWt, wt.size() * 8) != hipSuccess ||
        hipMalloc(&dT, (size_t)ntrig * N * nw * 8) != hipSuccess || hipMalloc(&dS, (size_t)ntrig * ntrig * nw * 8) != hipSuccess ||
        hipMalloc(&dCoef, (size_t)4 * nmm * nb2 * 2 * 8) != hipSuccess || hipMalloc(&dSum, sums_of(half)) != hipSuccess)
        return fail(EDUS_ERR_NOMEM, "coefficient generator buffers");
    if (hipMemcpy(dG, gd.data(), gd.size() * 8, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dWt, wt.data(), wt.size() * 8, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dTr, wtrig.data(), wtrig.size() * 8, hipMemcpyHostToDevice) != hipSuccess)
        return fail(EDUS_ERR_HIP, "coefficient generator upload");
    a.npair = npair; a.n_g = g->n_g; a.N = N; a.mode = 0;
    a.qtf2 = g->qtf * g->qtf; a.r0 = g->rytova_keldysh ? g->r0 : 0.0;
    int form = CG_GENERAL;
    {
        // the largest (q^2 + qTF^2) (|q| r0 + 1)^2 of the sums, and no lattice or screening
        // so small that its square is not a normal number
        double gx = 0, gy = 0;
        for (int ig = 0; ig < g->n_g; ig++) {
            gx = std::max(gx, std::fabs((double)g->g[2 * ig]));
            gy = std::max(gy, std::fabs((double)g->g[2 * ig + 1]));
        }
        const double b1 = (double)l11, b2 = std::hypot((double)l21, (double)l22), qm = (gx + 0.5) * b1 + (gy + 0.5) * b2, t = qm * a.r0 + 1.0;
        if (a.r0 >= 0.0 && (qm * qm + a.qtf2) * t * t < 1e300 && a.r0 < 1e100 && b1 > 1e-100 && l22 > 1e-100 &&
            (a.qtf2 == 0.0 || a.qtf2 > 1e-290))
            form = g->rytova_keldysh ? CG_RYTOVA : CG_PLAIN;
    }
    a.g = dG; a.qlist = nullptr;
    // sums over G of q numbers [q0, q0 + n) and W from them (of a set of ntot; mirror:
    // its second half comes from the first)
    auto lattice_sum = [&](CGenArgs c, long long q0, int n, long long ntot, bool mirror, double *W) {
        const int gs = split_of(n);
        c.gper = (g->n_g + gs - 1) / gs;
        const dim3 grid(blocks_of(n), gs), block(kCgThreads);
        auto go = [&](auto ptag) {
            constexpr int NPAIR = decltype(ptag)::value;
            if (form == CG_RYTOVA) hipLaunchKernelGGL((k_cgen_w<NPAIR, CG_RYTOVA>), grid, block, 0, 0, c, q0, n, dSum);
            else if (form == CG_PLAIN) hipLaunchKernelGGL((k_cgen_w<NPAIR, CG_PLAIN>), grid, block, 0, 0, c, q0, n, dSum);
            else hipLaunchKernelGGL((k_cgen_w<NPAIR, CG_GENERAL>), grid, block, 0, 0, c, q0, n, dSum);
        };
        if (npair == 0) go(std::integral_constant<int, 0>{});
        else if (npair == 1) go(std::integral_constant<int, 1>{});
        else if (npair == 3) go(std::integral_constant<int, 3>{});
        else go(std::integral_constant<int, 6>{});
        hipLaunchKernelGGL(k_cgen_finish, dim3((n + 255) / 256), dim3(256), 0, 0, c, q0, n, gs, ntot, mirror ? 1 : 0, (const double *)dSum, W);
    };
    // W on the Simpson grid, in chunks with a progress line each
    for (long long q0 = 0; q0 < half; q0 += chunk) {
        const int n = (int)std::min<long long>(chunk, half - q0);
        lattice_sum(a, q0, n, (long long)nq, gsym, dW);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) return fail(EDUS_ERR_HIP, "k_cgen_w");
        if (g->verbose) std::fprintf(stderr, "Coulomb coefficients: %lld / %lld q points\n", q0 + n, half);
    }
    {
        const int J = N * nw;
        hipLaunchKernelGGL(k_cgen_pass1, dim3((J + 15) / 16, ldt / (16 * kCgTT)), dim3(256), 0, 0, (const double *)dW, (const double *)dWt, N,
                           ldt, ntrig, J, dT);
        hipLaunchKernelGGL(k_cgen_pass2, dim3((ntrig * ntrig + 3) / 4), dim3(256), 0, 0, (const double *)dT, (const double *)dTr, N, ntrig, nw, dS);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) return fail(EDUS_ERR_HIP, "k_cgen_pass");
    }
    std::vector<double> S((size_t)ntrig * ntrig * nw);
    if (hipMemcpy(S.data(), dS, S.size() * 8, hipMemcpyDeviceToHost) != hipSuccess) return fail(EDUS_ERR_HIP, "download S");
    auto sv = [&](int t1, int t2, int c) { return S[((size_t)t1 * ntrig + t2) * nw + c]; };
    for (size_t i = 0; i < (size_t)nmm * nb2 * 2; i++) Ao[i] = Bo[i] = Co[i] = Do[i] = 0.0;
    for (int mm = 0; mm < nmm; mm++) {
        const int m = mm / nc, n = mm % nc;
        const double sc = 4.0 * ((m == 0 && n == 0) ? 0.25 : ((m == 0 || n == 0) ? 0.5 : 1.0));
        Ao[(size_t)mm * nb2 * 2] = sc * sv(m, n, 0);
        Do[(size_t)mm * nb2 * 2] = sc * sv(nc + m, nc + n, 0);
        for (int p = 0; p < npair; p++) {
            const size_t o = ((size_t)mm * nb2 + pic[p] * nb + pjc[p]) * 2;
            Ao[o] = sc * sv(m, n, 1 + 2 * p);
            Bo[o + 1] = sc * sv(m, nc + n, 2 + 2 * p);
            Co[o + 1] = sc * sv(nc + m, n, 2 + 2 * p);
            Do[o] = sc * sv(nc + m, nc + n, 1 + 2 * p);
        }
    }
    // correction around q = 0: points of the n_peak grid with 1e-17 < |q|^2 < q_peak^2
    for (int i = 0; i < nb2 * 2; i++) screen[i] = 0.0;
    const double hp = 2 * 0.5 / (Np - 1);
    std::vector<int> ql;
    {
        const double g11 = g->b1[0] * g->b1[0] + g->b1[1] * g->b1[1] + g->b1[2] * g->b1[2];
        const double g22 = g->b2[0] * g->b2[0] + g->b2[1] * g->b2[1] + g->b2[2] * g->b2[2];
        const double g12 = g->b1[0] * g->b2[0] + g->b1[1] * g->b2[1] + g->b1[2] * g->b2[2];
        const double lmin = 0.5 * (g11 + g22) - std::sqrt(0.25 * (g11 - g22) * (g11 - g22) + g12 * g12);
        const double rc = (lmin > 0) ? g->q_peak / std::sqrt(lmin) : 1.0;
        const int lo = std::max(0, (int)std::floor((0.5 - rc) / hp) - 2), hi = std::min(Np - 1, (int)std::ceil((0.5 + rc) / hp) + 2);
        const double qp2 = g->q_peak * g->q_peak, qmin2 = std::pow(10, -17);
        for (int ix = lo; ix <= hi; ix++)
            for (int iy = lo; iy <= hi; iy++) {
                const double qx = -0.5 + ix * hp, qy = -0.5 + iy * hp;
                double cart[3];
                for (int x = 0; x < 3; x++) cart[x] = g->b1[x] * qx + g->b2[x] * qy;
                const double q2 = cart[0] * cart[0] + cart[1] * cart[1] + cart[2] * cart[2];
                if (q2 < qp2 && q2 > qmin2) {
                    ql.push_back(ix);
                    ql.push_back(iy);
                }
            }
    }
    const int npk = (int)(ql.size() / 2);
    if (npk > 0) {
        const int nblk = (npk + kCgPeakThreads - 1) / kCgPeakThreads;
        std::vector<double> coef((size_t)4 * nmm * nb2 * 2);
        std::copy(Ao, Ao + (size_t)nmm * nb2 * 2, coef.begin());
        std::copy(Bo, Bo + (size_t)nmm * nb2 * 2, coef.begin() + (size_t)nmm * nb2 * 2);
        std::copy(Co, Co + (size_t)nmm * nb2 * 2, coef.begin() + (size_t)2 * nmm * nb2 * 2);
        std::copy(Do, Do + (size_t)nmm * nb2 * 2, coef.begin() + (size_t)3 * nmm * nb2 * 2);
        // the list runs through a disc around 0 in grid order: reversed, it is its mirror image
        bool qsym = gsym;
        for (int t = 0; t < npk && qsym; t++)
            qsym = ql[2 * t] + ql[2 * (npk - 1 - t)] == Np - 1 && ql[2 * t + 1] + ql[2 * (npk - 1 - t) + 1] == Np - 1;
        const long long phalf = qsym ? (npk + 1) / 2 : npk;
        (void)hipFree(dSum);
        dSum = nullptr;
        if (hipMalloc(&dQl, ql.size() * sizeof(int)) != hipSuccess || hipMalloc(&dW0, (size_t)npk * nw * 8) != hipSuccess ||
            hipMalloc(&dSum, sums_of(phalf)) != hipSuccess || hipMalloc(&dPart, (size_t)nblk * nb2 * 2 * 8) != hipSuccess)
            return fail(EDUS_ERR_NOMEM, "peak buffers");
        if (hipMemcpy(dQl, ql.data(), ql.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(dCoef, coef.data(), coef.size() * 8, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemset(dPart, 0, (size_t)nblk * nb2 * 2 * 8) != hipSuccess)
            return fail(EDUS_ERR_HIP, "peak upload");
        CGenArgs b = a;
        b.mode = 1; b.N = Np; b.qtf2 = 0.0; b.qlist = dQl;
        for (long long q0 = 0; q0 < phalf; q0 += chunk)
            lattice_sum(b, q0, (int)std::min(chunk, phalf - q0), npk, qsym, dW0);
        const size_t cs = (size_t)nmm * nb2 * 2;
        auto peak = [&](auto tag) {
            constexpr int NB = decltype(tag)::value;
            hipLaunchKernelGGL(k_cgen_peak<NB>, dim3(nblk), dim3(kCgPeakThreads), 0, 0, (const double *)dW0, (const int *)dQl, npk, nc, Np,
                               1. / ((double)Np * Np), (const double *)dCoef, (const double *)(dCoef + cs), (const double *)(dCoef + 2 * cs),
                               (const double *)(dCoef + 3 * cs), dPart);
        };
        if (nb == 1) peak(std::integral_constant<int, 1>{});
        else if (nb == 2) peak(std::integral_constant<int, 2>{});
        else if (nb == 3) peak(std::integral_constant<int, 3>{});
        else peak(std::integral_constant<int, 4>{});
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) return fail(EDUS_ERR_HIP, "peak kernels");
        std::vector<double> part((size_t)nblk * nb2 * 2);
        if (hipMemcpy(part.data(), dPart, part.size() * 8, hipMemcpyDeviceToHost) != hipSuccess) return fail(EDUS_ERR_HIP, "download peak");
        for (int b2i = 0; b2i < nblk; b2i++)
            for (int i = 0; i < nb2 * 2; i++) screen[i] += part[(size_t)b2i * nb2 * 2 + i];
        if (g->verbose) std::fprintf(stderr, "Coulomb coefficients: %d points in the q ~ 0 correction\n", npk);
    }
    cleanup();
    g_err.clear();
    return 0;
}

// Twiddles e^{2 pi i m / N_l} of the three grid directions, evaluated on the
// host in long double, and the offset of each direction's run.
static void wannier_twiddles(const int32_t nk3[3], std::vector<double> &tw, int offs[3]) {
    tw.clear();
    for (int l = 0; l < 3; l++) {
        offs[l] = (int)(tw.size() / 2);
        for (int m = 0; m < nk3[l]; m++) {
            long double ang = 2.0L * 3.14159265358979323846264338327950288L * (long double)m / (long double)nk3[l];
            tw.push_back((double)cosl(ang));
            tw.push_back((double)sinl(ang));
        }
    }
}

// One chunk of kc k (from kbase) of the FP64 contraction, the first nm of Val's ncol columns.
static void wannier_launch(const cd *PT, const cd *Val, const int2 *Col, const int32_t nk3[3], int nR, int nw2, int nm, int ncol, int kc,
                           int kbase, cd *H, cd *D) {
    hipLaunchKernelGGL(k_wannier_mfma, dim3((unsigned)((nm + 63) / 64), (unsigned)((kc + WMK - 1) / WMK)), dim3(256), 0, 0, PT, Val, Col,
                       nk3[0], nk3[1], nk3[2], nR, nw2, nm, ncol, kc, kbase, H, D);
}

// form: 0 FP64 matrix cores, 1 FP32, 2 BF16x3 split products.
static int wannier_hk(const int32_t nk3[3], int32_t nR, int32_t nw, const int32_t *R, const double *HR, const double *rR, double *H_out,
                     double *D_out, int form) {
    if (!nk3 || !R || !HR || !rR || !H_out || nR < 1 || nw < 1) return set_err(EDUS_ERR_INVALID, "bad Wannier arguments");
    for (int l = 0; l < 3; l++)
        if (nk3[l] < 1) return set_err(EDUS_ERR_INVALID, "bad grid");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(EDUS_ERR_NODEVICE, "no HIP device visible");
    const long long nk = (long long)nk3[0] * nk3[1] * nk3[2];
    const int nw2 = nw * nw, nm = D_out ? (int)wannier_cols(nw) : nw2, ncol = form ? 4 * nw2 : (int)wannier_cols(nw);
    std::vector<double> tw;
    int offs[3];
    wannier_twiddles(nk3, tw, offs);
    int *dR = nullptr;
    int2 *dCol = nullptr;
    double *dHR = nullptr, *drR = nullptr, *dVal = nullptr, *dTw = nullptr, *dPT = nullptr, *dH = nullptr, *dD = nullptr, *dOut = nullptr;
    auto cleanup = [&]() {
        for (void *q : {(void *)dOut, (void *)dR, (void *)dCol, (void *)dHR, (void *)drR, (void *)dVal, (void *)dTw, (void *)dPT, (void *)dH, (void *)dD})
            (void)hipFree(q);
    };
    Downloader down(Downloader::for_call((size_t)nk * nw2 * (D_out ? 64 : 16)));
    const size_t npt = (size_t)nR * (nk3[0] + nk3[1] + nk3[2]), nval = (size_t)nR * nw2;
    const size_t chunk = std::min<long long>(nk, std::max<long long>(64, (1LL << 28) / ((long long)nw2 * 64)));
    if (hipMalloc(&dR, (size_t)nR * 3 * sizeof(int)) != hipSuccess || hipMalloc(&dCol, (size_t)ncol * sizeof(int2)) != hipSuccess ||
        hipMalloc(&dHR, nval * 16) != hipSuccess || hipMalloc(&drR, nval * 48) != hipSuccess ||
        hipMalloc(&dVal, (size_t)nR * ncol * 16) != hipSuccess || hipMalloc(&dTw, tw.size() * sizeof(double)) != hipSuccess ||
        hipMalloc(&dPT, npt * 2 * sizeof(double)) != hipSuccess || hipMalloc(&dH, chunk * nw2 * 2 * sizeof(double)) != hipSuccess ||
        (form && hipMalloc(&dOut, chunk * ncol * 16) != hipSuccess) ||
        (D_out && hipMalloc(&dD, chunk * nw2 * 6 * sizeof(double)) != hipSuccess)) {
        cleanup();
        return set_err(EDUS_ERR_NOMEM, "Wannier buffers");
    }
    if (hipMemcpy(dR, R, (size_t)nR * 3 * sizeof(int), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dHR, HR, nval * 16, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(drR, rR, nval * 48, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dTw, tw.data(), tw.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        cleanup();
        return set_err(EDUS_ERR_HIP, "Wannier upload");
    }
    const dim3 gval((unsigned)((nval + 255) / 256));
    if (form) hipLaunchKernelGGL(k_wannier_val<true>, gval, dim3(256), 0, 0, (const cd *)dHR, (const cd *)drR, 0, nR, nw, ncol, (cd *)dVal, dCol);
    else hipLaunchKernelGGL(k_wannier_val<false>, gval, dim3(256), 0, 0, (const cd *)dHR, (const cd *)drR, 0, nR, nw, ncol, (cd *)dVal, dCol);
    hipLaunchKernelGGL(k_wannier_ptab, dim3((unsigned)std::min<size_t>((npt + 255) / 256, 65536)), dim3(256), 0, 0, (const int *)dR,
                       (const cd *)dTw, nR, nk3[0], nk3[1], nk3[2], offs[1], offs[2], (cd *)dPT);
    for (long long k0 = 0; k0 < nk; k0 += chunk) {
        const int kc = (int)std::min<long long>(chunk, nk - k0);
        const size_t nt = (size_t)kc * nw2;
        if (form == 0) {
            wannier_launch((const cd *)dPT, (const cd *)dVal, dCol, nk3, nR, nw2, nm, ncol, kc, (int)k0, (cd *)dH, (cd *)dD);
        } else {
            const dim3 grid((ncol + WMN - 1) / WMN, (unsigned)((kc + WMK - 1) / WMK));
            hipLaunchKernelGGL(form == 1 ? k_wannier_mfma32 : k_wannier_mfma_bf16x3, grid, dim3(256), 0, 0, (const cd *)dPT, (const cd *)dVal,
                               nk3[0], nk3[1], nk3[2], nR, ncol, kc, (int)k0, (cd *)dOut);
            hipLaunchKernelGGL(k_wannier_finish, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, 0, (const cd *)dOut, kc, nw, dH, dD);
        }
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = down.copy(H_out + (size_t)k0 * nw2 * 2, dH, nt * 16, 0);
        if (e == hipSuccess && D_out) e = down.copy(D_out + (size_t)k0 * nw2 * 6, dD, nt * 48, 0);
        if (e != hipSuccess) {
            cleanup();
            return set_err(EDUS_ERR_HIP, std::string("k_wannier: ") + hipGetErrorString(e));
        }
    }
    cleanup();
    g_err.clear();
    return 0;
}

int edus_wannier_hk(const int32_t nk3[3], int32_t nR, int32_t nw, const int32_t *R, const double *HR, const double *rR, double *H_out,
                    double *D_out) {
    return wannier_hk(nk3, nR, nw, R, HR, rR, H_out, D_out, 0);
}

int edus_wannier_hk_fp32(const int32_t nk3[3], int32_t nR, int32_t nw, const int32_t *R, const double *HR, const double *rR,
                         double *H_out, double *D_out) {
    return wannier_hk(nk3, nR, nw, R, HR, rR, H_out, D_out, 1);
}

int edus_wannier_hk_bf16x3(const int32_t nk3[3], int32_t nR, int32_t nw, const int32_t *R, const double *HR, const double *rR,
                           double *H_out, double *D_out) {
    return wannier_hk(nk3, nR, nw, R, HR, rR, H_out, D_out, 2);
}

// The contraction of edus_wannier_hk with every device buffer carved from the
// fixed scratch array: lattice vectors, twiddles, phase tables, H(R) and r(R)
// (packed on the device from copies passed through the output area), then the grid
// in as many k chunks as the rest of the array holds.  Nothing in the array needs
// clearing: every buffer is written before it is read.
int edus_wannier_hk_noalloc(const int32_t nk3[3], int32_t nR, int32_t nw, const int32_t *R, const double *HR, const double *rR,
                            double *H_out, double *D_out) {
    if (!nk3 || !R || !HR || !rR || !H_out || nR < 1 || nw < 1) return set_err(EDUS_ERR_INVALID, "bad Wannier arguments");
    for (int l = 0; l < 3; l++)
        if (nk3[l] < 1) return set_err(EDUS_ERR_INVALID, "bad grid");
    const long long nk = (long long)nk3[0] * nk3[1] * nk3[2];
    const long long nw2 = (long long)nw * nw, nm = 4 * nw2, nsum = (long long)nk3[0] + nk3[1] + nk3[2];
    auto al = [](long long b) { return (b + 255) / 256 * 256; };
    const long long oR = 0, oTw = al(oR + 12LL * nR), oPT = al(oTw + 16 * nsum), oVal = al(oPT + 16LL * nR * nsum),
                    oOut = al(oVal + 16LL * nR * nm);
    const long long per_k = 16 * nm + 16 * nw2 + (D_out ? 48 * nw2 : 0), slack = 512;
    const long long cap = EDUS_NOALLOC_SCRATCH_BYTES;
    if (oOut + per_k + slack > cap)
        return set_err(EDUS_ERR_UNSUPPORTED, "edus_wannier_hk_noalloc: the model needs " + std::to_string(oOut + per_k + slack) +
                                                 " bytes of scratch, above the " + std::to_string(cap) +
                                                 " of EDUS_NOALLOC_SCRATCH_BYTES (use edus_wannier_hk)");
    const long long chunk = std::min<long long>(nk, (cap - oOut - slack) / per_k);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_err(EDUS_ERR_NODEVICE, "no HIP device visible");
    void *base = nullptr;
    int rc = noalloc_scratch(&base);
    if (rc) return rc;
    char *b = static_cast<char *>(base);
    int *dR = reinterpret_cast<int *>(b + oR);
    double *dTw = reinterpret_cast<double *>(b + oTw), *dPT = reinterpret_cast<double *>(b + oPT);
    cd *dVal = reinterpret_cast<cd *>(b + oVal);
    const int ncol = (int)wannier_cols(nw), nform = D_out ? ncol : (int)nw2;
    // behind Val (smaller than the 4 nw^2 columns that the limit counts): the column
    // table, then the output chunk, which H(R) and r(R) pass through first
    const long long oCol = al(oVal + 16LL * nR * ncol), oH = al(oCol + 8LL * ncol), oD = al(oH + 16 * chunk * nw2);
    int2 *dCol = reinterpret_cast<int2 *>(b + oCol);
    cd *dH = reinterpret_cast<cd *>(b + oH), *dD = D_out ? reinterpret_cast<cd *>(b + oD) : nullptr;
    std::vector<double> tw;
    int offs[3];
    wannier_twiddles(nk3, tw, offs);
    HIP_TRY(hipMemcpy(dR, R, (size_t)nR * 3 * sizeof(int), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(dTw, tw.data(), tw.size() * sizeof(double), hipMemcpyHostToDevice));
    const int rchunk = (int)std::max<long long>(1, std::min<long long>(nR, (cap - oH - slack) / (64 * nw2)));
    for (int r0 = 0; r0 < nR; r0 += rchunk) {
        const int n = std::min(rchunk, nR - r0);
        cd *dHR = dH, *drR = dHR + (size_t)n * nw2;
        HIP_TRY(hipMemcpy(dHR, HR + (size_t)r0 * nw2 * 2, (size_t)n * nw2 * 16, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(drR, rR + (size_t)r0 * nw2 * 6, (size_t)n * nw2 * 48, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_wannier_val<false>, dim3((unsigned)(((long long)n * nw2 + 255) / 256)), dim3(256), 0, 0, (const cd *)dHR, (const cd *)drR,
                           r0, n, (int)nw, ncol, dVal, dCol);
        HIP_TRY(hipGetLastError());
    }
    const size_t npt = (size_t)nR * nsum;
    hipLaunchKernelGGL(k_wannier_ptab, dim3((unsigned)std::min<size_t>((npt + 255) / 256, 65536)), dim3(256), 0, 0, (const int *)dR,
                       (const cd *)dTw, nR, nk3[0], nk3[1], nk3[2], offs[1], offs[2], (cd *)dPT);
    HIP_TRY(hipGetLastError());
    for (long long k0 = 0; k0 < nk; k0 += chunk) {
        const int kc = (int)std::min<long long>(chunk, nk - k0);
        wannier_launch((const cd *)dPT, dVal, dCol, nk3, nR, (int)nw2, nform, ncol, kc, (int)k0, dH, dD);
        const long long nt = (long long)kc * nw2;
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipMemcpy(H_out + (size_t)k0 * nw2 * 2, dH, (size_t)nt * 16, hipMemcpyDeviceToHost));
        if (D_out) HIP_TRY(hipMemcpy(D_out + (size_t)k0 * nw2 * 6, dD, (size_t)nt * 48, hipMemcpyDeviceToHost));
    }
    g_err.clear();
    return 0;
}

}  // extern "C"
