// activation.hip — element-wise add / mul / SiLU / SwiGLU / GELU (tanh and erf
// forms) and the last-dimension bias add, for gfx950.
//
// Reference math (crates/sapient-backends/cpu/src/kernels/elementwise.rs):
//   add  a + b                        (:61-63, broadcast rule of binary_f32 :27-57)
//   mul  a * b                        (:67-69)
//   silu v / (1 + exp(-v))            (:141-143)
//   swiglu = silu(gate) * up          (llama.rs:531-532; wgpu analog elementwise.wgsl op1)
//   gelu 0.5 v (1 + tanh(0.79788456 (v + 0.044715 v v v)))   (:120-127)
//   gelu_erf 0.5 v (1 + erf_approx(v / √2))                  (:135-138, :163-174)
//   add_bias y[i] + bias[i % n]        (crates/sapient-models/src/forward/common.rs:556-569)
//
// Design: all streams are HBM-bound. Each thread moves 16-byte runs, one or two
// in flight per operand, at any element alignment; large launches pass the
// caches by (every byte is touched once), smaller ones use them (Policy). The
// grid is sized so each thread makes about one trip (up to 64K blocks) —
// measured on MI355X, a near-flat grid streams faster than a grid-stride loop
// over few blocks (SwiGLU f16: 125 → 114 µs).
//  - SiLU / SwiGLU return the reference's bits. f32 evaluates the reference's
//    expression (glibc's expf restated, see glibc_expf.h, then the IEEE
//    division) on every element: ~45 VALU ops, within the budget of 8-12
//    bytes per element. Half types (4-6 bytes per element) would be
//    VALU-bound that way, so they evaluate a fast SiLU (hardware exp2 /
//    reciprocal, ≤ 5 ulp — measured over every f32 input it serves) and run
//    the exact expression only where that error could change the rounding to
//    the half type (silu_certified).
//  - GELU: the reference's 1 + tanh(z) cancels for z < -3, so its result there
//    is glibc's rounding of tanh; only glibc's own algorithm reproduces it (see
//    glibc_tanhf.h). For f16 / bf16 inputs the op is a function of 16 bits, so
//    GELU is tabulated once per device — every input with |v| < 16 evaluated
//    on the GPU with that algorithm; outside that band the result is exactly
//    v, -0 or NaN — and each launch stages the 76 KiB table in LDS (two
//    resident blocks per CU in gfx950's 160 KiB) and streams the tensor through it:
//    bit-exact and bandwidth-bound. f32 inputs evaluate the algorithm per
//    element (VALU-bound).
//  - erf-GELU takes the same two routes: its erf_approx multiplies by glibc's
//    expf(-x²), restated in glibc_expf.h (double-precision evaluation with a
//    32-entry table of 2^(i/32), which each block stages in LDS). Outside
//    |v| < 16 expf(-x²) underflows to 0, so the band and the outside rule are
//    the ones of the tanh form.
//  - Bias add: a block owns a tile of up to 256 16-byte column runs over
//    two rows; each thread loads its bias vector once and adds it to both.
//    Narrow or small rows that no aligned vector fits go element by element.
#include <mutex>
#include <type_traits>

#include "glibc_expf.h"
#include "glibc_tanhf.h"
#include "sph_common.h"

namespace sph {
namespace {

constexpr int kThreads = 256;
constexpr int kUnroll = 2;       // vectors in flight per operand per thread
constexpr int64_t kMaxGrid = 65536;  // ~one loop trip per thread at the configuration sizes
// Launches of up to 2^20 16-byte vectors take one run per thread (a single trip, each thread's
// chain as short as it can be). Per launch, back to back on MI355X, against two vectors per thread:
// SwiGLU 64 x 14336 f32 3.99 -> 3.03 µs, f16 5.42 -> 3.53; 512 x 4864 f32 7.10 -> 6.46, f16 7.08 ->
// 5.16; 512 x 14336 f16 11.7 -> 11.2; GELU-tanh f32 512 x 4864 6.88 -> 6.60, but at 512 x 14336 f32
// (1.8 M vectors) 14.2 -> 16.1, and at larger launches both shapes run alike.
constexpr int64_t kFewVecs = int64_t(1) << 20;

// Smaller launches (decode steps, prefill chunks of small models) take one element per thread for
// the ops whose per-element work is long: a thread's chain is then one element's, and all CUs have
// work. Half-precision SiLU and SwiGLU up to 2^19 elements, then runs of eight: bf16 SwiGLU of 0.3 M
// elements 2.45 / 3.38 µs with one / eight, 3 M 6.88 / 5.73 (runs of four, 2.76, 3.41 / 3.72 at 1 M and
// 6.01, lose where the result is read next: f16 SwiGLU and an add 1 M 6.1 / 5.4, 2 M 8.3 / 6.8). GELU
// in f32 up to 2^18 (alone 0.3 M 2.41 µs against 3.07 with four and 1 M level, but between the bias that
// wrote its input and an add, the three 0.4 M 7.9 / 7.1 µs, 1 M 12.0 / 9.0, 2 M 19.7 / 13.9). f32 SiLU
// and SwiGLU from 2048 elements up to 2^18 (0.3 M 2.35 / 2.5, 1 M 3.70 / 3.39; below 2048 level or 0.3 %
// slower); adds and products never gain. Half-precision GELU reads its table from cache up to kFewElems
// instead of staging it per block (1 x 10240 f16 2.90 -> 1.79 µs). Results are the same bits either way.
constexpr int64_t kFewElems = int64_t(1) << 18;
constexpr int64_t kFewF32LightMin = 2048;

enum Op { OP_ADD = 0, OP_MUL = 1, OP_SILU = 2, OP_SWIGLU = 3, OP_GELU = 4, OP_GELU_ERF = 5 };

// 2^(i/32) for the expf restatement, staged per block into LDS by the kernels that need it.
__constant__ Exp2fTable kExp2f = exp2f_table();
enum Bcast { B_NONE = 0, B_SCALAR_B = 1, B_SCALAR_A = 2 };

// Fast SiLU for g >= -80: exp(-g) from the hardware exp2 on a split-precision
// argument, 1 / (1 + e) from the hardware reciprocal, ~12 VALU ops. From 64 on,
// exp(-g) < 2^-92, so 1 + e and its reciprocal are 1 and the result is g itself,
// as the reference's; the exponent is clamped there so that no product overflows.
__device__ __forceinline__ float silu_f(float g) {
    const float kL2eHi = 1.44269502162933349609375f;  // f32(log2 e)
    const float kL2eLo = 1.925963033500011e-08f;      // log2 e - kL2eHi
    const float kLn2 = 0.693147180559945309f;
    const float ng = -fminf(g, 64.0f);
    const float p = ng * kL2eHi;
    const float perr = __builtin_fmaf(ng, kL2eHi, -p) + ng * kL2eLo;  // -g·log2e - p
    const float e0 = __builtin_amdgcn_exp2f(p);
    const float e = __builtin_fmaf(e0, perr * kLn2, e0);            // 2^(p + perr)
    return g * __builtin_amdgcn_rcpf(1.0f + e);
}

// True when every f32 within 16 ulp of p rounds to the same T: p is far enough
// from the midpoint between two T values (a window around a midpoint never
// reaches a binade edge, so bit units are ulps). f16: the 13 bits below its
// mantissa, for |p| in [2^-14, 2^16) (normal f16 results and their overflow to
// inf); bf16: the 16 bits below its mantissa, anywhere in the finite range
// from 2^-125 on. Unsigned wrap-around makes each test one comparison.
template <typename T>
__device__ __forceinline__ bool rounding_is_clear(float p) {
    constexpr bool kF16 = std::is_same<T, f16>::value;
    constexpr uint32_t kBelow = kF16 ? 0x1FFFu : 0xFFFFu, kLow = kF16 ? 113u : 2u, kHigh = kF16 ? 142u : 254u;
    const uint32_t b = __builtin_bit_cast(uint32_t, p);
    const bool range = (b & 0x7FFFFFFFu) - (kLow << 23) < ((kHigh - kLow + 1) << 23);
    const bool far = (b & kBelow) - ((kBelow + 1) / 2 - 16) > 32u;
    return range & far;
}

// SiLU (times u for SwiGLU) of N values, whose rounding to the half type T equals
// the reference's: the fast silu_f is certified where it decides the result. Over
// every f32 g in [-80, 64] silu_f lies within 5 ulp of the exact
// silu_ref_order (measured on MI355X over all 2^31 such inputs). In ulps of
// the product that is < 10 ulp (ulp(s)·|u| < 2 ulp(s·u)), and the roundings
// RN(s·u), RN(s'·u) add one more, so the exact result lies within 11 ulp of the
// fast p. When every f32 within 16 ulp of p rounds to the same T value,
// rounding being monotonic, so does the exact result. Otherwise (about 0.4 %
// of elements), outside the measured domain, for non-finite values and for
// results outside the ranges rounding_is_clear covers, the exact expression
// runs inline: it touches only registers and the LDS copy of the 2^(i/32)
// table, so its rare divergent executions cost ~1 % (measured: fast-only
// 112 µs, certified 113 µs on f16 SwiGLU [8192, 14336]; a table load from
// global memory in the same branch stalls the wave on its stream traffic,
// 136 µs). The fast values and their tests are straight-line code, with one
// branch per value after them.
template <typename T, bool MUL, int N>
__device__ __forceinline__ void silu_certified(const float (&g)[N], const float (&u)[N], float (&o)[N],
                                               const uint64_t* exp_tab) {
    bool exact[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float s = silu_f(g[i]);
        o[i] = MUL ? s * u[i] : s;
        exact[i] = !((g[i] >= -80.0f) & rounding_is_clear<T>(o[i]));
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (exact[i]) {
            const float x = silu_ref_order(g[i], exp_tab);
            o[i] = MUL ? x * u[i] : x;
        }
    }
}

// T: the storage type. SiLU / SwiGLU give the reference's bits: f32 evaluates
// the reference's expression exactly (glibc's expf restated, IEEE division —
// within the bandwidth budget of 8-12 bytes per element); half types take the
// certified fast path (4-6 bytes per element leave no room for the exact
// expression on every element: f16 SwiGLU 149 µs instead of 113).
template <int OP, typename T>
__device__ __forceinline__ float apply_op(float a, float b, const uint64_t* exp_tab) {
    if constexpr (OP == OP_ADD) return a + b;
    if constexpr (OP == OP_MUL) return a * b;
    if constexpr (OP == OP_SILU) return silu_ref_order(a, exp_tab);
    if constexpr (OP == OP_SWIGLU) return silu_ref_order(a, exp_tab) * b;
    if constexpr (OP == OP_GELU) return gelu_tanh_ref_order(a);
    if constexpr (OP == OP_GELU_ERF) return gelu_erf_ref_order(a, exp_tab);
    return 0.0f;
}

template <int OP, typename T, int N>
__device__ __forceinline__ void apply_ops(const float (&a)[N], const float (&b)[N], float (&o)[N], const uint64_t* exp_tab) {
    if constexpr (sizeof(T) == 2 && (OP == OP_SILU || OP == OP_SWIGLU)) {
        silu_certified<T, OP == OP_SWIGLU>(a, b, o, exp_tab);
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) o[e] = apply_op<OP, T>(a[e], b[e], exp_tab);
    }
}

template <int OP, typename T> constexpr bool needs_exp_table() {
    return OP == OP_GELU_ERF || OP == OP_SILU || OP == OP_SWIGLU;
}

// Copy the 2^(i/32) table into LDS (block-wide; call before any use).
__device__ __forceinline__ void stage_exp_table(uint64_t* tab) {
    if (threadIdx.x < 32) tab[threadIdx.x] = kExp2f.tab[threadIdx.x];
    __syncthreads();
}

template <int OP> constexpr bool binary_op() { return OP == OP_ADD || OP == OP_MUL || OP == OP_SWIGLU; }

// How a launch's stream meets the caches, by the bytes it moves. Loads are cached below
// kCachedBytes (operands are mostly still in the 256 MB Infinity Cache from the kernel before);
// stores pass the caches by from 16 MB on, so that a launch does not end on writing back what it
// left dirty in the L2s. Per launch on MI355X, cached / non-temporal stores / both non-temporal:
// SwiGLU f32 512 x 4864 (30 MB) 7.1 / 6.5 / 6.9 µs, GELU-tanh f32 777 x 10240 (64 MB) 15.7 / 14.5 /
// 15.3, SwiGLU f16 8192 x 14336 (705 MB) 125 / 121 / 111.
enum Policy { P_CACHED = 0, P_NT_STORES = 1, P_NT = 2 };
inline int policy_for(int64_t bytes) {
    return bytes >= kCachedBytes ? P_NT : bytes >= (int64_t(1) << 24) ? P_NT_STORES : P_CACHED;
}

// `n` elements in runs of E (16 bytes of T), U runs in flight per thread, at any element
// alignment; the thread whose run crosses the end takes its elements in pieces, so odd sizes
// and odd addresses are one launch too (512 x 4864 + 3 f32 8.4 -> 6.4 µs, 3000 x 5001 f16 at an odd
// address, element by element before, 28.5 -> 18.0). B_SCALAR_B / B_SCALAR_A read element 0 of the
// broadcast operand. `out` may alias a full-length input: each element is read before it is
// written, by the same thread. U = 1: the grid covers all runs, fewer than 2^31. (Issuing the
// first loads before the exp table is staged costs 0.3 µs at 512 x 4864 f32 and 1.5 at bf16
// 333 x 14336.) TAIL: n is no multiple of E (the tail's code alone costs a small launch 0.2 µs).
template <typename T, int OP, int BC, int U, int POLICY, bool TAIL>
__global__ __launch_bounds__(kThreads) void ew_runs(const T* a, const T* b, T* out, int64_t n) {
    constexpr int E = vec16<T>::n;
    constexpr bool NTL = POLICY == P_NT, NTS = POLICY != P_CACHED;
    using Index = std::conditional_t<U == 1, int32_t, int64_t>;
    __shared__ uint64_t exp_tab[needs_exp_table<OP, T>() ? 32 : 1];
    if constexpr (needs_exp_table<OP, T>()) stage_exp_table(exp_tab);
    float sa = 0.0f, sb = 0.0f;
    if constexpr (BC == B_SCALAR_A) sa = widen(a[0]);
    if constexpr (BC == B_SCALAR_B) sb = widen(b[0]);
    const Index nrun = (Index)((n + E - 1) / E);
    // Elements of run i.
    auto left = [&](Index i) { return TAIL && i == nrun - 1 ? (int)(n - (int64_t)i * E) : E; };
    auto trip = [&](Index base) {
        float va[U][E], vb[U][E];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const Index i = base + u * kThreads;
            if (i < nrun) {
                if constexpr (BC != B_SCALAR_A) load_run_f32<T, E, NTL>(a + (int64_t)i * E, left(i), va[u]);
                if constexpr (binary_op<OP>() && BC != B_SCALAR_B)
                    load_run_f32<T, E, NTL>(b + (int64_t)i * E, left(i), vb[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const Index i = base + u * kThreads;
            if (i < nrun) {
                float o[E];
                if constexpr (BC != B_NONE) {
#pragma unroll
                    for (int e = 0; e < E; ++e) (BC == B_SCALAR_A ? va : vb)[u][e] = BC == B_SCALAR_A ? sa : sb;
                }
                apply_ops<OP, T, E>(va[u], vb[u], o, exp_tab);
                store_run_f32<T, E, NTS>(out + (int64_t)i * E, left(i), o);
            }
        }
    };
    const Index first = (Index)blockIdx.x * kThreads * U + (Index)threadIdx.x;
    if constexpr (U == 1) {
        trip(first);  // no loop: one that always breaks lets the compiler move the store out of it, less its nt bit
    } else {
        for (Index base = first; base < nrun; base += (Index)gridDim.x * kThreads * U) trip(base);
    }
}

// One element per thread: small launches (see kFewElems).
template <typename T, int OP, int BC>
__global__ __launch_bounds__(kThreads) void ew_scalar(const T* a, const T* b, T* out, int64_t n) {
    __shared__ uint64_t exp_tab[needs_exp_table<OP, T>() ? 32 : 1];
    if constexpr (needs_exp_table<OP, T>()) stage_exp_table(exp_tab);
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
        const float x[1] = {widen(a[BC == B_SCALAR_A ? 0 : i])};
        const float y[1] = {binary_op<OP>() ? widen(b[BC == B_SCALAR_B ? 0 : i]) : 0.0f};
        float o[1];
        apply_ops<OP, T, 1>(x, y, o, exp_tab);
        out[i] = narrow<T>(o[0]);
    }
}

inline unsigned grid_for(int64_t items, int64_t per_block, int64_t cap) {
    int64_t g = (items + per_block - 1) / per_block;
    if (g < 1) g = 1;
    return (unsigned)(g < cap ? g : cap);
}

template <typename T, int OP, int BC>
int launch_ew(const void* a, const void* b, void* out, int64_t n, hipStream_t stream) {
    if (n == 0) return SPH_OK;
    constexpr int E = vec16<T>::n;
    const T* ap = static_cast<const T*>(a);
    const T* bp = static_cast<const T*>(b);
    T* op = static_cast<T*>(out);
    constexpr bool kGelu = OP == OP_GELU || OP == OP_GELU_ERF;  // (half types: gelu_half)
    constexpr bool kHalfLong = sizeof(T) == 2 && (OP == OP_SILU || OP == OP_SWIGLU);
    constexpr bool kLong = kHalfLong || OP == OP_GELU;
    // (At addresses without 16-byte alignment runs pay off later: f32 GELU 0.5 M 3.3 µs in runs, 2.9 one by one, 1 M level;
    // f16 SwiGLU 0.8 M 3.8 / 3.4, 1.3 M 4.4 / 4.1, 1.6 M level.)
    const bool at16 = aligned(ap, 16) && aligned(op, 16) && (OP != OP_SWIGLU || aligned(bp, 16));
    const int64_t singles = kLong && !at16 ? kFewElems * 5 : kHalfLong ? kFewElems << 1 : kFewElems;
    if (n <= singles && (sizeof(T) == 2 || kGelu || n >= kFewF32LightMin))
        return launch(ew_scalar<T, OP, BC>, grid_for(n, kThreads, 8192), kThreads, stream, ap, bp, op, n);
    const int64_t streams = (BC != B_SCALAR_A) + (binary_op<OP>() && BC != B_SCALAR_B) + 1;
    const int policy = policy_for(n * (int64_t)sizeof(T) * streams);
    auto go = [&](auto u, auto p) {
        constexpr int U = decltype(u)::value;
        const unsigned grid = grid_for((n + E - 1) / E, (int64_t)kThreads * U, kMaxGrid);
        return n % E == 0 ? launch(ew_runs<T, OP, BC, U, decltype(p)::value, false>, grid, kThreads, stream, ap, bp, op, n)
                          : launch(ew_runs<T, OP, BC, U, decltype(p)::value, true>, grid, kThreads, stream, ap, bp, op, n);
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, kUnroll> two;
    const std::integral_constant<int, P_CACHED> cached;
    const std::integral_constant<int, P_NT_STORES> nt_stores;
    const std::integral_constant<int, P_NT> nt;
    // One run per thread: adds and products past 16 MB both ways non-temporal. They read what a kernel has just written,
    // and cached loads of that are slower: an add, then a product with a scalar, f32 3 M 12.1 against 9.1 µs, f16 8 M
    // 15.5 / 11.7; SwiGLU, then an add, f32 3 M 15.4 / 13.4. The activations keep cached loads: on inputs written longer
    // ago SwiGLU f32 512 x 4864 takes 6.8 µs against 7.6 non-temporal, bf16 333 x 14336 6.9 / 8.0.
    if ((n + E - 1) / E <= kFewVecs) {
        if (policy == P_CACHED) return go(one, cached);
        if constexpr (OP == OP_ADD || OP == OP_MUL) return go(one, nt);
        else return go(one, nt_stores);
    }
    return policy == P_NT ? go(two, nt) : go(two, nt_stores);
}

template <int OP>
int dispatch_unary(const void* x, void* out, int dt, int64_t n, hipStream_t stream) {
    if (n < 0) return SPH_EINVAL;
    if (n > 0 && (x == nullptr || out == nullptr)) return SPH_EINVAL;
    return with_float_type(dt, [&](auto t) -> int {
        using T = decltype(t);
        return launch_ew<T, OP, B_NONE>(x, nullptr, out, n, stream);
    });
}

template <int OP>
int dispatch_binary(const void* a, int64_t na, const void* b, int64_t nb, void* out, int dt, hipStream_t stream) {
    if (na < 0 || nb < 0) return SPH_EINVAL;
    if (a == nullptr || b == nullptr || out == nullptr) {
        if (na == 0 && nb == 0) return SPH_OK;
        return SPH_EINVAL;
    }
    return with_float_type(dt, [&](auto t) -> int {
        using T = decltype(t);
        if (na == nb) return launch_ew<T, OP, B_NONE>(a, b, out, na, stream);
        if (nb == 1) return launch_ew<T, OP, B_SCALAR_B>(a, b, out, na, stream);
        if (na == 1) return launch_ew<T, OP, B_SCALAR_A>(a, b, out, nb, stream);
        return SPH_EINVAL;  // the reference's ShapeMismatch
    });
}

// ─────────────────────────── GELU lookup tables ───────────────────────────
// For |v| >= 16 GELU is exact without a table: tanh(z) rounds to ±1, so the
// reference returns v itself for v >= 16 (and +inf), -0 for v <= -16, and
// NaN for -inf (-inf · 0) and NaN. The table therefore holds only |v| < 16:
// the 16-bit patterns below kLimit, for both signs — 76 KiB for f16 (68 KiB
// for bf16), which lets two 1024-thread blocks share a CU's 160 KiB of LDS.
template <typename T> struct gelu_band;
template <> struct gelu_band<f16> {   // 16.0 = 0x4C00; +inf 0x7C00; quiet-NaN bit 0x0200
    static constexpr uint32_t kLimit = 0x4C00u, kInf = 0x7C00u, kQuiet = 0x0200u;
};
template <> struct gelu_band<bf16> {  // 16.0 = 0x4180; +inf 0x7F80; quiet-NaN bit 0x0040
    static constexpr uint32_t kLimit = 0x4180u, kInf = 0x7F80u, kQuiet = 0x0040u;
};
constexpr uint32_t kLutEntries = 2 * gelu_band<f16>::kLimit;  // the larger of the two

// Table slot of a pattern inside the band: positives first, then negatives.
template <typename T>
__device__ __forceinline__ uint32_t gelu_slot(uint32_t h) {
    return (h & 0x8000u) ? gelu_band<T>::kLimit + (h & 0x7FFFu) : h;
}

// Result for a pattern outside the band (|v| >= 16, inf, NaN).
template <typename T>
__device__ __forceinline__ uint32_t gelu_outside(uint32_t h) {
    constexpr uint32_t inf = gelu_band<T>::kInf, quiet = gelu_band<T>::kQuiet;
    const bool neg = (h & 0x8000u) != 0;
    const uint32_t mag = h & 0x7FFFu;
    if (mag > inf) return h | quiet;                  // NaN stays NaN (quiet)
    if (!neg) return h;                               // v >= 16 and +inf: v
    if (mag == inf) return 0x8000u | inf | quiet;     // -inf: -inf * 0 = NaN
    return 0x8000u;                                   // v <= -16: -0
}

// Tables by index: form * 2 + type, form 0 = tanh, 1 = erf; type 0 = f16, 1 = bf16.
constexpr int kLutTables = 4;
__device__ __align__(16) uint16_t gelu_lut[kLutTables][kLutEntries];

template <typename T>
__global__ __launch_bounds__(kThreads) void gelu_lut_build(int which) {
    __shared__ uint64_t exp_tab[32];
    stage_exp_table(exp_tab);
    const uint32_t slot = blockIdx.x * kThreads + threadIdx.x;
    constexpr uint32_t L = gelu_band<T>::kLimit;
    if (slot >= 2 * L) return;
    const uint32_t h = slot < L ? slot : 0x8000u | (slot - L);
    const float v = widen(T{(uint16_t)h});
    const float g = which < 2 ? gelu_tanh_ref_order(v) : gelu_erf_ref_order(v, exp_tab);
    gelu_lut[which][slot] = narrow<T>(g).bits;
}

constexpr int kLutOneThreads = 1024, kLutTwoThreads = 512;  // one and two blocks per CU

template <typename T>
__device__ __forceinline__ uint32_t gelu_lookup(const uint16_t* tab, uint32_t h) {
    return (h & 0x7FFFu) < gelu_band<T>::kLimit ? (uint32_t)tab[gelu_slot<T>(h)] : gelu_outside<T>(h);
}

// Blocks of THREADS that each stage the band table in LDS once and then stream
// 16-byte runs, grid-stride, U per thread per trip, at any element alignment (the
// thread whose run crosses the end takes its elements in pieces), past the
// caches at every size: erf-GELU f16 after the bias that wrote its input, 1500 x
// 5120, 7.5 µs against 8.8 with cached loads and 3000 x 5120 14.2 against 17.2.
//  - Up to one trip of 1024 threads x 4 runs on every CU (8 M elements): one block
//    per CU, so the table is staged once, the fewest U that make it one trip, and
//    all of a thread's loads in flight beside the table's (AHEAD). In the same
//    sequence 400 x 5120 4.19 -> 3.72 µs, 800 x 5120 5.51 -> 4.85, 1500 x 5120 9.13 ->
//    7.54 (8.3 with the loads after the table, 9.1 with two blocks of 512).
//  - Larger: two 512-thread blocks per CU, both resident (LDS-bound), U = 2. At
//    [8192, 10240] f16, round-robin with a 16-byte copy of the same bytes (53.9 µs
//    in this loop shape, 53.1 as a flat grid): U = 2 56.8 µs, U = 3 58.6, U = 4 59.4,
//    U = 1 62.8; four blocks per CU (the table staged twice per slot) 59.4 at U = 2;
//    the first trip's loads issued before the table is staged: no change;
//    1024-thread blocks 58.5, the next trip's loads issued ahead 63-65.
template <typename T, int THREADS, int U, bool AHEAD>
__global__ __launch_bounds__(THREADS) void gelu_lut_apply(const T* in, T* out, int64_t n, int which) {
    constexpr int E = vec16<T>::n;
    __shared__ __align__(16) uint16_t tab[kLutEntries];
    const int64_t nrun = (n + E - 1) / E;
    const int64_t stride = (int64_t)gridDim.x * THREADS * U;
    const int64_t first = (int64_t)blockIdx.x * THREADS * U + threadIdx.x;
    // Elements of run i.
    auto left = [&](int64_t i) { return i == nrun - 1 ? (int)(n - i * E) : E; };
    uint32_t q[U][4];
    auto load = [&](int64_t base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = base + (int64_t)u * THREADS;
            if (i < nrun) load_run<T, E, true>(in + i * E, left(i), q[u]);
        }
    };
    {
        // The table is copied into LDS with gfx950's direct-to-LDS 16-byte
        // loads (global_load_lds_dwordx4: lane l of a wave writes the 16 bytes
        // at the wave's LDS base + 16 l, no register round trip), all of a
        // thread's chunks requested before the wait: one L2 round trip per block
        // (a load-wait-store loop through registers serialised ten of them; the
        // register-staged form of the same loop measured 0.2-0.4 us slower).
        constexpr int nq = (int)(2 * gelu_band<T>::kLimit * 2 / 16);  // 16-byte chunks of this type's table
        constexpr int per = (nq + THREADS - 1) / THREADS;
        // A wave loads 64 chunks from its base, and only waves whose base is below nq load.
        static_assert((nq + 63) / 64 * 64 <= (int)(kLutEntries * 2 / 16), "a wave's chunks stay inside tab");
        const u32x4* src = reinterpret_cast<const u32x4*>(gelu_lut[which]);
        const int wv = (int)threadIdx.x / 64;
#pragma unroll
        for (int i = 0; i < per; ++i) {
            const int base = i * THREADS + wv * 64;  // this wave's first chunk (wave-uniform)
            if (base < nq) {
                // Lanes past the table's end reload its last chunk into tab's
                // spare slots (in bounds: see the static_assert).
                const int k = (int)threadIdx.x + i * THREADS;
                __builtin_amdgcn_global_load_lds(src + (k < nq ? k : nq - 1), reinterpret_cast<u32x4*>(tab) + base,
                                                 16, 0, 0);
            }
        }
        if constexpr (AHEAD) load(first);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    for (int64_t base = first; base < nrun; base += stride) {
        if (!AHEAD || base != first) load(base);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = base + (int64_t)u * THREADS;
            if (i < nrun) {
                uint32_t r[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint32_t w = q[u][c];
                    r[c] = gelu_lookup<T>(tab, w & 0xFFFFu) | (gelu_lookup<T>(tab, w >> 16) << 16);
                }
                store_run_words<T, E, true>(out + i * E, left(i), r);
            }
        }
    }
}

// One element per thread, the table read from cache (see kFewElems).
template <typename T>
__global__ __launch_bounds__(kThreads) void gelu_lut_apply_scalar(const T* in, T* out, int64_t n, int which) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
        out[i].bits = (uint16_t)gelu_lookup<T>(gelu_lut[which], in[i].bits);
}

constexpr int kMaxDevices = 64;
std::mutex g_init_mu;
bool g_lut_ready[kMaxDevices];
int g_num_cus[kMaxDevices];

// Build the four tables on `stream` once per device and wait for them.
int ensure_device_ready(hipStream_t stream, int* cus) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return SPH_ENODEV;
    std::lock_guard<std::mutex> lock(g_init_mu);
    if (!g_lut_ready[dev]) {
        // The build waits for its kernels: under stream capture they would be
        // recorded instead of run and the wait would invalidate the capture.
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &cap) != hipSuccess) return SPH_EHIP;
        if (cap != hipStreamCaptureStatusNone) return SPH_ESTATE;
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            return SPH_ENODEV;
        g_num_cus[dev] = n;
        const dim3 grid((kLutEntries + kThreads - 1) / kThreads);
        for (int form = 0; form < 2; ++form) {
            if (launch(gelu_lut_build<f16>, grid, kThreads, stream, form * 2) != SPH_OK) return SPH_EHIP;
            if (launch(gelu_lut_build<bf16>, grid, kThreads, stream, form * 2 + 1) != SPH_OK) return SPH_EHIP;
        }
        if (hipStreamSynchronize(stream) != hipSuccess) return SPH_EHIP;
        g_lut_ready[dev] = true;
    }
    if (cus) *cus = g_num_cus[dev];
    return SPH_OK;
}

template <typename T>
int gelu_half(const void* x, void* out, int which, int64_t n, hipStream_t stream) {
    int cus = 0;
    const int st = ensure_device_ready(stream, &cus);
    if (st != SPH_OK) return st;
    const T* xp = static_cast<const T*>(x);
    T* op = static_cast<T*>(out);
    // At addresses without 16-byte alignment runs pay off later: f16 (bf16) at an odd address 300 K halves 2.4 (2.4) µs
    // element by element against 3.9 (3.9) in runs, 1 M 3.7 (3.4) / 4.3 (4.3), 2 M 5.3 (4.9) / 5.4 (5.4), 2.5 M 5.9
    // (5.4) / 5.7 (5.7).
    if (n <= kFewElems || (n <= kFewElems * 9 && !(aligned(xp, 16) && aligned(op, 16))))
        return launch(gelu_lut_apply_scalar<T>, grid_for(n, kThreads, 4096), kThreads, stream, xp, op, n, which);
    const int64_t nrun = (n + vec16<T>::n - 1) / vec16<T>::n;
    const int64_t trip = (int64_t)cus * kLutOneThreads;  // runs of one trip, one per thread
    auto one = [&](auto u) {
        constexpr int U = decltype(u)::value;
        return launch(gelu_lut_apply<T, kLutOneThreads, U, true>, grid_for(nrun, (int64_t)kLutOneThreads * U, cus),
                      kLutOneThreads, stream, xp, op, n, which);
    };
    if (nrun <= trip) return one(std::integral_constant<int, 1>{});
    if (nrun <= 2 * trip) return one(std::integral_constant<int, 2>{});
    if (nrun <= 4 * trip) return one(std::integral_constant<int, 4>{});
    return launch(gelu_lut_apply<T, kLutTwoThreads, 2, false>, grid_for(nrun, kLutTwoThreads * 2, 2 * cus),
                  kLutTwoThreads, stream, xp, op, n, which);
}

// GELU of either form: half types through the tables, f32 per element.
template <int OP>
int gelu_any(const void* x, void* out, int dtype, int64_t n, hipStream_t s) {
    if (n < 0) return SPH_EINVAL;
    if (n > 0 && (x == nullptr || out == nullptr)) return SPH_EINVAL;
    if (n == 0) return is_float_dtype(dtype) ? SPH_OK : SPH_EINVAL;
    const int form = OP == OP_GELU ? 0 : 1;
    if (dtype == SPH_F16) return gelu_half<f16>(x, out, form * 2, n, s);
    if (dtype == SPH_BF16) return gelu_half<bf16>(x, out, form * 2 + 1, n, s);
    return dispatch_unary<OP>(x, out, dtype, n, s);
}

// ───────────────────────────── bias add ─────────────────────────────
// Two rows per block, both in flight: measured on MI355X at 16384 x 4096 f32
// this runs at the speed of a plain two-stream add (16 rows per block: -15 %).
constexpr int kBiasRowsPerBlock = 2;

// Block b covers column tile b % ntiles (up to 256 16-byte runs of a row) over rows
// [(b / ntiles) · R, + R). A thread keeps its bias run in registers and streams y down the rows,
// RU rows in flight; any width and element alignment (TAIL: the row's last run is short). POLICY:
// see Policy (f16 1500 x 5120, 31 MB: 8.0 µs non-temporal, 7.0 cached, 6.5 with cached loads only).
template <typename T, typename TB, int POLICY, bool TAIL>
__global__ __launch_bounds__(kThreads) void bias_rows(const T* y, const TB* bias, T* out, int64_t rows, int n, int nvr,
                                                     int ntiles, int tile) {
    constexpr int E = vec16<T>::n;
    constexpr int RU = 2;
    constexpr bool NTL = POLICY == P_NT, NTS = POLICY != P_CACHED;
    const int t = (int)(blockIdx.x % (unsigned)ntiles);
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)ntiles) * kBiasRowsPerBlock;
    const int v = t * tile + (int)threadIdx.x;
    if ((int)threadIdx.x >= tile || v >= nvr) return;
    const int left = TAIL && v == nvr - 1 ? n - v * E : E;
    float bv[E];
    load_run_f32<TB, E, false>(bias + (size_t)v * E, left, bv);
    const int64_t r_end = r0 + kBiasRowsPerBlock < rows ? r0 + kBiasRowsPerBlock : rows;
    for (int64_t r = r0; r < r_end; r += RU) {
        float q[RU][E];
#pragma unroll
        for (int u = 0; u < RU; ++u)
            if (r + u < r_end) load_run_f32<T, E, NTL>(y + (size_t)(r + u) * n + (size_t)v * E, left, q[u]);
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            if (r + u < r_end) {
#pragma unroll
                for (int e = 0; e < E; ++e) q[u][e] = q[u][e] + bv[e];
                store_run_f32<T, E, NTS>(out + (size_t)(r + u) * n + (size_t)v * E, left, q[u]);
            }
        }
    }
}

// Rows too wide or too many for that grid, and small or narrow ragged launches: element-wise, one modulo per element.
template <typename T, typename TB>
__global__ __launch_bounds__(kThreads) void bias_scalar(const T* y, const TB* bias, T* out, int64_t total, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total; i += stride)
        out[i] = narrow<T>(widen(y[i]) + widen(bias[i % n]));
}

template <typename T, typename TB>
int launch_bias(const void* y, const void* bias, void* out, int64_t total, int64_t n, hipStream_t stream) {
    constexpr int E = vec16<T>::n;
    const T* yp = static_cast<const T*>(y);
    const TB* bp = static_cast<const TB*>(bias);
    T* op = static_cast<T*>(out);
    const int64_t rows = total / n;
    const int64_t nvr = (n + E - 1) / E;
    // Launches whose rows no aligned vector fits go element by element while they are small (bf16 500 x 1001 2.4 µs
    // against 3.1 in runs, 1000 x 1001 3.0 / 3.3, 2000 x 1001 4.1 / 3.7) or their rows narrow: a block holds two rows,
    // so few of its threads have a run. f32 16M / n x n: n = 1 31 µs against 1769 in runs, 63 31 / 41, 129 31 / 28,
    // 257 31 / 24 (at 2M, 129 4.8 / 5.7, 255 4.8 / 5.9, 257 4.8 / 4.5); f16 1 29 / 2035, 127 28 / 30 (at 64M
    // 76 / 135), 257 27 / 17 (at 64M 76 / 87), 300 27 / 14 (75 / 64).
    const bool by_element = !(n % E == 0 && aligned(y, 16) && aligned(out, 16) && aligned(bias, 16)) &&
                            (total <= (int64_t)1 << 20 || n <= (sizeof(T) == 2 ? 288 : 256));
    if (!by_element && nvr <= (int64_t)1 << 24) {
        const int tile = nvr >= kThreads ? kThreads : (int)((nvr + 63) / 64 * 64);
        const int ntiles = (int)((nvr + tile - 1) / tile);
        const int64_t groups = (rows + kBiasRowsPerBlock - 1) / kBiasRowsPerBlock;
        // The grid is one launch, of fewer than 2^32 work-items.
        if ((int64_t)ntiles * tile <= UINT32_MAX / groups) {
            auto go = [&](auto p) {
                constexpr int P = decltype(p)::value;
                const dim3 grid((unsigned)(ntiles * groups));
                return n % E == 0 ? launch(bias_rows<T, TB, P, false>, grid, tile, stream, yp, bp, op, rows, (int)n, (int)nvr,
                                           ntiles, tile)
                                  : launch(bias_rows<T, TB, P, true>, grid, tile, stream, yp, bp, op, rows, (int)n, (int)nvr,
                                           ntiles, tile);
            };
            switch (policy_for(2 * total * (int64_t)sizeof(T))) {
            case P_CACHED: return go(std::integral_constant<int, P_CACHED>{});
            case P_NT_STORES: return go(std::integral_constant<int, P_NT_STORES>{});
            default: return go(std::integral_constant<int, P_NT>{});
            }
        }
    }
    return launch(bias_scalar<T, TB>, grid_for(total, kThreads, 65536), kThreads, stream, yp, bp, op, total, n);
}

int dispatch_bias(const void* y, const void* bias, int b_dt, void* out, int dt, int64_t total, int64_t n,
                  hipStream_t stream) {
    if (total < 0 || n < 0) return SPH_EINVAL;
    if (!is_float_dtype(dt) || !is_float_dtype(b_dt)) return SPH_EINVAL;
    if (total == 0) return SPH_OK;
    if (n == 0 || total % n != 0) return SPH_EINVAL;
    if (y == nullptr || bias == nullptr || out == nullptr) return SPH_EINVAL;
    return with_float_type(dt, [&](auto ty) -> int {
        using T = decltype(ty);
        return with_float_type(b_dt, [&](auto tb) -> int {
            using TB = decltype(tb);
            return launch_bias<T, TB>(y, bias, out, total, n, stream);
        });
    });
}

}  // namespace
}  // namespace sph

extern "C" int sph_init(void* stream) { return sph::ensure_device_ready(static_cast<hipStream_t>(stream), nullptr); }

extern "C" int sph_add(const void* a, int64_t na, const void* b, int64_t nb, void* out, int dtype, void* stream) {
    return sph::dispatch_binary<sph::OP_ADD>(a, na, b, nb, out, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int sph_mul(const void* a, int64_t na, const void* b, int64_t nb, void* out, int dtype, void* stream) {
    return sph::dispatch_binary<sph::OP_MUL>(a, na, b, nb, out, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int sph_silu(const void* x, void* out, int dtype, int64_t n, void* stream) {
    return sph::dispatch_unary<sph::OP_SILU>(x, out, dtype, n, static_cast<hipStream_t>(stream));
}

extern "C" int sph_swiglu(const void* gate, const void* up, void* out, int dtype, int64_t n, void* stream) {
    if (n < 0) return SPH_EINVAL;
    return sph::dispatch_binary<sph::OP_SWIGLU>(gate, n, up, n, out, dtype, static_cast<hipStream_t>(stream));
}

extern "C" int sph_gelu_tanh(const void* x, void* out, int dtype, int64_t n, void* stream) {
    return sph::gelu_any<sph::OP_GELU>(x, out, dtype, n, static_cast<hipStream_t>(stream));
}

extern "C" int sph_gelu_erf(const void* x, void* out, int dtype, int64_t n, void* stream) {
    return sph::gelu_any<sph::OP_GELU_ERF>(x, out, dtype, n, static_cast<hipStream_t>(stream));
}

extern "C" int sph_add_bias(const void* y, const void* bias, int bias_dtype, void* out, int dtype, int64_t total,
                            int64_t n, void* stream) {
    return sph::dispatch_bias(y, bias, bias_dtype, out, dtype, total, n, static_cast<hipStream_t>(stream));
}
