// layout.hip — the device-resident decode helpers: head transposes and the
// KV-cache append, for gfx950.
//
// Reference (crates/sapient-backends/wgpu/src/resident.rs):
//   transpose_heads  [outer, inner, hd] → [inner, outer, hd]          (:420-458)
//   kv_append        src [n_kv, seq, hd] → cache[:, pos:pos+seq, :]
//                    of [n_kv, max_seq, hd], converted to the cache type (:645-711)
//
// Both are moves of hd-element rows between two row orders, so one kernel
// serves both: each thread moves 16 bytes of the narrower side (f32: 4
// elements, halves: 8; an f32 → half move reads two 16-byte words and writes
// one; 16 bytes of the wider side when hd is not a multiple of 8),
// non-temporal, with a per-row index map. The transpose walks 8 × 8 tiles of
// (outer, inner) rows, so a block's reads cover 8 runs of 8 consecutive
// source rows and its writes 8 runs of 8 consecutive output rows (measured at
// [8192, 32, 128] f32: 72 µs walking output rows with two 16-byte accesses per
// thread, 47.5 µs with one, 45.3 µs with tiles). The append walks source rows
// (reads contiguous, writes contiguous within each head's run of seq rows).
// Same-type moves copy raw bits (NaN payloads included); f32 → f16 / bf16
// rounds to nearest-even, the conversion the reference's host mirror applies
// (half::f16::from_f32). HBM-bound: read + write once per element.
#include <type_traits>

#include "sph_common.h"

namespace sph {
namespace {

constexpr int kThreads = 256;
constexpr uint32_t kTile = 8;  // transpose tiles: 8 outer x 8 inner rows

enum Map { M_TRANSPOSE = 0, M_KV = 1 };

// Row index map. TRANSPOSE: a = outer, b = inner, row = a tile-ordered row
// index (see tile_row). KV: walk source rows r = h·seq + s, destination row
// h·max_seq + pos + s (a = seq, b = max_seq, c = pos).
struct RowMap {
    uint32_t a, b;
    uint64_t c;
};

// Rows of one call number fewer than 2^32 (checked on the host), so the
// splits are 32-bit divisions. Returns false for the padding rows of edge tiles.
template <int MAP>
__device__ __forceinline__ bool map_row(uint32_t row, const RowMap& m, uint64_t& srow, uint64_t& drow) {
    if constexpr (MAP == M_TRANSPOSE) {
        // row = tile · 64 + w; tiles in output order (inner-tile major), and
        // inside a tile w = wi · 8 + wo, so consecutive rows are consecutive outputs.
        const uint32_t tiles_o = (m.a + kTile - 1) / kTile;
        const uint32_t tile = row / (kTile * kTile), w = row % (kTile * kTile);
        const uint32_t ti = tile / tiles_o, to = tile - ti * tiles_o;
        const uint32_t o = to * kTile + w % kTile, i = ti * kTile + w / kTile;
        if (o >= m.a || i >= m.b) return false;
        srow = (uint64_t)o * m.b + i;
        drow = (uint64_t)i * m.a + o;
    } else {
        const uint32_t hi = row / m.a, lo = row - hi * m.a;
        srow = row;
        drow = (uint64_t)hi * m.b + m.c + lo;
    }
    return true;
}

// Elements per thread of the vector path: 16 bytes of the narrower side (an
// f32 <-> half move reads or writes two 16-byte words, so both sides stay
// 16 bytes wide), or, when hd is not a multiple of that, 16 bytes of the wider side.
template <typename TS, typename TD>
struct MoveWidth {
    static constexpr int wide = 16 / (int)(sizeof(TS) < sizeof(TD) ? sizeof(TS) : sizeof(TD));
    static constexpr int narrow = 16 / (int)(sizeof(TS) > sizeof(TD) ? sizeof(TS) : sizeof(TD));
};

template <typename TS, typename TD, int E>
__device__ __forceinline__ void move_chunk(const TS* s, TD* d) {
    if constexpr (std::is_same<TS, TD>::value) {
        vstore<true>(reinterpret_cast<u32x4*>(d), vload<true>(reinterpret_cast<const u32x4*>(s)));
    } else {
        float v[E];
        load_f32<TS, E, true>(s, v);
        store_f32<TD, E, true>(d, v);
    }
}

// Vector path: hd a multiple of the chunk width E, both bases 16-byte aligned;
// rows [row0, row0 + items / cpr) of this launch, cpr chunks per row.
template <typename TS, typename TD, int MAP, int E>
__global__ __launch_bounds__(kThreads) void move_rows_vec(const TS* __restrict__ src, TD* __restrict__ dst,
                                                          uint32_t items, uint32_t cpr, uint32_t row0, RowMap m) {
    const uint32_t k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= items) return;
    const uint32_t r = k / cpr;
    const uint32_t c = (k - r * cpr) * E;
    uint64_t srow, drow;
    if (!map_row<MAP>(row0 + r, m, srow, drow)) return;
    const uint64_t hd = (uint64_t)cpr * E;
    move_chunk<TS, TD, E>(src + srow * hd + c, dst + drow * hd + c);
}

// Any hd / alignment: one element per thread.
template <typename TS, typename TD, int MAP>
__global__ __launch_bounds__(kThreads) void move_rows_scalar(const TS* __restrict__ src, TD* __restrict__ dst,
                                                             uint32_t items, uint32_t hd, uint32_t row0, RowMap m) {
    const uint32_t k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= items) return;
    const uint32_t r = k / hd;
    const uint32_t c = k - r * hd;
    uint64_t srow, drow;
    if (!map_row<MAP>(row0 + r, m, srow, drow)) return;
    if constexpr (std::is_same<TS, TD>::value) dst[drow * hd + c] = src[srow * hd + c];
    else dst[drow * hd + c] = narrow<TD>(widen(src[srow * hd + c]));
}

// `rows` = rows of the walk (the transpose's includes edge-tile padding).
template <typename TS, typename TD, int MAP>
int launch_move(const void* src, void* dst, uint64_t rows, uint64_t hd, RowMap m, hipStream_t stream) {
    if (rows == 0 || hd == 0) return SPH_OK;
    if (hd > (1u << 24) || rows > UINT32_MAX) return SPH_EINVAL;
    constexpr int EW = MoveWidth<TS, TD>::wide, EN = MoveWidth<TS, TD>::narrow;
    const TS* s = static_cast<const TS*>(src);
    TD* d = static_cast<TD*>(dst);
    const bool al = aligned(src, 16) && aligned(dst, 16);
    const int E = !al ? 0 : hd % EW == 0 ? EW : hd % EN == 0 ? EN : 0;  // 0: scalar path
    const uint64_t per_row = E ? hd / E : hd;  // work items per row
    // Each launch covers whole rows (whole tiles for the transpose) and fewer than 2^31 work items.
    uint64_t rows_per_launch = ((uint64_t)1 << 31) / per_row;
    if (MAP == M_TRANSPOSE) rows_per_launch -= rows_per_launch % (kTile * kTile);
    for (uint64_t r0 = 0; r0 < rows; r0 += rows_per_launch) {
        const uint64_t nr = rows - r0 < rows_per_launch ? rows - r0 : rows_per_launch;
        const uint32_t items = (uint32_t)(nr * per_row);
        const dim3 grid((items + kThreads - 1) / kThreads);
        const int st = E == EW ? launch(move_rows_vec<TS, TD, MAP, EW>, grid, kThreads, stream, s, d, items,
                                        (uint32_t)per_row, (uint32_t)r0, m)
                     : E == EN ? launch(move_rows_vec<TS, TD, MAP, EN>, grid, kThreads, stream, s, d, items,
                                        (uint32_t)per_row, (uint32_t)r0, m)
                               : launch(move_rows_scalar<TS, TD, MAP>, grid, kThreads, stream, s, d, items,
                                        (uint32_t)hd, (uint32_t)r0, m);
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

// Q8_0 cache: the quantizer of the reference's quantized KV cache
// (crates/sapient-models/src/forward/common.rs:336-348, the same steps as
// quant.rs:223-235) over each 32-element block of a (head, token) row: amax
// (NaN skipped, as f32::max folds), scale = amax / 127 in f32, d = f16(scale),
// q = clamp(round(v · 1/scale), ±127) with round half away from zero and NaN →
// 0 (the `as i8` cast), and 0 throughout for an all-zero block. Row layout:
// head_dim / 32 blocks of 34 bytes (f16 d, 32 × i8), rows of a head at
// positions 0 .. max_seq - 1.
// A block is read by kQ8Lanes neighbouring lanes, which share the amax through
// DPP moves: a wave's accesses are contiguous, where one thread per block
// walked its 128 bytes alone, 64 lanes 128 bytes apart.
// Bound by the quantizer's ~30 VALU operations per four elements as much as by
// its bytes: at f32 8 x 2048 x 128 (10.6 MB) 4.0 us one thread per block, 3.0
// with four lanes, 3.2 with two, 3.9 with eight (each lane divides twice), 4.3
// with eight and the packed blocks leaving through LDS in 16-byte stores; a
// decode step (8 x 1 x 128) 2.7 -> 1.9.
// items / kQ8Lanes / bpr rows from token s0 of the first head of src and cache.
constexpr uint32_t kQ8Lanes = 4;

// round(t), half away from zero, of |t| <= 127.5 (f32's predecessor of 1/2 is added, so that no sum
// below the next integer rounds up to it), clamped to ±127; NaN → 0.
__device__ __forceinline__ uint32_t q8_byte(float t) {
    t = t == t ? fminf(fmaxf(t, -127.0f), 127.0f) : 0.0f;
    return (uint32_t)(int32_t)(t + __builtin_copysignf(0x1.fffffep-2f, t)) & 0xFFu;
}

template <typename TS>
__global__ __launch_bounds__(kThreads) void kv_append_q8_0(const TS* __restrict__ src, uint8_t* __restrict__ cache,
                                                           uint32_t items, uint32_t bpr, uint32_t seq,
                                                           uint32_t max_seq, uint64_t pos, uint32_t s0) {
    constexpr uint32_t L = kQ8Lanes;
    constexpr int V = 32 / (int)L;  // values per lane
    const uint32_t i = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (i >= items) return;         // items is a multiple of L: a block's lanes leave together
    const uint32_t k = i / L, lane = i % L;
    const uint32_t r = k / bpr, blk = k - r * bpr;
    const uint32_t row = s0 + r;    // source row h · seq + s (below 2^32: see the launch)
    const uint32_t h = row / seq, s = row - h * seq;
    float v[V];
    load_f32<TS, V>(src + ((uint64_t)row * bpr + blk) * 32 + lane * V, v);
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < V; ++e) amax = fmaxf(amax, fabsf(v[e]));
    amax = fmaxf(amax, dpp_mov<0xb1>(amax));  // quad_perm [1,0,3,2]
    amax = fmaxf(amax, dpp_mov<0x4e>(amax));  // quad_perm [2,3,0,1]
    const float scale = amax / 127.0f;
    const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
    uint8_t* out = cache + (((uint64_t)h * max_seq + pos + s) * bpr + blk) * 34;  // 2-byte aligned
    if (lane == 0) *reinterpret_cast<uint16_t*>(out) = narrow<f16>(scale).bits;
    typedef uint32_t words __attribute__((ext_vector_type(V / 4)));
    typedef words words_at2 __attribute__((aligned(2)));
    words q;
#pragma unroll
    for (int w = 0; w < V / 4; ++w)
        q[w] = q8_byte(v[4 * w] * inv) | q8_byte(v[4 * w + 1] * inv) << 8 | q8_byte(v[4 * w + 2] * inv) << 16 |
               q8_byte(v[4 * w + 3] * inv) << 24;
    *reinterpret_cast<words_at2*>(out + 2 + lane * V) = q;
}

// Sliding-window shift of a KV cache (the trait path's update_kv_cache,
// crates/sapient-models/src/forward/common.rs:392-405 and :475-485): in every
// head, rows [shift, cur_len) move to [0, keep), keep = cur_len - shift, in
// place; the `shift` rows after them are then overwritten by the append. With
// X = rows [0, shift) and Y = rows [shift, cur_len), reversing Y and then the
// whole of [0, cur_len) turns X Y into Y rev(X): Y lands in [0, keep) and
// rev(X) in the rows the append overwrites. A reversal is a set of disjoint
// row swaps (row lo + j with row hi - 1 - j), so every thread swaps its units
// on its own — no ordering between blocks, no scratch memory — and the kernel
// boundary orders the two passes; the second writes the new rows too where the cache's
// rows split into 16-byte units (kv_reverse_append: f16 2 x 4096 x 64 7.7 -> 5.4 us, a launch
// less). Shifts of a few rows of a larger cache move in windows instead (Windows). Each pass reads and writes every row once
// (twice the bytes of a direct move) in whole rows, coalesced, over the whole
// GPU; a direct in-place move must keep each column of a head in one block,
// since a row is read by the row `shift` below it (16 bytes per row access,
// 128 blocks): a one-token update of a full 8 x 8192 x 128 f16 cache took
// 31.7 us that way and 16.0 us with the two passes, the append included.
template <typename UT>
__global__ __launch_bounds__(kThreads) void kv_reverse_rows(UT* cache, uint32_t units_per_row, uint64_t max_seq,
                                                            uint64_t lo, uint64_t hi, uint32_t items) {
    // items = (hi - lo) / 2 pairs x units_per_row, per head (blockIdx.y).
    const uint32_t i = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (i >= items) return;
    const uint32_t j = i / units_per_row, u = i - j * units_per_row;
    UT* base = cache + (uint64_t)blockIdx.y * max_seq * units_per_row + u;
    UT* a = base + (lo + j) * units_per_row;
    UT* b = base + (hi - 1 - j) * units_per_row;
    const UT va = *a, vb = *b;
    *a = vb;
    *b = va;
}

template <typename UT>
int launch_reverse(void* cache, uint64_t n_heads, uint64_t row_bytes, uint64_t max_seq, uint64_t lo, uint64_t hi,
                   hipStream_t stream) {
    const uint64_t upr = row_bytes / sizeof(UT);
    const uint64_t items = (hi - lo) / 2 * upr;
    if (items == 0) return SPH_OK;
    if (items > UINT32_MAX - kThreads || upr > UINT32_MAX) return SPH_EINVAL;
    constexpr uint64_t kMaxY = 65535;  // heads per launch (grid y)
    for (uint64_t h0 = 0; h0 < n_heads; h0 += kMaxY) {
        const uint64_t nh = n_heads - h0 < kMaxY ? n_heads - h0 : kMaxY;
        const dim3 grid((unsigned)((items + kThreads - 1) / kThreads), (unsigned)nh);
        const int st = launch(kv_reverse_rows<UT>, grid, kThreads, stream,
                              static_cast<UT*>(cache) + h0 * max_seq * upr, (uint32_t)upr, max_seq, lo, hi,
                              (uint32_t)items);
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

// The shift of a few rows (decode steps) in two launches: each row moves once, and `shift` rows of every window
// a second time. The rows [0, cur_len) of a head are cut into windows.
//  1. Every window's first `shift` rows (its slot) take the next window's: those are the rows that follow
//     the window, and the rows a slot held are the ones that the window before it takes. (The first slot's
//     rows are the dropped ones.)
//  2. Every window rotates left by `shift`: its own rows move down and the slot's end it. The last window's
//     end is the new rows' place.
// A block holds all it moves in registers between its loads and its stores, so the in-place moves need no
// order between blocks; only the two launches are ordered. HBM-bound: the second launch moves 33.5 MB in
// 5.5-7.5 us, the first waits on memory once (1.6-2.7 us). A one-token update against the reversal with its
// append, in turn on one MI355X: f16 32 x 4096 x 96 13.2 -> 10.7 us, 8 x 16384 x 128 20.8 -> 14.5; f32 31.3 -> 18.9,
// 38.8 -> 25.5; Q8_0 20.9 -> 15.6, 13.8 -> 12.8. Non-temporal accesses cost 1-3 us. Caches below kWindowBytes are
// bound by latency, the slots' launch above all, and reverse.
struct Windows {
    uint32_t count, shift;
    uint32_t step, rem;  // window c starts at row c * step + min(c, rem)
    __device__ __forceinline__ uint32_t start(uint32_t c) const { return c * step + (c < rem ? c : rem); }
};

// Units per thread of a window (64 f16 rows of 128 a block); 2 and 8 measured 0.2-5 us slower.
constexpr int kRotateUnits = 4;
constexpr int kSlotThreads = 1024, kSlotUnits = 4;  // step 1 (256 or 512 threads: within 1 us either way)

// Loads whose addresses another wave stores to after the barrier have to have arrived before it.
__device__ __forceinline__ void loads_landed() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// Step 1: a block owns `per_block` unit offsets of every slot of a head (count <= kSlotThreads * kSlotUnits).
template <typename UT>
__global__ __launch_bounds__(kSlotThreads) void kv_shift_slots(UT* cache, uint32_t upr, uint64_t max_seq, Windows w,
                                                              uint32_t per_block) {
    const uint32_t u0 = blockIdx.x * per_block, slot_units = w.shift * upr;
    const uint32_t nu = slot_units - u0 < per_block ? slot_units - u0 : per_block;
    const uint32_t n = (w.count - 1) * nu;
    UT* base = cache + (uint64_t)blockIdx.y * max_seq * upr + u0;
    UT v[kSlotUnits];
#pragma unroll
    for (int k = 0; k < kSlotUnits; ++k) {
        const uint32_t i = (uint32_t)k * kSlotThreads + threadIdx.x;
        const uint32_t c = i / nu;
        if (i < n) v[k] = base[(uint64_t)w.start(c + 1) * upr + (i - c * nu)];
    }
    loads_landed();
#pragma unroll
    for (int k = 0; k < kSlotUnits; ++k) {
        const uint32_t i = (uint32_t)k * kSlotThreads + threadIdx.x;
        const uint32_t c = i / nu;
        if (i < n) base[(uint64_t)w.start(c) * upr + (i - c * nu)] = v[k];
    }
}

// Step 2, window blockIdx.x of head blockIdx.y: `append` writes the new rows over the last window's end,
// once its rows are in registers (or is empty: a later launch writes them).
template <typename UT, typename F>
__device__ __forceinline__ void rotate_window(UT* head, uint32_t upr, const Windows& w, F&& append) {
    const uint32_t start = w.start(blockIdx.x);
    const uint32_t n = (w.start(blockIdx.x + 1) - start) * upr, sh = w.shift * upr;
    const bool last = blockIdx.x == w.count - 1;
    UT* base = head + (uint64_t)start * upr;
    UT v[kRotateUnits];
#pragma unroll
    for (int k = 0; k < kRotateUnits; ++k) {
        const uint32_t i = (uint32_t)k * kThreads + threadIdx.x;
        if (i < n) v[k] = base[i];
    }
    loads_landed();
#pragma unroll
    for (int k = 0; k < kRotateUnits; ++k) {
        const uint32_t i = (uint32_t)k * kThreads + threadIdx.x;
        if (i < n && i >= sh) base[i - sh] = v[k];
        if (i < sh && !last) base[i + n - sh] = v[k];
    }
    if (last) append();
}

template <typename UT>
__global__ __launch_bounds__(kThreads) void kv_rotate_windows(UT* cache, uint32_t upr, uint64_t max_seq, Windows w) {
    rotate_window(cache + (uint64_t)blockIdx.y * max_seq * upr, upr, w, [] {});
}

// Step 2 with the append: the last window's block writes the new rows on its own place, the blocks after it
// those past cur_len.
template <typename TS, typename TD>
__global__ __launch_bounds__(kThreads) void kv_rotate_append(TD* cache, const TS* __restrict__ src, uint32_t upr,
                                                             uint64_t max_seq, Windows w, uint64_t keep, uint32_t seq) {
    constexpr int E = vec16<TD>::n;
    TD* head = cache + (uint64_t)blockIdx.y * max_seq * upr * E;
    const TS* s = src + (uint64_t)blockIdx.y * seq * upr * E;
    TD* d = head + keep * upr * E;
    auto append = [&](uint32_t i) { move_chunk<TS, TD, E>(s + (uint64_t)i * E, d + (uint64_t)i * E); };
    if (blockIdx.x < w.count) {
        rotate_window(reinterpret_cast<u32x4*>(head), upr, w, [&] {
            for (uint32_t i = threadIdx.x; i < w.shift * upr; i += kThreads) append(i);
        });
    } else {
        const uint32_t i = w.shift * upr + (blockIdx.x - w.count) * kThreads + threadIdx.x;
        if (i < seq * upr) append(i);
    }
}

// Valid rows (bytes, all heads) from which a cache that is cut into windows slides faster so than by reversal, by
// shift: f16 2 x 4096 x 64 (1 MB) 1 row 5.0 us against 4.5, 4 5.2 / 4.4, 16 7.0 / 4.6; 8 x 2048 x 128 (4.2 MB) 5.5 /
// 5.3, 6.4 / 5.6, 7.7 / 6.4; 8 x 4096 x 128 (8.4 MB) 6.3 / 6.9, 8.1 / 7.0, 9.1 / 9.0; 40 x 4000 x 32 (10 MB) 6.5 /
// 7.6, 6.7 / 7.8, 7.0 / 8.1; Q8_0 8 x 4096 x 128 (4.5 MB) 8.1 / 7.8, 9.7 / 8.4, 10.1 / 9.5; 40 x 4000 x 32 (5.4 MB)
// 9.7 / 11.9, 11.3 / 12.3, 12.6 / 13.9. (8 MB at 4-8 rows, the reversal's by 1 us, is still the faster for what the
// two passes and the append took.) A head that one block holds has no slots: one launch, 2.3 us against 3.6.
constexpr uint64_t kWindowBytes = (uint64_t)5 << 20;

// The window cut for a shift; count = 0 where it does not apply: a window has to hold twice the shift, so
// that the slots' extra move stays well below the second move of every row that the reversal makes.
inline Windows cut_windows(uint64_t n_heads, uint64_t cur_len, uint64_t shift, uint64_t upr, uint64_t unit) {
    const uint64_t most = upr == 0 ? 0 : (uint64_t)kRotateUnits * kThreads / upr;  // rows a block holds
    if (cur_len <= shift || cur_len > INT32_MAX || 2 * shift + 2 > most) return Windows{0, 0, 0, 0};
    const uint64_t n = (cur_len + most - 1) / most;
    if (n > kSlotThreads * kSlotUnits) return Windows{0, 0, 0, 0};
    if (n > 1 && cur_len * upr * unit < (kWindowBytes + n_heads - 1) / n_heads) return Windows{0, 0, 0, 0};
    // n > 1: every window has at least cur_len / n > most / 2 > shift rows.
    return Windows{(uint32_t)n, (uint32_t)shift, (uint32_t)(cur_len / n), (uint32_t)(cur_len % n)};
}

// The shift in windows; with TS also the append.
template <typename UT, typename TS, typename TD>
int shift_by_windows(void* cache, const TS* src, uint64_t n_heads, uint64_t upr, uint64_t seq, uint64_t max_seq,
                     uint64_t keep, const Windows& w, hipStream_t stream) {
    constexpr uint64_t kMaxY = 65535;  // heads per launch (grid y)
    for (uint64_t h0 = 0; h0 < n_heads; h0 += kMaxY) {
        const unsigned nh = (unsigned)(n_heads - h0 < kMaxY ? n_heads - h0 : kMaxY);
        UT* base = static_cast<UT*>(cache) + h0 * max_seq * upr;
        int st = SPH_OK;
        if (w.count > 1) {
            const uint32_t slot_units = w.shift * (uint32_t)upr;
            uint32_t per_block = (uint32_t)(kSlotThreads * kSlotUnits) / (w.count - 1);
            if (per_block > slot_units) per_block = slot_units;
            st = launch(kv_shift_slots<UT>, dim3((slot_units + per_block - 1) / per_block, nh), kSlotThreads, stream, base,
                        (uint32_t)upr, max_seq, w, per_block);
            if (st != SPH_OK) return st;
        }
        if constexpr (!std::is_same<TS, void>::value) {
            constexpr uint64_t E = vec16<TD>::n;
            const uint64_t past = (seq - w.shift) * upr;  // units of new rows past cur_len
            st = launch(kv_rotate_append<TS, TD>, dim3(w.count + (unsigned)((past + kThreads - 1) / kThreads), nh), kThreads,
                        stream, reinterpret_cast<TD*>(base), src + h0 * seq * upr * E, (uint32_t)upr, max_seq, w, keep,
                        (uint32_t)seq);
        } else {
            st = launch(kv_rotate_windows<UT>, dim3(w.count, nh), kThreads, stream, base, (uint32_t)upr, max_seq, w);
        }
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

// Second reversal pass (the whole of [0, n)) with the append: a row that the pass would leave from `keep`
// on is written from src by the thread that has read it; rows [n, keep + seq) follow the pairs.
template <typename TS, typename TD>
__global__ __launch_bounds__(kThreads) void kv_reverse_append(TD* cache, const TS* __restrict__ src, uint32_t upr,
                                                              uint64_t max_seq, uint32_t n, uint32_t keep, uint32_t seq,
                                                              uint32_t items) {
    constexpr int E = vec16<TD>::n;
    const uint32_t i = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (i >= items) return;
    const uint32_t j = i / upr, u = i - j * upr;
    TD* head = cache + (uint64_t)blockIdx.y * max_seq * upr * E + (uint64_t)u * E;
    const TS* s = src + (uint64_t)blockIdx.y * seq * upr * E + (uint64_t)u * E;
    auto row = [&](uint32_t r) { return reinterpret_cast<u32x4*>(head + (uint64_t)r * upr * E); };
    auto append = [&](uint32_t r) {
        move_chunk<TS, TD, E>(s + (uint64_t)(r - keep) * upr * E, head + (uint64_t)r * upr * E);
    };
    const uint32_t pairs = (n + 1) / 2;
    if (j >= pairs) {
        append(n + (j - pairs));
        return;
    }
    const uint32_t b = n - 1 - j;  // j itself for the middle row of an odd n
    const u32x4 va = *row(j), vb = *row(b);
    if (j < keep) *row(j) = vb;
    else append(j);
    if (b == j) return;
    if (b < keep) *row(b) = va;
    else append(b);
}

// Shift and append of a float cache whose rows split into 16-byte units.
template <typename TS, typename TD>
int shift_append(const void* src, void* cache, uint64_t n_heads, uint64_t hd, uint64_t seq, uint64_t max_seq,
                 uint64_t shift, uint64_t cur_len, hipStream_t stream) {
    constexpr uint64_t E = vec16<TD>::n;
    const uint64_t upr = hd / E, keep = cur_len - shift;
    const TS* s = static_cast<const TS*>(src);
    const Windows w = cut_windows(n_heads, cur_len, shift, upr, 16);
    if (w.count > 0) return shift_by_windows<u32x4, TS, TD>(cache, s, n_heads, upr, seq, max_seq, keep, w, stream);
    int st = launch_reverse<u32x4>(cache, n_heads, hd * sizeof(TD), max_seq, shift, cur_len, stream);
    if (st != SPH_OK) return st;
    constexpr uint64_t kMaxY = 65535;  // heads per launch (grid y)
    const uint64_t items = ((cur_len + 1) / 2 + (keep + seq - cur_len)) * upr;
    for (uint64_t h0 = 0; h0 < n_heads; h0 += kMaxY) {
        const unsigned nh = (unsigned)(n_heads - h0 < kMaxY ? n_heads - h0 : kMaxY);
        st = launch(kv_reverse_append<TS, TD>, dim3((unsigned)((items + kThreads - 1) / kThreads), nh), kThreads, stream,
                    static_cast<TD*>(cache) + h0 * max_seq * hd, s + h0 * seq * hd, (uint32_t)upr, max_seq,
                    (uint32_t)cur_len, (uint32_t)keep, (uint32_t)seq, (uint32_t)items);
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

// The two passes, with the widest unit the row width and the cache's alignment allow.
// The second pass covers more rows than the first, so checking its item count
// before either launch means a rejected shift leaves the cache untouched.
template <typename UT>
int shift_window(void* cache, uint64_t n_heads, uint64_t row_bytes, uint64_t max_seq, uint64_t shift,
                 uint64_t cur_len, hipStream_t stream) {
    const uint64_t upr = row_bytes / sizeof(UT);
    if (upr > UINT32_MAX || cur_len / 2 * upr > UINT32_MAX - kThreads) return SPH_EINVAL;
    const Windows w = cut_windows(n_heads, cur_len, shift, upr, sizeof(UT));
    if (w.count > 0)
        return shift_by_windows<UT, void, void>(cache, nullptr, n_heads, upr, 0, max_seq, cur_len - shift, w, stream);
    const int st = launch_reverse<UT>(cache, n_heads, row_bytes, max_seq, shift, cur_len, stream);
    if (st != SPH_OK) return st;
    return launch_reverse<UT>(cache, n_heads, row_bytes, max_seq, 0, cur_len, stream);
}

// Out-of-place window update: row j < new_len of every head of `out` is cache
// row shift + j for j < keep, else src row j - keep converted to the cache type.
// Each kept row crosses HBM once each way (the in-place form's two reversal
// passes move it twice), and the new rows land in the same launch. An item is
// 16 bytes of the cache side (E elements of TD); each thread moves two, items
// i and i + stride (stride = the launch's threads per head, so every memory
// instruction of a wave stays one contiguous run); grid.y walks the heads.
// Same-type moves copy raw bits. Measured on a one-token update of a full
// 8 x 8192 x 128 f16 cache (back-to-back launches): one item per thread
// 7.9 us, two 7.3 us, four 7.5 us; 512- or 1024-thread blocks and grid-stride
// loops over 1024-2048 blocks no faster; a device-to-device hipMemcpyAsync of
// the kept rows alone 8.0 us.
template <typename TS, typename TD, int E>
__global__ __launch_bounds__(kThreads) void kv_window_into(const TD* __restrict__ cache, const TS* __restrict__ src,
                                                           TD* __restrict__ out, uint32_t cpr, uint32_t keep,
                                                           uint32_t seq, uint64_t max_seq, uint64_t shift,
                                                           uint32_t items, uint64_t h0) {
    const uint32_t stride = gridDim.x * (uint32_t)kThreads;
    const uint32_t i0 = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    const uint64_t h = h0 + blockIdx.y;
    const uint64_t hd = (uint64_t)cpr * E;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const uint32_t i = i0 + (uint32_t)u * stride;
        if (i >= items) return;
        const uint32_t j = i / cpr;
        const uint32_t c = (i - j * cpr) * E;
        TD* d = out + (h * max_seq + j) * hd + c;
        if (j < keep) {
            const TD* s = cache + (h * max_seq + shift + j) * hd + c;
            vstore<true>(reinterpret_cast<u32x4*>(d), vload<true>(reinterpret_cast<const u32x4*>(s)));
        } else {
            move_chunk<TS, TD, E>(src + (h * seq + (j - keep)) * hd + c, d);
        }
    }
}

// Rows [shift, shift + keep) of every head of cache → rows [0, keep) of out,
// as raw units of UT (any row width: the Q8_0 cache's 34-byte blocks, odd
// head dims); the new rows are appended by a second launch.
template <typename UT>
__global__ __launch_bounds__(kThreads) void kv_copy_rows(const UT* __restrict__ cache, UT* __restrict__ out,
                                                         uint32_t units_per_row, uint64_t max_seq, uint64_t shift,
                                                         uint32_t items, uint64_t h0) {
    const uint32_t i = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (i >= items) return;
    const uint32_t j = i / units_per_row, u = i - j * units_per_row;
    const uint64_t base = (h0 + blockIdx.y) * max_seq * units_per_row + u;
    out[base + (uint64_t)j * units_per_row] = cache[base + (shift + j) * units_per_row];
}

constexpr uint64_t kMaxGridY = 65535;  // heads per launch

template <typename TS, typename TD>
int launch_window_into(const void* cache, const void* src, void* out, uint64_t n_heads, uint64_t hd, uint64_t seq,
                       uint64_t max_seq, uint64_t shift, uint64_t keep, hipStream_t stream) {
    constexpr int E = vec16<TD>::n;
    const uint64_t cpr = hd / E;
    const uint64_t items = (keep + seq) * cpr;
    const uint64_t threads = (items + 1) / 2;  // two items per thread
    for (uint64_t h0 = 0; h0 < n_heads; h0 += kMaxGridY) {
        const uint64_t nh = n_heads - h0 < kMaxGridY ? n_heads - h0 : kMaxGridY;
        const dim3 grid((unsigned)((threads + kThreads - 1) / kThreads), (unsigned)nh);
        const int st = launch(kv_window_into<TS, TD, E>, grid, kThreads, stream, static_cast<const TD*>(cache),
                              static_cast<const TS*>(src), static_cast<TD*>(out), (uint32_t)cpr, (uint32_t)keep,
                              (uint32_t)seq, max_seq, shift, (uint32_t)items, h0);
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

template <typename UT>
int launch_copy_rows(const void* cache, void* out, uint64_t n_heads, uint64_t row_bytes, uint64_t max_seq,
                     uint64_t shift, uint64_t keep, hipStream_t stream) {
    const uint64_t upr = row_bytes / sizeof(UT);
    const uint64_t items = keep * upr;
    if (items == 0) return SPH_OK;
    for (uint64_t h0 = 0; h0 < n_heads; h0 += kMaxGridY) {
        const uint64_t nh = n_heads - h0 < kMaxGridY ? n_heads - h0 : kMaxGridY;
        const dim3 grid((unsigned)((items + kThreads - 1) / kThreads), (unsigned)nh);
        const int st = launch(kv_copy_rows<UT>, grid, kThreads, stream, static_cast<const UT*>(cache),
                              static_cast<UT*>(out), (uint32_t)upr, max_seq, shift, (uint32_t)items, h0);
        if (st != SPH_OK) return st;
    }
    return SPH_OK;
}

}  // namespace
}  // namespace sph

extern "C" int sph_transpose_heads(const void* x, void* out, int dtype, int64_t outer, int64_t inner,
                                   int64_t head_dim, void* stream) {
    if (outer < 0 || inner < 0 || head_dim < 0 || !sph::is_float_dtype(dtype)) return SPH_EINVAL;
    const uint64_t rows = (uint64_t)outer * (uint64_t)inner;
    if (rows == 0 || head_dim == 0) return SPH_OK;
    if (x == nullptr || out == nullptr || x == out) return SPH_EINVAL;
    if (outer > UINT32_MAX || inner > UINT32_MAX) return SPH_EINVAL;
    // The walk covers whole 8 x 8 tiles; padding rows are skipped in the kernel.
    const uint64_t t = sph::kTile;
    const uint64_t walk = (((uint64_t)outer + t - 1) / t) * (((uint64_t)inner + t - 1) / t) * t * t;
    const sph::RowMap m{(uint32_t)outer, (uint32_t)inner, 0};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SPH_F32) return sph::launch_move<float, float, sph::M_TRANSPOSE>(x, out, walk, head_dim, m, s);
    // Halves move as 16-bit patterns; the element type does not matter.
    return sph::launch_move<sph::f16, sph::f16, sph::M_TRANSPOSE>(x, out, walk, head_dim, m, s);
}

namespace {

// Every argument check of sph_kv_append: SPH_OK when the append would launch (or
// has nothing to do), else the error it returns. sph_kv_cache_update runs it
// before shifting, so a rejected call leaves the cache untouched.
int kv_append_check(const void* src, int src_dtype, const void* cache, int cache_dtype, int64_t n_kv, int64_t seq,
                    int64_t head_dim, int64_t max_seq, int64_t pos) {
    if (n_kv < 0 || seq < 0 || head_dim < 0 || max_seq < 0 || pos < 0) return SPH_EINVAL;
    const bool q8 = cache_dtype == SPH_Q8_0;
    if (!sph::is_float_dtype(src_dtype) || !(q8 || sph::is_float_dtype(cache_dtype))) return SPH_EINVAL;
    if (q8 && head_dim % 32 != 0) return SPH_EINVAL;
    if (pos > max_seq || seq > max_seq - pos) return SPH_ERANGE;
    const uint64_t rows = (uint64_t)n_kv * (uint64_t)seq;
    if (rows == 0 || head_dim == 0) return SPH_OK;
    if (src == nullptr || cache == nullptr) return SPH_EINVAL;
    if (seq > UINT32_MAX || max_seq > UINT32_MAX) return SPH_EINVAL;
    if (q8) {
        if (!sph::aligned(cache, 2) || !sph::aligned(src, 16) || head_dim / 32 > UINT32_MAX) return SPH_EINVAL;
        const uint64_t blocks = rows * ((uint64_t)head_dim / 32);
        if ((blocks + sph::kThreads - 1) / sph::kThreads > INT32_MAX) return SPH_EINVAL;
    } else if ((uint64_t)head_dim > (1u << 24) || rows > UINT32_MAX) {
        return SPH_EINVAL;  // launch_move's limits
    }
    return SPH_OK;
}

}  // namespace

extern "C" int sph_kv_append(const void* src, int src_dtype, void* cache, int cache_dtype, int64_t n_kv, int64_t seq,
                             int64_t head_dim, int64_t max_seq, int64_t pos, void* stream) {
    const int chk = kv_append_check(src, src_dtype, cache, cache_dtype, n_kv, seq, head_dim, max_seq, pos);
    if (chk != SPH_OK) return chk;
    const bool q8 = cache_dtype == SPH_Q8_0;
    const uint64_t rows = (uint64_t)n_kv * (uint64_t)seq;
    if (rows == 0 || head_dim == 0) return SPH_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (q8) {
        const uint64_t bpr = (uint64_t)head_dim / 32;
        return sph::with_float_type(src_dtype, [&](auto ts) -> int {
            using TS = decltype(ts);
            // Launches of fewer than 2^32 lanes: whole heads, or runs of one head's rows.
            constexpr uint64_t kItems = (uint64_t)1 << 31;
            const uint64_t row_items = bpr * sph::kQ8Lanes, head_items = row_items * (uint64_t)seq;
            const bool heads = head_items <= kItems;
            const uint64_t step_h = heads ? kItems / head_items : 1, step_s = heads ? (uint64_t)seq : kItems / row_items;
            if (step_s == 0) return SPH_EINVAL;
            for (uint64_t h0 = 0; h0 < (uint64_t)n_kv; h0 += step_h) {
                const uint64_t nh = (uint64_t)n_kv - h0 < step_h ? (uint64_t)n_kv - h0 : step_h;
                for (uint64_t s0 = 0; s0 < (uint64_t)seq; s0 += step_s) {
                    const uint64_t ns = (uint64_t)seq - s0 < step_s ? (uint64_t)seq - s0 : step_s;
                    const uint32_t items = (uint32_t)(nh * ns * row_items);
                    const int st = sph::launch(
                        sph::kv_append_q8_0<TS>, dim3((items + sph::kThreads - 1) / sph::kThreads), sph::kThreads, s,
                        static_cast<const TS*>(src) + h0 * (uint64_t)seq * (uint64_t)head_dim,
                        static_cast<uint8_t*>(cache) + h0 * (uint64_t)max_seq * bpr * 34, items, (uint32_t)bpr,
                        (uint32_t)seq, (uint32_t)max_seq, (uint64_t)pos, (uint32_t)s0);
                    if (st != SPH_OK) return st;
                }
            }
            return SPH_OK;
        });
    }
    const sph::RowMap m{(uint32_t)seq, (uint32_t)max_seq, (uint64_t)pos};
    return sph::with_float_type(src_dtype, [&](auto ts) -> int {
        using TS = decltype(ts);
        return sph::with_float_type(cache_dtype, [&](auto td) -> int {
            using TD = decltype(td);
            return sph::launch_move<TS, TD, sph::M_KV>(src, cache, rows, head_dim, m, s);
        });
    });
}

extern "C" int sph_kv_cache_update(const void* src, int src_dtype, void* cache, int cache_dtype, int64_t n_kv,
                                   int64_t seq, int64_t head_dim, int64_t max_seq, int64_t cur_len, int64_t* new_len,
                                   void* stream) {
    if (n_kv < 0 || seq < 0 || head_dim < 0 || max_seq < 0 || cur_len < 0 || new_len == nullptr) return SPH_EINVAL;
    const bool q8 = cache_dtype == SPH_Q8_0;
    if (!sph::is_float_dtype(src_dtype) || !(q8 || sph::is_float_dtype(cache_dtype))) return SPH_EINVAL;
    if (q8 && head_dim % 32 != 0) return SPH_EINVAL;
    if (seq > max_seq) return SPH_ERANGE;      // the reference's "new tokens exceeds max cache size"
    if (cur_len > max_seq) return SPH_EINVAL;  // more valid rows than the cache holds
    const int64_t total = cur_len + seq;
    const int64_t shift = total > max_seq ? total - max_seq : 0;
    const int64_t keep = cur_len - shift;
    const int chk = kv_append_check(src, src_dtype, cache, cache_dtype, n_kv, seq, head_dim, max_seq, keep);
    if (chk != SPH_OK) return chk;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (shift > 0 && keep > 0 && n_kv > 0 && head_dim > 0) {
        if (cache == nullptr) return SPH_EINVAL;
        const uint64_t row_bytes = q8 ? (uint64_t)head_dim / 32 * 34 : (uint64_t)head_dim * sph::dtype_size(cache_dtype);
        int st;
        // Float caches whose rows split into 16-byte units: the append rides in the shift's last launch (of fewer than 2^32
        // work-items, the windows' and the rounding of both counts to blocks included).
        if (!q8 && row_bytes % 16 == 0 && sph::aligned(cache, 16)) {
            const uint64_t e = 16 / sph::dtype_size(cache_dtype), src_access = e * sph::dtype_size(src_dtype);
            if (sph::aligned(src, src_access < 16 ? src_access : 16) &&
                ((uint64_t)cur_len / 2 + 1 + (uint64_t)seq) * ((uint64_t)head_dim / e) <= UINT32_MAX - 4 * sph::kThreads) {
                st = sph::with_float_type(src_dtype, [&](auto ts) -> int {
                    using TS = decltype(ts);
                    return sph::with_float_type(cache_dtype, [&](auto td) -> int {
                        using TD = decltype(td);
                        return sph::shift_append<TS, TD>(src, cache, n_kv, head_dim, seq, max_seq, shift, cur_len, s);
                    });
                });
                if (st == SPH_OK) *new_len = max_seq;
                return st;
            }
        }
        if (row_bytes % 16 == 0 && sph::aligned(cache, 16))
            st = sph::shift_window<sph::u32x4>(cache, n_kv, row_bytes, max_seq, shift, cur_len, s);
        else if (row_bytes % 8 == 0 && sph::aligned(cache, 8))
            st = sph::shift_window<sph::u32x2>(cache, n_kv, row_bytes, max_seq, shift, cur_len, s);
        else if (row_bytes % 4 == 0 && sph::aligned(cache, 4))
            st = sph::shift_window<uint32_t>(cache, n_kv, row_bytes, max_seq, shift, cur_len, s);
        else if (sph::aligned(cache, 2))
            st = sph::shift_window<uint16_t>(cache, n_kv, row_bytes, max_seq, shift, cur_len, s);
        else
            return SPH_EINVAL;
        if (st != SPH_OK) return st;
    }
    const int st = sph_kv_append(src, src_dtype, cache, cache_dtype, n_kv, seq, head_dim, max_seq, keep, stream);
    if (st != SPH_OK) return st;
    *new_len = total < max_seq ? total : max_seq;
    return SPH_OK;
}

namespace {

// [a, a + na) and [b, b + nb) share a byte.
bool overlaps(const void* a, uint64_t na, const void* b, uint64_t nb) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return na != 0 && nb != 0 && x < y + nb && y < x + na;
}

}  // namespace

extern "C" int sph_kv_cache_update_into(const void* src, int src_dtype, const void* cache, void* out, int cache_dtype,
                                        int64_t n_kv, int64_t seq, int64_t head_dim, int64_t max_seq,
                                        int64_t cur_len, int64_t* new_len, void* stream) {
    if (n_kv < 0 || seq < 0 || head_dim < 0 || max_seq < 0 || cur_len < 0 || new_len == nullptr) return SPH_EINVAL;
    const bool q8 = cache_dtype == SPH_Q8_0;
    if (!sph::is_float_dtype(src_dtype) || !(q8 || sph::is_float_dtype(cache_dtype))) return SPH_EINVAL;
    if (q8 && head_dim % 32 != 0) return SPH_EINVAL;
    if (seq > max_seq) return SPH_ERANGE;      // the reference's "new tokens exceeds max cache size"
    if (cur_len > max_seq) return SPH_EINVAL;  // more valid rows than the cache holds
    const int64_t total = cur_len + seq;
    const int64_t shift = total > max_seq ? total - max_seq : 0;
    const int64_t keep = cur_len - shift;
    const int64_t n_new = total < max_seq ? total : max_seq;
    // The append part's checks, against `out`.
    const int chk = kv_append_check(src, src_dtype, out, cache_dtype, n_kv, seq, head_dim, max_seq, keep);
    if (chk != SPH_OK) return chk;
    if (n_kv == 0 || head_dim == 0 || n_new == 0) {
        *new_len = n_new;
        return SPH_OK;
    }
    const uint64_t row_bytes = q8 ? (uint64_t)head_dim / 32 * 34 : (uint64_t)head_dim * sph::dtype_size(cache_dtype);
    const uint64_t cache_bytes = (uint64_t)n_kv * (uint64_t)max_seq * row_bytes;
    const uint64_t src_bytes = (uint64_t)n_kv * (uint64_t)seq * (uint64_t)head_dim * sph::dtype_size(src_dtype);
    if (out == nullptr || (keep > 0 && cache == nullptr)) return SPH_EINVAL;
    // out is written while cache and src are read.
    if ((keep > 0 && overlaps(cache, cache_bytes, out, cache_bytes)) || overlaps(src, src_bytes, out, cache_bytes))
        return SPH_EINVAL;
    hipStream_t s = static_cast<hipStream_t>(stream);

    // Float caches whose rows split into 16-byte units: one launch does the move and the append.
    if (!q8 && sph::aligned(cache, 16) && sph::aligned(out, 16)) {
        const int64_t e = 16 / (int64_t)sph::dtype_size(cache_dtype);
        const uint64_t src_access = (uint64_t)e * sph::dtype_size(src_dtype);
        const uint64_t items = (uint64_t)n_new * (uint64_t)(head_dim / e);
        if (head_dim % e == 0 && sph::aligned(src, src_access < 16 ? src_access : 16) &&
            items <= UINT32_MAX - 2 * sph::kThreads) {  // i0 + stride stays below 2^32
            const int st = sph::with_float_type(src_dtype, [&](auto ts) -> int {
                using TS = decltype(ts);
                return sph::with_float_type(cache_dtype, [&](auto td) -> int {
                    using TD = decltype(td);
                    return sph::launch_window_into<TS, TD>(cache, src, out, n_kv, head_dim, seq, max_seq, shift,
                                                           keep, s);
                });
            });
            if (st != SPH_OK) return st;
            *new_len = n_new;
            return SPH_OK;
        }
    }
    // Any other row: the kept rows as raw units of the widest width both buffers allow, then the append.
    if (keep > 0) {
        auto fits = [&](uint64_t unit) {
            return row_bytes % unit == 0 && sph::aligned(cache, unit) && sph::aligned(out, unit) &&
                   row_bytes / unit <= UINT32_MAX && (uint64_t)keep * (row_bytes / unit) <= UINT32_MAX - sph::kThreads;
        };
        int st;
        if (fits(16)) st = sph::launch_copy_rows<sph::u32x4>(cache, out, n_kv, row_bytes, max_seq, shift, keep, s);
        else if (fits(8)) st = sph::launch_copy_rows<sph::u32x2>(cache, out, n_kv, row_bytes, max_seq, shift, keep, s);
        else if (fits(4)) st = sph::launch_copy_rows<uint32_t>(cache, out, n_kv, row_bytes, max_seq, shift, keep, s);
        else if (fits(2)) st = sph::launch_copy_rows<uint16_t>(cache, out, n_kv, row_bytes, max_seq, shift, keep, s);
        else return SPH_EINVAL;
        if (st != SPH_OK) return st;
    }
    const int st = sph_kv_append(src, src_dtype, out, cache_dtype, n_kv, seq, head_dim, max_seq, keep, stream);
    if (st != SPH_OK) return st;
    *new_len = n_new;
    return SPH_OK;
}
