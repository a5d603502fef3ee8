// Device side of the layer-streaming path for MI355X (gfx950).
//
// Every kernel here is a streaming kernel: each byte is read once and
// written once, so the bound is HBM bandwidth (or the host link, for the
// copies), never the matrix cores.  The kernels therefore use
//   - 128-bit global loads and stores, 8 elements per lane per group,
//   - several independent groups per lane, or many workgroups of one group per
//     lane, to keep enough bytes in flight,
//   - 128- or 256-lane workgroups (2 or 4 wave64s): over HBM many thousands of
//     them, so that all 256 CUs over the 8 XCDs stay busy, over the host link a
//     few dozen, which fill it,
//   - no MFMA, and LDS only for the ids of the row gathers.
//
// The C ABI is declared in include/slidefsdp.h.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <hsa/hsa.h>
#include <hsa/hsa_ext_amd.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <chrono>
#include <mutex>
#include <thread>
#include <unordered_map>

#include "../../include/slidefsdp.h"

namespace {

constexpr int kThreads = 256;  // lanes per workgroup (4 wave64s)
constexpr int kUnroll = 4;     // 8-element groups per lane per workgroup tile
constexpr int kCastUnroll = 1; // the same for the flat cast (measured best, see below)
constexpr int kCastThreads = 128;  // lanes per workgroup of the flat cast (2 wave64s, see below)
constexpr int kGroup = 8;      // elements per 128-bit bf16 store
constexpr uint64_t kSizeUnit = 8192;  // elements; a segment table's size limit is counted in these

// Native vector types: the nontemporal builtins need them (HIP's float4 is a
// struct), and they map one-to-one onto 128-bit global_load/store_dwordx4.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// The same 128 bits at the alignment of one element: still one access.
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));

// fp32 -> bf16 with round-to-nearest-even on the bit pattern, NaN -> 0xFFFF.
// This is the arithmetic of torch's vectorised CPU cast that the reference
// calls at layer_state.py:301 (ATen cvtfp32_bf16: bias 0x7FFF plus the lsb
// of the kept half, and an all-ones pattern for unordered inputs); the
// tests pin it against that routine.  Denormals, infinities and signed
// zeros follow from the integer arithmetic.
__device__ __forceinline__ uint32_t rne_bf16(uint32_t u) {
    const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
    return ((u & 0x7FFFFFFFu) > 0x7F800000u) ? 0xFFFFu : r;
}

// fp32 -> fp16, IEEE round to nearest even with subnormals; overflow to
// infinity; NaN -> quiet NaN keeping the sign and the top 9 payload bits.
// This is what torch's CPU cast gives (`.to(torch.float16)`, the reference's
// staging of fp16 units, layer_state.py:301); the tests pin it against that
// routine.  v_cvt_f16_f32 does exactly this under the rounding and denormal
// modes that the compiler sets for every kernel (nearest even, fp16
// subnormals kept): compared with the same conversion in integer arithmetic
// over all 2^32 inputs, no bit differs, NaN payloads included.  The integer
// form took some 25 instructions per element and bound the cast: 12.6 M
// elements 17.8 us, with the instruction 14.2.
__device__ __forceinline__ uint32_t rne_f16(uint32_t u) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(__uint_as_float(u)));
}

__device__ __forceinline__ uint32_t pack2(uint32_t lo, uint32_t hi) {
    return lo | (hi << 16);
}

__device__ __forceinline__ u32x4 cast8(const f32x4 a, const f32x4 b) {
    u32x4 o;
    o.x = pack2(rne_bf16(__float_as_uint(a.x)), rne_bf16(__float_as_uint(a.y)));
    o.y = pack2(rne_bf16(__float_as_uint(a.z)), rne_bf16(__float_as_uint(a.w)));
    o.z = pack2(rne_bf16(__float_as_uint(b.x)), rne_bf16(__float_as_uint(b.y)));
    o.w = pack2(rne_bf16(__float_as_uint(b.z)), rne_bf16(__float_as_uint(b.w)));
    return o;
}

__device__ __forceinline__ u32x4 cast8_f16(const f32x4 a, const f32x4 b) {
    u32x4 o;
    o.x = pack2(rne_f16(__float_as_uint(a.x)), rne_f16(__float_as_uint(a.y)));
    o.y = pack2(rne_f16(__float_as_uint(a.z)), rne_f16(__float_as_uint(a.w)));
    o.z = pack2(rne_f16(__float_as_uint(b.x)), rne_f16(__float_as_uint(b.y)));
    o.w = pack2(rne_f16(__float_as_uint(b.z)), rne_f16(__float_as_uint(b.w)));
    return o;
}

// Elements between the 16-byte boundary at or before a 16-bit destination
// and the destination itself (0 to 7).
__host__ __device__ inline uint32_t lead_elems(uint64_t dst) { return uint32_t(dst & 15) >> 1; }

// Output formats of the flat cast.
struct ToBf16 {
    __device__ static u32x4 cast8(const f32x4 a, const f32x4 b) { return ::cast8(a, b); }
    __device__ static uint16_t cast1(float x) { return uint16_t(rne_bf16(__float_as_uint(x))); }
};
struct ToF16 {
    __device__ static u32x4 cast8(const f32x4 a, const f32x4 b) { return cast8_f16(a, b); }
    __device__ static uint16_t cast1(float x) { return uint16_t(rne_f16(__float_as_uint(x))); }
};

// ---------------------------------------------------------------------
// Flat cast, groups of 8 elements.
// Workgroup b owns groups [b*kCastThreads*kCastUnroll, (b+1)*kCastThreads*kCastUnroll);
// within it, unroll step k covers one contiguous run of kCastThreads groups,
// so every load/store instruction of a wave touches one contiguous 2 KiB
// span.  Loads and stores are nontemporal 128-bit accesses.  With cached
// loads the cast's rate depended on the work before it, falling with the
// bytes that work had written; with nontemporal loads it does not (one
// Llama layer, 10 casts per case, two rounds on one box, fraction of HBM
// peak):
//                         cached loads   nontemporal loads
//   back to back          0.759-0.763    0.777-0.780
//   after 20 bf16 GEMMs   0.733-0.738    0.766-0.768
//   after 4 x 1 GiB copy  0.676-0.680    0.767-0.769
// The sc0/sc1 bits changed nothing beside nt; plain stores were slower.
// Other shapes, one box each: 2 groups per lane 6.16 TB/s (then with
// nontemporal loads 5.61), 4 groups 6.04, 8 groups 5.70; one group per
// lane, measured in the training step: 0.2172-0.2182 ms per layer alone
// against 0.2245-0.2253 with 2 groups.  Workgroup size, one group per lane,
// two rounds on one box: 64 lanes 0.214 ms, 128 lanes 0.2124-0.2131 (6.15
// TB/s, 0.77 of peak), 256 lanes 0.2144-0.2157, 512 0.216-0.217, 1024
// 0.221-0.222; a plain fp32 copy of the same bytes reaches 0.79 of peak.
// Loads with every lane's 16 bytes contiguous across the wave (then 8-byte
// stores, or 16-byte stores after a lane-pair exchange), a blockIdx order
// that gives each XCD one contiguous eighth, and persistent grid-stride
// loops were no faster.
// ---------------------------------------------------------------------
// The groups start at the 16-byte boundary at or before dst, `lead` elements
// before it, so that every store is one aligned access; the source is loaded
// as 128-bit accesses at the alignment that leaves it.  Only the first and the
// last group of the array can be partial, and go element by element in the
// same launch.  Before, an array with either side off a boundary went through
// a scalar kernel (12.6 M elements to fp16: 23.2 us), and one whose length is
// no multiple of 8 needed a second launch for its tail (4,099 elements: 1.8 +
// 1.4 us of kernels and 5.5 us of host time for the two, 3.1 for one).
template <typename Fmt>
__device__ __forceinline__ void cast_flat_body(const float* __restrict__ src, uint16_t* __restrict__ dst,
                                               uint32_t lead, uint64_t n) {
    // Highest issue priority among the waves of its SIMD: staged units are
    // cast while the backward's GEMMs run on the same CUs, and the cast's few
    // instructions per byte then issue without queueing behind MFMA waves
    // (in a training step: 0.2537 -> 0.2492 ms per Llama layer).
    __builtin_amdgcn_s_setprio(3);
    const uint64_t end = n + lead;
    const uint64_t tile0 = uint64_t(blockIdx.x) * (kCastThreads * kCastUnroll * kGroup);
    // from the boundary on: never dereferenced below `lead`
    src -= lead;
    dst -= lead;
    if (tile0 >= lead && tile0 + kCastThreads * kCastUnroll * kGroup <= end) {
        // Full tile (every workgroup but the first and last): all loads are
        // issued before the first conversion, with no per-lane predicate
        // between them.
        f32x4 a[kCastUnroll], b[kCastUnroll];
#pragma unroll
        for (int k = 0; k < kCastUnroll; ++k) {
            const f32x4_any* p = reinterpret_cast<const f32x4_any*>(src + tile0 + (k * kCastThreads + threadIdx.x) * kGroup);
            a[k] = __builtin_nontemporal_load(p);
            b[k] = __builtin_nontemporal_load(p + 1);
        }
#pragma unroll
        for (int k = 0; k < kCastUnroll; ++k) {
            __builtin_nontemporal_store(Fmt::cast8(a[k], b[k]),
                reinterpret_cast<u32x4*>(dst + tile0 + (k * kCastThreads + threadIdx.x) * kGroup));
        }
    } else {
        for (int k = 0; k < kCastUnroll; ++k) {
            const uint64_t e = tile0 + (k * kCastThreads + threadIdx.x) * kGroup;
            if (e >= lead && e + kGroup <= end) {
                const f32x4_any* p = reinterpret_cast<const f32x4_any*>(src + e);
                __builtin_nontemporal_store(Fmt::cast8(__builtin_nontemporal_load(p), __builtin_nontemporal_load(p + 1)),
                                            reinterpret_cast<u32x4*>(dst + e));
            } else {
                for (uint64_t j = e < lead ? lead : e; j < e + kGroup && j < end; ++j) dst[j] = Fmt::cast1(src[j]);
            }
        }
    }
}

// The staging cast to bf16 (the default unit dtype) and to fp16.
__global__ __launch_bounds__(kCastThreads) void cast_flat_kernel(
    const float* __restrict__ src, uint16_t* __restrict__ dst, uint32_t lead, uint64_t n) {
    cast_flat_body<ToBf16>(src, dst, lead, n);
}

__global__ __launch_bounds__(kCastThreads) void cast_flat_f16_kernel(
    const float* __restrict__ src, uint16_t* __restrict__ dst, uint32_t lead, uint64_t n) {
    cast_flat_body<ToF16>(src, dst, lead, n);
}

// Scalar cast for pointers that are not aligned to their own elements.
template <typename Fmt>
__global__ __launch_bounds__(kThreads) void cast_scalar_kernel(
    const float* __restrict__ src, uint16_t* __restrict__ dst, uint64_t n) {
    const uint64_t stride = uint64_t(gridDim.x) * kThreads;
    for (uint64_t i = uint64_t(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride) {
        dst[i] = Fmt::cast1(src[i]);
    }
}

__global__ __launch_bounds__(kThreads) void fill_b16_kernel(
    uint16_t* __restrict__ dst, uint64_t n, uint16_t value) {
    const uint32_t v2 = uint32_t(value) | (uint32_t(value) << 16);
    const u32x4 v = {v2, v2, v2, v2};
    const uint64_t n8 = n / kGroup;
    const uint64_t base = uint64_t(blockIdx.x) * (kThreads * kUnroll) + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
        const uint64_t g = base + uint64_t(k) * kThreads;
        if (g < n8) reinterpret_cast<u32x4*>(dst)[g] = v;
    }
    // tail (< 8 elements): the first lanes of the first workgroup
    if (blockIdx.x == 0 && threadIdx.x < (n - n8 * kGroup)) dst[n8 * kGroup + threadIdx.x] = value;
}

// ---------------------------------------------------------------------
// Segment-table kernels.  The table travels in the kernel arguments
// (about 2 KiB for SF_MAX_SEGS segments), so no device allocation is
// needed.  Each workgroup owns one tile of kTile elements inside a single
// segment: tiles are numbered across segments and tile_start[s] is the first
// tile of segment s.  A workgroup finds its segment with a binary search
// over tile_start, whose loads are uniform (scalar).
//
// Bound by HBM (or, with a destination in host memory, by the host link).
// Tiles and groups of 8 are laid out from the 16-byte boundary at or before
// the segment's destination, so every store but those of a segment's two
// ends is one aligned 128-bit access whatever the destination's alignment;
// the source is loaded as 128-bit accesses too, at whatever alignment that
// leaves it (the hardware takes any multiple of the element size; within 2 %
// of aligned ones).  Elements of the partial groups at the two ends go one
// by one.  Before, a segment with either side off a 16-byte boundary went
// element by element: 61 tensors of odd sizes, 218 M elements in all, 257 ->
// 132 us (copy, 6.1 TB/s) and 278 -> 205 us (cast); 8.4 M elements 14.9 ->
// 9.5 us and 22.1 -> 12.0; packed into host memory 592 -> 327 us.
//
// Shape, 218 M elements aligned | 2.4 M | 8.4 M ragged, us: cast 64 lanes x 1
// group per lane 207.9 | 5.4 | 12.3, 128 x 1 205.8 | 5.5 | 12.1, 256 x 1 211.0
// | 5.2 | 12.0, 256 x 2 216.0 | 5.5 | 12.7, 256 x 4 (the shape before) 215.0 |
// 6.2 | 14.1, 512 x 1 207.6 | 5.6 | 12.2; copy 256 x 1 144.1 | 4.2 | 9.5, 256
// x 4 142.5 | 4.6 | 10.2.  Small tiles: few elements still fill the chip.  A
// capped grid instead has few workgroups, each with kHostUnroll groups per
// lane in flight: one layer into host memory with 16 workgroups of 256 x 8
// 7802 us, 256 x 4 7926, 256 x 2 8062, 512 x 1 8145.  A capped unpack of host
// memory takes kReadUnroll, whose requests fill the link already and whose
// smaller tiles end together (us, 8 | 4 groups with 16 workgroups: 2 M elements
// 77.9 | 74.6, one layer 7705 | 7583; with 8, 2 M 82.8 | 75.7).
// ---------------------------------------------------------------------
struct SegTable {
    uint64_t src[SF_MAX_SEGS];
    uint64_t dst[SF_MAX_SEGS];
    uint64_t n[SF_MAX_SEGS];
    uint64_t tile_start[SF_MAX_SEGS + 1];
    uint32_t nsegs;
};

__device__ __forceinline__ uint32_t find_seg(const SegTable& t, uint64_t tile) {
    uint32_t lo = 0, hi = t.nsegs;  // tile_start[lo] <= tile < tile_start[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (t.tile_start[mid] <= tile) lo = mid; else hi = mid;
    }
    return lo;
}

// Element operations: fp32 -> bf16 cast, or 16-bit copy.  Raw is what a lane
// holds of a group between its loads and its store.
struct OpCast {
    using S = float;
    struct Raw {
        f32x4 a, b;
    };
    __device__ static Raw load(const S* p) {
        const f32x4_any* q = reinterpret_cast<const f32x4_any*>(p);
        return {__builtin_nontemporal_load(q), __builtin_nontemporal_load(q + 1)};
    }
    // a load that the caches may keep
    __device__ static Raw load_kept(const S* p) {
        const f32x4_any* q = reinterpret_cast<const f32x4_any*>(p);
        return {q[0], q[1]};
    }
    __device__ static u32x4 convert(const Raw& r) { return cast8(r.a, r.b); }
    __device__ static uint16_t convert1(S x) { return uint16_t(rne_bf16(__float_as_uint(x))); }
};

struct OpCopy16 {
    using S = uint16_t;
    using Raw = u32x4;
    __device__ static Raw load(const S* p) {
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
    }
    __device__ static Raw load_kept(const S* p) { return *reinterpret_cast<const u32x4_any*>(p); }
    __device__ static u32x4 convert(const Raw& r) { return r; }
    __device__ static uint16_t convert1(S x) { return x; }
};

// One group of 8 at element offset e (a multiple of 8 from the boundary the
// pointers start at) of a run occupying [lead, end): the whole group, or its
// elements inside the run one by one.
template <typename Op>
__device__ __forceinline__ void move_group(const typename Op::S* src, uint16_t* dst, int64_t e, int64_t lead,
                                           int64_t end) {
    if (e >= lead && e + kGroup <= end) {
        __builtin_nontemporal_store(Op::convert(Op::load(src + e)), reinterpret_cast<u32x4*>(dst + e));
    } else {
        for (int64_t j = e < lead ? lead : e; j < e + kGroup && j < end; ++j) dst[j] = Op::convert1(src[j]);
    }
}

constexpr int kSegUnroll = 1;   // groups per lane and tile: one workgroup per tile
constexpr int kHostUnroll = 8;  // the same for a capped grid
constexpr int kReadUnroll = 4;  // and for one that unpacks host memory
constexpr int kStageBlocks = 48;   // workgroups that read one array over the host link

template <typename Op, int kU>
__device__ __forceinline__ void store_tile(const typename Op::Raw (&v)[kU], uint16_t* out) {
#pragma unroll
    for (int k = 0; k < kU; ++k)
        __builtin_nontemporal_store(Op::convert(v[k]), reinterpret_cast<u32x4*>(out + (k * kThreads + threadIdx.x) * kGroup));
}

template <typename Op, int kU>
__global__ __launch_bounds__(kThreads) void seg_kernel(const SegTable t) {
    using S = typename Op::S;
    constexpr int64_t kTile = int64_t(kThreads) * kU * kGroup;
    const uint64_t ntiles = t.tile_start[t.nsegs];
    typename Op::Raw v[kU];       // the last whole tile read
    uint16_t* out = nullptr;      // and where it goes
    // Grid-stride over tiles: one workgroup per tile when the grid covers
    // them all, or a capped grid (e.g. a copy into host memory, which only
    // needs enough workgroups to keep the host link busy).
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint32_t s = find_seg(t, tile);
        const int64_t lead = lead_elems(t.dst[s]);
        const int64_t end = int64_t(t.n[s]) + lead;
        // from the boundary on: never dereferenced below `lead`
        const S* src = reinterpret_cast<const S*>(t.src[s] - uint64_t(lead) * sizeof(S));
        uint16_t* dst = reinterpret_cast<uint16_t*>(t.dst[s] - uint64_t(lead) * 2);
        const int64_t first = int64_t(tile - t.tile_start[s]) * kTile;
        if (((t.dst[s] & 1) | (t.src[s] & (sizeof(S) - 1))) != 0) {
            // not aligned to its own elements: byte-exact element accesses
            for (int64_t j = first + threadIdx.x; j < first + kTile && j < end; j += kThreads)
                if (j >= lead) dst[j] = Op::convert1(src[j]);
        } else if (first >= lead && first + kTile <= end) {
            // Whole tile: unpredicated loads, all in flight together.  With a
            // capped grid they are issued before the stores of the tile before
            // it, so that they don't wait for those to be acknowledged.
            typename Op::Raw next[kU];
#pragma unroll
            for (int k = 0; k < kU; ++k) next[k] = Op::load(src + first + (k * kThreads + threadIdx.x) * kGroup);
            if (kU > 1 && out != nullptr) store_tile<Op, kU>(v, out);
#pragma unroll
            for (int k = 0; k < kU; ++k) v[k] = next[k];
            out = dst + first;
            if (kU == 1) store_tile<Op, kU>(v, out);
        } else {
            for (int k = 0; k < kU; ++k)
                move_group<Op>(src, dst, first + (k * kThreads + threadIdx.x) * kGroup, lead, end);
        }
    }
    if (kU > 1 && out != nullptr) store_tile<Op, kU>(v, out);
}

// ---------------------------------------------------------------------
// Row gather: dst row t = src row ids[t] (rows of row_len elements), cast
// fp32 -> bf16 or copied as 16-bit values.  src may be pinned host memory
// (the row-sparse embedding load) and dst may be pinned host memory (the
// row-sparse gradient offload, then with a capped grid).  An id outside
// [0, nrows) yields a row of 0xFFFF (a NaN in bf16) and sets *bad.
//
// A row is per_row groups of 8 elements, laid out from the 16-byte boundary
// at or before its destination (kVec: every row starts on one and ends on
// one), and a workgroup's tile is kU groups per lane of the rows put end to
// end, so rows of any length fill its lanes.  All loads of a whole tile are
// issued before its first store, without a per-lane predicate: under one, the
// compiler waits for all outstanding memory operations before each store,
// and each store into host memory would wait for the previous one to be
// acknowledged over the link.  Bound by the link (about 57 GB/s; a DMA copy
// of 128 MB reaches 55-57) or, inside HBM, by HBM.  Before, a workgroup took
// one row at a time, so that short rows left it idle, and rows of a length
// that is no multiple of 8 went element by element.  us, before -> now, fp32
// rows from host memory: 4,096 rows of 4096 1250 -> 1125; 8,192 of 8192 4842
// -> 3730.  16-bit rows into host memory, 16 workgroups: 8,192 of 64 139 ->
// 26; 3,000 of 1003 224 -> 123; 4,096 of 4096 616 either way.
// ---------------------------------------------------------------------
struct RowShape {
    uint64_t row_len, nrows;
    uint64_t per_row;    // groups per row
    uint32_t recip;      // ceil(2^31 / per_row), read where per_row < a tile
};

// Group x of rows put end to end, x - (row0 * per_row) = loc + rem0 < per_row
// + kTile: its row past row0 and its place in that row.  A division by
// multiplication: exact for loc + rem0 < 2^12 and per_row < 2^12.
template <uint32_t kTile>
__device__ __forceinline__ void split_group(const RowShape& s, uint64_t rem0, uint32_t loc, uint32_t& row,
                                            uint64_t& j) {
    static_assert(kTile <= 2048, "split_group's product");
    if (s.per_row >= kTile) {
        const uint64_t x = rem0 + loc;
        row = x >= s.per_row ? 1u : 0u;
        j = row ? x - s.per_row : x;
    } else {
        const uint32_t x = uint32_t(rem0) + loc;
        row = __umulhi(2 * x, s.recip);
        j = x - row * uint32_t(s.per_row);
    }
}

// How rows lie: every one starts and ends on a 16-byte boundary of the
// destination (and the source is aligned so), rows of at least 8 elements
// that start anywhere, or what is left: shorter rows, and a source that is
// not aligned to its own elements.
enum RowMode { kWhole, kEdges, kElements };

// A tile between its loads and its stores (kWhole, kEdges).
template <typename Op, int kU, RowMode kMode>
struct Held {
    typename Op::Raw v[kU];
    uint16_t* out[kU];
    uint32_t part[kMode == kEdges ? kU : 1];   // bit d: element d of v goes to out + d
    bool ok[kU];
};

// Loads of a tile that starts at group rem0 of row row0; lanes past its group
// `last` load that one again.  row_of(i, t, id): destination row and id of
// row i.  kEdges: of a row's first and last group, which can be partial, the
// nearest 8 elements of the row are loaded.
template <typename Op, int kU, RowMode kMode, typename RowOf>
__device__ __forceinline__ void load_rows(Held<Op, kU, kMode>& h, const typename Op::S* src, uint16_t* dst,
                                          const RowShape& s, uint64_t row0, uint64_t rem0, uint32_t last,
                                          RowOf row_of) {
#pragma unroll
    for (int k = 0; k < kU; ++k) {
        const uint32_t loc = k * kThreads + threadIdx.x;
        uint32_t i;
        uint64_t j, t;
        int64_t id;
        split_group<kThreads * kU>(s, rem0, loc < last ? loc : last, i, j);
        row_of(row0 + i, t, id);
        h.ok[k] = id >= 0 && uint64_t(id) < s.nrows;
        uint16_t* row = dst + t * s.row_len;
        int64_t at = int64_t(j) * kGroup;
        if (kMode == kEdges) {
            const int64_t e = at - int64_t(lead_elems(reinterpret_cast<uint64_t>(row)));
            const int64_t n = int64_t(s.row_len);
            at = e < 0 ? 0 : (e + kGroup <= n ? e : n - kGroup);
            // the group is [e, e + 8) of the row, the 8 loaded elements [at, at + 8)
            const int64_t d = at - e;
            h.part[k] = d >= kGroup || d <= -kGroup ? 0u : d >= 0 ? 0xFFu >> d : (0xFFu << -d) & 0xFFu;
        }
        h.out[k] = row + at;
        h.v[k] = Op::load_kept(src + (h.ok[k] ? uint64_t(id) : 0) * s.row_len + at);
    }
}

// Its stores: of all groups (kAll) or of the first n.
template <typename Op, int kU, RowMode kMode, bool kAll>
__device__ __forceinline__ bool store_rows(const Held<Op, kU, kMode>& h, uint32_t n) {
    const u32x4 nan = {~0u, ~0u, ~0u, ~0u};
    bool any_bad = false;
#pragma unroll
    for (int k = 0; k < kU; ++k) {
        const u32x4 c = Op::convert(h.v[k]);
        const u32x4 o = h.ok[k] ? c : nan;
        any_bad |= !h.ok[k];
        if (!kAll && k * kThreads + threadIdx.x >= n) continue;
        if (kMode == kWhole || h.part[k] == 0xFFu) {
            __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(h.out[k]));
        } else {
#pragma unroll
            for (int d = 0; d < kGroup; ++d)
                if (h.part[k] >> d & 1) h.out[k][d] = uint16_t(o[d / 2] >> (d % 2 * 16));
        }
    }
    return any_bad;
}

// One tile of n groups (up to kThreads * kU) from group rem0 of row row0 on.
template <typename Op, int kU, RowMode kMode, typename RowOf>
__device__ __forceinline__ bool gather_tile(const typename Op::S* src, uint16_t* dst, const RowShape& s, uint64_t row0,
                                            uint64_t rem0, uint32_t n, RowOf row_of) {
    constexpr uint32_t kTile = kThreads * kU;
    bool any_bad = false;
    if (kMode != kElements) {
        Held<Op, kU, kMode> h;
        load_rows<Op, kU, kMode>(h, src, dst, s, row0, rem0, n - 1, row_of);
        return n == kTile ? store_rows<Op, kU, kMode, true>(h, n) : store_rows<Op, kU, kMode, false>(h, n);
    }
    for (uint32_t loc = threadIdx.x; loc < n; loc += kThreads) {
        uint32_t i;
        uint64_t j, t;
        int64_t id;
        split_group<kTile>(s, rem0, loc, i, j);
        row_of(row0 + i, t, id);
        const bool ok = id >= 0 && uint64_t(id) < s.nrows;
        any_bad |= !ok;
        const typename Op::S* from = src + (ok ? uint64_t(id) * s.row_len : 0);
        uint16_t* row = dst + t * s.row_len;
        for (uint64_t q = j * kGroup; q < (j + 1) * kGroup && q < s.row_len; ++q)
            row[q] = ok ? Op::convert1(from[q]) : uint16_t(0xFFFFu);
    }
    return any_bad;
}

// Rows of a table in HBM; short rows, or rows of fewer than 8 elements, of one
// in host memory.  A workgroup takes span groups, up to one per lane.
template <bool kCast> struct GatherOp { using T = OpCopy16; };
template <> struct GatherOp<true> { using T = OpCast; };

template <bool kCast, RowMode kMode>
__global__ __launch_bounds__(kThreads) void gather_rows_kernel(const void* __restrict__ src,
                                                               const int64_t* __restrict__ ids, uint64_t ntok,
                                                               RowShape s, uint32_t span, uint16_t* __restrict__ dst,
                                                               uint32_t* __restrict__ bad) {
    using Op = typename GatherOp<kCast>::T;
    const uint64_t total = ntok * s.per_row;
    bool any_bad = false;
    for (uint64_t b = blockIdx.x; b * span < total; b += gridDim.x) {
        const uint64_t tile0 = b * span, row0 = span == s.per_row ? b : tile0 / s.per_row;
        any_bad |= gather_tile<Op, 1, kMode>(static_cast<const typename Op::S*>(src), dst, s, row0,
                                             tile0 - row0 * s.per_row,
                                             uint32_t(total - tile0 < span ? total - tile0 : span),
                                             [&](uint64_t i, uint64_t& t, int64_t& id) { t = i; id = ids[i]; });
    }
    if (any_bad && bad != nullptr) bad[0] = 1u;
}

// Rows that cross the host link: of a table in pinned host memory, with at
// most kLinkBlocks workgroups, or into pinned host memory with the caller's
// cap; kU groups per lane in flight.  A few workgroups keep the link busy, and
// more requests at once only get into each other's way (us, 1 workgroup per
// tile | 128 | 64 | 32 | 16: 4,096 rows of 4096 fp32 1237 | 1198 | 1175 | 1171
// | 1210; 1,581 of 480 74 | 72.5 | 61.6 | 59.4 | 59.8).  The ids are taken
// from LDS, so that no second latency stands before the rows' own.  Host rows
// shorter than kLinkRow bytes go one per workgroup instead, as fast or faster
// (us, link | one per workgroup: 3,000 fp32 rows of 320 77.3 | 71.7, of 500
// 120.8 | 116.3, of 640 140.2 | 139.9, of 1000 221 | 225), unless they are at
// most kShortRow bytes and there are many (65,536 16-bit rows of 8 21 | 43, of 64
// 42 | 57, fp32 59 | 76, of 160 81 | 78).
//
// kOnce: a row that several tokens ask for crosses the link once.  The first
// token of each window of kWindow that asks for it gathers it, and
// repeat_gather_rows_kernel copies it to the others inside HBM.  Both find
// the first token by a hash table of the window's ids in LDS, which every
// workgroup makes for itself (some 5 us; no memory beside the operands).
//
// A cap decides where it leaves few workgroups: below kManyBlocks for a table in
// host memory, up to kLinkBlocks for rows into host memory (us, here |
// gather_rows_kernel: 20,000 16-bit rows of 1024 with 16 workgroups 762 | 846,
// with 64 795 | 757) and up to kFewBlocks inside HBM, for the loads in flight:
// a workgroup walks over all windows for its share of each, so many workgroups
// pay that walk for a few rows (at a cap of 4096: 1 M 16-bit rows of 64 1269 |
// 27, 200,000 of 1024 269 | 101, 65,536 of 4096 129 | 122).
constexpr uint32_t kLinkBlocks = 32;
constexpr uint64_t kFewBlocks = 256, kManyBlocks = 4096;
constexpr size_t kLinkRow = 2560, kShortRow = 256;
constexpr size_t kManyTokens = 8192;
constexpr uint32_t kWindow = 8192;
constexpr uint32_t kSlots = 2 * kWindow;   // of the hash table, at most half full
constexpr uint32_t kEmpty = ~0u;
// A table entry is id * kWindow + token, so that entries of one id are
// ordered by token.  nrows < kOnceRows leaves kNoRow free for ids outside the
// table and keeps every entry different from kEmpty.
constexpr uint64_t kOnceRows = (uint64_t(1) << 32) / kWindow - 1;
constexpr uint32_t kNoRow = uint32_t(kOnceRows);

__device__ __forceinline__ uint32_t first_slot(uint32_t id) { return id * 2654435761u >> (32 - 14); }
static_assert(kSlots == 1u << 14, "first_slot");

// slots[] = for every id of the window its first token.
__device__ __forceinline__ void index_window(uint32_t* slots, const int64_t* ids, uint32_t n, uint64_t nrows) {
    for (uint32_t i = threadIdx.x; i < kSlots; i += blockDim.x) slots[i] = kEmpty;
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < n; t += blockDim.x) {
        const int64_t id = ids[t];
        if (id < 0 || uint64_t(id) >= nrows) continue;
        const uint32_t entry = uint32_t(id) * kWindow + t;
        for (uint32_t h = first_slot(uint32_t(id));; h = (h + 1) % kSlots) {
            const uint32_t old = atomicCAS(&slots[h], kEmpty, entry);
            if (old == kEmpty) break;
            if (old / kWindow == uint32_t(id)) {
                atomicMin(&slots[h], entry);
                break;
            }
        }
    }
    __syncthreads();
}

// The first token of the window that asks for row id, which is in the table.
__device__ __forceinline__ uint32_t first_token(const uint32_t* slots, uint32_t id) {
    uint32_t h = first_slot(id);
    while (slots[h] / kWindow != id) h = (h + 1) % kSlots;
    return slots[h] % kWindow;
}

template <bool kCast, int kU, RowMode kMode, bool kOnce>
__global__ __launch_bounds__(kThreads) void link_gather_rows_kernel(const void* __restrict__ src,
                                                                    const int64_t* __restrict__ ids, uint64_t ntok,
                                                                    RowShape s, uint16_t* __restrict__ dst,
                                                                    uint32_t* __restrict__ bad) {
    using Op = typename GatherOp<kCast>::T;
    // this workgroup's tokens of the window: every gridDim.x-th
    constexpr uint32_t kMine = kOnce ? kWindow / kLinkBlocks : kWindow;
    __shared__ uint32_t slots[kOnce ? kSlots : 1];
    __shared__ uint32_t own[kMine];   // kOnce: entries of the tokens to gather; else ids, ~0 outside the table
    __shared__ uint32_t count;
    const auto* table = static_cast<const typename Op::S*>(src);
    const uint64_t tile_rows = kThreads * kU / s.per_row, tile_rem = kThreads * kU - tile_rows * s.per_row;
    bool any_bad = false;
    for (uint64_t w0 = 0; w0 < ntok; w0 += kWindow) {
        const uint32_t n = uint32_t(ntok - w0 < kWindow ? ntok - w0 : kWindow);
        const uint32_t mine = n > blockIdx.x ? (n - blockIdx.x + gridDim.x - 1) / gridDim.x : 0;
        if (kOnce) {
            if (threadIdx.x == 0) count = 0;
            index_window(slots, ids + w0, n, s.nrows);
        }
        for (uint32_t i = threadIdx.x; i < mine; i += kThreads) {
            const uint32_t t = blockIdx.x + i * gridDim.x;
            const int64_t id = ids[w0 + t];
            const bool ok = id >= 0 && uint64_t(id) < s.nrows;
            if (!kOnce) own[i] = ok ? uint32_t(id) : ~0u;
            else if (!ok || first_token(slots, uint32_t(id)) == t)
                own[atomicAdd(&count, 1u)] = (ok ? uint32_t(id) : kNoRow) * kWindow + t;
        }
        __syncthreads();
        const auto row_of = [&](uint64_t i, uint64_t& t, int64_t& id) {
            const uint32_t e = own[i];
            t = w0 + (kOnce ? e % kWindow : blockIdx.x + uint32_t(i) * gridDim.x);
            id = kOnce ? e / kWindow : e;   // past the last row for one outside the table
        };
        constexpr uint32_t kTile = kThreads * kU;
        uint64_t left = uint64_t(kOnce ? count : mine) * s.per_row, row0 = 0, rem0 = 0;
        if (left > 0) {
            // A tile's loads are issued before the stores of the one before it,
            // so that they don't wait for those to be acknowledged.
            Held<Op, kU, kMode> h;
            uint32_t n = uint32_t(left < kTile ? left : kTile);
            load_rows<Op, kU, kMode>(h, table, dst, s, row0, rem0, n - 1, row_of);
            while (left > kTile) {
                left -= kTile;
                row0 += tile_rows;
                rem0 += tile_rem;
                if (rem0 >= s.per_row) {
                    rem0 -= s.per_row;
                    ++row0;
                }
                n = uint32_t(left < kTile ? left : kTile);
                Held<Op, kU, kMode> next;
                load_rows<Op, kU, kMode>(next, table, dst, s, row0, rem0, n - 1, row_of);
                any_bad |= store_rows<Op, kU, kMode, true>(h, kTile);
                h = next;
            }
            any_bad |= n == kTile ? store_rows<Op, kU, kMode, true>(h, n) : store_rows<Op, kU, kMode, false>(h, n);
        }
        __syncthreads();   // before the next window's ids
    }
    if (any_bad && bad != nullptr) bad[0] = 1u;
}

// The rows that link_gather_rows_kernel<kOnce> left out, from the row it
// gathered: one wave per token.
constexpr int kRepeatThreads = 1024;
constexpr uint32_t kRepeatBlocks = 256;
__global__ __launch_bounds__(kRepeatThreads) void repeat_gather_rows_kernel(const int64_t* __restrict__ ids,
                                                                            uint64_t ntok, RowShape s, uint16_t* dst) {
    __shared__ uint32_t slots[kSlots];
    for (uint64_t w0 = 0; w0 < ntok; w0 += kWindow) {
        const uint32_t n = uint32_t(ntok - w0 < kWindow ? ntok - w0 : kWindow);
        index_window(slots, ids + w0, n, s.nrows);
        for (uint32_t t = blockIdx.x * (kRepeatThreads / 64) + (threadIdx.x >> 6); t < n;
             t += gridDim.x * (kRepeatThreads / 64)) {
            const int64_t id = ids[w0 + t];
            if (id < 0 || uint64_t(id) >= s.nrows) continue;
            const uint32_t f = first_token(slots, uint32_t(id));
            if (f == t) continue;
            const uint16_t* from = dst + (w0 + f) * s.row_len;
            uint16_t* row = dst + (w0 + t) * s.row_len;
            const int64_t lead = lead_elems(reinterpret_cast<uint64_t>(row));
            for (uint64_t j = threadIdx.x & 63; j < s.per_row; j += 64)
                move_group<OpCopy16>(from - lead, row - lead, int64_t(j) * kGroup, lead, int64_t(s.row_len) + lead);
        }
        __syncthreads();   // before the next window's table
    }
}

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Upper bound on workgroups per launch; the grids below stay far under the
// 2^32-1 lanes per dimension that the dispatch packet allows.
constexpr uint64_t kMaxBlocks = (uint64_t(1) << 31) / kThreads;

template <typename Op>
int launch_segs(const sf_seg* segs, int nsegs, int max_workgroups, hipStream_t stream, int host_unroll = kHostUnroll) {
    if (nsegs < 0 || (nsegs > 0 && segs == nullptr)) return SF_EINVAL;
    const bool capped = max_workgroups > 0;
    const int unroll = capped ? host_unroll : kSegUnroll;
    const auto kernel = unroll == kHostUnroll ? seg_kernel<Op, kHostUnroll>
                        : unroll == kReadUnroll ? seg_kernel<Op, kReadUnroll>
                                                : seg_kernel<Op, kSegUnroll>;
    const uint64_t tile_elems = uint64_t(kThreads) * kGroup * uint64_t(unroll);
    // Tables longer than SF_MAX_SEGS are split into several launches.
    for (int base = 0; base < nsegs; base += SF_MAX_SEGS) {
        const int cnt = (nsegs - base < SF_MAX_SEGS) ? (nsegs - base) : SF_MAX_SEGS;
        SegTable t;
        memset(&t, 0, sizeof(t));
        uint64_t tiles = 0, size_units = 0;
        uint32_t m = 0;
        for (int i = 0; i < cnt; ++i) {
            const sf_seg& g = segs[base + i];
            if (g.n == 0) continue;
            if (g.src == 0 || g.dst == 0) return SF_EINVAL;
            size_units += ceil_div(g.n, kSizeUnit);
            t.src[m] = g.src;
            t.dst[m] = g.dst;
            t.n[m] = g.n;
            t.tile_start[m] = tiles;
            tiles += ceil_div(g.n + lead_elems(g.dst), tile_elems);
            ++m;
        }
        if (m == 0) continue;
        t.tile_start[m] = tiles;
        t.nsegs = m;
        if (size_units > kMaxBlocks) return SF_EINVAL;  // > 68e9 elements: not a real layer
        uint64_t grid = tiles < kMaxBlocks ? tiles : kMaxBlocks;
        if (capped && grid > uint64_t(max_workgroups)) grid = uint64_t(max_workgroups);
        hipLaunchKernelGGL(kernel, dim3(uint32_t(grid)), dim3(kThreads), 0, stream, t);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return int(e);
    }
    return SF_OK;
}

}  // namespace

namespace {
// Status of a failed runtime call, handed to the caller.  The runtime also
// keeps it as the thread's last error, where the next library that checks
// for errors (torch after its own calls) would report it as its own: clear it.
inline int hip_status(hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    return int(e);
}
}  // namespace

namespace {
// The memory type the runtime records for ptr, or -1 for memory it does
// not know (pageable host memory).
int pointer_attributes(const void* p, hipPointerAttribute_t* a) {
    const hipError_t e = hipPointerGetAttributes(a, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return -1;
    }
    return int(a->type);
}

int memory_type(const void* p) {
    hipPointerAttribute_t a;
    return pointer_attributes(p, &a);
}

// Bytes that a gather over the host link would read again for ids it has met
// before, were the ids drawn uniformly (those of text repeat more often).  A
// table that fits the L2s crosses the link at most once for each of the 8.
inline double repeated_bytes(size_t ntok, size_t nrows, size_t row_bytes) {
    const double n = double(ntok < kWindow ? ntok : kWindow), v = double(nrows);
    const double met = v * -expm1(-n / v) * (double(ntok) / n);
    const double read = double(ntok) < 8.0 * v ? double(ntok) : 8.0 * v;
    return (read - met) * double(row_bytes);
}

// Reading rows once pays from here on: 2 MiB are 37 us on the link; a window's
// hash tables and the second kernel cost 5 (1,024 tokens) to 25 us (8,192), so
// every full window has to save that much.  65,536 tokens of 30,000 16-bit rows
// of 160, 2.7 MB to save in 8 windows, 393 -> 499 us; 16,384 of 1,000 fp32 rows
// of 160, 3.8 MB in 2, 88 -> 57.  fp32
// rows of 4096: 4,096 tokens of 32,000 rows 1168 -> 1125 us, of 2,000 rows
// 1076 -> 533; 1,024 of 32,000 rows, 0.3 MiB to save, 298 -> 306.  8,192
// tokens of 256 rows of 1024 160 -> 45 us, of 256 rows of 64, 0.4 MiB, 15 -> 24.
constexpr double kOnceBytes = 2 << 20, kOnceWindowBytes = 3 << 19;

template <bool kCast, RowMode kMode>
int launch_gather(const void* src, const int64_t* ids, uint64_t ntok, const RowShape& s, uint16_t* dst, uint32_t* bad,
                  uint64_t cap, bool from_host, bool link, bool once, hipStream_t st) {
    if constexpr (kMode != kElements) {
        if (link) {
            constexpr int kU = kCast ? 4 : 8;   // 128 bytes per lane in flight
            hipLaunchKernelGGL((once ? link_gather_rows_kernel<kCast, kU, kMode, true>
                                     : link_gather_rows_kernel<kCast, kU, kMode, false>),
                               dim3(uint32_t(ntok < cap ? ntok : cap)), dim3(kThreads), 0, st, src, ids, ntok, s, dst,
                               bad);
            if (once) {
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return hip_status(e);
                hipLaunchKernelGGL(repeat_gather_rows_kernel, dim3(kRepeatBlocks), dim3(kRepeatThreads), 0, st, ids,
                                   ntok, s, dst);
            }
            return hip_status(hipGetLastError());
        }
    }
    const uint32_t span = from_host && s.per_row < uint64_t(kThreads) ? uint32_t(s.per_row) : uint32_t(kThreads);
    const uint64_t tiles = ceil_div(ntok * s.per_row, span);
    hipLaunchKernelGGL((gather_rows_kernel<kCast, kMode>), dim3(uint32_t(tiles < cap ? tiles : cap)), dim3(kThreads), 0,
                       st, src, ids, ntok, s, span, dst, bad);
    return hip_status(hipGetLastError());
}

template <bool kCast>
int launch_gather_rows(const void* src, const int64_t* ids, size_t ntok, size_t row_len, size_t nrows,
                       uint16_t* dst, uint32_t* bad, int max_workgroups, hipStream_t st, size_t src_elem) {
    if (ntok == 0 || row_len == 0) return SF_OK;
    if (src == nullptr || ids == nullptr || dst == nullptr) return SF_EINVAL;
    if ((reinterpret_cast<uintptr_t>(dst) & 1) != 0) return SF_EINVAL;
    // the destination rows must not overlap the source table
    const uintptr_t s0 = reinterpret_cast<uintptr_t>(src), d0 = reinterpret_cast<uintptr_t>(dst);
    if (s0 < d0 + 2 * ntok * row_len && d0 < s0 + src_elem * nrows * row_len) return SF_EOVERLAP;
    const RowMode mode = nrows == 0 || row_len < size_t(kGroup) || (s0 & (src_elem - 1)) != 0 ? kElements
                         : row_len % kGroup == 0 && ((s0 | d0) & 15) == 0                     ? kWhole
                                                                                              : kEdges;
    RowShape s;
    s.row_len = row_len;
    s.nrows = nrows;
    s.per_row = mode == kEdges ? (uint64_t(row_len) + 2 * kGroup - 2) / kGroup : ceil_div(row_len, kGroup);
    s.recip = uint32_t(ceil_div(uint64_t(1) << 31, s.per_row));
    uint64_t cap = max_workgroups > 0 && uint64_t(max_workgroups) < kMaxBlocks ? uint64_t(max_workgroups) : kMaxBlocks;
    const bool from_host = memory_type(src) == int(hipMemoryTypeHost);
    const size_t row_bytes = row_len * src_elem;
    const bool once = from_host && mode != kElements && cap > kLinkBlocks && ntok >= kLinkBlocks &&
                      nrows < kOnceRows &&
                      repeated_bytes(ntok, nrows, row_bytes) >=
                          fmax(kOnceBytes, kOnceWindowBytes * double(ntok / kWindow)) &&
                      memory_type(dst) == int(hipMemoryTypeDevice);
    const bool few = from_host ? cap < kManyBlocks || row_bytes >= kLinkRow ||
                                     (row_bytes <= kShortRow && ntok >= kManyTokens)
                               : cap <= kLinkBlocks ||
                                     (cap <= kFewBlocks && memory_type(dst) == int(hipMemoryTypeDevice));
    const bool link = (once || few) && nrows < (uint64_t(1) << 31);
    if (link && from_host && cap > kLinkBlocks) cap = kLinkBlocks;
    switch (mode) {
        case kWhole: return launch_gather<kCast, kWhole>(src, ids, ntok, s, dst, bad, cap, from_host, link, once, st);
        case kEdges: return launch_gather<kCast, kEdges>(src, ids, ntok, s, dst, bad, cap, from_host, link, once, st);
        default: return launch_gather<kCast, kElements>(src, ids, ntok, s, dst, bad, cap, from_host, link, once, st);
    }
}
}  // namespace

extern "C" {

const char* sf_error_string(int status) {
    switch (status) {
        case SF_OK: return "success";
        case SF_EINVAL: return "sf: invalid argument (null pointer, bad size or enum)";
        case SF_ETOOMANY: return "sf: too many segments for one call";
        case SF_EDTYPE: return "sf: dtype combination not supported";
        case SF_ENOOPT: return "sf: unknown optimizer id";
        case SF_EOVERLAP: return "sf: source and destination overlap";
        case SF_EALIGN: return "sf: array not aligned as the entry point requires";
        case SF_ETOOBIG: return "sf: piece larger than the library's device scratch (SF_STAGE_SCRATCH_ELEMS)";
        case SF_ETIMEDOUT: return "sf: wait ended at its deadline with work still pending";
        default:
            if (status >= SF_EDMA_BASE && status < SF_EDMA_BASE + 0x1000) return "sf: ROCr DMA call failed";
            return hipGetErrorString(hipError_t(status));
    }
}

int sf_abi_version(void) { return SF_ABI_VERSION; }

}  // extern "C"

namespace {

// The flat cast's launch.  ``start`` / ``stop`` (may be null) are stamped by
// the runtime around the launch's own dispatch, so they time the kernel alone,
// not what the stream waited for before it.
int cast_launch(const float* src, uint16_t* dst, size_t n, hipStream_t st, hipEvent_t start, hipEvent_t stop,
                bool to_f16 = false) {
    if (n == 0) {
        // nothing to launch: the events still mark the (empty) interval
        if (start != nullptr) {
            const hipError_t e = hipEventRecord(start, st);
            if (e != hipSuccess) return hip_status(e);
        }
        if (stop != nullptr) {
            const hipError_t e = hipEventRecord(stop, st);
            if (e != hipSuccess) return hip_status(e);
        }
        return SF_OK;
    }
    if (src == nullptr || dst == nullptr) return SF_EINVAL;
    const uintptr_t s = reinterpret_cast<uintptr_t>(src), d = reinterpret_cast<uintptr_t>(dst);
    // fp32 source [s, s+4n) and bf16 destination [d, d+2n) must not overlap:
    // workgroups run in no particular order.
    if (s < d + 2 * n && d < s + 4 * n) return SF_EOVERLAP;
    const uint32_t lead = lead_elems(d);
    const uint64_t blocks = ceil_div(n + lead, uint64_t(kCastThreads) * kCastUnroll * kGroup);
    // > 8.6e9 elements: not a real unit; the limit counts whole groups, so up to
    // 7 elements more need one workgroup more
    if (((s | d) & 15) == 0 && ceil_div(n / kGroup, uint64_t(kCastThreads) * kCastUnroll) > kMaxBlocks) return SF_EINVAL;
    if ((s & 3) == 0 && (d & 1) == 0 && blocks <= kMaxBlocks + 1) {
        hipExtLaunchKernelGGL(to_f16 ? cast_flat_f16_kernel : cast_flat_kernel, dim3(uint32_t(blocks)),
                              dim3(kCastThreads), 0, st, start, stop, 0, src, dst, lead, uint64_t(n));
    } else {
        const uint64_t grid = ceil_div(n, kThreads);
        hipExtLaunchKernelGGL(to_f16 ? cast_scalar_kernel<ToF16> : cast_scalar_kernel<ToBf16>,
                              dim3(uint32_t(grid > 65536 ? 65536 : grid)), dim3(kThreads), 0, st, start, stop, 0, src, dst, uint64_t(n));
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SF_OK : int(e);
}

}  // namespace

extern "C" {

int sf_cast_f32_bf16(const float* src, uint16_t* dst, size_t n, sf_stream_t stream) {
    return cast_launch(src, dst, n, reinterpret_cast<hipStream_t>(stream), nullptr, nullptr);
}

int sf_cast_f32_bf16_timed(const float* src, uint16_t* dst, size_t n, sf_stream_t stream, sf_event_t start,
                           sf_event_t stop) {
    if ((start == nullptr) != (stop == nullptr)) return SF_EINVAL;
    return cast_launch(src, dst, n, reinterpret_cast<hipStream_t>(stream), reinterpret_cast<hipEvent_t>(start),
                       reinterpret_cast<hipEvent_t>(stop));
}

int sf_cast_f32_f16(const float* src, uint16_t* dst, size_t n, sf_stream_t stream) {
    return cast_launch(src, dst, n, reinterpret_cast<hipStream_t>(stream), nullptr, nullptr, true);
}

int sf_cast_f32_f16_timed(const float* src, uint16_t* dst, size_t n, sf_stream_t stream, sf_event_t start,
                          sf_event_t stop) {
    if ((start == nullptr) != (stop == nullptr)) return SF_EINVAL;
    return cast_launch(src, dst, n, reinterpret_cast<hipStream_t>(stream), reinterpret_cast<hipEvent_t>(start),
                       reinterpret_cast<hipEvent_t>(stop), true);
}

int sf_event_create(sf_event_t* ev) {
    if (ev == nullptr) return SF_EINVAL;
    hipEvent_t e = nullptr;
    const int rc = hip_status(hipEventCreate(&e));
    *ev = rc == SF_OK ? reinterpret_cast<sf_event_t>(e) : nullptr;
    return rc;
}

int sf_event_destroy(sf_event_t ev) {
    if (ev == nullptr) return SF_OK;
    return hip_status(hipEventDestroy(reinterpret_cast<hipEvent_t>(ev)));
}

int sf_event_elapsed_ms(sf_event_t start, sf_event_t stop, float* ms) {
    if (start == nullptr || stop == nullptr || ms == nullptr) return SF_EINVAL;
    return hip_status(hipEventElapsedTime(ms, reinterpret_cast<hipEvent_t>(start), reinterpret_cast<hipEvent_t>(stop)));
}

int sf_cast_scatter_f32_bf16(const sf_seg* segs, int nsegs, sf_stream_t stream) {
    return launch_segs<OpCast>(segs, nsegs, 0, reinterpret_cast<hipStream_t>(stream));
}

int sf_copy_segs_b16(const sf_seg* segs, int nsegs, int max_workgroups, sf_stream_t stream) {
    return launch_segs<OpCopy16>(segs, nsegs, max_workgroups, reinterpret_cast<hipStream_t>(stream));
}

int sf_pack_b16(const sf_seg* segs, int nsegs, uint16_t* dst, int max_workgroups, sf_stream_t stream) {
    if (nsegs < 0 || (nsegs > 0 && (segs == nullptr || dst == nullptr))) return SF_EINVAL;
    sf_seg local[SF_MAX_SEGS];
    uint64_t off = 0;
    for (int base = 0; base < nsegs; base += SF_MAX_SEGS) {
        const int cnt = (nsegs - base < SF_MAX_SEGS) ? (nsegs - base) : SF_MAX_SEGS;
        for (int i = 0; i < cnt; ++i) {
            local[i].src = segs[base + i].src;
            local[i].dst = reinterpret_cast<uint64_t>(dst + off);
            local[i].n = segs[base + i].n;
            off += segs[base + i].n;
        }
        int rc = launch_segs<OpCopy16>(local, cnt, max_workgroups, reinterpret_cast<hipStream_t>(stream));
        if (rc != SF_OK) return rc;
    }
    return SF_OK;
}

int sf_unpack_b16(const uint16_t* src, const sf_seg* segs, int nsegs, int max_workgroups,
                  sf_stream_t stream) {
    if (nsegs < 0 || (nsegs > 0 && (segs == nullptr || src == nullptr))) return SF_EINVAL;
    const int unroll = max_workgroups > 0 && memory_type(src) == int(hipMemoryTypeHost) ? kReadUnroll : kHostUnroll;
    sf_seg local[SF_MAX_SEGS];
    uint64_t off = 0;
    for (int base = 0; base < nsegs; base += SF_MAX_SEGS) {
        const int cnt = (nsegs - base < SF_MAX_SEGS) ? (nsegs - base) : SF_MAX_SEGS;
        for (int i = 0; i < cnt; ++i) {
            local[i].src = reinterpret_cast<uint64_t>(src + off);
            local[i].dst = segs[base + i].dst;
            local[i].n = segs[base + i].n;
            off += segs[base + i].n;
        }
        int rc = launch_segs<OpCopy16>(local, cnt, max_workgroups, reinterpret_cast<hipStream_t>(stream), unroll);
        if (rc != SF_OK) return rc;
    }
    return SF_OK;
}

int sf_gather_rows_f32_bf16(const float* src, const int64_t* ids, size_t ntok, size_t row_len, size_t nrows,
                            uint16_t* dst, uint32_t* bad, int max_workgroups, sf_stream_t stream) {
    return launch_gather_rows<true>(src, ids, ntok, row_len, nrows, dst, bad, max_workgroups,
                                    reinterpret_cast<hipStream_t>(stream), 4);
}

int sf_gather_rows_b16(const uint16_t* src, const int64_t* ids, size_t ntok, size_t row_len, size_t nrows,
                       uint16_t* dst, uint32_t* bad, int max_workgroups, sf_stream_t stream) {
    return launch_gather_rows<false>(src, ids, ntok, row_len, nrows, dst, bad, max_workgroups,
                                     reinterpret_cast<hipStream_t>(stream), 2);
}

int sf_fill_b16(uint16_t* dst, size_t n, uint16_t value, sf_stream_t stream) {
    if (n == 0) return SF_OK;
    if (dst == nullptr) return SF_EINVAL;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if ((reinterpret_cast<uintptr_t>(dst) & 1) != 0) return SF_EINVAL;  // not 16-bit aligned
    if ((reinterpret_cast<uintptr_t>(dst) & 15) != 0) {
        // Fill the head up to the next 16-byte boundary (< 8 elements) with a
        // one-workgroup launch whose vector part is empty, then the rest.
        const uint64_t head = (16 - (reinterpret_cast<uintptr_t>(dst) & 15)) / 2;
        const uint64_t h = head < n ? head : n;
        hipLaunchKernelGGL(fill_b16_kernel, dim3(1), dim3(kThreads), 0, st, dst, h, value);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return int(e);
        dst += h;
        n -= h;
        if (n == 0) return SF_OK;
    }
    const uint64_t n8 = n / kGroup;
    uint64_t blocks = ceil_div(n8 > 0 ? n8 : 1, uint64_t(kThreads) * kUnroll);
    if (blocks > kMaxBlocks) return SF_EINVAL;
    hipLaunchKernelGGL(fill_b16_kernel, dim3(uint32_t(blocks)), dim3(kThreads), 0, st, dst, n, value);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? SF_OK : int(e);
}

}  // extern "C"

// ---------------------------------------------------------------------
// Staging: pinned fp32 host array -> bf16 device array.
//
// Up to kStageDirect elements the segment cast reads the host array over the
// link: one kernel, which the link bounds.  With kStageBlocks workgroups of
// kHostUnroll groups per lane it reads as fast as a DMA copy, starts sooner and
// leaves no cast to follow: 147,712 elements 30.1 -> 14.3 us, 600,000 61 -> 48,
// 8 M 587 -> 572.  One workgroup per tile reads 2 M elements in 181 us, 64 of 4
// groups per lane in 146, 16 to 96 of 8 in 146 to 153.
//
// Larger arrays go piece by piece through a device fp32 buffer, all on one
// stream: each piece is copied into the buffer by DMA and cast from it by the
// flat cast; the next piece's copy into the same buffer follows that cast in
// stream order.  There the kernel's head start is 2 % and less, and it holds
// its compute units for the whole transfer, which a caller wants beside other
// work: 12 x 32 M elements beside 40 products of 8192^3 ended after 40.4 ms
// (products 36.0 of 34.7 alone) by DMA and after 45.2 by the kernel (45.2, the
// staging 31).  Pieces under kStagePiece elements leave the kernel the faster
// way at any size: each ends with a cast that nothing runs beside (6 M elements
// in pieces of 2 M 480 us, by the kernel 426).
// ---------------------------------------------------------------------
namespace {

constexpr size_t kStageDirect = size_t(4) << 20;
constexpr size_t kStagePiece = size_t(4) << 20;

// Whether n elements are read by one kernel, with pieces of `chunk` otherwise.
inline bool stage_direct(size_t n, size_t chunk) { return n <= kStageDirect || chunk < kStagePiece; }

int stage_launch(const float* host, uint16_t* dst, size_t n, float* buf, size_t chunk, hipStream_t st) {
    if (n == 0) return SF_OK;
    hipPointerAttribute_t a;
    // pinned host memory, which a kernel and an asynchronous copy can read; the cast writes device memory
    if (pointer_attributes(host, &a) != int(hipMemoryTypeHost) || memory_type(dst) != int(hipMemoryTypeDevice))
        return SF_EINVAL;
    if (stage_direct(n, chunk)) {
        // Whether the runtime reports the addresses of the pointer or of its
        // allocation is not documented: the two belong together either way.
        const ptrdiff_t inside = reinterpret_cast<const char*>(host) - static_cast<const char*>(a.hostPointer);
        const sf_seg seg = {reinterpret_cast<uint64_t>(a.devicePointer) + uint64_t(inside),
                            reinterpret_cast<uint64_t>(dst), n};
        return launch_segs<OpCast>(&seg, 1, kStageBlocks, st);
    }
    chunk -= chunk % kGroup;  // every piece starts 16-byte aligned in dst if dst does
    for (size_t off = 0; off < n; off += chunk) {
        const size_t c = n - off < chunk ? n - off : chunk;
        const hipError_t e = hipMemcpyAsync(buf, host + off, c * sizeof(float), hipMemcpyHostToDevice, st);
        if (e != hipSuccess) return hip_status(e);
        const int rc = cast_launch(buf, dst + off, c, st, nullptr, nullptr);
        if (rc != SF_OK) return rc;
    }
    return SF_OK;
}

}  // namespace

extern "C" {

int sf_stage_f32_bf16(const float* host_src, uint16_t* dst, size_t n, float* workspace, size_t workspace_elems,
                      sf_stream_t stream) {
    if (n == 0) return SF_OK;
    if (host_src == nullptr || dst == nullptr || workspace == nullptr || workspace_elems < size_t(kGroup) ||
        memory_type(workspace) != int(hipMemoryTypeDevice))
        return SF_EINVAL;
    return stage_launch(host_src, dst, n, workspace, workspace_elems, reinterpret_cast<hipStream_t>(stream));
}

}  // extern "C"

// ---------------------------------------------------------------------
// Staging without allocating: the pieces go through the library's own
// device buffer instead of a caller workspace.  `scratch` is a static
// device array, so every device the library's code object is loaded on
// holds one for the life of the process.  In host code its name is not a
// device address: the address comes from hipGetSymbolAddress, looked up
// once per device with that device current, and only that address is
// passed to the copies and the cast.
// ---------------------------------------------------------------------
namespace {

__device__ __align__(256) float scratch[SF_STAGE_SCRATCH_ELEMS];

constexpr int kMaxDevices = 64;
// Per device: the address of `scratch`, and an event recorded after the last
// cast of the previous call (the next call's stream waits on it).  The
// mutex is held from the wait to the record, so the calls of several host
// threads are ordered one after the other.
struct ScratchState {
    float* ptr = nullptr;
    hipEvent_t last = nullptr;
    bool recorded = false;
};
std::mutex g_scratch_mu;
ScratchState g_scratch[kMaxDevices];

// The current device, which must be the device of `st` (the null stream:
// the current device).
int device_for_stream(hipStream_t st, int* dev) {
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return hip_status(e);
    if (st != nullptr) {
        hipDevice_t sd = 0;
        e = hipStreamGetDevice(st, &sd);
        if (e != hipSuccess) return hip_status(e);
        if (int(sd) != cur) return SF_EINVAL;
    }
    *dev = cur;
    return SF_OK;
}

// The device's scratch state, set up on its first use; g_scratch_mu is held.
int scratch_state(int dev, ScratchState** out) {
    if (dev < 0 || dev >= kMaxDevices) return SF_EINVAL;
    ScratchState& s = g_scratch[dev];
    if (s.ptr == nullptr) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_status(e);
        if (p == nullptr) return SF_EINVAL;
        if (s.last == nullptr) {
            e = hipEventCreateWithFlags(&s.last, hipEventDisableTiming);
            if (e != hipSuccess) return hip_status(e);
        }
        s.ptr = static_cast<float*>(p);
    }
    *out = &s;
    return SF_OK;
}

}  // namespace

extern "C" {

int sf_stage_f32_bf16_noalloc(const float* host_src, uint16_t* dst, size_t n, size_t chunk_elems,
                              sf_stream_t stream) {
    if (chunk_elems > SF_STAGE_SCRATCH_ELEMS) return SF_ETOOBIG;
    if (n == 0) return SF_OK;
    if (host_src == nullptr || dst == nullptr || (chunk_elems != 0 && chunk_elems < size_t(kGroup))) return SF_EINVAL;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int dev = 0;
    int rc = device_for_stream(st, &dev);
    if (rc != SF_OK) return rc;
    const size_t chunk = chunk_elems == 0 ? SF_STAGE_SCRATCH_ELEMS : chunk_elems;
    if (stage_direct(n, chunk)) return stage_launch(host_src, dst, n, nullptr, chunk, st);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    ScratchState* s = nullptr;
    rc = scratch_state(dev, &s);
    if (rc != SF_OK) return rc;
    if (s->recorded) {
        const hipError_t e = hipStreamWaitEvent(st, s->last, 0);
        if (e != hipSuccess) return hip_status(e);
    }
    rc = stage_launch(host_src, dst, n, s->ptr, chunk, st);
    // Recorded also after a failed launch: whatever was enqueued before the
    // failure still uses the scratch buffer and must precede the next call.
    const hipError_t e = hipEventRecord(s->last, st);
    if (e == hipSuccess) s->recorded = true;
    if (rc != SF_OK) return rc;
    return hip_status(e);
}

int sf_memcpy_async(void* dst, const void* src, size_t bytes, int kind, sf_stream_t stream) {
    if (bytes == 0) return SF_OK;
    if (dst == nullptr || src == nullptr) return SF_EINVAL;
    hipMemcpyKind k;
    switch (kind) {
        case SF_COPY_H2D: k = hipMemcpyHostToDevice; break;
        case SF_COPY_D2H: k = hipMemcpyDeviceToHost; break;
        case SF_COPY_D2D: k = hipMemcpyDeviceToDevice; break;
        default: return SF_EINVAL;
    }
    return hip_status(hipMemcpyAsync(dst, src, bytes, k, reinterpret_cast<hipStream_t>(stream)));
}

int sf_host_alloc(void** out, size_t bytes) {
    if (out == nullptr) return SF_EINVAL;
    *out = nullptr;
    if (bytes == 0) return SF_OK;
    return hip_status(hipHostMalloc(out, bytes, hipHostMallocDefault));
}

int sf_host_free(void* ptr) {
    if (ptr == nullptr) return SF_OK;
    return hip_status(hipHostFree(ptr));
}

int sf_host_device_pointer(void* host_ptr, void** device_ptr) {
    if (host_ptr == nullptr || device_ptr == nullptr) return SF_EINVAL;
    *device_ptr = nullptr;
    return hip_status(hipHostGetDevicePointer(device_ptr, host_ptr, 0));
}

// ---------------------------------------------------------------------
// SDMA copies device -> pinned host, issued through the ROCr runtime.
//
// hipMemcpyAsync performs device-to-host copies with a shader blit kernel;
// a kernel writing over PCIe slows every HBM-bound kernel running beside it
// (the staging cast takes 5-10x longer), wherever its waves are placed.  An
// SDMA engine moves the same bytes at the same link rate without touching
// the shader memory path.  These copies are not ordered with HIP streams:
// the caller makes sure the source is complete (an event synchronised on the
// host) before sf_dma_copy and reads the destination only after sf_dma_wait.
// ---------------------------------------------------------------------
namespace {
struct DmaAgents {
    hsa_agent_t gpu{0};
    hsa_agent_t cpu{0};
    int device = -1;
    bool ok = false;
    uint32_t engine_mask = 0;  // one SDMA engine bit; 0: runtime's choice
    uint64_t ts_freq = 0;      // HSA system timestamp ticks per second
    int avoid_held = 0;        // route around engines another client holds:
                               // 0 no (default), 1 onto free engines 0-3,
                               // 2 also 4 and up
    // Copies issued here and not yet released by sf_dma_wait: signal handle
    // -> engine bit (0 for a runtime-chosen engine).
    std::unordered_map<uint64_t, uint32_t> outstanding;
};
DmaAgents g_dma;
std::mutex g_dma_mu;

struct AgentScan {
    uint32_t want_bdf;
    hsa_agent_t gpu{0};
    hsa_agent_t first_gpu{0};
    hsa_agent_t cpu{0};
};

hsa_status_t scan_agent(hsa_agent_t a, void* data) {
    AgentScan* sc = static_cast<AgentScan*>(data);
    hsa_device_type_t t;
    if (hsa_agent_get_info(a, HSA_AGENT_INFO_DEVICE, &t) != HSA_STATUS_SUCCESS) return HSA_STATUS_SUCCESS;
    if (t == HSA_DEVICE_TYPE_CPU && sc->cpu.handle == 0) sc->cpu = a;
    if (t == HSA_DEVICE_TYPE_GPU) {
        if (sc->first_gpu.handle == 0) sc->first_gpu = a;
        uint32_t bdf = 0;
        if (hsa_agent_get_info(a, static_cast<hsa_agent_info_t>(HSA_AMD_AGENT_INFO_BDFID), &bdf) ==
                HSA_STATUS_SUCCESS && bdf == sc->want_bdf && sc->gpu.handle == 0)
            sc->gpu = a;
    }
    return HSA_STATUS_SUCCESS;
}

int hsa_status_to_sf(hsa_status_t s) { return s == HSA_STATUS_SUCCESS ? SF_OK : SF_EDMA_BASE + int(s & 0xFFF); }
}  // namespace

// The runtime reports an engine as unavailable while any copy is pending on
// it: ours, or one of HIP's.  A HIP copy ordered after an event that has not
// fired yet sits on its engine until the event fires, and a copy of ours
// queued on that engine waits behind it (measured: 190 ms behind one such
// H2D).  So an engine of the preferred set that is busy while none of our
// copies is pending on it is held by another client: use the free engines
// among the first four in its place.  Engines 4 and up move host copies at a
// fraction of the rate; mode 2 takes them (twice as many) only when no
// engine among the first four can be had (measured in the fp32 Qwen2.5-14B
// step: gradient copies had waited ~300 ms behind held engines, and the host
// AdamW with them).  An engine that holds a copy of ours counts as ours even
// if another client's copy waits behind it; that client's copy then blocks
// only what is queued after it.
uint32_t sf_dma_choose_engines(uint32_t preferred, uint32_t avail, uint32_t ours, int mode) {
    preferred &= 0xFFFFu;
    if (preferred == 0 || mode <= 0) return preferred;
    const uint32_t held = ~avail & ~ours & 0xFFFFu;
    if ((preferred & held) == 0) return preferred;
    uint32_t use = preferred & ~held;
    const int want = __builtin_popcount(preferred);
    for (int e = 0; e < 4 && __builtin_popcount(use) < want; ++e) {
        const uint32_t b = 1u << e;
        if ((avail & b) && !(use & b)) use |= b;
    }
    if (use == 0 && mode >= 2) {
        for (int e = 4; e < 16 && __builtin_popcount(use) < 2 * want; ++e)
            if (avail & (1u << e)) use |= 1u << e;
    }
    return use != 0 ? use : preferred;
}

namespace {
// Engines for the next device -> host copies, from the runtime's engine
// status and this library's pending copies.  Called with g_dma_mu held.
uint32_t pick_engines_locked(uint32_t preferred, hsa_agent_t cpu, hsa_agent_t gpu) {
    if (preferred == 0 || g_dma.avoid_held <= 0) return preferred;
    uint32_t avail = 0;
    if (hsa_amd_memory_copy_engine_status(cpu, gpu, &avail) != HSA_STATUS_SUCCESS) return preferred;
    uint32_t ours = 0;
    for (const auto& kv : g_dma.outstanding)
        if (hsa_signal_load_scacquire(hsa_signal_t{kv.first}) >= 1) ours |= kv.second;
    return sf_dma_choose_engines(preferred, avail, ours, g_dma.avoid_held);
}
}  // namespace

int sf_dma_init(int device) {
    std::lock_guard<std::mutex> lk(g_dma_mu);
    if (g_dma.ok && g_dma.device == device) return SF_OK;
    hsa_status_t st = hsa_init();  // reference-counted; HIP holds its own reference
    if (st != HSA_STATUS_SUCCESS) return hsa_status_to_sf(st);
    // Match the HIP device to its ROCr agent by PCI location.
    int bus = 0, dev = 0, dom = 0;
    hipError_t e = hipDeviceGetAttribute(&bus, hipDeviceAttributePciBusId, device);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&dev, hipDeviceAttributePciDeviceId, device);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&dom, hipDeviceAttributePciDomainID, device);
    if (e != hipSuccess) return int(e);
    AgentScan sc;
    sc.want_bdf = (uint32_t(bus) << 8) | (uint32_t(dev) << 3);  // function 0
    st = hsa_iterate_agents(scan_agent, &sc);
    if (st != HSA_STATUS_SUCCESS) return hsa_status_to_sf(st);
    if (sc.gpu.handle == 0) sc.gpu = sc.first_gpu;  // single-GPU fallback
    if (sc.gpu.handle == 0 || sc.cpu.handle == 0) return SF_EINVAL;
    g_dma.gpu = sc.gpu;
    g_dma.cpu = sc.cpu;
    g_dma.device = device;
    // Copy profiling times come in system timestamp ticks.
    uint64_t freq = 0;
    if (hsa_system_get_info(HSA_SYSTEM_INFO_TIMESTAMP_FREQUENCY, &freq) != HSA_STATUS_SUCCESS) freq = 0;
    g_dma.ts_freq = freq;
    g_dma.ok = true;
    // Engine for device -> host copies.  HIP puts each of its own
    // host<->device copies on the first SDMA engine that is free: engine 0,
    // then 1 while 0 is held, then 2.  A HIP copy whose stream waits on an
    // event holds its engine until the event completes, and a copy queued
    // behind it on that engine waits as long (measured on MI355X: with
    // engines 0 and 1 held, a HIP copy waiting for 250 ms of GEMMs took
    // engine 2, and a 1 GiB device -> host copy split over engines 2 and 3
    // took 206 ms instead of 19-21; in the Qwen2.5-14B step the gradient
    // copies on engines 2 and 3 moved 20-28 GB/s while busy, on engine 3
    // alone 52-53).  Engines 0-3 each move 57 GB/s device -> host alone and
    // 52 beside a host -> device copy on another engine, as much as two of
    // them; engines 4-7 move ~25 GB/s together.  So the copies use engine 3
    // alone, the last fast engine HIP reaches, else engine 2, else the
    // runtime's choice.
    // An engine the status reports busy may only be running a copy at this
    // moment: ask again for up to 100 ms before settling for another one.
    g_dma.engine_mask = 0;
    uint32_t seen = 0;
    for (int tries = 0; tries < 100; ++tries) {
        uint32_t avail = 0;
        if (hsa_amd_memory_copy_engine_status(g_dma.cpu, g_dma.gpu, &avail) != HSA_STATUS_SUCCESS) break;
        seen |= avail;
        if (seen & (1u << 3)) break;
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
    }
    if (seen & (1u << 3))
        g_dma.engine_mask = 1u << 3;
    else if (seen & (1u << 2))
        g_dma.engine_mask = 1u << 2;
    return SF_OK;
}

int sf_dma_set_engines(uint32_t engine_mask) {
    std::lock_guard<std::mutex> lk(g_dma_mu);
    if (!g_dma.ok) return SF_EINVAL;
    g_dma.engine_mask = engine_mask & 0xFFFFu;
    return SF_OK;
}

int sf_dma_set_avoid_held(int mode) {
    std::lock_guard<std::mutex> lk(g_dma_mu);
    if (!g_dma.ok) return SF_EINVAL;
    if (mode < 0 || mode > 2) return SF_EINVAL;
    g_dma.avoid_held = mode;
    return SF_OK;
}

int sf_dma_get_engines(uint32_t* engine_mask) {
    std::lock_guard<std::mutex> lk(g_dma_mu);
    if (!g_dma.ok || engine_mask == nullptr) return SF_EINVAL;
    *engine_mask = g_dma.engine_mask;
    return SF_OK;
}

// On an error after some copies were issued, *nsignals holds their number and
// signals[0 .. *nsignals) their handles: those copies run to completion, and
// the caller waits for them (sf_dma_wait) before reusing the destination.
int sf_dma_copy_d2h(const sf_seg* segs, int nsegs, uint64_t* signals, int max_signals, int* nsignals) {
    if (nsegs < 0 || (nsegs > 0 && (segs == nullptr || signals == nullptr)) || nsignals == nullptr) return SF_EINVAL;
    *nsignals = 0;
    uint32_t mask = 0;
    hsa_agent_t cpu{0}, gpu{0};
    {
        std::lock_guard<std::mutex> lk(g_dma_mu);
        if (!g_dma.ok) return SF_EINVAL;
        // Every segment is checked before the first copy is issued.
        for (int i = 0; i < nsegs; ++i)
            if (segs[i].n != 0 && (segs[i].src == 0 || segs[i].dst == 0)) return SF_EINVAL;
        cpu = g_dma.cpu;
        gpu = g_dma.gpu;
        mask = pick_engines_locked(g_dma.engine_mask, cpu, gpu);
    }
    // Engines to spread over: the set bits of the engine mask, or one
    // runtime-chosen engine.
    uint32_t engines[16];
    int nengines = 0;
    for (int e = 0; e < 16; ++e)
        if (mask & (1u << e)) engines[nengines++] = 1u << e;
    if (nengines == 0) engines[nengines++] = 0;
    constexpr uint64_t kSplit = uint64_t(4) << 20;  // split copies above 4 MiB
    int rr = 0;
    for (int i = 0; i < nsegs; ++i) {
        const uint64_t bytes = segs[i].n;
        if (bytes == 0) continue;
        const int parts = (bytes >= kSplit && nengines > 1) ? nengines : 1;
        const uint64_t chunk = (bytes / parts) & ~uint64_t(4095);
        for (int k = 0; k < parts; ++k) {
            const uint64_t off = chunk * k;
            const uint64_t n = (k == parts - 1) ? bytes - off : chunk;
            if (*nsignals >= max_signals) return SF_ETOOMANY;
            hsa_signal_t sig;
            hsa_status_t st = hsa_signal_create(1, 0, nullptr, &sig);
            if (st != HSA_STATUS_SUCCESS) return hsa_status_to_sf(st);
            void* dst = reinterpret_cast<char*>(segs[i].dst) + off;
            const void* src = reinterpret_cast<const char*>(segs[i].src) + off;
            const uint32_t eng = engines[rr++ % nengines];
            if (eng != 0)
                st = hsa_amd_memory_async_copy_on_engine(dst, cpu, src, gpu, size_t(n), 0, nullptr, sig,
                                                         static_cast<hsa_amd_sdma_engine_id_t>(eng), true);
            else
                st = hsa_amd_memory_async_copy(dst, cpu, src, gpu, size_t(n), 0, nullptr, sig);
            if (st != HSA_STATUS_SUCCESS) {
                hsa_signal_destroy(sig);
                return hsa_status_to_sf(st);
            }
            {
                std::lock_guard<std::mutex> lk(g_dma_mu);
                g_dma.outstanding[sig.handle] = eng;
            }
            signals[(*nsignals)++] = sig.handle;
        }
    }
    return SF_OK;
}

int sf_dma_wait(const uint64_t* signals, int nsignals, uint64_t timeout_ns, uint64_t* start_ns,
                uint64_t* end_ns) {
    if (nsignals < 0 || (nsignals > 0 && signals == nullptr)) return SF_EINVAL;
    // Every copy must be complete before any handle is released, so that a
    // wait that ends at its deadline leaves all of them valid.  Poll with
    // short sleeps: an SDMA completion does not reliably wake a thread
    // blocked in the runtime's interrupt wait (measured: a blocked wait
    // returned 350 ms after the copy had finished).
    // at most ~30 years: the signed duration cannot wrap to a deadline in the past
    const uint64_t capped_ns = timeout_ns < (uint64_t(1) << 60) ? timeout_ns : (uint64_t(1) << 60);
    const auto deadline = std::chrono::steady_clock::now() + std::chrono::nanoseconds(int64_t(capped_ns));
    for (int i = 0; i < nsignals; ++i) {
        if (signals[i] == 0) continue;
        const hsa_signal_t sig{signals[i]};
        while (hsa_signal_load_scacquire(sig) >= 1) {
            if (timeout_ns != 0 && std::chrono::steady_clock::now() >= deadline) return SF_ETIMEDOUT;
            std::this_thread::sleep_for(std::chrono::microseconds(50));
        }
    }
    uint64_t t0 = UINT64_MAX, t1 = 0;
    int rc = SF_OK;
    for (int i = 0; i < nsignals; ++i) {
        if (signals[i] == 0) continue;
        hsa_signal_t sig{signals[i]};
        if (start_ns != nullptr && end_ns != nullptr) {
            hsa_amd_profiling_async_copy_time_t tm;
            if (hsa_amd_profiling_get_async_copy_time(sig, &tm) == HSA_STATUS_SUCCESS && tm.end > 0) {
                if (tm.start < t0) t0 = tm.start;
                if (tm.end > t1) t1 = tm.end;
            }
        }
        {
            // forget the copy before its signal handle can be reused
            std::lock_guard<std::mutex> lk(g_dma_mu);
            g_dma.outstanding.erase(signals[i]);
        }
        hsa_status_t st = hsa_signal_destroy(sig);
        if (st != HSA_STATUS_SUCCESS && rc == SF_OK) rc = hsa_status_to_sf(st);
    }
    if (start_ns != nullptr && end_ns != nullptr) {
        if (t0 == UINT64_MAX || g_dma.ts_freq == 0) {
            *start_ns = *end_ns = 0;
        } else {
            // system timestamp ticks -> ns on the same clock
            const long double scale = 1e9L / (long double)g_dma.ts_freq;
            *start_ns = uint64_t((long double)t0 * scale);
            *end_ns = uint64_t((long double)t1 * scale);
        }
    }
    return rc;
}

int sf_dma_query(const uint64_t* signals, int nsignals, int* done) {
    if (done == nullptr || nsignals < 0 || (nsignals > 0 && signals == nullptr)) return SF_EINVAL;
    *done = 1;
    for (int i = 0; i < nsignals; ++i) {
        if (signals[i] == 0) continue;
        if (hsa_signal_load_scacquire(hsa_signal_t{signals[i]}) >= 1) {
            *done = 0;
            break;
        }
    }
    return SF_OK;
}

int sf_dma_clock_ns(uint64_t* ns) {
    if (ns == nullptr) return SF_EINVAL;
    uint64_t freq = 0;
    {
        std::lock_guard<std::mutex> lk(g_dma_mu);
        if (!g_dma.ok || g_dma.ts_freq == 0) return SF_EINVAL;
        freq = g_dma.ts_freq;
    }
    uint64_t ticks = 0;
    const hsa_status_t st = hsa_system_get_info(HSA_SYSTEM_INFO_TIMESTAMP, &ticks);
    if (st != HSA_STATUS_SUCCESS) return hsa_status_to_sf(st);
    *ns = uint64_t((long double)ticks * (1e9L / (long double)freq));
    return SF_OK;
}

int sf_dma_enable_timing(int on) {
    if (!g_dma.ok) return SF_EINVAL;
    return hsa_status_to_sf(hsa_amd_profiling_async_copy_enable(on != 0));
}

}  // extern "C"
