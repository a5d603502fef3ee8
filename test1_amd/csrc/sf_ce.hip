// Cross entropy of the output unit over one chunk of logits, and the scaling
// of its gradients, for MI355X (gfx950).
//
// The three products around these kernels (logits, hidden and weight
// gradient) are library GEMMs; what lies between them moves bytes, and as
// separate elementwise and reduction passes it cost more than the products
// themselves: widening, logsumexp (three passes), gather, subtract, exp, the
// one-hot update, the mask and the rounding back moved some 25 bytes per
// logit and launched about 20 kernels per chunk.  ce_rows_kernel reads every
// logit once and writes its gradient over it: 4 bytes per 16-bit logit.
// Measured at 4092 rows of 128256 bf16 logits: ce_rows_kernel 0.43-0.45 ms
// (4.7 to 4.9 TB/s; a device copy reaches 5.1), ce_scale16_kernel for the 128256 x 4096
// weight and 4092 x 4096 hidden gradients 0.52 ms (6.0 TB/s).  The same steps as
// torch operations took 7.2 ms, and adding the chunks' weight gradients into the
// fp32 sum 8.1 ms more; loss with both gradients 35.1 -> 11.3 ms.  With the
// hidden rows transposed for the weight gradient's product (ce_hidden_kernel)
// 10.3, of which 9.5 are the products.  At 510 rows of 4096 (hidden 512) 450 ->
// 165 to 260 us with the host, 60 of them on the GPU, the rest host time of the
// launches.
//
// The C ABI is declared in include/slidefsdp.h.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/slidefsdp.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLog2eLo = 1.92596299e-8f;   // log2(e) - kLog2e
constexpr int kGroup = 8;   // 16-bit elements per 128-bit access

// 16-bit formats: a pair in a 32-bit word <-> two floats.  The conversions
// back round to nearest even (v_cvt_pk_bf16_f32, v_cvt_f16_f32), as torch's.
struct Bf16 {
    static constexpr uint32_t kNegInf2 = 0xFF80FF80u;
    static constexpr uint32_t kNegInf = 0xFF80u;
    static constexpr uint32_t kNan2 = 0x7FC07FC0u;
    __device__ static float lo(uint32_t w) { return __uint_as_float(w << 16); }
    __device__ static float hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
    __device__ static uint32_t pack(float a, float b) {
        const f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
};
struct F16 {
    static constexpr uint32_t kNegInf2 = 0xFC00FC00u;
    static constexpr uint32_t kNegInf = 0xFC00u;
    static constexpr uint32_t kNan2 = 0x7E007E00u;
    __device__ static float lo(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).x); }
    __device__ static float hi(uint32_t w) { return float(__builtin_bit_cast(f16x2, w).y); }
    __device__ static uint32_t pack(float a, float b) {
        const f32x2 f = {a, b};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
};

// exp(t) for t <= 0 as 2^(t log2 e), the product rounded: relative error up to
// |t| 2^-24 and no subnormal results.  For the terms of a row's sum alone:
// against the lane's own maximum |t| is small, and the sum's logarithm comes
// out as close to 64 bits as with expf (mean relative error of the row losses
// 3.3e-8 | 3.9e-8 at 4092 x 128256, 3.8e-8 | 4.2e-8 at 510 x 4096).
__device__ __forceinline__ float exp_term(float t) { return __builtin_amdgcn_exp2f(t * kLog2e); }

// exp(t) for finite t <= 0 or so and t = -inf, to an ulp or two, subnormal
// results included: 2^n times 2^f, f the rest of t log2 e in two parts.  What
// becomes a probability takes this one: with exp_term 1.1e-4 of the bf16
// results at 4092 x 128256 were not the nearest to the exact ones, with it
// 0.4e-4 to 0.9e-4, as with expf, which needs 5 instructions more.  us with
// exp_term | this, bf16 rows: 4092 x 128256 403 | 427, 4092 x 32000 80 | 83,
// 1023 x 50257 47 | 51, 20000 x 4096 49 | 54.
__device__ __forceinline__ float exp_full(float t) {
    t = fmaxf(t, -200.0f);   // 2^f of an infinite t would be NaN
    const float n = rintf(t * kLog2e);
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(fmaf(t, kLog2eLo, fmaf(t, kLog2e, -n))), int(n));
}

// A partial logsumexp: the maximum so far and the sum of exp(x - base(max)).
// base() is the maximum itself, or 0 where that is infinite, so that rows
// with infinities give what logsumexp gives: +inf, or -inf for a row of them.
struct Lse {
    float m, s;
};
__device__ __forceinline__ float base(float m) { return __builtin_isinf(m) ? 0.0f : m; }

// The same over groups of kN neighbouring lanes of a wave, in every lane: the
// maximum first, so that each lane rescales its part once (merging pairs costs
// two exponentials a step: 300,000 rows of 2000 bf16 1,030 us, so 694), then the
// sums.
template <int kN>
__device__ __forceinline__ Lse lane_lse(Lse p) {
    float m = p.m;
#pragma unroll
    for (int d = kN / 2; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    // an empty part stays empty whatever the bases are; a NaN sum stays NaN
    float s = p.s == 0.0f ? 0.0f : p.s * expf(base(p.m) - base(m));
#pragma unroll
    for (int d = kN / 2; d > 0; d >>= 1) s += __shfl_xor(s, d);
    return {m, s};
}

// logsumexp over a row's kT lanes, the same value in every one: in one wave
// without a barrier, else through LDS.
template <int kT>
__device__ __forceinline__ float block_lse(Lse p, Lse* parts) {
    p = lane_lse<(kT < 64 ? kT : 64)>(p);
    if constexpr (kT > 64) {
        if ((threadIdx.x & 63) == 0) parts[threadIdx.x >> 6] = p;
        __syncthreads();
        p = lane_lse<kT / 64>(parts[threadIdx.x % (kT / 64)]);
    }
    return base(p.m) + logf(p.s);
}

// Rows of one workgroup: rows that one wave or less reads share it.
template <int kT>
constexpr int kRowsOf = kT <= 64 ? 256 / kT : 1;

// What a row's label asks for.
enum RowKind { kValid, kIgnored, kBadLabel };
__device__ __forceinline__ RowKind row_kind(int64_t y, int64_t ignore_index, uint32_t vocab) {
    if (y == ignore_index) return kIgnored;
    return (y < 0 || y >= int64_t(vocab)) ? kBadLabel : kValid;
}

// Make the compiler forget what the packed words were made of, so that it
// unpacks them again in the next phase instead of keeping two floats alive
// for each word (that is 152 VGPRs more at kG = 19, and it spilled).
template <int kG>
__device__ __forceinline__ void keep_packed(u32x4 (&v)[kG]) {
#pragma unroll
    for (int k = 0; k < kG; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t w = v[k][j];
            asm volatile("" : "+v"(w));
            v[k][j] = w;
        }
}

// ---------------------------------------------------------------------
// kT lanes per row, the whole row in registers as packed 16-bit pairs:
// kG groups of 8 per lane, so 4 kG VGPRs, up to 76 of the 128 a lane of a
// 1024-lane workgroup has.  Read once, written once; between the two only
// one barrier, since each lane sums against its own maximum and the parts
// are merged with both.  All loads are issued before the first use (lanes
// past the end of the row load its last group again and drop it).  The host
// picks kG so that the row has more than kT kFull groups: the first kFull
// groups of every lane need no check.
// ---------------------------------------------------------------------
template <typename Fmt, int kT, int kG, int kFull>
__global__ __launch_bounds__(kT * kRowsOf<kT>) void ce_rows_kernel(uint16_t* __restrict__ logits, uint64_t ld,
                                                                   uint64_t rows, uint32_t vocab,
                                                                   const int64_t* __restrict__ labels,
                                                                   int64_t ignore_index, float* __restrict__ row_loss) {
    __shared__ Lse parts[kT > 64 ? kT / 64 : 1];
    __shared__ float first;
    const uint32_t lane = threadIdx.x % kT;
    const uint64_t row = uint64_t(blockIdx.x) * kRowsOf<kT> + threadIdx.x / kT;
    if (kRowsOf<kT> > 1 && row >= rows) return;   // no barrier below for these
    uint16_t* x = logits + row * ld;
    u32x4* xv = reinterpret_cast<u32x4*>(x);
    const int64_t y = labels[row];
    const uint32_t groups = (vocab + kGroup - 1) / kGroup;
    const RowKind kind = row_kind(y, ignore_index, vocab);
    if (kind != kValid) {
        const uint32_t w = kind == kIgnored ? 0u : Fmt::kNan2;
        const u32x4 fill = {w, w, w, w};
        for (uint32_t g = lane; g < groups; g += kT) xv[g] = fill;
        if (lane == 0) row_loss[row] = kind == kIgnored ? 0.0f : __builtin_nanf("");
        return;
    }
    u32x4 v[kG];
#pragma unroll
    for (int k = 0; k < kG; ++k) {
        const uint32_t g = uint32_t(k) * kT + lane;
        v[k] = xv[k < kFull || g < groups ? g : groups - 1];
    }
    // Read before any lane writes: the barrier in block_lse stands between, or
    // the row's lanes are one wave's.
    float target = 0.0f;
    if (lane == 0) target = Fmt::lo(x[y]);
    if (kT > 64) {
        if (lane == 0) first = target;
    } else {
        target = __shfl(target, 0, kT < 64 ? kT : 64);
    }
    const uint32_t rem = vocab % kGroup;
#pragma unroll
    for (int k = kFull; k < kG; ++k) {
        const uint32_t g = uint32_t(k) * kT + lane;
        if (g >= groups) {
            v[k] = u32x4{Fmt::kNegInf2, Fmt::kNegInf2, Fmt::kNegInf2, Fmt::kNegInf2};
        } else if (rem != 0 && g == groups - 1) {
            // the row's last, partial group: what follows it is padding
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (2 * uint32_t(j) >= rem) v[k][j] = Fmt::kNegInf2;
                else if (2 * uint32_t(j) + 1 >= rem) v[k][j] = (v[k][j] & 0xFFFFu) | (Fmt::kNegInf << 16);
            }
        }
    }
    float m = -__builtin_inff();
#pragma unroll
    for (int k = 0; k < kG; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) m = fmaxf(fmaxf(m, Fmt::lo(v[k][j])), Fmt::hi(v[k][j]));
    keep_packed<kG>(v);
    const float c = base(m);
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int k = 0; k < kG; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s0 += exp_term(Fmt::lo(v[k][j]) - c);
            s1 += exp_term(Fmt::hi(v[k][j]) - c);
        }
    keep_packed<kG>(v);
    const float lse = block_lse<kT>({m, s0 + s1}, parts);
    if (kT > 64) target = first;
    if (lane == 0) row_loss[row] = lse - target;
    if (!__builtin_isfinite(lse)) {
        // a row with NaN or infinities: what softmax gives, from memory again
        for (uint32_t g = lane; g < groups; g += kT) {
            const u32x4 r = xv[g];
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = Fmt::pack(expf(Fmt::lo(r[j]) - lse), expf(Fmt::hi(r[j]) - lse));
            xv[g] = o;
        }
        if (lane == uint32_t(y) / kGroup % kT) x[y] = uint16_t(Fmt::pack(expf(target - lse) - 1.0f, 0.0f));
        return;
    }
#pragma unroll
    for (int k = 0; k < kG; ++k) {
        const uint32_t g = uint32_t(k) * kT + lane;
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            o[j] = Fmt::pack(exp_full(Fmt::lo(v[k][j]) - lse), exp_full(Fmt::hi(v[k][j]) - lse));
        if (k < kFull || g < groups) xv[g] = o;
    }
    // The label's element, over what the same lane has just stored with its group.
    if (lane == uint32_t(y) / kGroup % kT)
        x[y] = uint16_t(Fmt::pack(exp_full(target - lse) - 1.0f, 0.0f));
}

// Element access of the streaming kernel below.
struct Elem32 {
    using S = float;
    __device__ static float load(const S* p) { return *p; }
    __device__ static void store(S* p, float f) { *p = f; }
};
template <typename Fmt>
struct Elem16 {
    using S = uint16_t;
    __device__ static float load(const S* p) { return Fmt::lo(*p); }
    __device__ static void store(S* p, float f) { *p = uint16_t(Fmt::pack(f, 0.0f)); }
};

// Rows that do not fit the registers (16-bit rows of more than 155,648
// elements) and fp32 rows: kT lanes per row, two passes, the second one over
// what the caches still hold.
template <typename El, int kT>
__global__ __launch_bounds__(kT * kRowsOf<kT>) void ce_rows_stream_kernel(typename El::S* __restrict__ logits,
                                                                          uint64_t ld, uint64_t rows, uint32_t vocab,
                                                                          const int64_t* __restrict__ labels,
                                                                          int64_t ignore_index,
                                                                          float* __restrict__ row_loss) {
    __shared__ Lse parts[kT > 64 ? kT / 64 : 1];
    __shared__ float first;
    const uint32_t lane = threadIdx.x % kT;
    const uint64_t row = uint64_t(blockIdx.x) * kRowsOf<kT> + threadIdx.x / kT;
    if (kRowsOf<kT> > 1 && row >= rows) return;   // no barrier below for these
    typename El::S* x = logits + row * ld;
    const int64_t y = labels[row];
    const RowKind kind = row_kind(y, ignore_index, vocab);
    if (kind != kValid) {
        const float f = kind == kIgnored ? 0.0f : __builtin_nanf("");
        for (uint32_t i = lane; i < vocab; i += kT) El::store(x + i, f);
        if (lane == 0) row_loss[row] = f;
        return;
    }
    float target = 0.0f;
    if (lane == 0) target = El::load(x + y);
    if (kT > 64) {
        if (lane == 0) first = target;
    } else {
        target = __shfl(target, 0, kT < 64 ? kT : 64);
    }
    constexpr int kU = 4;
    Lse p = {-__builtin_inff(), 0.0f};
    for (uint32_t i = lane; i < vocab; i += kT * kU) {
        float f[kU];
#pragma unroll
        for (int k = 0; k < kU; ++k) f[k] = i + k * kT < vocab ? El::load(x + i + k * kT) : -__builtin_inff();
        float m = p.m;
#pragma unroll
        for (int k = 0; k < kU; ++k) m = fmaxf(m, f[k]);
        const float c = base(m);
        float s = p.s == 0.0f ? 0.0f : p.s * expf(base(p.m) - c);
#pragma unroll
        for (int k = 0; k < kU; ++k) s += expf(f[k] - c);
        p = {m, s};
    }
    const float lse = block_lse<kT>(p, parts);
    if (kT > 64) target = first;
    if (lane == 0) row_loss[row] = lse - target;
    for (uint32_t i = lane; i < vocab; i += kT) {
        const float q = expf(El::load(x + i) - lse);
        El::store(x + i, int64_t(i) == y ? q - 1.0f : q);
    }
}

// Mean of the rows' losses and the number of rows it is taken over, each row
// once, in an order fixed by n alone: one workgroup, or, for many rows,
// kLossParts of them into `parts` and one more over those (us, one | parts:
// 32,768 rows 7.3 | 10.4, 65,536 12.0 | 10.4, 300,000 46 | 10.4, 2 M 633 | 10.1).
struct LossSum {
    double sum, count;
};
template <int kT>
__device__ __forceinline__ LossSum block_sum(LossSum p, LossSum* waves) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        p.sum += __shfl_xor(p.sum, d);
        p.count += __shfl_xor(p.count, d);
    }
    if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = p;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < kT / 64; ++w) {
            p.sum += waves[w].sum;
            p.count += waves[w].count;
        }
    return p;   // the whole sum in lane 0
}

__device__ __forceinline__ LossSum sum_rows(const float* __restrict__ row_loss, const int64_t* __restrict__ labels,
                                            uint64_t n, int64_t ignore_index, uint64_t first, uint64_t step) {
    LossSum p = {0.0, 0.0};
#pragma unroll 4
    for (uint64_t i = first; i < n; i += step) {
        p.sum += double(row_loss[i]);
        p.count += labels[i] != ignore_index ? 1.0 : 0.0;
    }
    return p;
}

constexpr int kLossThreads = 1024;
__global__ __launch_bounds__(kLossThreads) void ce_loss_kernel(const float* __restrict__ row_loss,
                                                               const int64_t* __restrict__ labels, uint64_t n,
                                                               int64_t ignore_index, float* __restrict__ loss,
                                                               float* __restrict__ n_valid) {
    __shared__ LossSum waves[kLossThreads / 64];
    const LossSum p = block_sum<kLossThreads>(
        sum_rows(row_loss, labels, n, ignore_index, threadIdx.x, kLossThreads), waves);
    if (threadIdx.x != 0) return;
    *loss = float(p.sum / p.count);
    *n_valid = float(p.count);
}

constexpr int kLossParts = SF_CE_LOSS_PARTS;
constexpr int kPartThreads = 256;
__global__ __launch_bounds__(kPartThreads) void ce_loss_parts_kernel(const float* __restrict__ row_loss,
                                                                     const int64_t* __restrict__ labels, uint64_t n,
                                                                     int64_t ignore_index, LossSum* __restrict__ parts) {
    __shared__ LossSum waves[kPartThreads / 64];
    const LossSum p = block_sum<kPartThreads>(
        sum_rows(row_loss, labels, n, ignore_index, blockIdx.x * kPartThreads + threadIdx.x,
                               uint64_t(kLossParts) * kPartThreads),
        waves);
    if (threadIdx.x == 0) parts[blockIdx.x] = p;
}

__global__ __launch_bounds__(kLossParts) void ce_loss_total_kernel(const LossSum* __restrict__ parts,
                                                                   float* __restrict__ loss,
                                                                   float* __restrict__ n_valid) {
    __shared__ LossSum waves[kLossParts / 64];
    const LossSum p = block_sum<kLossParts>(parts[threadIdx.x], waves);
    if (threadIdx.x != 0) return;
    *loss = float(p.sum / p.count);
    *n_valid = float(p.count);
}

// out = in * (grad_loss / n_valid) for both gradients in one launch: the
// hidden gradient (n_h elements) and the fp32 weight gradient (n_w), each
// rounded once into the output type.  Streaming, 8 elements per lane, one
// group per lane as the staging cast; the weight's groups come first.
constexpr int kScaleThreads = 128;
template <typename Fmt>
__device__ __forceinline__ u32x4 pack8(const f32x4 a, const f32x4 b) {
    return u32x4{Fmt::pack(a.x, a.y), Fmt::pack(a.z, a.w), Fmt::pack(b.x, b.y), Fmt::pack(b.z, b.w)};
}

template <typename Fmt>
__global__ __launch_bounds__(kScaleThreads) void ce_scale16_kernel(
    const float* __restrict__ grad_loss, const float* __restrict__ n_valid, const uint16_t* __restrict__ h,
    uint16_t* __restrict__ h_out, uint64_t n_h, const float* __restrict__ w, uint16_t* __restrict__ w_out,
    uint64_t n_w, uint64_t w_blocks, uint64_t first_block) {
    const float scale = *grad_loss / *n_valid;
    const uint64_t block = first_block + blockIdx.x;
    if (block < w_blocks) {
        const uint64_t i = (block * kScaleThreads + threadIdx.x) * kGroup;
        if (i + kGroup <= n_w) {
            const f32x4* p = reinterpret_cast<const f32x4*>(w + i);
            const f32x4 a = __builtin_nontemporal_load(p), b = __builtin_nontemporal_load(p + 1);
            __builtin_nontemporal_store(pack8<Fmt>(a * scale, b * scale), reinterpret_cast<u32x4*>(w_out + i));
        } else {
            for (uint64_t j = i; j < n_w; ++j) w_out[j] = uint16_t(Fmt::pack(w[j] * scale, 0.0f));
        }
        return;
    }
    const uint64_t i = ((block - w_blocks) * kScaleThreads + threadIdx.x) * kGroup;
    if (i + kGroup <= n_h) {
        const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(h + i));
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = Fmt::pack(Fmt::lo(v[j]) * scale, Fmt::hi(v[j]) * scale);
        __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(h_out + i));
    } else {
        for (uint64_t j = i; j < n_h; ++j) h_out[j] = uint16_t(Fmt::pack(Fmt::lo(h[j]) * scale, 0.0f));
    }
}

// fp32 gradients, 67 M elements: element by element 317 us, by 128-bit accesses
// 96 (5.6 TB/s).
__global__ __launch_bounds__(kScaleThreads) void ce_scale32_kernel(
    const float* __restrict__ grad_loss, const float* __restrict__ n_valid, const float* __restrict__ h,
    float* __restrict__ h_out, uint64_t n_h, const float* __restrict__ w, float* __restrict__ w_out, uint64_t n_w,
    uint64_t w_blocks, uint64_t first_block) {
    const float scale = *grad_loss / *n_valid;
    const uint64_t block = first_block + blockIdx.x;
    const bool is_w = block < w_blocks;
    const float* src = is_w ? w : h;
    float* dst = is_w ? w_out : h_out;
    const uint64_t n = is_w ? n_w : n_h;
    const uint64_t b = is_w ? block : block - w_blocks;
    const uint64_t i = (b * kScaleThreads + threadIdx.x) * kGroup;
    if (i + kGroup <= n) {
        const f32x4* p = reinterpret_cast<const f32x4*>(src + i);
        const f32x4 u = __builtin_nontemporal_load(p), v = __builtin_nontemporal_load(p + 1);
        __builtin_nontemporal_store(u * scale, reinterpret_cast<f32x4*>(dst + i));
        __builtin_nontemporal_store(v * scale, reinterpret_cast<f32x4*>(dst + i) + 1);
    } else {
        for (uint64_t j = i; j < n; ++j) dst[j] = src[j] * scale;
    }
}

// The chunk's hidden rows transposed, [hidden, tokens], for the product of the
// weight gradient, whose sum runs over the tokens: with one operand laid out
// along the sum, and the sum's length a multiple of 64, the product is up to a
// third faster.  us, hidden rows as they are | transposed and padded, at tokens
// x hidden x vocabulary: 4092 x 4096 x 128256 4198 | 3490, 2046 x 2560 x 151936
// 1773 | 1474, 3001 x 5120 x 65000 2001 | 1662, 1023 x 4096 x 128256 1438 |
// 1217, 777 x 1024 x 32000 79.9 | 68.6, 127 x 4096 x 128256 708 | 474.  (The
// gradient of the logits transposed too: 3355, which its 0.4 ms does not pay.)
//
// Bound by HBM: 4 bytes per element, 67 MB and 17 us at the first of these sizes.  A
// workgroup takes a tile of 64 x 64 through LDS, 128-bit accesses on both
// sides.  Rows of 66 elements in LDS put the 8 lanes that read 8 rows each, and
// the 8 columns beside each other in a wave, into banks of their own.  The
// same launch clears the rows of the gradient of the logits that pad the sum
// (workgroups from `tiles` on).
constexpr int kTr = 64;
constexpr int kTrThreads = 256;
constexpr int kTrLd = kTr + 2;
template <bool kVec>   // rows on 16-byte boundaries, hidden a multiple of 8
__global__ __launch_bounds__(kTrThreads) void ce_hidden_kernel(const uint16_t* __restrict__ hidden, uint64_t ldh,
                                                               uint64_t rows, uint64_t cols, uint16_t* __restrict__ out,
                                                               uint64_t ldt, uint32_t tiles, u32x4* __restrict__ tail,
                                                               uint64_t tail_groups) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[kTr * kTrLd];
    if (blockIdx.x >= tiles) {
        const uint64_t stride = uint64_t(gridDim.x - tiles) * kTrThreads;
        for (uint64_t g = uint64_t(blockIdx.x - tiles) * kTrThreads + threadIdx.x; g < tail_groups; g += stride)
            tail[g] = u32x4{0, 0, 0, 0};
        return;
    }
    const uint32_t across = uint32_t(ldt / kTr);
    const uint64_t row0 = uint64_t(blockIdx.x % across) * kTr, col0 = uint64_t(blockIdx.x / across) * kTr;
#pragma unroll
    for (int k = 0; k < kTr * kTr / kGroup / kTrThreads; ++k) {
        const uint32_t g = k * kTrThreads + threadIdx.x, r = g / (kTr / kGroup), c = g % (kTr / kGroup) * kGroup;
        u32x4 v = {0, 0, 0, 0};
        if (row0 + r < rows) {
            const uint16_t* p = hidden + (row0 + r) * ldh + col0 + c;
            if (kVec) {
                if (col0 + c < cols) v = *reinterpret_cast<const u32x4*>(p);
            } else {
#pragma unroll
                for (int j = 0; j < kGroup; ++j)
                    if (col0 + c + j < cols) v[j / 2] |= uint32_t(p[j]) << (j % 2 * 16);
            }
        }
        uint32_t* t = reinterpret_cast<uint32_t*>(tile + r * kTrLd + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = v[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTr * kTr / kGroup / kTrThreads; ++k) {
        const uint32_t g = k * kTrThreads + threadIdx.x, c = g / (kTr / kGroup), r = g % (kTr / kGroup) * kGroup;
        if (col0 + c >= cols) continue;
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = uint32_t(tile[(r + 2 * j) * kTrLd + c]) | uint32_t(tile[(r + 2 * j + 1) * kTrLd + c]) << 16;
        *reinterpret_cast<u32x4*>(out + (col0 + c) * ldt + row0 + r) = v;
    }
}

// The hidden gradient's product sums over the vocabulary, and for most shapes
// [tokens, hidden] has too few tiles for the chip: the sum is taken in kParts
// parts side by side (one batched product into fp32), and this kernel adds
// them up and rounds once.  A part's length is a multiple of 8, so that every
// operand starts on a 16-byte boundary; the up to 8 kParts - 1 terms that
// leaves are summed here.  A whole call, one product | parts and this kernel,
// us, tokens x hidden x vocabulary: 1023 x 4096 x 128256 4200 | 3504, 777 x
// 1024 x 32000 371 | 285.  Bound by the parts' reads, at most 134 MB, which the
// last-level cache still holds in part.
constexpr int kSumThreads = 128;
template <typename Fmt, int kParts>
__global__ __launch_bounds__(kSumThreads) void ce_sum_kernel(const float* __restrict__ parts, uint32_t count,
                                                             uint32_t cols, uint16_t* __restrict__ out,
                                                             const uint16_t* __restrict__ g, uint64_t ld,
                                                             const uint16_t* __restrict__ w, uint32_t tail) {
    const uint32_t i = (blockIdx.x * kSumThreads + threadIdx.x) * kGroup;
    if (i >= count) return;
    f32x4 a[kParts], b[kParts];
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
        const f32x4* p = reinterpret_cast<const f32x4*>(parts + uint64_t(s) * count + i);
        a[s] = __builtin_nontemporal_load(p);
        b[s] = __builtin_nontemporal_load(p + 1);
    }
    // neighbours first: a tree, whose rounding error grows with log2(kParts)
#pragma unroll
    for (int d = 1; d < kParts; d *= 2)
#pragma unroll
        for (int s = 0; s < kParts; s += 2 * d) {
            a[s] += a[s + d];
            b[s] += b[s + d];
        }
    if (tail > 0) {
        const uint32_t row = i / cols, col = i - row * cols;
        f32x4 ta = {0.0f, 0.0f, 0.0f, 0.0f}, tb = ta;
#pragma unroll 4
        for (uint32_t k = 0; k < tail; ++k) {
            const float f = Fmt::lo(g[row * ld + k]);
            const u32x4 v = *reinterpret_cast<const u32x4*>(w + uint64_t(k) * cols + col);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                ta[2 * j] = fmaf(f, Fmt::lo(v[j]), ta[2 * j]);
                ta[2 * j + 1] = fmaf(f, Fmt::hi(v[j]), ta[2 * j + 1]);
                tb[2 * j] = fmaf(f, Fmt::lo(v[j + 2]), tb[2 * j]);
                tb[2 * j + 1] = fmaf(f, Fmt::hi(v[j + 2]), tb[2 * j + 1]);
            }
        }
        a[0] += ta;
        b[0] += tb;
    }
    *reinterpret_cast<u32x4*>(out + i) = pack8<Fmt>(a[0], b[0]);
}

// The weight gradient of up to 256 tokens, [vocabulary, hidden], by the matrix
// cores with the scaling at the end, and the hidden gradient's scaling in the
// same launch.  With so few tokens its operands are small beside it and it is
// bound by its own bytes; as a product into fp32 that another kernel scales
// and rounds, it cost 10 bytes an element instead of 2.  Loss with both
// gradients, product and scaling | this, us, tokens x hidden x vocabulary: 4 x
// 4096 x 128256 1461 | 847, 1 x 5120 x 65000 906 | 565, 32 x 768 x 152064 398 |
// 304, 127 x 4096 x 128256 1455 | 1033, 200 x 4096 x 32000 467 | 380, 256 x 4096
// x 128256 1757 | 1555, 250 x 1024 x 32000 240 | 233.  Beyond, the operands no
// longer fit the registers of two waves per SIMD with four tiles each, and with
// two the loads of the hidden rows bind it: 300 x 2560 x 50257 591 | 658, 510 x
// 4096 x 32000 635 | 852.
//
// A wave owns 16 kV columns of the gradient of the logits, all tokens of them,
// as operands in registers, and walks over the hidden dimension 32 at a time
// with the transposed hidden rows (from the caches: at most 256 tokens by
// hidden).  Both index maps are permuted for wide accesses: the column of
// lane l in tile t is kV (l % 16) + t, so that a lane reads kV neighbours of a
// token at once, and the four hidden rows of lane l in tile u start at 8 (l /
// 16) + 4 u, so that it ends up with 8 neighbours and stores 16 bytes.
// Products of 16 x 16 x 32: operand lanes hold row or column l % 16, terms 8
// (l / 16) to + 7; result lanes column l % 16, rows 4 (l / 16) to + 3.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x4 mfma(Bf16, u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}
__device__ __forceinline__ f32x4 mfma(F16, u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

constexpr int kWgThreads = 256;
constexpr int kWgTokens = 256;
constexpr int kWgStep = 32;   // hidden rows a wave takes at once
constexpr int kV = 4;         // tiles of 16 columns a wave owns
constexpr int kWgColumns = kWgThreads / 64 * 16 * kV;   // of a workgroup

template <typename Fmt, int kSteps>   // at least tokens / 32
__global__ __launch_bounds__(kWgThreads, 2) void ce_weight_grad_kernel(
    const float* __restrict__ grad_loss, const float* __restrict__ n_valid, const uint16_t* __restrict__ g, uint64_t ld,
    uint32_t vocab, const uint16_t* __restrict__ hidden_t, uint32_t tokens, uint32_t hidden, uint16_t* __restrict__ out,
    uint32_t col_blocks, uint32_t per_block, uint32_t w_blocks, const uint16_t* __restrict__ h,
    uint16_t* __restrict__ h_out, uint64_t n_h) {
    const float scale = *grad_loss / *n_valid;
    if (blockIdx.x >= w_blocks) {
        const uint64_t i = (uint64_t(blockIdx.x - w_blocks) * kWgThreads + threadIdx.x) * kGroup;
        if (i < n_h) {   // a multiple of 8 elements
            const u32x4 v = *reinterpret_cast<const u32x4*>(h + i);
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = Fmt::pack(Fmt::lo(v[j]) * scale, Fmt::hi(v[j]) * scale);
            *reinterpret_cast<u32x4*>(h_out + i) = o;
        }
        return;
    }
    const uint32_t lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const uint32_t col = (blockIdx.x % col_blocks) * uint32_t(kWgColumns) + (threadIdx.x >> 6) * (16 * kV) + l16 * kV;
    const uint32_t steps = tokens / 32;   // <= kSteps
    u32x4 b[kSteps][kV];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        u32x2 e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            // ld and col are multiples of 4: all of a lane's columns lie inside the row or none
            e[j] = uint32_t(s) < steps && col < ld
                       ? *reinterpret_cast<const u32x2*>(g + uint64_t(s * 32 + quad * 8 + j) * ld + col)
                       : u32x2{0, 0};
#pragma unroll
        for (int t = 0; t < kV; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t lo = e[2 * j][t / 2] >> (t % 2 * 16), hi = e[2 * j + 1][t / 2] >> (t % 2 * 16);
                b[s][t][j] = (lo & 0xFFFFu) | hi << 16;
            }
    }
    const uint32_t first = blockIdx.x / col_blocks * per_block;
    const uint32_t last = first + per_block < hidden ? first + per_block : hidden;
    for (uint32_t h0 = first; h0 < last; h0 += kWgStep) {
        f32x4 acc[2][kV];
        const uint16_t* row[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t r = h0 + (l16 >> 2) * 8 + u * 4 + (l16 & 3);
            row[u] = hidden_t + uint64_t(r < hidden ? r : hidden - 1) * tokens + quad * 8;
#pragma unroll
            for (int t = 0; t < kV; ++t) acc[u][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            if (uint32_t(s) < steps) {
                const u32x4 a0 = *reinterpret_cast<const u32x4*>(row[0] + s * 32);
                const u32x4 a1 = *reinterpret_cast<const u32x4*>(row[1] + s * 32);
#pragma unroll
                for (int t = 0; t < kV; ++t) {
                    acc[0][t] = mfma(Fmt{}, a0, b[s][t], acc[0][t]);
                    acc[1][t] = mfma(Fmt{}, a1, b[s][t], acc[1][t]);
                }
            }
        }
        const uint32_t hr = h0 + quad * 8;
        if (hr < hidden) {   // a multiple of 8
#pragma unroll
            for (int t = 0; t < kV; ++t)
                if (col + t < vocab)
                    *reinterpret_cast<u32x4*>(out + uint64_t(col + t) * hidden + hr) =
                        pack8<Fmt>(acc[0][t] * scale, acc[1][t] * scale);
        }
    }
}

inline int status() {
    // the runtime keeps a failed launch as the thread's last error: reading it clears it
    return int(hipGetLastError());
}

inline bool misaligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; }

// Lanes of one launch: a dispatch takes fewer than 2^32 along a dimension.
constexpr uint64_t kMaxLanes = uint64_t(1) << 31;

// A kernel of kT lanes per row, over as many launches as the rows need.
template <int kT, typename Kernel, typename S>
int launch_rows(Kernel kernel, S* x, uint64_t ld, uint64_t rows, uint32_t vocab, const int64_t* labels, int64_t ignore,
                float* row_loss, hipStream_t st) {
    constexpr uint64_t kMax = kMaxLanes / kT;
    for (uint64_t r = 0; r < rows; r += kMax) {
        const uint64_t n = rows - r < kMax ? rows - r : kMax;
        hipLaunchKernelGGL(kernel, dim3(uint32_t((n + kRowsOf<kT> - 1) / kRowsOf<kT>)), dim3(kT * kRowsOf<kT>), 0, st,
                           x + r * ld, ld, n, vocab, labels + r, ignore, row_loss + r);
        const int e = status();
        if (e != SF_OK) return e;
    }
    return SF_OK;
}

// The scaling of both gradients, in as many launches as its blocks need.
template <typename S, typename Kernel>
int launch_scale(Kernel kernel, const float* grad_loss, const float* n_valid, const void* h, void* h_out, uint64_t n_h,
                 const float* w, void* w_out, uint64_t n_w, uint64_t w_blocks, uint64_t blocks, hipStream_t st) {
    constexpr uint64_t kMax = kMaxLanes / kScaleThreads;
    for (uint64_t first = 0; first < blocks; first += kMax) {
        hipLaunchKernelGGL(kernel, dim3(uint32_t(blocks - first < kMax ? blocks - first : kMax)), dim3(kScaleThreads), 0,
                           st, grad_loss, n_valid, static_cast<const S*>(h), static_cast<S*>(h_out), n_h, w,
                           static_cast<S*>(w_out), n_w, w_blocks, first);
        const int e = status();
        if (e != SF_OK) return e;
    }
    return SF_OK;
}

template <typename Fmt>
int launch_sum(int nparts, const float* parts, uint32_t count, uint32_t cols, void* out, const void* g, size_t ld,
               const void* w, uint32_t tail, hipStream_t st) {
    const auto kernel = nparts == 2   ? ce_sum_kernel<Fmt, 2>
                        : nparts == 4 ? ce_sum_kernel<Fmt, 4>
                        : nparts == 8 ? ce_sum_kernel<Fmt, 8>
                                      : ce_sum_kernel<Fmt, 16>;
    hipLaunchKernelGGL(kernel, dim3((count / kGroup + kSumThreads - 1) / kSumThreads), dim3(kSumThreads), 0, st, parts,
                       count, cols, static_cast<uint16_t*>(out), static_cast<const uint16_t*>(g), uint64_t(ld),
                       static_cast<const uint16_t*>(w), tail);
    return status();
}

template <typename Fmt>
int launch_weight_grad(const float* grad_loss, const float* n_valid, const void* g, uint64_t ld, uint32_t vocab,
                       const void* hidden_t, uint32_t tokens, uint32_t hidden, void* out, const void* h, void* h_out,
                       uint64_t n_h, hipStream_t st) {
    const uint32_t col_blocks = (vocab + kWgColumns - 1) / kWgColumns;
    // some 1,024 workgroups, the hidden dimension split where the columns give fewer
    const uint32_t steps = (hidden + kWgStep - 1) / kWgStep, want = (1024 + col_blocks - 1) / col_blocks;
    const uint32_t per = (steps + want - 1) / want, splits = (steps + per - 1) / per;
    const uint64_t h_blocks = (n_h / kGroup + kWgThreads - 1) / kWgThreads;
    const uint64_t w_blocks = uint64_t(col_blocks) * splits;
    if (w_blocks + h_blocks > (uint64_t(1) << 31) / kWgThreads) return SF_EINVAL;
    const auto kernel = tokens <= 64    ? ce_weight_grad_kernel<Fmt, 2>
                        : tokens <= 128 ? ce_weight_grad_kernel<Fmt, 4>
                                        : ce_weight_grad_kernel<Fmt, 8>;
    hipLaunchKernelGGL(kernel, dim3(uint32_t(w_blocks + h_blocks)), dim3(kWgThreads), 0, st, grad_loss, n_valid,
                       static_cast<const uint16_t*>(g), ld, vocab, static_cast<const uint16_t*>(hidden_t), tokens,
                       hidden, static_cast<uint16_t*>(out), col_blocks, per * kWgStep, uint32_t(w_blocks),
                       static_cast<const uint16_t*>(h), static_cast<uint16_t*>(h_out), n_h);
    return status();
}

// The fewest lanes that hold the row (up to 1024), then groups per lane, so
// that short rows keep many of them on a CU and long ones all their loads in
// flight at once.
template <typename Fmt>
int dispatch_rows16(uint16_t* x, uint64_t ld, uint64_t rows, uint32_t vocab, const int64_t* labels, int64_t ignore,
                    float* row_loss, hipStream_t st) {
    const uint32_t groups = (vocab + kGroup - 1) / kGroup;
    // (lanes, groups per lane, of them full: what the line above could not hold)
#define SF_ROWS(T, G, FULL)         \
    if (groups <= uint32_t(T) * G) \
        return launch_rows<T>(ce_rows_kernel<Fmt, T, G, FULL>, x, ld, rows, vocab, labels, ignore, row_loss, st);
    // (16 lanes: 2 M rows of 64 932 -> 216 us, rows of a wave each before)
    SF_ROWS(16, 1, 0)
    SF_ROWS(64, 2, 0)
    SF_ROWS(256, 2, 0)
    SF_ROWS(256, 4, 2)
    SF_ROWS(512, 4, 2)
    SF_ROWS(1024, 4, 2)
    SF_ROWS(1024, 8, 4)
    SF_ROWS(1024, 12, 8)
    SF_ROWS(1024, 16, 12)
    SF_ROWS(1024, 19, 16)
#undef SF_ROWS
    return launch_rows<1024>(ce_rows_stream_kernel<Elem16<Fmt>, 1024>, x, ld, rows, vocab, labels, ignore, row_loss, st);
}

// fp32 rows: as many lanes as have a whole step of the loop to do.  us, 1024
// lanes for every row | so: 2 M rows of 4 15,325 | 160, 500,000 of 512 4,205 |
// 557, 65,536 of 512 555 | 69.
int dispatch_rows32(float* x, uint64_t ld, uint64_t rows, uint32_t vocab, const int64_t* labels, int64_t ignore,
                    float* row_loss, hipStream_t st) {
    if (vocab <= 64)
        return launch_rows<16>(ce_rows_stream_kernel<Elem32, 16>, x, ld, rows, vocab, labels, ignore, row_loss, st);
    if (vocab <= 512)
        return launch_rows<64>(ce_rows_stream_kernel<Elem32, 64>, x, ld, rows, vocab, labels, ignore, row_loss, st);
    if (vocab <= 8192)
        return launch_rows<256>(ce_rows_stream_kernel<Elem32, 256>, x, ld, rows, vocab, labels, ignore, row_loss, st);
    return launch_rows<1024>(ce_rows_stream_kernel<Elem32, 1024>, x, ld, rows, vocab, labels, ignore, row_loss, st);
}

}  // namespace

extern "C" {

int sf_ce_rows(void* logits, int dtype, size_t ld, size_t rows, size_t vocab, const int64_t* labels,
               int64_t ignore_index, float* row_loss, sf_stream_t stream) {
    if (rows == 0) return SF_OK;
    if (logits == nullptr || labels == nullptr || row_loss == nullptr) return SF_EINVAL;
    if (vocab == 0 || vocab > (size_t(1) << 31) || rows >= (size_t(1) << 31) || ld < vocab) return SF_EINVAL;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == SF_DTYPE_F32) {
        if (misaligned(logits, 4)) return SF_EINVAL;
        return dispatch_rows32(static_cast<float*>(logits), ld, rows, uint32_t(vocab), labels, ignore_index, row_loss,
                               st);
    }
    if (dtype != SF_DTYPE_BF16 && dtype != SF_DTYPE_F16) return SF_EDTYPE;
    // whole 128-bit groups: every row starts on one and its last one is inside the row's ld elements
    if (misaligned(logits, 16) || ld % kGroup != 0) return SF_EALIGN;
    uint16_t* x = static_cast<uint16_t*>(logits);
    return dtype == SF_DTYPE_BF16
               ? dispatch_rows16<Bf16>(x, ld, rows, uint32_t(vocab), labels, ignore_index, row_loss, st)
               : dispatch_rows16<F16>(x, ld, rows, uint32_t(vocab), labels, ignore_index, row_loss, st);
}

int sf_ce_hidden(const void* hidden, size_t ldh, size_t rows, size_t cols, void* hidden_t, size_t ldt, void* tail,
                 size_t ld_tail, sf_stream_t stream) {
    if (rows == 0 || cols == 0) return SF_OK;
    if (hidden == nullptr || hidden_t == nullptr || ldh < cols || ldt % kTr != 0 || ldt < rows || ldt - rows >= kTr)
        return SF_EINVAL;
    if (ldt > rows && (tail == nullptr || ld_tail == 0)) return SF_EINVAL;
    if (misaligned(hidden, 2)) return SF_EINVAL;
    if (misaligned(hidden_t, 16) || (ldt > rows && (misaligned(tail, 16) || ld_tail % kGroup != 0))) return SF_EALIGN;
    const uint64_t tiles = uint64_t(ldt / kTr) * ((cols + kTr - 1) / kTr);
    const uint64_t groups = uint64_t(ldt - rows) * (ldt > rows ? ld_tail / kGroup : 0);
    // one group per lane of the cleared rows, in at most 2,048 workgroups
    const uint64_t want = (groups + kTrThreads - 1) / kTrThreads, clear = want < 2048 ? want : 2048;
    if (tiles + clear > (uint64_t(1) << 31) / kTrThreads) return SF_EINVAL;
    const bool vec = !misaligned(hidden, 16) && ldh % kGroup == 0 && cols % kGroup == 0;
    hipLaunchKernelGGL((vec ? ce_hidden_kernel<true> : ce_hidden_kernel<false>), dim3(uint32_t(tiles + clear)),
                       dim3(kTrThreads), 0, reinterpret_cast<hipStream_t>(stream), static_cast<const uint16_t*>(hidden),
                       uint64_t(ldh), uint64_t(rows), uint64_t(cols), static_cast<uint16_t*>(hidden_t), uint64_t(ldt),
                       uint32_t(tiles), static_cast<u32x4*>(tail), groups);
    return status();
}

int sf_ce_sum(const float* parts, int nparts, size_t rows, size_t cols, void* out, int dtype, const void* g_tail,
              size_t ld, const void* w_tail, size_t tail, sf_stream_t stream) {
    if (rows == 0 || cols == 0) return SF_OK;
    if (parts == nullptr || out == nullptr || (nparts != 2 && nparts != 4 && nparts != 8 && nparts != 16))
        return SF_EINVAL;
    if (tail >= size_t(kGroup) * size_t(nparts) || (tail > 0 && (g_tail == nullptr || w_tail == nullptr || ld < tail)))
        return SF_EINVAL;
    if (cols > (size_t(1) << 31) || rows > (size_t(1) << 31) / cols) return SF_EINVAL;
    if (cols % kGroup != 0 || misaligned(parts, 16) || misaligned(out, 16) || (tail > 0 && misaligned(w_tail, 16)) ||
        (tail > 0 && misaligned(g_tail, 2)))
        return SF_EALIGN;
    const uint32_t count = uint32_t(rows * cols);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == SF_DTYPE_BF16)
        return launch_sum<Bf16>(nparts, parts, count, uint32_t(cols), out, g_tail, ld, w_tail, uint32_t(tail), st);
    if (dtype == SF_DTYPE_F16)
        return launch_sum<F16>(nparts, parts, count, uint32_t(cols), out, g_tail, ld, w_tail, uint32_t(tail), st);
    return SF_EDTYPE;
}

int sf_ce_loss(const float* row_loss, const int64_t* labels, size_t n, int64_t ignore_index, float* loss,
               float* n_valid, sf_stream_t stream) {
    if (loss == nullptr || n_valid == nullptr || (n > 0 && (row_loss == nullptr || labels == nullptr)))
        return SF_EINVAL;
    hipLaunchKernelGGL(ce_loss_kernel, dim3(1), dim3(kLossThreads), 0, reinterpret_cast<hipStream_t>(stream),
                       row_loss, labels, uint64_t(n), ignore_index, loss, n_valid);
    return status();
}

int sf_ce_loss_parts(const float* row_loss, const int64_t* labels, size_t n, int64_t ignore_index, void* parts,
                     float* loss, float* n_valid, sf_stream_t stream) {
    if (loss == nullptr || n_valid == nullptr || parts == nullptr ||
        (n > 0 && (row_loss == nullptr || labels == nullptr)))
        return SF_EINVAL;
    if (misaligned(parts, sizeof(double))) return SF_EALIGN;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    LossSum* p = static_cast<LossSum*>(parts);
    hipLaunchKernelGGL(ce_loss_parts_kernel, dim3(kLossParts), dim3(kPartThreads), 0, st, row_loss, labels, uint64_t(n),
                       ignore_index, p);
    const int e = status();
    if (e != SF_OK) return e;
    hipLaunchKernelGGL(ce_loss_total_kernel, dim3(1), dim3(kLossParts), 0, st, p, loss, n_valid);
    return status();
}

int sf_ce_scale(const float* grad_loss, const float* n_valid, const void* grad_h, void* grad_h_out, size_t n_h,
                const float* grad_w, void* grad_w_out, size_t n_w, int dtype, sf_stream_t stream) {
    if (n_h == 0 && n_w == 0) return SF_OK;
    if (grad_loss == nullptr || n_valid == nullptr) return SF_EINVAL;
    if ((n_h > 0 && (grad_h == nullptr || grad_h_out == nullptr)) ||
        (n_w > 0 && (grad_w == nullptr || grad_w_out == nullptr)))
        return SF_EINVAL;
    if (misaligned(grad_h, 16) || misaligned(grad_h_out, 16) || misaligned(grad_w, 16) || misaligned(grad_w_out, 16))
        return SF_EALIGN;
    constexpr uint64_t kPer = uint64_t(kScaleThreads) * kGroup;
    const uint64_t wb = (n_w + kPer - 1) / kPer, hb = (n_h + kPer - 1) / kPer;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
        case SF_DTYPE_F32:
            return launch_scale<float>(ce_scale32_kernel, grad_loss, n_valid, grad_h, grad_h_out, n_h, grad_w,
                                       grad_w_out, n_w, wb, wb + hb, st);
        case SF_DTYPE_BF16:
            return launch_scale<uint16_t>(ce_scale16_kernel<Bf16>, grad_loss, n_valid, grad_h, grad_h_out, n_h, grad_w,
                                          grad_w_out, n_w, wb, wb + hb, st);
        case SF_DTYPE_F16:
            return launch_scale<uint16_t>(ce_scale16_kernel<F16>, grad_loss, n_valid, grad_h, grad_h_out, n_h, grad_w,
                                          grad_w_out, n_w, wb, wb + hb, st);
        default: return SF_EDTYPE;
    }
}

int sf_ce_weight_grad(const float* grad_loss, const float* n_valid, const void* g, size_t ld, size_t vocab,
                      const void* hidden_t, size_t tokens, size_t hidden, void* grad_w_out, const void* grad_h,
                      void* grad_h_out, size_t n_h, int dtype, sf_stream_t stream) {
    if (grad_loss == nullptr || n_valid == nullptr || g == nullptr || hidden_t == nullptr || grad_w_out == nullptr ||
        (n_h > 0 && (grad_h == nullptr || grad_h_out == nullptr)))
        return SF_EINVAL;
    if (tokens == 0 || tokens % 64 != 0 || tokens > size_t(kWgTokens) || vocab == 0 || vocab > (size_t(1) << 31) ||
        hidden == 0 || hidden > (size_t(1) << 31) || ld < vocab)
        return SF_EINVAL;
    if (ld % kGroup != 0 || hidden % kGroup != 0 || n_h % kGroup != 0 || misaligned(g, 16) || misaligned(hidden_t, 16) ||
        misaligned(grad_w_out, 16) || misaligned(grad_h, 16) || misaligned(grad_h_out, 16))
        return SF_EALIGN;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == SF_DTYPE_BF16)
        return launch_weight_grad<Bf16>(grad_loss, n_valid, g, ld, uint32_t(vocab), hidden_t, uint32_t(tokens),
                                        uint32_t(hidden), grad_w_out, grad_h, grad_h_out, n_h, st);
    if (dtype == SF_DTYPE_F16)
        return launch_weight_grad<F16>(grad_loss, n_valid, g, ld, uint32_t(vocab), hidden_t, uint32_t(tokens),
                                       uint32_t(hidden), grad_w_out, grad_h, grad_h_out, n_h, st);
    return SF_EDTYPE;
}

}  // extern "C"
