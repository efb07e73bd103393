// kernels.hpp - gfx950 kernels of the quantized histogram / partition / split path.
//
// Compiled with -ffp-contract=off and without fast math: every f32/f64 operation below is the IEEE operation
// silvic's CPU path performs, in the same order, so quantized values and split decisions are bit-identical.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "exp_f64.hpp"
#include "packed_word.hpp"

namespace srocm {

constexpr double K_EPSILON = static_cast<double>(1e-15f);  // split.rs:37 (a float literal widened)
constexpr int WAVE = 64;

// ---------------------------------------------------------------------------------------------------------
// Rust numeric semantics on the device
// ---------------------------------------------------------------------------------------------------------

// `x as i32` for f32: truncation toward zero, saturating, NaN -> 0.
__device__ __forceinline__ int32_t sat_i32(float x) {
    if (x != x) return 0;
    if (x >= 2147483648.0f) return 2147483647;
    if (x <= -2147483648.0f) return (-2147483647 - 1);
    return static_cast<int32_t>(x);
}

// `x as i64` for f64.
__device__ __forceinline__ int64_t sat_i64(double x) {
    if (x != x) return 0;
    if (x >= 9223372036854775807.0) return INT64_MAX;
    if (x <= -9223372036854775808.0) return INT64_MIN;
    return static_cast<int64_t>(x);
}

// f64::max (IEEE maxNum: a NaN operand yields the other).
__device__ __forceinline__ double max_num(double a, double b) {
    if (a != a) return b;
    if (b != b) return a;
    return a > b ? a : b;
}

// ---------------------------------------------------------------------------------------------------------
// quantize.rs:14-31 counter hash and quantize.rs:100-136 stochastic rounding
// ---------------------------------------------------------------------------------------------------------

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352dU;
    x ^= x >> 15;
    x *= 0x846ca68bU;
    x ^= x >> 16;
    return x;
}

__device__ __forceinline__ float uniform(uint32_t seed, uint32_t stream, uint32_t iteration, uint64_t row) {
    uint32_t row_hash = mix32(static_cast<uint32_t>(row) ^ mix32(static_cast<uint32_t>(row >> 32)));
    uint32_t h = mix32(seed ^ mix32(stream ^ mix32(iteration ^ row_hash)));
    return static_cast<float>(h >> 8) * (1.0f / 16777216.0f);
}

struct QuantDev {
    float inv_grad_scale, inv_hess_scale;
    int32_t grad_max_q, hess_max_q;
    uint32_t constant_hessian, stochastic, seed, iteration;
};

__device__ __forceinline__ int32_t clamp_i32(int32_t v, int32_t lo, int32_t hi) { return v < lo ? lo : (v > hi ? hi : v); }

// quantize.rs:103-136 quantize_row
__device__ __forceinline__ int32_t quantize_row(const QuantDev &s, float grad, float hess, uint64_t row) {
    float q;
    if (s.stochastic) {
        float u = uniform(s.seed, 0u, s.iteration, row);
        q = grad >= 0.0f ? __builtin_truncf(__builtin_fmaf(grad, s.inv_grad_scale, u))
                         : __builtin_truncf(__builtin_fmaf(grad, s.inv_grad_scale, -u));
    } else {
        q = __builtin_rintf(grad * s.inv_grad_scale);
    }
    int32_t g = clamp_i32(sat_i32(q), -s.grad_max_q, s.grad_max_q);
    int32_t h;
    if (s.constant_hessian) {
        h = 1;
    } else {
        float p;
        if (s.stochastic) {
            float u = uniform(s.seed, 1u, s.iteration, row);
            p = __builtin_truncf(__builtin_fmaf(hess, s.inv_hess_scale, u));
        } else {
            p = __builtin_rintf(hess * s.inv_hess_scale);
        }
        h = clamp_i32(sat_i32(p), 0, s.hess_max_q);
    }
    return static_cast<int32_t>(static_cast<uint32_t>(h) * 65536u + static_cast<uint32_t>(g));
}

__global__ void k_quantize(const float *__restrict__ grad, const float *__restrict__ hess, int32_t *__restrict__ packed,
                           uint64_t n, uint64_t row_offset, QuantDev spec) {
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x)
        packed[r] = quantize_row(spec, grad[r], hess[r], row_offset + r);
}

// The gradient maxima live in MAX_SLOTS pairs of words: block b adds its own to pair b mod MAX_SLOTS, so at most
// ceil(blocks / MAX_SLOTS) atomics meet at one address (atomics on one address are served one at a time, about
// 11 ns each: 2048 blocks on one pair took 49 us where the loads took 4), and readers take the largest pair-wise.
constexpr uint32_t MAX_SLOTS = 64;

// An iteration's quantization made on the device from the gradient maxima, so the boosting loop never waits for
// them: the scales of quantize.rs:56-84 and the fixed-point scales of quantize.rs:153-159, in the host's double
// operations (ceil(log2 x) from the exponent: exact for the float maxima these are).
struct DevScales {
    double sg, sh;    // grad_scale, hess_scale
    float gsc, hsc;   // the leaf sums' fixed-point scales
    QuantDev q;
};

__device__ __forceinline__ double positive_or_one_d(double v) { return v > 0.0 && __builtin_isfinite(v) ? v : 1.0; }

__device__ __forceinline__ float fixed_point_scale_d(double max_abs) {
    if (!__builtin_isfinite(max_abs) || max_abs <= 0.0) return 1.0f;
    int ex = 0;
    const double m = __builtin_frexp(max_abs, &ex);  // max_abs = m * 2^ex, m in [0.5, 1)
    int e = 30 - (m == 0.5 ? ex - 1 : ex);
    e = e < -126 ? -126 : (e > 127 ? 127 : e);
    return __builtin_ldexpf(1.0f, e);
}

// What an iteration's quantization is made from besides the gradient maxima.
struct SpecArgs {
    uint32_t num_bins, constant_hessian;
    double constant;
    uint32_t stochastic, seed, iteration;
};
__device__ __forceinline__ DevScales make_scales(uint32_t max_g, uint32_t max_h, const SpecArgs &a) {
    const double mg = static_cast<double>(__uint_as_float(max_g)), mh = static_cast<double>(__uint_as_float(max_h));
    DevScales d;
    d.q.grad_max_q = static_cast<int32_t>(a.num_bins / 2);
    d.q.hess_max_q = static_cast<int32_t>(a.num_bins);
    d.sg = positive_or_one_d(mg / static_cast<double>(d.q.grad_max_q));
    d.sh = a.constant_hessian ? positive_or_one_d(a.constant) : positive_or_one_d(mh / static_cast<double>(d.q.hess_max_q));
    d.q.inv_grad_scale = static_cast<float>(1.0 / d.sg);
    d.q.inv_hess_scale = static_cast<float>(1.0 / d.sh);
    d.q.constant_hessian = a.constant_hessian;
    d.q.stochastic = a.stochastic;
    d.q.seed = a.seed;
    d.q.iteration = a.iteration;
    d.gsc = fixed_point_scale_d(mg);
    d.hsc = fixed_point_scale_d(mh);
    return d;
}

// The boosting loop's quantization in one pass: every block makes the scales from the maxima (MAX_SLOTS pairs), block 0
// leaves them for the kernels after it and clears the other gradients' maxima (`clear`: the two buffers take turns, so
// the next gradients start from zero without a fill); then each row's packed word and, when given, the partition in row
// order (`part`) and the rows' gradient codes (`codes`, packed_code). Bound by memory: 8 B read and 4 to 9 B written a row,
// four rows a thread a load. Four launches before (scales, words, row ids, codes): 60 us at 10M rows, 36 now; on small
// tables it is the three launches that count.
__global__ __launch_bounds__(256) void k_quantize_dev(const float *__restrict__ grad, const float *__restrict__ hess,
                                                      int32_t *__restrict__ packed, uint64_t n, uint64_t row_offset,
                                                      const uint32_t *maxima, uint32_t *clear, DevScales *out, SpecArgs a,
                                                      uint32_t *__restrict__ part, uint8_t *__restrict__ codes) {
    __shared__ QuantDev s_q;
    static_assert(MAX_SLOTS == 64, "one slot pair a lane");
    if (threadIdx.x < MAX_SLOTS) {
        uint32_t ug = maxima[2u * threadIdx.x], uh = maxima[2u * threadIdx.x + 1u];
        for (int o = 32; o >= 1; o >>= 1) {
            const uint32_t x = __shfl_xor(ug, o), y = __shfl_xor(uh, o);
            ug = ug > x ? ug : x;
            uh = uh > y ? uh : y;
        }
        const DevScales d = make_scales(ug, uh, a);
        if (threadIdx.x == 0) s_q = d.q;
        if (blockIdx.x == 0) {
            clear[2u * threadIdx.x] = 0u;
            clear[2u * threadIdx.x + 1u] = 0u;
            if (threadIdx.x == 0) *out = d;
        }
    }
    __syncthreads();
    const QuantDev spec = s_q;
    const uint64_t quads = n / 4;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < quads; i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const float4 g = reinterpret_cast<const float4 *>(grad)[i], h = reinterpret_cast<const float4 *>(hess)[i];
        const uint64_t r = row_offset + 4 * i;
        const int4 w = make_int4(quantize_row(spec, g.x, h.x, r), quantize_row(spec, g.y, h.y, r + 1),
                                 quantize_row(spec, g.z, h.z, r + 2), quantize_row(spec, g.w, h.w, r + 3));
        reinterpret_cast<int4 *>(packed)[i] = w;
        const uint32_t id = static_cast<uint32_t>(4 * i);
        if (part) reinterpret_cast<uint4 *>(part)[i] = make_uint4(id, id + 1, id + 2, id + 3);
        if (codes) reinterpret_cast<uchar4 *>(codes)[i] = make_uchar4(packed_code(w.x), packed_code(w.y), packed_code(w.z), packed_code(w.w));
    }
    if (blockIdx.x == 0 && threadIdx.x < n % 4) {
        const uint64_t r = 4 * quads + threadIdx.x;
        const int32_t w = quantize_row(spec, grad[r], hess[r], row_offset + r);
        packed[r] = w;
        if (part) part[r] = static_cast<uint32_t>(r);
        if (codes) codes[r] = packed_code(w);
    }
}

// ---------------------------------------------------------------------------------------------------------
// gradients (objective/regression.rs:70-93: f32 arithmetic) and their maxima (cpu.rs:774)
// ---------------------------------------------------------------------------------------------------------

// max |v| as the bits of a non-negative float (order-preserving as unsigned), NaN skipped.
__device__ __forceinline__ uint32_t abs_bits(float v) {
    float a = __builtin_fabsf(v);
    return (a != a) ? 0u : __float_as_uint(a);
}

// Block-wide max of two per-thread values, one atomicMax each per block into its slot pair (blockDim 256).
__device__ __forceinline__ void block_max2(uint32_t a, uint32_t b, uint32_t *out) {
    __shared__ uint32_t sa[4], sb[4];
    for (int o = 32; o >= 1; o >>= 1) {
        uint32_t x = __shfl_xor(a, o), y = __shfl_xor(b, o);
        a = a > x ? a : x;
        b = b > y ? b : y;
    }
    if ((threadIdx.x & 63) == 0) {
        sa[threadIdx.x >> 6] = a;
        sb[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) {
            a = a > sa[w] ? a : sa[w];
            b = b > sb[w] ? b : sb[w];
        }
        uint32_t *slot = out + 2u * (blockIdx.x % MAX_SLOTS);
        atomicMax(slot, a);
        atomicMax(slot + 1, b);
    }
}

__global__ void k_grad_regression(const float *__restrict__ scores, const float *__restrict__ label,
                                  const float *__restrict__ weight, float *__restrict__ grad, float *__restrict__ hess,
                                  uint64_t n, uint32_t *maxima) {
    uint32_t mg = 0, mh = 0;
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x) {
        float g, h;
        float residual = scores[r] - label[r];
        if (weight) {
            g = residual * weight[r];
            h = weight[r];
        } else {
            g = residual;
            h = 1.0f;
        }
        grad[r] = g;
        hess[r] = h;
        uint32_t a = abs_bits(g), b = abs_bits(h);
        mg = mg > a ? mg : a;
        mh = mh > b ? mh : b;
    }
    block_max2(mg, mh, maxima);
}

// objective/binary.rs:27-50: f64 logloss gradients with an exp equal to the C library's, stored as f32
__global__ void k_grad_binary(const float *__restrict__ scores, const float *__restrict__ label,
                              const float *__restrict__ weight, float *__restrict__ grad, float *__restrict__ hess,
                              uint64_t n, double sigmoid, uint32_t *maxima) {
    uint32_t mg = 0, mh = 0;
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x) {
        double sign = label[r] > 0.0f ? 1.0 : -1.0;
        double response = -sign * sigmoid / (1.0 + srocm_exp::exp(sign * sigmoid * static_cast<double>(scores[r])));
        double abs_response = __builtin_fabs(response);
        double w = weight ? static_cast<double>(weight[r]) : 1.0;
        float g = static_cast<float>(response * w);
        float h = static_cast<float>(abs_response * (sigmoid - abs_response) * w);
        grad[r] = g;
        hess[r] = h;
        uint32_t a = abs_bits(g), b = abs_bits(h);
        mg = mg > a ? mg : a;
        mh = mh > b ? mh : b;
    }
    block_max2(mg, mh, maxima);
}

__global__ void k_max_abs(const float *__restrict__ grad, const float *__restrict__ hess, uint64_t n, uint32_t *maxima) {
    uint32_t mg = 0, mh = 0;
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t a = abs_bits(grad[r]), b = abs_bits(hess[r]);
        mg = mg > a ? mg : a;
        mh = mh > b ? mh : b;
    }
    block_max2(mg, mh, maxima);
}

__global__ void k_fill_f32(float *__restrict__ out, uint64_t n, float v) {
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x)
        out[r] = v;
}

__global__ void k_zero_i64(int64_t *__restrict__ out, uint64_t n) {
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x)
        out[r] = 0;
}

// Column-major bins, one byte per bin, or two (little-endian u16) when the dataset has features of more than 256
// bins (`col16`).
__device__ __forceinline__ uint32_t col_bin(const uint8_t *col, uint32_t col16, size_t i) {
    return col16 ? static_cast<uint32_t>(reinterpret_cast<const uint16_t *>(col)[i]) : static_cast<uint32_t>(col[i]);
}

// Whether a split sends `bin` left: a byte feature's split is its 256-bit mask (BinSplit::goes_left,
// backend/mod.rs:34-37); a feature of more than 256 bins (`wide`) carries its numerical rule in the words instead:
// lb[0] the threshold, lb[1] the NaN bin + 1 when missing values go left (0 otherwise).
__device__ __forceinline__ bool rule_left(const uint32_t *lb, uint32_t wide, uint32_t bin) {
    if (wide) return bin <= lb[0] || (lb[1] != 0u && bin == lb[1] - 1u);
    return ((lb[bin >> 5] >> (bin & 31u)) & 1u) != 0u;
}

__global__ void k_iota(uint32_t *__restrict__ out, uint64_t n) {
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < n; r += (uint64_t)gridDim.x * blockDim.x)
        out[r] = static_cast<uint32_t>(r);
}

// ---------------------------------------------------------------------------------------------------------
// Histogram of a leaf over one slab (a run of up to W features stored as W-byte rows).
//
// LDS holds the slab's histogram bin-major: word (bin * W + column), one packed i32 (h_q << 16) + g_q per bin
// (quantize.rs:100-107). A wave covers 64 / (W/4) rows, each lane one dword (4 columns) of a row. At step k a
// lane adds byte x = (k + (lane%32)/8) % 4 of its dword, so the 32 lanes of each half-wave hit the 32 LDS banks
// (bank = column mod 32 = 4 * (lane%8) + x) exactly once: every ds_add_u32 is conflict-free whatever the bins.
// Every `flush_rows` rows (at most 32767 / max |g| and 65535 / max h: the low half holds g as a signed 16-bit
// value, the high half h, which is never negative, as an unsigned one) the packed words are unpacked into per-thread
// registers (i32 g and h sums) and zeroed. Each workgroup writes its sums as a partial
// histogram `partial[wg][bin * W + column] = {g, h}`, or, when its rows never need a flush, the packed words themselves (half
// the bytes: 128 columns, 202k rows over 98 workgroups 32.0 -> 26.7 us with the reduce); k_hist_reduce adds the partials.
// ---------------------------------------------------------------------------------------------------------

struct HistArgs {
    const uint8_t *bins;      // slab rows: row r at bins + r * W
    const uint32_t *rows;     // partition buffer; the leaf's rows start at `begin`
    const int32_t *gh;        // packed quantized gradients per row
    int32_t *partial;         // [groups][256 * W] {g, h} pairs, or packed words in the first half of each
    const uint32_t *dev_left; // when non-null: the leaf is the `side` child of [begin, begin+count) split at *dev_left
    uint32_t begin, count, side;
    uint32_t flush_rows;
    uint32_t max_groups;      // row ranges at most
    uint32_t min_rows_per_group;
    const uint32_t *pos_word; // dense slab: per row byte, its LDS word at bin 0 (segment base * W + column)
    uint32_t dw_row;          // dense slab: dwords per row
};

// The rows of the leaf after resolving a device-side left count; identical in every kernel that calls it.
__device__ __forceinline__ void leaf_rows(const uint32_t *dev_left, uint32_t begin, uint32_t count, uint32_t side,
                                          uint32_t &b, uint32_t &n) {
    if (dev_left) {
        uint32_t left = *dev_left;
        if (side == 0) {
            b = begin;
            n = left;
        } else {
            b = begin + left;
            n = count - left;
        }
    } else {
        b = begin;
        n = count;
    }
}

// Workgroups used for n rows and rows per workgroup (a multiple of 64); identical in k_hist and k_hist_reduce.
__device__ __forceinline__ void hist_split(uint32_t n, uint32_t max_groups, uint32_t min_rows, uint32_t &groups,
                                           uint32_t &per) {
    uint32_t want = (n + min_rows - 1) / min_rows;
    groups = want < max_groups ? want : max_groups;
    if (groups == 0) groups = 1;
    per = (n + groups - 1) / groups;
    per = (per + 63u) & ~63u;
    if (per == 0) per = 64;
    groups = (n + per - 1) / per;
    if (groups == 0) groups = 1;
}

// A lane's four adds per row dword, in the conflict-free order: at step k byte x = (k + rot) % 4, i.e. bits 8x..8x+7
// (xs[k] = 8x), is the row's byte i = 4d + x and goes to column i (cols[k]). In a packed slab (PACK features of at
// most 256 / PACK bins a column) byte i goes to column i % W, in the rows of its segment i / W: cols[k] is then
// the word offset of that segment's column, and a bin b adds to word b * W + cols[k] as in a byte slab (the bank
// is still the column's).
template <int W, int PACK>
__device__ __forceinline__ void row_bin_lanes(uint32_t d, uint32_t rot, uint32_t (&xs)[4], uint32_t (&cols)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t x = (k + rot) & 3u;
        const uint32_t i = 4u * d + x;
        xs[k] = 8u * x;
        cols[k] = PACK == 1 ? i : (i / W) * (256u / PACK) * W + i % W;
    }
}

// Adds gv to the LDS words (bin * W + column) of the four bins in a row dword: each bin is extracted in place (one
// bit-field extract) and scaled into its word address with the column added (one shift-add). Q32: the LDS holds
// separate 32-bit g and h counters (g words first, then 256 * W h words), and gv, hv are the row's g and h.
template <int W, int PACK = 1, bool Q32 = false>
__device__ __forceinline__ void add_row_bins(int32_t *lds, uint32_t dw, int32_t gv, int32_t hv, const uint32_t (&xs)[4],
                                             const uint32_t (&cols)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t b = __builtin_amdgcn_ubfe(dw, xs[k], 8u);
        if constexpr (PACK > 1) b &= 256u / PACK - 1u;  // a packed column's segment: invalid bins stay in it
        atomicAdd(&lds[b * W + cols[k]], gv);
        if constexpr (Q32) atomicAdd(&lds[256 * W + b * W + cols[k]], hv);
    }
}

// A wide slab (two-byte bins of up to 1024, W / 4 features) keeps the byte slab's LDS and partial shape: bin b of
// its column c is word (b >> 2) * W + (b & 3) * (W / 4) + c, i.e. a wide column is four virtual byte columns (bins
// congruent to 0, 1, 2, 3 mod 4). A lane's dword holds the bins of columns 2d and 2d + 1.
template <int W, bool Q32 = false>
__device__ __forceinline__ void add_row_bins_wide(int32_t *lds, uint32_t dw, int32_t gv, int32_t hv, uint32_t d) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t b = min((dw >> (16 * k)) & 0xffffu, 1023u);  // clamped: invalid bins stay inside the LDS
        const uint32_t w = (b >> 2) * W + (b & 3u) * (W / 4) + 2u * d + k;
        atomicAdd(&lds[w], gv);
        if constexpr (Q32) atomicAdd(&lds[256 * W + w], hv);
    }
}

// A row's quantized pair as the LDS adds take it: the packed word itself, or (Q32) its g and h apart.
template <bool Q32>
__device__ __forceinline__ void row_units(int32_t word, bool on, int32_t &gv, int32_t &hv) {
    if constexpr (Q32) {
        const int32_t g = packed_g(word);
        gv = on ? g : 0;
        hv = on ? packed_h(word, g) : 0;
    } else {
        gv = on ? word : 0;
        hv = 0;
    }
}

// A dense slab (DP passes): features stacked in the LDS columns by their bin counts, W = 128 columns of 256 bin rows
// and a spare row 256. The feature at row byte i is in column i % 128 at rows [base, base + bins) of it; pos_word[i]
// = base * W + i % 128, and positions past the slab's features point at the spare row (their bytes are 0). A row of
// up to 64 * DP dwords is read by the whole wave, lane l taking dwords l, l + 64, ... (pass p): byte x of dword
// 64p + l is position 256p + 4l + x, so the 32 lanes of a half-wave add to 32 distinct columns, as in a byte slab.
template <int DP>
__device__ __forceinline__ void dense_lanes(const uint32_t *pos_word, uint32_t lane, uint32_t (&xs)[4],
                                            uint32_t (&cols)[DP][4]) {
    const uint32_t rot = (lane & 31u) >> 3;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t x = (k + rot) & 3u;
        xs[k] = 8u * x;
#pragma unroll
        for (int p = 0; p < DP; ++p) cols[p][k] = pos_word[256u * p + 4u * lane + x];
    }
}

// The rows list[c0 .. c1) of a dense slab into the LDS, UNROLL rows a wave at a time over NW waves (`wave` among
// them); dwords past the row (dw_row) read as 0, i.e. bin 0 of spare positions. 16 dwords a lane are in flight whatever the
// row's length (UNROLL = 16 / DP): what bounds it is the latency of the rows' gathers. A step's row ids and gradients are
// one load each (lane u: row u, read across lanes as scalars), the ids a step ahead. With 4 passes for every row of up to
// 1024 bytes, a 256-byte row took three passes of spare adds: 1M x 136 in 256-byte rows, root k_hist 172 -> 71 us,
// k_step_rows 72.3 -> 29.1 us a launch.
template <int DP> constexpr int dense_unroll() { return 16 / DP; }
template <int W, int DP, int NW = 16, bool CODES = false>
__device__ __forceinline__ void hist_list_dense(int32_t *lds, const uint32_t *list, uint32_t c0, uint32_t c1,
                                                const int32_t *gh, const uint32_t *bins32, uint32_t dw_row,
                                                const uint32_t (&xs)[4], const uint32_t (&cols)[DP][4],
                                                uint32_t wave = threadIdx.x >> 6, const uint8_t *codes = nullptr) {
    constexpr int UNROLL = dense_unroll<DP>();
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t base = c0 + __builtin_amdgcn_readfirstlane(wave) * UNROLL;
    if (base >= c1) return;
    const uint32_t last = c1 - 1, mine = lane < UNROLL ? lane : UNROLL - 1;
    uint32_t cidx = list[min(base + mine, last)];
    for (; base < c1; base += NW * UNROLL) {
        int32_t gl;
        if constexpr (CODES) gl = code_word(codes[min(base + mine, last)]);
        else gl = gh[cidx];
        uint32_t r[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) r[u] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(cidx), u));
        cidx = list[min(base + NW * UNROLL + mine, last)];
        uint32_t dw[UNROLL][DP];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t *row = bins32 + static_cast<size_t>(r[u]) * dw_row;
#pragma unroll
            for (int p = 0; p < DP; ++p) {
                const uint32_t d = 64u * p + lane;
                dw[u][p] = d < dw_row ? row[d] : 0u;
            }
        }
        if (base + mine >= c1) gl = 0;
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int32_t gv = __builtin_amdgcn_readlane(gl, u);
#pragma unroll
            for (int p = 0; p < DP; ++p) add_row_bins<W>(lds, dw[u][p], gv, 0, xs, cols[p]);
        }
    }
}

// Loads are branch-free: row positions past the range are clamped to its last row and their gradients
// zeroed, so the compiler issues every load of a step back to back instead of one masked load at a time. A
// wave fetches the row ids of its next step in one coalesced load (lane l: id l) while it works on the current
// step, and hands them out with a shuffle. WIDE: the slab's rows are W / 4 two-byte bins. PACK: the slab's rows
// are W * PACK bytes, PACK features of at most 256 / PACK bins to an LDS column. SUB: the columns a workgroup takes of its
// rows; W / SUB workgroups share a row range, each reading its dwords of every row.
template <int W, bool WIDE = false, int PACK = 1, bool Q32 = false, int DP = 0, int SUB = W>
__global__ __launch_bounds__(1024) void k_hist(HistArgs a) {
    static_assert(PACK == 1 || (!WIDE && W * PACK <= 256), "a packed row is at most 64 dwords");
    static_assert(!Q32 || W <= 64, "separate g and h counters take twice the LDS");
    static_assert(DP == 0 || (W == 128 && !WIDE && PACK == 1 && !Q32), "a dense slab has 128 byte columns");
    static_assert(SUB == W || (!WIDE && PACK == 1 && !Q32 && DP == 0), "only byte slabs go by column parts");
    constexpr int PARTS = W / SUB;                      // workgroups that share a row range, each with SUB of the columns
    constexpr int ROW = WIDE ? W / 8 : W * PACK / 4;    // dwords per row
    constexpr int DW = ROW / PARTS;                     // of them, this workgroup's
    constexpr int RPW = WAVE / DW;            // rows per wave step
    // row ids of one step fit one wave-wide load; at W = 128 the 64 accumulator registers leave room for 8
    constexpr int UNROLL = SUB == 128 ? 8 : (64 / RPW < 16 ? 64 / RPW : 16);
    constexpr uint32_t STEP = 16u * RPW * UNROLL;          // rows per block step (16 waves)
    constexpr int SLOTS = 256 * SUB / 1024;
    constexpr int LDS_WORDS = (Q32 ? 2 : 1) * 256 * SUB + (DP ? W : 0);  // a dense slab's spare row
    __shared__ int32_t lds[LDS_WORDS];

    uint32_t lb, n;
    leaf_rows(a.dev_left, a.begin, a.count, a.side, lb, n);
    uint32_t groups, per;
    hist_split(n, a.max_groups, a.min_rows_per_group, groups, per);
    // the parts of a row range 8 workgroups apart, so on one XCD: its L2 serves a row's line to all but the first
    const uint32_t group = PARTS == 1 ? blockIdx.x : blockIdx.x / (8u * PARTS) * 8u + blockIdx.x % 8u;
    const uint32_t part = PARTS == 1 ? 0u : blockIdx.x / 8u % PARTS;
    if (group >= groups) return;
    const bool packed = !Q32 && per <= a.flush_rows;  // the partial is the packed words themselves
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = tid; k < static_cast<uint32_t>(LDS_WORDS); k += 1024) lds[k] = 0;
    int32_t accg[SLOTS], acch[SLOTS];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) accg[j] = acch[j] = 0;
    __syncthreads();

    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const uint32_t d = lane % DW, rsub = lane / DW;
    const uint32_t rot = (lane & 31u) >> 3;
    uint32_t xs[4], cols[4];
    row_bin_lanes<SUB, PACK>(d, rot, xs, cols);
    const uint32_t *rows = a.rows + lb;
    const uint32_t *bins32 = reinterpret_cast<const uint32_t *>(a.bins) + part * DW;
    uint32_t start = group * per;
    uint32_t end = start + per < n ? start + per : n;
    uint32_t dcols[DP ? DP : 1][4];
    if constexpr (DP > 0) dense_lanes<DP>(a.pos_word, lane, xs, dcols);

    for (uint32_t chunk = start; chunk < end; chunk += a.flush_rows) {
        uint32_t cend = end - chunk > a.flush_rows ? chunk + a.flush_rows : end;
        if constexpr (DP > 0) {
            hist_list_dense<W, DP>(lds, rows, chunk, cend, a.gh, bins32, a.dw_row, xs, dcols);
        } else {
            uint32_t last = cend - 1;
            uint32_t base = chunk + wave * RPW * UNROLL;
            uint32_t cidx = rows[min(base + lane, last)];
            for (; base < cend; base += STEP) {
                uint32_t r[UNROLL];
#pragma unroll
                for (int u = 0; u < UNROLL; ++u) r[u] = __shfl(cidx, u * RPW + rsub);
                cidx = rows[min(base + STEP + lane, last)];
                uint32_t dw[UNROLL];
                int32_t g[UNROLL];
#pragma unroll
                for (int u = 0; u < UNROLL; ++u) {
                    g[u] = a.gh[r[u]];
                    dw[u] = bins32[(size_t)r[u] * ROW + d];
                }
#pragma unroll
                for (int u = 0; u < UNROLL; ++u) {
                    int32_t gv, hv;
                    row_units<Q32>(g[u], base + u * RPW + rsub < cend, gv, hv);
                    if constexpr (WIDE) add_row_bins_wide<W, Q32>(lds, dw[u], gv, hv, d);
                    else add_row_bins<SUB, PACK, Q32>(lds, dw[u], gv, hv, xs, cols);
                }
            }
        }
        __syncthreads();
        if (packed) break;  // the only chunk
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) {
            int32_t v = lds[tid + j * 1024];
            lds[tid + j * 1024] = 0;
            if constexpr (Q32) {
                accg[j] += v;
                acch[j] += lds[256 * W + tid + j * 1024];
                lds[256 * W + tid + j * 1024] = 0;
            } else {
                const int32_t gq = packed_g(v);
                accg[j] += gq;
                acch[j] += packed_h(v, gq);
            }
        }
        __syncthreads();
    }
    // the slot of LDS word k: bin k / SUB, column part * SUB + k % SUB
    int32_t *mine = a.partial + static_cast<size_t>(group) * (2 * 256 * W);
    if (packed) {
#pragma unroll
        for (int j = 0; j < SLOTS; ++j) {
            const uint32_t k = tid + j * 1024;
            mine[k / SUB * W + part * SUB + k % SUB] = lds[k];
        }
        return;
    }
    int2 *out = reinterpret_cast<int2 *>(mine);
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
        const uint32_t k = tid + j * 1024;
        out[k / SUB * W + part * SUB + k % SUB] = make_int2(accg[j], acch[j]);
    }
}

// Adds the partials of one slab into the leaf histogram (i64 {g, h} per bin, flat layout). Thread per slab slot
// (bin * W + column); `col_offset[column]` is the column's feature's first bin in the flat histogram,
// `col_bins[column]` its bin count (0 for padding). When `parent` is non-null, also writes the sibling:
// sibling[bin] = parent[bin] - built[bin] (learner.rs:356-371), in place of the parent.
struct ReduceArgs {
    const int32_t *partial;
    const uint32_t *col_offset;
    const uint32_t *col_bins;
    const uint32_t *col_stride;  // flat-histogram bins between a column's consecutive bins: 1, or 4 (wide slab)
    int64_t *out;       // built child's histogram
    int64_t *parent;    // parent's histogram, overwritten with the sibling's (or null)
    const uint32_t *dev_left;
    uint32_t begin, count, side;
    uint32_t max_groups, min_rows_per_group;
    uint32_t packed_rows; // partials of at most this many rows are packed words (k_hist)
    uint32_t width;     // W
    uint32_t seg_shift; // a packed slab's column holds a feature each 2^seg_shift bins: 8 (one feature), 7 or 6
    const uint32_t *slot_flat;  // a dense slab: per slot (bin * W + column) its flat-histogram bin + 1, 0 for none
};

// A block takes 32 slots (bin * W + column) and splits the workgroups' partials of each into 8 stripes that meet in
// LDS. grid: ceil(256 * W / 32) blocks of 256 threads.
__global__ __launch_bounds__(256) void k_hist_reduce(ReduceArgs a) {
    __shared__ int64_t red[2][8][32];
    uint32_t lb, n;
    leaf_rows(a.dev_left, a.begin, a.count, a.side, lb, n);
    uint32_t groups, per;
    hist_split(n, a.max_groups, a.min_rows_per_group, groups, per);
    const uint32_t slots = 256u * a.width;
    const uint32_t tid = threadIdx.x, lane = tid & 31u, stripe = tid >> 5;
    const uint32_t s = blockIdx.x * 32u + lane, col = s % a.width, bin = s / a.width;
    // the slot's feature: segment bin >> seg_shift of the column (its index in the per-feature arrays), its bin;
    // in a dense slab the slot's flat bin from the table
    const uint32_t vb = bin & ((1u << a.seg_shift) - 1u), fs = (bin >> a.seg_shift) * a.width + col;
    const uint32_t flat1 = a.slot_flat && s < slots ? a.slot_flat[s] : 0u;
    const bool on = s < slots && (a.slot_flat ? flat1 != 0u : vb < a.col_bins[fs]);
    int64_t g = 0, h = 0;
    if (on) {
        if (per <= a.packed_rows) {
            const int32_t *p = a.partial + s;
#pragma unroll 8
            for (uint32_t w = stripe; w < groups; w += 8u) {
                const int32_t v = p[2 * static_cast<size_t>(w) * slots], gq = packed_g(v);
                g += gq;
                h += packed_h(v, gq);
            }
        } else {
            const int2 *p = reinterpret_cast<const int2 *>(a.partial) + s;
#pragma unroll 8
            for (uint32_t w = stripe; w < groups; w += 8u) {
                const int2 v = p[static_cast<size_t>(w) * slots];
                g += v.x;
                h += v.y;
            }
        }
    }
    red[0][stripe][lane] = g;
    red[1][stripe][lane] = h;
    __syncthreads();
    if (stripe == 0 && on) {
#pragma unroll
        for (int k = 1; k < 8; ++k) {
            g += red[0][k][lane];
            h += red[1][k][lane];
        }
        const size_t o = a.slot_flat ? 2 * static_cast<size_t>(flat1 - 1u)
                                     : 2 * (static_cast<size_t>(a.col_offset[fs]) + static_cast<size_t>(vb) * a.col_stride[fs]);
        a.out[o] = g;
        a.out[o + 1] = h;
        if (a.parent) {
            a.parent[o] -= g;
            a.parent[o + 1] -= h;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// Stable partition (cpu.rs:556-599) of a leaf's rows by a BinSplit, through a second buffer.
// Pass 1 counts each block's left rows; pass 2 recomputes every block's offset from those counts, compacts
// stably within the block (wave ballots + an LDS prefix over waves) and scatters; pass 3 copies back.
// Predicate: the bin of the split feature (column-major bins `col`) is set in `left_bins`; or, for bagging,
// quantize.rs:147-149 `in_bag` of the row.
// ---------------------------------------------------------------------------------------------------------

struct PartArgs {
    const uint32_t *src;   // rows
    uint32_t *dst;
    const uint8_t *col;    // column-major bins of the split feature (null: bagging predicate)
    uint32_t col16, wide;  // u16 column-major bins; the split is a wide feature's numerical rule
    uint32_t *block_left;  // [grid]
    uint32_t *dev_left;    // total left count (written by block 0 of pass 2)
    uint32_t *host_left;   // and in the host's pinned memory (or null)
    uint32_t begin, count;
    uint32_t left_bins[8];
    // bagging
    uint32_t bag_seed, bag_round;
    uint64_t row_offset;
    double fraction;
};

// Rows per block for `count` rows over the launch's blocks: a multiple of 256, the same in both passes.
__device__ __forceinline__ uint32_t part_per_block(uint32_t count, uint32_t blocks) {
    uint32_t per = (count + blocks - 1) / blocks;
    per = (per + 1023u) & ~1023u;
    return per < 1024u ? 1024u : per;
}

__device__ __forceinline__ bool part_left(const PartArgs &a, uint32_t row) {
    if (a.col) return rule_left(a.left_bins, a.wide, col_bin(a.col, a.col16, row));
    return static_cast<double>(uniform(a.bag_seed, 2u, a.bag_round, a.row_offset + row)) < a.fraction;
}

// Tiles of 1024 rows: thread t takes rows t, t+256, t+512, t+768 of the tile (four sub-tiles of 256 in order),
// with every load of the tile issued before any is used (positions past the range are clamped and ignored).
__global__ __launch_bounds__(256) void k_part_count(PartArgs a) {
    __shared__ uint32_t wsum[4];
    const uint32_t per_block = part_per_block(a.count, gridDim.x);
    const uint32_t active = (a.count + per_block - 1) / per_block;
    if (blockIdx.x >= active && blockIdx.x > 0) return;
    const uint32_t start = blockIdx.x * per_block;
    const uint32_t end = start + per_block < a.count ? start + per_block : a.count;
    uint32_t c = 0;
    for (uint32_t tile = start; tile < end; tile += 1024) {
        uint32_t row[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) row[j] = a.src[a.begin + min(tile + j * 256 + threadIdx.x, end - 1)];
#pragma unroll
        for (int j = 0; j < 4; ++j) c += (tile + j * 256 + threadIdx.x < end && part_left(a, row[j])) ? 1u : 0u;
    }
    for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) a.block_left[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
}

__global__ __launch_bounds__(256) void k_part_scatter(PartArgs a) {
    __shared__ uint32_t red[2][4];
    __shared__ uint32_t wl[4][4];  // [sub-tile][wave] left counts
    const uint32_t per_block = part_per_block(a.count, gridDim.x);
    uint32_t active = (a.count + per_block - 1) / per_block;
    if (active == 0) active = 1;
    if (blockIdx.x >= active) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    // lefts before this block, and in total
    uint32_t before = 0, total = 0;
    for (uint32_t j = tid; j < active; j += 256) {
        uint32_t v = a.block_left[j];
        total += v;
        if (j < blockIdx.x) before += v;
    }
    for (int o = 32; o >= 1; o >>= 1) {
        before += __shfl_xor(before, o);
        total += __shfl_xor(total, o);
    }
    if (lane == 0) {
        red[0][wave] = before;
        red[1][wave] = total;
    }
    __syncthreads();
    before = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    total = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    if (blockIdx.x == 0 && tid == 0) {
        *a.dev_left = total;
        if (a.host_left) *a.host_left = total;
    }
    const uint32_t start = blockIdx.x * per_block;
    const uint32_t end = start + per_block < a.count ? start + per_block : a.count;
    uint32_t lpos = before;                    // next left slot (relative to begin)
    uint32_t rpos = total + (start - before);  // next right slot
    const uint64_t below_mask = (1ull << lane) - 1ull;
    for (uint32_t tile = start; tile < end; tile += 1024) {
        uint32_t row[4];
        bool ok[4], left[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t i = tile + j * 256 + tid;
            ok[j] = i < end;
            row[j] = a.src[a.begin + min(i, end - 1)];
        }
        uint32_t below[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            left[j] = ok[j] && part_left(a, row[j]);
            uint64_t m = __ballot(left[j]);
            below[j] = __popcll(m & below_mask);
            if (lane == 0) wl[j][wave] = static_cast<uint32_t>(__popcll(m));
        }
        __syncthreads();
        uint32_t lsub = 0;  // lefts in the sub-tiles before j
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t sub_start = tile + j * 256;
            uint32_t sub_valid = sub_start < end ? (end - sub_start < 256u ? end - sub_start : 256u) : 0u;
            uint32_t lbefore = 0, sub_left = 0;
            for (uint32_t w = 0; w < 4; ++w) {
                if (w < wave) lbefore += wl[j][w];
                sub_left += wl[j][w];
            }
            if (ok[j]) {
                uint32_t lrank = lsub + lbefore + below[j];  // lefts before this row in the tile
                if (left[j]) {
                    a.dst[a.begin + lpos + lrank] = row[j];
                } else {
                    uint32_t rrank = (sub_start - tile) + tid - lrank;  // rights before this row in the tile
                    a.dst[a.begin + rpos + rrank] = row[j];
                }
            }
            lsub += sub_left;
            (void)sub_valid;
        }
        uint32_t tile_valid = end - tile < 1024u ? end - tile : 1024u;
        lpos += lsub;
        rpos += tile_valid - lsub;
        __syncthreads();
    }
}

__global__ void k_copy_u32(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, uint32_t begin, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        dst[begin + i] = src[begin + i];
}

// ---------------------------------------------------------------------------------------------------------
// leaf_sums (cpu.rs:886-908): exact fixed-point sums rint(v * scale) per leaf (quantize.rs:163-165)
// ---------------------------------------------------------------------------------------------------------

__device__ __forceinline__ int64_t to_fixed(float v, float scale) {
    float p = __builtin_rintf(v * scale);
    return sat_i64(static_cast<double>(p));
}

// A block's share of one leaf: at most LEAF_SUM_ROWS of its rows.
struct LeafJob {
    uint32_t begin, count, leaf;
};

// Eight rows a thread, their ids and then their gathers all in flight, met in LDS and added by one pair of atomics a block:
// what bounds it is the latency of the gathers (blocks of 8192 rows, one row a thread at a time, one block a compute unit:
// 2.25M rows in 2 leaves 57 -> 24 us, 7.5k rows 11.3 -> 4.5 us). grid: the jobs, 256 threads.
constexpr uint32_t LEAF_SUM_ROWS = 2048;
__global__ __launch_bounds__(256) void k_leaf_sums(const float *__restrict__ grad, const float *__restrict__ hess,
                                                   const uint32_t *__restrict__ partition, const LeafJob *jobs,
                                                   float gs, float hs, unsigned long long *out) {
    constexpr uint32_t RPT = LEAF_SUM_ROWS / 256u;
    __shared__ int64_t part[2][4];
    const LeafJob j = jobs[blockIdx.x];
    uint32_t r[RPT];
    float g[RPT], h[RPT];
#pragma unroll
    for (uint32_t k = 0; k < RPT; ++k) r[k] = partition[j.begin + min(threadIdx.x + 256u * k, j.count - 1u)];
#pragma unroll
    for (uint32_t k = 0; k < RPT; ++k) {
        g[k] = grad[r[k]];
        h[k] = hess[r[k]];
    }
    int64_t sg = 0, sh = 0;
#pragma unroll
    for (uint32_t k = 0; k < RPT; ++k) {
        if (threadIdx.x + 256u * k >= j.count) continue;
        sg += to_fixed(g[k], gs);
        sh += to_fixed(h[k], hs);
    }
    for (int o = 32; o >= 1; o >>= 1) {
        sg += __shfl_xor(sg, o);
        sh += __shfl_xor(sh, o);
    }
    if ((threadIdx.x & 63u) == 0u) {
        part[0][threadIdx.x >> 6] = sg;
        part[1][threadIdx.x >> 6] = sh;
    }
    __syncthreads();
    if (threadIdx.x < 2u) {
        const int64_t *p = part[threadIdx.x];
        atomicAdd(out + 2 * j.leaf + threadIdx.x, static_cast<unsigned long long>(p[0] + p[1] + p[2] + p[3]));
    }
}

// ---------------------------------------------------------------------------------------------------------
// add_tree (cpu.rs:666-695): walk each row down the tree on column-major bins, score += leaf value (f32)
// ---------------------------------------------------------------------------------------------------------

struct DevNode {
    uint32_t left_bins[8];
    uint32_t feature;  // index of the feature's column-major bins
    int32_t left, right;
    uint32_t wide;     // left_bins hold a numerical rule (rule_left)
};

// `gate` (when set): the leaves of the tree to add, 0 for none (k_tree_nodes).
__global__ void k_add_tree(const uint8_t *__restrict__ colbins, uint32_t col16, uint64_t rows,
                           const DevNode *__restrict__ nodes, const float *__restrict__ leaf_values,
                           float *__restrict__ scores, const uint32_t *gate) {
    if (gate && *gate == 0u) return;
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x) {
        int32_t node = 0;
        while (node >= 0) {
            const DevNode &nd = nodes[node];
            const uint32_t bin = col_bin(colbins, col16, (size_t)nd.feature * rows + r);
            node = rule_left(nd.left_bins, nd.wide, bin) ? nd.left : nd.right;
        }
        scores[r] += leaf_values[~node];
    }
}

// Each row's leaf from a walk down the tree (nodes in LDS; several rows per thread in flight: the walk is a chain
// of dependent gathers), in row order, and the leaves' exact fixed-point sums rint(v * scale) of the in-bag rows'
// gradients: the sums k_leaf_sums makes over the final partition (integers, so the order does not matter;
// cpu.rs:886-908). grid: any, tl_threads<MAXL>() threads.
struct TreeLeavesArgs {
    const uint8_t *colbins;            // column-major bins [feature][rows]
    uint32_t col16;                    // two bytes per bin
    uint64_t rows;
    const DevNode *nodes;
    uint32_t nn, nl;                   // internal nodes, leaves (nn >= 1, nl <= the kernel's MAXL)
    uint16_t *leaf_of;                 // [rows]
    const float *grad, *hess;          // null: no sums
    float gs, hs;
    unsigned long long *sums;          // [nl][2], zeroed before
    uint32_t bag, bag_seed, bag_round; // bag != 0: only rows in the bag (quantize.rs:147-149) are summed
    uint64_t row_offset;
    double fraction;
    const uint32_t *gate;              // when set: the leaves (nn, nl from it), 0 for no tree (k_tree_nodes)
    const DevScales *dsc;              // when set: gs and hs are its fixed-point scales
};
// Instantiated for trees of up to 512 leaves (28 KiB of LDS: several blocks per compute unit) and up to 2048 (112 KiB:
// one block per compute unit, of 1024 threads, so that 16 waves walk at once). The walk is a chain of dependent
// LDS reads and gathers; its rate is set by the rows in flight, which the register file bounds: 8 rows a thread
// keeps the 512-leaf kernel at 70 registers (7 waves a SIMD), 12 the 2048-leaf one at 124 (4 waves a SIMD, which
// its one block a compute unit fills).
constexpr uint32_t LEAVES_SMALL = 512;
template <uint32_t MAXL> constexpr uint32_t tl_threads() { return MAXL > LEAVES_SMALL ? 1024u : 512u; }
template <uint32_t MAXL> constexpr int tl_rows() { return MAXL > LEAVES_SMALL ? 12 : 8; }

// RPT rows a thread walked down the tree to their leaves (nd: 0 for a row to walk, -1 for none; ~leaf after). A level is
// branch-free over the rows, so that their LDS reads and gathers issue back to back and each kind waits once: every row
// reads its node's head (x: its feature's column, bit 31 set for a numerical rule; y: its left and right children as two
// i16, a leaf l as ~l), gathers its bin, then reads the rule word the bin selects. A row already at its leaf reads node 0
// and row 0 and keeps its leaf. The rule words are word-major (word w of node n at w * NN + n).
template <int RPT, bool COL16, uint32_t NN>
__device__ __forceinline__ void walk_rows(const uint2 *head, const uint32_t *rule, const uint8_t *__restrict__ colbins, uint32_t rows,
                                          const uint32_t (&r)[RPT], int32_t (&nd)[RPT]) {
    for (;;) {
        uint2 h[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) h[k] = head[nd[k] < 0 ? 0 : nd[k]];
        uint32_t b[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const size_t i = static_cast<size_t>(h[k].x & 0x7fffffffu) * rows + (nd[k] < 0 ? 0u : r[k]);
            b[k] = COL16 ? static_cast<uint32_t>(reinterpret_cast<const uint16_t *>(colbins)[i]) : static_cast<uint32_t>(colbins[i]);
        }
        uint32_t m0[RPT], m1[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const uint32_t n = nd[k] < 0 ? 0u : static_cast<uint32_t>(nd[k]);
            const uint32_t w = COL16 ? (h[k].x >> 31 ? 0u : min(b[k] >> 5, 7u)) : b[k] >> 5;
            m0[k] = rule[w * NN + n];
            if (COL16) m1[k] = rule[NN + n];
        }
        bool any = false;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            bool left = ((m0[k] >> (b[k] & 31u)) & 1u) != 0u;
            // rule_left's numerical rule: word 0 the threshold, word 1 the NaN bin + 1 or 0
            if (COL16 && (h[k].x >> 31)) left = b[k] <= m0[k] || (m1[k] != 0u && b[k] == m1[k] - 1u);
            const int32_t c = static_cast<int32_t>(static_cast<int16_t>(left ? h[k].y & 0xffffu : h[k].y >> 16));
            nd[k] = nd[k] < 0 ? nd[k] : c;
            any = any || nd[k] >= 0;
        }
        if (!any) break;
    }
}

// The tree's nodes into LDS as walk_rows reads them, by the whole block.
template <uint32_t NN>
__device__ __forceinline__ void stage_nodes(const DevNode *nodes, uint32_t nn, uint2 *head, uint32_t *rule) {
    for (uint32_t k = threadIdx.x; k < nn; k += blockDim.x) {
        const DevNode &x = nodes[k];
        head[k] = make_uint2(x.feature | (x.wide ? 0x80000000u : 0u),
                             (static_cast<uint32_t>(x.left) & 0xffffu) | (static_cast<uint32_t>(x.right) << 16));
#pragma unroll
        for (int w = 0; w < 8; ++w) rule[w * NN + k] = x.left_bins[w];
    }
}

// COL16: two-byte column-major bins (the only kind with numerical rules, `wide`).
template <uint32_t MAXL, bool COL16>
__global__ __launch_bounds__(tl_threads<MAXL>()) void k_tree_leaves(TreeLeavesArgs a) {
    constexpr int RPT = tl_rows<MAXL>();
    constexpr uint32_t NN = MAXL - 1;
    __shared__ uint2 head[NN];
    __shared__ uint32_t rule[8 * NN];
    __shared__ unsigned long long ls[MAXL][2];
    uint32_t nn = a.nn, nl = a.nl;
    const float gs = a.dsc ? a.dsc->gsc : a.gs, hs = a.dsc ? a.dsc->hsc : a.hs;
    if (a.gate) {
        nl = *a.gate;
        if (nl == 0u || nl > MAXL) return;
        nn = nl - 1u;
    }
    stage_nodes<NN>(a.nodes, nn, head, rule);
    if (a.grad)
        for (uint32_t l = threadIdx.x; l < nl; l += blockDim.x) ls[l][0] = ls[l][1] = 0ull;
    __syncthreads();
    const uint32_t rows = static_cast<uint32_t>(a.rows);  // rows < 2^32 (row ids are u32)
    const uint32_t step = gridDim.x * blockDim.x;
    for (uint64_t base = blockIdx.x * blockDim.x + threadIdx.x; base < rows; base += static_cast<uint64_t>(RPT) * step) {
        uint32_t r[RPT];
        int32_t nd[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const uint64_t row = base + static_cast<uint64_t>(k) * step;
            r[k] = row < rows ? static_cast<uint32_t>(row) : 0u;
            nd[k] = row < rows ? 0 : -1;
        }
        walk_rows<RPT, COL16, NN>(head, rule, a.colbins, rows, r, nd);
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            if (base + static_cast<uint64_t>(k) * step >= rows) continue;
            const uint32_t leaf = static_cast<uint32_t>(~nd[k]);
            a.leaf_of[r[k]] = static_cast<uint16_t>(leaf);
            if (!a.grad) continue;
            if (a.bag && !(static_cast<double>(uniform(a.bag_seed, 2u, a.bag_round, a.row_offset + r[k])) < a.fraction)) continue;
            atomicAdd(&ls[leaf][0], static_cast<unsigned long long>(to_fixed(a.grad[r[k]], gs)));
            atomicAdd(&ls[leaf][1], static_cast<unsigned long long>(to_fixed(a.hess[r[k]], hs)));
        }
    }
    if (!a.grad) return;
    __syncthreads();
    for (uint32_t l = threadIdx.x; l < nl; l += blockDim.x) {
        if (ls[l][0]) atomicAdd(&a.sums[2 * l], ls[l][0]);
        if (ls[l][1]) atomicAdd(&a.sums[2 * l + 1], ls[l][1]);
    }
}

// k_add_tree for many rows and trees of up to 512 leaves: the walk of k_tree_leaves, the scores read before it and the
// leaves' values in LDS, where k_add_tree waits for three dependent loads a level for one row (3M x 40: 127 leaves 87 -> 38 us,
// 511 leaves 109 -> 50 us). grid: any, tl_threads<LEAVES_SMALL>() threads.
template <bool COL16>
__global__ __launch_bounds__(tl_threads<LEAVES_SMALL>()) void k_add_tree_walk(const uint8_t *__restrict__ colbins, uint32_t rows,
                                                                              const DevNode *nodes, uint32_t nl,
                                                                              const float *__restrict__ leaf_values,
                                                                              float *__restrict__ scores, const uint32_t *gate) {
    constexpr uint32_t MAXL = LEAVES_SMALL;
    constexpr int RPT = tl_rows<MAXL>();
    constexpr uint32_t NN = MAXL - 1;
    __shared__ uint2 head[NN];
    __shared__ uint32_t rule[8 * NN];
    __shared__ float value[MAXL];
    if (gate) nl = *gate;
    if (nl == 0u || nl > MAXL) return;
    stage_nodes<NN>(nodes, nl - 1u, head, rule);
    for (uint32_t l = threadIdx.x; l < nl; l += blockDim.x) value[l] = leaf_values[l];
    __syncthreads();
    const uint32_t step = gridDim.x * blockDim.x;
    for (uint64_t base = blockIdx.x * blockDim.x + threadIdx.x; base < rows; base += static_cast<uint64_t>(RPT) * step) {
        uint32_t r[RPT];
        int32_t nd[RPT];
        float old[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const uint64_t row = base + static_cast<uint64_t>(k) * step;
            r[k] = row < rows ? static_cast<uint32_t>(row) : 0u;
            nd[k] = row < rows ? 0 : -1;
            old[k] = scores[r[k]];
        }
        walk_rows<RPT, COL16, NN>(head, rule, colbins, rows, r, nd);
#pragma unroll
        for (int k = 0; k < RPT; ++k)
            if (base + static_cast<uint64_t>(k) * step < rows) scores[r[k]] = old[k] + value[~nd[k]];
    }
}

// scores[r] += the value of row r's leaf: the f32 add of k_add_tree, in row order. Four rows of the grid-stride loop
// at once, their loads (then their leaves' values) issued together: one row an iteration waited on its loads and then
// on its leaf's value (21.0 -> 18.4 us at 10M rows; the gradient kernels, bound by their f64 arithmetic, were slower
// so).
__global__ void k_add_leaf_values(const uint16_t *__restrict__ leaf_of, const float *__restrict__ leaf_values,
                                  float *__restrict__ scores, uint64_t rows, const uint32_t *gate) {
    constexpr int RA = 4;
    if (gate && *gate == 0u) return;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t r0 = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r0 < rows; r0 += RA * stride) {
        uint32_t l[RA];
        float s[RA], v[RA];
#pragma unroll
        for (int k = 0; k < RA; ++k) {
            const uint64_t r = r0 + k * stride;
            l[k] = r < rows ? leaf_of[r] : 0u;
            s[k] = r < rows ? scores[r] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < RA; ++k) v[k] = r0 + k * stride < rows ? leaf_values[l[k]] : 0.0f;
#pragma unroll
        for (int k = 0; k < RA; ++k) {
            const uint64_t r = r0 + k * stride;
            if (r < rows) scores[r] = s[k] + v[k];
        }
    }
}

// a -= b over n int64 values (a histogram slot minus another, learner.rs:365-367)
__global__ void k_sub_i64(int64_t *__restrict__ a, const int64_t *__restrict__ b, uint64_t n) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        a[i] -= b[i];
}

__global__ void k_add_const(float *__restrict__ scores, uint64_t rows, float v) {
    for (uint64_t r = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x)
        scores[r] += v;
}

// ---------------------------------------------------------------------------------------------------------
// Best-split search (split.rs:201-961) for numerical features, one wave per (leaf, feature).
//
// A scan's running sums are sums of exact integers (quantized units and rounded per-bin counts), so a parallel
// prefix over the wave gives the same f64/i64 values as the reference's sequential loop. Every per-candidate
// value (hessians, constraints, the stopping candidate, gains) is then the same IEEE operation on the same
// operands; the best is the first maximum (NaN never wins), as ScanBuffer::best (split.rs:508-531).
// ---------------------------------------------------------------------------------------------------------

struct SplitCfgDev {
    int64_t min_data_in_leaf;
    double min_sum_hessian_in_leaf, lambda_l1, lambda_l2, min_gain_to_split;
    uint64_t max_cat_to_onehot, max_cat_threshold;
    double cat_l2, cat_smooth;
    int64_t min_data_per_group;
};

struct Ctx {
    double units_grad, units_hess;
    int64_t num_data;
    double scale_grad, scale_hess;
    double sum_grad, sum_hess, cnt_factor, min_gain_shift;
    bool valid;
};

// split.rs:159-162
__device__ __forceinline__ double leaf_gain(double g, double h, double l1, double l2) {
    double r = max_num(__builtin_fabs(g) - l1, 0.0);
    return r * r / (h + l2);
}

// split.rs:145-154, 190-192
__device__ __forceinline__ double leaf_output(double g, double h, double l1, double l2) {
    double reg = max_num(__builtin_fabs(g) - l1, 0.0);
    double sign = static_cast<double>(static_cast<int>(g > 0.0) - static_cast<int>(g < 0.0));
    return -(sign * reg) / (h + l2);
}

// The renewed leaf values of a grown tree from its leaves' fixed-point sums (learner.rs:376-404), shrunk by the
// learning rate (tree.rs:180-185) and, for the first tree, moved by the initial score (tree.rs:188-193, with the
// f32 values added to the scores taken without it: replay.rs:38-40): the host's double operations, in its order.
// One block; leaf l: value[l], weight[l] (double) and lv[l] (the f32 added to the scores).
struct LeafValueArgs {
    const unsigned long long *sums;  // [nl][2] i64 fixed-point {g, h}
    const uint32_t *gate;            // when set: nl from it, 0 for no tree (k_tree_nodes)
    const DevScales *dsc;            // when set: gs and hs are its fixed-point scales
    uint32_t nl, add_bias;
    float gs, hs;                    // the fixed-point scales
    double l1, l2, rate, bias;
    double *value, *weight;
    float *lv;
};

__device__ __forceinline__ double round_to_zero_d(double v) { return fabs(v) > static_cast<double>(1e-35f) ? v : 0.0; }

__global__ void k_leaf_values(LeafValueArgs a) {
    const uint32_t nl = a.gate ? *a.gate : a.nl;
    const float gs = a.dsc ? a.dsc->gsc : a.gs, hs = a.dsc ? a.dsc->hsc : a.hs;
    for (uint32_t l = threadIdx.x; l < nl; l += blockDim.x) {
        const double sg = static_cast<double>(static_cast<int64_t>(a.sums[2 * l])) / static_cast<double>(gs);
        const double sh = static_cast<double>(static_cast<int64_t>(a.sums[2 * l + 1])) / static_cast<double>(hs);
        double v = round_to_zero_d(leaf_output(sg, sh, a.l1, a.l2));
        v = round_to_zero_d(v * a.rate);
        float f = static_cast<float>(v);
        if (a.add_bias) {
            v = round_to_zero_d(v + a.bias);
            f = static_cast<float>(v - a.bias);
        }
        a.value[l] = v;
        a.weight[l] = sh;
        a.lv[l] = f;
    }
}


// split.rs:214-233 LeafCtx::new
__device__ __forceinline__ Ctx make_ctx(const SplitCfgDev &cfg, double sg, double sh, double ug, double uh, int64_t count) {
    Ctx c;
    c.valid = !(uh != uh || uh <= 0.0 || count <= 0);
    c.units_grad = ug;
    c.units_hess = uh;
    c.num_data = count;
    c.scale_grad = sg;
    c.scale_hess = sh;
    c.sum_grad = ug * sg;
    c.sum_hess = uh * sh + 2.0 * K_EPSILON;
    double gain_shift = leaf_gain(c.sum_grad, c.sum_hess, cfg.lambda_l1, cfg.lambda_l2);
    c.cnt_factor = static_cast<double>(count) / c.sum_hess;
    c.min_gain_shift = gain_shift + cfg.min_gain_to_split;
    return c;
}

// A feature's best candidate (split.rs:298-317) as the search writes it per (leaf, feature).
struct FeatCand {
    int32_t found;        // a candidate exists
    int32_t splittable;   // any scan had a valid candidate
    double gain;          // best.gain - min_gain_shift
    double best_gain;     // the candidate's own split gain
    uint32_t threshold;
    uint32_t default_left;
    double left_grad, left_hess;
    int64_t left_count;
    double left_units_g, left_units_h;
    uint32_t col;         // the feature's column-major index (its bins for the partition)
    uint32_t nan_idx;     // its NaN bin, or NO_BIN
    uint32_t wide;        // it has two-byte bins (rule_left)
    uint32_t rule;        // RULE_NUMERICAL, RULE_ONEHOT or RULE_SORTED
    uint32_t cat_forward; // sorted categorical: the run went from the low end of the sorted order
    uint32_t cat_count;   // categorical: bins going left
    uint32_t cat_mask[8]; // categorical: the bins going left
};

constexpr uint32_t NO_BIN = 0xffffffffu;
constexpr uint32_t RULE_NUMERICAL = 0, RULE_ONEHOT = 1, RULE_SORTED = 2;  // split.rs:112-117, 694-844

struct Grown {
    uint32_t bin;
    double ug, uh;
    int64_t count;
    double gain;
};

// Wave-wide inclusive scans with DPP row operations (gfx9: row_shr within rows of 16 lanes, then row_bcast:15
// and row_bcast:31 across rows): each step is a VALU move, not an LDS permute.
constexpr int DPP_ROW_SHR1 = 0x111, DPP_ROW_SHR2 = 0x112, DPP_ROW_SHR4 = 0x114, DPP_ROW_SHR8 = 0x118;
constexpr int DPP_ROW_BCAST15 = 0x142, DPP_ROW_BCAST31 = 0x143;

// The value of the lane the DPP step reads (0 where the step has no source or leaves the lane unwritten).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROW_MASK, 0xf, true));
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
    uint32_t lo = dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(v));
    uint32_t hi = dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}
__device__ __forceinline__ uint64_t bits_of(double x) { return __builtin_bit_cast(uint64_t, x); }
__device__ __forceinline__ double double_of(uint64_t x) { return __builtin_bit_cast(double, x); }

// Whether step CTRL/ROW_MASK gives `lane` a source lane (the steps of an inclusive scan, in order).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ bool dpp_has_source(uint32_t lane) {
    const uint32_t row = lane >> 4, in_row = lane & 15u;
    if (CTRL >= DPP_ROW_SHR1 && CTRL <= DPP_ROW_SHR1 + 14) return in_row >= static_cast<uint32_t>(CTRL - 0x110);
    return (ROW_MASK >> row) & 1u;
}

// Inclusive sums over the wave of three exact (integer-valued) quantities.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void scan_add_step(double &g, double &h, int64_t &c) {
    g += double_of(dpp_u64<CTRL, ROW_MASK>(bits_of(g)));
    h += double_of(dpp_u64<CTRL, ROW_MASK>(bits_of(h)));
    c += static_cast<int64_t>(dpp_u64<CTRL, ROW_MASK>(static_cast<uint64_t>(c)));
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, uint32_t lane) {
    uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v)), lane));
    uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v >> 32)), lane));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// (gain, feature) order of split.rs:866-880 for reductions: a beats b on higher gain, then lower feature; -1 is
// "no candidate".
__device__ __forceinline__ bool cand_better(double ga, int fa, double gb, int fb) {
    return fa >= 0 && (fb < 0 || ga > gb || (ga == gb && fa < fb));
}

// Wave-wide all-reductions through the DPP scan steps; every lane ends with the result.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void best_step(double &g, int &i, uint32_t lane) {
    double og = double_of(dpp_u64<CTRL, ROW_MASK>(bits_of(g)));
    int oi = static_cast<int>(dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(i)));
    if (dpp_has_source<CTRL, ROW_MASK>(lane) && cand_better(og, oi, g, i)) {
        g = og;
        i = oi;
    }
}
// The best (gain, index) pair: higher gain, then the lower index; index < 0 is "none".
__device__ __forceinline__ void wave_best(double &g, int &i) {
    const uint32_t lane = threadIdx.x & 63u;
    best_step<DPP_ROW_SHR1, 0xf>(g, i, lane);
    best_step<DPP_ROW_SHR2, 0xf>(g, i, lane);
    best_step<DPP_ROW_SHR4, 0xf>(g, i, lane);
    best_step<DPP_ROW_SHR8, 0xf>(g, i, lane);
    best_step<DPP_ROW_BCAST15, 0xa>(g, i, lane);
    best_step<DPP_ROW_BCAST31, 0xc>(g, i, lane);
    i = __builtin_amdgcn_readlane(i, 63);
    g = double_of(readlane_u64(bits_of(g), 63));
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void min_step(int &v, uint32_t lane) {
    int o = static_cast<int>(dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(v)));
    if (dpp_has_source<CTRL, ROW_MASK>(lane) && o < v) v = o;
}
__device__ __forceinline__ int wave_min(int v) {
    const uint32_t lane = threadIdx.x & 63u;
    min_step<DPP_ROW_SHR1, 0xf>(v, lane);
    min_step<DPP_ROW_SHR2, 0xf>(v, lane);
    min_step<DPP_ROW_SHR4, 0xf>(v, lane);
    min_step<DPP_ROW_SHR8, 0xf>(v, lane);
    min_step<DPP_ROW_BCAST15, 0xa>(v, lane);
    min_step<DPP_ROW_BCAST31, 0xc>(v, lane);
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ double readlane_f64(double v, uint32_t lane) { return double_of(readlane_u64(bits_of(v), lane)); }

// Branch-free all-reductions: a lane without a source in a DPP step reads the reduction's identity (the `old`
// operand with bound_ctrl off), so every step is one move and one max or min.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_min_step(int v) {
    const int o = __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, ROW_MASK, 0xf, false);
    return o < v ? o : v;
}
__device__ __forceinline__ int wave_min_i32(int v) {
    v = dpp_min_step<DPP_ROW_SHR1, 0xf>(v);
    v = dpp_min_step<DPP_ROW_SHR2, 0xf>(v);
    v = dpp_min_step<DPP_ROW_SHR4, 0xf>(v);
    v = dpp_min_step<DPP_ROW_SHR8, 0xf>(v);
    v = dpp_min_step<DPP_ROW_BCAST15, 0xa>(v);
    v = dpp_min_step<DPP_ROW_BCAST31, 0xc>(v);
    return __builtin_amdgcn_readlane(v, 63);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_max_step(double v) {  // v is never NaN
    const uint64_t b = bits_of(v), id = bits_of(-__builtin_inf());
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(static_cast<uint32_t>(id)),
                                                                          static_cast<int>(static_cast<uint32_t>(b)), CTRL, ROW_MASK, 0xf, false));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(static_cast<uint32_t>(id >> 32)),
                                                                          static_cast<int>(static_cast<uint32_t>(b >> 32)), CTRL, ROW_MASK, 0xf, false));
    const double o = double_of((static_cast<uint64_t>(hi) << 32) | lo);
    return o > v ? o : v;
}
__device__ __forceinline__ double wave_max_f64(double v) {
    v = dpp_max_step<DPP_ROW_SHR1, 0xf>(v);
    v = dpp_max_step<DPP_ROW_SHR2, 0xf>(v);
    v = dpp_max_step<DPP_ROW_SHR4, 0xf>(v);
    v = dpp_max_step<DPP_ROW_SHR8, 0xf>(v);
    v = dpp_max_step<DPP_ROW_BCAST15, 0xa>(v);
    v = dpp_max_step<DPP_ROW_BCAST31, 0xc>(v);
    return readlane_f64(v, 63);
}
// wave_best for gains that are never NaN: the highest gain, then the lowest index among the lanes holding it.
__device__ __forceinline__ void wave_argmax(double &g, int &i) {
    const double m = wave_max_f64(i >= 0 ? g : -__builtin_inf());
    const int w = wave_min_i32(i >= 0 && g == m ? i : 0x7fffffff);
    g = m;
    i = w == 0x7fffffff ? -1 : w;
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_max_u32_step(uint32_t v) {
    const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROW_MASK, 0xf, false));
    return o > v ? o : v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = dpp_max_u32_step<DPP_ROW_SHR1, 0xf>(v);
    v = dpp_max_u32_step<DPP_ROW_SHR2, 0xf>(v);
    v = dpp_max_u32_step<DPP_ROW_SHR4, 0xf>(v);
    v = dpp_max_u32_step<DPP_ROW_SHR8, 0xf>(v);
    v = dpp_max_u32_step<DPP_ROW_BCAST15, 0xa>(v);
    v = dpp_max_u32_step<DPP_ROW_BCAST31, 0xc>(v);
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_max_u64_step(uint64_t v) {
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(static_cast<uint32_t>(v)), CTRL, ROW_MASK, 0xf, false));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(static_cast<uint32_t>(v >> 32)), CTRL, ROW_MASK, 0xf, false));
    const uint64_t o = (static_cast<uint64_t>(hi) << 32) | lo;
    return o > v ? o : v;
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
    v = dpp_max_u64_step<DPP_ROW_SHR1, 0xf>(v);
    v = dpp_max_u64_step<DPP_ROW_SHR2, 0xf>(v);
    v = dpp_max_u64_step<DPP_ROW_SHR4, 0xf>(v);
    v = dpp_max_u64_step<DPP_ROW_SHR8, 0xf>(v);
    v = dpp_max_u64_step<DPP_ROW_BCAST15, 0xa>(v);
    v = dpp_max_u64_step<DPP_ROW_BCAST31, 0xc>(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v)), 63));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(static_cast<uint32_t>(v >> 32)), 63));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}
// wave_max_u64 by the high words first: their u32 maximum, then the low word of the one lane holding it, or the low
// words' maximum over the lanes holding it when several do (half the DPP work of wave_max_u64 when the high words
// rarely tie). All lanes active.
__device__ __forceinline__ uint64_t wave_max_u64_hi(uint64_t v) {
    const uint32_t hi = static_cast<uint32_t>(v >> 32), lo = static_cast<uint32_t>(v);
    const uint32_t mh = wave_max_u32(hi);
    const unsigned long long at = __ballot(hi == mh);
    const uint32_t ml = (at & (at - 1ull)) == 0ull
                            ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lo), static_cast<int>(__builtin_ctzll(at))))
                            : wave_max_u32(hi == mh ? lo : 0u);
    return (static_cast<uint64_t>(mh) << 32) | ml;
}

struct FeatDev {
    uint32_t num_bins, hist_offset, kind, nan_bin;
    uint32_t col;   // column-major index among the non-trivial features
    uint32_t wide;  // two-byte bins (up to 1024, numerical): splits carry a numerical rule (rule_left)
};

struct ScanJob {
    const int64_t *hist;  // the leaf's histogram
    double units_grad, units_hess;
    int64_t count;
    FeatCand *out;        // [num_features]
};

// split.rs:584-620 find_numerical: the reverse scan (split.rs:557-567: missing values go left) always; the forward
// scan over the bins before the NaN bin (split.rs:571-580) only for a feature with a NaN bin and more than two bins.
__device__ __forceinline__ bool scan_searched(const Ctx &c, const FeatDev &m, bool evaluate) {
    return c.valid && evaluate && m.num_bins >= 2 && (m.kind == 1 || m.kind == 2);
}
__device__ __forceinline__ bool scan_two_way(const FeatDev &m) { return m.nan_bin && m.num_bins > 2; }

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_max_i32_step(int v) {
    const int o = __builtin_amdgcn_update_dpp(static_cast<int>(0x80000000u), v, CTRL, ROW_MASK, 0xf, false);
    return o > v ? o : v;
}
__device__ __forceinline__ int wave_max_i32(int v) {
    v = dpp_max_i32_step<DPP_ROW_SHR1, 0xf>(v);
    v = dpp_max_i32_step<DPP_ROW_SHR2, 0xf>(v);
    v = dpp_max_i32_step<DPP_ROW_SHR4, 0xf>(v);
    v = dpp_max_i32_step<DPP_ROW_SHR8, 0xf>(v);
    v = dpp_max_i32_step<DPP_ROW_BCAST15, 0xa>(v);
    v = dpp_max_i32_step<DPP_ROW_BCAST31, 0xc>(v);
    return __builtin_amdgcn_readlane(v, 63);
}

// One candidate of a scan (split.rs:420-462): the accumulated side's exact units and rows; returns its gain, -inf
// when the candidate is skipped (that side too small) or NaN (split.rs:508-531), and sets `stop` when the other side
// is too small while this one is not (the reference's `break`).
__device__ __forceinline__ double candidate_gain(const Ctx &c, const SplitCfgDev &cfg, double ug, double uh, int64_t cnt,
                                                int64_t min_count, bool &stop) {
    const double hh = K_EPSILON + uh * c.scale_hess;
    const bool skip = cnt < min_count || hh < cfg.min_sum_hessian_in_leaf || uh <= 0.0;
    const bool other_small = c.num_data - cnt < min_count || c.sum_hess - hh < cfg.min_sum_hessian_in_leaf ||
                             c.units_hess - uh <= 0.0;
    stop = other_small && !skip;
    const double gg = ug * c.scale_grad;
    const double gain = leaf_gain(c.sum_grad - gg, c.sum_hess - hh, cfg.lambda_l1, cfg.lambda_l2) +
                        leaf_gain(gg, hh, cfg.lambda_l1, cfg.lambda_l2);
    return (skip || gain != gain) ? -__builtin_inf() : gain;
}

// A candidate's stop test alone (candidate_gain's `stop`, without the gain).
__device__ __forceinline__ bool candidate_stop(const Ctx &c, const SplitCfgDev &cfg, double uh, int64_t cnt,
                                               int64_t min_count) {
    const double hh = K_EPSILON + uh * c.scale_hess;
    const bool skip = cnt < min_count || hh < cfg.min_sum_hessian_in_leaf || uh <= 0.0;
    const bool other_small = c.num_data - cnt < min_count || c.sum_hess - hh < cfg.min_sum_hessian_in_leaf ||
                             c.units_hess - uh <= 0.0;
    return other_small && !skip;
}

// Where a scan reads a feature's units from: planes of doubles in LDS, g and h apart, every value an exact integer.
struct LdsUnits {
    const double *pg, *ph;
    __device__ __forceinline__ double g(int b) const { return pg[b]; }
    __device__ __forceinline__ double h(int b) const { return ph[b]; }
};
// The same with a gap each 16 bins, for the wide scan, whose lanes read bins 16 apart.
struct PadUnits {
    const double *pg, *ph;
    __device__ __forceinline__ double g(int b) const { return pg[b + (b >> 4)]; }
    __device__ __forceinline__ double h(int b) const { return ph[b + (b >> 4)]; }
};

// A wave's LDS planes of one feature's units: up to 256 bins, or 1024 (two-byte bins) with PadUnits' gaps.
template <bool WIDE> struct UnitPlanes {
    static constexpr int BINS = WIDE ? 1024 : 256;
    double g[WIDE ? BINS + BINS / 16 : BINS], h[WIDE ? BINS + BINS / 16 : BINS];
};
// Fills them from a histogram ({g, h} per bin, in memory) with whole-line loads, all in flight together: lane l takes bins
// l, l + 64, ... (a scan's own lanes hold 4 or 16 neighbouring bins, so reading memory by them touched a line a lane and
// load: k_step_scan 64 -> 48 us a step on 6M x 32 two-byte bins). T: int64_t, or double for a histogram of the host's.
// Within the wave.
template <bool WIDE, class T>
__device__ __forceinline__ auto stage_units(const T *hist, const FeatDev &m, UnitPlanes<WIDE> &pl) {
    struct alignas(16) Pair {
        T g, h;
    };
    const uint32_t lane = threadIdx.x & 63u;
    const Pair *p = reinterpret_cast<const Pair *>(hist) + m.hist_offset;
    const uint32_t nb = m.num_bins;
    constexpr int N = UnitPlanes<WIDE>::BINS / 64;
    Pair v[N];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p[min(lane + 64u * i, nb ? nb - 1u : 0u)];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t b = lane + 64u * i, at = WIDE ? b + (b >> 4) : b;
        pl.g[at] = static_cast<double>(static_cast<int64_t>(v[i].g));
        pl.h[at] = static_cast<double>(static_cast<int64_t>(v[i].h));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (WIDE) return PadUnits{pl.g, pl.h};
    else return LdsUnits{pl.g, pl.h};
}

constexpr uint32_t UNIT_FEATS = 16;  // features a scan unit holds at most (segments of 4 lanes)

// A scan's lanes: the wave (SEGL = 64), or segments of SEGL = 16 or 4 lanes, each scanning its own feature of at most
// 4 * SEGL bins (t = lane % SEGL holds bins 4t .. 4t + 3). The wave-wide operations below, taken over a segment:
// inclusive sums (DPP row shifts stay inside a row of 16 lanes; a 4-lane segment masks the lanes below the shift),
// the segment's last value, maxima and minima, and a lane's value read by its segment.
template <int SEGL>
__device__ __forceinline__ void seg_scan_add(double &g, double &h, int64_t &c) {
    if constexpr (SEGL == 64) {
        scan_add_step<DPP_ROW_SHR1, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR2, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR4, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR8, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_BCAST15, 0xa>(g, h, c);
        scan_add_step<DPP_ROW_BCAST31, 0xc>(g, h, c);
    } else if constexpr (SEGL == 16) {
        scan_add_step<DPP_ROW_SHR1, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR2, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR4, 0xf>(g, h, c);
        scan_add_step<DPP_ROW_SHR8, 0xf>(g, h, c);
    } else {
        static_assert(SEGL == 4, "segments of 64, 16 or 4 lanes");
        const uint32_t t = threadIdx.x & 3u;
        const double g1 = double_of(dpp_u64<DPP_ROW_SHR1, 0xf>(bits_of(g))), h1 = double_of(dpp_u64<DPP_ROW_SHR1, 0xf>(bits_of(h)));
        const int64_t c1 = static_cast<int64_t>(dpp_u64<DPP_ROW_SHR1, 0xf>(static_cast<uint64_t>(c)));
        if (t >= 1) {
            g += g1;
            h += h1;
            c += c1;
        }
        const double g2 = double_of(dpp_u64<DPP_ROW_SHR2, 0xf>(bits_of(g))), h2 = double_of(dpp_u64<DPP_ROW_SHR2, 0xf>(bits_of(h)));
        const int64_t c2 = static_cast<int64_t>(dpp_u64<DPP_ROW_SHR2, 0xf>(static_cast<uint64_t>(c)));
        if (t >= 2) {
            g += g2;
            h += h2;
            c += c2;
        }
    }
}
template <int SEGL>
__device__ __forceinline__ double seg_read_f64(double v, uint32_t t) {
    if constexpr (SEGL == 64) return readlane_f64(v, t);
    else return __shfl(v, static_cast<int>(t), SEGL);
}
template <int SEGL>
__device__ __forceinline__ int64_t seg_read_i64(int64_t v, uint32_t t) {
    if constexpr (SEGL == 64) return static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(v), t));
    else return static_cast<int64_t>(__shfl(static_cast<long long>(v), static_cast<int>(t), SEGL));
}
template <int SEGL>
__device__ __forceinline__ int seg_max_i32(int v) {
    if constexpr (SEGL == 64) {
        return wave_max_i32(v);
    } else {
#pragma unroll
        for (int o = SEGL / 2; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, SEGL));
        return v;
    }
}
template <int SEGL>
__device__ __forceinline__ int seg_min_i32(int v) {
    if constexpr (SEGL == 64) {
        return wave_min_i32(v);
    } else {
#pragma unroll
        for (int o = SEGL / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, SEGL));
        return v;
    }
}
template <int SEGL>
__device__ __forceinline__ double seg_max_f64(double v) {  // v is never NaN
    if constexpr (SEGL == 64) {
        return wave_max_f64(v);
    } else {
#pragma unroll
        for (int o = SEGL / 2; o > 0; o >>= 1) {
            const double w = __shfl_xor(v, o, SEGL);
            v = w > v ? w : v;
        }
        return v;
    }
}

// scan_numerical for a feature of up to 1024 bins (two-byte bins, an extension): lane l holds bins
// 16l .. 16l + 15. The same candidates, stops and ties as scan_numerical, in two passes over the lane's bins so that
// only the units stay in registers: the first finds both directions' stops, the second evaluates the candidates in
// range, re-forming the exact prefix sums as it goes.
__device__ __forceinline__ void scan_numerical_wide(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m, const PadUnits &u,
                                                    bool &rf, Grown &rg, bool &ff, Grown &fg) {
    constexpr int NPB = 16;
    const int lane = static_cast<int>(threadIdx.x & 63u);
    const int nb = static_cast<int>(m.num_bins);
    const bool two = scan_two_way(m);
    const int top = two ? nb - 2 : nb - 1;
    double gu[NPB], hu[NPB];
#pragma unroll
    for (int j = 0; j < NPB; ++j) {
        const int b = NPB * lane + j;
        const int t = b <= top ? b : 0;
        gu[j] = b <= top ? u.g(t) : 0.0;
        hu[j] = b <= top ? u.h(t) : 0.0;
    }
    // per-bin counts (split.rs:196-198): `(x + 0.5) as i64`
    auto count_of = [&](int j) {
        return NPB * lane + j <= top ? sat_i64(hu[j] * c.scale_hess * c.cnt_factor + 0.5) : int64_t{0};
    };
    double lg = 0.0, lh = 0.0;
    int64_t lc = 0;
#pragma unroll
    for (int j = 0; j < NPB; ++j) {
        lg += gu[j];
        lh += hu[j];
        lc += count_of(j);
    }
    double eg = lg, eh = lh;
    int64_t ec = lc;
    scan_add_step<DPP_ROW_SHR1, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR2, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR4, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR8, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_BCAST15, 0xa>(eg, eh, ec);
    scan_add_step<DPP_ROW_BCAST31, 0xc>(eg, eh, ec);
    const double tg = readlane_f64(eg, 63), th = readlane_f64(eh, 63);
    const int64_t tc = static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(ec), 63));
    eg -= lg;
    eh -= lh;
    ec -= lc;
    const int64_t min_count = cfg.min_data_in_leaf > 1 ? cfg.min_data_in_leaf : 1;
    // pass 1: the stops (reverse: the highest stopping bin; forward: the lowest)
    int stop_r = -1, stop_f = 0x7fffffff;
    {
        double pg = eg, ph = eh;
        int64_t pc = ec;
        for (int j = 0; j < NPB; ++j) {
            const int b = NPB * lane + j;
            const int64_t cj = count_of(j);
            const double bg = pg, bh = ph;  // the prefix below b
            const int64_t bc = pc;
            pg += gu[j];
            ph += hu[j];
            pc += cj;
            if (b > top) continue;
            if (b >= 1 && candidate_stop(c, cfg, th - bh, tc - bc, min_count)) stop_r = b;
            if (two && stop_f == 0x7fffffff && candidate_stop(c, cfg, ph, pc, min_count)) stop_f = b;
            (void)bg;
        }
    }
    const int lo = wave_max_i32(stop_r) + 1;
    const int hi = two ? wave_min_i32(stop_f) : 0;
    // pass 2: the candidates in range; each lane keeps its best of each direction with its accumulated side
    double brg = -__builtin_inf(), bfg = -__builtin_inf();
    int brb = -1, bfb = -1;
    double rug = 0.0, ruh = 0.0, fug = 0.0, fuh = 0.0;
    int64_t ruc = 0, fuc = 0;
    {
        double pg = eg, ph = eh;
        int64_t pc = ec;
        for (int j = 0; j < NPB; ++j) {
            const int b = NPB * lane + j;
            const int64_t cj = count_of(j);
            const double ag = tg - pg, ah = th - ph;  // the right side from b up
            const int64_t ac = tc - pc;
            pg += gu[j];
            ph += hu[j];
            pc += cj;
            if (b > top) continue;
            bool stop;
            if (b >= 1 && b >= lo) {
                const double gv = candidate_gain(c, cfg, ag, ah, ac, min_count, stop);
                if (brb < 0 || gv >= brg) {  // visited downward: the highest b on equal gains
                    brg = gv;
                    brb = b;
                    rug = ag;
                    ruh = ah;
                    ruc = ac;
                }
            }
            if (two && b < hi) {
                const double gv = candidate_gain(c, cfg, pg, ph, pc, min_count, stop);
                if (bfb < 0 || gv > bfg) {  // visited upward: the lowest b on equal gains
                    bfg = gv;
                    bfb = b;
                    fug = pg;
                    fuh = ph;
                    fuc = pc;
                }
            }
        }
    }
    rf = false;
    ff = false;
    {
        const double best = wave_max_f64(brb >= 0 ? brg : -__builtin_inf());
        const int first = wave_max_i32(brb >= 0 && brg == best ? brb : -1);
        if (first >= 0 && best > c.min_gain_shift) {
            const uint32_t owner = static_cast<uint32_t>(first) / NPB;
            rg.ug = readlane_f64(rug, owner);
            rg.uh = readlane_f64(ruh, owner);
            rg.count = static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(ruc), owner));
            rg.gain = best;
            rg.bin = static_cast<uint32_t>(first);
            rf = true;
        }
    }
    if (two) {
        const double best = wave_max_f64(bfb >= 0 ? bfg : -__builtin_inf());
        const int first = wave_min_i32(bfb >= 0 && bfg == best ? bfb : 0x7fffffff);
        if (first != 0x7fffffff && best > c.min_gain_shift) {
            const uint32_t owner = static_cast<uint32_t>(first) / NPB;
            fg.ug = readlane_f64(fug, owner);
            fg.uh = readlane_f64(fuh, owner);
            fg.count = static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(fuc), owner));
            fg.gain = best;
            fg.bin = static_cast<uint32_t>(first);
            ff = true;
        }
    }
}

// Both scan directions of a numerical feature (split.rs:555-620) from one pass over its bins, wave-wide. Lane l
// holds bins 4l .. 4l + 3 in natural order; the scanned bins are 0 .. top, top being the last bin before the NaN bin
// when the feature scans both ways and the last bin otherwise. Every accumulated side is a sum of exact integers
// (histogram units, per-bin counts rounded as split.rs:196-198), so the reverse scan's right side from bin b up is
// the total minus the prefix below b, the same values the reference's running sums reach.
// - Reverse (missing values go left): visits b = top .. 1; stops at the first b, in that order the highest, where
//   the other side is too small while the accumulated one is not; keeps the first maximum in its order, so the
//   highest b on equal gains. Threshold b - 1.
// - Forward (missing values go right; two-way features only): visits b = 0 .. top; stops at the lowest such b;
//   keeps the lowest b on equal gains. Threshold b.
template <int SEGL = 64, class Units>
__device__ __forceinline__ void scan_numerical(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m, const Units &u, bool &rf,
                                               Grown &rg, bool &ff, Grown &fg) {
    const int lane = static_cast<int>(threadIdx.x & static_cast<uint32_t>(SEGL - 1));  // the lane in its segment
    const int nb = static_cast<int>(m.num_bins);
    const bool two = scan_two_way(m);
    const int top = two ? nb - 2 : nb - 1;
    double gu[4], hu[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int b = 4 * lane + j;
        const int t = b <= top ? b : 0;
        gu[j] = b <= top ? u.g(t) : 0.0;
        hu[j] = b <= top ? u.h(t) : 0.0;
    }
    // per-bin counts: `(x + 0.5) as i64`, one conversion when the wave's are all in u32
    double xc[4];
    bool small = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        xc[j] = 4 * lane + j <= top ? hu[j] * c.scale_hess * c.cnt_factor + 0.5 : 0.0;
        small = small && xc[j] >= 0.0 && xc[j] < 4294967296.0;
    }
    int64_t ci[4];
    if (__all(small)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) ci[j] = static_cast<int64_t>(static_cast<uint32_t>(xc[j]));
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) ci[j] = sat_i64(xc[j]);
    }
    // inclusive prefix P(b) over bins 0 .. top, after the lane's exclusive one: p[j] is below bin 4 lane + j, p[j + 1]
    // up to it
    double pg[5], ph[5];
    int64_t pc[5];
    double lg = 0.0, lh = 0.0;
    int64_t lc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        lg += gu[j];
        lh += hu[j];
        lc += ci[j];
    }
    double eg = lg, eh = lh;
    int64_t ec = lc;
    seg_scan_add<SEGL>(eg, eh, ec);
    const double tg = seg_read_f64<SEGL>(eg, SEGL - 1), th = seg_read_f64<SEGL>(eh, SEGL - 1);
    const int64_t tc = seg_read_i64<SEGL>(ec, SEGL - 1);
    pg[0] = eg - lg;
    ph[0] = eh - lh;
    pc[0] = ec - lc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        pg[j + 1] = pg[j] + gu[j];
        ph[j + 1] = ph[j] + hu[j];
        pc[j + 1] = pc[j] + ci[j];
    }
    const int64_t min_count = cfg.min_data_in_leaf > 1 ? cfg.min_data_in_leaf : 1;
    rf = false;
    ff = false;
    {  // reverse: the right side from bin b up; candidates above the highest stop, the highest b among equal gains
        double gain[4];
        int stop_b = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = 4 * lane + j;
            bool stop = false;
            gain[j] = candidate_gain(c, cfg, tg - pg[j], th - ph[j], tc - pc[j], min_count, stop);
            if (stop && b >= 1 && b <= top) stop_b = b;  // b grows with j: the lane's highest
        }
        const int lo = max(seg_max_i32<SEGL>(stop_b) + 1, 1);
        double bg = -__builtin_inf();
        int bb = -1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = 4 * lane + j;
            if (b >= lo && b <= top && (bb < 0 || gain[j] >= bg)) {
                bg = gain[j];
                bb = b;
            }
        }
        const double best = seg_max_f64<SEGL>(bg);
        const int first = seg_max_i32<SEGL>(bb >= 0 && bg == best ? bb : -1);
        if (first >= 0 && best > c.min_gain_shift) {
            const uint32_t owner = static_cast<uint32_t>(first) >> 2;
            const int jj = first & 3;
            double og = pg[0], oh = ph[0];
            int64_t oc = pc[0];
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (j == jj) {
                    og = pg[j];
                    oh = ph[j];
                    oc = pc[j];
                }
            rg.ug = tg - seg_read_f64<SEGL>(og, owner);
            rg.uh = th - seg_read_f64<SEGL>(oh, owner);
            rg.count = tc - seg_read_i64<SEGL>(oc, owner);
            rg.gain = best;
            rg.bin = static_cast<uint32_t>(first);
            rf = true;
        }
    }
    if (two) {  // forward: candidates below the lowest stop, the lowest b among equal gains
        double gain[4];
        int stop_b = 0x7fffffff;
#pragma unroll
        for (int j = 3; j >= 0; --j) {
            const int b = 4 * lane + j;
            bool stop = false;
            gain[j] = candidate_gain(c, cfg, pg[j + 1], ph[j + 1], pc[j + 1], min_count, stop);
            if (stop && b <= top) stop_b = b;  // b falls with j: the lane's lowest
        }
        const int hi = seg_min_i32<SEGL>(stop_b);
        double bg = -__builtin_inf();
        int bb = -1;
#pragma unroll
        for (int j = 3; j >= 0; --j) {
            const int b = 4 * lane + j;
            if (b < hi && b <= top && (bb < 0 || gain[j] >= bg)) {
                bg = gain[j];
                bb = b;
            }
        }
        const double best = seg_max_f64<SEGL>(bg);
        const int first = seg_min_i32<SEGL>(bb >= 0 && bg == best ? bb : 0x7fffffff);
        if (first != 0x7fffffff && best > c.min_gain_shift) {
            const uint32_t owner = static_cast<uint32_t>(first) >> 2;
            const int jj = first & 3;
            double og = pg[1], oh = ph[1];
            int64_t oc = pc[1];
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (j == jj) {
                    og = pg[j + 1];
                    oh = ph[j + 1];
                    oc = pc[j + 1];
                }
            fg.ug = seg_read_f64<SEGL>(og, owner);
            fg.uh = seg_read_f64<SEGL>(oh, owner);
            fg.count = seg_read_i64<SEGL>(oc, owner);
            fg.gain = best;
            fg.bin = static_cast<uint32_t>(first);
            ff = true;
        }
    }
}

// The feature's candidate from its scans' results (rf/rg reverse, ff/fg forward).
__device__ FeatCand feature_candidate(const Ctx &c, const FeatDev &m, bool rf, const Grown &rg, bool ff, const Grown &fg) {
    FeatCand r = {};
    bool have = false;
    r.splittable = rf || ff;
    double output_gain = -__builtin_inf();
    if (rf) {  // split.rs:557-567 reverse_best
        double right_hess = K_EPSILON + rg.uh * c.scale_hess;
        r.best_gain = rg.gain;
        r.threshold = rg.bin - 1;
        r.left_grad = c.sum_grad - rg.ug * c.scale_grad;
        r.left_hess = c.sum_hess - right_hess;
        r.left_count = c.num_data - rg.count;
        r.left_units_g = c.units_grad - rg.ug;
        r.left_units_h = c.units_hess - rg.uh;
        r.default_left = scan_two_way(m) ? 1 : (m.nan_bin ? 0 : 1);
        output_gain = rg.gain - c.min_gain_shift;
        have = true;
    }
    if (ff && fg.gain > output_gain + c.min_gain_shift) {  // split.rs:571-580 forward_best
        r.best_gain = fg.gain;
        r.threshold = fg.bin;
        r.left_grad = fg.ug * c.scale_grad;
        r.left_hess = K_EPSILON + fg.uh * c.scale_hess;
        r.left_count = fg.count;
        r.left_units_g = fg.ug;
        r.left_units_h = fg.uh;
        r.default_left = 0;
        have = true;
    }
    if (have) {
        r.found = 1;
        r.gain = r.best_gain - c.min_gain_shift;
        r.col = m.col;
        r.nan_idx = m.nan_bin ? m.num_bins - 1 : NO_BIN;
        r.wide = m.wide;
    }
    return r;
}

// ---------------------------------------------------------------------------------------------------------
// Categorical features (split.rs:694-844): one-hot for at most max_cat_to_onehot bins, otherwise the bins with
// enough rows sorted by their smoothed gradient ratio and scanned from both ends. One wave per feature.
// ---------------------------------------------------------------------------------------------------------

// split.rs:243-258 check for a growing side (rows, hessian, hessian units) against the other side:
// 0 skip the candidate (Continue), 1 stop the scan (Break), 2 evaluate it.
__device__ __forceinline__ int side_check(const Ctx &c, const SplitCfgDev &cfg, int64_t cnt, double hess, double units_h,
                                          int64_t other_cnt, double other_hess) {
    if (cnt < cfg.min_data_in_leaf || cnt <= 0 || hess < cfg.min_sum_hessian_in_leaf || units_h <= 0.0) return 0;
    if (other_cnt < cfg.min_data_in_leaf || other_cnt <= 0) return 1;
    if (other_hess < cfg.min_sum_hessian_in_leaf || c.units_hess - units_h <= 0.0) return 1;
    return 2;
}

__device__ __forceinline__ int64_t bin_rows(const Ctx &c, double units_h) {  // split.rs:236-238 bin_count
    return sat_i64(units_h * c.scale_hess * c.cnt_factor + 0.5);
}

__device__ __forceinline__ void mask_set(uint32_t (&mask)[8], uint32_t bin) {
#pragma unroll
    for (uint32_t w = 0; w < 8; ++w)
        if ((bin >> 5) == w) mask[w] |= 1u << (bin & 31u);
}

// split.rs:695-736 find_onehot: every bin 1..num_bins on its own against the rest; the first strict maximum above
// min_gain_shift (NaN never counts). Lane l takes bins 1 + l + 64 j.
template <class Units>
__device__ FeatCand onehot_scan(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m, const Units &u) {
    const uint32_t lane = threadIdx.x & 63u;
    const int nb = static_cast<int>(m.num_bins);
    double bg = 0.0, bu_g = 0.0, bu_h = 0.0;
    int bt = -1;
    int64_t bcnt = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = 1 + static_cast<int>(lane) + 64 * j;
        if (t >= nb) continue;
        const double ug = u.g(t), uh = u.h(t);
        const int64_t cnt = bin_rows(c, uh);
        const double raw_hess = uh * c.scale_hess;
        const int64_t other_cnt = c.num_data - cnt;
        const double other_hess = c.sum_hess - raw_hess - K_EPSILON;
        if (side_check(c, cfg, cnt, raw_hess, uh, other_cnt, other_hess) != 2) continue;
        const double grad = ug * c.scale_grad;
        const double gain = leaf_gain(c.sum_grad - grad, other_hess, cfg.lambda_l1, cfg.lambda_l2) +
                            leaf_gain(grad, raw_hess + K_EPSILON, cfg.lambda_l1, cfg.lambda_l2);
        if (gain != gain || gain <= c.min_gain_shift) continue;
        if (bt < 0 || gain > bg) {
            bg = gain;
            bt = t;
            bu_g = ug;
            bu_h = uh;
            bcnt = cnt;
        }
    }
    const bool any = __ballot(bt >= 0) != 0;
    double wg = bg;
    int wt = bt;
    wave_best(wg, wt);
    FeatCand r = {};
    r.splittable = any ? 1 : 0;
    if (wt >= 0) {
        const uint32_t owner = static_cast<uint32_t>(wt - 1) & 63u;
        const double ug = readlane_f64(bu_g, owner), uh = readlane_f64(bu_h, owner);
        const int64_t cnt = static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(bcnt), owner));
        r.found = 1;
        r.best_gain = wg;
        r.gain = wg - c.min_gain_shift;
        r.threshold = static_cast<uint32_t>(wt);
        r.left_grad = ug * c.scale_grad;
        r.left_hess = uh * c.scale_hess + K_EPSILON;
        r.left_count = cnt;
        r.left_units_g = ug;
        r.left_units_h = uh;
        r.col = m.col;
        r.nan_idx = NO_BIN;
        r.rule = RULE_ONEHOT;
        r.cat_count = 1;
        mask_set(r.cat_mask, static_cast<uint32_t>(wt));
    }
    return r;
}

// A wave's LDS for the sorted categorical scan.
struct CatScratch {
    unsigned long long key[256];  // total-order bits of each bin's ratio (bin-indexed)
    uint32_t order[256];          // the sorted bins
    uint8_t eligible[256];        // the bin has at least cat_smooth rows
};

// f64 total order (split.rs:754 total_cmp) as an unsigned integer order. A ratio that is NaN (0 / 0 with
// cat_smooth = 0) orders by its sign bit; the reference computes it on x86-64, whose invalid-operation result is the
// default NaN with the sign set, so the device's NaN is replaced by that one.
__device__ __forceinline__ unsigned long long total_order_bits(double x) {
    unsigned long long b = x != x ? 0xfff8000000000000ull : __builtin_bit_cast(unsigned long long, x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

// One run of split.rs:795-843 SortedScan::run over the first `steps` positions of the sorted order, from the low
// end (forward) or the high end. Positions i = lane + 64 j; the stateful min_data_per_group walk is uniform.
// Returns whether a candidate passed; (gain, pos) the best, and its left sums.
template <class Units>
__device__ bool sorted_run(const Ctx &c, const SplitCfgDev &cfg, const Units &u, const CatScratch &sc, int used,
                           int steps, bool forward, double l2, bool &splittable, double &best_gain, int &best_pos,
                           double &lug, double &luh, int64_t &lcnt) {
    const uint32_t lane = threadIdx.x & 63u;
    double pg[4], ph[4];
    int64_t pc[4], ci[4];
    double lg = 0.0, lh = 0.0;
    int64_t lc = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = static_cast<int>(lane) * 4 + j;  // contiguous positions per lane: the prefix below is in order
        double gu = 0.0, hu = 0.0;
        int64_t cn = 0;
        if (i < steps) {
            const uint32_t t = sc.order[forward ? i : used - 1 - i];
            gu = u.g(static_cast<int>(t));
            hu = u.h(static_cast<int>(t));
            cn = bin_rows(c, hu);
        }
        ci[j] = cn;
        lg += gu;
        lh += hu;
        lc += cn;
        pg[j] = lg;
        ph[j] = lh;
        pc[j] = lc;
    }
    double eg = lg, eh = lh;
    int64_t ec = lc;
    scan_add_step<DPP_ROW_SHR1, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR2, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR4, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_SHR8, 0xf>(eg, eh, ec);
    scan_add_step<DPP_ROW_BCAST15, 0xa>(eg, eh, ec);
    scan_add_step<DPP_ROW_BCAST31, 0xc>(eg, eh, ec);
    eg -= lg;
    eh -= lh;
    ec -= lc;
    // per position: 1 skip (Continue), 2 stop (Break, or the other side below min_data_per_group), 0 candidate
    uint32_t flags = 0;  // 2 bits per position j
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        pg[j] += eg;
        ph[j] += eh;
        pc[j] += ec;
        const int i = static_cast<int>(lane) * 4 + j;
        if (i >= steps) continue;
        const double lhess = K_EPSILON + ph[j] * c.scale_hess;
        const int64_t rcnt = c.num_data - pc[j];
        const double rhess = c.sum_hess - lhess;
        const int chk = side_check(c, cfg, pc[j], lhess, ph[j], rcnt, rhess);
        uint32_t f = chk == 0 ? 1u : (chk == 1 || rcnt < cfg.min_data_per_group ? 2u : 0u);
        flags |= f << (2 * j);
    }
    // the walk (split.rs:806-823): rows since the last evaluated candidate must reach min_data_per_group
    uint32_t mine = 0;  // bit j: this lane's position 4 lane + j is evaluated
    int64_t group = 0;
    for (int i = 0; i < steps; ++i) {
        const uint32_t src = static_cast<uint32_t>(i) >> 2, jj = static_cast<uint32_t>(i) & 3u;
        const int64_t cij = jj == 0 ? ci[0] : (jj == 1 ? ci[1] : (jj == 2 ? ci[2] : ci[3]));
        group += static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(cij), src));
        const uint32_t f = (static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(flags), src)) >> (2 * jj)) & 3u;
        if (f == 1u) continue;
        if (f == 2u) break;
        if (group < cfg.min_data_per_group) continue;
        group = 0;
        if (lane == src) mine |= 1u << jj;
    }
    double bg = 0.0;
    int bp = -1;
    double b_g = 0.0, b_h = 0.0;
    int64_t b_c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (!((mine >> j) & 1u)) continue;
        const double lgrad = pg[j] * c.scale_grad;
        const double lhess = K_EPSILON + ph[j] * c.scale_hess;
        const double rhess = c.sum_hess - lhess;
        const double gain = leaf_gain(lgrad, lhess, cfg.lambda_l1, l2) + leaf_gain(c.sum_grad - lgrad, rhess, cfg.lambda_l1, l2);
        if (gain != gain || gain <= c.min_gain_shift) continue;
        if (bp < 0 || gain > bg) {
            bg = gain;
            bp = static_cast<int>(lane) * 4 + j;
            b_g = pg[j];
            b_h = ph[j];
            b_c = pc[j];
        }
    }
    splittable = splittable || (__ballot(bp >= 0) != 0);
    double wg = bg;
    int wp = bp;
    wave_best(wg, wp);
    if (wp < 0) return false;
    const uint32_t owner = static_cast<uint32_t>(wp) >> 2;
    best_gain = wg;
    best_pos = wp;
    lug = readlane_f64(b_g, owner);
    luh = readlane_f64(b_h, owner);
    lcnt = static_cast<int64_t>(readlane_u64(static_cast<uint64_t>(b_c), owner));
    return true;
}

// split.rs:740-784: sorted categorical. `order_out` (when given) receives the left bins in the rule's order.
template <class Units>
__device__ FeatCand sorted_scan(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m, const Units &u, CatScratch &sc,
                                uint8_t *order_out) {
    const uint32_t lane = threadIdx.x & 63u;
    const int nb = static_cast<int>(m.num_bins < 256 ? m.num_bins : 256);
    // split.rs:740-760: bins with at least cat_smooth (estimated) rows, by (g / (h + cat_smooth), bin)
    bool ok[4];
    unsigned long long key[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = 1 + static_cast<int>(lane) + 64 * j;
        ok[j] = false;
        key[j] = 0;
        if (t < nb) {
            const double gu = u.g(t), hu = u.h(t);
            ok[j] = static_cast<double>(bin_rows(c, hu)) >= cfg.cat_smooth;
            key[j] = total_order_bits((gu * c.scale_grad) / (hu * c.scale_hess + cfg.cat_smooth));
        }
        if (t < 256) {
            sc.key[t] = key[j];
            sc.eligible[t] = ok[j] ? 1 : 0;
        }
    }
    if (lane == 0) sc.eligible[0] = 0;
    int used = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) used += __popcll(__ballot(ok[j]));
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    // rank = eligible bins before this one in (key, bin) order
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = 1 + static_cast<int>(lane) + 64 * j;
        int rank = 0;
        if (ok[j])
            for (int v = 1; v < nb; ++v) {
                const unsigned long long kv = sc.key[v];
                rank += (sc.eligible[v] && (kv < key[j] || (kv == key[j] && v < t))) ? 1 : 0;
            }
        __builtin_amdgcn_wave_barrier();
        if (ok[j]) sc.order[rank] = static_cast<uint32_t>(t);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    FeatCand r = {};
    const int max_num_cat = static_cast<int>(cfg.max_cat_threshold < static_cast<uint64_t>((used + 1) / 2)
                                                 ? cfg.max_cat_threshold : static_cast<uint64_t>((used + 1) / 2));
    const int steps = used < max_num_cat ? used : max_num_cat;
    const double l2 = cfg.lambda_l2 + cfg.cat_l2;
    bool splittable = false;
    double fg = 0.0, bgn = 0.0, flg = 0.0, flh = 0.0, blg = 0.0, blh = 0.0;
    int fp = -1, bpz = -1;
    int64_t flc = 0, blc = 0;
    const bool ff = steps > 0 && sorted_run(c, cfg, u, sc, used, steps, true, l2, splittable, fg, fp, flg, flh, flc);
    const bool bf = steps > 0 && sorted_run(c, cfg, u, sc, used, steps, false, l2, splittable, bgn, bpz, blg, blh, blc);
    r.splittable = splittable ? 1 : 0;
    if (!ff && !bf) return r;
    const bool fwd = ff && !(bf && bgn > fg);  // split.rs:775-781: the backward run replaces only a lower gain
    const double gain = fwd ? fg : bgn;
    const int pos = fwd ? fp : bpz;
    const double ug = fwd ? flg : blg, uh = fwd ? flh : blh;
    r.found = 1;
    r.best_gain = gain;
    r.gain = gain - c.min_gain_shift;
    r.threshold = static_cast<uint32_t>(pos);
    r.left_grad = ug * c.scale_grad;
    r.left_hess = K_EPSILON + uh * c.scale_hess;
    r.left_count = fwd ? flc : blc;
    r.left_units_g = ug;
    r.left_units_h = uh;
    r.col = m.col;
    r.nan_idx = NO_BIN;
    r.rule = RULE_SORTED;
    r.cat_forward = fwd ? 1u : 0u;
    r.cat_count = static_cast<uint32_t>(pos + 1);
    for (int k = 0; k <= pos; ++k) {
        const uint32_t t = sc.order[fwd ? k : used - 1 - k];
        mask_set(r.cat_mask, t);
        if (order_out && lane == 0) order_out[k] = static_cast<uint8_t>(t);
    }
    return r;
}

// The candidate of a categorical feature (split.rs:847-862).
template <class Units>
__device__ __forceinline__ FeatCand categorical_candidate(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m,
                                                          const Units &u, CatScratch &sc, uint8_t *order_out) {
    if (m.num_bins <= cfg.max_cat_to_onehot) return onehot_scan(c, cfg, m, u);
    return sorted_scan(c, cfg, m, u, sc, order_out);
}

// One feature's candidate from a leaf's histogram, by one wave: split.rs:584-620 find_numerical, or a categorical search.
template <bool WIDE, class T>
__device__ __forceinline__ FeatCand scan_feature(const Ctx &c, const SplitCfgDev &cfg, const FeatDev &m, const T *hist, bool evaluate,
                                                 UnitPlanes<WIDE> &planes, CatScratch *cats, uint8_t *order_out) {
    if (!scan_searched(c, m, evaluate)) return FeatCand{};
    const auto u = stage_units<WIDE>(hist, m, planes);
    Grown rg = {}, fg = {};
    bool rf, ff;
    if constexpr (WIDE) {
        scan_numerical_wide(c, cfg, m, u, rf, rg, ff, fg);
    } else {
        if (m.kind == 2) return categorical_candidate(c, cfg, m, u, *cats, order_out);
        scan_numerical(c, cfg, m, u, rf, rg, ff, fg);
    }
    return feature_candidate(c, m, rf, rg, ff, fg);
}

// split.rs:919-961 over one leaf's histogram, a wave a feature: split.rs:584-620 find_numerical, or a categorical search.
// WIDE: the features of two-byte bins (numerical, up to 1024), in an instance of their own, so the wide scan's registers do
// not lower the occupancy of the byte-bin scan. T: the histogram's units, int64_t, or double (a histogram of the host's,
// read where the host put it). One wave a feature whatever its bins: all of a leaf's features are on the chip at once.
// grid: ceil(num_features / 4); 256 threads.
template <bool WIDE, class T>
__global__ __launch_bounds__(256) void k_split_scan(ScanJob job, const FeatDev *__restrict__ feats,
                                                    const uint8_t *__restrict__ evaluate, uint32_t num_features,
                                                    SplitCfgDev cfg, double sg, double sh,
                                                    uint8_t *cat_order /* [feature][256] or null */) {
    __shared__ UnitPlanes<WIDE> planes[4];
    __shared__ __align__(16) uint8_t cats[WIDE ? 16 : 4 * sizeof(CatScratch)];
    const uint32_t wave = threadIdx.x >> 6, f = blockIdx.x * 4 + wave;
    if (f >= num_features) return;
    const FeatDev m = feats[f];
    const bool ev = evaluate[f] != 0;
    if ((m.wide != 0) != WIDE) return;  // the other instance's feature
    const Ctx c = make_ctx(cfg, sg, sh, job.units_grad, job.units_hess, job.count);
    const FeatCand r = scan_feature<WIDE>(c, cfg, m, reinterpret_cast<const T *>(job.hist), ev, planes[wave],
                                          reinterpret_cast<CatScratch *>(cats) + (WIDE ? 0u : wave),
                                          cat_order ? cat_order + static_cast<size_t>(f) * 256 : nullptr);
    if ((threadIdx.x & 63) == 0) job.out[f] = r;
}

// The leaf's SplitInfo (split.rs:631-651 finish) and splittable flags from the per-feature candidates: the
// highest gain, NaN as -inf, ties to the lower feature (split.rs:866-880). One block per job.
struct SplitOut {
    int32_t found, feature;
    double gain;
    uint32_t threshold, default_left;
    double left_grad, left_hess;
    int64_t left_count;
    double right_grad, right_hess;
    int64_t right_count;
    double left_output, right_output;
    uint32_t col, nan_idx;  // the feature's column-major index and NaN bin (NO_BIN: none)
    uint32_t rule;          // RULE_*: categorical rules send exactly the bins of cat_mask left
    uint32_t wide;          // the feature has two-byte bins
    uint32_t cat_count;
    uint32_t cat_mask[8];
};

// The best split over the per-feature candidates of `job` (highest gain, NaN as -inf, ties to the lower feature,
// split.rs:866-880) as the leaf's SplitOut (split.rs:631-651 finish), and its splittable flags. Block-wide (up
// to 1024 threads).
// split.rs:631-651 finish: the leaf's SplitInfo from its best feature's candidate.
__device__ __forceinline__ SplitOut split_out(const FeatCand &c, int f, const Ctx &x, const SplitCfgDev &cfg) {
    SplitOut o = {};
    o.found = 1;
    o.feature = f;
    o.gain = c.best_gain - x.min_gain_shift;
    o.threshold = c.threshold;
    o.default_left = c.default_left;
    o.left_grad = c.left_units_g;
    o.left_hess = c.left_units_h;
    o.left_count = c.left_count;
    o.right_grad = x.units_grad - c.left_units_g;
    o.right_hess = x.units_hess - c.left_units_h;
    o.right_count = x.num_data - c.left_count;
    const double l2 = c.rule == RULE_SORTED ? cfg.lambda_l2 + cfg.cat_l2 : cfg.lambda_l2;  // split.rs:667-680
    o.left_output = leaf_output(c.left_grad, c.left_hess, cfg.lambda_l1, l2);
    o.right_output = leaf_output(x.sum_grad - c.left_grad, x.sum_hess - c.left_hess, cfg.lambda_l1, l2);
    o.col = c.col;
    o.nan_idx = c.nan_idx;
    o.rule = c.rule;
    o.wide = c.wide;
    o.cat_count = c.cat_count;
    for (int w = 0; w < 8; ++w) o.cat_mask[w] = c.cat_mask[w];
    if (c.rule != RULE_NUMERICAL) {
        o.threshold = 0;
        o.default_left = 0;
    }
    return o;
}

__device__ void select_split(const ScanJob &job, int64_t count, uint32_t num_features, const SplitCfgDev &cfg, double sg,
                             double sh, SplitOut *out, uint8_t *splittable) {
    __shared__ double wgain[16];
    __shared__ int wfeat[16];
    const uint32_t nw = blockDim.x >> 6;
    double best = 0.0;
    int bf = -1;
    for (uint32_t f = threadIdx.x; f < num_features; f += blockDim.x) {
        const FeatCand &c = job.out[f];
        splittable[f] = static_cast<uint8_t>(c.splittable);
        if (!c.found) continue;
        double g = (c.gain != c.gain) ? -__builtin_inf() : c.gain;
        if (cand_better(g, static_cast<int>(f), best, bf)) {
            best = g;
            bf = static_cast<int>(f);
        }
    }
    for (int o = 32; o >= 1; o >>= 1) {
        double og = __shfl_xor(best, o);
        int of = __shfl_xor(bf, o);
        if (cand_better(og, of, best, bf)) {
            best = og;
            bf = of;
        }
    }
    if ((threadIdx.x & 63) == 0) {
        wgain[threadIdx.x >> 6] = best;
        wfeat[threadIdx.x >> 6] = bf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < nw; ++w)
            if (cand_better(wgain[w], wfeat[w], best, bf)) {
                best = wgain[w];
                bf = wfeat[w];
            }
        SplitOut o = {};
        if (bf >= 0) o = split_out(job.out[bf], bf, make_ctx(cfg, sg, sh, job.units_grad, job.units_hess, count), cfg);
        *out = o;
    }
    __syncthreads();
}

// The trait's split search's end: the leaf's SplitOut, its splittable flags and, for a sorted categorical rule, its bins in
// order, written where the host reads them. One block.
__global__ __launch_bounds__(256) void k_split_select(ScanJob job, uint32_t num_features, SplitCfgDev cfg, double sg, double sh,
                                                      const uint8_t *cat_order, SplitOut *out, uint8_t *order_out,
                                                      uint8_t *splittable) {
    __shared__ SplitOut o;
    select_split(job, job.count, num_features, cfg, sg, sh, &o, splittable);
    __syncthreads();
    static_assert(sizeof(SplitOut) % 4 == 0 && sizeof(SplitOut) / 4 <= 256, "a split copies in one pass");
    if (threadIdx.x < sizeof(SplitOut) / 4)
        reinterpret_cast<uint32_t *>(out)[threadIdx.x] = reinterpret_cast<const uint32_t *>(&o)[threadIdx.x];
    if (o.found && o.rule == RULE_SORTED) order_out[threadIdx.x] = cat_order[static_cast<size_t>(o.feature) * 256 + threadIdx.x];
}

// A histogram's units as the doubles the trait returns, and a partition's left count (when given), written to the host's
// pinned memory. A thread a bin.
__global__ __launch_bounds__(256) void k_hist_to_host(const int64_t *__restrict__ hist, double *__restrict__ out, uint64_t bins,
                                                      const uint32_t *left, uint32_t *left_out) {
    if (left && blockIdx.x == 0 && threadIdx.x == 0) *left_out = *left;
    for (uint64_t b = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; b < bins; b += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const longlong2 v = reinterpret_cast<const longlong2 *>(hist)[b];
        reinterpret_cast<double2 *>(out)[b] = make_double2(static_cast<double>(v.x), static_cast<double>(v.y));
    }
}

// ---------------------------------------------------------------------------------------------------------
// Device-driven growth (learner.rs:121-352) with speculative expansion.
//
// The reference grows leaf-wise: each split takes the leaf with the highest best gain (learner.rs:418-429), and
// a leaf's best split depends only on its own rows, its depth and its parent's splittable flags, never on when
// the leaf is split. So one split step here expands several leaves at once: the leaf the reference splits next
// (the blocker) and the highest-gain other leaves of the speculative tree. After each step, `advance` replays
// the reference's order over the gains known so far: it commits expansions while the leaf the reference splits
// next has been expanded (nodes and leaves get the reference's numbers), and plans the next step from the leaf
// where it stopped. Expansions the order has not reached when the tree is complete are dropped: their rows are
// merged back into ascending order (every leaf's rows are ascending, since the root's are and every partition
// is stable).
// ---------------------------------------------------------------------------------------------------------

// learner.rs:432-452 bin_split: word w of the bins that go left; numerical: bins 0..=threshold and the NaN bin when
// missing values go left; categorical: the rule's bins. A wide feature's split carries its rule instead (threshold,
// NaN bin + 1 when missing values go left; rule_left).
__device__ __forceinline__ uint32_t left_bins_word(const SplitOut &info, uint32_t w, uint32_t wide) {
    if (wide) {
        if (w == 0) return info.threshold;
        return w == 1 && info.default_left && info.nan_idx != NO_BIN ? info.nan_idx + 1u : 0u;
    }
    if (info.rule != RULE_NUMERICAL) return info.cat_mask[w];
    const uint32_t upto = info.threshold + 1;
    const uint32_t lo = 32 * w;
    uint32_t word = upto >= lo + 32 ? 0xffffffffu : (upto > lo ? (1u << (upto - lo)) - 1u : 0u);
    if (info.default_left && info.nan_idx != NO_BIN && (info.nan_idx >> 5) == w) word |= 1u << (info.nan_idx & 31u);
    return word;
}

constexpr uint32_t STEP_TILE = 4096;          // rows per partition tile: TILE_RPT per thread of a 1024-thread block
constexpr int TILE_RPT = STEP_TILE / 1024;
constexpr uint32_t CG_COLS = 4;               // slab columns per column group (k_step_reduce, k_step_scan)
// A split step's partials: workgroup b of a slab owns step_partial_stride(W) {g, h} pairs from pair b * stride,
// whether it writes 256 * W pairs or 256 * W packed words (a step can mix both). The stride is padded so that
// the same slot of consecutive partials does not fall at a power-of-two distance (which maps it to the same
// memory channel and bank).
constexpr uint32_t STEP_PARTIAL_PAD = 288;
__host__ __device__ constexpr size_t step_partial_stride(uint32_t w) { return 256u * static_cast<size_t>(w) + STEP_PARTIAL_PAD; }
constexpr uint32_t ST_AGG = 1, ST_INCL = 2;   // tile status: its own left count / lefts up to and including it
constexpr uint32_t LOOKBACK_SPINS = 1u << 20; // ~0.1 s of polling before a step gives up with an error

// Stripes of a job's `groups` partials that k_step_reduce adds on separate threads (combined through LDS), so that
// a thread adds about 8 partials (one round of loads): a power of two up to 32.
__device__ __forceinline__ uint32_t reduce_ways(uint32_t groups) {
    uint32_t w = 1;
    while (w < 32 && w * 8 < groups) w <<= 1;
    return w;
}

// Wave-wide sums of one value per lane (every lane active): inclusive and exclusive prefix, total. DPP steps: the plan's
// nine prefixes on one wave took 54 dependent LDS permutes by __shfl_up.
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v) {
    v += dpp_u32<DPP_ROW_SHR1, 0xf>(v);
    v += dpp_u32<DPP_ROW_SHR2, 0xf>(v);
    v += dpp_u32<DPP_ROW_SHR4, 0xf>(v);
    v += dpp_u32<DPP_ROW_SHR8, 0xf>(v);
    v += dpp_u32<DPP_ROW_BCAST15, 0xa>(v);
    v += dpp_u32<DPP_ROW_BCAST31, 0xc>(v);
    return v;
}
__device__ __forceinline__ uint32_t wave_excl_sum(uint32_t v) { return wave_incl_sum(v) - v; }
__device__ __forceinline__ uint32_t wave_total(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(wave_incl_sum(v)), 63));
}
__device__ __forceinline__ float wave_total_f32(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

constexpr uint32_t JMAX = 64;              // leaves expanded by one step at most (the plan's capacity)
// a step's jobs at most (GrowState::jcap): trees of up to LEAVES_SMALL leaves take 32, where a longer speculation
// mostly expands leaves the tree commits late or never; larger trees take JMAX, their steps being bound by the job count
__host__ __device__ constexpr uint32_t grow_jcap(uint32_t num_leaves) { return num_leaves <= LEAVES_SMALL ? 32u : JMAX; }
constexpr uint32_t SPEC_FEW = 8;           // at most this many: picked by repeated wave maxima (top_few)
constexpr uint32_t GROW_MAX_LEAVES = 2048;  // num_leaves of a device-grown tree at most
// Speculative leaves of a tree of num_leaves: 4 per leaf up to 512 leaves, then 2 per further leaf (the expansions
// a tree keeps need 2 per leaf; the rest is the room for speculating ahead, which advance keeps within it).
__host__ __device__ constexpr uint32_t grow_tcap(uint32_t num_leaves) {
    return num_leaves <= 512 ? 4 * num_leaves + 64 : 2 * num_leaves + 1088;
}

constexpr uint32_t T_LEAF = 0, T_PLANNED = 1, T_EXPANDED = 2;  // a speculative leaf's state

// A leaf of the speculative tree: the committed leaves and the children of every expansion.
struct TLeaf {
    uint32_t begin, count;   // rows in the partition
    double ug, uh;           // sums in histogram units
    int64_t cnt;             // exact row count
    int32_t slot;            // histogram slot, -1: none
    uint32_t has_best;
    uint32_t buf;            // partition buffer holding the rows
    uint32_t rev;            // the rows are stored last-first (right children of a split step)
    int32_t depth;
    uint32_t state;          // T_LEAF, T_PLANNED (expanded by the running step), T_EXPANDED
    int32_t kid;             // the children kid (left) and kid + 1 (right), once planned; -1 before
    uint32_t pad_;
    double value, weight;    // the leaf's output and hessian weight in the tree (from its parent's split)
    SplitOut best;
};

// The part of a speculative leaf that advance reads for every leaf, kept apart for one coalesced load.
struct TKey {
    double gain;  // best gain, when `has`
    uint32_t has;
    uint32_t state;
    int32_t kid;
    uint32_t pad_;
};

struct TreeDev {
    int32_t *split_feature;
    uint32_t *threshold_bin;
    uint8_t *default_left;
    int32_t *left_child, *right_child;
    float *split_gain;
    double *internal_value, *internal_weight;
    int64_t *internal_count;
    double *leaf_value, *leaf_weight;
    int64_t *leaf_count;
    int32_t *leaf_parent, *leaf_depth;
    uint32_t *left_bins;  // [node][8]: the bins that go left (BinSplit::left_bins)
    uint32_t *leaf_range; // [leaf][2]: the leaf's rows in the partition (begin, count)
};

// One leaf expanded by a split step (learner.rs:249-290): written by advance, read by the step's kernels.
struct JobPlan {
    uint32_t t;                   // the speculative leaf expanded
    uint32_t begin, count;        // its rows in the partition
    uint32_t col;                 // column-major index of the split feature
    uint32_t left_bins[8];
    uint32_t wide;                // left_bins hold a wide feature's numerical rule (rule_left)
    uint32_t built_side;          // 0: the left child is histogrammed, 1: the right (learner.rs:271-275)
    uint32_t hist;                // the built child is histogrammed (learner.rs:266-268)
    int32_t parent_slot, built_slot;
    uint32_t src_buf, src_rev;    // the buffer holding the leaf's rows (its children go to the other) and order
    uint32_t ntiles, tile_base;   // partition tiles and the first one's status word
    uint32_t groups, group_base;  // k_step_rows workgroups, one partial each
    uint32_t packed;              // the partials are packed 16/16 LDS words (one tile per workgroup)
    uint32_t ways;                // k_step_reduce stripes of the partials (reduce_ways)
    uint32_t red_base;            // k_step_reduce work items: per column group of two-byte slabs, `ways`
    uint32_t scan_base;           // k_step_scan work items: one per two-byte feature
    uint32_t ticket;              // next partition tile to hand out
    uint32_t left;                // rows going left, written by the last tile
    int32_t kid;                  // the children's speculative leaves
    int64_t parent_count;
    double child_ug[2], child_uh[2];  // the children's sums in histogram units (left, right)
    double child_out[2];          // their outputs
    int32_t depth;                // and depth
    uint32_t pad_;
};

// What k_step_children needs of a histogrammed job, found by its item's index alone (item / column groups), so that a
// block's first loads do not wait for a search of the jobs. A job of more than CHILD_SPLIT partials has a record for each
// of `ways` shares of about CHILD_SHARE partials, whose sums meet in scratch: in a tree's first step one job has a partial
// a compute unit, and one block a column group left most of the chip idle (88 us a launch on
// 10M x 128, 39 with shares; at 100 partials a job, the meeting cost more than it saved: 24 us against 34).
constexpr uint32_t CHILD_SPLIT = 160, CHILD_SHARE = 32, CHILD_WAYS = 16;  // a job's shares at most
constexpr uint32_t CHILD_MAX = JMAX + 64;                                // records of a step at most
struct ChildJob {
    uint32_t j, t, built_side;      // the job, its leaf, the histogrammed child
    uint32_t group_base, groups;    // the share's partials
    uint32_t ways, way, scratch;    // the job's shares, this one, the first one's scratch and counter row
    int32_t parent_slot, built_slot, kid;
    int64_t parent_count;
    double child_ug[2], child_uh[2];
};

// A split step: the plan of step s is plans[s % 2], written by the step before it.
struct StepPlan {
    uint32_t njobs;
    uint32_t total_groups;  // k_step_rows workgroups in use
    uint32_t total_child;   // k_step_children work items
    uint32_t total_red;     // k_step_reduce work items
    uint32_t total_scan;    // k_step_scan work items
    uint32_t epoch;         // tags the step's tile status words
    uint32_t pad_[2];
    // the jobs' first workgroup and work items side by side (a job search reads one run of words)
    uint32_t group_base[JMAX], red_base[JMAX], scan_base[JMAX];
    uint32_t pairs[JMAX];   // some partial of the job is {g, h} pairs (set by k_step_rows)
    ChildJob child[CHILD_MAX];  // the histogrammed jobs' shares
    JobPlan jobs[JMAX];
};

// The job whose range of work holds x: the last whose first element (bases[k]) is at or below it. The bases are read
// as one unrolled run, so the search is one round of loads: of the first 32 when the step has no more jobs (the
// whole run cost the latency-bound k_step_reduce 15% in such steps).
template <uint32_t N>
__device__ __forceinline__ uint32_t job_search(const uint32_t (&bases)[JMAX], uint32_t njobs, uint32_t x) {
    uint32_t j = 0;
#pragma unroll
    for (uint32_t k = 1; k < N; ++k)
        if (k < njobs && x >= bases[k]) j = k;
    return j;
}
__device__ __forceinline__ uint32_t job_of(const uint32_t (&bases)[JMAX], uint32_t njobs, uint32_t x) {
    return njobs <= 32u ? job_search<32>(bases, njobs, x) : job_search<JMAX>(bases, njobs, x);
}

struct GrowCtl {
    uint32_t num_leaves;   // committed leaves
    uint32_t done;         // no further step this tree
    uint32_t error;        // an invariant failed: 1 a child without rows, 3 a look-back gave up, 4 no room for a step
    uint32_t ntent;        // speculative leaves in use
    uint32_t next_slot;    // next free histogram slot
    uint32_t pending;      // expanded leaves not yet committed
    uint32_t epoch;        // split steps planned so far (kept across trees; tags tile status words)
    uint32_t steps;        // split steps planned this tree
    uint32_t expansions;   // leaves expanded this tree
    uint32_t pad_;
    uint32_t err_info[8];  // error 1: the job, its leaf, rows, left rows, tiles, workgroups, packed, jobs
    double hist_rows;      // rows histogrammed (built children), and rows x evaluated features
    double hist_bins;
    double hist_builds;    // child histograms built
    double part_rows;      // rows partitioned by the split steps
};

// Histogram slots: the root's is slot 0, each expansion that histograms takes the next free slot for its built
// child, and the other child keeps its parent's slot (a slot is never reused within a tree).
struct GrowState {
    GrowCtl *ctl;
    StepPlan *plans;          // [2]
    TLeaf *tl;                // [tcap], 0 is the root
    TKey *tk;                 // [tcap]
    int32_t *leaf_t;          // [num_leaves]: each committed leaf's speculative leaf
    uint8_t *leaf_left;       // [num_leaves]: the committed leaf is its parent's left child
    uint8_t *splittable;      // [tcap][nf]
    ScanJob *jobs;            // [1]: the root's search
    FeatCand *root_cands;     // [nf]: the root's search
    FeatCand *cands;          // [JMAX][2][nslot]: a step's children's candidates, the best of each column group of byte
                              // slabs, then each two-byte feature's
    double *cand_gain;        // their gains (NaN as -inf) and features (-1: none), apart for coalesced loads
    int32_t *cand_feat;
    const uint8_t *mask;      // [nf], the tree's feature mask
    const FeatDev *feats;
    TreeDev tree;
    int64_t *pool;
    uint64_t slot_stride;
    uint32_t nf, num_leaves, sums_feature;
    uint32_t tcap, nslots;    // speculative leaves and histogram slots available
    int32_t max_depth;
    SplitCfgDev cfg;
    double sg, sh;
    const struct DevScales *dsc;  // when set, the scales are these (made on the device), not sg and sh
    uint32_t target_groups;   // k_step_rows workgroups a step is spread over
    uint32_t jcap;            // jobs a step at most: grow_jcap(num_leaves)
    uint32_t ncgb;            // column groups of byte slabs (k_step_children), the first ones
    uint32_t ncgw;            // column groups of two-byte slabs (k_step_reduce)
    uint32_t nwide;           // two-byte features (k_step_scan, a wave per feature and child)
    uint32_t nslot;           // ncgb + nwide
    uint32_t flush_rows;      // rows a packed 16/16 LDS word can take
    uint32_t tile_cap;        // k_step_rows tiles a workgroup may take (its i32 sums of the quantized units)
    uint32_t count_work;      // keep the control block's byte-count totals (hist_rows ... part_rows)
    float hist_weight;        // the planner's cost of a tile of histogrammed rows, in partitioned tiles of a dense
    float sparse_weight;      // leaf, and the most a tile of a sparse leaf costs more
};

__device__ __forceinline__ double grow_sg(const GrowState &g) { return g.dsc ? g.dsc->sg : g.sg; }
__device__ __forceinline__ double grow_sh(const GrowState &g) { return g.dsc ? g.dsc->sh : g.sh; }

__device__ __forceinline__ bool depth_allows(const GrowState &g, int32_t d) { return g.max_depth <= 0 || d < g.max_depth; }

// Brings each listed run of rows into the first partition buffer in ascending order: copied from the second
// buffer (reversed when stored last-first), or reversed in place. grid: (x, runs).
struct RowRun {
    uint32_t begin, count, buf, rev;
};

__global__ void k_consolidate(const RowRun *__restrict__ runs, const uint32_t *__restrict__ buf1, uint32_t *__restrict__ buf0) {
    const RowRun l = runs[blockIdx.y];
    const uint32_t b = l.begin, n = l.count;
    const uint32_t stride = gridDim.x * blockDim.x;
    if (l.buf) {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
            buf0[b + i] = buf1[l.rev ? b + n - 1 - i : b + i];
    } else if (l.rev) {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n / 2; i += stride) {
            uint32_t x = buf0[b + i], y = buf0[b + n - 1 - i];
            buf0[b + i] = y;
            buf0[b + n - 1 - i] = x;
        }
    }
}

// A leaf whose expansion was dropped holds its rows as ascending runs (its speculative descendants' rows), which
// pairwise merge rounds bring back into one ascending run: in round t, runs 2m and 2m + 1 of the level-t runs (each
// the merge of 2^t consecutive original runs, its start starts[min(p << t, runs)]) become one, a row's place being
// its place in its run plus the rows below it in the partner run (a binary search; the rows of a leaf are distinct).
// ceil(log2(runs)) rounds, each moving every row once from `src` to `dst`, so a leaf costs its rows times the rounds,
// not times its runs. grid: (x, leaves).
struct MergeJob {
    uint32_t begin, count;
    uint32_t first, runs;  // the runs' starts (relative to begin) are starts[first, first + runs], then `count`
};

__global__ void k_merge_round(const MergeJob *__restrict__ jobs, const uint32_t *__restrict__ starts, uint32_t t,
                              const uint32_t *__restrict__ src, uint32_t *__restrict__ dst) {
    const MergeJob m = jobs[blockIdx.y];
    const uint32_t *s = starts + m.first;
    const uint32_t *leaf = src + m.begin;
    const uint32_t nr = (m.runs + (1u << t) - 1u) >> t;  // level-t runs
    auto start = [&](uint32_t p) { return s[min(p << t, m.runs)]; };
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m.count; i += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = nr;  // the run holding i: the last p with start(p) <= i
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (start(mid) <= i) lo = mid;
            else hi = mid;
        }
        const uint32_t p = lo, q = p ^ 1u;
        const uint32_t v = leaf[i];
        uint32_t pos = i;
        if (q < nr) {
            uint32_t a = start(q), b = start(q + 1);  // rows of run q below v: the first position holding more
            const uint32_t base = a;
            while (a < b) {
                const uint32_t mid = (a + b) >> 1;
                if (leaf[mid] < v) a = mid + 1;
                else b = mid;
            }
            pos = start(p & ~1u) + (i - start(p)) + (a - base);
        }
        dst[m.begin + pos] = v;
    }
}

__global__ void k_copy_back(const MergeJob *__restrict__ jobs, const uint32_t *__restrict__ buf1, uint32_t *__restrict__ buf0) {
    const MergeJob m = jobs[blockIdx.y];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < m.count; i += gridDim.x * blockDim.x)
        buf0[m.begin + i] = buf1[m.begin + i];
}

// The tree at its start: one leaf holding the root rows, its histogram in slot 0 when it is searched.
// A tree's state before its root is searched (or, `searched` 0, for a root that is not): by one thread.
__device__ __forceinline__ void grow_init(const GrowState &g, uint32_t root_begin, uint32_t root_count, int64_t root_cnt,
                                          uint32_t searched, double ug, double uh) {
    GrowCtl &c = *g.ctl;
    c.num_leaves = 1;
    c.done = searched ? 0u : 1u;
    c.error = 0;
    c.ntent = 1;
    c.next_slot = 1;
    c.pending = 0;
    c.steps = 0;
    c.expansions = 0;
    c.hist_rows = 0.0;
    c.hist_bins = 0.0;
    c.hist_builds = 0.0;
    c.part_rows = 0.0;
    TLeaf l = {};
    l.begin = root_begin;
    l.count = root_count;
    l.ug = ug;
    l.uh = uh;
    l.cnt = root_cnt;
    l.slot = searched ? 0 : -1;
    l.state = T_LEAF;
    l.kid = -1;
    g.tl[0] = l;
    g.tk[0] = TKey{0.0, 0u, T_LEAF, -1, 0u};
    g.leaf_t[0] = 0;
    g.leaf_left[0] = 0;
    g.tree.leaf_value[0] = 0.0;
    g.tree.leaf_weight[0] = 0.0;
    g.tree.leaf_count[0] = 0;
    g.tree.leaf_parent[0] = -1;
    g.tree.leaf_depth[0] = 0;
    g.tree.leaf_range[0] = root_begin;
    g.tree.leaf_range[1] = root_count;
    // both step plans empty until advance writes one: a step launched on an empty plan does nothing
    for (int k = 0; k < 2; ++k) {
        g.plans[k].njobs = 0;
        g.plans[k].total_groups = 0;
        g.plans[k].total_child = 0;
        g.plans[k].total_red = 0;
        g.plans[k].total_scan = 0;
    }
}
__global__ void k_grow_init(GrowState g, uint32_t root_begin, uint32_t root_count, int64_t root_cnt) {
    if (threadIdx.x == 0) grow_init(g, root_begin, root_count, root_cnt, 0u, 0.0, 0.0);
}

// The root's search (learner.rs:143-157): its sums from the sums feature's bins (split.rs:101-108) and every feature's
// candidate, a wave a feature; block 0 of the instance with `first` also makes the tree's initial state. The root's sums
// are those of one feature's bins taken in bin order as f64; every bin and every partial sum is an integer of magnitude
// below 2^53 (rows times units stays below 2^48), so each of those additions is exact and the result is the exact integer
// sum, which every wave adds in i64 and converts once (one more round of loads, against the two launches this took
// before). WIDE as k_split_scan's. grid: ceil(nf / 4), 256 threads.
template <bool WIDE>
__global__ __launch_bounds__(256) void k_root_scan(GrowState g, uint32_t root_begin, uint32_t root_count, int64_t root_cnt,
                                                   uint32_t first) {
    __shared__ UnitPlanes<WIDE> planes[4];
    __shared__ __align__(16) uint8_t cats[WIDE ? 16 : 4 * sizeof(CatScratch)];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u, f = blockIdx.x * 4 + wave;
    const int64_t *hist = g.pool;  // the root's slot is 0
    const FeatDev sums = g.feats[g.sums_feature];
    const FeatDev m = f < g.nf ? g.feats[f] : FeatDev{};
    const bool ev = f < g.nf && g.mask[f] != 0;
    const double scale_g = grow_sg(g), scale_h = grow_sh(g);
    const longlong2 *h = reinterpret_cast<const longlong2 *>(hist) + sums.hist_offset;
    int64_t sg = 0, sh = 0;
    for (uint32_t b = lane; b < sums.num_bins; b += 64u) {
        const longlong2 v = h[b];
        sg += v.x;
        sh += v.y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        sg += static_cast<int64_t>(__shfl_xor(static_cast<long long>(sg), o));
        sh += static_cast<int64_t>(__shfl_xor(static_cast<long long>(sh), o));
    }
    const double dg = static_cast<double>(sg), dh = static_cast<double>(sh);
    if (first && blockIdx.x == 0 && threadIdx.x == 0) {
        grow_init(g, root_begin, root_count, root_cnt, 1u, dg, dh);
        g.jobs[0] = ScanJob{hist, dg, dh, root_cnt, g.root_cands};
    }
    if (f >= g.nf || (m.wide != 0) != WIDE) return;
    const Ctx c = make_ctx(g.cfg, scale_g, scale_h, dg, dh, root_cnt);
    const FeatCand r = scan_feature<WIDE>(c, g.cfg, m, hist, ev, planes[wave], reinterpret_cast<CatScratch *>(cats) + (WIDE ? 0u : wave), nullptr);
    if (lane == 0) g.root_cands[f] = r;
}

// ---------------------------------------------------------------------------------------------------------
// advance: the reference's order over the known gains, then the next step's plan. Block-wide (1024 threads);
// `scratch` is LDS of at least sizeof(AdvShared) bytes.
// ---------------------------------------------------------------------------------------------------------

template <uint32_t MAXL>
struct AdvShared {
    static constexpr uint32_t TCAP = grow_tcap(MAXL);
    static constexpr uint32_t CAND = (TCAP + 1) / 2 + 1;  // unexpanded leaves: E + 1 of the 2E + 1 of E expansions
    double gain[TCAP];                    // speculative leaves' best gains
    uint32_t meta[TCAP];                  // bit 0: has a best split; bits 1-2: state; bits 3..: kid + 1
    uint16_t leaf_t[MAXL];                // committed leaf -> speculative leaf, as the replay goes
    int16_t pnode[MAXL];                  // committed leaf -> the internal node above it (-1: the root)
    uint8_t is_left[MAXL];                // committed leaf is its node's left child
    uint8_t touched[MAXL];                // committed leaf changed by this replay
    // committed leaf's replay key (0: none): replay_key64 in trees of more than 512 leaves, where 32-bit keys meet
    // the winner's gain prefix often; replay_key<11> in the others, where its u32 wave max is the cheaper
    std::conditional_t<(MAXL > LEAVES_SMALL), uint64_t, uint32_t> key[MAXL];
    // trees of up to 512 leaves (replay_reg): an expanded speculative leaf's children, left then right, as their
    // replay_key<11> without the id bits (0: no key), bit 0 set when the child has a split and a NaN gain
    uint2 crec[MAXL > LEAVES_SMALL ? 1 : TCAP];
    uint32_t leaf_m[MAXL > LEAVES_SMALL ? MAXL : 1];  // trees of more than 512 leaves: committed leaf's s.meta word
    uint16_t ck[MAXL];                    // commit c: the speculative leaf split (node n0 - 1 + c)
    uint16_t cx[MAXL];                    // commit c: the leaf id split
    int16_t cpn[MAXL];                    // commit c: the split leaf's node above
    uint8_t cleft[MAXL];                  // commit c: the split leaf was its node's left child
    uint64_t ckey[CAND];                  // speculation candidates' keys (higher bound, gain, then lower leaf);
                                          // before them, frontier_bounds' parent links
    uint32_t crank[CAND];                 // and their ranks
    uint16_t cand[CAND];                  // speculation candidates
    uint16_t job_t[JMAX];
    uint64_t skey[JMAX];                  // select_top: the selected candidates' keys
    uint16_t scand[JMAX];                 // and leaves
    uint32_t ncand, ncommit, n, blocker, done, njobs, band, above, nsel, neligible;
    uint32_t nnan;                        // committed leaves whose best gain is NaN (replay_lds)
};

__device__ __forceinline__ uint32_t key_meta(const TKey &k) {
    return (k.has ? 1u : 0u) | (k.state << 1) | (static_cast<uint32_t>(k.kid + 1) << 3);
}

// A committed leaf's replay key: the top 32 - IDB bits of its positive gain (a positive double's bits order as its
// value), then the lower leaf id (2^IDB - 1 - id); 0 for a leaf without a split or a positive gain. One u32 max over
// the wave finds the highest key; it is best_leaf's choice unless another leaf shares its gain prefix, which the
// replay then settles on the exact gains. IDB = 9 takes trees of up to 512 leaves, 11 up to 2048.
template <int IDB>
__device__ __forceinline__ uint32_t replay_key(double gain, uint32_t meta, uint32_t id) {
    if (!(meta & 1u) || !(gain > 0.0)) return 0u;
    uint32_t p = static_cast<uint32_t>(__builtin_bit_cast(uint64_t, gain) >> (31 + IDB));
    p = p ? p : 1u;
    return (p << IDB) | ((1u << IDB) - 1u - id);
}

// replay_key in 64 bits for trees of up to 2048 leaves (replay_lds): the positive gain's bits without their low 11
// (its exponent and 41 bits of mantissa) above 2047 - leaf id. Two gains share that prefix only when they agree to
// about 5e-13 (32-bit keys kept 21 bits, and at 2047 leaves a third of the commits met a leaf with the winner's
// prefix, each settled by an exact f64 argmax).
__device__ __forceinline__ uint64_t replay_key64(double gain, uint32_t meta, uint32_t id) {
    if (!(meta & 1u) || !(gain > 0.0)) return 0ull;
    uint64_t p = __builtin_bit_cast(uint64_t, gain) >> 11;
    p = p ? p : 1ull;
    return (p << 11) | (2047u - id);
}

// replay_lds's key of a leaf, in the width of the key array (Key)
template <class Key>
__device__ __forceinline__ Key leaf_key(double gain, uint32_t meta, uint32_t id) {
    if constexpr (sizeof(Key) == 8) return replay_key64(gain, meta, id);
    else return replay_key<11>(gain, meta, id);
}

// The replay of advance (learner.rs:158-163 with best_leaf, learner.rs:418-429) on one wave. Lane l owns committed
// leaves l, l + 64, ... (NPL of them, NPL * 64 >= num_leaves); their state is in LDS (speculative leaf, node above,
// its state word, left and changed flags, and the replay key in s.key) and only the lane's largest key is in a
// register. A commit is one wave max of those (the reference's argmax only matters while the best gain is positive:
// otherwise the tree stops), with an exact f64 argmax only when two leaves share the winner's gain prefix: a lane
// other than the winner's holds such a key exactly when its largest key has the prefix, and the winner's own keys
// are read from s.key by NPL lanes at once, with the winner's state, and serve again for that lane's new largest key
// after the commit. So a commit waits on two LDS reads: those, then its children's gains and state words. The rule
// that the first leaf with a split decides when its gain is NaN takes a wave minimum, only while some leaf has a NaN
// gain (they are counted). Leaves the commits, the committed-leaf arrays and the outcome in `s`.
template <int NPL, typename S>
__device__ __forceinline__ void replay_lds(S &s, uint32_t n0, uint32_t L) {
    constexpr int IDB = 11;
    static_assert(NPL * 64 <= (1 << IDB) && NPL * 64 <= static_cast<int>(GROW_MAX_LEAVES) && NPL <= 64, "leaf ids fit");
    constexpr uint64_t IDM = (1u << IDB) - 1u;
    static_assert(sizeof(s.leaf_m) >= sizeof(uint32_t) * NPL * 64, "the committed leaves' state words");
    using Key = std::remove_cv_t<std::remove_reference_t<decltype(s.key[0])>>;
    constexpr bool K64 = sizeof(Key) == 8;
    auto key_of = [](double gain, uint32_t meta, uint32_t id) -> Key { return leaf_key<Key>(gain, meta, id); };
    auto wave_max_key = [](Key v) -> Key {  // 64-bit keys: two gains share the high word when within about 1e-6
        if constexpr (K64) return wave_max_u64_hi(v);
        else return wave_max_u32(v);
    };
    const uint32_t lane = threadIdx.x & 63u;
    // the keys (0 past the committed leaves) and the NaN count were made by the whole block (advance)
    Key lk = 0;
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const Key key = s.key[lane + 64u * j];
        lk = key > lk ? key : lk;
    }
    uint32_t nan_leaves = s.nnan;
    uint32_t n = n0, nc = 0, blocker = 0;
    bool done = false;
    for (;;) {
        if (n >= L) {
            done = true;
            break;
        }
        // best_leaf: the first leaf with a split decides when its gain is NaN (nothing beats NaN under `>`)
        if (nan_leaves) {
            int lfirst = 1 << 30;
            for (int j = NPL - 1; j >= 0; --j) {  // descending, so the lowest id is the one kept
                const uint32_t id = lane + 64u * j;
                if (id >= n) continue;
                const uint32_t t = s.leaf_t[id];
                const double gj = s.gain[t];
                if (s.meta[t] & 1u) lfirst = 2 * static_cast<int>(id) + (gj != gj ? 1 : 0);
            }
            const int first = wave_min_i32(lfirst);
            if (first < (1 << 30) && (first & 1)) {
                done = true;
                break;
            }
        }
        const Key best = wave_max_key(lk);
        if (best == 0u) {
            done = true;
            break;
        }
        uint32_t x = static_cast<uint32_t>(IDM - (best & IDM));
        // the winner's lane's keys (0 past the leaves) and the winner's state, read together
        Key kk = lane < static_cast<uint32_t>(NPL) ? s.key[(x & 63u) + 64u * lane] : Key{0};
        uint32_t k = s.leaf_t[x], m = s.leaf_m[x];
        int32_t pn = s.pnode[x];
        uint32_t xl = s.is_left[x];
        {  // another leaf with the winner's gain prefix: the exact gains decide (then the lower id)
            const Key bp = best >> IDB;
            const bool other = (lane != (x & 63u) && (lk >> IDB) == bp) || ((kk >> IDB) == bp && kk != best);
            if (__ballot(other)) {
                double kg = 0.0;
                int ki = -1;
                for (int j = NPL - 1; j >= 0; --j) {  // descending, so the lowest id is kept on equal gains
                    const uint32_t id = lane + 64u * j;
                    if ((s.key[id] >> IDB) != bp) continue;
                    const double gj = s.gain[s.leaf_t[id]];
                    if (ki < 0 || gj >= kg) {
                        kg = gj;
                        ki = static_cast<int>(id);
                    }
                }
                wave_argmax(kg, ki);
                x = static_cast<uint32_t>(ki);
                kk = lane < static_cast<uint32_t>(NPL) ? s.key[(x & 63u) + 64u * lane] : Key{0};
                k = s.leaf_t[x];
                m = s.leaf_m[x];
                pn = s.pnode[x];
                xl = s.is_left[x];
            }
        }
        if (((m >> 1) & 3u) != T_EXPANDED) {
            blocker = k;
            break;
        }
        const uint32_t kid = (m >> 3) - 1u;
        const double g0 = s.gain[kid], g1 = s.gain[kid + 1];
        const uint32_t m0 = s.meta[kid], m1 = s.meta[kid + 1];
        const Key k0 = key_of(g0, m0, x), k1 = key_of(g1, m1, n);
        // leaf x becomes the left child, leaf n the right one, both under node n - 1
        const int32_t node = static_cast<int32_t>(n) - 1;
        if (lane == 0) {
            s.ck[nc] = static_cast<uint16_t>(k);
            s.cx[nc] = static_cast<uint16_t>(x);
            s.cpn[nc] = static_cast<int16_t>(pn);
            s.cleft[nc] = static_cast<uint8_t>(xl);
            s.leaf_t[x] = static_cast<uint16_t>(kid);
            s.leaf_m[x] = m0;
            s.pnode[x] = static_cast<int16_t>(node);
            s.is_left[x] = 1;
            s.touched[x] = 1;
            s.key[x] = k0;
            s.leaf_t[n] = static_cast<uint16_t>(kid + 1);
            s.leaf_m[n] = m1;
            s.pnode[n] = static_cast<int16_t>(node);
            s.is_left[n] = 0;
            s.touched[n] = 1;
            s.key[n] = k1;
        }
        nan_leaves += ((m0 & 1u) && g0 != g0 ? 1u : 0u) + ((m1 & 1u) && g1 != g1 ? 1u : 0u);
        // the lanes' largest keys: x's lane (its largest was x's old key) from its keys as read, with x's key now k0
        // (and n's k1 when n is in that lane); n's lane takes k1 as well
        const uint32_t lx = x & 63u, ln = n & 63u;
        Key kv = lane == (x >> 6) ? k0 : kk;
        kv = ln == lx && lane == (n >> 6) ? k1 : kv;
        const Key mx = wave_max_key(kv);
        if (lane == lx) lk = mx;
        else if (lane == ln) lk = k1 > lk ? k1 : lk;
        ++nc;
        ++n;
    }
    if (lane == 0) {
        s.ncommit = nc;
        s.n = n;
        s.done = done ? 1u : 0u;
        s.blocker = blocker;
    }
}

// replay_lds for trees of up to 512 leaves (NPL 4 or 8) with the replay keys and speculative leaves of lane l's
// committed leaves (l, l + 64, ...) in its registers: the test for another leaf with the winner's gain prefix
// needs no LDS, the winner's speculative leaf is a read of its lane, and its children's keys come from one read
// of s.crec (their key prefixes, made by the whole block), so a commit waits on one LDS read (that record with the
// state word) where replay_lds waits on five. Lane 0 keeps the committed-leaf arrays in LDS up to date for
// apply_commits and the NaN rule, which reads them; s.key is left as the block made it.
template <int NPL, typename S>
__device__ __forceinline__ void replay_reg(S &s, uint32_t n0, uint32_t L) {
    constexpr int IDB = 11;
    static_assert(NPL * 64 <= static_cast<int>(LEAVES_SMALL) && sizeof(s.key[0]) == 4, "u32 keys of 512 leaves at most");
    constexpr uint32_t IDM = (1u << IDB) - 1u;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t rk[NPL], rt[NPL], lk = 0;
#pragma unroll
    for (int j = 0; j < NPL; ++j) {  // keys are 0 past the committed leaves, whose speculative leaf is then unused
        const uint32_t id = lane + 64u * j;
        rk[j] = s.key[id];
        rt[j] = s.leaf_t[id];
        lk = rk[j] > lk ? rk[j] : lk;
    }
    uint32_t nan_leaves = s.nnan;
    uint32_t n = n0, nc = 0, blocker = 0;
    bool done = false;
    for (;;) {
        if (n >= L) {
            done = true;
            break;
        }
        // best_leaf: the first leaf with a split decides when its gain is NaN (nothing beats NaN under `>`)
        if (nan_leaves) {
            int lfirst = 1 << 30;
            for (int j = NPL - 1; j >= 0; --j) {  // descending, so the lowest id is the one kept
                const uint32_t id = lane + 64u * j;
                if (id >= n) continue;
                const uint32_t t = s.leaf_t[id];
                const double gj = s.gain[t];
                if (s.meta[t] & 1u) lfirst = 2 * static_cast<int>(id) + (gj != gj ? 1 : 0);
            }
            const int first = wave_min_i32(lfirst);
            if (first < (1 << 30) && (first & 1)) {
                done = true;
                break;
            }
        }
        const uint32_t best = wave_max_u32(lk);
        if (best == 0u) {
            done = true;
            break;
        }
        uint32_t x = IDM - (best & IDM);
        {  // another leaf with the winner's gain prefix: the exact gains decide (then the lower id)
            const uint32_t bp = best >> IDB;
            bool other = false;
            if (lane == (x & 63u)) {
#pragma unroll
                for (int j = 0; j < NPL; ++j) other = other || (rk[j] != best && (rk[j] >> IDB) == bp);
            } else {
                other = (lk >> IDB) == bp;
            }
            if (__ballot(other)) {
                double kg = 0.0;
                int ki = -1;
#pragma unroll
                for (int j = NPL - 1; j >= 0; --j) {  // descending, so the lowest id is kept on equal gains
                    if ((rk[j] >> IDB) != bp) continue;
                    const double gj = s.gain[rt[j]];
                    if (ki < 0 || gj >= kg) {
                        kg = gj;
                        ki = static_cast<int>(lane + 64u * j);
                    }
                }
                wave_argmax(kg, ki);
                x = static_cast<uint32_t>(ki);
            }
        }
        const uint32_t jx = x >> 6, lx = x & 63u, jn = n >> 6, ln = n & 63u;
        uint32_t tv = rt[0];
#pragma unroll
        for (int j = 1; j < NPL; ++j) tv = jx == static_cast<uint32_t>(j) ? rt[j] : tv;
        const uint32_t k = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tv), static_cast<int>(lx)));
        const uint32_t m = s.meta[k];
        const uint2 c = s.crec[k];
        const int32_t pn = s.pnode[x];
        const uint32_t xl = s.is_left[x];
        if (((m >> 1) & 3u) != T_EXPANDED) {
            blocker = k;
            break;
        }
        const uint32_t kid = (m >> 3) - 1u;
        const uint32_t k0 = (c.x >> IDB) ? ((c.x & ~IDM) | (IDM - x)) : 0u;
        const uint32_t k1 = (c.y >> IDB) ? ((c.y & ~IDM) | (IDM - n)) : 0u;
        // leaf x becomes the left child, leaf n the right one, both under node n - 1
        const int32_t node = static_cast<int32_t>(n) - 1;
        if (lane == 0) {
            s.ck[nc] = static_cast<uint16_t>(k);
            s.cx[nc] = static_cast<uint16_t>(x);
            s.cpn[nc] = static_cast<int16_t>(pn);
            s.cleft[nc] = static_cast<uint8_t>(xl);
            s.leaf_t[x] = static_cast<uint16_t>(kid);
            s.pnode[x] = static_cast<int16_t>(node);
            s.is_left[x] = 1;
            s.touched[x] = 1;
            s.leaf_t[n] = static_cast<uint16_t>(kid + 1);
            s.pnode[n] = static_cast<int16_t>(node);
            s.is_left[n] = 0;
            s.touched[n] = 1;
        }
        nan_leaves += (c.x & 1u) + (c.y & 1u);
        uint32_t nk = 0;
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            if (jx == static_cast<uint32_t>(j) && lane == lx) {
                rk[j] = k0;
                rt[j] = kid;
            }
            if (jn == static_cast<uint32_t>(j) && lane == ln) {
                rk[j] = k1;
                rt[j] = kid + 1u;
            }
            nk = rk[j] > nk ? rk[j] : nk;
        }
        lk = nk;
        ++nc;
        ++n;
    }
    if (lane == 0) {
        s.ncommit = nc;
        s.n = n;
        s.done = done ? 1u : 0u;
        s.blocker = blocker;
    }
}

// The replay of replay_lds for trees of up to 128 leaves (NPL 1 or 2), where registers beat LDS: lane l holds committed
// leaves l, l + 64, ... (NPL of them, NPL * 64 >= num_leaves) in registers (replay key, meta, speculative leaf, node
// above, left / has-split / NaN-gain flags). A commit is one u32 wave max of the keys (the reference's argmax only
// matters while the best gain is positive: otherwise the tree stops), with an exact f64 argmax only when two
// leaves share the winner's gain prefix; the rule that the first leaf with a split decides when its gain is NaN
// takes a wave minimum, only while some leaf has a NaN gain. Leaves the commits, the committed-leaf arrays and the
// outcome in `s`.
template <int NPL, typename S>
__device__ __forceinline__ void replay(S &s, uint32_t n0, uint32_t L) {
    constexpr int IDB = 9;
    static_assert(NPL * 64 <= (1 << IDB), "leaf ids fit the key");
    constexpr uint32_t IDM = (1u << IDB) - 1u;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t rk[NPL], rm[NPL], rt[NPL];
    int32_t rp[NPL];
    uint32_t rl = 0, rtouch = 0, rhas = 0, rnan = 0;  // bit j: leaf lane + 64 j is a left child / changed / ...
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const uint32_t id = lane + 64u * j;
        rk[j] = 0;
        rm[j] = 0;
        rt[j] = 0;
        rp[j] = -1;
        if (id < n0) {
            rt[j] = s.leaf_t[id];
            const double gj = s.gain[rt[j]];
            rm[j] = s.meta[rt[j]];
            rk[j] = replay_key<IDB>(gj, rm[j], id);
            rp[j] = s.pnode[id];
            rl |= s.is_left[id] ? 1u << j : 0u;
            rhas |= (rm[j] & 1u) ? 1u << j : 0u;
            rnan |= (rm[j] & 1u) && gj != gj ? 1u << j : 0u;
        }
    }
    uint32_t n = n0, nc = 0, blocker = 0;
    bool done = false;
    for (;;) {
        if (n >= L) {
            done = true;
            break;
        }
        // best_leaf: the first leaf with a split decides when its gain is NaN (nothing beats NaN under `>`)
        if (__ballot(rnan != 0u)) {
            int lfirst = 1 << 30;
#pragma unroll
            for (int j = NPL - 1; j >= 0; --j)  // descending, so the lowest id is the one kept
                if ((rhas >> j) & 1u) lfirst = 2 * static_cast<int>(lane + 64u * j) + static_cast<int>((rnan >> j) & 1u);
            const int first = wave_min_i32(lfirst);
            if (first < (1 << 30) && (first & 1)) {
                done = true;
                break;
            }
        }
        // otherwise the first highest gain among the rest (a NaN later never wins); none positive ends the tree
        uint32_t lk = 0;
#pragma unroll
        for (int j = 0; j < NPL; ++j) lk = rk[j] > lk ? rk[j] : lk;
        const uint32_t best = wave_max_u32(lk);
        if (best == 0u) {
            done = true;
            break;
        }
        uint32_t x = IDM - (best & IDM);
        {  // another leaf with the winner's gain prefix: the exact gains decide (then the lower id)
            const uint32_t bp = best >> IDB;
            uint32_t same = 0;
#pragma unroll
            for (int j = 0; j < NPL; ++j) same += (rk[j] >> IDB) == bp && rk[j] != best ? 1u : 0u;
            if (__ballot(same != 0u)) {
                double kg = 0.0;
                int ki = -1;
#pragma unroll
                for (int j = NPL - 1; j >= 0; --j) {  // descending, so the lowest id is kept on equal gains
                    if ((rk[j] >> IDB) != bp) continue;
                    const double gj = s.gain[rt[j]];
                    if (ki < 0 || gj >= kg) {
                        kg = gj;
                        ki = static_cast<int>(lane + 64u * j);
                    }
                }
                wave_argmax(kg, ki);
                x = static_cast<uint32_t>(ki);
            }
        }
        const uint32_t jx = x >> 6, lx = x & 63u;
        // jx is wave-uniform: indexed register reads
        const uint32_t vm = rm[jx], vt = rt[jx];
        const int32_t vp = rp[jx];
        const uint32_t m = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(vm), lx));
        const uint32_t k = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(vt), lx));
        if (((m >> 1) & 3u) != T_EXPANDED) {
            blocker = k;
            break;
        }
        const int32_t pn = __builtin_amdgcn_readlane(vp, lx);
        const uint32_t xl = (static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(rl), lx)) >> jx) & 1u;
        const uint32_t kid = (m >> 3) - 1u;
        const double g0 = s.gain[kid], g1 = s.gain[kid + 1];
        const uint32_t m0 = s.meta[kid], m1 = s.meta[kid + 1];
        if (lane == 0) {
            s.ck[nc] = static_cast<uint16_t>(k);
            s.cx[nc] = static_cast<uint16_t>(x);
            s.cpn[nc] = static_cast<int16_t>(pn);
            s.cleft[nc] = static_cast<uint8_t>(xl);
        }
        // leaf x becomes the left child, leaf n the right one, both under node n - 1
        const int32_t node = static_cast<int32_t>(n) - 1;
        const uint32_t jn = n >> 6, ln = n & 63u;
        // (jx and jn are wave-uniform: indexed register moves, one slot each)
        if (lane == lx) {
            rt[jx] = kid;
            rk[jx] = replay_key<IDB>(g0, m0, x);
            rm[jx] = m0;
            rp[jx] = node;
        }
        if (lane == ln) {
            rt[jn] = kid + 1;
            rk[jn] = replay_key<IDB>(g1, m1, n);
            rm[jn] = m1;
            rp[jn] = node;
        }
        const uint32_t bx = 1u << jx, bn = 1u << jn;
        if (lane == lx) {
            rl |= bx;
            rtouch |= bx;
            rhas = (rhas & ~bx) | ((m0 & 1u) ? bx : 0u);
            rnan = (rnan & ~bx) | ((m0 & 1u) && g0 != g0 ? bx : 0u);
        }
        if (lane == ln) {
            rl &= ~bn;
            rtouch |= bn;
            rhas = (rhas & ~bn) | ((m1 & 1u) ? bn : 0u);
            rnan = (rnan & ~bn) | ((m1 & 1u) && g1 != g1 ? bn : 0u);
        }
        ++nc;
        ++n;
    }
#pragma unroll
    for (int j = 0; j < NPL; ++j) {
        const uint32_t id = lane + 64u * j;
        if (id < n) {
            s.leaf_t[id] = static_cast<uint16_t>(rt[j]);
            s.pnode[id] = static_cast<int16_t>(rp[j]);
            s.is_left[id] = static_cast<uint8_t>((rl >> j) & 1u);
            s.touched[id] = static_cast<uint8_t>((rtouch >> j) & 1u);
        }
    }
    if (lane == 0) {
        s.ncommit = nc;
        s.n = n;
        s.done = done ? 1u : 0u;
        s.blocker = blocker;
    }
}

// The `spec` highest candidate keys for a few expansions (spec <= SPEC_FEW), on one wave: `spec` rounds of a wave
// maximum over the keys below the last one taken. The keys are distinct and end in 8191 - leaf, so round r finds the key
// ranked r and its leaf: jobs 1 .. spec in descending key order, as the ranking orders them.
template <typename S>
__device__ __forceinline__ void top_few(S &s, uint32_t ncand, uint32_t spec) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t first = lane < ncand ? s.ckey[lane] : 0ull;  // the only one of a lane up to 64 candidates
    uint64_t last = ~0ull;
    for (uint32_t r = 0; r < spec; ++r) {
        uint64_t best = first < last ? first : 0ull;
        for (uint32_t i = lane + 64u; i < ncand; i += 64u) {
            const uint64_t k = s.ckey[i];
            best = k < last && k > best ? k : best;
        }
        last = wave_max_u64_hi(best);
        if (lane == 0) s.job_t[1 + r] = static_cast<uint16_t>(8191u - (static_cast<uint32_t>(last) & 8191u));
    }
}

// The `spec` highest of the `ncand` candidate keys s.ckey (distinct 64-bit keys) into s.job_t[1 .. spec], in key
// order, by a radix selection over the keys' 64 bits, 8 at a time from the top: a 256-bucket count of the
// candidates that still match the prefix found so far, the bucket where the count from the top reaches what is
// left to take, and the candidates above it taken. Every key is distinct, so after at most 8 rounds the prefix
// is a whole key. Block-wide; s.crank holds the counts.
template <uint32_t MAXL>
__device__ void select_top(AdvShared<MAXL> &s, uint32_t ncand, uint32_t spec) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, nt = blockDim.x;
    uint32_t *count = s.crank;  // 256 buckets
    uint64_t prefix = 0, mask = 0;  // the bits fixed so far
    uint32_t taken = 0;             // candidates above the prefix, all taken
    if (tid == 0) s.nsel = 0;
    for (int shift = 56; shift >= 0 && taken < spec; shift -= 8) {
        for (uint32_t i = tid; i < 256u; i += nt) count[i] = 0;
        __syncthreads();
        for (uint32_t i = tid; i < ncand; i += nt) {
            const uint64_t k = s.ckey[i];
            if ((k & mask) == prefix) atomicAdd(&count[static_cast<uint32_t>(k >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (tid < 64) {  // lane l: buckets 255 - 4 l down to 252 - 4 l
            uint32_t c = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) c += count[255u - 4u * lane - static_cast<uint32_t>(q)];
            const uint32_t incl = wave_incl_sum(c), before = incl - c;
            const unsigned long long hit = __ballot(taken + incl >= spec);
            if (lane == static_cast<uint32_t>(__builtin_ctzll(hit))) {  // the total reaches it: some lane hits
                uint32_t above = before, b = 255u - 4u * lane;
                for (int q = 0; q < 4; ++q, --b) {
                    if (taken + above + count[b] >= spec) break;
                    above += count[b];
                }
                s.band = b;
                s.above = above;
            }
        }
        __syncthreads();
        const uint32_t b = s.band, above = s.above, cb = count[b];  // read before the counts are cleared again
        // every matching candidate above bucket b is in
        for (uint32_t i = tid; i < ncand; i += nt) {
            const uint64_t k = s.ckey[i];
            if ((k & mask) == prefix && (static_cast<uint32_t>(k >> shift) & 255u) > b) {
                const uint32_t at = atomicAdd(&s.nsel, 1u);
                s.skey[at] = k;
                s.scand[at] = s.cand[i];
            }
        }
        taken += above;
        prefix |= static_cast<uint64_t>(b) << shift;
        mask |= uint64_t(255) << shift;
        __syncthreads();
        if (taken + cb == spec) {  // uniform: bucket b completes the selection (always so once the key is whole)
            for (uint32_t i = tid; i < ncand; i += nt) {
                const uint64_t k = s.ckey[i];
                if ((k & mask) == prefix) {
                    const uint32_t at = atomicAdd(&s.nsel, 1u);
                    s.skey[at] = k;
                    s.scand[at] = s.cand[i];
                }
            }
            taken = spec;
            __syncthreads();
        }
    }
    if (tid < spec) {  // the selected ones in key order
        const uint64_t ki = s.skey[tid];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < spec; ++j) rank += s.skey[j] > ki ? 1u : 0u;
        s.job_t[1 + rank] = s.scand[tid];
    }
}

// The commits applied to the tree (tree.rs:143-177) by waves w0 .. w0 + nw - 1 of the block (nw >= 2): wave w0
// writes the new nodes and then, once they have landed, the links into nodes split again (a later commit of the step
// may split a leaf a node of the same step points to); the other waves write the changed leaves.
template <uint32_t MAXL>
__device__ void apply_commits(const GrowState &g, const AdvShared<MAXL> &s, uint32_t n0, uint32_t nc, uint32_t n,
                              uint32_t w0, uint32_t nw) {
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const TreeDev &t = g.tree;
    if (wave == w0) {
        for (uint32_t c = lane; c < nc; c += 64u) {
            const TLeaf &p = g.tl[s.ck[c]];
            const SplitOut &info = p.best;
            const uint32_t node = n0 - 1 + c;
            t.split_feature[node] = info.feature;
#pragma unroll
            for (uint32_t w = 0; w < 8; ++w) t.left_bins[static_cast<size_t>(node) * 8 + w] = left_bins_word(info, w, info.wide);
            t.split_gain[node] = static_cast<float>(info.gain + g.cfg.min_gain_to_split);
            t.threshold_bin[node] = info.threshold;
            t.default_left[node] = static_cast<uint8_t>(info.default_left);
            t.left_child[node] = ~static_cast<int32_t>(s.cx[c]);
            t.right_child[node] = ~static_cast<int32_t>(n0 + c);
            t.internal_weight[node] = p.weight;
            t.internal_value[node] = p.value;
            t.internal_count[node] = p.cnt;
        }
        __builtin_amdgcn_s_waitcnt(0);  // the nodes' children have landed before the links overwrite some
        for (uint32_t c = lane; c < nc; c += 64u) {
            const int32_t pn = s.cpn[c];
            if (pn < 0) continue;
            if (s.cleft[c]) t.left_child[pn] = static_cast<int32_t>(n0 - 1 + c);
            else t.right_child[pn] = static_cast<int32_t>(n0 - 1 + c);
        }
        return;
    }
    if (wave <= w0 || wave >= w0 + nw) return;
    for (uint32_t id = (wave - w0 - 1) * 64u + lane; id < n; id += (nw - 1) * 64u) {
        if (!s.touched[id]) continue;
        const uint32_t k = s.leaf_t[id];
        const TLeaf &l = g.tl[k];
        t.leaf_value[id] = l.value;
        t.leaf_weight[id] = l.weight;
        t.leaf_count[id] = l.cnt;
        t.leaf_parent[id] = s.pnode[id];
        t.leaf_depth[id] = l.depth;
        t.leaf_range[2 * id] = l.begin;
        t.leaf_range[2 * id + 1] = l.count;
        g.leaf_t[id] = static_cast<int32_t>(k);
        g.leaf_left[id] = s.is_left[id];
    }
}

// Each speculative leaf's bound after the replay: the smallest gain (as f32) on its path from the committed leaf
// above it (that leaf included) down to it, the order in which best_leaf would reach it (a leaf is committed before
// another whose bound is lower, since every leaf on its path must be committed first and each is the largest gain
// when it is). Into the .x half of each leaf's s.gain word (the replay's exact gains are no longer read), the leaf's
// gain as f32 in .y; leaves not below a committed leaf (the committed tree's nodes) get -1. Pointer jumping over
// parent links kept in the s.ckey words: a leaf's link is its parent until it meets a committed leaf, each round
// takes the minimum with its link's and doubles the link's reach, so ceil(log2(depth)) + 1 rounds end it (at most
// 16, which covers any tree of the sizes here). Before the rounds, each leaf walks up to BOUND_WALK links by itself, which
// ends most trees' without a round (a round is two barriers). Block-wide.
constexpr int BOUND_WALK = 8;
template <uint32_t MAXL>
__device__ void frontier_bounds(AdvShared<MAXL> &s, uint32_t ntent, uint32_t n) {
    constexpr uint32_t PER = (AdvShared<MAXL>::TCAP + 511) / 512;  // leaves a thread (blocks of at least 512)
    constexpr uint32_t NONE = 0xffffu, UNDER = 1u << 16;             // link: bits 0-15; bit 16: below a committed leaf
    static_assert(AdvShared<MAXL>::TCAP < NONE, "leaf links fit 16 bits");
    static_assert(sizeof(s.ckey) >= sizeof(uint32_t) * AdvShared<MAXL>::TCAP, "the links fit the key words");
    uint32_t *link = reinterpret_cast<uint32_t *>(s.ckey);
    float2 *bw = reinterpret_cast<float2 *>(s.gain);
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    for (uint32_t k = tid; k < ntent; k += nt) link[k] = NONE;
    __syncthreads();
    for (uint32_t k = tid; k < ntent; k += nt) {
        const uint32_t m = s.meta[k];
        const double gk = s.gain[k];
        if (((m >> 1) & 3u) != T_LEAF && (m >> 3) != 0u) {  // expanded or planned: its children are kid, kid + 1
            const uint32_t kid = (m >> 3) - 1u;
            link[kid] = k;
            link[kid + 1] = k;
        }
        const float gf = (m & 1u) && gk == gk ? static_cast<float>(gk) : -1.0f;
        bw[k] = make_float2(gf, gf);  // read after the barrier below
    }
    __syncthreads();
    for (uint32_t id = tid; id < n; id += nt) link[s.leaf_t[id]] = UNDER | NONE;  // the committed leaves: the path's top
    __syncthreads();
    for (int round = -1; round < 16; ++round) {
        uint32_t nl[PER];
        float nb[PER];
        bool moved = false;
        if (round < 0) {
#pragma unroll
            for (uint32_t i = 0; i < PER; ++i) {
                const uint32_t k = tid + nt * i;
                nl[i] = NONE;
                nb[i] = 0.0f;
                if (k >= ntent) continue;
                uint32_t l = link[k];
                float b = bw[k].x;
                for (int w = 0; w < BOUND_WALK && (l & NONE) != NONE; ++w) {
                    const uint32_t u = l & NONE, lu = link[u];
                    b = fminf(b, bw[u].y);  // .y: the leaf's own gain, which no round changes
                    l = (l & UNDER) | lu;
                }
                nl[i] = l;
                nb[i] = b;
                moved = moved || (l & NONE) != NONE;
            }
        } else
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t k = tid + nt * i;
            nl[i] = NONE;
            nb[i] = 0.0f;
            if (k >= ntent) continue;
            const uint32_t l = link[k];
            nl[i] = l;
            nb[i] = bw[k].x;
            if ((l & NONE) != NONE) {
                const uint32_t u = l & NONE, lu = link[u];
                nb[i] = fminf(nb[i], bw[u].x);
                nl[i] = (l & UNDER) | (lu & UNDER) | (lu & NONE);
                moved = true;
            }
        }
        const bool any = __syncthreads_or(moved ? 1 : 0) != 0;
#pragma unroll
        for (uint32_t i = 0; i < PER; ++i) {
            const uint32_t k = tid + nt * i;
            if (k < ntent) {
                link[k] = nl[i];
                bw[k].x = nb[i];
            }
        }
        __syncthreads();
        if (!any) break;
    }
    for (uint32_t k = tid; k < ntent; k += nt)
        if (!(link[k] & UNDER)) bw[k].x = -1.0f;
    __syncthreads();
}

// The bits of the R-th highest bound (frontier_bounds, positive f32 bits order as the values) among the leaves the
// tree may still commit: the unexpanded leaves with a split and a positive gain (the blocker among them) and the
// expanded ones not yet committed; 0 when there are fewer than R of them. best_leaf commits a leaf before any of
// lower bound, so a leaf below this bound is not among the next R commits and expanding it now is wasted. A radix
// selection over the bound bits, 8 at a time from the top (s.crank: 256 counts). Block-wide.
template <uint32_t MAXL>
__device__ uint32_t pool_threshold(AdvShared<MAXL> &s, uint32_t ntent, uint32_t R) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, nt = blockDim.x;
    const float2 *bw = reinterpret_cast<const float2 *>(s.gain);
    uint32_t *count = s.crank;
    auto bound_bits = [&](uint32_t k) -> uint32_t {  // 0: not in the pool
        const uint32_t m = s.meta[k], st = (m >> 1) & 3u;
        const float2 b = bw[k];
        const bool in = b.x > 0.0f && (st == T_EXPANDED || (st == T_LEAF && (m & 1u) && b.y > 0.0f));
        return in ? __float_as_uint(b.x) : 0u;
    };
    // fewer than R in the pool (early in a tree): every candidate may be committed
    if (tid == 0) s.band = 0;
    __syncthreads();
    uint32_t mine = 0;
    for (uint32_t k = tid; k < ntent; k += nt) mine += bound_bits(k) ? 1u : 0u;
    mine = wave_total(mine);
    if (lane == 0 && mine) atomicAdd(&s.band, mine);
    __syncthreads();
    if (s.band < R) return 0u;  // uniform
    __syncthreads();  // s.band is read before the rounds below set it
    uint32_t prefix = 0, mask = 0, above = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (uint32_t i = tid; i < 256u; i += nt) count[i] = 0;
        __syncthreads();
        for (uint32_t k = tid; k < ntent; k += nt) {
            const uint32_t v = bound_bits(k);
            if (v && (v & mask) == prefix) atomicAdd(&count[(v >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (tid < 64) {  // lane l: buckets 255 - 4 l down to 252 - 4 l
            uint32_t c = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) c += count[255u - 4u * lane - static_cast<uint32_t>(q)];
            const uint32_t incl = wave_incl_sum(c), before = incl - c;
            const unsigned long long hit = __ballot(above + incl >= R);
            if (!hit) {
                if (lane == 0) s.band = 256u;  // fewer than R in the pool
            } else if (lane == static_cast<uint32_t>(__builtin_ctzll(hit))) {
                uint32_t acc = above + before, b = 255u - 4u * lane;
                for (int q = 0; q < 4; ++q, --b) {
                    if (acc + count[b] >= R) break;
                    acc += count[b];
                }
                s.band = b;
                s.above = acc;
            }
        }
        __syncthreads();
        const uint32_t b = s.band;
        if (b == 256u) return 0u;  // uniform
        above = s.above;
        prefix |= b << shift;
        mask |= 255u << shift;
        __syncthreads();  // the counts are read before the next round clears them
    }
    return prefix;
}

// The control block's words that advance reads.
struct AdvState {
    uint32_t n0, ntent, pending0, slot0, epoch0, expansions0, steps0;
};
__device__ __forceinline__ AdvState adv_state(const GrowCtl *ctl) {
    return AdvState{ctl->num_leaves, ctl->ntent, ctl->pending, ctl->next_slot, ctl->epoch, ctl->expansions, ctl->steps};
}

// advance's LDS copies of the first `ntk` speculative leaves' keys and of the committed leaves. Block-wide; the caller
// synchronizes.
template <uint32_t MAXL>
__device__ __forceinline__ void advance_load(const GrowState &g, AdvShared<MAXL> &s, uint32_t n0, uint32_t ntk) {
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    for (uint32_t k = tid; k < ntk; k += nt) {
        const TKey key = g.tk[k];
        s.gain[k] = key.gain;
        s.meta[k] = key_meta(key);
    }
    for (uint32_t id = tid; id < n0; id += nt) {
        s.leaf_t[id] = static_cast<uint16_t>(g.leaf_t[id]);
        s.pnode[id] = static_cast<int16_t>(g.tree.leaf_parent[id]);
        s.is_left[id] = g.leaf_left[id];
        s.touched[id] = 0;
    }
    if (tid == 0) {
        s.ncand = 0;
        s.nnan = 0;
    }
}

// With every key in LDS (advance_load), after a barrier.
template <uint32_t MAXL>
__device__ void advance(const GrowState &g, StepPlan &next, AdvShared<MAXL> &s, const AdvState &st) {
    GrowCtl *ctl = g.ctl;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, nt = blockDim.x;
    const uint32_t n0 = st.n0, ntent = st.ntent, L = g.num_leaves;
    const uint32_t pending0 = st.pending0, slot0 = st.slot0, epoch0 = st.epoch0;
    const uint32_t expansions0 = st.expansions0, steps0 = st.steps0;
    // the replay keys of the committed leaves for replay_lds and replay_reg (trees of more than 128 leaves), by the
    // whole block
    if (MAXL > LEAVES_SMALL || L > 128) {
        using Key = std::remove_cv_t<std::remove_reference_t<decltype(s.key[0])>>;
        for (uint32_t id = tid; id < MAXL; id += nt) {
            Key key = 0;
            if (id < n0) {
                const uint32_t t = s.leaf_t[id];
                const double gj = s.gain[t];
                const uint32_t m = s.meta[t];
                key = leaf_key<Key>(gj, m, id);
                if ((m & 1u) && gj != gj) atomicAdd(&s.nnan, 1u);
                if constexpr (MAXL > LEAVES_SMALL) s.leaf_m[id] = m;
            }
            s.key[id] = key;
        }
        if constexpr (MAXL <= LEAVES_SMALL) {  // replay_reg's records of the expanded speculative leaves
            for (uint32_t k = tid; k < ntent; k += nt) {
                const uint32_t m = s.meta[k];
                if (((m >> 1) & 3u) != T_EXPANDED) continue;
                const uint32_t kid = (m >> 3) - 1u;
                uint32_t c[2];
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    const double gc = s.gain[kid + i];
                    const uint32_t mc = s.meta[kid + i];
                    c[i] = (replay_key<11>(gc, mc, 0) & ~2047u) | ((mc & 1u) && gc != gc ? 1u : 0u);
                }
                s.crec[k] = make_uint2(c[0], c[1]);
            }
        }
        __syncthreads();
    }

    // -- the replay, one wave, with as few leaves per lane as the tree needs
    if (tid < 64) {
        if constexpr (MAXL <= LEAVES_SMALL) {
            if (L <= 64) replay<1>(s, n0, L);
            else if (L <= 128) replay<2>(s, n0, L);
            else if (L <= 256) replay_reg<4>(s, n0, L);
            else replay_reg<LEAVES_SMALL / 64>(s, n0, L);
        } else {
            if (L <= 1024) replay_lds<16>(s, n0, L);
            else replay_lds<MAXL / 64>(s, n0, L);
        }
    }
    __syncthreads();
    const uint32_t nc = s.ncommit, n = s.n;
    const bool done = s.done != 0;

    if (tid == 0) {
        ctl->num_leaves = n;
        ctl->pending = pending0 - nc;
        if (done) ctl->done = 1;
    }
    if (done) {
        apply_commits(g, s, n0, nc, n, 0, nt >> 6);
        return;
    }

    // -- speculation candidates: unexpanded leaves with a positive gain, the blocker aside, in the order best_leaf
    // would reach them: by bound (frontier_bounds), then gain, then lower leaf
    const uint32_t blocker = s.blocker;
    frontier_bounds<MAXL>(s, ntent, n);
    const uint32_t R = L - n;  // splits left, this step's blocker included
    // The pool holds the candidates, the blocker and the expanded leaves not yet committed (pending0 - nc). With
    // R >= that last count + jcap, fewer than R of them lie above the (jcap - 1)-th highest candidate's bound, so the
    // R-th highest bound cannot leave out any of the candidates a step takes: no selection is needed.
    const uint32_t cut = R >= pending0 - nc + g.jcap ? 0u : pool_threshold<MAXL>(s, ntent, R);
    if (tid == 0) s.neligible = 0;
    __syncthreads();
    const float2 *bw = reinterpret_cast<const float2 *>(s.gain);
    for (uint32_t k = tid; k < ntent; k += nt) {
        const uint32_t m = s.meta[k];
        const float2 b = bw[k];
        if ((m & 1u) && ((m >> 1) & 3u) == T_LEAF && b.y > 0.0f && b.x > 0.0f && k != blocker) {
            if (__float_as_uint(b.x) >= cut) atomicAdd(&s.neligible, 1u);
            const uint32_t at = atomicAdd(&s.ncand, 1u);
            s.cand[at] = static_cast<uint16_t>(k);
            // positive f32 bits order as the values: bound, then the top 19 bits of the gain below the sign, then
            // the lower leaf (13 bits: leaf ids are below 8192)
            s.ckey[at] = (static_cast<uint64_t>(__float_as_uint(b.x)) << 32) |
                         (static_cast<uint64_t>(__float_as_uint(b.y) >> 12) << 13) | (8191u - k);
            s.crank[at] = 0;
        }
    }
    __syncthreads();
    const uint32_t ncand = s.ncand;
    const uint32_t pending = pending0 - nc;
    // the candidates among the R leaves of highest bound (pool_threshold), at most jcap - 1; being the highest keys,
    // the ones the selection below takes are exactly those
    uint32_t spec = s.neligible;
    if (spec > g.jcap - 1) spec = g.jcap - 1;
    // room for this step and every later blocker (each commits, so at most R of them in all)
    const uint32_t free_t = g.tcap - ntent, free_s = g.nslots - slot0;
    const uint32_t room_t = free_t >= 2 * R ? (free_t - 2 * R) / 2 : 0u, room_s = free_s >= R ? free_s - R : 0u;
    if (spec > room_t) spec = room_t;
    if (spec > room_s) spec = room_s;
    if (spec > ncand) spec = ncand;
    // The spec highest keys; the blocker is job 0. Which leaves are expanded early changes no result (every
    // expansion is the one its leaf gets when the replay reaches it), only the work done ahead. Up to 512 candidates,
    // each one's rank (keys above its own) is summed over `nsl` slices of the others, one thread each; beyond that
    // (trees of thousands of leaves), a radix selection finds the spec-th key in linear passes.
    if (spec <= SPEC_FEW) {
        if (tid < 64) top_few(s, ncand, spec);
    } else if (ncand <= 512u) {
        const uint32_t nsl = ncand && ncand < nt ? nt / ncand : 1u;
        for (uint32_t w = tid; w < ncand * nsl; w += nt) {
            const uint32_t i = w % ncand, sl = w / ncand;
            const uint64_t ki = s.ckey[i];
            uint32_t rank = 0;
#pragma unroll 8
            for (uint32_t j = sl; j < ncand; j += nsl) rank += s.ckey[j] > ki ? 1u : 0u;
            atomicAdd(&s.crank[i], rank);
        }
        __syncthreads();
        for (uint32_t i = tid; i < ncand; i += nt)
            if (s.crank[i] < spec) s.job_t[1 + s.crank[i]] = s.cand[i];
    } else {
        select_top<MAXL>(s, ncand, spec);
    }
    if (tid == 0) {
        s.job_t[0] = static_cast<uint16_t>(blocker);
        s.njobs = 1 + spec;
    }
    __syncthreads();
    const uint32_t njobs = s.njobs;
    if (free_t < 2 || free_s < 1) {  // no room even for the blocker: the sizes above make this unreachable
        if (tid == 0) {
            ctl->error = 4;
            ctl->done = 1;
        }
        apply_commits(g, s, n0, nc, n, 0, nt >> 6);
        return;
    }

    // -- the jobs (learner.rs:249-290), one lane each; then prefix sums over the jobs on the same wave. The other
    // waves meanwhile apply the commits to the tree (nothing the plan reads).
    if (tid >= 64) apply_commits(g, s, n0, nc, n, 1, (nt >> 6) - 1);
    if (tid < 64) {
        const bool on = lane < njobs;
        JobPlan J = {};
        uint32_t hist = 0, ntiles = 0;
        float cost = 0.0f;
        if (on) {
            const uint32_t tt = s.job_t[lane];
            const TLeaf &l = g.tl[tt];
            const SplitOut &info = l.best;
            J.t = tt;
            J.begin = l.begin;
            J.count = l.count;
            J.col = info.col;
            J.wide = info.wide;
#pragma unroll
            for (uint32_t w = 0; w < 8; ++w) J.left_bins[w] = left_bins_word(info, w, J.wide);
            J.built_side = info.left_count <= info.right_count ? 0u : 1u;
            hist = (l.slot >= 0 && depth_allows(g, l.depth + 1)) ? 1u : 0u;
            J.hist = hist;
            J.parent_slot = l.slot;
            J.src_buf = l.buf;
            J.src_rev = l.rev;
            ntiles = (l.count + STEP_TILE - 1) / STEP_TILE;
            J.ntiles = ntiles;
            // the job's k_step_rows work in tiles: every tile partitions, its rows' split bins costing more the sparser
            // the leaf's rows lie (a line a row once they are sparser than one in 128: sparse_weight at most), and the
            // built child's share of its rows is histogrammed besides (hist_weight a tile of built rows)
            const double lc = static_cast<double>(info.left_count), rc = static_cast<double>(info.right_count);
            const double built = hist && lc + rc > 0.0 ? (lc <= rc ? lc : rc) / (lc + rc) : 0.0;
            const double spread = static_cast<double>(g.tl[0].count) / (128.0 * static_cast<double>(l.count ? l.count : 1u));
            cost = static_cast<float>(ntiles) * (1.0f + g.sparse_weight * static_cast<float>(spread < 1.0 ? spread : 1.0) +
                                                 g.hist_weight * static_cast<float>(built));
            J.parent_count = l.cnt;
            J.child_ug[0] = info.left_grad;
            J.child_uh[0] = info.left_hess;
            J.child_ug[1] = info.right_grad;
            J.child_uh[1] = info.right_hess;
            J.child_out[0] = info.left_output;
            J.child_out[1] = info.right_output;
            J.depth = l.depth + 1;
            J.kid = static_cast<int32_t>(ntent + 2 * lane);
        }
        // exclusive prefixes over lanes 0..njobs-1 (one wave)
        const uint32_t hist_before = wave_excl_sum(hist);
        const uint32_t tiles_before = wave_excl_sum(ntiles);
        const uint32_t total_tiles = wave_total(ntiles);
        const float total_cost = wave_total_f32(cost);
        uint32_t groups = 0;
        if (on) {  // workgroups in proportion to the jobs' work (a job's tiles go to its workgroups by ticket), so that
            // no job's workgroups run long; the rounding up in each job costs at most one workgroup a job, so with
            // target - njobs for the shares the step fits in one round of workgroups (one per compute unit). At most
            // tile_cap tiles a workgroup (its i32 sums), and no more workgroups than tiles.
            const uint32_t share = g.target_groups > njobs ? g.target_groups - njobs : 1u;
            if (total_tiles <= g.target_groups) {
                groups = ntiles;
            } else {
                const float per_cost = total_cost / static_cast<float>(share);
                groups = static_cast<uint32_t>(__builtin_ceilf(cost / per_cost));
                const uint32_t least = (ntiles + g.tile_cap - 1) / g.tile_cap;
                groups = groups < least ? least : groups;
                groups = groups > ntiles ? ntiles : groups;
            }
            if (groups == 0) groups = 1;
        }
        const uint32_t groups_before = wave_excl_sum(groups);
        const uint32_t total_groups = wave_total(groups);
        uint32_t red = 0;
        if (on) {
            J.tile_base = tiles_before;
            J.groups = groups;
            J.group_base = groups_before;
            J.packed = (ntiles <= groups && g.flush_rows >= STEP_TILE) ? 1u : 0u;
            J.ways = reduce_ways(groups);
            red = hist ? g.ncgw * J.ways : 0u;
            J.built_slot = hist ? static_cast<int32_t>(slot0 + hist_before) : -1;
        }
        const uint32_t red_before = wave_excl_sum(red), total_red = wave_total(red);
        const uint32_t nhist = wave_total(hist);
        uint32_t ways = hist ? (groups > CHILD_SPLIT ? min(CHILD_WAYS, (groups + CHILD_SHARE - 1) / CHILD_SHARE) : 1u) : 0u;
        if (wave_total(ways) > CHILD_MAX) ways = hist;  // uniform
        const uint32_t share_before = wave_excl_sum(ways), total_shares = wave_total(ways);
        const uint32_t scratch_before = wave_excl_sum(ways > 1u ? ways : 0u);
        if (on) {
            J.red_base = red_before;
            const uint32_t scan_before = hist_before * g.nwide;
            J.scan_base = scan_before;
            next.group_base[lane] = J.group_base;
            next.red_base[lane] = red_before;
            next.scan_base[lane] = scan_before;
            J.ticket = 0;
            J.left = 0;
            next.jobs[lane] = J;
            next.pairs[lane] = 0;
            const uint32_t per = ways ? (groups + ways - 1) / ways : 0u;
            for (uint32_t w = 0; w < ways; ++w) {
                const uint32_t b = min(w * per, groups);
                next.child[share_before + w] = ChildJob{lane, J.t, J.built_side, J.group_base + b, min(per, groups - b), ways, w, scratch_before,
                                                        J.parent_slot, J.built_slot, J.kid, J.parent_count,
                                                        {J.child_ug[0], J.child_ug[1]}, {J.child_uh[0], J.child_uh[1]}};
            }
            g.tl[J.t].state = T_PLANNED;
            g.tl[J.t].kid = J.kid;
            g.tk[J.t].state = T_PLANNED;
            g.tk[J.t].kid = J.kid;
        }
        if (lane == 0) {
            next.njobs = njobs;
            next.total_groups = total_groups;
            next.total_child = total_shares * g.ncgb;
            next.total_red = total_red;
            next.total_scan = nhist * g.nwide;
            next.epoch = epoch0 + 1;
            ctl->epoch = epoch0 + 1;
            ctl->ntent = ntent + 2 * njobs;
            ctl->next_slot = slot0 + nhist;
            ctl->pending = pending + njobs;
            ctl->expansions = expansions0 + njobs;
            ctl->steps = steps0 + 1;
        }
    }
}

// After a grown tree's steps: when the tree is complete with at least one split, its nodes for k_tree_leaves and
// k_add_tree (as the host builds them from the tree it reads back: the split's bins, the column of its feature,
// the children), its leaf sums zeroed, and *gate = its leaves; *gate = 0 otherwise (an unfinished tree or one
// that never split: the gated kernels after it do nothing). Every node is checked as the host checks an uploaded
// tree (a known feature; an internal child after its parent, a leaf child among the leaves), so the walks over it
// end; a malformed tree flags ctl->error = 6 and closes the gate. *gate_out: the gate, for the host. A nonzero
// *veto (when given: the iteration's gradients are to be made again) closes the gate too. One block.
__global__ void k_tree_nodes(GrowState g, DevNode *nodes, unsigned long long *sums, uint32_t *gate, double *gate_out,
                             const uint32_t *veto) {
    __shared__ uint32_t bad;
    GrowCtl *ctl = g.ctl;
    const uint32_t n = ctl->done && !ctl->error && !(veto && *veto) ? ctl->num_leaves : 0u;
    const uint32_t nl = n > 1u && n <= GROW_MAX_LEAVES ? n : 0u, nn = nl ? nl - 1u : 0u;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nn; k += blockDim.x) {
        DevNode d;
#pragma unroll
        for (int w = 0; w < 8; ++w) d.left_bins[w] = g.tree.left_bins[static_cast<size_t>(k) * 8 + w];
        const int32_t f = g.tree.split_feature[k];
        d.feature = f >= 0 && static_cast<uint32_t>(f) < g.nf ? g.feats[f].col : 0u;
        d.left = g.tree.left_child[k];
        d.right = g.tree.right_child[k];
        d.wide = f >= 0 && static_cast<uint32_t>(f) < g.nf ? g.feats[f].wide : 0u;
        nodes[k] = d;
        bool ok = f >= 0 && static_cast<uint32_t>(f) < g.nf;
        for (const int32_t c : {d.left, d.right})
            ok = ok && (c >= 0 ? static_cast<uint32_t>(c) > k && static_cast<uint32_t>(c) < nn : static_cast<uint32_t>(~c) < nl);
        if (!ok) atomicOr(&bad, 1u);
    }
    for (uint32_t i = threadIdx.x; i < 2u * nl; i += blockDim.x) sums[i] = 0ull;
    __syncthreads();
    if (threadIdx.x == 0) {
        if (bad) ctl->error = 6;
        *gate = bad ? 0u : nl;
        *gate_out = static_cast<double>(bad ? 0u : nl);
    }
}

// The root's best split (learner.rs:157-163), then the first step's plan. One block of 512 threads; MAXL: the
// largest tree it takes (LEAVES_SMALL or GROW_MAX_LEAVES).
template <uint32_t MAXL>
__global__ __launch_bounds__(512) void k_root_select(GrowState g) {
    __shared__ SplitOut o;
    __shared__ __align__(16) uint8_t scratch[sizeof(AdvShared<MAXL>)];
    AdvShared<MAXL> &s = *reinterpret_cast<AdvShared<MAXL> *>(scratch);
    const AdvState st = adv_state(g.ctl);
    const uint32_t done = g.ctl->done;
    ScanJob job = g.jobs[0];
    select_split(job, job.count, g.nf, g.cfg, grow_sg(g), grow_sh(g), &o, g.splittable);
    if (threadIdx.x == 0) {
        g.tl[0].best = o;
        g.tl[0].has_best = o.found ? 1u : 0u;
        g.tk[0].gain = o.gain;
        g.tk[0].has = o.found ? 1u : 0u;
    }
    if (done) return;
    __syncthreads();
    advance_load(g, s, st.n0, st.ntent);
    __syncthreads();
    advance<MAXL>(g, g.plans[0], s, st);
}

// ---------------------------------------------------------------------------------------------------------
// A split step in two kernels: every job of the step's plan (learner.rs:249-352 for each leaf it expands).
//
// k_step_rows: the stable partition of each job's rows by its BinSplit (cpu.rs:556-599) in one pass, fused with
// its built child's histogram. A job's workgroups take its tiles of STEP_TILE rows in order; a tile's left
// count is published at once, its offset comes from a look-back over the job's earlier tiles (no second pass
// over the rows), its rows are scattered, then its rows of the built child (kept in LDS) are histogrammed as
// k_hist does. Left rows are written first-first from the range's start, right rows last-first from its end, so
// both children are stable; a leaf stored last-first is read back to front by the step that expands it and by
// k_consolidate. Launches for a second or later slab only histogram.
//
// Then, one launch each: k_step_children adds each job's partials, writes the built child's histogram, forms the sibling
// by subtraction (learner.rs:356-371) and scans every (job, feature, child) of the byte slabs (k_step_reduce and
// k_step_scan do so for two-byte slabs); k_step_select, one block, selects both children's splits of every job and runs
// advance.
// ---------------------------------------------------------------------------------------------------------

// A launch takes one slab, or (histogram only) several slabs of one kernel, k1 workgroups each: slab s of the
// launch is the first one's buffers moved by s strides (its rows by bins_stride bytes, its partials by k1
// partials, its formats by k1 entries, its column bins by W * PACK entries).
struct StepArgs {
    const uint8_t *bins;         // the first slab's rows: row r at bins + r * row bytes
    uint64_t bins_stride;
    int32_t *partial;            // its partials, step_partial_stride(W) pairs apart, one per workgroup
    uint32_t *fmt;               // per workgroup: its partial is packed (1) or {g, h} pairs (0)
    const uint32_t *col_bins;    // per slab column: its feature's bins (0 for padding)
    const uint32_t *pos_word;    // a dense slab: per row byte, its LDS word at bin 0 (256 * DP entries a slab)
    uint32_t dw_row;             // a dense slab: dwords per row
    uint32_t k1;                 // workgroups a slab
    const int32_t *gh;           // packed quantized gradients per row
    const uint8_t *colbase;      // column-major bins [feature][rows]
    uint32_t col16;              // two bytes per column-major bin
    uint64_t rows;
    uint32_t *buf0, *buf1;       // the partition buffers
    unsigned long long *status;  // per-tile status words
    StepPlan *plan;              // this step's plan
    GrowCtl *ctl;
    uint32_t flush_rows;
    uint32_t partition;          // 1: this launch partitions (the first slab's alone); 0: histogram only
    uint32_t tile_cap;           // tiles a workgroup takes at most (its i32 sums of the quantized units)
    uint8_t *codes0, *codes1;    // each row's one-byte gradient code beside its id in buf0 / buf1 (packed_code), or
                                 // null: the histograms gather the packed words
};

__device__ __forceinline__ unsigned long long status_word(uint32_t epoch, uint32_t flag, uint32_t value) {
    return (static_cast<unsigned long long>(((epoch & 0x3fffffffu) << 2) | flag) << 32) | value;
}

// Lefts in the tiles before `t`: wave-wide over up to 64 earlier tiles at a time, nearest first, summing
// aggregates until an inclusive prefix. Tile 0 always publishes an inclusive one, and every earlier tile was
// handed to a running block that publishes its aggregate before any wait, so the polling ends; a step that
// still sees no status after LOOKBACK_SPINS polls flags an error instead of waiting on.
__device__ uint32_t lookback(const unsigned long long *status, uint32_t t, uint32_t epoch, GrowCtl *ctl) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t want = epoch & 0x3fffffffu;
    uint32_t prefix = 0, spins = 0;
    int64_t hi = static_cast<int64_t>(t) - 1;
    while (hi >= 0) {
        const int64_t idx = hi - static_cast<int64_t>(lane);
        unsigned long long w = 0;
        if (idx >= 0) w = __hip_atomic_load(status + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t tag = static_cast<uint32_t>(w >> 32);
        const bool ready = idx >= 0 && (tag >> 2) == want && (tag & 3u) != 0u;
        const unsigned long long waiting = __ballot(idx >= 0 && !ready);
        const unsigned long long incl = __ballot(ready && (tag & 3u) == ST_INCL);
        const uint32_t first_incl = incl ? static_cast<uint32_t>(__builtin_ctzll(incl)) : 64u;
        const uint32_t first_wait = waiting ? static_cast<uint32_t>(__builtin_ctzll(waiting)) : 64u;
        if (first_wait < first_incl) {
            if (++spins > LOOKBACK_SPINS) {
                if (lane == 0) ctl->error = 3;
                return prefix;
            }
            __builtin_amdgcn_s_sleep(2);
            continue;
        }
        const uint32_t take = first_incl < 64u ? first_incl + 1u : 64u;
        uint32_t v = (lane < take && idx >= 0) ? static_cast<uint32_t>(w) : 0u;
        for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
        prefix += v;
        if (first_incl < 64u) break;
        hi -= 64;
    }
    return prefix;
}

// The 4 x 4 transpose of a quad of lanes' v[0 .. 3]: lane c4 = lane % 4 leaves with v[c4] of lanes 0 .. 3 of its quad. At
// level b a lane keeps the elements whose index bit b matches its own and swaps the other two with lane c4 ^ b; every
// choice is one select on a lane bit.
__device__ __forceinline__ int4 quad_transpose(int32_t v0, int32_t v1, int32_t v2, int32_t v3) {
    const uint32_t c4 = threadIdx.x & 3u;
    {
        const bool hi = (c4 & 1u) != 0;
        const int32_t t0 = __builtin_amdgcn_update_dpp(0, hi ? v0 : v1, 0xB1, 0xf, 0xf, false);
        const int32_t t1 = __builtin_amdgcn_update_dpp(0, hi ? v2 : v3, 0xB1, 0xf, 0xf, false);
        const int32_t n0 = hi ? t0 : v0, n1 = hi ? v1 : t0, n2 = hi ? t1 : v2, n3 = hi ? v3 : t1;
        v0 = n0;
        v1 = n1;
        v2 = n2;
        v3 = n3;
    }
    {
        const bool hi = (c4 & 2u) != 0;
        const int32_t t0 = __builtin_amdgcn_update_dpp(0, hi ? v0 : v2, 0x4E, 0xf, 0xf, false);
        const int32_t t1 = __builtin_amdgcn_update_dpp(0, hi ? v1 : v3, 0x4E, 0xf, 0xf, false);
        const int32_t n0 = hi ? t0 : v0, n1 = hi ? t1 : v1, n2 = hi ? v2 : t0, n3 = hi ? v3 : t1;
        v0 = n0;
        v1 = n1;
        v2 = n2;
        v3 = n3;
    }
    return make_int4(v0, v1, v2, v3);
}

// Moves the packed 16/16 LDS words (Q32: the separate g and h counters) into a workgroup's {g, h} partial (stored, or
// added to what an earlier flush stored) and zeroes them. The partial is two planes, the g sums then (64 W int4s on) the
// h sums, each in the order of a packed partial (store_packed_partial), so that a reduce's wave reads either in whole
// lines (as {g, h} pairs bin-major, each thread's 32 bytes lay in a line of its own: the first step of a 10M x 128 tree,
// one job over 288 such partials, took k_step_children 165 us, 88 in planes). `col_bins`: the most bins of the thread's quad
// of columns; bins past them are not stored. Block-wide.
template <int W, bool Q32 = false>
__device__ __forceinline__ void flush_pairs(int32_t *lds, int4 *planes, uint32_t col_bins, bool add) {
    constexpr int SLOTS = 256 * W / 1024;
    const uint32_t tid = threadIdx.x;
    __syncthreads();
#pragma unroll 2
    for (int it = 0; it < SLOTS / 4; ++it) {
        const uint32_t k = tid + 1024u * it, c = k % W, q = k / W;
        int32_t gq[4], hq[4];
#pragma unroll
        for (uint32_t b = 0; b < 4; ++b) {
            const uint32_t slot = (4 * q + b) * W + c;
            const int32_t v = lds[slot];
            lds[slot] = 0;
            if constexpr (Q32) {
                gq[b] = v;
                hq[b] = lds[256 * W + slot];
                lds[256 * W + slot] = 0;
            } else {
                gq[b] = packed_g(v);
                hq[b] = packed_h(v, gq[b]);
            }
        }
        int4 g4 = quad_transpose(gq[0], gq[1], gq[2], gq[3]), h4 = quad_transpose(hq[0], hq[1], hq[2], hq[3]);
        if (4 * q + (tid & 3u) < col_bins) {
            int4 *pg = planes + q * W + c, *ph = pg + 64 * W;
            if (add) {
                const int4 og = *pg, oh = *ph;
                g4 = make_int4(g4.x + og.x, g4.y + og.y, g4.z + og.z, g4.w + og.w);
                h4 = make_int4(h4.x + oh.x, h4.y + oh.y, h4.z + oh.z, h4.w + oh.w);
            }
            *pg = g4;
            *ph = h4;
        }
    }
    __syncthreads();
}
// The most bins of the thread's quad of columns (tid % W and its three neighbours), for flush_pairs.
template <int W>
__device__ __forceinline__ uint32_t quad_bins(const uint32_t *col_bins) {
    const uint4 b = *reinterpret_cast<const uint4 *>(col_bins + (threadIdx.x % W & ~3u));
    return max(max(b.x, b.y), max(b.z, b.w));
}

// A job of the step as one workgroup of k_step_rows sees it.
struct StepView {
    JobPlan *job;
    unsigned long long *status;  // the job's tile status words
    uint32_t begin, count, ntiles, groups;
    const uint32_t *src;
    uint32_t *dst;
    bool rev, hist, partition;
    const uint8_t *col;
    uint32_t col16;       // column-major bins are two bytes
    uint32_t wide;        // the split is a wide feature's numerical rule
    uint32_t built_left;  // 1: the left child is histogrammed
    uint32_t epoch;
    const uint8_t *csrc;  // the rows' gradient codes beside src, and beside dst (CODES)
    uint8_t *cdst;
};

struct StepShared {
    uint32_t list[STEP_TILE];  // the tile's rows of the built child
    uint8_t codes[STEP_TILE];  // and their gradient codes (CODES)
    uint32_t wl[TILE_RPT][16];  // left counts per (sub-tile, wave)
    uint32_t left_bins[8];     // the split's bins that go left
    uint32_t tile, tile2, prefix;
};

// One partition tile in parts. tile_rows and tile_bins read its rows in the leaf's order (TILE_RPT per thread:
// positions tid, 1024 + tid, ...) and their split-feature bins, so that a workgroup can load its next tile while
// it works on this one; tile_front ranks the lefts, publishes the tile's left count and lists its rows of the built
// child in sh.list, in order; tile_lookback (wave 0) takes the tile's offset from the look-back; tile_scatter
// writes its rows, left first-first and right last-first. Between the last two the other waves histogram the
// listed rows.
struct TileRows {
    uint32_t row[TILE_RPT], bin[TILE_RPT];
    uint32_t codes;  // CODES: row j's gradient code in byte j
};

template <bool CODES>
__device__ __forceinline__ void tile_rows(const StepView &v, uint32_t t, TileRows &r) {
    const uint32_t t0 = t * STEP_TILE;
    static_assert(TILE_RPT <= 4, "a tile's codes fit one word a thread");
    if constexpr (CODES) r.codes = 0;
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) {
        const uint32_t i = t0 + j * 1024 + threadIdx.x;
        const uint32_t ic = i < v.count ? i : v.count - 1;
        const uint32_t at = v.rev ? v.begin + v.count - 1 - ic : v.begin + ic;
        r.row[j] = v.src[at];
        if constexpr (CODES) r.codes |= static_cast<uint32_t>(v.csrc[at]) << (8 * j);
    }
}

__device__ __forceinline__ void tile_bins(const StepView &v, TileRows &r) {
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) r.bin[j] = col_bin(v.col, v.col16, r.row[j]);
}

struct TileState {
    uint32_t row[TILE_RPT], lrank[TILE_RPT];  // lrank: lefts before the row in the tile
    uint32_t codes;                           // CODES: row j's gradient code in byte j
    bool ok[TILE_RPT], left[TILE_RPT];
    uint32_t tile_left;
};

// Returns the rows listed. Block-wide; the list is complete on return.
template <bool CODES>
__device__ __forceinline__ uint32_t tile_front(const StepView &v, uint32_t t, const TileRows &r, TileState &st,
                                               StepShared &sh) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint64_t below_mask = (1ull << lane) - 1ull;
    const uint32_t t0 = t * STEP_TILE;
    const uint32_t valid = v.count - t0 < STEP_TILE ? v.count - t0 : STEP_TILE;
    if constexpr (CODES) st.codes = r.codes;
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) {
        st.ok[j] = t0 + j * 1024 + tid < v.count;
        st.row[j] = r.row[j];
        st.left[j] = st.ok[j] && rule_left(sh.left_bins, v.wide, r.bin[j]);
    }
    uint32_t below[TILE_RPT];
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) {
        unsigned long long m = __ballot(st.left[j]);
        below[j] = static_cast<uint32_t>(__popcll(m & below_mask));
        if (lane == 0) sh.wl[j][wave] = static_cast<uint32_t>(__popcll(m));
    }
    __syncthreads();
    // lefts before each row of the tile (rows in order: sub-tile, wave, lane)
    uint32_t sub[TILE_RPT], before[TILE_RPT];
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) sub[j] = before[j] = 0;
    for (uint32_t w = 0; w < 16; ++w) {
#pragma unroll
        for (int j = 0; j < TILE_RPT; ++j) {
            const uint32_t c = sh.wl[j][w];
            sub[j] += c;
            before[j] += w < wave ? c : 0u;
        }
    }
    st.tile_left = 0;
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) {
        st.lrank[j] = st.tile_left + before[j] + below[j];
        st.tile_left += sub[j];
    }
    if (v.partition && tid == 0)
        __hip_atomic_store(v.status + t, status_word(v.epoch, t == 0 ? ST_INCL : ST_AGG, st.tile_left), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    if (v.hist) {  // the tile's rows of the built child, in order
#pragma unroll
        for (int j = 0; j < TILE_RPT; ++j) {
            uint32_t pos = j * 1024 + tid;
            if (st.ok[j] && (st.left[j] ? 1u : 0u) == v.built_left) {
                const uint32_t at = v.built_left ? st.lrank[j] : pos - st.lrank[j];
                sh.list[at] = st.row[j];
                if constexpr (CODES) sh.codes[at] = static_cast<uint8_t>(st.codes >> (8 * j));
            }
        }
    }
    __syncthreads();  // the list is complete
    return v.built_left ? st.tile_left : valid - st.tile_left;
}

// The tile's offset into sh.prefix, published as its inclusive count. Wave 0 of a partition launch.
__device__ __forceinline__ void tile_lookback(const StepView &v, const StepArgs &a, uint32_t t, const TileState &st,
                                              StepShared &sh) {
    const uint32_t prefix = t == 0 ? 0u : lookback(v.status, t, v.epoch, a.ctl);
    if ((threadIdx.x & 63u) == 0) {
        if (t > 0)
            __hip_atomic_store(v.status + t, status_word(v.epoch, ST_INCL, prefix + st.tile_left), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        sh.prefix = prefix;
        if (t == v.ntiles - 1) v.job->left = prefix + st.tile_left;
    }
}

// The tile's rows written from the offset in sh.prefix (after a barrier that follows tile_lookback).
template <bool CODES>
__device__ __forceinline__ void tile_scatter(const StepView &v, uint32_t t, const TileState &st, const StepShared &sh) {
    const uint32_t tid = threadIdx.x;
    const uint32_t lp = sh.prefix, rp = t * STEP_TILE - lp;  // lefts and rights before the tile
#pragma unroll
    for (int j = 0; j < TILE_RPT; ++j) {
        if (!st.ok[j]) continue;
        uint32_t at;
        if (st.left[j]) {
            const uint32_t k = lp + st.lrank[j];
            if (k >= v.count) continue;
            at = v.begin + k;
        } else {
            const uint32_t k = rp + (j * 1024 + tid - st.lrank[j]);
            if (k >= v.count) continue;
            at = v.begin + v.count - 1 - k;
        }
        v.dst[at] = st.row[j];
        if constexpr (CODES) v.cdst[at] = static_cast<uint8_t>(st.codes >> (8 * j));
    }
}

// The histogram of rows list[c0, c1) into the packed LDS words: a wave covers RPW = 64 / (W/4) rows per step, a
// lane one dword (4 columns) of a row, with the conflict-free byte rotation of k_hist. Loads are branch-free. NW
// waves take part; `wave` is this one's index among them.
template <int W, bool WIDE, int PACK, bool Q32, int UNROLL, int NW = 16, bool CODES = false>
__device__ __forceinline__ void hist_list(int32_t *lds, const uint32_t *list, uint32_t c0, uint32_t c1, const int32_t *gh,
                                          const uint32_t *bins32, uint32_t wave = threadIdx.x >> 6,
                                          const uint8_t *codes = nullptr) {
    constexpr int DW = WIDE ? W / 8 : W * PACK / 4;
    constexpr int RPW = WAVE / DW;
    constexpr uint32_t STEP = NW * RPW * UNROLL;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t d = lane % DW, rsub = lane / DW;
    const uint32_t rot = (lane & 31u) >> 3;
    uint32_t xs[4], cols[4];
    row_bin_lanes<W, PACK>(d, rot, xs, cols);
    const uint32_t last = c1 - 1;
    for (uint32_t base = c0 + wave * RPW * UNROLL; base < c1; base += STEP) {
        uint32_t r[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) r[u] = list[min(base + u * RPW + rsub, last)];
        uint32_t dw[UNROLL];
        int32_t gq[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            if constexpr (CODES) gq[u] = code_word(codes[min(base + u * RPW + rsub, last)]);
            else gq[u] = gh[r[u]];
            dw[u] = bins32[static_cast<size_t>(r[u]) * DW + d];
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            int32_t gv, hv;
            row_units<Q32>(gq[u], base + u * RPW + rsub < c1, gv, hv);
            if constexpr (WIDE) add_row_bins_wide<W, Q32>(lds, dw[u], gv, hv, d);
            else add_row_bins<W, PACK, Q32>(lds, dw[u], gv, hv, xs, cols);
        }
    }
}

// A workgroup's packed LDS words (every row added, none flushed) stored as its partial: int4 q * W + c holds bin
// 4q + c % 4 of columns (c & ~3) .. (c & ~3) + 3. Task k takes column c = k % W and bins 4q..4q+3 (q = k / W),
// reads LDS across the wave without bank conflicts, and a butterfly transpose in each quad of lanes (the group's 4
// columns) leaves lane c % 4 with bin 4q + c % 4 of all four columns: a wave stores 1 KiB contiguously. The LDS
// words must be complete (after a barrier). Block-wide, 1024 threads.
template <int W>
__device__ __forceinline__ void store_packed_partial(const int32_t *lds, int32_t *partial) {
    constexpr int SLOTS = 256 * W / 1024;
    int4 *out = reinterpret_cast<int4 *>(partial);
    const uint32_t tid = threadIdx.x;
#pragma unroll
    for (int it = 0; it < SLOTS / 4; ++it) {
        const uint32_t k = tid + 1024u * it, c = k % W, q = k / W;
        // column (c & ~3) + j at bin 4q + c % 4
        out[q * W + c] = quad_transpose(lds[(4 * q + 0) * W + c], lds[(4 * q + 1) * W + c], lds[(4 * q + 2) * W + c], lds[(4 * q + 3) * W + c]);
    }
}

// hist_list for a 128-column byte slab with 8 columns a lane: a wave covers 4 rows a step, lane l the dword pair
// l % 16 of row l / 16, so a row is one 128-byte line read by 16 lanes and a wave has 4 * UNROLL rows in flight for
// the registers that 2 * UNROLL rows take at a dword a lane. Each lane rotates its pair right by `rot` bytes once a
// row, so that its k-th add takes byte (k + rot) % 8 (column 8d + (k + rot) % 8). The LDS serves an instruction a
// half-wave (32 lanes, two rows) at a time; with rot = d / 4 + 4 * (row % 2) the 8 lanes of a half-wave whose
// columns share a bank group (d % 4 alike) take 8 different bytes, so no two of its lanes meet in a bank.
template <int UNROLL, int NW = 16, bool CODES = false>
__device__ __forceinline__ void hist_list_pairs(int32_t *lds, const uint32_t *list, uint32_t c0, uint32_t c1,
                                                const int32_t *gh, const uint32_t *bins32, uint32_t wave,
                                                const uint8_t *codes = nullptr) {
    constexpr uint32_t W = 128, RPW = 4;
    constexpr uint32_t STEP = NW * RPW * UNROLL;
    const uint32_t lane = threadIdx.x & 63u, d = lane & 15u, rsub = lane >> 4;
    const uint32_t rot = ((d >> 2) + 4u * (rsub & 1u)) & 7u;
    const bool swap = rot >= 4u;
    const uint32_t sh = 8u * (rot & 3u);
    uint32_t cols[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) cols[k] = 8u * d + ((static_cast<uint32_t>(k) + rot) & 7u);
    const uint2 *rows2 = reinterpret_cast<const uint2 *>(bins32);
    const uint32_t last = c1 - 1;
    for (uint32_t base = c0 + wave * RPW * UNROLL; base < c1; base += STEP) {
        uint32_t r[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) r[u] = list[min(base + u * RPW + rsub, last)];
        uint2 v[UNROLL];
        int32_t gq[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            if constexpr (CODES) gq[u] = code_word(codes[min(base + u * RPW + rsub, last)]);
            else gq[u] = gh[r[u]];
            v[u] = rows2[static_cast<size_t>(r[u]) * (W / 8) + d];
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int32_t gv = base + u * RPW + rsub < c1 ? gq[u] : 0;
            const uint32_t a = swap ? v[u].y : v[u].x, b = swap ? v[u].x : v[u].y;  // the pair rotated by 4 bytes
            const uint32_t lo = __builtin_amdgcn_alignbit(b, a, sh), hi = __builtin_amdgcn_alignbit(a, b, sh);
#pragma unroll
            for (int k = 0; k < 4; ++k) atomicAdd(&lds[__builtin_amdgcn_ubfe(lo, 8u * k, 8u) * W + cols[k]], gv);
#pragma unroll
            for (int k = 0; k < 4; ++k) atomicAdd(&lds[__builtin_amdgcn_ubfe(hi, 8u * k, 8u) * W + cols[4 + k]], gv);
        }
    }
}

// A split step's histogram of list[c0 .. c1): hist_list, or hist_list_dense for a dense slab (DP passes).
template <int W, bool WIDE, int PACK, bool Q32, int DP, int UNROLL, int NW = 16, bool CODES = false>
__device__ __forceinline__ void step_hist(int32_t *lds, const uint32_t *list, uint32_t c0, uint32_t c1, const int32_t *gh,
                                          const uint32_t *bins32, uint32_t dw_row, const uint32_t (&xs)[4],
                                          const uint32_t (&dcols)[DP ? DP : 1][4], uint32_t wave = threadIdx.x >> 6,
                                          const uint8_t *codes = nullptr) {
    if constexpr (DP > 0)
        hist_list_dense<W, DP, NW, CODES>(lds, list, c0, c1, gh, bins32, dw_row, xs, dcols, wave, codes);
    else if constexpr (W == 128 && !WIDE && PACK == 1 && !Q32)
        hist_list_pairs<UNROLL * 3 / 4, NW, CODES>(lds, list, c0, c1, gh, bins32, wave, codes);
    else hist_list<W, WIDE, PACK, Q32, UNROLL, NW, CODES>(lds, list, c0, c1, gh, bins32, wave, codes);
}

// The one-byte gradient codes of a tree's root rows, beside their ids: codes[i] = packed_code(gh[part[i]]) for i in
// [begin, begin + count). The split steps then move each code with its row. Four rows a thread, their loads issued
// together (one row a thread waited on two dependent loads a row).
__global__ void k_gh_codes(const uint32_t *__restrict__ part, const int32_t *__restrict__ gh, uint32_t begin,
                           uint32_t count, uint8_t *__restrict__ codes) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < count; i += 4u * stride) {
        uint32_t r[4];
        int32_t w[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) r[k] = i + k * stride < count ? part[begin + i + k * stride] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) w[k] = i + k * stride < count ? gh[r[k]] : 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (i + k * stride < count) codes[begin + i + k * stride] = packed_code(w[k]);
    }
}

// The LDS words of a k_step_rows instance: the histogram (twice for separate counters) and a dense slab's spare row.
template <int W, bool Q32, int DP>
constexpr int step_lds_words() { return (Q32 ? 2 : 1) * 256 * W + (DP ? W : 0); }

// k_step_rows' work, with the built rows' gradients read from their carried codes (CODES) or gathered.
template <int W, bool WIDE, int PACK, bool Q32, int DP, bool CODES>
__device__ __forceinline__ void step_rows_body(const StepArgs &a, int32_t *lds, StepShared &sh) {
    static_assert(PACK == 1 || (!WIDE && W * PACK <= 256), "a packed row is at most 64 dwords");
    static_assert(!Q32 || W <= 64, "separate g and h counters take twice the LDS");
    static_assert(DP == 0 || (W == 128 && !WIDE && PACK == 1 && !Q32), "a dense slab has 128 byte columns");
    static_assert(!(CODES && Q32), "codes hold small units only");
    constexpr int DW = WIDE ? W / 8 : W * PACK / 4;
    constexpr int RPW = WAVE / DW;
    // rows per lane in multi-tile workgroups (16 at W = 32 with packed columns spills)
    constexpr int UNROLL = (W == 128 || (W == 32 && PACK > 1)) ? 8 : (64 / RPW < 16 ? 64 / RPW : 16);
    constexpr int SLOTS = 256 * W / 1024;
    constexpr int LDS_WORDS = step_lds_words<W, Q32, DP>();

    // a launch of histogram-only slabs takes k1 workgroups a slab: wg is the workgroup within its slab
    const uint32_t sl = blockIdx.x / a.k1, wg = blockIdx.x - sl * a.k1;
    struct {
        const uint8_t *bins;
        int32_t *partial;
        uint32_t *fmt;
        const uint32_t *col_bins;
        const uint32_t *pos_word;
    } R = {a.bins + sl * a.bins_stride, a.partial + static_cast<size_t>(sl) * a.k1 * 2 * step_partial_stride(W),
           a.fmt + sl * a.k1, a.col_bins + sl * (W * PACK), a.pos_word + sl * 256u * (DP ? DP : 1)};
    StepPlan &P = *a.plan;  // empty once the tree is done (k_step_select)
    if (wg >= P.total_groups) return;
    const uint32_t j = job_of(P.group_base, P.njobs, wg);
    JobPlan &J = P.jobs[j];
    StepView v;
    v.job = &J;
    v.hist = J.hist != 0;
    v.partition = a.partition != 0;
    if (!v.hist && !v.partition) return;
    v.status = a.status + J.tile_base;
    v.begin = J.begin;
    v.count = J.count;
    v.ntiles = J.ntiles;
    v.groups = J.groups;
    const uint32_t gi = wg - J.group_base;  // the workgroup within its job
    const bool packed = J.packed != 0;  // then one tile per workgroup
    v.src = J.src_buf ? a.buf1 : a.buf0;
    v.dst = J.src_buf ? a.buf0 : a.buf1;
    v.rev = J.src_rev != 0;
    v.col16 = a.col16;
    v.wide = J.wide;
    v.col = a.colbase + static_cast<size_t>(J.col) * a.rows * (a.col16 ? 2u : 1u);
    v.built_left = J.built_side == 0 ? 1u : 0u;
    v.epoch = P.epoch;
    v.csrc = J.src_buf ? a.codes1 : a.codes0;
    v.cdst = J.src_buf ? a.codes0 : a.codes1;
    const uint32_t tid = threadIdx.x;
    if (tid < 8) sh.left_bins[tid] = J.left_bins[tid];  // visible after the first barrier below
    const uint32_t *bins32 = reinterpret_cast<const uint32_t *>(R.bins);
    if (v.hist)
        for (uint32_t k = tid; k < static_cast<uint32_t>(LDS_WORDS); k += 1024) lds[k] = 0;
    uint32_t dxs[4], dcols[DP ? DP : 1][4];
    if constexpr (DP > 0) dense_lanes<DP>(R.pos_word, tid & 63u, dxs, dcols);

    if (!v.partition) {
        // A later slab: the built child's rows as the partition launch (an earlier kernel) left them in dst, the left
        // child first-first from begin, the right one after the left rows (any order sums alike), a workgroup
        // taking an equal share; no tile is ranked again. Whenever flush_rows rows have gone into the packed words
        // they are added into the partial as {g, h} pairs; a workgroup that never flushes stores them packed.
        const uint32_t nb = v.built_left ? J.left : v.count - J.left;
        const uint32_t b0 = v.begin + (v.built_left ? 0u : J.left);
        const uint32_t per = (nb + v.groups - 1) / v.groups;
        const uint32_t c0 = min(nb, gi * per), c1 = min(nb, c0 + per);
        const uint32_t *list = v.dst + b0;
        const uint8_t *codes = CODES ? v.cdst + b0 : nullptr;
        int4 *pairs = reinterpret_cast<int4 *>(R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
        const uint32_t col_bins = (PACK > 1 || DP > 0) ? 256u : quad_bins<W>(R.col_bins);
        __syncthreads();  // the LDS histogram is zeroed
        bool flushed = false;
        for (uint32_t ca = c0; ca < c1;) {
            const uint32_t cb = c1 - ca < a.flush_rows ? c1 : ca + a.flush_rows;
            if (ca > c0) {
                flush_pairs<W, Q32>(lds, pairs, col_bins, flushed);
                flushed = true;
            }
            step_hist<W, WIDE, PACK, Q32, DP, UNROLL, 16, CODES>(lds, list, ca, cb, a.gh, bins32, a.dw_row, dxs, dcols,
                                                                threadIdx.x >> 6, codes);
            ca = cb;
        }
        if (!flushed && !Q32) {
            __syncthreads();
            store_packed_partial<W>(lds, R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
            if (tid == 0) R.fmt[wg] = 1u;
            return;
        }
        flush_pairs<W, Q32>(lds, pairs, col_bins, flushed);
        if (tid == 0) {
            R.fmt[wg] = 0u;
            P.pairs[j] = 1u;
        }
        return;
    }

    if (packed) {  // one tile; the partial is the LDS words themselves
        __syncthreads();
        if (tid == 0) sh.tile = v.partition ? atomicAdd(&J.ticket, 1u) : gi;
        __syncthreads();
        const uint32_t t = sh.tile;
        TileRows r;
        tile_rows<CODES>(v, t, r);
        tile_bins(v, r);
        TileState st;
        const uint32_t nb = tile_front<CODES>(v, t, r, st, sh);
        // wave 0 resolves the tile's offset while the other waves histogram it (wv: the wave, uniform)
        const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        if (v.partition) {
            if (wv == 0) tile_lookback(v, a, t, st, sh);
            else if (v.hist) step_hist<W, WIDE, PACK, Q32, DP, 16, 15, CODES>(lds, sh.list, 0, nb, a.gh, bins32, a.dw_row, dxs, dcols, wv - 1, sh.codes);
        } else if (v.hist) {
            step_hist<W, WIDE, PACK, Q32, DP, 16, 16, CODES>(lds, sh.list, 0, nb, a.gh, bins32, a.dw_row, dxs, dcols, threadIdx.x >> 6, sh.codes);
        }
        __syncthreads();  // the offset and the histogram are complete
        if (v.partition) tile_scatter<CODES>(v, t, st, sh);
        if (!v.hist) return;
        if constexpr (Q32) {  // the counters as a {g, h} pair partial
            int4 *pairs = reinterpret_cast<int4 *>(R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
            flush_pairs<W, true>(lds, pairs, 256u, false);
            if (tid == 0) {
            R.fmt[wg] = 0u;
            P.pairs[j] = 1u;
        }
            return;
        }
        store_packed_partial<W>(lds, R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
        if (tid == 0) R.fmt[wg] = 1u;
        return;
    }

    // several tiles per workgroup: whenever flush_rows rows have gone into the packed words they are added into the
    // partial as {g, h} pairs; a workgroup that never flushes stores its partial packed instead
    int4 *pairs = reinterpret_cast<int4 *>(R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
    // slot tid + 1024 j is bin (tid + 1024 j) / W of column tid % W; a packed column's features are all stored
    const uint32_t col_bins = (PACK > 1 || DP > 0) ? 256u : quad_bins<W>(R.col_bins);
    uint32_t pending = 0;  // rows added to the packed LDS words since they were last flushed
    bool flushed = false;
    // partition launches take tiles in ticket order, the next ticket drawn while the current tile is worked on (a
    // look-back only ever waits on lower tiles, so holding a later one cannot block it); histogram-only launches
    // take tiles gi, gi + groups, ...
    // A workgroup holds the tickets of its current and next tiles, and loads the next tile's rows while it
    // histograms the current one (their split bins after it).
    // At most a.tile_cap tickets a workgroup, whatever the others' pace (its i32 sums; the planner gives every job
    // enough workgroups for its tiles at that many each).
    __syncthreads();  // the LDS histogram is zeroed
    uint32_t taken = 0;  // tickets this workgroup drew (thread 0's count)
    if (tid == 0) {
        sh.tile = v.partition ? atomicAdd(&J.ticket, 1u) : gi;
        sh.tile2 = v.partition ? (a.tile_cap > 1u ? atomicAdd(&J.ticket, 1u) : v.ntiles) : gi + v.groups;
        taken = a.tile_cap > 1u ? 2u : 1u;
    }
    __syncthreads();
    uint32_t t = sh.tile, tn = sh.tile2;
    uint32_t next = gi + 2 * v.groups;
    TileRows r;
    if (t < v.ntiles) {
        tile_rows<CODES>(v, t, r);
        tile_bins(v, r);
    }
    while (t < v.ntiles) {
        TileState st;
        const uint32_t nb = tile_front<CODES>(v, t, r, st, sh);
        uint32_t ticket = next;
        if (v.partition && tid == 0) {
            ticket = taken < a.tile_cap ? atomicAdd(&J.ticket, 1u) : v.ntiles;
            ++taken;
        }
        next += v.groups;
        if (tn < v.ntiles) tile_rows<CODES>(v, tn, r);
        // a tile that takes the packed words past flush_rows rows is histogrammed by all waves around the flushes
        // (block-wide); otherwise wave 0 resolves the tile's offset while the other waves histogram it
        const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        bool hist_done = !v.hist;
        if (v.hist && pending + nb > a.flush_rows) {
            uint32_t c0 = 0;
            while (c0 < nb) {
                if (pending >= a.flush_rows) {
                    flush_pairs<W, Q32>(lds, pairs, col_bins, flushed);
                    pending = 0;
                    flushed = true;
                }
                uint32_t room = a.flush_rows - pending;
                uint32_t c1 = nb - c0 < room ? nb : c0 + room;
                step_hist<W, WIDE, PACK, Q32, DP, UNROLL, 16, CODES>(lds, sh.list, c0, c1, a.gh, bins32, a.dw_row, dxs, dcols, threadIdx.x >> 6, sh.codes);
                pending += c1 - c0;
                c0 = c1;
            }
            hist_done = true;
        }
        if (v.partition) {
            if (wv == 0) tile_lookback(v, a, t, st, sh);
            else if (!hist_done) step_hist<W, WIDE, PACK, Q32, DP, UNROLL, 15, CODES>(lds, sh.list, 0, nb, a.gh, bins32, a.dw_row, dxs, dcols, wv - 1, sh.codes);
            __syncthreads();  // the offset is in sh.prefix
            tile_scatter<CODES>(v, t, st, sh);
        } else if (!hist_done) {
            step_hist<W, WIDE, PACK, Q32, DP, UNROLL, 16, CODES>(lds, sh.list, 0, nb, a.gh, bins32, a.dw_row, dxs, dcols, threadIdx.x >> 6, sh.codes);
        }
        if (!hist_done) pending += nb;
        if (tn < v.ntiles) tile_bins(v, r);
        __syncthreads();  // the tile's list is consumed
        if (tid == 0) sh.tile = ticket;
        __syncthreads();
        t = tn;
        tn = sh.tile;
    }
    if (!v.hist) return;
    if (!flushed && !Q32) {  // every row still in the packed words: the partial is packed, as a one-tile workgroup's
        __syncthreads();
        store_packed_partial<W>(lds, R.partial + 2 * static_cast<size_t>(wg) * step_partial_stride(W));
        if (tid == 0) R.fmt[wg] = 1u;
        return;
    }
    flush_pairs<W, Q32>(lds, pairs, col_bins, flushed);
    if (tid == 0) {
            R.fmt[wg] = 0u;
            P.pairs[j] = 1u;
        }
}

// CODES: the built rows' gradients come from the codes beside their ids (a.codes0 / a.codes1), else gathered. The
// two are separate instances: in one kernel behind a branch, the register allocator spilled both.
template <int W, bool WIDE = false, int PACK = 1, bool Q32 = false, int DP = 0, bool CODES = false>
__global__ __launch_bounds__(1024) void k_step_rows(StepArgs a) {
    __shared__ int32_t lds[step_lds_words<W, Q32, DP>()];
    __shared__ StepShared sh;
    step_rows_body<W, WIDE, PACK, Q32, DP, CODES>(a, lds, sh);
}

// Measurement only (profile mode): the distinct 128-byte lines (the size of every L2 miss's request to memory) a
// split step's gathers must touch, from the step's own plan and partition buffers, right after its k_step_rows
// launches. Per job, over the parent's rows (ascending in row id, whatever order they are stored in): the lines of
// the column-major split-feature array their bins lie in (128 rows a line, 64 for two-byte bins) and, over the built
// child's rows (sorted too), the lines of the packed gradient array (32 rows a line). A sorted run of rows touches as
// many lines as it has distinct row / rows-per-line values, so each is a count of the positions where that value
// changes. `shared`, when set, is one bit per (column-major feature, split-bin line), or-ed over every job of the
// step: the lines the step would touch if jobs that split on the same feature shared them. counters: [0] parent
// rows, [1] their split-bin lines, [2] built rows, [3] their gradient lines, [5] partials written (the first slab's
// workgroups of histogrammed jobs), [6] of those, packed (`fmt`: the first slab's partial formats), [7]-[9] parent
// rows, split-bin lines and built rows of the sparse jobs (fewer than two parent rows a split-bin line). grid: (x,
// JMAX); one block per job when `sparse_split` is needed (x = 1).
__global__ __launch_bounds__(256) void k_sector_model(const StepPlan *plan, const uint32_t *buf0, const uint32_t *buf1,
                                                      uint32_t col16, uint32_t *shared, uint64_t lines_per_col,
                                                      const uint32_t *fmt, unsigned long long *counters) {
    __shared__ unsigned long long part[4];
    const StepPlan &P = *plan;
    const uint32_t j = blockIdx.y;
    if (threadIdx.x < 4) part[threadIdx.x] = 0;
    if (j < P.njobs && blockIdx.x == 0 && threadIdx.x == 0 && P.jobs[j].hist) {
        const JobPlan &J = P.jobs[j];
        unsigned long long packed = 0;
        for (uint32_t k = 0; k < J.groups; ++k) packed += fmt[J.group_base + k] ? 1ull : 0ull;
        atomicAdd(counters + 5, static_cast<unsigned long long>(J.groups));
        atomicAdd(counters + 6, packed);
    }
    __syncthreads();
    if (j < P.njobs) {
        const JobPlan &J = P.jobs[j];
        const uint32_t *src = J.src_buf ? buf1 : buf0, *dst = J.src_buf ? buf0 : buf1;
        const uint32_t sshift = col16 ? 6u : 7u;
        unsigned long long prow = 0, psec = 0, brow = 0, bsec = 0;
        for (uint32_t i = threadIdx.x; i < J.count; i += blockDim.x) {
            const uint32_t at = J.src_rev ? J.begin + J.count - 1 - i : J.begin + i;
            const uint32_t r = src[at];
            ++prow;
            if (i == 0 || (src[J.src_rev ? at + 1 : at - 1] >> sshift) != (r >> sshift)) ++psec;
            if (shared) {
                const uint64_t bit = static_cast<uint64_t>(J.col) * lines_per_col + (r >> sshift);
                atomicOr(shared + (bit >> 5), 1u << (bit & 31u));
            }
        }
        if (J.hist) {
            // the built child: the left one first-first at begin, the right one last-first after the left rows
            const uint32_t b = J.built_side == 0 ? J.begin : J.begin + J.left;
            const uint32_t n = J.built_side == 0 ? J.left : J.count - J.left;
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
                const uint32_t r = dst[b + i];
                ++brow;
                if (i == 0 || (dst[b + i - 1] >> 5) != (r >> 5)) ++bsec;
            }
        }
        atomicAdd(&part[0], prow);
        atomicAdd(&part[1], psec);
        atomicAdd(&part[2], brow);
        atomicAdd(&part[3], bsec);
    }
    __syncthreads();
    if (threadIdx.x < 4 && part[threadIdx.x]) atomicAdd(counters + threadIdx.x, part[threadIdx.x]);
    if (threadIdx.x == 0 && part[1] * 2 > part[0]) {  // a sparse job (one block a job)
        atomicAdd(counters + 7, part[0]);
        atomicAdd(counters + 8, part[1]);
        atomicAdd(counters + 9, part[2]);
    }
}

// Measurement only: the set bits of k_sector_model's shared-line bitmap into counters[4], the bitmap cleared.
__global__ __launch_bounds__(256) void k_sector_bits(uint32_t *bits, uint64_t words, unsigned long long *counters) {
    unsigned long long c = 0;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < words;
         i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const uint32_t w = bits[i];
        if (w) {
            c += static_cast<unsigned long long>(__popc(w));
            bits[i] = 0;
        }
    }
    for (int o = 32; o > 0; o >>= 1) c += static_cast<unsigned long long>(__shfl_xor(static_cast<long long>(c), o));
    if ((threadIdx.x & 63u) == 0 && c) atomicAdd(counters + 4, c);
}

// Four columns of one slab: a work unit of k_step_children (byte slabs) or k_step_reduce (two-byte slabs).
struct ColGroup {
    uint64_t partial;  // the slab's partials, in {g, h} pairs from the start of the step partial buffer
    uint32_t width;    // the slab's W
    uint32_t c0;       // first column of the group in the slab
    uint32_t fmt;      // the slab's first k_step_rows workgroup in the partial-format flags
    uint32_t offset[4][4];  // per segment and column: its feature's first bin in the flat histogram
    uint32_t bins[4][4];    // per segment and column: the feature's bins (0 for padding)
    uint32_t seg_shift;     // a column holds a feature each 2^seg_shift bins (8: one; 7 or 6 in a packed slab)
    uint32_t dense;         // a dense slab: the slots' flat bins come from the slot table at slot_base
    uint32_t slot_base;
    uint32_t pairs;         // the slab's partials are always {g, h} pairs (separate 32-bit counters)
    uint32_t unit_first, unit_count;  // the columns' scan units (k_step_children); CG_COLS a group unless segmented
};

// Block-wide hand-off through `counter`: true in every thread of the block that arrives last of `target` blocks,
// which then sees the global stores every arriving block made before arriving; that block returns the counter
// to 0. Each thread first waits for its own stores to reach L2, so thread 0's release fence (an L2 write-back,
// waited for before the increment) covers the whole block, and its acquire fence covers the last block's reads.
__device__ __forceinline__ bool arrive_last(uint32_t *counter, uint32_t target) {
    __shared__ uint32_t s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __builtin_amdgcn_s_waitcnt(0);
        bool last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == target - 1u;
        if (last) {
            __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        s_last = last ? 1u : 0u;
    }
    __syncthreads();
    return s_last != 0;
}

// One feature of a scan unit (k_step_children): a unit is one wave's scan of a child's histogram, of one feature (64
// lanes), or of 4 features of at most 64 bins (16 lanes each) or 16 of at most 16 bins (4 lanes each), a segment of lanes
// each (UNIT_FEATS records a unit). `at`: the feature's bin 0 in a child's LDS planes, 256 * (column in its group) + the
// column's row.
struct UnitRec {
    int32_t feat;  // -1: padding
    uint32_t at;
    FeatDev m;
};

struct ChildArgs {
    const int32_t *partial;     // the step partial buffer
    const uint32_t *fmt;        // the partials' formats (per slab, per k_step_rows workgroup: 1 packed, 0 pairs)
    const ColGroup *cgs;        // [ncgb]
    const uint32_t *slot_flat;  // dense slabs: per slot, its flat-histogram bin + 1 (0: none)
    const UnitRec *recs;        // [units][UNIT_FEATS]; when no unit holds several features, [ncgb][CG_COLS]
    const uint32_t *unit_segl;  // per unit, its lanes a feature: 64, 16 or 4
    StepPlan *plan;
    int64_t *scratch;           // the shares' sums: [scratch row][column group][4][512]
    uint32_t *counters;         // [scratch row][column group] arrivals, returned to 0
};

struct ScanStepArgs {
    const int32_t *wide_feats;  // the two-byte features
    StepPlan *plan;
};

struct SelectArgs {
    StepPlan *plan;             // this step's plan
    StepPlan *next;             // the next step's
};

struct ReduceStepArgs {
    const int32_t *partial;     // the step partial buffer
    const uint32_t *fmt;        // the partials' formats (per slab, per k_step_rows workgroup: 1 packed, 0 pairs)
    const ColGroup *cgs;        // [ncgw], the two-byte slabs'
    StepPlan *plan;
};

// The children's histograms and candidates of each job over its byte slabs, one work item per (job, column group): the
// built child's histogram of the group's four columns from the job's partials and its sibling's by subtraction in place
// of the parent's (learner.rs:356-371), both kept in LDS, then every feature of the group scanned in both children
// (split.rs:584-620, 694-844) from there, a wave a scan unit and child, and the group's best candidate of each child
// written. Reducing and scanning in one launch saves the second one's start (a launch, the plan, then each scan's
// dependent loads of a histogram another XCD just wrote): k_step_reduce 6.5 us + k_step_scan 13.7 us a step on 100k x 28
// are 11.7 us here; 22.7 + 37.5 us in the 32-job steps of 10M x 128 are 38 us.
// Threads: bin tid % 256, stripe tid / 256 of the partials (two stripes that meet in LDS, each then finishing two of the
// four columns), 8 partials' loads in flight a thread. One item a block, its job found by the item's index (ChildJob):
// with a loop over items every load of the plan came after some store, so all went through vector registers, and the
// kernel spilled. SEG: some units hold several features; CAT: some a categorical one (apart for the registers of the plain
// scan: two blocks a compute unit need at most 128). grid: the most items a step can have, 512 threads.
// The sums of one bin of four columns over N partials w, w + step, ... below `groups`, their loads in flight together.
// add_packed: packed partials. add_pairs: {g, h} pairs (PAIRS: the slab has no others), or, format by format, a mix.
template <uint32_t N>
__device__ __forceinline__ void add_packed(const int4 *src, size_t stride4, uint32_t w, uint32_t step, uint32_t groups, int64_t (&sg)[4],
                                           int64_t (&sh)[4]) {
    int4 x[N];
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        const uint32_t wk = w + step * k;
        x[k] = src[static_cast<size_t>(wk < groups ? wk : w) * stride4];
    }
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        if (w + step * k >= groups) continue;
        const int32_t v4[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int32_t gq = packed_g(v4[c]);
            sg[c] += gq;
            sh[c] += packed_h(v4[c], gq);
        }
    }
}
template <uint32_t N, bool PAIRS>
__device__ __forceinline__ void add_pairs(const int4 *src, size_t stride4, size_t plane, const uint32_t *fmt, uint32_t w,
                                          uint32_t step, uint32_t groups, int64_t (&sg)[4], int64_t (&sh)[4]) {
    int4 a0[N], a1[N];
    bool pk[N];
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        const uint32_t wk = w + step * k;
        pk[k] = !PAIRS && fmt[wk < groups ? wk : w] != 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        const uint32_t wk = w + step * k;
        const int4 *p = src + static_cast<size_t>(wk < groups ? wk : w) * stride4;
        a0[k] = p[0];
        a1[k] = p[pk[k] ? 0 : plane];
    }
#pragma unroll
    for (uint32_t k = 0; k < N; ++k) {
        if (w + step * k >= groups) continue;
        if (pk[k]) {
            const int32_t v4[4] = {a0[k].x, a0[k].y, a0[k].z, a0[k].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int32_t gq = packed_g(v4[c]);
                sg[c] += gq;
                sh[c] += packed_h(v4[c], gq);
            }
        } else {
            sg[0] += a0[k].x;
            sg[1] += a0[k].y;
            sg[2] += a0[k].z;
            sg[3] += a0[k].w;
            sh[0] += a1[k].x;
            sh[1] += a1[k].y;
            sh[2] += a1[k].z;
            sh[3] += a1[k].w;
        }
    }
}

template <bool SEG, bool CAT>
__global__ __launch_bounds__(512, 4) void k_step_children(GrowState g, ChildArgs a) {
    __shared__ double plane_g[2][4 * 256], plane_h[2][4 * 256];  // [built, sibling][column * 256 + bin]
    __shared__ int64_t red[4][512];                              // the two columns a stripe hands to the other
    __shared__ FeatCand s_cand[8];                               // each wave's best candidate
    __shared__ double s_gain[8];
    __shared__ int32_t s_feat[8];
    __shared__ __align__(16) uint8_t s_cats[CAT ? 8 * sizeof(CatScratch) : 16];
    const StepPlan &P = *a.plan;  // empty once the tree is done (k_step_select)
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // one item a block: nothing is stored before the plan is read, so its loads are scalar ones
    const uint32_t item = blockIdx.x, total = P.total_child;
    const uint32_t k = item / g.ncgb, r = item - k * g.ncgb;  // the share and its item
    uint32_t cgi = r;
    if ((g.ncgb & 15u) == 0u) {
        // column groups 2p and 2p + 1 (one 128-byte line of a packed partial) 8 items apart, so on one XCD (blocks
        // go to the 8 XCDs in turn): the second reads the line from that XCD's L2
        const uint32_t w = r & 15u;
        cgi = 2u * ((r >> 4) * 8u + (w & 7u)) + (w >> 3);
    }
    const ChildJob &J = P.child[k < CHILD_MAX ? k : 0u];
    const ColGroup &cg = a.cgs[cgi];  // read in place: a column is picked per thread
    // wave w scans units w / 2, w / 2 + 4, ... of child w % 2: its first unit's record comes with the job
    const uint32_t child = wave & 1u, units = SEG ? cg.unit_count : CG_COLS;
    const uint32_t first = SEG ? cg.unit_first : CG_COLS * cgi;
    uint32_t segl = 64u;
    UnitRec rec;
    auto load_rec = [&](uint32_t u) {
        if constexpr (SEG) {
            segl = a.unit_segl[first + u];  // wave-uniform
            rec = a.recs[static_cast<size_t>(first + u) * UNIT_FEATS + lane / segl];
        } else {
            rec = a.recs[first + u];
        }
    };
    if (item >= total) return;
    if (wave >> 1 < units) load_rec(wave >> 1);
    else rec = UnitRec{-1, 0u, FeatDev{}};
    const uint32_t left = P.jobs[J.j].left, mixed = P.pairs[J.j];
    const uint8_t *prow = g.splittable + static_cast<size_t>(J.t) * g.nf;
    bool sev = rec.feat >= 0 && g.mask[rec.feat] != 0 && prow[rec.feat] != 0;
    int64_t *built = g.pool + static_cast<size_t>(J.built_slot) * g.slot_stride;
    int64_t *parent = g.pool + static_cast<size_t>(J.parent_slot) * g.slot_stride;
    {
        const size_t stride4 = step_partial_stride(cg.width) / 2;  // int4s from one partial to the next
        const uint32_t q = wave >> 2, bin = tid & 255u;            // this thread's stripe (wave-uniform) and bin
        // bin `bin` of the group's columns in a partial: int4 (bin / 4) * W + c0 + bin % 4, of packed words or, in a
        // partial of pairs, of its g plane, the h plane's 64 W int4s on
        const int4 *src = reinterpret_cast<const int4 *>(a.partial + 2 * cg.partial) + static_cast<size_t>(J.group_base) * stride4 +
                          static_cast<size_t>(bin / 4u) * cg.width + cg.c0 + bin % 4u;
        const size_t plane = 64u * static_cast<size_t>(cg.width);
        const uint32_t *fmt = a.fmt + cg.fmt + J.group_base;
        // this thread finishes columns 2q and 2q + 1: their slots' flat bins + 1 (0: none) and the parent's units,
        // loaded with the partials
        const uint32_t seg = bin >> cg.seg_shift, vb = bin & ((1u << cg.seg_shift) - 1u);
        uint32_t fl[2];
        if (cg.dense) {
            const uint2 t = *reinterpret_cast<const uint2 *>(a.slot_flat + cg.slot_base + static_cast<size_t>(bin) * cg.width + cg.c0 + 2u * q);
            fl[0] = t.x;
            fl[1] = t.y;
        } else {
#pragma unroll
            for (uint32_t c = 0; c < 2; ++c)
                fl[c] = vb < cg.bins[seg][2u * q + c] ? cg.offset[seg][2u * q + c] + vb + 1u : 0u;
        }
        longlong2 par[2];
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c)
            par[c] = *reinterpret_cast<const longlong2 *>(parent + 2 * static_cast<size_t>(fl[c] ? fl[c] - 1u : 0u));
        int64_t sg[4] = {0, 0, 0, 0}, sh[4] = {0, 0, 0, 0};
        if (cg.pairs) {
            for (uint32_t w = q; w < J.groups; w += 16u) add_pairs<8, true>(src, stride4, plane, fmt, w, 2u, J.groups, sg, sh);
        } else if (mixed) {
            for (uint32_t w = q; w < J.groups; w += 16u) add_pairs<8, false>(src, stride4, plane, fmt, w, 2u, J.groups, sg, sh);
        } else {
            uint32_t w = q;
            for (; w + 2u < J.groups; w += 16u) add_packed<8>(src, stride4, w, 2u, J.groups, sg, sh);
            if (w < J.groups) add_packed<1>(src, stride4, w, 2u, J.groups, sg, sh);
        }
        int64_t mg[2], mh[2];
        const uint32_t to = q * 256u + bin, from = (1u - q) * 256u + bin;
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) {
            red[2 * c][to] = q == 0u ? sg[2 + c] : sg[c];
            red[2 * c + 1][to] = q == 0u ? sh[2 + c] : sh[c];
            mg[c] = q == 0u ? sg[c] : sg[2 + c];
            mh[c] = q == 0u ? sh[c] : sh[2 + c];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) {
            mg[c] += red[2 * c][from];
            mh[c] += red[2 * c + 1][from];
        }
        if (J.ways > 1u) {  // the last of the job's shares to arrive adds them all up and goes on (exact integers)
            int64_t *mine = a.scratch + ((static_cast<size_t>(J.scratch) + J.way) * g.ncgb + cgi) * 2048 + tid;
#pragma unroll
            for (uint32_t c = 0; c < 2; ++c) {
                mine[(2 * c) * 512] = mg[c];
                mine[(2 * c + 1) * 512] = mh[c];
            }
            if (!arrive_last(a.counters + static_cast<size_t>(J.scratch) * g.ncgb + cgi, J.ways)) return;
            const int64_t *all = a.scratch + (static_cast<size_t>(J.scratch) * g.ncgb + cgi) * 2048 + tid;
            for (uint32_t w = 0; w < J.ways; ++w) {
                if (w == J.way) continue;
                const int64_t *o = all + static_cast<size_t>(w) * g.ncgb * 2048;
#pragma unroll
                for (uint32_t c = 0; c < 2; ++c) {
                    mg[c] += o[(2 * c) * 512];
                    mh[c] += o[(2 * c + 1) * 512];
                }
            }
        }
#pragma unroll
        for (uint32_t c = 0; c < 2; ++c) {
            const uint32_t at = (2u * q + c) * 256u + bin;
            const int64_t og = par[c].x - mg[c], oh = par[c].y - mh[c];
            plane_g[0][at] = static_cast<double>(mg[c]);
            plane_h[0][at] = static_cast<double>(mh[c]);
            plane_g[1][at] = static_cast<double>(og);
            plane_h[1][at] = static_cast<double>(oh);
            if (fl[c]) {
                const size_t o = 2 * static_cast<size_t>(fl[c] - 1u);
                *reinterpret_cast<longlong2 *>(built + o) = make_longlong2(mg[c], mh[c]);
                *reinterpret_cast<longlong2 *>(parent + o) = make_longlong2(og, oh);
            }
        }
    }
    const uint32_t which = child == J.built_side ? 0u : 1u;
    const int64_t cnt = child == 0 ? static_cast<int64_t>(left) : J.parent_count - static_cast<int64_t>(left);
    const Ctx c = make_ctx(g.cfg, grow_sg(g), grow_sh(g), child ? J.child_ug[1] : J.child_ug[0],
                           child ? J.child_uh[1] : J.child_uh[0], cnt);
    uint8_t *row = g.splittable + static_cast<size_t>(J.kid + static_cast<int32_t>(child)) * g.nf;
    __syncthreads();
    double best = 0.0;
    int bf = -1;
    for (uint32_t u = wave >> 1; u < units; u += 4u) {
        if (u >= 4u) {
            load_rec(u);
            sev = rec.feat >= 0 && g.mask[rec.feat] != 0 && prow[rec.feat] != 0;
        }
        const LdsUnits h{&plane_g[which][rec.at], &plane_h[which][rec.at]};
        FeatCand cand = {};
        bool rf = false, ff = false;
        Grown rg = {}, fg = {};
        const bool on = scan_searched(c, rec.m, sev);
        if (CAT && segl == 64u && rec.m.kind == 2) {
            if (on) cand = categorical_candidate(c, g.cfg, rec.m, h, reinterpret_cast<CatScratch *>(s_cats)[wave], nullptr);
        } else {
            if (segl == 64u) {
                if (on) scan_numerical<64>(c, g.cfg, rec.m, h, rf, rg, ff, fg);
            } else if (SEG) {
                if (segl == 16u) scan_numerical<16>(c, g.cfg, rec.m, h, rf, rg, ff, fg);
                else scan_numerical<4>(c, g.cfg, rec.m, h, rf, rg, ff, fg);
            }
            if (on) cand = feature_candidate(c, rec.m, rf, rg, ff, fg);
        }
        const bool lead = rec.feat >= 0 && (lane & (segl - 1u)) == 0u;
        if (lead) row[rec.feat] = static_cast<uint8_t>(cand.splittable);
        // the unit's best by (gain, lower feature), against the wave's so far
        double wg = lead && cand.found ? (cand.gain != cand.gain ? -__builtin_inf() : cand.gain) : 0.0;
        int wf = lead && cand.found ? rec.feat : -1;
        const int mine = wf;
        if (SEG && segl != 64u) {
            wave_best(wg, wf);
        } else {
            wg = readlane_f64(wg, 0);
            wf = __builtin_amdgcn_readlane(wf, 0);
        }
        if (cand_better(wg, wf, best, bf)) {
            best = wg;
            bf = wf;
            if (mine == wf) s_cand[wave] = cand;
        }
    }
    if (lane == 0) {
        s_gain[wave] = best;
        s_feat[wave] = bf;
    }
    __syncthreads();
    if (wave < 2) {  // child `wave`'s best over its four waves
        double wg = lane < 4 ? s_gain[wave + 2 * lane] : 0.0;
        int wf = lane < 4 ? s_feat[wave + 2 * lane] : -1;
        const int mine = wf;
        wave_best(wg, wf);
        const size_t slot = (static_cast<size_t>(J.j) * 2 + wave) * g.nslot + cgi;
        if (lane == 0) {
            g.cand_gain[slot] = wg;
            g.cand_feat[slot] = wf;
        }
        static_assert(sizeof(FeatCand) % 4 == 0 && sizeof(FeatCand) / 4 <= 64, "a candidate copies in one wave");
        if (wf >= 0) {
            const uint32_t owner = wave + 2u * static_cast<uint32_t>(__builtin_ctzll(__ballot(mine == wf)));
            if (lane < sizeof(FeatCand) / 4)
                reinterpret_cast<uint32_t *>(&g.cands[slot])[lane] = reinterpret_cast<const uint32_t *>(&s_cand[owner])[lane];
        }
    }
}

// The two-byte slabs' histograms of each job: the built child's from its workgroups' partials, and its sibling's by
// subtraction in place of the parent's (learner.rs:356-371). Work items (job, column group, bin range) in a grid-stride
// loop: a thread adds one stripe of the workgroups' partials of one bin of the group's four columns, reading each partial
// in its own format (packed: one 16-byte load; {g, h} pairs: two), and the stripes meet in LDS. (A two-byte feature's
// bins lie in four column groups, so its scan is a launch of its own.) An item takes neighbouring bins of four features
// across their four column groups, so that a wave reads and writes whole lines of the histograms: by column group a lane's
// bins were 64 bytes from the next one's and each line was written by four items (6M x 32 at 2047 leaves 56 -> 38 us a
// step). grid: any, 256 threads.
__global__ __launch_bounds__(256) void k_step_reduce(GrowState g, ReduceStepArgs a) {
    __shared__ int64_t red[8][256];  // the stripes' sums, [value][thread]: conflict-free
    const StepPlan &P = *a.plan;  // empty once the tree is done (k_step_select)
    const uint32_t tid = threadIdx.x;
    for (uint32_t item = blockIdx.x; item < P.total_red; item += gridDim.x) {
        const uint32_t j = job_of(P.red_base, P.njobs, item);
        const JobPlan &J = P.jobs[j];
        const uint32_t ways = J.ways, groups = J.groups;
        const uint32_t r = item - J.red_base;
        uint32_t cgi, sub;
        if ((g.ncgw & 15u) == 0u) {
            // column groups 2p and 2p + 1 (one 128-byte line of a packed partial) 8 items apart, so on one XCD (blocks
            // go to the 8 XCDs in turn): the second reads the line from that XCD's L2
            const uint32_t w = r & 15u, pi = (r >> 4) * 8u + (w & 7u), pair = pi / ways;
            sub = pi - pair * ways;
            cgi = 2u * pair + (w >> 3);
        } else {
            cgi = r / ways;
            sub = r - cgi * ways;
        }
        const ColGroup &cg = a.cgs[cgi];
        int64_t *built = g.pool + static_cast<size_t>(J.built_slot) * g.slot_stride;
        int64_t *parent = g.pool + static_cast<size_t>(J.parent_slot) * g.slot_stride;
        const size_t stride4 = step_partial_stride(cg.width) / 2;  // int4s from one partial to the next
        const uint32_t ns = 256u / ways;                           // the item's bins
        const uint32_t q = tid / ns;                               // this thread's stripe
        // the slab's column group l stands for four features (quad) and a quarter of their 1024 bins; bin b lies in the
        // column group of its phase b % 4, as bin b / 4 of the group's columns
        const uint32_t l = cg.c0 / CG_COLS, nq = cg.width / (4u * CG_COLS), quad = l % nq;
        const uint32_t b = (l / nq * ways + sub) * ns + tid % ns, bin = b / 4u, lb = (b % 4u) * nq + quad;
        const ColGroup &cb = a.cgs[cgi - l + lb];
        // bin `bin` of the group's columns in a partial: int4 (bin / 4) * W + c0 + bin % 4, of packed words or, in a
        // partial of pairs, of its g plane, the h plane's 64 W int4s on
        const int4 *src = reinterpret_cast<const int4 *>(a.partial + 2 * cg.partial) + static_cast<size_t>(J.group_base) * stride4 +
                          static_cast<size_t>(bin / 4u) * cg.width + CG_COLS * lb + bin % 4u;
        const size_t plane = 64u * static_cast<size_t>(cg.width);
        const uint32_t *fmt = a.fmt + cg.fmt + J.group_base;
        // the parent's bins are loaded with the partials (the writes below need them); fl: the flat bin + 1 of each of the
        // four features' bin b (0: none)
        uint32_t fl[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) fl[c] = bin < cb.bins[0][c] ? cb.offset[0][c] + bin * 4u + 1u : 0u;
        longlong2 par[4];
        if (q == 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) par[c] = *reinterpret_cast<const longlong2 *>(parent + 2 * static_cast<size_t>(fl[c] ? fl[c] - 1u : 0u));
        }
        int64_t sg[4] = {0, 0, 0, 0}, sh[4] = {0, 0, 0, 0};
        for (uint32_t w = q; w < groups; w += 8u * ways) {
            if (cg.pairs) add_pairs<8, true>(src, stride4, plane, fmt, w, ways, groups, sg, sh);
            else if (P.pairs[j]) add_pairs<8, false>(src, stride4, plane, fmt, w, ways, groups, sg, sh);
            else add_packed<8>(src, stride4, w, ways, groups, sg, sh);
        }
        if (ways > 1u) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                red[2 * c][tid] = sg[c];
                red[2 * c + 1][tid] = sh[c];
            }
            __syncthreads();
            if (q == 0)
                for (uint32_t k = 1; k < ways; ++k) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        sg[c] += red[2 * c][tid + k * ns];
                        sh[c] += red[2 * c + 1][tid + k * ns];
                    }
                }
        }
        if (q == 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (fl[c]) {
                    const size_t o = 2 * static_cast<size_t>(fl[c] - 1u);
                    *reinterpret_cast<longlong2 *>(built + o) = make_longlong2(sg[c], sh[c]);
                    *reinterpret_cast<longlong2 *>(parent + o) = make_longlong2(par[c].x - sg[c], par[c].y - sh[c]);
                }
            }
        }
        __syncthreads();  // the LDS is free for the next item
    }
}

// Scan items (job, two-byte feature, child), a wave each in a grid-stride loop: the feature scanned in both directions
// (split.rs:584-620) over the child's histogram (the built one, or the sibling k_step_reduce formed in the parent's slot)
// and its candidate written to its own slot. A wave a block: the planes of four would leave one block a compute unit.
// grid: any, 64 threads.
__global__ __launch_bounds__(64) void k_step_scan(GrowState g, ScanStepArgs a) {
    __shared__ UnitPlanes<true> planes;
    const StepPlan &P = *a.plan;  // empty once the tree is done (k_step_select)
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t total = P.total_scan * 2u;  // scan items count features: a wave per feature and child
    for (uint32_t item = blockIdx.x; item < total; item += gridDim.x) {
        const uint32_t gi = item >> 1, child = item & 1u;
        const uint32_t j = job_of(P.scan_base, P.njobs, gi);
        const JobPlan &J = P.jobs[j];
        const uint32_t u = gi - J.scan_base;
        const int32_t sf = a.wide_feats[u];
        const FeatDev sm = g.feats[sf];
        const bool sev = g.mask[sf] != 0 && g.splittable[static_cast<size_t>(J.t) * g.nf + sf] != 0;
        const int64_t *hist = g.pool + static_cast<size_t>(child == J.built_side ? J.built_slot : J.parent_slot) * g.slot_stride;
        const int64_t cnt = child == 0 ? static_cast<int64_t>(J.left) : J.parent_count - static_cast<int64_t>(J.left);
        const Ctx c = make_ctx(g.cfg, grow_sg(g), grow_sh(g), J.child_ug[child], J.child_uh[child], cnt);
        FeatCand r = {};
        if (scan_searched(c, sm, sev)) {
            Grown rg = {}, fg = {};
            bool rf, ff;
            scan_numerical_wide(c, g.cfg, sm, stage_units<true>(hist, sm, planes), rf, rg, ff, fg);
            r = feature_candidate(c, sm, rf, rg, ff, fg);
        }
        if (lane == 0) {
            const size_t slot = (static_cast<size_t>(j) * 2 + child) * g.nslot + g.ncgb + u;
            g.cands[slot] = r;
            g.cand_gain[slot] = r.gain != r.gain ? -__builtin_inf() : r.gain;
            g.cand_feat[slot] = r.found ? sf : -1;
            g.splittable[static_cast<size_t>(J.kid + static_cast<int32_t>(child)) * g.nf + sf] = static_cast<uint8_t>(r.splittable);
        }
    }
}

// The end of a step, by one block: each job's children take their best splits (learner.rs:294-352, split.rs:866-880) and
// become leaves of the speculative tree, then advance replays and plans the next step. What bounds it is the chain of
// dependent loads of what other XCDs just wrote (about 1 us each), not its work: so one block does all jobs (a block a job
// met through a counter, whose fences alone took several microseconds), loads everything whose address does not depend on
// another load at once, keeps the new leaves' keys in LDS for the replay, and a plan carries what its children need of
// their parent. 20.6 -> 15.4 us a step on 100k x 28, 37.4 -> 34.6 us on 10M x 128. One block, of 1024 threads for trees of
// more than 512 leaves (up to 128 children a step: 76.5 us at 2047 leaves against 82.6 with 512 threads). MAXL: the
// largest tree it takes.
template <uint32_t MAXL> constexpr uint32_t select_threads() { return MAXL > LEAVES_SMALL ? 1024u : 512u; }
template <uint32_t MAXL>
__global__ __launch_bounds__(select_threads<MAXL>()) void k_step_select(GrowState g, SelectArgs a) {
    constexpr uint32_t NW = select_threads<MAXL>() / 64, BATCH = 4;
    __shared__ __align__(16) uint8_t scratch[sizeof(AdvShared<MAXL>)];
    __shared__ int32_t s_feat[2 * JMAX];   // per (job, child), its best feature (-1: none) and that candidate's slot
    __shared__ uint32_t s_slot[2 * JMAX];
    __shared__ uint32_t s_bad;
    AdvShared<MAXL> &s = *reinterpret_cast<AdvShared<MAXL> *>(scratch);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const StepPlan &P = *a.plan;
    const AdvState st = adv_state(g.ctl);
    const uint32_t done = g.ctl->done, njobs = P.njobs, pairs = 2u * njobs;
    const uint32_t pj = tid < 2u * JMAX ? tid >> 1 : 0u, ch = tid & 1u;
    const JobPlan &J = P.jobs[pj];  // thread p < pairs: child p % 2 of job p / 2
    if (done || njobs == 0) {
        // the next plan stays empty: the steps after a finished tree do nothing without reading the control block
        if (tid == 0) {
            a.next->njobs = 0;
            a.next->total_groups = 0;
            a.next->total_child = 0;
            a.next->total_red = 0;
            a.next->total_scan = 0;
        }
        return;
    }
    if (tid == 0) s_bad = 0;
    // the keys of the leaves before this step's children; the children's are made below
    advance_load(g, s, st.n0, st.ntent - pairs);
    // each child's best candidate over its slots by (gain, lower feature), a wave BATCH children at a time
    for (uint32_t p0 = wave; p0 < pairs; p0 += NW * BATCH) {
        double gv[BATCH];
        int fv[BATCH];
#pragma unroll
        for (uint32_t i = 0; i < BATCH; ++i) {
            const uint32_t p = p0 + NW * i < pairs ? p0 + NW * i : p0;
            const size_t at = static_cast<size_t>(p) * g.nslot + (lane < g.nslot ? lane : 0u);
            gv[i] = g.cand_gain[at];
            fv[i] = g.cand_feat[at];
        }
#pragma unroll
        for (uint32_t i = 0; i < BATCH; ++i) {
            const uint32_t p = p0 + NW * i;
            if (p >= pairs) continue;  // uniform
            double best = gv[i];
            int bf = lane < g.nslot ? fv[i] : -1;
            uint32_t bs = lane;
            for (uint32_t x = lane + 64u; x < g.nslot; x += 64u) {
                const double gx = g.cand_gain[static_cast<size_t>(p) * g.nslot + x];
                const int fx = g.cand_feat[static_cast<size_t>(p) * g.nslot + x];
                if (cand_better(gx, fx, best, bf)) {
                    best = gx;
                    bf = fx;
                    bs = x;
                }
            }
            int wf = bf;
            wave_best(best, wf);
            const unsigned long long at = __ballot(bf == wf);  // a feature is in one slot
            if (wf >= 0 && lane == static_cast<uint32_t>(__builtin_ctzll(at))) s_slot[p] = bs;
            if (lane == 0) s_feat[p] = wf;
        }
    }
    if (g.count_work)  // the jobs' evaluated features (learner.rs:262-265), for the byte counts
        for (uint32_t j = wave; j < njobs; j += NW) {
            const JobPlan &Q = P.jobs[j];
            const uint8_t *prow = g.splittable + static_cast<size_t>(Q.t) * g.nf;
            uint32_t used = 0;
            for (uint32_t f0 = 0; f0 < g.nf; f0 += 64u)
                used += static_cast<uint32_t>(__popcll(__ballot(f0 + lane < g.nf && g.mask[f0 + lane] != 0 && prow[f0 + lane] != 0)));
            if (lane == 0) {
                if (Q.hist) {  // the built child's histogram was made, searched or not
                    const double built = static_cast<double>(Q.built_side == 0 ? Q.left : Q.count - Q.left);
                    atomicAdd(&g.ctl->hist_rows, built);
                    atomicAdd(&g.ctl->hist_bins, built * static_cast<double>(used));
                    atomicAdd(&g.ctl->hist_builds, 1.0);
                }
                atomicAdd(&g.ctl->part_rows, static_cast<double>(Q.count));
            }
        }
    __syncthreads();
    if (tid < pairs) {
        const int64_t left = static_cast<int64_t>(J.left), right = J.parent_count - left;
        if (!(left > 0 && right > 0)) {
            if (ch == 0 && atomicExch(&s_bad, 1u) == 0u) {
                const uint32_t info[8] = {pj, J.t, J.count, J.left, J.ntiles, J.groups, J.packed, 0u};
                for (int k = 0; k < 8; ++k) g.ctl->err_info[k] = info[k];
            }
        } else {
            const int64_t min_pair = 2 * g.cfg.min_data_in_leaf, cnt = ch == 0 ? left : right;
            const bool searched = J.hist && depth_allows(g, J.depth) && (left >= min_pair || right >= min_pair);
            const double ug = ch == 0 ? J.child_ug[0] : J.child_ug[1], uh = ch == 0 ? J.child_uh[0] : J.child_uh[1];
            const uint32_t kid = static_cast<uint32_t>(J.kid) + ch;
            TLeaf c;
            c.best = SplitOut{};
            const int bf = searched ? s_feat[tid] : -1;
            if (bf >= 0)
                c.best = split_out(g.cands[static_cast<size_t>(tid) * g.nslot + s_slot[tid]], bf,
                                   make_ctx(g.cfg, grow_sg(g), grow_sh(g), ug, uh, cnt), g.cfg);
            const uint32_t has = c.best.found ? 1u : 0u;
            c.begin = ch == 0 ? J.begin : J.begin + J.left;
            c.count = ch == 0 ? J.left : J.count - J.left;
            c.ug = ug;
            c.uh = uh;
            c.cnt = cnt;
            // the built child's histogram goes to the job's new slot, the other child keeps its parent's
            c.slot = searched ? ((J.built_side == ch) ? J.built_slot : J.parent_slot) : -1;
            c.has_best = has;
            c.buf = 1u - J.src_buf;
            c.rev = ch;  // the split step writes the left child first-first and the right child last-first
            c.depth = J.depth;
            c.state = T_LEAF;
            c.kid = -1;
            c.pad_ = 0;
            const double v = ch == 0 ? J.child_out[0] : J.child_out[1];
            c.value = v != v ? 0.0 : v;
            c.weight = uh * grow_sh(g);
            const TKey key{c.best.gain, has, T_LEAF, -1, 0u};
            g.tl[kid] = c;
            g.tk[kid] = key;
            s.gain[kid] = key.gain;
            s.meta[kid] = key_meta(key);
            if (ch == 0) {  // the job's leaf, which has a split and is expanded now
                g.tl[J.t].state = T_EXPANDED;
                g.tk[J.t].state = T_EXPANDED;
                s.meta[J.t] = key_meta(TKey{0.0, 1u, T_EXPANDED, J.kid, 0u});
            }
        }
    }
    __syncthreads();
    if (tid == 0) {  // empty unless advance writes it
        a.next->njobs = 0;
        a.next->total_groups = 0;
        a.next->total_child = 0;
        a.next->total_red = 0;
        a.next->total_scan = 0;
        if (s_bad) {
            g.ctl->error = 1;
            g.ctl->done = 1;
        }
    }
    if (s_bad) return;  // uniform
    advance<MAXL>(g, *a.next, s, st);
}

}  // namespace srocm
