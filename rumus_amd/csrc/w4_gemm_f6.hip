// INT4 engine: dequant-fused GEMM on the six-bit-float matrix cores, for large batches.
//
//   y[m,n] = sum_g scale[g,n] * ( sum_{k in g} x[m,k] (q[k,n] - z[g,n])  -  rest[g,n] * sum_{k in g} x[m,k] )
//
// with z the zero-point's nearest integer (within 0..15) and rest = zp - z.  v_mfma_scale_f32_32x32x64_f8f6f4 runs
// operands of six bits (e2m3: sign, 0 .. 7.5, integers up to 16 in units of 1/8 .. 1/2) at four times the f16 rate:
//   - q - z is -15 .. 15: exact as (q - z) / 2;
//   - x becomes six six-bit digits.  Per row and 32 consecutive k, x 2^-e (largest magnitude below 7.5) is rounded to
//     the nearest e2m3, the exact remainder, at most 1/4, is rounded again in units of 2^-4, the remainder of that, at
//     most 2^-7, in units of 2^-9, then 2^-14, 2^-19 and 2^-24: what is left is below 2^-27, i.e. 29 bits below the largest of
//     the 32 values.  The exponent e is the MFMA's own block scale (one E8M0 byte per row and 32 k), and the
//     digits' constant offsets ride on the block scale of the weight operand, so all six products add up in one f32
//     accumulator.
// Why six: the f16 tiles (w4_gemm_tile.hip) keep 22 bits of every element, and so does this down to 2^-7 of the largest of the
// 32.  Five digits, 24 bits below the largest, took 12 % less time and were further off than those: the split's own error against
// float64, as a share of the result, with some channels 20 times as large 5.5e-8 (f16 tiles 4.3e-8, six digits 1.0e-9), with
// SwiGLU outputs 5.4e-8 (4.4e-8, 0.9e-9), with every eighth channel 2^4 as large and met by weights of zero 3.4e-7 (4.4e-8, 0.7e-8).
// Whole calls, 2048 x 4096 -> 11008 on such inputs, sums included: 3.4e-7 (f16 tiles 4.7e-7 to 5.8e-7).
// The weights' codes (3/4 of a byte each) are made once per call, in the launch that prepares the activations, where the workspace has room;
// otherwise every block of 128 rows converts them for itself, five vector instructions per MFMA instead of two.  One box in turn, by
// every block -> once (us): 2048 x 4096 -> 11008 act-order 324 -> 305, 4096 x 4096 -> 12288 655 -> 625, -> 22016 1226 -> 1157, 4096 x 11008 -> 4096
// 690 -> 661, 512 x 4096 -> 11008 111 -> 107.  The matmul itself 300 -> 265: its matrix cores are busy 65 % of a workgroup's cycles (55 before),
// vector issue 33 % (52), at 1.87 GHz (1.93); six-bit MFMAs alone on random operands run at 1.41 GHz, the power limit.
// Six products at four times the rate are 3/4 of the matrix work of the two f16 products of the hi/lo split.  One box in turn, f16
// tiles -> this (us): 2048 x 4096 -> 11008 344 -> 298 with integer zero-points, 370 -> 325 with fractional ones, groups of 64
// 383 -> 332; 4096 x 4096 -> 22016 1312 -> 1086, 4096 x 11008 -> 4096 707 -> 610, 4096 x 4096 -> 4096 267 -> 219.
//
// Elements that tower over some of their 32 neighbours would still cost those their low bits: where an octet of the 32 lies 2^8
// or more below the largest, or kF6Small of the 32 (not counting zeros) 2^9 or more, the run is marked, and a second pass over such
// steps, after the main loop, multiplies two more digits (2^-29, 2^-34: 39 bits below the largest).  N(0,1) marks no run in
// 10^7, SwiGLU outputs of gates N(0,4) fewer than one in 10^4, of gates N(0,16) one in 200; a call in which every step has marks takes
// 2.4 times as long.  The split's error with every second, eighth or 32nd channel 2^p as large and met by weights of zero, p = 2 to 16: at
// most 1.6e-7 of the result.
// Why q - z in halves: codes below 1 have no leading bit, and the instruction seems to align its sum as if they had one.  With
// q - z in eighths, most of them such codes, a sum of few small products lost low bits of the accumulator: 1.5e-6 of the result
// where the small elements of those inputs come to half a unit of a digit (p = 6, 10 and 16), in halves 4.7e-7, f16 tiles 4.5e-7 to
// 4.8e-7 throughout.  It costs 1.5 % of a call (2048 x 4096 -> 11008 307 -> 312 us); quarters 6.2e-7 and nothing.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "w4.h"

namespace rumus {

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v32h __attribute__((ext_vector_type(32)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef uint32_t v6u __attribute__((ext_vector_type(6)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v3fa4 __attribute__((ext_vector_type(3), aligned(4)));

typedef const void __attribute__((address_space(1)))* gptr_t;
typedef void __attribute__((address_space(3)))* lptr_t;

constexpr int kF6BM = 128;                      // rows per workgroup
constexpr int kF6Tiles = kF6BM / 32;            // row tiles of 32 per workgroup
constexpr int kF6Digits = 6;
constexpr int kF6Tile = kF6Digits * 1536;       // bytes of one row tile and one step of 64 k: 64 lanes x 24 bytes per digit
constexpr int kF6Step = kF6Tiles * kF6Tile;     // 36 KB
constexpr int kF6Lo = kF6Digits * 1024;         // inside a tile: the lanes' first 16 bytes of every digit, then their last 8
constexpr int kF6BTile = 1024 + 512 + 32;       // the same for 32 columns of weights; 32 bytes of skew against bank conflicts
constexpr uint32_t kF6Band = 4;                 // row blocks that a die works on at a time
constexpr uint32_t kF6MaxK = 16384;             // padded to whole groups: a thread of the preparation per 32 k of a row, a row in LDS
constexpr uint32_t kF6Flags = 256;              // parts of the zero-point table, one flag word each
constexpr int kF6Deep = 2;                      // further digits where a run of 32 k spans many binades
constexpr uint32_t kF6Small = 12;               // elements 2^9 or more below the largest of a run that mark it
constexpr uint32_t kF6DeepBit = 0x80;           // of an exponent byte: the run needs them (the exponents themselves stay below 128)
// digit d counts in units of 2^-shift
constexpr int kF6Shift[kF6Digits + kF6Deep] = {0, 4, 9, 14, 19, 24, 29, 34};

struct F6Args {
    const uint32_t* packed;
    const float* scales;
    const float* zp;
    const uint32_t* zp4;
    const float* bias;
    const uint8_t* planes;     // [row block][step][kF6Step]
    const uint8_t* codes;      // PRE: the weights' six-bit codes, [block of 128 TN columns][step][4 TN tiles][1536]
    const uint16_t* exps;      // [row block][pair of steps][row tile][64 lanes]: two E8M0 bytes
    const float* sums;         // [row block][step][kF6BM rows]: sum of x over the step's 64 k
    const float* x;            // for the further digits of marked runs, with what the preparation does to its rows
    const int32_t* perm;
    const float* norm_w;
    bool glu;
    const float* rinv;         // [row], RMSNorm: 1 / rms
    const float* rfac;         // [row]: back to the row's own scale (NaN: the row holds a NaN or an infinity)
    const float* least;        // [column]: the smallest unit of its accumulators (NaN: a scale is)
    const uint32_t* zflags;    // kF6Flags words, nonzero where a part of the zero-point table holds a value that is no integer in 0..15
    float* y;
    uint32_t m, k, n, steps, steps_per_group, num_groups;
    const float* residual;     // [m][n], added to the result, or null; may be y
    uint32_t row_blocks, col_blocks;
};

__device__ __forceinline__ v8i f6_operand(const v6u& a) {
    return v8i{(int)a[0], (int)a[1], (int)a[2], (int)a[3], (int)a[4], (int)a[5], 0, 0};
}

// Fragment order of the weights (nibble conversion): field 8 w + {0..7} of a lane holds k offsets 8 w + {0,4,1,5,2,6,3,7}:
// even fields come from one register vector, odd ones from the other.
__device__ __forceinline__ void f6_order(const float (&v)[32], v16f& ev, v16f& od) {
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            ev[4 * w + j] = v[8 * w + j];
            od[4 * w + j] = v[8 * w + 4 + j];
        }
}
// the next digit of 32 values, in units of `unit`, and what it leaves (exact)
__device__ __forceinline__ v6u f6_digit(v16f& ev, v16f& od, float unit) {
    const v6u code = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ev, od, unit);
    const v32f back = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(code, unit);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        ev[i] -= back[2 * i];
        od[i] -= back[2 * i + 1];
    }
    return code;
}

// ---- weights -> six-bit codes, once per call ---------------------------------------------------------------------
// one packed word -> eight f16, k order 0,4,1,5,2,6,3,7, the integer z taken off on the way (1024 + n - (1024 + z), and
// (1024 + 16 n) / 16 - (64 + z)): exact
__device__ __forceinline__ v8h f6_nibbles(uint32_t w, v2h big, v2h small) {
    const v2h k16th = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u, magic = 0x64006400u;
    const uint32_t w8 = w >> 8;
    uint32_t t0, t1, t2, t3;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t0) : "v"(w), "v"(m_lo), "s"(magic));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t1) : "v"(w), "v"(m_hi), "s"(magic));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t2) : "v"(w8), "v"(m_lo), "s"(magic));
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(t3) : "v"(w8), "v"(m_hi), "s"(magic));
    const v2h h0 = __builtin_bit_cast(v2h, t0) - big;
    const v2h h1 = __builtin_elementwise_fma(__builtin_bit_cast(v2h, t1), k16th, small);
    const v2h h2 = __builtin_bit_cast(v2h, t2) - big;
    const v2h h3 = __builtin_elementwise_fma(__builtin_bit_cast(v2h, t3), k16th, small);
    return v8h{h0[0], h0[1], h1[0], h1[1], h2[0], h2[1], h3[0], h3[1]};
}

// TN adjacent columns' floats (TN = 2, 3 or 4; 8-byte aligned)
template <int TN> struct F6Floats { float v[TN]; };
template <int TN>
__device__ __forceinline__ void f6_cols_store(float* p, const F6Floats<TN>& o) {
    if constexpr (TN == 4) *reinterpret_cast<float4*>(p) = make_float4(o.v[0], o.v[1], o.v[2], o.v[3]);
    else if constexpr (TN == 3) *reinterpret_cast<v3fa4*>(p) = v3fa4{o.v[0], o.v[1], o.v[2]};
    else *reinterpret_cast<float2*>(p) = make_float2(o.v[0], o.v[1]);
}
// An array as a buffer resource: addresses are an offset that is the same for the whole wave (scalar) plus one per lane,
// and reads beyond its end give zeros.  (gfx9 descriptor: no swizzle, raw 32-bit data.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t f6_array(const void* p, uint64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)min(bytes, (uint64_t)0xffffffffu), 0x00027000);
}
template <int TN>
__device__ __forceinline__ F6Floats<TN> f6_cols_at(__amdgpu_buffer_rsrc_t p, uint32_t lane_bytes, uint32_t uniform) {
    F6Floats<TN> o;
    if constexpr (TN == 4) {
        const v4u f = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(p, (int)lane_bytes, (int)uniform, 0));
#pragma unroll
        for (int j = 0; j < 4; j++) o.v[j] = __uint_as_float(f[j]);
    } else if constexpr (TN == 3) {
        const auto f = __builtin_amdgcn_raw_buffer_load_b96(p, (int)lane_bytes, (int)uniform, 0);
#pragma unroll
        for (int j = 0; j < 3; j++) o.v[j] = __uint_as_float(f[j]);
    } else {
        const v2u f = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(p, (int)lane_bytes, (int)uniform, 0));
        o.v[0] = __uint_as_float(f[0]);
        o.v[1] = __uint_as_float(f[1]);
    }
    return o;
}
// The codes of a step in the order in which the matmul copies them into LDS: [block of 128 TN columns][step][4 TN tiles of 32
// columns][1536].  A wave takes 32 TN columns (a lane TN adjacent ones of one half of a step, 4 TN bytes of a word row per
// load) and two steps; eight waves a block of columns and four steps.  Memory bound: 4096 x 11008 reads 25 and writes 34 MB.
struct F6Weights {
    const uint32_t* packed;
    const float* zp;
    const uint32_t* zp4;
    uint8_t* codes;                // or null: the matmul converts the weights itself
    uint32_t n, steps, steps_per_group, num_groups, tn;
};
constexpr uint32_t kF6CodeSteps = 4;
template <int TN, bool ZP4>
__device__ __forceinline__ void f6_codes(const F6Weights& a, uint32_t part) {
    constexpr int U = 2;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), set = wave & 3, half = lane >> 5;
    const uint32_t chunks = (a.steps + kF6CodeSteps - 1) / kF6CodeSteps, block = part / chunks;
    const uint32_t col = (block * 4 + set) * (32 * TN) + TN * (lane & 31), s0 = part % chunks * kF6CodeSteps + (wave >> 2) * U;
    const uint32_t row_bytes = a.n * 4;                           // (columns past n: codes of anything, never stored)
    const auto b_packed = f6_array(a.packed, (uint64_t)a.steps * 8 * row_bytes);
    const auto b_zp = ZP4 ? f6_array(a.zp4, (uint64_t)a.num_groups * (a.n / 2)) : f6_array(a.zp, (uint64_t)a.num_groups * row_bytes);
    F6Floats<TN> raw[U][4], z[U];
    uint32_t z4[U][2];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t s = min(s0 + u, a.steps - 1), g = s / a.steps_per_group;
#pragma unroll
        for (int i = 0; i < 4; i++) raw[u][i] = f6_cols_at<TN>(b_packed, half * 4 * row_bytes + col * 4, (8 * s + i) * row_bytes);
        if constexpr (ZP4) {                                     // (three columns from col = 6 mod 8 on lie in two words)
            z4[u][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_zp, (int)(col / 8 * 4), (int)(g * (a.n / 2)), 0);
            z4[u][1] = TN == 3 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_zp, (int)((col + 2) / 8 * 4), (int)(g * (a.n / 2)), 0) : z4[u][0];
        } else {
            z[u] = f6_cols_at<TN>(b_zp, col * 4, g * row_bytes);
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        if (s0 + u >= a.steps) return;
        uint8_t* const to = a.codes + (((uint64_t)block * a.steps + s0 + u) * 4 + set) * (TN * 1536);
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const float zj = ZP4 ? (float)((((col & 7u) + j > 7u ? z4[u][1] : z4[u][0]) >> (4 * ((col + j) & 7u))) & 15u)
                                 : fminf(fmaxf(rintf(z[u].v[j]), 0.0f), 15.0f);   // (a NaN becomes 0 and stays whole in the rest)
            const _Float16 b = (_Float16)(1024.0f + zj), sm = (_Float16)(-64.0f - zj);
            v32h halves;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const v8h f = f6_nibbles(__float_as_uint(raw[u][i].v[j]), v2h{b, b}, v2h{sm, sm});
#pragma unroll
                for (int e = 0; e < 8; e++) halves[8 * i + e] = f[e];
            }
            const v6u code = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(halves, 2.0f);
            *reinterpret_cast<uint4*>(to + j * 1536 + lane * 16) = make_uint4(code[0], code[1], code[2], code[3]);
            *reinterpret_cast<uint2*>(to + j * 1536 + 1024 + lane * 8) = make_uint2(code[4], code[5]);
        }
    }
}
__device__ __forceinline__ void f6_codes_of(const F6Weights& a, uint32_t part) {
    if (a.zp4) {
        if (a.tn == 2) f6_codes<2, true>(a, part);
        else if (a.tn == 3) f6_codes<3, true>(a, part);
        else f6_codes<4, true>(a, part);
    } else if (a.tn == 2) f6_codes<2, false>(a, part);
    else if (a.tn == 3) f6_codes<3, false>(a, part);
    else f6_codes<4, false>(a, part);
}

// ---- activations -> digits ---------------------------------------------------------------------------
// A workgroup takes `rows` rows (a power of two up to 8): copies them into LDS with contiguous reads, finding each row's
// largest magnitude on the way, and then every thread turns one unit, 32 consecutive k of one row, into six digits
// (rows * units <= 512 threads).  The gather of act-order weights happens on the way out of LDS: from global memory a wave
// instruction would touch 64 cache lines for 256 bytes.  Memory bound: 2048 x 4096 reads 33.5 and writes 38 MB.
// LDS: row r at r * pitch floats, 4 floats of padding after every 32, so that the 16-byte reads of threads 32 floats
// apart fall on different banks (likewise rows: pitch / 4 is odd).
// Beyond the row groups, more workgroups look at the columns' scales, 64 columns each, kF6Flags at f32 zero-points, and the last
// ones convert the weights.
__device__ __forceinline__ uint32_t f6_padded(uint32_t j) { return j + (j >> 5) * 4; }

// What the rows of x go through on their way into LDS (a decoder block's operators in front of a projection; k % 4 == 0 and
// 16-byte aligned then): RMSNorm with `norm_w`, or SwiGLU of rows gate | up of 2 k floats.  Their results are written
// nowhere: for marked runs the matmul computes them once more, in the same operations.
// 4096 rows: SwiGLU of 2 x 11008 125 + 113 us as two kernels, 163 as one; RMSNorm of 4096 25 + 27 us, 35 as one.
enum F6In { kF6Plain, kF6Perm, kF6Norm, kF6Glu };
__device__ __forceinline__ float f6_norm(float v, float inv, float w) { return v * inv * w; }
__device__ __forceinline__ float f6_glu(float a, float b) { return a / (1.0f + expf(-a)) * b; }

template <F6In IN>
__global__ __launch_bounds__(512) void w4_f6_prepare_kernel(const float* __restrict__ x, const int32_t* __restrict__ perm,
                                                            uint8_t* __restrict__ planes, uint8_t* __restrict__ exps,
                                                            float* __restrict__ sums, float* __restrict__ rfac,
                                                            uint32_t m, uint32_t k, uint32_t steps, uint32_t rows,
                                                            uint32_t pitch, const float4* __restrict__ zp, uint32_t zp_count4,
                                                            uint32_t* __restrict__ zflags, const float* __restrict__ scales,
                                                            uint32_t num_groups, uint32_t n, float* __restrict__ least,
                                                            uint32_t row_groups,
                                                            const float* __restrict__ norm_w, float eps,
                                                            float* __restrict__ rinv, F6Weights weights) {
    constexpr bool PERM = IN == kF6Perm;
    extern __shared__ __attribute__((aligned(16))) float lds_x[];
    __shared__ uint32_t rowmax[8];
    __shared__ float squares[8];
    constexpr uint32_t T = 512;
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x >= row_groups) {
        uint32_t part = blockIdx.x - row_groups;
        if (part < (n + 63) / 64) {                            // eight waves share the groups
            const uint32_t col = part * 64 + (tid & 63), at = min(col, n - 1);
            uint32_t top = 0;                                    // bit patterns without their sign: a NaN sorts highest
            for (uint32_t g = tid >> 6; g < num_groups; g += 64) {
                uint32_t v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = __float_as_uint(scales[(uint64_t)min(g + 8 * u, num_groups - 1) * n + at]);
#pragma unroll
                for (int u = 0; u < 8; u++) top = max(top, v[u] & 0x7fffffffu);
            }
            uint32_t* const tops = reinterpret_cast<uint32_t*>(lds_x);   // [8][64]
            tops[tid] = top;
            __syncthreads();
            if (tid < 64 && col < n) {
#pragma unroll
                for (int w = 1; w < 8; w++) top = max(top, tops[64 * w + tid]);
                const float t = __uint_as_float(top);
                least[col] = t != t ? t : fmaxf(t * 0x1p-60f, 0x1p-126f);
            }
            return;
        }
        part -= (n + 63) / 64;
        const uint32_t flags = weights.zp4 ? 0 : kF6Flags;
        if (part >= flags) return f6_codes_of(weights, part - flags);
        bool mine = false;
        for (uint32_t i = part * T + tid; i < zp_count4; i += kF6Flags * T) {
            const float4 z = zp[i];
            const float v[4] = {z.x, z.y, z.z, z.w};
#pragma unroll
            for (int j = 0; j < 4; j++) mine = mine || !(v[j] == rintf(v[j]) && v[j] >= 0.0f && v[j] <= 15.0f);   // a NaN counts
        }
        const int any = __syncthreads_or(mine);
        if (tid == 0) zflags[part] = any ? 1u : 0u;
        return;
    }
    const uint32_t row0 = xcd_contiguous(blockIdx.x, row_groups) * rows;   // neighbours fill the same cache lines of the planes
    const uint32_t live = row0 < m ? min(rows, m - row0) : 0;
    if (tid < 8) rowmax[tid] = 0;
    const uint32_t units = 2 * steps, r = tid % rows, unit = tid / rows, row = row0 + r;
    const bool mine = unit < units;
    int4 from[PERM ? 8 : 1];                                     // act-order: where the unit's values come from
    if constexpr (PERM) {                                                // (k is a multiple of the group size then, and so of 64)
#pragma unroll
        for (int q = 0; q < 8; q++) from[q] = reinterpret_cast<const int4*>(perm)[mine ? 8 * unit + q : q];
    }
    __syncthreads();
    // rows into LDS, largest magnitudes on the bit patterns (a NaN or an infinity sorts highest)
    const bool vec = k % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    const uint32_t per_row = T / rows, r1 = tid / per_row, t1 = tid % per_row;   // (a wave's threads share a row)
    {
        uint32_t am = 0;
        auto look = [&](const float4& v) __attribute__((always_inline)) {
            am = max(max(am, __float_as_uint(v.x) & 0x7fffffffu), __float_as_uint(v.y) & 0x7fffffffu);
            am = max(max(am, __float_as_uint(v.z) & 0x7fffffffu), __float_as_uint(v.w) & 0x7fffffffu);
        };
        const float* const src = x + (uint64_t)(row0 + r1) * k * (IN == kF6Glu ? 2 : 1);
        float* const dst = lds_x + r1 * pitch;
        const uint32_t last = k / 4 - 1;
        if constexpr (IN == kF6Glu) {
            if (r1 < live) {
                for (uint32_t i0 = t1; i0 <= last; i0 += 8 * per_row) {
                    float4 g[8], v[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        g[u] = reinterpret_cast<const float4*>(src)[min(i0 + u * per_row, last)];
                        v[u] = reinterpret_cast<const float4*>(src + k)[min(i0 + u * per_row, last)];
                    }
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const float4 y = make_float4(f6_glu(g[u].x, v[u].x), f6_glu(g[u].y, v[u].y), f6_glu(g[u].z, v[u].z), f6_glu(g[u].w, v[u].w));
                        *reinterpret_cast<float4*>(dst + f6_padded(4 * min(i0 + u * per_row, last))) = y;
                        look(y);
                    }
                }
            }
        } else if constexpr (IN == kF6Norm) {
            float ss = 0.0f;
            if (r1 < live) {
                for (uint32_t i0 = t1; i0 <= last; i0 += 8 * per_row) {
                    float4 v[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) v[u] = reinterpret_cast<const float4*>(src)[min(i0 + u * per_row, last)];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        if (i0 + u * per_row > last) continue;
                        *reinterpret_cast<float4*>(dst + f6_padded(4 * (i0 + u * per_row))) = v[u];
                        ss = fmaf(v[u].x, v[u].x, fmaf(v[u].y, v[u].y, fmaf(v[u].z, v[u].z, fmaf(v[u].w, v[u].w, ss))));
                    }
                }
            }
            ss = wave_sum(ss);
            if ((tid & 63) == 0) squares[tid >> 6] = ss;
            __syncthreads();
            const uint32_t waves = per_row / 64;                     // of a row, neighbours
            float total = 0.0f;
            for (uint32_t w = 0; w < waves; w++) total += squares[r1 * waves + w];
            const float inv = 1.0f / sqrtf(total / (float)k + eps);
            if (r1 < live) {
                if (t1 == 0) rinv[row0 + r1] = inv;
                for (uint32_t i = t1; i <= last; i += per_row) {     // every thread's own elements
                    const float4 w = reinterpret_cast<const float4*>(norm_w)[i];
                    float4* const at = reinterpret_cast<float4*>(dst + f6_padded(4 * i));
                    const float4 v = *at, y = make_float4(f6_norm(v.x, inv, w.x), f6_norm(v.y, inv, w.y), f6_norm(v.z, inv, w.z), f6_norm(v.w, inv, w.w));
                    *at = y;
                    look(y);
                }
            }
        } else if (r1 < live) {
            if (vec) {
                for (uint32_t i0 = t1; i0 <= last; i0 += 8 * per_row) {
                    float4 v[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) v[u] = reinterpret_cast<const float4*>(src)[min(i0 + u * per_row, last)];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        *reinterpret_cast<float4*>(dst + f6_padded(4 * min(i0 + u * per_row, last))) = v[u];
                        look(v[u]);
                    }
                }
            } else {
                for (uint32_t i = t1; i < k; i += per_row) {
                    const float v = src[i];
                    dst[f6_padded(i)] = v;
                    am = max(am, __float_as_uint(v) & 0x7fffffffu);
                }
            }
        }
        am = wave_max(am);
        if ((tid & 63) == 0) atomicMax(&rowmax[r1], am);
    }
    __syncthreads();
    // 2^(113 - E) brings the row's largest magnitude into [2^-14, 2^-13) (rows beyond 2^112: below 4): the accumulators then
    // stay inside f32's range whatever the row's own size; the factor and its reciprocal are normal numbers
    const uint32_t e8 = rowmax[r] >> 23, fb = e8 == 0 || e8 == 255 ? 127u : 240u > e8 ? 240u - e8 : 1u;
    const bool filled = mine && row < m && e8 != 255;
    float v[32];
    {
        const float rv = __uint_as_float(fb << 23);
        const float* lr = lds_x + r * pitch;
        const uint32_t left = filled && k > 32 * unit ? k - 32 * unit : 0;   // columns past k are zeros
        if constexpr (PERM) {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                v[4 * q] = lr[f6_padded((uint32_t)from[q].x)]; v[4 * q + 1] = lr[f6_padded((uint32_t)from[q].y)];
                v[4 * q + 2] = lr[f6_padded((uint32_t)from[q].z)]; v[4 * q + 3] = lr[f6_padded((uint32_t)from[q].w)];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float4 f = *reinterpret_cast<const float4*>(lr + (mine ? unit * 36 : 0) + 4 * q);
                v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
            }
        }
#pragma unroll
        for (int j = 0; j < 32; j++) v[j] = (uint32_t)j < left ? v[j] * rv : 0.0f;
    }
    float o4[4], top = 0.0f, low = 3.4e38f;                      // the octets' largest magnitudes, over all of them: largest and smallest
#pragma unroll
    for (int o = 0; o < 4; o++) {
        o4[o] = fabsf(v[8 * o]);
#pragma unroll
        for (int j = 1; j < 8; j++) o4[o] = fmaxf(o4[o], fabsf(v[8 * o + j]));
        top = fmaxf(top, o4[o]);
        low = o4[o] > 0.0f ? fminf(low, o4[o]) : low;            // (octets of zeros have nothing to lose)
    }
    uint32_t small = 0;
#pragma unroll
    for (int j = 0; j < 32; j++) small += v[j] != 0.0f && fabsf(v[j]) < top * 0x1p-9f ? 1u : 0u;
    const bool is_deep = low < top * 0x1p-8f || small >= kF6Small;
    if (!mine) return;                                           // whole waves or the tail of one: no barrier follows
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; j++) sum += v[j];
    // the other half of the step: threads tid and tid ^ rows (rows divides 64, units is even)
    sum += __shfl_xor(sum, (int)rows);
    // 2^e with top 2^-e in [3.75, 7.5); units far below the row's size keep a floor
    const uint32_t eb = max(__float_as_uint(top * (8.0f / 7.5f)) >> 23, 37u) - 2;
    v16f ev, od;
    f6_order(v, ev, od);
    const uint32_t step = unit >> 1, half = unit & 1, blk = row / kF6BM, rt = row / 32 % kF6Tiles, ln = half * 32 + (row & 31);
    uint8_t* const tile = planes + ((uint64_t)blk * steps + step) * kF6Step + rt * kF6Tile;
#pragma unroll
    for (int d = 0; d < kF6Digits; d++) {
        const v6u code = f6_digit(ev, od, __uint_as_float((eb - kF6Shift[d]) << 23));
        *reinterpret_cast<uint4*>(tile + d * 1024 + ln * 16) = make_uint4(code[0], code[1], code[2], code[3]);
        *reinterpret_cast<uint2*>(tile + kF6Lo + d * 512 + ln * 8) = make_uint2(code[4], code[5]);
    }
    uint8_t* const e_at = exps + ((((uint64_t)blk * ((steps + 1) / 2) + step / 2) * kF6Tiles + rt) * 64 + ln) * 2;
    e_at[step & 1] = (uint8_t)(eb | (is_deep ? kF6DeepBit : 0u));
    if ((steps & 1) && step + 1 == steps) e_at[1] = 0;           // a step that does not exist is not marked either
    if (half == 0) sums[((uint64_t)blk * steps + step) * kF6BM + row % kF6BM] = sum;
    if (unit == 0 && row < m) {
        rfac[row] = e8 == 255 ? __uint_as_float(0x7fc00000u) : __uint_as_float((254u - fb) << 23);
    }
}

// ---- the matmul ----------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t lds_offset(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p; }

// Loads into LDS (16 bytes per lane, to `to` + 16 * lane) and writes to it, spelled out: the compiler would make every
// LDS access wait for all loads into LDS in flight (it cannot see that they go to another buffer).  The waits that it counts
// for its own accesses only get longer for operations it does not know of; the barrier that publishes a buffer waits for
// these explicitly.
__device__ __forceinline__ void lds_load16(uint32_t to, const uint8_t* from, uint32_t lane_bytes) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(lane_bytes), "s"(from));
}
template <int OFF>
__device__ __forceinline__ void lds_write24(uint32_t hi_at, uint32_t lo_at, const v6u& v) {
    const v4u hi = {v[0], v[1], v[2], v[3]};
    const v2u lo = {v[4], v[5]};
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(hi_at), "v"(hi), "n"(OFF));
    asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(lo_at), "v"(lo), "n"(OFF));
}

// s_waitcnt vmcnt(n) lgkmcnt(0)
#define RUMUS_F6_WAIT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x70)

// Eight waves as 2 (rows) x 4 (columns); a wave owns 64 rows (two row tiles) and 32 TN columns, lane l's columns being
// TN adjacent ones per tile set.  The accumulators (32 TN registers) set the tile: with 128 TN columns by 128 rows every
// converted weight serves two row tiles and every activation digit TN column tiles, two steps of both take 129 KB
// of LDS at TN = 4, and one workgroup runs per compute unit; w4_launch_gemm_f6 picks TN.
template <int TN, int FOLD, bool ZP4, bool PRE>
__global__ __launch_bounds__(512, 2) void w4_gemm_f6_kernel(F6Args a) {
    constexpr int BN = 128 * TN, CPT = TN == 2 ? 1 : 2;          // columns per workgroup; columns each thread converts per step
    constexpr int BTILE = PRE ? 1536 : kF6BTile, BBYTES = 4 * TN * BTILE;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // A[2][kF6Step], B[2][BBYTES], 16 bytes per thread
    uint8_t* const lds_b = lds + 2 * kF6Step;

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 2, wn = wave & 3, l32 = lane & 31, kb = lane >> 5;
    // Each die gets a contiguous run of workgroups in the order: kF6Band row blocks by column blocks, column by column.  The 32 that it
    // works on at a time are then 4 row blocks by 8 column blocks (288 KB per step out of 4 MB of L2) instead of 9 by 29 (850 KB):
    // misses 7.4 M -> 3.1 M lines at 2048 x 4096 -> 11008, the call 297 -> 291 us.
    const uint32_t tile = xcd_contiguous(blockIdx.x, gridDim.x), band = tile / (kF6Band * a.col_blocks), in_band = tile % (kF6Band * a.col_blocks);
    const uint32_t band_rows = min(kF6Band, a.row_blocks - band * kF6Band);
    const uint32_t blk = band * kF6Band + in_band % band_rows, cblk = in_band / band_rows, m0 = blk * kF6BM, n0 = cblk * BN;
    // whether some zero-point of the table is no integer in 0..15 (found by w4_f6_prepare_kernel)
    uint4 zflag = make_uint4(0, 0, 0, 0);
    if constexpr (!ZP4) zflag = reinterpret_cast<const uint4*>(a.zflags)[lane];
    const uint32_t my_col = n0 + wn * (32 * TN) + TN * l32;       // first of the lane's TN output columns
    const uint32_t my_col_c = my_col < a.n ? my_col : 0;          // n % 4 == 0

    // ---- weights: thread converts CPT adjacent columns of one half (32 k) of a step --------------------
    // (TN = 3: 192 pairs of columns, the last 64 threads of a half repeat the last pair)
    const uint32_t c_half = wave >> 2, c_first = CPT * min(tid & 255, (uint32_t)(BN / CPT - 1)), c_col = n0 + c_first;
    const uint32_t c_col_c = c_col < a.n ? c_col : 0;
    uint32_t c_hi[CPT], c_lo[CPT];                                 // where the column's codes go
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        const uint32_t w = (c_first + c) / (32 * TN), r = (c_first + c) % (32 * TN);
        const uint32_t tile = lds_offset(lds_b) + (w * TN + r % TN) * BTILE, ln = c_half * 32 + r / TN;
        c_hi[c] = tile + ln * 16;
        c_lo[c] = tile + 1024 + ln * 8;
    }
    const uint32_t row_bytes = a.n * 4;
    const auto b_packed = f6_array(a.packed, (uint64_t)a.steps * 8 * row_bytes), b_scales = f6_array(a.scales, (uint64_t)a.num_groups * row_bytes);
    const auto b_zp = ZP4 ? f6_array(a.zp4, (uint64_t)a.num_groups * (a.n / 2)) : f6_array(a.zp, (uint64_t)a.num_groups * row_bytes);
    const uint32_t c_bytes = c_col_c * 4;
    uint32_t raw[2][4][CPT];                                       // words of an even and an odd step
    auto word_load = [&](uint32_t s, int set, int i) __attribute__((always_inline)) {
        const uint32_t row = min(s, a.steps - 1) * 8 + c_half * 4 + i;
        if constexpr (CPT == 2) {
            const v2u w = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(b_packed, (int)c_bytes, (int)(row * row_bytes), 0));
            raw[set][i][0] = w[0]; raw[set][i][1] = w[1];
        } else {
            raw[set][i][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_packed, (int)c_bytes, (int)(row * row_bytes), 0);
        }
    };
    constexpr int ZSETS = FOLD == 1 ? 2 : 1;                       // zero-points in flight: of every step, or of every even one
    float raw_zp[ZSETS][CPT];
    uint32_t raw_zp4[ZSETS];
    auto zp_load = [&](uint32_t s, int set) __attribute__((always_inline)) {
        const uint32_t g = min(s, a.steps - 1) / a.steps_per_group;
        if constexpr (ZP4) {
            raw_zp4[set] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_zp, (int)(c_col_c / 8 * 4), (int)(g * (a.n / 2)), 0);
        } else if constexpr (CPT == 2) {
            const v2u z = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(b_zp, (int)c_bytes, (int)(g * row_bytes), 0));
            raw_zp[set][0] = __uint_as_float(z[0]); raw_zp[set][1] = __uint_as_float(z[1]);
        } else {
            raw_zp[set][0] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_zp, (int)c_bytes, (int)(g * row_bytes), 0));
        }
    };
    v2h z_big[CPT], z_small[CPT];
    auto zero_points = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            float z;
            if constexpr (ZP4) {
                z = (float)((raw_zp4[set] >> (4 * (c_col_c & 7u) + 4 * c)) & 15u);
            } else {
                z = fminf(fmaxf(rintf(raw_zp[set][c]), 0.0f), 15.0f);    // (a NaN becomes 0 and stays whole in the rest)
            }
            const _Float16 b = (_Float16)(1024.0f + z), sm = (_Float16)(-64.0f - z);
            z_big[c] = v2h{b, b};
            z_small[c] = v2h{sm, sm};
        }
    };
    v32h halves;
    auto convert_words = [&](int set, int c, int first) __attribute__((always_inline)) {   // two of the four words of column c
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const v8h f = f6_nibbles(raw[set][first + i][c], z_big[c], z_small[c]);
#pragma unroll
            for (int e = 0; e < 8; e++) halves[8 * (first + i) + e] = f[e];
        }
    };
    auto column_store = [&](int c, auto buf_tag) __attribute__((always_inline)) {
        constexpr int OFF = decltype(buf_tag)::value * BBYTES;
        const v6u code = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(halves, 2.0f);
        lds_write24<OFF>(c_hi[c], c_lo[c], code);
    };

    // ---- activations: a step is 36 KB, straight into LDS; wave w takes KB w, w + 8, w + 16, w + 24, w + 32 (the last four waves
    // repeat the last: same bytes to the same place, so that every wave counts the same loads) ------------------
    const uint8_t* const a_blk = a.planes + (uint64_t)blk * a.steps * kF6Step;
    const uint32_t a_lds = lds_offset(lds), a_lane = lane * 16;
    auto digits_load = [&](uint32_t s, uint32_t buf) __attribute__((always_inline)) {
        const uint8_t* src = a_blk + (uint64_t)min(s, a.steps - 1) * kF6Step;
#pragma unroll
        for (uint32_t q = 0; q < (kF6Step / 1024 + 7) / 8; q++) {
            const uint32_t c = min(wave + 8 * q, kF6Step / 1024 - 1u) * 1024;
            lds_load16(a_lds + buf * kF6Step + c, src + c, a_lane);
        }
    };
    uint32_t exps[2], exps_next[2];                                // E8M0 bytes of two steps, per row tile of this wave
    const uint32_t e_pairs = (a.steps + 1) / 2;
    const auto b_exps = f6_array(a.exps + (uint64_t)blk * e_pairs * (kF6Tiles * 64), (uint64_t)e_pairs * (kF6Tiles * 128));
    auto exps_load = [&](uint32_t s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++)
            exps_next[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(
                b_exps, (int)(lane * 2), (int)(min(s, a.steps - 1) / 2 * (kF6Tiles * 128) + (wm * 2 + i) * 128), 0);
    };

    uint32_t deep = 0;                                             // kF6DeepBit of any run seen
    auto take_exps = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            deep |= exps_next[i];
            exps[i] = exps_next[i] & (0x0101u * (kF6DeepBit - 1));
        }
    };

    v16f acc[2][TN];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    auto scales_of = [&](uint32_t g) __attribute__((always_inline)) {
        return f6_cols_at<TN>(b_scales, my_col_c * 4, min(g, a.num_groups - 1) * row_bytes);
    };
    // The accumulators are kept in units of the current group's scale.  A scale far below the column's others would take them
    // out of f32's range (and a zero or a subnormal its reciprocal): the unit is 2^-60 of the column's largest scale, and
    // 2^-126, at least (w4_f6_prepare_kernel finds it), and a smaller group counts with that.  It lies in LDS, a slot per lane
    // (no registers are left): with the largest scale so far kept there from group to group a call took 2 to 3 % longer.
    float* const unit_slot = reinterpret_cast<float*>(lds + 2 * (kF6Step + BBYTES)) + tid * 4;
    auto units_read = [&]() __attribute__((always_inline)) {
        F6Floats<TN> o;
#pragma unroll
        for (int j = 0; j < TN; j++) o.v[j] = unit_slot[j];
        return o;
    };
    auto unit_of = [](float s, float least) __attribute__((always_inline)) { return copysignf(fmaxf(fabsf(s), least), s); };
    F6Floats<TN> sc_cur, sc_next, least, ratio;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        ratio.v[j] = 1.0f;
        unit_slot[j] = a.least[min(my_col_c + j, a.n - 1)];
    }

    constexpr int kB0 = 128 | (124 << 8) | (119 << 16) | (114 << 24), kB1 = 109 | (104 << 8);   // 2 / 2^shift of every digit

    auto read6 = [&](const uint8_t* hi, const uint8_t* lo) __attribute__((always_inline)) {
        const uint4 h = *reinterpret_cast<const uint4*>(hi + lane * 16);
        const uint2 l = *reinterpret_cast<const uint2*>(lo + lane * 8);
        return v6u{h.x, h.y, h.z, h.w, l.x, l.y};
    };

    // Step s from buffer P, in twelve sections of TN MFMAs (row tile i, digit d): a section's A fragment is read one section
    // ahead, and the vector work of a step is dealt out over its sections so that every MFMA has its share: the change of
    // the accumulators from one group's scale to the next (a row tile undergoes it while the other one multiplies, in the
    // second half of an odd step and the first half of an even one), and in the other halves the next step's weights.
    auto step = [&](uint32_t s, auto p_tag) __attribute__((always_inline)) {
        constexpr int P = decltype(p_tag)::value;
        constexpr bool ENDS = P == 1 || FOLD == 1, STARTS = P == 0 || FOLD == 1;   // a group may end / start with this step
        constexpr int D = kF6Digits, C0 = P == 0 ? D : 0;                       // first section of the conversion
        constexpr int SET = P ^ 1;                               // of step s + 1
        typedef std::integral_constant<int, P ^ 1> other;
        const uint8_t* const pa = lds + P * kF6Step + wm * 2 * kF6Tile;
        const uint8_t* const pb = lds_b + P * BBYTES + wn * TN * BTILE;
        v6u bf[TN], af[2];
        af[0] = read6(pa, pa + kF6Lo);
#pragma unroll
        for (int j = 0; j < TN; j++) bf[j] = read6(pb + j * BTILE, pb + j * BTILE + 1024);
#pragma unroll
        for (int t = 0; t < 2 * D; t++) {
            const int i = t / D, d = t % D;
            if (t + 1 < 2 * D) {
                const int i2 = (t + 1) / D, d2 = (t + 1) % D;
                af[(t + 1) & 1] = read6(pa + i2 * kF6Tile + d2 * 1024, pa + i2 * kF6Tile + kF6Lo + d2 * 512);
            }
            if (t == 0) digits_load(s + 1, P ^ 1);
            if (P == 1 && t == 1) exps_load(s + 1);
            if (t == C0 && ENDS) zero_points(FOLD == 1 ? SET : 0);
            if (t == C0 + 1 && ENDS) zp_load(s + 3, FOLD == 1 ? SET : 0);
            if (t == C0 || t == C0 + 1) convert_words(SET, 0, 2 * (t - C0));
            if (t == C0 + 2) column_store(0, other{});
            if (CPT == 2 && (t == C0 + 2 || t == C0 + 3)) convert_words(SET, 1, 2 * (t - C0 - 2));
            if (CPT == 2 && t == C0 + 4) column_store(1, other{});
            if (t == C0 + 3) { word_load(s + 3, SET, 0); word_load(s + 3, SET, 1); }
            if (t == C0 + 4) { word_load(s + 3, SET, 2); word_load(s + 3, SET, 3); }
            if (STARTS && t >= 1 && t <= TN) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[1][t - 1][r] *= ratio.v[t - 1];
            }
            // the scales of this step's group and the next step's
            if (ENDS && t == 1) {
                sc_cur = scales_of(min(s, a.steps - 1) / a.steps_per_group);
                sc_next = scales_of(min(s + 1, a.steps - 1) / a.steps_per_group);
            }
            if (ENDS && t == D - 1) least = units_read();
            if (ENDS && t == D) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const float sc = unit_of(sc_cur.v[j], least.v[j]), sn = unit_of(sc_next.v[j], least.v[j]);
                    const float rc = __builtin_amdgcn_rcpf(sn);
                    const float q = sc * rc;
                    ratio.v[j] = fmaf(fmaf(-q, sn, sc), rc, q);   // one correction step: within an ulp of the quotient, and 1 for the same group
                }
            }
            if (ENDS && t > D && t <= D + TN) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[0][t - D - 1][r] *= ratio.v[t - D - 1];
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const v8i fa = f6_operand(af[t & 1]), fb = f6_operand(bf[j]);
                // (the byte selectors are immediates)
                if (d == 0) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 0, kB0);
                if (d == 1) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 1, kB0);
                if (d == 2) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 2, kB0);
                if (d == 3) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 3, kB0);
                if (d == 4) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 0, kB1);
                if (d == 5) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 1, kB1);
            }
            // the reads of the next section, then MFMAs with a share of the vector work behind each
            if (t + 1 < 2 * D) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, FOLD == 1 ? 10 : 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (P == 1) take_exps();
        // this step's digits have landed once only the loads issued behind them are outstanding: words, exponents,
        // zero-points, scales
        RUMUS_F6_WAIT(4 + (ENDS ? 3 : 0) + (P == 1 ? 2 : 0));
        __builtin_amdgcn_s_barrier();
    };

    // PRE: digits and codes of a step, 36 + 6 TN KB, straight into LDS, chunk c of 1 KB by wave c % 8 (the last ones by several)
    constexpr uint32_t CHUNKS = (kF6Step + BBYTES) / 1024;
    const uint8_t* const c_blk = a.codes + (uint64_t)cblk * a.steps * BBYTES;
    auto step_load = [&](uint32_t s, uint32_t buf) __attribute__((always_inline)) {
        const uint64_t at = min(s, a.steps - 1);
        const uint8_t* const sa = a_blk + at * kF6Step, * const sb = c_blk + at * BBYTES;
#pragma unroll
        for (uint32_t q = 0; q < (CHUNKS + 7) / 8; q++) {
            const uint32_t c = min(wave + 8 * q, CHUNKS - 1u);
            constexpr uint32_t A = kF6Step / 1024;
            const bool of_a = c < A;
            lds_load16(a_lds + (of_a ? buf * kF6Step + c * 1024 : 2 * kF6Step + buf * BBYTES + (c - A) * 1024),
                       of_a ? sa + c * 1024 : sb + (c - A) * 1024, a_lane);
        }
    };
    auto codes_load = [&](uint32_t s, uint32_t buf) __attribute__((always_inline)) {   // the codes alone
#pragma unroll
        for (uint32_t q = 0; q < (BBYTES / 1024 + 7) / 8; q++) {
            const uint32_t c = min(wave + 8 * q, (uint32_t)BBYTES / 1024 - 1) * 1024;
            lds_load16(a_lds + 2 * kF6Step + buf * BBYTES + c, c_blk + (uint64_t)s * BBYTES + c, a_lane);
        }
    };
    v6u bq[2][TN], aq[3];                                          // fragments in flight: weights of two steps, three digits
    auto read_b = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const uint8_t* const p = lds_b + buf * BBYTES + (wn * TN + j) * BTILE;
            bq[buf][j] = read6(p, p + 1024);
        }
    };
    auto read_a = [&](int buf, int t) __attribute__((always_inline)) {
        const uint8_t* const p = lds + buf * kF6Step + (wm * 2 + t / kF6Digits) * kF6Tile;
        const int d = t % kF6Digits;
        aq[t % 3] = read6(p + d * 1024, p + kF6Lo + d * 512);
    };
    auto group_scales = [&](uint32_t s) __attribute__((always_inline)) {   // of step s and the one after it
        sc_cur = scales_of(min(s, a.steps - 1) / a.steps_per_group);
        sc_next = scales_of(min(s + 1, a.steps - 1) / a.steps_per_group);
    };
    // PRE: step s from buffer P, in twelve sections of TN MFMAs.  The digits are read two sections ahead; with the last of them read
    // a wave is done with the buffer, so the barrier stands two sections before the step's end: it publishes the next step, whose
    // first fragments arrive under the remaining MFMAs, and frees this one's buffer for the loads of step s + 2.
    auto step_pre = [&](uint32_t s, auto p_tag) __attribute__((always_inline)) {
        constexpr int P = decltype(p_tag)::value;
        constexpr bool ENDS = P == 1 || FOLD == 1, STARTS = P == 0 || FOLD == 1;
        constexpr int D = kF6Digits;
#pragma unroll
        for (int t = 0; t < 2 * D; t++) {
            const int i = t / D, d = t % D;
            if (t == 2 * D - 2) {
                RUMUS_F6_WAIT(0);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                read_b(P ^ 1);
                step_load(s + 2, P);
            }
            if (t < 2 * D - 2) read_a(P, t + 2);
            else read_a(P ^ 1, t + 2 - 2 * D);
            if (P == 1 && t == 1) exps_load(s + 1);
            if (FOLD == 2 && P == 0 && t == 1) group_scales(s + 1);
            if (FOLD == 1 && t == D + 1) group_scales(s + 1);
            if (STARTS && t >= 1 && t <= TN) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[1][t - 1][r] *= ratio.v[t - 1];
            }
            if (ENDS && t == D - 1) least = units_read();
            if (ENDS && t == D) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const float sc = unit_of(sc_cur.v[j], least.v[j]), sn = unit_of(sc_next.v[j], least.v[j]);
                    const float rc = __builtin_amdgcn_rcpf(sn);
                    const float q = sc * rc;
                    ratio.v[j] = fmaf(fmaf(-q, sn, sc), rc, q);
                }
            }
            if (ENDS && t > D && t <= D + TN) {
#pragma unroll
                for (int r = 0; r < 16; r++) acc[0][t - D - 1][r] *= ratio.v[t - D - 1];
            }
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const v8i fa = f6_operand(aq[t % 3]), fb = f6_operand(bq[P][j]);
                if (d == 0) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 0, kB0);
                if (d == 1) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 1, kB0);
                if (d == 2) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 2, kB0);
                if (d == 3) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 3, kB0);
                if (d == 4) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 0, kB1);
                if (d == 5) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa, fb, acc[i][j], 2, 2, P, (int)exps[i], 1, kB1);
            }
            if (t == 2 * D - 2) __builtin_amdgcn_sched_group_barrier(0x100, 2 * TN + 2, 0);
            else __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int j = 0; j < TN; j++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, FOLD == 1 ? 10 : 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (P == 1) take_exps();
    };

    uint32_t s = 0;
    if constexpr (PRE) {
        exps_load(0);
        if constexpr (FOLD == 1) group_scales(0);
        step_load(0, 0);
        step_load(1, 1);
        RUMUS_F6_WAIT(0);
        take_exps();
        __builtin_amdgcn_s_barrier();
        read_b(0);
        read_a(0, 0);
        read_a(0, 1);
        __builtin_amdgcn_sched_barrier(0);
        for (; s + 1 < a.steps; s += 2) {
            step_pre(s, std::integral_constant<int, 0>{});
            step_pre(s + 1, std::integral_constant<int, 1>{});
        }
        if (s < a.steps) step_pre(s, std::integral_constant<int, 0>{});
    } else {
    digits_load(0, 0);
    exps_load(0);
    take_exps();
    if constexpr (FOLD == 1) zp_load(1, 1);
    zp_load(0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) word_load(0, 0, i);
#pragma unroll
    for (int i = 0; i < 4; i++) word_load(1, 1, i);
    zero_points(0);
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        convert_words(0, c, 0);
        convert_words(0, c, 2);
        column_store(c, std::integral_constant<int, 0>{});
    }
#pragma unroll
    for (int i = 0; i < 4; i++) word_load(2, 0, i);
    zp_load(2, 0);
    RUMUS_F6_WAIT(0);
    __builtin_amdgcn_s_barrier();
    for (; s + 1 < a.steps; s += 2) {
        step(s, std::integral_constant<int, 0>{});
        step(s + 1, std::integral_constant<int, 1>{});
    }
    if (s < a.steps) step(s, std::integral_constant<int, 0>{});
    }
    RUMUS_F6_WAIT(0);                                              // the loads past the last step have landed: the LDS is free
    __syncthreads();

    // the last unit of every column; the slots hold these from now on
    sc_cur = scales_of(a.num_groups - 1);
    least = units_read();
#pragma unroll
    for (int j = 0; j < TN; j++) {
        sc_cur.v[j] = least.v[j] != least.v[j] ? least.v[j] : unit_of(sc_cur.v[j], least.v[j]);   // (the column holds a NaN)
        unit_slot[j] = sc_cur.v[j];
    }

    // ---- the further digits of marked runs; ordinary data has none --------------------------------------------------
    if (__syncthreads_or((deep & (0x0101u * kF6DeepBit)) != 0)) {
        // LDS: the codes of the further digits, the step's values of x and RMSNorm weights, and which steps have marks
        constexpr int DTILE = kF6Deep * 1536;
        constexpr uint32_t PITCH = 64 + 4;
        static_assert(kF6Tiles * DTILE + (kF6BM * PITCH + 64 + kF6MaxK / 64) * 4 <= 2 * kF6Step, "they fit the buffers of the planes");
        float* const values = reinterpret_cast<float*>(lds + kF6Tiles * DTILE);
        float* const weights = values + kF6BM * PITCH;
        uint32_t* const has_marks = reinterpret_cast<uint32_t*>(weights + 64);
        if (tid < kF6MaxK / 64) has_marks[tid] = 0;
        __syncthreads();
        {
            const uint32_t* const e2 = reinterpret_cast<const uint32_t*>(a.exps) + (uint64_t)blk * e_pairs * (kF6Tiles * 32);
            for (uint32_t i = tid; i < e_pairs * (kF6Tiles * 32); i += 512) {   // two lanes of a pair of steps
                const uint32_t e = e2[i];
                if (e & 0x00010001u * kF6DeepBit) has_marks[i / (kF6Tiles * 32) * 2] = 1;
                if (e & 0x01000100u * kF6DeepBit) has_marks[i / (kF6Tiles * 32) * 2 + 1] = 1;
            }
        }
        __syncthreads();
        // a thread per run: its row's factors
        const uint32_t d_row = m0 + tid % kF6BM, d_half = tid / kF6BM, d_tile = tid % kF6BM / 32, d_lane = d_half * 32 + (tid & 31);
        const uint32_t d_rowc = min(d_row, a.m - 1);
        const float d_rv = __uint_as_float((254u - (__float_as_uint(a.rfac[d_rowc]) >> 23)) << 23), d_inv = a.norm_w ? a.rinv[d_rowc] : 0.0f;
        for (uint32_t s = 0; s < a.steps; s++) {
            if (!has_marks[s]) continue;
            const uint32_t e_shift = 8 * (s & 1);
            // everything that the step reads from memory at once: its weights and values once more, exponents, scales
            const uint32_t kk = 64 * s + lane, from = kk >= a.k ? 0 : a.perm ? (uint32_t)a.perm[kk] : kk;
            if constexpr (PRE) {
                codes_load(s, 0);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) word_load(s, 0, i);
                zp_load(s, 0);
            }
            exps_load(s);
            const uint32_t e = a.exps[(((uint64_t)blk * e_pairs + s / 2) * kF6Tiles + d_tile % kF6Tiles) * 64 + d_lane % 64] >> e_shift & 0xffu;
            const F6Floats<TN> sc = scales_of(s / a.steps_per_group);
            constexpr int ROWS = kF6BM / 8;                        // of a wave, 64 values each
            const uint32_t width = a.glu ? 2 * a.k : a.k;
            float xv[ROWS];
#pragma unroll
            for (int i = 0; i < ROWS; i++) xv[i] = a.x[(uint64_t)min(m0 + wave + 8 * i, a.m - 1) * width + from];
            if (a.glu) {
                float up[ROWS];
#pragma unroll
                for (int i = 0; i < ROWS; i++) up[i] = a.x[(uint64_t)min(m0 + wave + 8 * i, a.m - 1) * width + a.k + from];
#pragma unroll
                for (int i = 0; i < ROWS; i++) xv[i] = f6_glu(xv[i], up[i]);
            }
            if (a.norm_w && wave == 0) weights[lane] = kk < a.k ? a.norm_w[from] : 0.0f;
#pragma unroll
            for (int i = 0; i < ROWS; i++) values[(wave + 8 * i) * PITCH + lane] = kk < a.k ? xv[i] : 0.0f;
            if constexpr (!PRE) {
                zero_points(0);
#pragma unroll
                for (int c = 0; c < CPT; c++) {
                    convert_words(0, c, 0);
                    convert_words(0, c, 2);
                    column_store(c, std::integral_constant<int, 0>{});
                }
            }
            __syncthreads();
            // the runs' digits past those that the planes hold
            if (tid < 2 * kF6BM) {
                const bool marked = (e & kF6DeepBit) != 0;        // (rows past m are not)
                const uint32_t rt = d_tile, ln = d_lane;
                uint8_t* const to = lds + rt * DTILE;
                v16f ev, od;
                if (marked) {
                    float v[32];
#pragma unroll
                    for (int j = 0; j < 32; j++) v[j] = values[tid % kF6BM * PITCH + 32 * d_half + j];
                    if (a.norm_w) {
#pragma unroll
                        for (int j = 0; j < 32; j++) v[j] = f6_norm(v[j], d_inv, weights[32 * d_half + j]);
                    }
#pragma unroll
                    for (int j = 0; j < 32; j++) v[j] *= d_rv;
                    f6_order(v, ev, od);
#pragma unroll
                    for (int d = 0; d < kF6Digits; d++) (void)f6_digit(ev, od, __uint_as_float(((e & (kF6DeepBit - 1)) - kF6Shift[d]) << 23));
                } else {
#pragma unroll
                    for (int j = 0; j < 16; j++) ev[j] = od[j] = 0.0f;
                }
#pragma unroll
                for (int d = 0; d < kF6Deep; d++) {
                    // (unmarked: zeros in any unit)
                    const v6u code = f6_digit(ev, od, marked ? __uint_as_float(((e & (kF6DeepBit - 1)) - kF6Shift[kF6Digits + d]) << 23) : 1.0f);
                    *reinterpret_cast<uint4*>(to + d * 1536 + ln * 16) = make_uint4(code[0], code[1], code[2], code[3]);
                    *reinterpret_cast<uint2*>(to + d * 1536 + 1024 + ln * 8) = make_uint2(code[4], code[5]);
                }
            }
            RUMUS_F6_WAIT(0);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int ea = (int)(exps_next[i] >> e_shift & (kF6DeepBit - 1));
                const uint8_t* const pa = lds + (wm * 2 + i) * DTILE;
                v8i da[kF6Deep];
#pragma unroll
                for (int d = 0; d < kF6Deep; d++) da[d] = f6_operand(read6(pa + d * 1536, pa + d * 1536 + 1024));
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const uint8_t* const pb = lds_b + (wn * TN + j) * BTILE;
                    const v8i fb = f6_operand(read6(pb, pb + 1024));
                    v16f t;
#pragma unroll
                    for (int r = 0; r < 16; r++) t[r] = 0.0f;
                    t = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(da[0], fb, t, 2, 2, 0, ea, 0, 128 - kF6Shift[kF6Digits]);
                    t = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(da[1], fb, t, 2, 2, 0, ea, 0, 128 - kF6Shift[kF6Digits + 1]);
                    const float ratio_s = sc.v[j] / sc_cur.v[j];
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(t[r], ratio_s, acc[i][j][r]);
                }
            }
            __syncthreads();                                       // before the next step's codes
        }
    }

    // ---- what integer zero-points left over: - sum over g of scale (zp - z) (sum of x over the group) ----------------
    if constexpr (!ZP4) {
        if (__builtin_amdgcn_ballot_w64((zflag.x | zflag.y | zflag.z | zflag.w) != 0) != 0) {   // the same in every wave
            // A product of two f32 tables over the groups, exact to 24 bits on the bf16 matrix cores: both factors split into
            // three bf16 parts, eight of the nine products; the 16 k slots of an instruction are two groups of eight
            // products, lane half h carries group g + h.  The tables go through LDS, GROUPS groups at a time: read from
            // memory by every wave for itself, one trip per few groups, they cost 17 us a launch instead of 12.
            constexpr uint32_t GROUPS = 32;
            static_assert(GROUPS * (BN + kF6BM) * 4 <= 2 * (kF6Step + BBYTES), "the tables fit the LDS");
            float* const t_y = reinterpret_cast<float*>(lds);          // [GROUPS][BN], in the accumulators' unit
            float* const t_x = t_y + GROUPS * BN;                      // [GROUPS][kF6BM]
            auto parts = [](float v, short (&p)[3]) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    const uint32_t hi = __float_as_uint(v) & 0xffff0000u;
                    p[q] = (short)(hi >> 16);
                    v -= __uint_as_float(hi);
                }
            };
            const uint32_t spg = a.steps_per_group, gb = a.num_groups - 1;
            const uint32_t t_col = min(n0 + tid, a.n - 1);             // BN <= 512: a column per thread
            __syncthreads();
            const uint32_t t_c = min(tid, (uint32_t)BN - 1);
            const float last = reinterpret_cast<const float*>(lds + 2 * (kF6Step + BBYTES))[(t_c / (32 * TN) * 64 + t_c % (32 * TN) / TN) * 4 + t_c % TN];
            const float t_unit = 1.0f / last;
            for (uint32_t g0 = 0; g0 <= gb; g0 += GROUPS) {
                const uint32_t count = min(GROUPS, gb - g0 + 1);
                if (tid < BN) {
                    for (uint32_t g = 0; g < GROUPS; g += 8) {
                        float sv[8], zv[8];
#pragma unroll
                        for (int u = 0; u < 8; u++) {
                            const uint32_t at = min(g0 + g + u, gb) * a.n + t_col;
                            sv[u] = a.scales[at];
                            zv[u] = a.zp[at];
                        }
#pragma unroll
                        for (int u = 0; u < 8; u++) {
                            const float z = fminf(fmaxf(rintf(zv[u]), 0.0f), 15.0f);
                            t_y[(g + u) * BN + tid] = g + u < count ? -(zv[u] - z) * sv[u] * t_unit : 0.0f;
                        }
                    }
                }
                for (uint32_t e = tid; e < GROUPS * kF6BM; e += 512) {
                    const uint32_t g = min(g0 + e / kF6BM, gb), sa = g * spg, sb = min(g * spg + spg, a.steps);
                    const float* p = a.sums + ((uint64_t)blk * a.steps + sa) * kF6BM + e % kF6BM;
                    float v = p[0] + (sb - sa > 1 ? p[kF6BM] : 0.0f);
                    for (uint32_t s = sa + 2; s < sb; s++) v += p[(s - sa) * kF6BM];
                    t_x[e] = e / kF6BM < count ? v : 0.0f;
                }
                __syncthreads();
                for (uint32_t g2 = 0; g2 < count; g2 += 2) {
                    const uint32_t g = g2 + kb;                        // (rows past count hold zeros)
                    v8s fb[TN];
                    short p[3];
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        parts(t_y[g * BN + wn * (32 * TN) + TN * l32 + j], p);
                        fb[j] = v8s{p[0], p[1], p[2], p[0], p[1], p[0], p[2], p[1]};
                    }
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        parts(t_x[g * kF6BM + (wm * 2 + i) * 32 + l32], p);
                        const v8s fa = v8s{p[0], p[0], p[0], p[1], p[1], p[2], p[1], p[2]};
#pragma unroll
                        for (int j = 0; j < TN; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, fa), __builtin_bit_cast(v8bf, fb[j]), acc[i][j], 0, 0, 0);
                    }
                }
                __syncthreads();
            }
        }
    }

    // ---- store -------------------------------------------------------------------------------------------------
    // All row factors first (rfac holds whole blocks of rows): a load in front of every store would cost a trip to memory per
    // row, since its wait includes the stores before it.
    float rf[2][16];                                              // back to the rows' own scale: exact, powers of two
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4 f = *reinterpret_cast<const float4*>(a.rfac + m0 + (wm * 2 + i) * 32 + 8 * q + 4 * kb);
            rf[i][4 * q] = f.x; rf[i][4 * q + 1] = f.y; rf[i][4 * q + 2] = f.z; rf[i][4 * q + 3] = f.w;
        }
    float bv[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) bv[j] = a.bias && my_col + j < a.n ? a.bias[my_col + j] : 0.0f;
    if (my_col >= a.n) return;
    const bool whole = m0 + kF6BM <= a.m, inside = TN != 3 || my_col + TN <= a.n;   // (otherwise the right edge: n % 4 == 0)
    auto row_of = [&](int i, int r) { return m0 + (wm * 2 + i) * 32 + 8 * (r / 4) + 4 * kb + (r % 4); };
    auto put = [&](int i, int r, const F6Floats<TN>& add) __attribute__((always_inline)) {
        F6Floats<TN> o;
#pragma unroll
        for (int j = 0; j < TN; j++) o.v[j] = fmaf(acc[i][j][r] * rf[i][r], sc_cur.v[j], bv[j]);
        if (a.residual)
#pragma unroll
            for (int j = 0; j < TN; j++) o.v[j] += add.v[j];
        float* p = a.y + (uint64_t)row_of(i, r) * a.n + my_col;
        if (inside) {
            f6_cols_store<TN>(p, o);
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
                if (my_col + j < a.n) p[j] = o.v[j];
        }
    };
    if (a.residual) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) {                         // four rows at a time: their loads, then their stores
                F6Floats<TN> add[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float* p = a.residual + (uint64_t)min(row_of(i, 4 * q + r), a.m - 1) * a.n + my_col;
#pragma unroll
                    for (int j = 0; j < TN; j++) add[r].v[j] = p[inside || my_col + j < a.n ? j : 0];
                }
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (whole || row_of(i, 4 * q + r) < a.m) put(i, 4 * q + r, add[r]);
            }
        return;
    }
    const F6Floats<TN> none = {};
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            if (whole || row_of(i, r) < a.m) put(i, r, none);
}

// How a call runs: columns per workgroup / 128, and whether the weights are converted once, before the matmul, or by every
// block of rows for itself.  `us`: the time of a call in microseconds: workgroups run one per compute unit, in rounds of 256.
// A round's steps (of 64 k) take L at least, and with more than about 170 workgroups at work each is slower: a launch as a whole
// does not beat P per 256 workgroup-steps.  16 is a round's start and end, the rest the preparation, of the weights too where it does those.
// The form was fitted to 252 timings with five digits, each width forced (130 .. 4096 rows; seven weights), L, P and the preparation
// then to 50 calls with six (512 to 4096 rows, 1024 -> 2816 to 8192 -> 8192 and 4096 -> 22016), with converted weights to 240 of
// 288 to 4096 rows, as a ratio to the same call without: within 5 %, up to 10 % too low at k = 11008.
struct F6Plan {
    int tn;
    bool codes;
    double us;
};
// Converted weights take 3/4 of a byte per weight of the workspace: a call asks for at most this much on top of what it needs.
constexpr uint64_t kF6MostCodes = uint64_t(256) << 20;
static uint64_t f6_codes_bytes(uint32_t k, uint32_t n, int tn) { return (uint64_t)ceil_div(n, 128 * tn) * ceil_div(k, 64) * (tn * 4 * 1536); }

static F6Plan f6_plan(uint32_t m, uint32_t k, uint32_t n, bool may_convert) {
    static const double L[2][3] = {{1.24, 1.59, 1.87}, {1.00, 1.34, 1.70}}, P[2][3] = {{1.31, 2.00, 2.58}, {1.27, 1.92, 2.46}};
    const double steps = ceil_div(k, 64);
    F6Plan best{4, false, 1e30};
    for (int codes = 0; codes <= (may_convert ? 1 : 0); codes++)
        for (int tn = 4; tn >= 2; tn--) {
            if (codes && f6_codes_bytes(k, n, tn) > kF6MostCodes) continue;
            const double wgs = (double)ceil_div(m, kF6BM) * ceil_div(n, 128 * tn), rounds = std::ceil(wgs / 256.0);
            const double chain = rounds * (steps * L[codes][tn - 2] + 16.0), power = wgs / 256.0 * steps * P[codes][tn - 2];
            const double t = std::sqrt(std::sqrt(chain * chain * chain * chain + power * power * power * power)) + 3.0 + 2.0e-6 * m * k +
                             (codes ? 0.2e-6 * k * n : 0.0);
            if (t < best.us) best = F6Plan{tn, codes != 0, t};
        }
    return best;
}

static size_t f6_up(size_t v) { return (v + 255) & ~size_t(255); }

struct F6Workspace {
    uint32_t blocks, steps;
    size_t planes, exps, sums, rfac, rinv, least, flags, total;   // bytes
    F6Workspace(uint32_t m, uint32_t padded_k, uint32_t n) : blocks(ceil_div(m, kF6BM)), steps(padded_k / 64) {
        planes = (size_t)blocks * steps * kF6Step;
        exps = f6_up((size_t)blocks * ((steps + 1) / 2) * kF6Tiles * 64 * 2);
        sums = (size_t)blocks * steps * kF6BM * 4;
        rfac = (size_t)blocks * kF6BM * 4;
        rinv = rfac;
        least = f6_up((size_t)n * 4);
        flags = kF6Flags * 4;
        total = planes + exps + sums + rfac + rinv + least + flags;
    }
};

// Six digits park 4.6 bytes per element of x, the f16 tiles 4.25.  What those run within the fixed scratch array (w4_gemv.hip),
// and what a caller reserved by the documented bound, has to do for this kernel too: such a call runs as two halves of its rows.
constexpr uint64_t kF6Array = uint64_t(32) << 20;
static bool f6_array_fits(uint32_t m, uint32_t padded_k) { return (uint64_t)m * padded_k * 17 / 4 <= kF6Array; }
static uint32_t f6_rows_at_once(uint32_t m, uint32_t padded_k, uint32_t n) {
    const F6Workspace w(m, padded_k, n);
    uint64_t limit = (uint64_t)5 * (m + 64) * (padded_k + 128);
    if (f6_array_fits(m, padded_k)) limit = std::min(limit, kF6Array);
    return w.total <= limit ? m : ceil_div(w.blocks, 2) * kF6BM;
}

// More than 256 rows (blocks of 128 rows: up to there the integer kernel's blocks of 64 fit as well or better, and K would have to be
// shared over workgroups), where its time is below what the other two kernels are expected to take.  The two estimates of
// those are loosest upwards for the integer kernel (8192 -> 8192 at 640 rows: 201 us expected, 164 measured, 185 here), hence its
// margin.  Over 45 calls above 512 rows the choice takes 10 % less time than the older kernels alone, 24 % at best (1000 rows
// 4096 -> 11008 199 -> 152 us), and 6 % more at worst (1400 rows 11008 -> 4096 283 -> 293).
bool w4_gemm_f6_chosen(const W4Args& a) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(a.packed) | reinterpret_cast<uintptr_t>(a.scales) |
                           reinterpret_cast<uintptr_t>(a.zp) | reinterpret_cast<uintptr_t>(a.y) |
                           reinterpret_cast<uintptr_t>(a.perm) | reinterpret_cast<uintptr_t>(a.bias);
    if (!(a.m > 256 && a.m <= 65535u * kF6BM && a.n % 4 == 0 && (bits & 15) == 0 && !a.g_idx && !a.tiled &&
          a.group_size % 64 == 0 && (!a.zp4 || a.n % 8 == 0) && a.k >= 1024 &&                    // (what the estimates were fitted to)
          a.padded_k <= kF6MaxK &&
          (a.x != a.y || !a.x) &&                              // (marked runs read x again while other workgroups store)
          (uint64_t)a.padded_k / 8 * a.n * 4 < (1ull << 32) && (uint64_t)a.m * a.n < (1ull << 32)))
        return false;
    double other = 0.0;
    // (the time without codes, for every call: whether there is room for them must not change the kernel, that is the bits.  With
    // them it is 6 to 10 % less, so where it is close the call goes to a slower kernel.)
    const double us = f6_plan(a.m, a.k, a.n, false).us;
    const bool i8 = w4_gemm_i8_supported(a, &other);
    // what the integer kernel runs within the fixed scratch array (w4_gemv.hip), 3.1 bytes per element of x, has to go on running there
    if (i8 && !f6_array_fits(a.m, a.padded_k)) return false;
    return us < (i8 ? 0.92 : 1.0) * other;
}

template <int TN, int FOLD, bool ZP4, bool PRE>
static int launch_f6(F6Args f, uint32_t blocks, hipStream_t s) {
    f.row_blocks = blocks;
    f.col_blocks = ceil_div(f.n, 128 * TN);
    constexpr size_t lds_bytes = 2 * (size_t)(kF6Step + 4 * TN * (PRE ? 1536 : kF6BTile)) + 512 * 16;
    static_assert(lds_bytes <= 160 * 1024, "two steps fit the LDS");
    static bool attr_set = false;   // benign race: setting the attribute is idempotent
    if (!attr_set) {
        if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&w4_gemm_f6_kernel<TN, FOLD, ZP4, PRE>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes),
                               "hipFuncSetAttribute"))
            return rc;
        attr_set = true;
    }
    hipLaunchKernelGGL((w4_gemm_f6_kernel<TN, FOLD, ZP4, PRE>), dim3(f.col_blocks * blocks), dim3(512), lds_bytes, s, f);
    return check_launch("w4_gemm_f6_kernel");
}

template <int TN, bool ZP4>
static int launch_f6_groups(const F6Args& f, const W4Args& a, uint32_t blocks, uint8_t* codes, hipStream_t s) {
    const bool wide = a.group_size % 128 == 0;
    if (!codes) return wide ? launch_f6<TN, 2, ZP4, false>(f, blocks, s) : launch_f6<TN, 1, ZP4, false>(f, blocks, s);
    return wide ? launch_f6<TN, 2, ZP4, true>(f, blocks, s) : launch_f6<TN, 1, ZP4, true>(f, blocks, s);
}

static int launch_f6_rows(const W4Args& a, hipStream_t s, const W4BlockArgs& block, const F6Plan& plan) {
    const F6Workspace w(a.m, a.padded_k, a.n);
    const size_t codes_bytes = plan.codes ? f6_codes_bytes(a.padded_k, a.n, plan.tn) : 0;
    void* ws = nullptr;
    WorkspaceLease lease;                                    // until the last kernel of this call is queued
    if (int rc = workspace_get(s, w.total + codes_bytes, &ws, lease)) return rc;
    uint8_t* p = static_cast<uint8_t*>(ws);
    uint8_t* const planes = p; p += w.planes;
    uint8_t* const exps = p; p += w.exps;
    float* const sums = reinterpret_cast<float*>(p); p += w.sums;
    float* const rfac = reinterpret_cast<float*>(p); p += w.rfac;
    float* const rinv = reinterpret_cast<float*>(p); p += w.rinv;
    float* const least = reinterpret_cast<float*>(p); p += w.least;
    uint32_t* const zflags = reinterpret_cast<uint32_t*>(p); p += w.flags;
    uint8_t* const codes = codes_bytes ? p : nullptr;
    // rows per workgroup of the preparation: at most 512 units and 80 KB of LDS (two workgroups per compute unit), and enough workgroups
    const uint32_t units = 2 * w.steps, pitch = units * 36 + 4, rows_pad = w.blocks * kF6BM;
    uint32_t rows = 8;
    while (rows > 1 && ((size_t)rows * pitch * 4 > 80 * 1024 || rows * units > 512 || rows_pad / rows < 256)) rows /= 2;
    static bool attr_set = false;   // benign race: setting the attribute is idempotent
    if (!attr_set) {
        for (const void* f : {reinterpret_cast<const void*>(&w4_f6_prepare_kernel<kF6Plain>), reinterpret_cast<const void*>(&w4_f6_prepare_kernel<kF6Perm>),
                              reinterpret_cast<const void*>(&w4_f6_prepare_kernel<kF6Norm>), reinterpret_cast<const void*>(&w4_f6_prepare_kernel<kF6Glu>)})
            if (int rc = check_hip(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024), "hipFuncSetAttribute"))
                return rc;
        attr_set = true;
    }
    const F6Weights weights{a.packed, a.zp, a.zp4, codes, a.n, w.steps, a.group_size / 64, a.num_groups, (uint32_t)plan.tn};
    const dim3 pgrid(rows_pad / rows + ceil_div(a.n, 64) + (a.zp4 ? 0 : kF6Flags) +
                     (codes ? ceil_div(a.n, 128 * plan.tn) * ceil_div(w.steps, kF6CodeSteps) : 0));
#define RUMUS_F6_PREPARE(IN)                                                                                             \
    hipLaunchKernelGGL(w4_f6_prepare_kernel<IN>, pgrid, dim3(512), (size_t)rows * pitch * 4, s, a.x, a.perm, planes, exps, sums, \
                       rfac, a.m, a.k, w.steps, rows, pitch, reinterpret_cast<const float4*>(a.zp),                        \
                       (uint32_t)((uint64_t)a.num_groups * a.n / 4), zflags, a.scales, a.num_groups, a.n, least, rows_pad / rows, block.norm_w, block.eps, rinv, weights)
    if (a.perm) RUMUS_F6_PREPARE(kF6Perm);
    else if (block.norm_w) RUMUS_F6_PREPARE(kF6Norm);
    else if (a.glu) RUMUS_F6_PREPARE(kF6Glu);
    else RUMUS_F6_PREPARE(kF6Plain);
#undef RUMUS_F6_PREPARE
    if (int rc = check_launch("w4_f6_prepare_kernel")) return rc;
    const F6Args f{a.packed, a.scales, a.zp, a.zp4, a.bias, planes, codes, reinterpret_cast<const uint16_t*>(exps), sums, a.x, a.perm, block.norm_w, a.glu, rinv,
                   rfac, least, zflags, a.y, a.m, a.k, a.n, w.steps, a.group_size / 64, a.num_groups, block.residual};
    switch (plan.tn) {
        case 2: return a.zp4 ? launch_f6_groups<2, true>(f, a, w.blocks, codes, s) : launch_f6_groups<2, false>(f, a, w.blocks, codes, s);
        case 3: return a.zp4 ? launch_f6_groups<3, true>(f, a, w.blocks, codes, s) : launch_f6_groups<3, false>(f, a, w.blocks, codes, s);
        default: return a.zp4 ? launch_f6_groups<4, true>(f, a, w.blocks, codes, s) : launch_f6_groups<4, false>(f, a, w.blocks, codes, s);
    }
}

int w4_launch_gemm_f6(const W4Args& a, hipStream_t s, const W4BlockArgs& block) {
    RUMUS_REQUIRE(a.padded_k <= kF6MaxK, "qmatmul_int4: padded_k %u is beyond the six-bit kernel's %u", a.padded_k, kF6MaxK);
    // With the weights converted where the workspace has room for that or may grow; the same bits without.  A size that the caller
    // set holds what is taken without: the digits of `rows` rows, which may be half of all.
    const uint32_t rows = f6_rows_at_once(a.m, a.padded_k, a.n);
    const F6Plan plan = f6_plan(a.m, a.padded_k, a.n, true);
    if (plan.codes) {
        const size_t least = F6Workspace(min(rows, a.m), a.padded_k, a.n).total;
        const size_t all = F6Workspace(a.m, a.padded_k, a.n).total + f6_codes_bytes(a.padded_k, a.n, plan.tn);
        size_t got = 0;
        void* ws = nullptr;
        WorkspaceLease lease;
        if (int rc = workspace_get_upto(s, least, all, &got, &ws, lease)) return rc;
        if (got == all) return launch_f6_rows(a, s, block, plan);
    }
    for (uint32_t r0 = 0; r0 < a.m; r0 += rows) {
        W4Args part = a;
        W4BlockArgs around = block;
        part.m = min(rows, a.m - r0);
        part.x = a.x + (uint64_t)r0 * a.k * (a.glu ? 2 : 1);
        part.y = a.y + (uint64_t)r0 * a.n;
        if (block.residual) around.residual = block.residual + (uint64_t)r0 * a.n;
        if (int rc = launch_f6_rows(part, s, around, f6_plan(part.m, part.padded_k, part.n, false))) return rc;
    }
    return RUMUS_HIP_OK;
}

}  // namespace rumus
