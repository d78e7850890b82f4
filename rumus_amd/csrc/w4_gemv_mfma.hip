// INT4 engine: the decode-shape kernel for 2 to 8 rows (group_size % 32 == 0), on the int8 matrix cores in one launch.
//
//   y[m,n] = sum_c 2^-e[m,c] sum_{g in c} scale[g,n] * ( sum_{k in g} X[m,k] q[k,n]  -  zp[g,n] * sum_{k in g} X[m,k] )
//
// over units c of 128 or 256 consecutive k, with X = rint(x 2^e), e from the unit's largest magnitude, whose X is 2^21 to 2^22 (all but: w4m_digits).
// X = d0 + 2^8 d1 + 2^16 d2 in signed bytes, and the sixteen rows of v_mfma_i32_16x16x64_i8 are three digits of four rows of x and, fourth, ones.
// In its accumulator layout a lane then holds all digits' sums of one output, so folding a group takes eight vector instructions per
// output and no exchange, and four rows cost the matrix cores what one does.
//
// Why beside w4_gemv_dot8.hip: there the activations become nibble planes in every lane for sixteen columns, 62 vector instructions per row and 128 k
// of a wave, which made every row cost a microsecond at 4096 x 4096, and the code of a row of its own; here 128 k cost 55 for four rows.
// From HBM, us, there -> here: 4 x 1024 x 1024 6.8 -> 2.9, 4 x 4096 x 4096 7.8 -> 5.4, 4 x 1152 x 8064 12.0 -> 4.5, 8 x 2048 x 2048 11.9 -> 4.9, groups of 32 the same
// shape 11.4 -> 4.1 (1024); act-order 4 x 4096 x 4096 17.4 -> 8.9, 8 x 512 x 11008 82 -> 6.4; f16 rows 4 x 4096 x 4096 11.9 (with two launches that convert) -> 5.9.
// What bounds it: vector issue of the conversion (half of the launch at 4 x 4096 x 4096), then latency.  Error against float64 with some channels 20
// times as large 3.3e-6 -> 1.1e-6, N(0,1) 2.0e-6 -> 0.3e-6.
//
// A workgroup owns 16 Q columns over the whole of K (no partial sums in memory); its eight waves take units in turn, all loads of U units
// in flight, activations first.  Every activation is loaded and converted once per workgroup; the byte transposition that the digits need
// is a trip through the wave's own part of LDS, without a barrier.
//
// Elements that tower over their unit: where all of one lane's elements (8 or 16 of a unit) lie 2^8 below the unit's largest, the row's part is multiplied on
// its own, and what its digits left of the elements is taken for further digits, 22 bits at a time until nothing is left of them: sums of exact
// products, whatever their spread.
#include <atomic>
#include <type_traits>

#include "w4.h"

namespace rumus {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

constexpr int kW4mWaves = 8, kW4mThreads = 64 * kW4mWaves;
constexpr uint32_t kW4mLds = 128 * 1024;      // dynamic LDS: digits, and rows of an act-order call

// Where the activations come from.  kW4mAny reads them one by one (any k, any alignment, act-order rows beyond LDS).
enum W4mIn { kW4mVec, kW4mHalf, kW4mPerm, kW4mAny, kW4mNorm, kW4mGlu };

#define W4M_DPP(v, ctrl) __builtin_amdgcn_update_dpp(0, (int)(v), (ctrl), 0xF, 0xF, true)

struct W4mArgs {
    const uint32_t* packed;
    const float* scales;
    const uint32_t* zps;          // f32 [groups, n], or packed u4
    const void* x;
    void* y;
    const float* bias;
    const int32_t* perm;
    const float* norm_w;
    const float* resid;           // may be y
    uint32_t m, k, n, padded_k, group_size;
    float eps;
    uint32_t per_group;           // ceil(2^32 / (group_size / 16))
    bool zp4, tiled;              // packed u4 zero-points; tile-major copies (w4_decode_layout)
};

// silu(g) * u, the expression of swiglu_kernel (block_glue.hip): the same bits
__device__ __forceinline__ float w4m_silu(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Four values x 2^e (k 0, 2, 4, 6 or 1, 3, 5, 7 of a packed word) -> dword b: digit b of each, k ascending.  Adding 1.5 * 2^23 + 0x8080
// leaves X + 0x408080 in the low bits: bytes 128 + d0, 128 + d1, 64 + d2.  The 64 stays (w4m_sum takes it off again), the fourth dword is ones.
__device__ __forceinline__ v4i w4m_digits(const float (&v)[4], float f) {
    uint32_t Z[4];
#pragma unroll
    for (int j = 0; j < 4; j++) Z[j] = __float_as_uint(fmaf(v[j], f, 12615808.0f));
    const uint32_t e0 = __builtin_amdgcn_perm(Z[1], Z[0], 0x05010400u), e1 = __builtin_amdgcn_perm(Z[1], Z[0], 0x0c0c0602u);
    const uint32_t f0 = __builtin_amdgcn_perm(Z[3], Z[2], 0x05010400u), f1 = __builtin_amdgcn_perm(Z[3], Z[2], 0x06020c0cu);
    return v4i{(int)(__builtin_amdgcn_perm(f0, e0, 0x05040100u) ^ 0x80808080u), (int)(__builtin_amdgcn_perm(f0, e0, 0x07060302u) ^ 0x80808080u),
               (int)(e1 | f1), 0x01010101};
}
// the largest magnitude of four, as bits: a NaN sorts highest
__device__ __forceinline__ uint32_t w4m_largest(const float (&v)[4]) {
    float top = __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(v[0]), fabsf(v[1])), fabsf(v[2]));
    return __float_as_uint(__builtin_elementwise_maximum(top, fabsf(v[3]))) & 0x7fffffffu;
}
__device__ __forceinline__ float w4m_sum(const v4i& c) {      // of the digits' sums: exact but for two roundings
    return fmaf((float)(c[2] - 64 * c[3]), 65536.0f, (float)((c[1] << 8) + c[0]));
}
// the same where zero-points of up to 1023 have been taken off: 128 products of a digit then make up to 2^24, and not 256 times that in 32 bits
__device__ __forceinline__ float w4m_wide_sum(const v4i& c) {
    return fmaf((float)(c[2] - 64 * c[3]), 65536.0f, fmaf((float)c[1], 256.0f, (float)c[0]));
}

// MB: blocks of four rows.  Q: column tiles of 16.  S: steps of 64 k per unit.  G: groups per 128 k that a fold tells apart, 1, 2 or 4 (a group
// of 32: the halves of a step are multiplied with the other half's digits zeroed).  U: units in flight.  The last unit may reach beyond K.
//
// The conversion is a rolled loop over the units: unrolled, a launch waited longer for its instructions than for its data.
template <int MB, int Q, int G, W4mIn IN, int S, int U>
__global__ __launch_bounds__(kW4mThreads) void w4_gemv_mfma_kernel(W4mArgs a) {
    constexpr int kFolds = S * G / 2;                              // per unit
    constexpr bool kGather = IN == kW4mPerm;
    constexpr int kSrc = IN == kW4mGlu ? 2 : 1;                    // words per activation that wait in LDS
    constexpr int kPart = S * 256;                                 // 4-byte words of one (unit, block of rows)
    extern __shared__ __attribute__((aligned(16))) uint32_t w4m_lds[];
    // [wave][unit][rows' block][source][step][quad][16], the digits in the place of the activations; then the staged rows of an act-order call
    __shared__ float back_of[kW4mWaves][U * MB][4];                // 2^-e per row
    __shared__ float red[kW4mWaves][MB * Q][64];
    __shared__ float squares[IN == kW4mNorm ? kW4mWaves * MB * 4 : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c16 = lane & 15, kb = lane >> 4, d = lane & 3, r4 = c16 >> 2;
    const uint32_t word_rows = a.padded_k / 8, num_groups = a.padded_k / a.group_size;
    const uint32_t units = (a.padded_k + 64 * S - 1) / (64 * S);
    const uint32_t tile = xcd_contiguous(blockIdx.x, (a.n + 16 * Q - 1) / (16 * Q));
    // All arrays are read as buffers: an offset per lane that stays, and zeros where it lies beyond the end.  (gfx9 descriptor: no
    // swizzle, raw 32-bit data.)  A scalar offset is no part of that check, so what a step of K adds is taken off the buffer
    // itself; of one past the end nothing is left.  Per lane: where its column starts (a column past n: that of the last).
    const auto array = [](const void* p, uint32_t bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
    };
    const auto beyond = [&](const void* p, uint32_t bytes, uint32_t from) __attribute__((always_inline)) {
        from = min(from, bytes);
        return array(static_cast<const uint8_t*>(p) + from, bytes - from);
    };
    const uint32_t row_bytes = a.n * 4, word_row = a.tiled ? 64 : row_bytes, zp_row = a.zp4 ? word_row / 8 : word_row;
    const uint32_t packed_bytes = word_rows * row_bytes;
    const auto b_scales = array(a.scales, num_groups * row_bytes), b_zps = array(a.zps, num_groups * (a.zp4 ? row_bytes / 8 : row_bytes));
    uint32_t words_at[Q], meta_at[Q], zp_at[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const uint32_t col = min((tile * Q + q) * 16 + c16, a.n - 1);
        words_at[q] = (a.tiled ? (col >> 4) * word_rows * 64 + (col & 15) * 4 : col * 4) + 2 * kb * word_row;
        meta_at[q] = a.tiled ? (col >> 4) * num_groups * 64 + (col & 15) * 4 : col * 4;
        zp_at[q] = a.zp4 ? (a.tiled ? (col >> 4) * num_groups * 8 + ((col & 15) >> 3) * 4 : (col >> 3) * 4) : meta_at[q];
    }
    const uint32_t row_of[2] = {min(r4, a.m - 1), min(r4 + 4, a.m - 1)};
    uint32_t* const mine = w4m_lds + wave * (U * MB * kSrc * kPart);
    // A quad's sixteen k in LDS: first the activations, the even and the odd k of the two packed words in turn; then their digits, digit after
    // digit, turned by the quad's number so that the four writes of a wave fall on all banks.  At `lane * 4` a lane reads the four
    // activations that it converts, at `digit_at` the operand of the digit that it multiplies.
    const uint32_t quad = lane >> 2, digit_at = quad * 16 + ((d + kb) & 3) * 4;
    uint32_t digit_to[4];
#pragma unroll
    for (int i = 0; i < 4; i++) digit_to[i] = quad * 16 + ((i + kb) & 3) * 4 + d;
    const uint32_t even_at = quad * 16 + (d >> 1) * 8 + (d & 1) * 2, k_of = kb * 16 + (d >> 1) * 8 + (d & 1);   // k of a step: k_of + 0, 2, 4, 6
    const uint32_t k_in = kb * 16 + 4 * d;                         // what a lane reads of a step: k_in + 0, 1, 2, 3
    constexpr uint32_t kBytes = IN == kW4mHalf ? 2 : 4;
    const uint32_t x_bytes = a.m * (kSrc * a.k) * kBytes;
    const uint32_t x_at[2] = {(row_of[0] * (kSrc * a.k) + k_in) * kBytes, (row_of[1] * (kSrc * a.k) + k_in) * kBytes};
    float* const staged = reinterpret_cast<float*>(w4m_lds + kW4mWaves * U * MB * kSrc * kPart);

    if constexpr (kGather) {                  // (k % 32 == 0, 16-byte aligned rows)
        const uint32_t count = a.m * (a.k / 4);
        const float4* const src = static_cast<const float4*>(a.x);
        for (uint32_t i0 = tid; i0 < count; i0 += 8 * kW4mThreads) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = src[min(i0 + u * kW4mThreads, count - 1)];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (i0 + u * kW4mThreads < count) reinterpret_cast<float4*>(staged)[i0 + u * kW4mThreads] = v[u];
        }
        __syncthreads();
    }

    float acc[MB][Q];
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
        for (int q = 0; q < Q; q++) acc[b][q] = 0.0f;
    float ssq[MB] = {};

    // element kk of a row, as the kernel multiplies it (rare path and kW4mAny: one by one)
    auto element = [&](uint32_t row, uint32_t kk) __attribute__((always_inline)) {
        const uint32_t at = min(kk, a.k - 1);
        float v;
        if constexpr (IN == kW4mHalf) v = (float)static_cast<const _Float16*>(a.x)[(uint64_t)row * a.k + at];
        else if constexpr (IN == kW4mGlu) {
            const float* const x = static_cast<const float*>(a.x) + (uint64_t)row * 2 * a.k;
            v = w4m_silu(x[at], x[a.k + at]);
        } else {
            v = static_cast<const float*>(a.x)[(uint64_t)row * a.k + ((IN == kW4mPerm || IN == kW4mAny) && a.perm ? (uint32_t)a.perm[at] : at)];
            if constexpr (IN == kW4mNorm) v *= a.norm_w[at];
        }
        return kk < a.k ? v : 0.0f;
    };
    // the scaling of a unit of one row from its lanes' largest bits: 2^e and its reciprocal (NaN for a row with an infinity or a NaN)
    auto scaling = [&](uint32_t top, float& f, float& back) __attribute__((always_inline)) {
        top = max(top, (uint32_t)W4M_DPP(top, 0xB1));              // over the lanes of the row: the quad, then the four of k
        top = max(top, (uint32_t)W4M_DPP(top, 0x4E));
        const auto r = __builtin_amdgcn_permlane16_swap(top, top, false, false);
        top = max(r[0], r[1]);
        const auto h = __builtin_amdgcn_permlane32_swap(top, top, false, false);
        top = max(h[0], h[1]);
        // 2^(21 - E) for a largest magnitude in [2^E, 2^(E+1)), half of that from 2^(E+1) (1 - 2^-6) on: |X| stays below 2^22 - 2^16, and byte 2
        // of what w4m_digits adds up below 128.  At most 2^126, its reciprocal is a normal number then.
        const uint32_t bits = min((275u << 23) - ((top + (1u << 18)) & 0x7f800000u), 253u << 23);
        f = __uint_as_float(bits);
        back = top >= 0x7f800000u ? __uint_as_float(0x7fc00000u) : __uint_as_float((254u << 23) - bits);
        return top;
    };
    auto towering = [](uint32_t top, uint32_t least_1) __attribute__((always_inline)) {
        return top - (8u << 23) < (255u << 23) - (8u << 23) && least_1 < top - (8u << 23);
    };
    auto any_of_row = [](uint32_t any) __attribute__((always_inline)) {
        any |= (uint32_t)W4M_DPP(any, 0xB1);
        any |= (uint32_t)W4M_DPP(any, 0x4E);
        any |= (uint32_t)__shfl_xor((int)any, 16);
        return any | (uint32_t)__shfl_xor((int)any, 32);
    };
    auto widen = [&](uint32_t w0, uint32_t w1) __attribute__((always_inline)) {
        return v4i{(int)(w0 & 0x0f0f0f0fu), (int)((w0 >> 4) & 0x0f0f0f0fu), (int)(w1 & 0x0f0f0f0fu), (int)((w1 >> 4) & 0x0f0f0f0fu)};
    };
    // one unit's digits A with its weights, into `to`.  EXACT: the zero-point's nearest integer is taken off the sums as integers, so that an
    // element as large as it likes leaves nothing behind where its weight is zero.
    auto multiply = [&](auto EXACT, const v4i (&A)[S], const uint32_t (&w)[S][2][Q], const float (&sc)[kFolds][Q], const uint32_t (&zw)[kFolds][Q], float back,
                        float (&to)[Q]) __attribute__((always_inline)) {
        const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int p = 0; p < kFolds; p++) {
            constexpr int kSteps = G == 1 ? 2 : 1;
            v4i part[kSteps];
#pragma unroll
            for (int s = 0; s < kSteps; s++)
#pragma unroll
                for (int i = 0; i < 4; i++) part[s][i] = G == 4 && (kb >> 1) != (uint32_t)(p & 1) ? 0 : A[G == 1 ? 2 * p + s : p * 2 / G][i];
            v4i sx = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < kSteps; s++) sx = __builtin_amdgcn_mfma_i32_16x16x64_i8(part[s], ones, sx, 0, 0, 0);
            const float sum = w4m_sum(sx);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                v4i sq = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < kSteps; s++) {
                    const int at = G == 1 ? 2 * p + s : p * 2 / G;
                    sq = __builtin_amdgcn_mfma_i32_16x16x64_i8(part[s], widen(w[at][0][q], w[at][1][q]), sq, 0, 0, 0);
                }
                const float z = a.zp4 ? (float)((zw[p][q] >> (4 * (c16 & 7))) & 15u) : __uint_as_float(zw[p][q]);
                float rest = z;
                if constexpr (EXACT.value) {
                    const float whole = fabsf(z) < 1024.0f ? rintf(z) : 0.0f;
                    rest = z - whole;
#pragma unroll
                    for (int i = 0; i < 4; i++) sq[i] -= (int)whole * sx[i];
                }
                to[q] = fmaf(fmaf(-rest, sum, EXACT.value ? w4m_wide_sum(sq) : w4m_sum(sq)) * sc[p][q], back, to[q]);
            }
        }
    };
    auto load_weights = [&](uint32_t c, uint32_t (&w)[S][2][Q], float (&sc)[kFolds][Q], uint32_t (&z)[kFolds][Q]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            const uint32_t step = c * S + s;               // (word rows come in fours: a lane's second is there if its first is)
            const auto b_packed = beyond(a.packed, packed_bytes, step * 64 < a.padded_k ? step * 8 * word_row : packed_bytes);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int q = 0; q < Q; q++)
                    w[s][i][q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_packed, (int)words_at[q], (int)(i * word_row), 0);
        }
#pragma unroll
        for (int p = 0; p < kFolds; p++) {
            const uint32_t k32 = c * (2 * S) + p * (4 / G);
            const uint32_t g = min(__umulhi(2 * k32, a.per_group), num_groups - 1);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                sc[p][q] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_scales, (int)meta_at[q], (int)(g * word_row), 0));
                z[p][q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b_zps, (int)zp_at[q], (int)(g * zp_row), 0);
            }
        }
    };

    for (uint32_t base = 0; base < units; base += kW4mWaves * U) {
        const uint32_t c0 = base + wave;                           // and every eighth after it: the same units whatever U
        // ---- loads of U units: activations first (their digits are made while the weights are on their way)
        v4i raw[U][S][MB][kSrc], nw[IN == kW4mNorm ? U : 1][S];
        uint32_t word[U][S][2][Q], zp[U][kFolds][Q];
        float scale[U][kFolds][Q];
        if (base == 0) __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int s = 0; s < S; s++) {
                const uint32_t step = ((c0 + kW4mWaves * u) * S + s) * 64, in_row = min(step, a.k);   // (a row's end: the next one's start, or the end)
                const auto b_x = beyond(a.x, x_bytes, step < a.k ? step * kBytes : x_bytes);
#pragma unroll
                for (int b = 0; b < MB; b++) {
                    v4i& v = raw[u][s][b][0];
                    if constexpr (kGather) {
                        if (b == 0) v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(beyond(a.perm, a.k * 4, in_row * 4), (int)(k_in * 4), 0, 0));
                    } else if constexpr (IN == kW4mHalf) {
                        const v4h f = __builtin_bit_cast(v4h, __builtin_amdgcn_raw_buffer_load_b64(b_x, (int)x_at[b], 0, 0));
                        v = v4i{__float_as_int((float)f[0]), __float_as_int((float)f[1]), __float_as_int((float)f[2]), __float_as_int((float)f[3])};
                    } else if constexpr (IN == kW4mAny) {
                        const uint32_t k0 = step + k_in;
                        v = v4i{__float_as_int(element(row_of[b], k0)), __float_as_int(element(row_of[b], k0 + 1)),
                                __float_as_int(element(row_of[b], k0 + 2)), __float_as_int(element(row_of[b], k0 + 3))};
                    } else {                                       // (k % 4 == 0)
                        v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(b_x, (int)x_at[b], 0, 0));
                        if constexpr (IN == kW4mGlu)
                            raw[u][s][b][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                beyond(a.x, x_bytes, step < a.k ? (step + a.k) * 4 : x_bytes), (int)x_at[b], 0, 0));
                    }
                }
                if constexpr (IN == kW4mNorm)
                    nw[u][s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(beyond(a.norm_w, a.k * 4, in_row * 4), (int)(k_in * 4), 0, 0));
            }
        if (base == 0) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < U; u++) load_weights(c0 + kW4mWaves * u, word[u], scale[u], zp[u]);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int b = 0; b < MB; b++)
#pragma unroll
                for (int s = 0; s < S; s++)
#pragma unroll
                    for (int i = 0; i < kSrc; i++) {
                        if (kGather && b) continue;
                        v4i v = raw[u][s][b][i];
                        if constexpr (IN == kW4mNorm) {
                            const bool in = ((c0 + kW4mWaves * u) * S + s) * 64 + k_in < a.k;
#pragma unroll
                            for (int j = 0; j < 4; j++) {
                                const float f = __int_as_float(v[j]);
                                ssq[b] = in ? fmaf(f, f, ssq[b]) : ssq[b];
                                v[j] = __float_as_int(f * __int_as_float(nw[u][s][j]));
                            }
                        }
                        uint32_t* const to = mine + ((u * MB + b) * kSrc + i) * kPart + s * 256 + even_at;
                        *reinterpret_cast<v2i*>(to) = v2i{v[0], v[2]};
                        *reinterpret_cast<v2i*>(to + 4) = v2i{v[1], v[3]};
                    }

        // ---- digits, in the place of the activations
        const uint32_t live = c0 < units ? min((uint32_t)U, (units - c0 + kW4mWaves - 1) / kW4mWaves) : 0;
        if (lane < U * MB * 4) back_of[wave][0][lane] = 0.0f;      // (a unit that is not there adds nothing)
        uint32_t deep = 0;                                         // bit per (unit, block) with towering elements
#pragma unroll 1
        for (uint32_t i = 0; i < live * MB; i++) {
            const uint32_t u = i / MB, b = i % MB;
            uint32_t* const at = mine + i * (kSrc * kPart);
            float t[S][4];
            uint32_t top = 0, least = 0xffffffffu;                 // on the bit patterns without their sign
#pragma unroll
            for (int s = 0; s < S; s++) {
                const v4i v = *reinterpret_cast<const v4i*>((kGather ? mine + u * MB * kPart : at) + s * 256 + lane * 4);
                if constexpr (kGather) {
                    const float* const row = staged + (b ? row_of[1] : row_of[0]) * a.k;
#pragma unroll
                    for (int j = 0; j < 4; j++) t[s][j] = row[(uint32_t)v[j]];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) t[s][j] = __int_as_float(v[j]);
                }
                if constexpr (IN == kW4mGlu) {
                    const v4i up = *reinterpret_cast<const v4i*>(at + kPart + s * 256 + lane * 4);
#pragma unroll
                    for (int j = 0; j < 4; j++) t[s][j] = w4m_silu(t[s][j], __int_as_float(up[j]));
                }
            }
            if ((c0 + kW4mWaves * u + 1) * (64 * S) > a.k) {
#pragma unroll
                for (int s = 0; s < S; s++)
#pragma unroll
                    for (int j = 0; j < 4; j++) t[s][j] = ((c0 + kW4mWaves * u) * S + s) * 64 + k_of + 2 * j < a.k ? t[s][j] : 0.0f;
            }
#pragma unroll
            for (int s = 0; s < S; s++) top = max(top, w4m_largest(t[s]));
            least = top - 1u;                                      // (a lane of zeros, as beyond k, has nothing to lose)
            float f, back;
            top = scaling(top, f, back);
            if (__builtin_expect(__any(towering(top, least)), 0)) {
                deep |= 1u << i;
                back = any_of_row(towering(top, least)) ? 0.0f : back;     // (all of such a row is multiplied below)
            }
            if (kb == 0 && d == 0) back_of[wave][i][r4] = back;
            // (act-order: the last block of rows takes the place of the unit's indices)
#pragma unroll
            for (int s = 0; s < S; s++) {
                const v4i T = w4m_digits(t[s], f);
                uint32_t* const to = (kGather ? mine + (u * MB + MB - 1 - b) * kPart : at) + s * 256;
#pragma unroll
                for (int j = 0; j < 4; j++) to[digit_to[j]] = (uint32_t)T[j];
            }
        }
        // ---- unit by unit
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int b = 0; b < MB; b++) {
                v4i A[S];
#pragma unroll
                for (int s = 0; s < S; s++)
                    A[s] = *reinterpret_cast<const v4i*>(mine + (kGather ? (u * MB + MB - 1 - b) * kPart : (u * MB + b) * kSrc * kPart) + s * 256 + digit_at);
                multiply(std::false_type{}, A, word[u], scale[u], zp[u], back_of[wave][u * MB + b][kb], acc[b]);
            }
        // ---- rows with towering elements: digits, and of what they leave, scaled by 2^22, digits again until nothing is left (exact)
        if (__builtin_expect(deep != 0, 0)) {
#pragma unroll 1
            for (uint32_t i = 0; i < live * MB; i++) {
                if (!((deep >> i) & 1)) continue;
                const uint32_t c = c0 + kW4mWaves * (i / MB), b = i % MB, row = b ? row_of[1] : row_of[0];
                uint32_t w[S][2][Q], z[kFolds][Q];
                float sc[kFolds][Q];
                load_weights(c, w, sc, z);
                float rest[S][4], f, back;
                uint32_t top = 0;
#pragma unroll
                for (int s = 0; s < S; s++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) rest[s][j] = element(row, (c * S + s) * 64 + k_of + 2 * j);
                    top = max(top, w4m_largest(rest[s]));
                }
                const uint32_t least = top - 1u;
                top = scaling(top, f, back);
                const bool whole = any_of_row(towering(top, least)) != 0;
#pragma unroll
                for (int s = 0; s < S; s++)
#pragma unroll
                    for (int j = 0; j < 4; j++) rest[s][j] = whole ? rest[s][j] : 0.0f;
                // the accumulators' row is lane >> 4: what belongs to that row sits in lanes 4 (lane >> 4) of the first sixteen
                float unit = __uint_as_float(__builtin_amdgcn_ds_bpermute((int)(16 * kb), (int)__float_as_uint(back))), sum[Q] = {};
#pragma unroll 1
                for (int pass = 0; pass < 14; pass++) {
                    bool more = false;
                    v4i A[S];
#pragma unroll
                    for (int s = 0; s < S; s++) {
                        const v4i T = w4m_digits(rest[s], f);
                        uint32_t* const to = mine + s * 256;       // (every unit's digits have been multiplied)
#pragma unroll
                        for (int j = 0; j < 4; j++) to[digit_to[j]] = (uint32_t)T[j];
                        A[s] = *reinterpret_cast<const v4i*>(to + digit_at);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float v = rest[s][j] * f;
                            rest[s][j] = v - rintf(v);
                            more = more || rest[s][j] != 0.0f;
                        }
                    }
                    multiply(std::true_type{}, A, w, sc, z, unit, sum);
                    if (!__any(more)) break;
                    f = 0x1p22f;
                    unit *= 0x1p-22f;
                }
#pragma unroll
                for (int bb = 0; bb < MB; bb++)
#pragma unroll
                    for (int q = 0; q < Q; q++) acc[bb][q] += (uint32_t)bb == b ? sum[q] : 0.0f;
            }
        }
    }

    // ---- the waves' shares of K
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
        for (int q = 0; q < Q; q++) red[wave][b * Q + q][lane] = acc[b][q];
    if constexpr (IN == kW4mNorm) {
#pragma unroll
        for (int b = 0; b < MB; b++) {
            float v = ssq[b];
            v += __uint_as_float(W4M_DPP(__float_as_uint(v), 0xB1));
            v += __uint_as_float(W4M_DPP(__float_as_uint(v), 0x4E));
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (kb == 0 && d == 0) squares[(wave * MB + b) * 4 + r4] = v;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < MB * Q * 64; i += kW4mThreads) {
        const uint32_t j = i >> 6, b = j / Q, q = j % Q, row = b * 4 + (i & 63) / 16, oc = (tile * Q + q) * 16 + (i & 15);
        if (row >= a.m || oc >= a.n) continue;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kW4mWaves; w++) v += red[w][j][i & 63];
        if constexpr (IN == kW4mNorm) {
            float q2 = 0.0f;
#pragma unroll
            for (int w = 0; w < kW4mWaves; w++) q2 += squares[(w * MB + b) * 4 + (row & 3)];
            v *= rsqrtf(q2 / (float)a.k + a.eps);
        }
        if (a.bias) v += a.bias[oc];
        if (a.resid) v += a.resid[(uint64_t)row * a.n + oc];
        if constexpr (IN == kW4mHalf) static_cast<_Float16*>(a.y)[(uint64_t)row * a.n + oc] = (_Float16)v;
        else static_cast<float*>(a.y)[(uint64_t)row * a.n + oc] = v;
    }
}

template <auto KERNEL>
static int w4m_queue(dim3 grid, dim3 block, size_t lds, const W4mArgs& a, hipStream_t s) {
    static std::atomic<bool> allowed{false};
    if (lds > 64 * 1024 && !allowed.load(std::memory_order_relaxed)) {
        if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kW4mLds),
                               "hipFuncSetAttribute")) return rc;
        allowed.store(true, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL(KERNEL, grid, block, lds, s, a);
    return RUMUS_HIP_OK;
}
template <int MB, int Q, W4mIn IN, int S, int U>
static int w4m_launch(const W4mArgs& a, hipStream_t s) {
    const dim3 grid(ceil_div(a.n, 16 * Q)), block(kW4mThreads);
    const size_t lds = (size_t)kW4mWaves * U * MB * (IN == kW4mGlu ? 2 : 1) * S * 1024 + (IN == kW4mPerm ? (size_t)a.m * a.k * sizeof(float) : 0);
    if (a.group_size % 128 == 0) return w4m_queue<&w4_gemv_mfma_kernel<MB, Q, 1, IN, S, U>>(grid, block, lds, a, s);
    if (a.group_size % 64 == 0) return w4m_queue<&w4_gemv_mfma_kernel<MB, Q, 2, IN, S, U>>(grid, block, lds, a, s);
    if constexpr (U == 1) return w4m_queue<&w4_gemv_mfma_kernel<MB, Q, 4, IN, S, U>>(grid, block, lds, a, s);
    return set_error(RUMUS_HIP_EINVAL, "w4 gemv: groups of 32 take one unit at a time");
}
// Of one launch's LDS: digits of the units in flight, and an act-order call's rows.
static size_t w4m_gather_lds(uint32_t m, uint32_t k, uint32_t flight) {
    return (size_t)kW4mWaves * flight * (m > 4 ? 2 : 1) * 4096 + (size_t)m * k * sizeof(float);
}
// Two units in flight for up to four rows where the eight waves have more than that and the rows of an act-order call leave room for both.  Not for
// eight rows, whose digits of two units are 128 KB, one workgroup a compute unit, nor for groups of 32, whose folds take the registers (us with two
// and one: 8 x 4096 x 5632 12.7 and 10.1, 8 x 5120 x 5120 18.1 and 12.2, 8 x 4096 x 22016 24.7 and 21.6; groups of 32, 3 x 4096 x 12288 16.2 and 14.1, 5 x
// 4096 x 12288 through RMSNorm 28.7 and 22.3).
// Units of 128 k where 256 would leave waves without one, and for groups of 32 where there are more workgroups than compute units: half the registers
// let two share one (3 x 4096 x 12288 14.1 -> 12.0, 5 x 4096 x 5632 15.8 -> 13.9, 8 x 5120 x 5120 20.5 -> 16.6; but 3 x 4096 x 8192, 256 of them, 8.3 -> 9.1).
// The rows of an act-order call hold the LDS of a compute unit anyway.  None of it depends on the number of rows but the units in flight, which
// leave a wave its units in their order: a row's bits are the same in calls of three to eight.
template <int MB, int Q, W4mIn IN>
static int w4m_sweep(const W4mArgs& a, hipStream_t s) {
    const uint32_t units = ceil_div(a.padded_k, 256), columns = a.n >= 8192 ? 32 : 16;     // of a workgroup (w4m_pick)
    const bool shared = IN != kW4mPerm && a.group_size % 64 != 0 && ceil_div(a.n, columns) > 256;
    if (2 * units <= kW4mWaves || shared) return w4m_launch<MB, Q, IN, 2, 1>(a, s);
    if constexpr (MB == 1) {
        if (a.group_size % 64 == 0 && units > kW4mWaves && (IN != kW4mPerm || w4m_gather_lds(a.m, a.k, 2) <= kW4mLds)) return w4m_launch<MB, Q, IN, 4, 2>(a, s);
    }
    return w4m_launch<MB, Q, IN, 4, 1>(a, s);
}
// (f16 rows come with row-major arrays: pieces of 128 bytes only where the rows of all columns begin on the same memory channels, us with 16 and 32
// columns 4 x 4096 x 8192 9.0 and 7.8, 4 x 8192 x 8192 14.4 and 12.3, but 4 x 4096 x 11008 11.1 and 12.1)
template <W4mIn IN>
static int w4m_pick(const W4mArgs& a, hipStream_t s) {
    constexpr bool kWide = IN == kW4mVec || IN == kW4mHalf || IN == kW4mNorm || IN == kW4mGlu;
    if constexpr (kWide) {
        if (a.n >= 8192 && (IN != kW4mHalf || a.n % 2048 == 0)) return a.m <= 4 ? w4m_sweep<1, 2, IN>(a, s) : w4m_sweep<2, 2, IN>(a, s);
    }
    return a.m <= 4 ? w4m_sweep<1, 1, IN>(a, s) : w4m_sweep<2, 1, IN>(a, s);
}

// Arrays that 32-bit offsets reach, and group numbers from a product: x / by = mulhi(x, ceil(2^32 / by)) while x by < 2^32.
bool w4_gemv_mfma_reaches(const W4Args& a) {
    const uint64_t by = a.group_size / 16, most = a.padded_k / 16 + 256;
    return ((uint64_t)a.padded_k + 4096) * (a.n + 64) / 2 < (uint64_t(1) << 31) && (uint64_t)a.num_groups * a.n < (uint64_t(1) << 29) &&
           ((uint64_t)a.k + 4096) * a.m < (uint64_t(1) << 28) && most * by < (uint64_t(1) << 32);
}

// 2 to 8 rows, group_size % 32 == 0, no g_idx: y = f(x) . dequant(W) + bias + resid, f = RMSNorm with `norm_w`, SwiGLU (a.glu) or nothing
// (the caller has checked: k % 4 == 0, 16-byte aligned x and norm_w, no perm for those two).
int w4_launch_gemv_mfma(const W4Args& a, const float* norm_w, float eps, const float* resid, hipStream_t s) {
    const W4mArgs b{a.packed, a.scales, a.zp4 ? a.zp4 : reinterpret_cast<const uint32_t*>(a.zp), a.x16 ? static_cast<const void*>(a.x16) : a.x,
                    a.y16 ? static_cast<void*>(a.y16) : a.y, a.bias, a.perm, norm_w, resid, a.m, a.k, a.n, a.padded_k, a.group_size, eps,
                    (uint32_t)(((uint64_t(1) << 32) + a.group_size / 16 - 1) / (a.group_size / 16)), a.zp4 != nullptr, a.tiled};
    const bool rows = a.k % 4 == 0 && (reinterpret_cast<uintptr_t>(b.x) & 15) == 0;
    if (a.glu && !(rows && a.tiled && !a.zp4))
        return set_error(RUMUS_HIP_EINVAL, "w4 gemv: the SwiGLU input needs the decode layout, f32 zero-points, "
                                           "k %% 8 == 0 and 16-byte aligned rows");
    // act-order rows are gathered from LDS; where all of them do not fit beside the digits, fewer at a time
    uint32_t part = a.m;
    if (a.perm && rows && (reinterpret_cast<uintptr_t>(a.perm) & 15) == 0) {
        auto fits = [&](uint32_t m) { return w4m_gather_lds(m, a.k, 1) <= kW4mLds; };
        if (!fits(part)) part = fits(4) ? 4 : fits(2) ? 2 : fits(1) ? 1 : 0;
    } else if (a.perm) {
        part = 0;
    }
    int rc = RUMUS_HIP_OK;
    if (a.x16) rc = w4m_pick<kW4mHalf>(b, s);
    else if (a.glu) rc = w4m_pick<kW4mGlu>(b, s);
    else if (norm_w) rc = w4m_pick<kW4mNorm>(b, s);
    else if (!a.perm && rows) rc = w4m_pick<kW4mVec>(b, s);
    else if (!a.perm || part == 0) rc = w4m_pick<kW4mAny>(b, s);
    else
        for (uint32_t r0 = 0; r0 < a.m && rc == RUMUS_HIP_OK; r0 += part) {
            W4mArgs c = b;
            c.m = min(part, a.m - r0);
            c.x = a.x + (uint64_t)r0 * a.k;
            c.y = a.y + (uint64_t)r0 * a.n;
            rc = w4m_pick<kW4mPerm>(c, s);
        }
    return rc ? rc : check_launch("w4_gemv_mfma_kernel");
}

}  // namespace rumus
