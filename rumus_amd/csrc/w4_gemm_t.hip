// grad_x of the INT4 Linear for batches, on the f16 matrix cores:
//   out[m, k] = sum_n gy[m, n] * (q[k, n] - zp[g, n]) * s[g, n],   g = k / group_size
// (custom_forward(&QMatMulINT4TransposeOp, ..) quant.rs:262-317; qmatmul_int4_transpose.wgsl:37-74
// computes the same sums one output per thread with n as the serial loop).
//
// The sum runs over n, and scale and zero-point change with n, so they cannot be taken out of the
// sum the way the forward kernel takes them out per group.  They can be moved to the other operand:
//   out[m, k] = sum_n A_g[m, n] * (q[k, n] - z0[g, n])  -  c[m, g],
//   A_g[m, n] = gy[m, n] s[g, n],   z0 = rint(zp),   c[m, g] = sum_n A_g[m, n] (zp[g, n] - z0[g, n])
// so the matrix cores multiply small integers (exact in f16) with activations that are re-scaled once
// per group of output columns.  (Taking the whole zero-point out, q against c = sum A zp, costs
// accuracy: the 2^-23 the f16 planes lose of A is then multiplied by q instead of by q - zp, which
// near-zero weights make many times larger than the term itself.)  A workgroup owns 64 rows x 128 consecutive k of one
// group (group_size % 128 == 0; 64 or 32 k for groups of 64 or 32) and walks n in steps of 32:
//   * conversion (all 256 threads, 8 values each): a = (gy f_row) (s / S) with f_row and S powers of two
//     that put |a| below 2^14 (w4t_prepare_kernel: row maxima of gy, maximum of the scales), split into
//     hi + lo f16 (22 bits), written to LDS in A-fragment rows of 64 bytes; c accumulates in f32;
//   * every wave owns 32 of the 128 k: lane (k = lane % 32, half = lane / 32) reads the 8 consecutive
//     words of word row k / 8 that hold its 8 values of n, takes nibble k % 8 of each, and splices them
//     under the mantissa of 1024 (minus 1024, two at a time): 16 instructions per B fragment, which
//     serves 4 MFMAs (two row tiles x hi, lo);
//   * v_mfma_f32_32x32x16_f16 accumulates in f32; the epilogue subtracts c and undoes f_row and S.
// Few tiles: n is shared out over blockIdx.z as well and the partial results are added in a fixed order.
#include "common.h"
#include "i8_gemm.h"

#include <algorithm>
#include <type_traits>

namespace rumus {

typedef _Float16 t8h __attribute__((ext_vector_type(8)));
typedef _Float16 t2h __attribute__((ext_vector_type(2)));
typedef float t16f __attribute__((ext_vector_type(16)));

constexpr int kTMaxSplits = 16;

// Per call, before the GEMM:
//   blocks [0, m): f_row = 2^(140 - e) for a row maximum a 2^(e - 127), 1 <= a < 2, so |gy f| < 2^14
//       (0 for an all-zero or tiny row, NaN marker for a row with inf / nan);
//   blocks [m, m + groups): for group g, S_g = the power of two at or above its largest scale, and per
//       column the three things the GEMM needs of scale and zero-point: s / S_g (f32, at most 1),
//       zp - z0 (f32) and 1024 + z0 (f16), z0 = rint(zp) held within +-1000, so that no workgroup works
//       them out again.
//       sgrp[g] = S_g; 0 when every scale of the group is zero or denormal, NaN when one is not finite
//       or S_g or 1 / S_g would leave the normal range: the GEMM then writes zeros / NaNs for the group.
// BLOCKS: the three lie together, 16 columns at a time (w4t_wide_kernel, n % 16 == 0): 16 s / S_g, 16 products of that with zp - z0,
// 16 times 1024 + z0, kTBlock bytes in sp; zf and zo are not used.
constexpr uint32_t kTBlock = 160;
template <bool BLOCKS>
__global__ __launch_bounds__(256) void w4t_prepare_kernel(const float* __restrict__ gy, const float* __restrict__ scales,
                                                          const float* __restrict__ zp, float* __restrict__ rowf,
                                                          float* __restrict__ sgrp, float* __restrict__ sp,
                                                          float* __restrict__ zf, _Float16* __restrict__ zo,
                                                          uint32_t m, uint32_t n) {
    __shared__ uint32_t red[4];
    const uint32_t tid = threadIdx.x;
    const bool is_row = blockIdx.x < m;
    const float* r = is_row ? gy + (uint64_t)blockIdx.x * n : scales + (uint64_t)(blockIdx.x - m) * n;   // n % 4 == 0, aligned
    // The first kPrepCache steps of a thread (n up to 12288) stay in registers between the pass that finds the maximum
    // and the pass that writes the tables, and the zero-points are asked for together with them: one trip to memory
    // instead of one per four steps and pass.
    constexpr int kPrepCache = 12;
    const uint32_t g = is_row ? 0 : blockIdx.x - m;
    const float* zr = zp + (uint64_t)g * n;
    float4 cs[kPrepCache], cz[kPrepCache];
#pragma unroll
    for (int i = 0; i < kPrepCache; i++) {
        const uint32_t j = min(4 * tid + 1024 * i, n - 4);      // clamped: no load under a branch
        cs[i] = *reinterpret_cast<const float4*>(r + j);
        cz[i] = *reinterpret_cast<const float4*>(zr + j);       // a row's workgroup reads group 0's and drops them
    }
    auto max4 = [](uint32_t a, const float4& t) {
        return max(max(a, max(__float_as_uint(t.x) & 0x7FFFFFFFu, __float_as_uint(t.y) & 0x7FFFFFFFu)),
                   max(__float_as_uint(t.z) & 0x7FFFFFFFu, __float_as_uint(t.w) & 0x7FFFFFFFu));
    };
    uint32_t amax = 0;
#pragma unroll
    for (int i = 0; i < kPrepCache; i++)
        if (4 * tid + 1024 * i < n) amax = max4(amax, cs[i]);
#pragma unroll 4
    for (uint32_t j = 4 * tid + 1024 * kPrepCache; j < n; j += 1024) amax = max4(amax, *reinterpret_cast<const float4*>(r + j));
    amax = wave_max(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = max(max(red[0], red[1]), max(red[2], red[3]));
    if (is_row) {
        const uint32_t e = amax >> 23;
        if (tid == 0)
            rowf[blockIdx.x] = e >= 255 ? __uint_as_float(0x7FC00000u) : e < 14 ? 0.0f : __uint_as_float((267u - e) << 23);
        return;
    }
    const uint32_t se = (amax >> 23) + ((amax & 0x7FFFFFu) ? 1u : 0u);      // S_g = 2^(se - 127)
    const bool ok = se >= 1 && se <= 253;                      // S_g and 1 / S_g are normal floats
    const float s_inv = ok ? __uint_as_float((254u - se) << 23) : 0.0f;
    if (tid == 0) sgrp[g] = ok ? __uint_as_float(se << 23) : (amax >= 0x7F000000u ? __uint_as_float(0x7FC00000u) : 0.0f);
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    auto emit = [&](uint32_t j, const float4& sv, const float4& z) {
        // zero-points are 0 .. 15 unless a group's weights sit far from zero (zp = -min / scale); beyond
        // +-1000 the integer part stops growing and the rest goes into the f32 correction with the fraction
        auto whole = [](float v) { return fminf(fmaxf(rintf(v), -1000.0f), 1000.0f); };
        const float4 z0 = make_float4(whole(z.x), whole(z.y), whole(z.z), whole(z.w));
        // s / S_g is exact (a power of two); 1024 + z0 is exact in f16 for |z0| <= 1024
        if constexpr (BLOCKS) {
            uint8_t* const at = reinterpret_cast<uint8_t*>(sp) + ((uint64_t)g * (n / 16) + j / 16) * kTBlock;
            const float4 sc = make_float4(sv.x * s_inv, sv.y * s_inv, sv.z * s_inv, sv.w * s_inv);
            *reinterpret_cast<float4*>(at + j % 16 * 4) = sc;
            *reinterpret_cast<float4*>(at + 64 + j % 16 * 4) = make_float4(sc.x * (z.x - z0.x), sc.y * (z.y - z0.y), sc.z * (z.z - z0.z), sc.w * (z.w - z0.w));
            *reinterpret_cast<v4h*>(at + 128 + j % 16 * 2) =
                v4h{(_Float16)(1024.0f + z0.x), (_Float16)(1024.0f + z0.y), (_Float16)(1024.0f + z0.z), (_Float16)(1024.0f + z0.w)};
            return;
        }
        *reinterpret_cast<float4*>(sp + (uint64_t)g * n + j) = make_float4(sv.x * s_inv, sv.y * s_inv, sv.z * s_inv, sv.w * s_inv);
        *reinterpret_cast<float4*>(zf + (uint64_t)g * n + j) = make_float4(z.x - z0.x, z.y - z0.y, z.z - z0.z, z.w - z0.w);
        *reinterpret_cast<v4h*>(zo + (uint64_t)g * n + j) =
            v4h{(_Float16)(1024.0f + z0.x), (_Float16)(1024.0f + z0.y), (_Float16)(1024.0f + z0.z), (_Float16)(1024.0f + z0.w)};
    };
#pragma unroll
    for (int i = 0; i < kPrepCache; i++)
        if (4 * tid + 1024 * i < n) emit(4 * tid + 1024 * i, cs[i], cz[i]);
#pragma unroll 4
    for (uint32_t j = 4 * tid + 1024 * kPrepCache; j < n; j += 1024)   // independent iterations: their loads overlap
        emit(j, *reinterpret_cast<const float4*>(r + j), *reinterpret_cast<const float4*>(zr + j));
}

// One workgroup: rows [64 y, 64 y + 64), k [128 x, 128 x + 128), n steps [z steps_per, ..).
//
// Operands travel global -> LDS by direct-to-LDS loads, kTStages steps deep: per step the raw tile of
// grad_y (64 rows x 32 floats), the 16 word rows x 32 words of the weights and the group's 32 scaled
// scales, 32 zero-point fractions and 32 f16 zero-point integers, 10.5 KB.  The raw tile of step t+1
// is converted into the A-fragment buffer (double-buffered) while the MFMAs of step t run; one barrier
// per step.
constexpr int kTRawGy = 64 * 128, kTRawW = 16 * 128, kTRawSz = 256, kTRawZo = 256;   // 64 bytes of zero-point integers used
constexpr int kTRawWt = kTRawW + kTRawSz + kTRawZo;           // weights and tables of one step
constexpr int kTAbuf = 2 * 64 * 64;                           // hi, lo planes
constexpr int kTSlots = 12;                                   // wave-wide loads per step: 8 grad_y, 1-2 weights, 2 tables
// The raw tile of grad_y of step t is dead once it has been converted (during step t - 1), the weights and tables of
// step t are read during step t: one slot fewer for grad_y than for the rest, at the same depth of loads in flight.
constexpr size_t w4t_lds_bytes(int stages) {
    return (size_t)(stages - 1) * kTRawGy + (size_t)stages * kTRawWt + 2 * kTAbuf + 2 * 64 * sizeof(float);
}

// Direct-to-LDS loads and the barrier that publishes a step, spelled out.  With the compiler's own loads every LDS read that
// follows waits for all of them (it cannot see that they go to another slot): the two steps meant to be in flight were waited
// for within the step that had asked for them.  The barrier waits for the step it publishes, and for the wave's LDS writes.
// With that, the loop in two scheduled halves and the shorter nibble cut below, same bits (4096 x 11008, whole call): 16 rows
// 31.8 -> 27.8 us, 128 rows 52.3 -> 49.5, 512 rows 150.9 -> 145.4, 1024 rows 316 -> 293, 2048 rows 541 -> 522; groups of 64 and 32 6 %.
// What bounds it now: vector issue (103 instructions per wave and step of 8 MFMAs, four waves per SIMD).
__device__ __forceinline__ uint32_t w4t_lds_offset(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p; }
__device__ __forceinline__ void w4t_load16(uint32_t to, const void* from, uint32_t lane_bytes) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(lane_bytes), "s"(from) : "memory");
}
__device__ __forceinline__ void w4t_load4(uint32_t to, const void* from, uint32_t lane_bytes) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(to), "v"(lane_bytes), "s"(from) : "memory");
}
template <int LOADS>
__device__ __forceinline__ void w4t_publish() {               // all but the youngest LOADS loads of the wave have landed
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
}

// KW = waves per workgroup = 32-column slices of k per tile: 4 when groups are multiples of 128, 2 for
// groups of 64, 1 for groups of 32 (a tile must lie inside one group, since the activations are re-scaled
// per group; the smaller workgroups convert the same 64 x 32 activations for fewer output columns).
// HALF: at most 32 rows (one row tile, half full): the loads, the conversion and the MFMAs of rows 32..63 are
// left out (4096 x 11008 at 16 rows: the call 44.6 -> 40.7 us; groups of 64 at 24 rows 56.1 -> 47.4 us).
template <int kTStages, int KW, bool HALF = false>
__global__ __launch_bounds__(64 * KW, 2) void w4t_gemm_kernel(
    const float* __restrict__ gy, const uint32_t* __restrict__ packed, const float* __restrict__ sp,
    const float* __restrict__ zf, const _Float16* __restrict__ zo, const float* __restrict__ rowf,
    const float* __restrict__ sgrp, float* __restrict__ out, uint32_t m, uint32_t k, uint32_t n, uint32_t gs,
    uint32_t steps_per) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint8_t* const raw_gy = lds;                               // [kTStages - 1][kTRawGy]
    uint8_t* const raw_wt = lds + (kTStages - 1) * kTRawGy;    // [kTStages][kTRawWt]
    uint8_t* const abuf = raw_wt + kTStages * kTRawWt;         // [2][kTAbuf]
    float* const lds_c = reinterpret_cast<float*>(abuf + 2 * kTAbuf);
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kTLoads = (HALF ? kTSlots - 4 : kTSlots) / KW;   // per wave and step
    constexpr int RTILES = HALF ? 1 : 2;                       // 32-row tiles of the accumulators
    constexpr int WS = KW == 4 ? 2 : 1;                        // slots of weight words (8 word rows each)
    const uint32_t k0 = blockIdx.x * (32 * KW), m0 = blockIdx.y * 64;
    const uint32_t g = k0 / gs;
    const uint32_t nsteps = (n + 31) / 32;
    const uint32_t st0 = blockIdx.z * steps_per, st1 = min(nsteps, st0 + steps_per);   // st0 < st1 by the launch

    // ---- global side of the direct-to-LDS loads: load q = 4 i + wave of a step --------------------------
    //   q 0..7: rows 8 q .. 8 q + 7 of grad_y (lane: row lane / 8, floats 4 (lane % 8) .. + 3)
    //   q 8 (and 9 when KW = 4): word rows 8 (q - 8) .. + 7 of the weights (lane: row lane / 8, words
    //         4 (lane % 8) .. + 3)
    //   next: lanes 0..31 scaled scale, 32..63 zero-point fraction of column lane % 32
    //   last (and any slot left over): lanes 0..15 two f16 zero-point integers each (columns 2 lane,
    //         2 lane + 1); the other lanes fetch the same words again, into the unused tail of the stage
    const uint32_t l8 = lane >> 3, p8 = lane & 7;
    // Address of a load = a base that is the same for the whole wave (array, tile, and the step's columns: scalar
    // registers, advanced by scalar arithmetic) + a 32-bit offset per lane that never changes (row, column inside the
    // step): no vector instruction per load and step.  Only a step that reaches past n (the last one when n % 32 != 0)
    // works its addresses out lane by lane, to send the columns past n to column 0.
    const uint8_t* ubase[kTLoads];                             // wave-uniform
    uint32_t voff[kTLoads], colw[kTLoads];                     // per lane; colw: the lane's first column inside a step
    uint32_t dst[kTLoads], esz[kTLoads];                       // dst: offset inside the slot of its kind
    bool wide[kTLoads], is_gy[kTLoads];
    const uint32_t zf_off = (uint32_t)(reinterpret_cast<const uint8_t*>(zf) - reinterpret_cast<const uint8_t*>(sp));   // one workspace: < 2^32
#pragma unroll
    for (int i = 0; i < kTLoads; i++) {
        uint32_t q = KW * i + wave;
        if (HALF && q >= 4) q += 4;                            // no loads of rows 32..63 of grad_y
        is_gy[i] = q < 8;
        if (q < 8) {
            const uint32_t row = min(m0 + 8 * q + l8, m - 1) - m0;
            ubase[i] = reinterpret_cast<const uint8_t*>(gy + (uint64_t)m0 * n);
            // rows two apart would put the conversion's 128-bit reads two to a bank: every other pair of rows
            // holds its 16-byte pieces swapped in twos (LDS piece p of row r = piece p ^ (r / 2 % 2) of the tile)
            dst[i] = q * 1024; colw[i] = 4 * (p8 ^ ((l8 >> 1) & 1)); wide[i] = true; esz[i] = 4;
            voff[i] = (row * n + colw[i]) * 4;                 // < 64 n 4
        } else if (q < 8 + WS) {
            // the tile's 4 KW word rows (< padded_k / 8: whole groups exist in the arrays); lanes past them
            // fetch its last row again, into room the stage keeps for that
            const uint32_t wr = min(8 * (q - 8) + l8, 4u * KW - 1);
            ubase[i] = reinterpret_cast<const uint8_t*>(packed + (uint64_t)(k0 / 8) * n);
            dst[i] = (q - 8) * 1024; colw[i] = 4 * p8; wide[i] = true; esz[i] = 4;
            voff[i] = (wr * n + colw[i]) * 4;
        } else if (q == 8 + WS) {
            ubase[i] = reinterpret_cast<const uint8_t*>(sp + (uint64_t)g * n);   // zf lies zf_off behind sp
            dst[i] = kTRawW; colw[i] = lane & 31; wide[i] = false; esz[i] = 4;
            voff[i] = colw[i] * 4 + (lane < 32 ? 0 : zf_off);
        } else {
            ubase[i] = reinterpret_cast<const uint8_t*>(zo + (uint64_t)g * n);
            dst[i] = kTRawW + kTRawSz; colw[i] = 2 * (lane & 15); wide[i] = false; esz[i] = 2;
            voff[i] = colw[i] * 2;
        }
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(w4t_lds_offset(lds));
    auto issue = [&](uint32_t st, uint32_t gslot, uint32_t wslot) {
        const uint32_t gbase = lds0 + gslot * kTRawGy, wbase = lds0 + (kTStages - 1) * kTRawGy + wslot * kTRawWt;
        const uint32_t c0 = min(st, st1 - 1) * 32;
        const bool inside = c0 + 32 <= n;
#pragma unroll
        for (int i = 0; i < kTLoads; i++) {
            constexpr int skip = HALF ? 4 : 0;
            const bool all_wide = KW * (i + 1) - 1 + skip < 8 + WS;    // whatever the wave
            const uint32_t to = (is_gy[i] ? gbase : wbase) + dst[i];
            const uint8_t* from = ubase[i];
            uint32_t at = voff[i];
            if (inside) {
                from += (uint64_t)c0 * esz[i];
            } else {
                // columns past n are fetched from column 0: the conversion turns them into zeros
                const uint32_t col = c0 + colw[i] < n ? c0 + colw[i] : 0;
                at += (col - colw[i]) * esz[i];
            }
            if (all_wide || wide[i]) w4t_load16(to, from, at);
            else w4t_load4(to, from, at);
        }
    };

    // ---- conversion role: row tid / KW, its chunks of 8 consecutive n: 4 / KW of them from (tid % KW) 4 / KW ----
    constexpr int CPT = 4 / KW;
    const uint32_t s_row = tid / KW, s_ch0 = (tid % KW) * CPT;
    const float frow_raw = rowf[min(m0 + s_row, m - 1)];
    const float frow = frow_raw != frow_raw ? 0.0f : frow_raw; // inf / nan in the row: NaN times 0 poisons it below
    const uint32_t n_end = min(n, st1 * 32);
    float csum = 0.0f;
    auto convert_chunk = [&](uint32_t st, uint32_t gslot, uint32_t wslot, int buf, uint32_t s_ch) {
        const uint32_t s_lds = s_row * 64 + ((s_ch ^ row_swizzle(s_row)) & 3) * 16;
        const uint8_t* gbase = raw_gy + gslot * kTRawGy;
        const uint8_t* tbase = raw_wt + wslot * kTRawWt + kTRawW;
        const uint32_t sw = (s_row >> 1) & 1;                  // see the loads: pieces swapped in twos
        const float4 g0 = *reinterpret_cast<const float4*>(gbase + s_row * 128 + ((2 * s_ch) ^ sw) * 16);
        const float4 g1 = *reinterpret_cast<const float4*>(gbase + s_row * 128 + ((2 * s_ch + 1) ^ sw) * 16);
        const float4 s0 = *reinterpret_cast<const float4*>(tbase + s_ch * 32);
        const float4 s1 = *reinterpret_cast<const float4*>(tbase + s_ch * 32 + 16);
        const float4 z0 = *reinterpret_cast<const float4*>(tbase + 128 + s_ch * 32);
        const float4 z1 = *reinterpret_cast<const float4*>(tbase + 128 + s_ch * 32 + 16);
        const uint32_t c0 = st * 32 + s_ch * 8;                // (and past the workgroup's share nothing is added to its sum)
        // n % 4 == 0: four columns are all-in or all-out; the columns past n hold values of column 0
        const float f0 = c0 < n_end ? frow : 0.0f, f1 = c0 + 4 < n_end ? frow : 0.0f;
        // powers of two first: gy f is exact, the product with s / S is rounded once
        const float a[8] = {(g0.x * f0) * s0.x, (g0.y * f0) * s0.y, (g0.z * f0) * s0.z, (g0.w * f0) * s0.w,
                            (g1.x * f1) * s1.x, (g1.y * f1) * s1.y, (g1.z * f1) * s1.z, (g1.w * f1) * s1.w};
        const float zv[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            csum = fmaf(a[e], zv[e], csum);
            csum = fmaf(a[e + 1], zv[e + 1], csum);
            // hi = a cut to 11 bits (one instruction for two values), lo = the rest cut to 11 bits: 2^-21 of a
            // is lost at most.  The explicit conversion also keeps the compiler from rounding a product
            // to f16 in two different ways (v_fma_mixlo_f16 of the exact product here, a conversion of the
            // rounded f32 there), which on a tie differ by a whole f16 step that hi + lo then misses.
            const auto h2 = __builtin_amdgcn_cvt_pkrtz(a[e], a[e + 1]);
            // a - hi is exact (the low bits of a): one mixed-precision fma each (the f16 half read in place) instead of
            // a conversion and a subtraction, which is what the compiler makes of the plain expression
            const uint32_t h2b = __builtin_bit_cast(uint32_t, h2);
            float r0, r1;
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(h2b), "v"(a[e]));
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(h2b), "v"(a[e + 1]));
            const auto l2 = __builtin_amdgcn_cvt_pkrtz(r0, r1);
            hi[e / 2] = __builtin_bit_cast(uint32_t, h2);
            lo[e / 2] = __builtin_bit_cast(uint32_t, l2);
        }
        uint8_t* ab = abuf + buf * kTAbuf;
        *reinterpret_cast<uint4*>(ab + s_lds) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        *reinterpret_cast<uint4*>(ab + 64 * 64 + s_lds) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    };
    auto convert = [&](uint32_t st, uint32_t gslot, uint32_t wslot, int buf) {
        if (HALF && s_row >= 32) return;                       // whole waves when KW >= 2
#pragma unroll
        for (int cc = 0; cc < CPT; cc++) convert_chunk(st, gslot, wslot, buf, s_ch0 + cc);
    };

    // ---- B role: lane (k = 32 wave + lane % 32, half = lane / 32): 8 words of word row 4 wave + k / 8 ----
    const uint32_t bc = lane & 31, bh = lane >> 5;
    // Nibble k % 8 lies in byte k % 8 / 2 of its word: one v_perm_b32 puts that byte of two words into the halves of a third,
    // one shift (by 0 or 4) brings the nibbles down, one v_and_or_b32 masks them and adds the mantissa of 1024: four instructions
    // for two values with the subtraction, where a field extract per word, a shift-or and an or took five (111 -> 103 vector
    // instructions per step).  Mask and constant sit in vector registers: the instruction reads one scalar operand only.
    const uint32_t shift = 4 * (bc & 1), pick = (0x0C040C00u) + ((bc & 7) >> 1) * 0x00010001u;
    uint32_t mask = 0x000F000Fu, magic = 0x64006400u;
    asm("" : "+v"(mask), "+v"(magic));
    const uint32_t b_off = (4 * wave + (bc >> 3)) * 128 + bh * 32;
    uint4 bw[4];
    t8h boff[2];                                               // 1024 + z0
    auto b_read = [&](uint32_t wslot) {
        const uint8_t* sb = raw_wt + wslot * kTRawWt;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            bw[2 * t] = *reinterpret_cast<const uint4*>(sb + b_off + t * 64);
            bw[2 * t + 1] = *reinterpret_cast<const uint4*>(sb + b_off + t * 64 + 16);
            boff[t] = *reinterpret_cast<const t8h*>(sb + kTRawW + kTRawSz + 32 * t + 16 * bh);
        }
    };
    auto b_cut = [&](int j, t8h (&to)[2]) {                    // the four values of word quad j, j = 0 .. 3
        const uint32_t w[4] = {bw[j].x, bw[j].y, bw[j].z, bw[j].w};
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t q = ((__builtin_amdgcn_perm(w[2 * i + 1], w[2 * i], pick) >> shift) & mask) | magic;
            const int e = 4 * (j & 1) + 2 * i;
            const t2h h = __builtin_bit_cast(t2h, q) - t2h{boff[j >> 1][e], boff[j >> 1][e + 1]};   // (1024 + q) - (1024 + z0): exact
            to[j >> 1][e] = h[0];
            to[j >> 1][e + 1] = h[1];
        }
    };

    // ---- A fragment reads: lane (row fr, half fh), MFMA step t: logical chunk 2 t + fh -----------------
    const uint32_t fr = lane & 31, fh = lane >> 5, fsw = row_swizzle(fr);
    uint32_t a_off[2];
#pragma unroll
    for (int t = 0; t < 2; t++) a_off[t] = fr * 64 + (((2 * t + fh) ^ fsw) & 3) * 16;

    t16f acc[RTILES];
#pragma unroll
    for (int i = 0; i < RTILES; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

    // ---- pipeline -----------------------------------------------------------------------------------------
    // Every step issues exactly kTLoads loads per wave, also past the end (the last step again, into a
    // stage nobody reads any more), so the counter arithmetic has no tail cases.
#pragma unroll
    for (int s = 0; s < kTStages - 1; s++) issue(st0 + s, s, s);
    w4t_publish<(kTStages - 2) * kTLoads>();                  // step st0 has landed
    convert(st0, 0, 0, 0);
    // The B fragments of a step are cut out of its words while the MFMAs of the step before run (a wave issues
    // nothing while it waits to issue an MFMA: fragments and MFMAs of the same step one after the other leave the
    // vector ALU idle during the MFMAs and the matrix cores idle during the cutting).
    t8h first[2];
    b_read(0);
#pragma unroll
    for (int j = 0; j < 4; j++) b_cut(j, first);
    t8h b0 = first[0], b1 = first[1];
    uint32_t cur = 0, gcur = 0;                                // slots of step st: weights and tables, grad_y
    for (uint32_t st = st0; st < st1; st++) {
        const int ab = (st - st0) & 1;
        const uint32_t nxt = cur + 1 == kTStages ? 0 : cur + 1, prv = cur == 0 ? kTStages - 1 : cur - 1;
        const uint32_t gnxt = gcur + 1 == kTStages - 1 ? 0 : gcur + 1;
        // step st+1 has landed once only the kTStages-3 younger steps are outstanding; past the barrier
        // the A fragments of step st are visible, the weight slot of step st-1 is free and so is the grad_y
        // slot of step st itself (converted during step st-1)
        w4t_publish<(kTStages - 3) * kTLoads>();
        issue(st + (kTStages - 1), gcur, prv);
        // Tile by tile: the fragments of a tile are read in one go, and between its MFMAs stand a share of the next step's B
        // fragments (first tile; after the last step: that step's words again, unused) and of its A fragments (after the last
        // step: zeros that nobody reads), held there by the scheduling barriers.
        const uint8_t* abp = abuf + ab * kTAbuf;
        t8h nb[2];
#pragma unroll
        for (int i = 0; i < RTILES; i++) {
            const uint8_t* hi = abp + i * 32 * 64;
            const uint8_t* lo = abp + 64 * 64 + i * 32 * 64;
            const t8h f[4] = {*reinterpret_cast<const t8h*>(hi + a_off[0]), *reinterpret_cast<const t8h*>(lo + a_off[0]),
                              *reinterpret_cast<const t8h*>(hi + a_off[1]), *reinterpret_cast<const t8h*>(lo + a_off[1])};
            if (i == 0) {
                b_read(nxt);
            } else {
                convert(st + 1, gnxt, nxt, ab ^ 1);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], j < 2 ? b0 : b1, acc[i], 0, 0, 0);
                if (i == 0) b_cut(j, nb);
            }
            if (i == 0) {
                __builtin_amdgcn_sched_group_barrier(0x100, 10, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                }
            } else {
                __builtin_amdgcn_sched_group_barrier(0x100, 10, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 13, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (RTILES == 1) convert(st + 1, gnxt, nxt, ab ^ 1);
        b0 = nb[0];
        b1 = nb[1];
        cur = nxt;
        gcur = gnxt;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct-to-LDS write may outlive the workgroup

    // ---- c[row]: the KW conversion threads of a row are neighbours in a wave ---------------------------
    if (KW >= 2) csum += __shfl_xor(csum, 1);
    if (KW == 4) csum += __shfl_xor(csum, 2);
    // and 1 / f_row = 2^(e - 140), from the bits of f (f = 2^(140 - e), biased exponent 267 - e), fetched when the kernel began: a
    // load in front of every store would cost a trip to memory per row (its wait includes the stores before it)
    if (tid % KW == 0) {
        lds_c[s_row] = csum;
        lds_c[64 + s_row] = frow_raw != frow_raw ? frow_raw
                            : frow_raw == 0.0f   ? 0.0f
                                                 : __uint_as_float((254u - (__float_as_uint(frow_raw) >> 23)) << 23);
    }
    __syncthreads();

    // ---- register r of lane l is row 8 (r/4) + 4 (l/32) + r%4, column l%32 of its 32 x 32 tile -------
    const uint32_t col = k0 + 32 * wave + bc;
    const float s_big = sgrp[g];
    if (col >= k) return;
    float* const dst_out = out + (uint64_t)blockIdx.z * m * k + (uint64_t)m0 * k + col;
    auto value = [&](int i, int r, uint32_t lr) { return ((acc[i][r] - lds_c[lr]) * lds_c[64 + lr]) * s_big; };
    const uint32_t live = m - m0;
    if (live >= 32u * RTILES) {
#pragma unroll
        for (int i = 0; i < RTILES; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t lr = 32 * i + 8 * (r / 4) + 4 * fh + (r % 4);
                dst_out[(uint64_t)lr * k] = value(i, r, lr);
            }
    } else {
#pragma unroll
        for (int i = 0; i < RTILES; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t lr = 32 * i + 8 * (r / 4) + 4 * fh + (r % 4);
                if (lr < live) dst_out[(uint64_t)lr * k] = value(i, r, lr);
            }
    }
}

// ---- batches: the activations are converted in registers, once per group ---------------------------------------------
// Above, four waves share 64 x 32 converted activations through LDS for 32 columns each: 103 vector instructions and 24 KB of LDS
// traffic per wave and 8 MFMAs.  Here a wave owns 64 rows x all 128 columns of a group (128 accumulator registers) over its own
// range of n, and nothing in its loop is shared, so there is no barrier in it either:
//   * an A fragment is built where it is used: lane (row = lane % 32, half = lane / 32) reads its 8 floats of grad_y from LDS (where
//     direct loads put them, since 32 rows apart they are no coalesced load) and makes hi and lo of them, once per group, with
//     c += p (s (zp - z0)), p = gy f, six instructions an element;
//   * the nibbles of a word serve one lane alone: lane l takes word row l % 16 of the group's 16 and the half l / 16 of its words,
//     i.e. column 8 (l % 16) + 4 (l / 16) + j of the tile for column tile j = 0 .. 3.  Two words give the halves of a register with
//     one v_perm_b32 and that 8 values with one shift, four v_and_or_b32 and four subtractions: 1.25 instructions a value (2 above).
// Together 8 vector instructions per MFMA and 16 KB of LDS traffic per 16.  The workgroup's four waves take a quarter of its steps
// of 16 columns each and add their tiles through LDS at the end; lane l's four columns are adjacent, so a row is stored in 16-byte pieces.
// One box in turn, above -> here (us, 4096 x 11008): 48 rows 34.1 -> 26.8, 128 rows 48.4 -> 39, 512 rows 143 -> 113, 1024 rows 292 -> 207, 2048
// rows 518 -> 403; 11008 x 4096 at 512 rows 146 -> 111.  Error against float64 4.3e-7 -> 2.9e-7 of a row at 512 rows (shorter sums, and
// hi and lo rounded instead of cut).  What bounds it: vector issue 65 % and matrix cores 49 % of the cycles at 1.76 GHz; neither hides behind
// the other (one wave per SIMD is as fast as two), without the conversions a call would take 20 % less, without the loads 20 %.
// Tried: 128 rows per wave (a wave per SIMD, 256 accumulators) 5 % faster at 4096 x 11008 from 512 rows on, up to 18 % slower elsewhere; the
// fragments' LDS reads one row tile ahead: 2 % slower.
constexpr int kTWStages = 3, kTWLoads = 6;                    // loads per wave and step: 4 grad_y, 1 words, 1 tables
constexpr uint32_t kTWGy = 64 * 64, kTWWords = 16 * 64, kTWStage = kTWGy + kTWWords + 256;   // per wave and step; kTBlock of the last 256 bytes
constexpr uint32_t kTWLds = 4 * 16384;                        // the stages of four waves; afterwards half of each one's tile
static_assert(4 * kTWStages * kTWStage <= kTWLds && 2 * (kTWLds + 1024) <= 160 * 1024, "they fit, and two workgroups a compute unit");

// kTBlock bytes, 16 per lane of the first ten
__device__ __forceinline__ void w4t_load_tables(uint32_t to, const void* from, uint32_t lane_bytes) {
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, 0x3ff\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                 ::"s"(to), "v"(lane_bytes), "s"(from) : "memory");
}

__global__ __launch_bounds__(256, 2) void w4t_wide_kernel(
    const float* __restrict__ gy, const uint32_t* __restrict__ packed, const uint8_t* __restrict__ tables,
    const float* __restrict__ rowf, const float* __restrict__ sgrp, float* __restrict__ out, uint32_t m, uint32_t k, uint32_t n,
    uint32_t gs, uint32_t shares) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float lds_c[4][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t l32 = lane & 31, half = lane >> 5, l4 = lane >> 2, p4 = lane & 3;
    const uint32_t k0 = blockIdx.x * 128, m0 = blockIdx.y * 64, g = k0 / gs;
    const uint32_t nsteps = n / 16, part = blockIdx.z * 4 + wave, parts = 4 * shares;
    const uint32_t st0 = (uint32_t)((uint64_t)nsteps * part / parts), st1 = (uint32_t)((uint64_t)nsteps * (part + 1) / parts);

    // ---- loads into LDS: a base that is the same for the whole wave plus an offset per lane that never changes ------------
    // (piece p of 16 bytes of row r lies at place p ^ row_swizzle(r): the fragments' reads then fall on different banks)
    uint32_t gy_off[4];
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        const uint32_t r = 16 * q + l4;
        gy_off[q] = ((min(m0 + r, m - 1) - m0) * n + 4 * ((p4 ^ row_swizzle(r)) & 3)) * 4;
    }
    const uint32_t w_off = (l4 * n + 4 * ((p4 ^ row_swizzle(l4)) & 3)) * 4, t_off = lane * 16;
    const float* const gy0 = gy + (uint64_t)m0 * n;
    const uint32_t* const words0 = packed + (uint64_t)(k0 / 8) * n;
    const uint8_t* const tables0 = tables + (uint64_t)g * nsteps * kTBlock;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(w4t_lds_offset(lds)) + wave * (kTWStages * kTWStage);
    auto issue = [&](uint32_t st, uint32_t slot) __attribute__((always_inline)) {
        const uint32_t at = min(st, nsteps - 1), to = lds0 + slot * kTWStage;   // past the end: the last one, for nobody
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) w4t_load16(to + q * 1024, gy0 + (uint64_t)at * 16, gy_off[q]);
        w4t_load16(to + kTWGy, words0 + (uint64_t)at * 16, w_off);
        w4t_load_tables(to + kTWGy + kTWWords, tables0 + (uint64_t)at * kTBlock, t_off);
    };

    // ---- fragments ---------------------------------------------------------------------------------------------------
    const uint8_t* const mine = lds + wave * (kTWStages * kTWStage);
    uint32_t a_at[2], w_at[2];                                 // where the lane's two pieces lie (row_swizzle repeats after 16 rows)
#pragma unroll
    for (uint32_t e = 0; e < 2; e++) {
        a_at[e] = l32 * 64 + (((2 * half + e) ^ row_swizzle(l32)) & 3) * 16;
        w_at[e] = kTWGy + (lane & 15) * 64 + (((2 * half + e) ^ row_swizzle(lane & 15)) & 3) * 16;
    }
    float frow[2], csum[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float f = rowf[min(m0 + 32 * i + l32, m - 1)];
        frow[i] = f != f ? 0.0f : f;                           // inf / nan in the row: NaN times 0 poisons it below
        csum[i] = 0.0f;
    }
    const uint32_t pick = (lane & 16) ? 0x07060302u : 0x05040100u;
    uint32_t mask_lo = 0x000F000Fu, mask_hi = 0x00F000F0u, magic = 0x64006400u;
    asm("" : "+v"(mask_lo), "+v"(mask_hi));
    asm("" : "+s"(magic));

    uint4 fa[2][2][2];                                         // [step's parity][row tile][hi, lo]
    uint4 fb[2][4];                                            // [step's parity][column tile]
    struct { float4 sc[2], cz[2]; uint32_t words[8]; t8h zo; } in;
    auto read_step = [&](uint32_t slot) __attribute__((always_inline)) {
        const uint8_t* const at = mine + slot * kTWStage;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const uint4 w = *reinterpret_cast<const uint4*>(at + w_at[e]);
            in.words[4 * e] = w.x; in.words[4 * e + 1] = w.y; in.words[4 * e + 2] = w.z; in.words[4 * e + 3] = w.w;
            in.sc[e] = *reinterpret_cast<const float4*>(at + kTWGy + kTWWords + half * 32 + e * 16);
            in.cz[e] = *reinterpret_cast<const float4*>(at + kTWGy + kTWWords + 64 + half * 32 + e * 16);
        }
        in.zo = *reinterpret_cast<const t8h*>(at + kTWGy + kTWWords + 128 + half * 16);
    };
    float4 raw[2];
    auto read_rows = [&](uint32_t slot, int i) __attribute__((always_inline)) {
        raw[0] = *reinterpret_cast<const float4*>(mine + slot * kTWStage + a_at[0] + i * 2048);
        raw[1] = *reinterpret_cast<const float4*>(mine + slot * kTWStage + a_at[1] + i * 2048);
    };
    auto convert = [&](int i, float f, uint4 (&to)[2]) __attribute__((always_inline)) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float4 v = raw[e >> 1], s4 = in.sc[e >> 1], z4 = in.cz[e >> 1];
            const float p0 = ((e & 1) ? v.z : v.x) * f, p1 = ((e & 1) ? v.w : v.y) * f;
            const float a0 = p0 * ((e & 1) ? s4.z : s4.x), a1 = p1 * ((e & 1) ? s4.w : s4.y);
            csum[i] = fmaf(p0, (e & 1) ? z4.z : z4.x, csum[i]);
            csum[i] = fmaf(p1, (e & 1) ? z4.w : z4.y, csum[i]);
            // (v_fma_mixlo_f16 / _mixhi_f16 would save an instruction per element, and issue at half the rate)
            float r0, r1;
            asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(hi[e]) : "v"(a0), "v"(a1));
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(hi[e]), "v"(a0));
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(hi[e]), "v"(a1));
            asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(lo[e]) : "v"(r0), "v"(r1));
        }
        to[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        to[1] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    };
    auto cut = [&](int e, uint4 (&to)[4]) __attribute__((always_inline)) {   // words 2 e and 2 e + 1
        const t2h k16th = {(_Float16)0.0625f, (_Float16)0.0625f}, c960 = {(_Float16)960.0f, (_Float16)960.0f};
        const t2h big = {in.zo[2 * e], in.zo[2 * e + 1]}, small = c960 - big;   // 1024 + z0, -64 - z0
        const uint32_t u = __builtin_amdgcn_perm(in.words[2 * e + 1], in.words[2 * e], pick), u8 = u >> 8;
        const uint32_t t0 = (u & mask_lo) | magic, t1 = (u & mask_hi) | magic, t2 = (u8 & mask_lo) | magic, t3 = (u8 & mask_hi) | magic;
        // (1024 + q) - (1024 + z0) and (1024 + 16 q) / 16 - (64 + z0): exact
        const uint32_t h[4] = {__builtin_bit_cast(uint32_t, __builtin_bit_cast(t2h, t0) - big),
                               __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(t2h, t1), k16th, small)),
                               __builtin_bit_cast(uint32_t, __builtin_bit_cast(t2h, t2) - big),
                               __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(t2h, t3), k16th, small))};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (e == 0) to[j].x = h[j];
            else if (e == 1) to[j].y = h[j];
            else if (e == 2) to[j].z = h[j];
            else to[j].w = h[j];
        }
    };
    t16f acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = t16f{};

    // ---- pipeline: while the MFMAs of a step run, the fragments of the next one are made, half of them beside each row tile's ------
    uint32_t slot = 0;                                         // of the step whose MFMAs run
    if (st0 < st1) {
#pragma unroll
        for (uint32_t u = 0; u < kTWStages; u++) issue(st0 + u, u);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kTWStages - 1) * kTWLoads) : "memory");
        read_step(0);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            read_rows(0, i);
            convert(i, frow[i], fa[0][i]);
            cut(2 * i, fb[0]);
            cut(2 * i + 1, fb[0]);
        }
    }
    auto step = [&](uint32_t st, auto p_tag) __attribute__((always_inline)) {
        constexpr int P = decltype(p_tag)::value;
        const uint32_t next = slot == kTWStages - 1 ? 0 : slot + 1;
        // the next step has landed once only the one after it is outstanding; this one's slot was read out during the last step
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kTWLoads) : "memory");
        issue(st + kTWStages, slot);
        read_step(next);
        const float live = st + 1 < st1 ? 1.0f : 0.0f;         // past the wave's share nothing is added to its sums
#pragma unroll
        for (int i = 0; i < 2; i++) {
            read_rows(next, i);
            convert(i, frow[i] * live, fa[P ^ 1][i]);
            cut(2 * i, fb[P ^ 1]);
            cut(2 * i + 1, fb[P ^ 1]);
#pragma unroll
            for (int d = 0; d < 2; d++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(t8h, fa[P][i][d]), __builtin_bit_cast(t8h, fb[P][j]), acc[i][j], 0, 0, 0);
            if (i == 0) __builtin_amdgcn_sched_group_barrier(0x100, 9, 0);
            else __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int d = 0; d < 8; d++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        slot = next;
    };
    uint32_t st = st0;
    for (; st + 1 < st1; st += 2) {
        step(st, std::integral_constant<int, 0>{});
        step(st + 1, std::integral_constant<int, 1>{});
    }
    if (st < st1) step(st, std::integral_constant<int, 0>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // no load into LDS may outlive this
    __syncthreads();

    // ---- the four waves' tiles: wave w ends up with rows 16 (w / 2) .. + 15 of row tile w % 2: first the waves of a pair exchange --
    // a row tile, then the pairs half of one (registers 8 h .. + 7 are rows 16 h .. + 15)
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float c = csum[i] + __shfl_xor(csum[i], 32);
        if (half == 0) lds_c[wave][32 * i + l32] = c;
    }
    float4* const box = reinterpret_cast<float4*>(lds);        // [wave][half row tile][4 column tiles][2][64 lanes]
    float sum[4][8];
    auto columns = [&](auto f) __attribute__((always_inline)) {   // (indexes as constants: the accumulators have to stay registers)
        f(std::integral_constant<int, 0>{});
        f(std::integral_constant<int, 1>{});
        f(std::integral_constant<int, 2>{});
        f(std::integral_constant<int, 3>{});
    };
    auto put = [&](auto i_tag, auto h_tag, uint32_t place) __attribute__((always_inline)) {
        constexpr int I = decltype(i_tag)::value, R = 8 * decltype(h_tag)::value;
        columns([&](auto j) __attribute__((always_inline)) {
            const t16f& t = acc[I][j.value];
            float4* const at = box + (place * 8 + 2 * j.value) * 64 + lane;
            at[0] = make_float4(t[R], t[R + 1], t[R + 2], t[R + 3]);
            at[64] = make_float4(t[R + 4], t[R + 5], t[R + 6], t[R + 7]);
        });
    };
    auto take = [&](auto i_tag, auto h_tag, uint32_t place, auto into) __attribute__((always_inline)) {
        constexpr int I = decltype(i_tag)::value, R = 8 * decltype(h_tag)::value;
        columns([&](auto j) __attribute__((always_inline)) {
            const t16f& t = acc[I][j.value];
            const float4* const at = box + (place * 8 + 2 * j.value) * 64 + lane;
            const float4 v = at[0], w = at[64];
            const float o[8] = {t[R] + v.x, t[R + 1] + v.y, t[R + 2] + v.z, t[R + 3] + v.w, t[R + 4] + w.x, t[R + 5] + w.y, t[R + 6] + w.z, t[R + 7] + w.w};
            into(j, o);
        });
    };
    typedef std::integral_constant<int, 0> zero;
    typedef std::integral_constant<int, 1> one;
    auto exchange = [&](auto keep, auto send) __attribute__((always_inline)) {
        constexpr int I = decltype(keep)::value;
        put(send, zero{}, 2 * wave);
        put(send, one{}, 2 * wave + 1);
        __syncthreads();
        auto back = [&](auto h) __attribute__((always_inline)) {
            take(keep, h, 2 * (wave ^ 1) + h.value, [&](auto j, const float (&o)[8]) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < 8; r++) acc[I][j.value][8 * h.value + r] = o[r];
            });
        };
        back(zero{});
        back(one{});
        __syncthreads();
        auto halves = [&](auto mine_h, auto other_h) __attribute__((always_inline)) {
            put(keep, other_h, wave);
            __syncthreads();
            take(keep, mine_h, wave ^ 2, [&](auto j, const float (&o)[8]) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < 8; r++) sum[j.value][r] = o[r];
            });
            asm volatile("; half %0 of row tile %1" ::"n"(decltype(mine_h)::value), "n"(I));   // (merged, the variants would index the accumulators)
        };
        if (wave < 2) halves(zero{}, one{});
        else halves(one{}, zero{});
        asm volatile("; row tile %0" ::"n"(I));
    };
    if ((wave & 1) == 0) exchange(zero{}, one{});
    else exchange(one{}, zero{});

    // ---- register r of lane l is row 8 (r/4) + 4 (l/32) + r%4 of a row tile ---------------------------------------------------
    const uint32_t col = k0 + 8 * (lane & 15) + 4 * ((lane >> 4) & 1), row0 = 32 * (wave & 1) + 16 * (wave >> 1);
    const float s_big = sgrp[g];
    float c8[8], f8[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint32_t lr = row0 + 8 * (r / 4) + 4 * half + (r % 4);
        c8[r] = (lds_c[0][lr] + lds_c[1][lr]) + (lds_c[2][lr] + lds_c[3][lr]);
        // 1 / f_row = 2^(e - 140), from the bits of f (f = 2^(140 - e), biased exponent 267 - e)
        const float f = rowf[min(m0 + lr, m - 1)];
        f8[r] = f != f ? f : f == 0.0f ? 0.0f : __uint_as_float((254u - (__float_as_uint(f) >> 23)) << 23);
    }
    if (col >= k) return;                                      // k % 4 == 0
    float* const dst = out + (uint64_t)blockIdx.z * m * k + (uint64_t)m0 * k + col;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint32_t lr = row0 + 8 * (r / 4) + 4 * half + (r % 4);
        auto value = [&](int j) { return ((sum[j][r] - c8[r]) * f8[r]) * s_big; };
        if (m0 + lr < m) *reinterpret_cast<float4*>(dst + (uint64_t)lr * k) = make_float4(value(0), value(1), value(2), value(3));
    }
}

// out = sum over the shares of n of their partial results, in share order
__global__ __launch_bounds__(256) void w4t_add_shares_kernel(const float4* __restrict__ part, float4* __restrict__ out,
                                                             uint32_t count4, uint32_t shares) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= count4) return;
    float4 v = part[i];
    for (uint32_t z = 1; z < shares; z++) {
        const float4 t = part[(uint64_t)z * count4 + i];
        v.x += t.x; v.y += t.y; v.z += t.z; v.w += t.w;
    }
    out[i] = v;
}

bool w4_gemm_t_supported(uint32_t m, uint32_t k, uint32_t n, uint32_t group_size, const void* gy, const void* packed,
                         const void* scales, const void* zp, const void* out) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(gy) | reinterpret_cast<uintptr_t>(packed) |
                           reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(zp) |
                           reinterpret_cast<uintptr_t>(out);
    return (group_size % 128 == 0 || group_size == 64 || group_size == 32) && n % 4 == 0 && k % 4 == 0 && (bits & 15) == 0 &&
           (uint64_t)m * k < (1ull << 32) && (uint64_t)m * n < (1ull << 40);
}

// Shares of n of the wide kernel.  A step of 16 columns takes a compute unit 0.48 us per workgroup that it holds (two side by side
// take twice as long: the vector unit and the matrix cores are busy all the time with one), so what counts is the most that any
// gets; every share's partial result is written and read once, by one more launch.  Over 35 shapes (16 to 2048 rows) the choice is
// within 3 % of the best of 1 .. 16: 4096 x 11008 at 512 rows 1 share 113.5 us, 4 shares 118.8; at 100 rows 91.5 and 37.5.
struct W4tShares { uint32_t shares; double us; };
static W4tShares w4t_wide_shares(uint32_t tiles, uint32_t m, uint32_t k, uint32_t n) {
    W4tShares best{1, 1e30};
    for (uint32_t shares = 1; shares == 1 || (shares <= (uint32_t)kTMaxSplits && n / 16 >= 8 * shares); shares++) {
        const double us = 8.7 + (double)ceil_div(tiles * shares, 256) * ceil_div(n / 16, 4 * shares) * 0.48 + (shares > 1 ? 3.0 + (shares + 1.0) * m * k * 4 / 4.5e6 : 0.0);
        if (us < best.us) best = W4tShares{shares, us};
    }
    return best;
}

// Shares of n of the narrow kernel.  Four workgroups share a compute unit; a step of 32 columns then takes them `step` us, `beside` more for each
// neighbour, and a round of them `start` us besides; partial results are added by one more launch (`add`, and 0.3 a share).  Fitted to 241 calls with
// groups of 32, 64 and 128 (13 to 1024 rows, k and n 512 to 11008, 1 to 16 shares each; 3 to 5 % rms near the best): the choice is 1 % slower than
// the best of a shape on average, 10 % at worst.  Shares of at least sixteen steps, as before, left weights of few columns on a few workgroups: groups of 32 1.25, of 64 1.13 times
// as fast now, us: 50 x 1728 x 688 (k, n) groups of 32 37.1 -> 17.1, of 64 26.7 -> 15.4; 126 x 1024 x 1024 31.6 -> 19.1, 23.9 -> 17.0; 200 x 4096 x 4096 179.8 ->
// 100.8 (groups of 32); 24 x 6912 x 688 22.3 -> 15.5 (64), 18.3 -> 13.6 (128).
static W4tShares w4t_narrow_shares(uint32_t tiles, int kw, uint32_t m, uint32_t k, uint32_t n) {
    struct Cost { double step, beside, start, add; };
    const Cost c = kw == 1 ? Cost{1.26, 0.07, 2.8, 1.9} : kw == 4 ? (m <= 32 ? Cost{0.50, 0.19, 0.8, 1.8} : Cost{0.62, 0.25, 1.6, 2.0})
                                                        : (m <= 32 ? Cost{0.65, 0.13, 2.0, 1.9} : Cost{0.84, 0.12, 1.5, 2.7});
    const uint32_t nsteps = ceil_div(n, 32);
    W4tShares best{1, 1e30};
    for (uint32_t want = 1; want <= min((uint32_t)kTMaxSplits, nsteps); want++) {
        const uint32_t steps = ceil_div(nsteps, want), shares = ceil_div(nsteps, steps);
        const uint64_t on_one = ((uint64_t)tiles * shares + 255) / 256, last = on_one % 4;
        double us = 6.0 + (double)(on_one / 4) * (steps * (c.step + 3 * c.beside) + c.start) + (last ? steps * (c.step + (last - 1) * c.beside) + c.start : 0.0);
        if (shares > 1) us += c.add + 0.3 * shares + (shares + 1.0) * m * k * 4 / 4.5e6;
        if (us < best.us) best = W4tShares{shares, us};
    }
    return best;
}

// Up to 32 rows half of the wide kernel's rows would be empty (11008 x 4096 at 16 rows 24.1 us on the narrow one, 24.6 there).
static bool w4t_takes_wide(uint32_t m, uint32_t n, uint32_t group_size) { return group_size % 128 == 0 && n % 16 == 0 && m > 32; }

static int w4t_waves(uint32_t group_size) { return group_size % 128 == 0 ? 4 : (int)group_size / 32; }

static W4tShares w4t_shares(uint32_t m, uint32_t k, uint32_t n, uint32_t padded_k, uint32_t group_size) {
    const int kw = w4t_waves(group_size);
    const uint64_t tiles = (uint64_t)(padded_k / (32 * kw)) * ceil_div(m, 64);
    if (tiles >= 1u << 20) return W4tShares{1, 0.0};
    if (w4t_takes_wide(m, n, group_size)) {
        if (tiles >= 512) return W4tShares{1, 0.0};
        return w4t_wide_shares((uint32_t)tiles, m, k, n);
    }
    return w4t_narrow_shares((uint32_t)tiles, kw, m, k, n);
}

double w4_gemm_t_us(uint32_t m, uint32_t k, uint32_t n, uint32_t padded_k, uint32_t group_size) { return w4t_shares(m, k, n, padded_k, group_size).us; }

template <int NS, int KW, bool HALF = false>
static int launch_w4t(uint32_t ktiles, uint32_t mtiles, uint32_t shares, hipStream_t s, const float* gy,
                      const uint32_t* packed, const float* sp, const float* zf, const _Float16* zo, const float* rowf,
                      const float* sgrp, float* out, uint32_t m, uint32_t k, uint32_t n, uint32_t gs, uint32_t steps_per) {
    constexpr size_t lds_bytes = w4t_lds_bytes(NS);
    static bool attr_set = false;   // benign race: setting the attribute is idempotent
    if (!attr_set && lds_bytes > 64 * 1024) {
        if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&w4t_gemm_kernel<NS, KW, HALF>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes),
                               "hipFuncSetAttribute"))
            return rc;
        attr_set = true;
    }
    hipLaunchKernelGGL((w4t_gemm_kernel<NS, KW, HALF>), dim3(ktiles, mtiles, shares), dim3(64 * KW), lds_bytes, s, gy, packed, sp, zf, zo,
                       rowf, sgrp, out, m, k, n, gs, steps_per);
    return check_launch("w4t_gemm_kernel");
}

#define RUMUS_W4T_LAUNCH(NS, KW)                                                                                  \
    (m <= 32 ? launch_w4t<NS, KW, true>(ktiles, mtiles, shares, s, gy, packed, sp, zf, zo, rowf, sgrp,              \
                                        shares > 1 ? part : out, m, k, n, group_size, steps_per)                   \
             : launch_w4t<NS, KW>(ktiles, mtiles, shares, s, gy, packed, sp, zf, zo, rowf, sgrp,                    \
                                  shares > 1 ? part : out, m, k, n, group_size, steps_per))

int w4_launch_gemm_t(const float* gy, const uint32_t* packed, const float* scales, const float* zp, float* out,
                     uint32_t m, uint32_t k, uint32_t n, uint32_t padded_k, uint32_t group_size, uint32_t num_groups,
                     hipStream_t s) {
    const int kw = w4t_waves(group_size);                    // waves per workgroup: 32-column slices of one group
    const uint32_t ktiles = padded_k / (32 * kw), mtiles = ceil_div(m, 64), nsteps = ceil_div(n, 32);
    RUMUS_REQUIRE(mtiles <= 65535, "qmatmul_int4_t: m %u is beyond the grid limit", m);
    const bool wide = w4t_takes_wide(m, n, group_size);
    // n is shared out too where that is the faster
    uint32_t shares = w4t_shares(m, k, n, padded_k, group_size).shares;
    // Without room for the partial results of those shares: no more than the workspace has always had room for, which is what a capture
    // may have been prepared with (tiles for less than two workgroups per compute unit, shares of at least 16 steps, 16 of one row tile, 8 of more).
    uint32_t fewest = 1;
    const uint64_t tiles = (uint64_t)ktiles * mtiles;
    if (tiles < 512) fewest = max(1u, min(min((uint32_t)(1024 / tiles), nsteps / 16), (uint32_t)(mtiles == 1 ? kTMaxSplits : kTMaxSplits / 2)));
    fewest = min(fewest, shares);
    auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
    const size_t gn = (size_t)num_groups * n;
    const size_t rowf_bytes = up((size_t)m * sizeof(float)), sgrp_bytes = up((size_t)num_groups * sizeof(float));
    const size_t sp_bytes = up(gn * sizeof(float)), zo_bytes = up(gn * sizeof(_Float16) + 64);
    auto bytes = [&](uint32_t parts) {
        return rowf_bytes + sgrp_bytes + 2 * sp_bytes + zo_bytes + (parts > 1 ? (size_t)parts * m * k * sizeof(float) : 0);
    };
    void* ws = nullptr;
    size_t got = 0;
    WorkspaceLease lease;                                    // until the last kernel of this call is queued
    if (int rc = workspace_get_upto(s, bytes(fewest), bytes(shares), &got, &ws, lease)) return rc;
    if (got < bytes(shares)) shares = fewest;
    const uint32_t steps_per = ceil_div(nsteps, shares);
    if (!wide) shares = ceil_div(nsteps, steps_per);
    uint8_t* b = static_cast<uint8_t*>(ws);
    float* rowf = reinterpret_cast<float*>(b);
    float* sgrp = reinterpret_cast<float*>(b + rowf_bytes);
    float* sp = reinterpret_cast<float*>(b + rowf_bytes + sgrp_bytes);
    float* zf = reinterpret_cast<float*>(b + rowf_bytes + sgrp_bytes + sp_bytes);
    _Float16* zo = reinterpret_cast<_Float16*>(b + rowf_bytes + sgrp_bytes + 2 * sp_bytes);
    float* part = reinterpret_cast<float*>(b + rowf_bytes + sgrp_bytes + 2 * sp_bytes + zo_bytes);
    auto add_shares = [&] {
        const uint32_t count4 = (uint32_t)((uint64_t)m * k / 4);
        hipLaunchKernelGGL(w4t_add_shares_kernel, dim3(ceil_div(count4, 256)), dim3(256), 0, s,
                           reinterpret_cast<const float4*>(part), reinterpret_cast<float4*>(out), count4, shares);
        return check_launch("w4t_add_shares_kernel");
    };
    if (wide) {
        hipLaunchKernelGGL(w4t_prepare_kernel<true>, dim3(m + num_groups), dim3(256), 0, s, gy, scales, zp, rowf, sgrp, sp, zf, zo, m, n);
        if (int rc = check_launch("w4t_prepare_kernel")) return rc;
        static bool attr_set = false;   // benign race: setting the attribute is idempotent
        if (!attr_set) {
            if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&w4t_wide_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)kTWLds), "hipFuncSetAttribute"))
                return rc;
            attr_set = true;
        }
        hipLaunchKernelGGL(w4t_wide_kernel, dim3(ktiles, mtiles, shares), dim3(256), kTWLds, s, gy, packed, reinterpret_cast<const uint8_t*>(sp), rowf, sgrp,
                           shares > 1 ? part : out, m, k, n, group_size, shares);
        if (int rc = check_launch("w4t_wide_kernel")) return rc;
        return shares == 1 ? RUMUS_HIP_OK : add_shares();
    }
    hipLaunchKernelGGL(w4t_prepare_kernel<false>, dim3(m + num_groups), dim3(256), 0, s, gy, scales, zp, rowf, sgrp, sp, zf, zo, m,
                       n);
    if (int rc = check_launch("w4t_prepare_kernel")) return rc;
    // Three weight slots and two grad_y slots: 39.75 KB of LDS, four workgroups per compute unit.  Workgroups run in
    // rounds of that many per CU and a round lasts almost the same whether it is full or not, so what matters is how
    // many fit: with four stages (three per CU) 2048 rows x 4096 took 0.70 ms for 1024 workgroups on 768 places, with
    // three stages 0.57 ms on 1024 places, and the four-stage form was faster for no batch from 256 to 4096 rows.
    const int rc = kw == 4 ? RUMUS_W4T_LAUNCH(3, 4) : kw == 2 ? RUMUS_W4T_LAUNCH(3, 2) : RUMUS_W4T_LAUNCH(3, 1);
    if (rc) return rc;
    return shares == 1 ? RUMUS_HIP_OK : add_shares();
}

}  // namespace rumus
