// W8A8 layer for a few rows: f32 activations in, one launch.
//
//   y[m, n] = (f32(sum_k xq[m, k] wq[n, k]) * sx[m]) * sw[n] (+ bias[n]),   xq, sx = the row quantizer's (i8_quant.hip)
//
// The same bits as rumus_hip_i8_quantize_rows and rumus_hip_i8_gemm on its result; every workgroup quantizes all of the rows for itself.
// What bounds it: the weights' stream where they are large (8 x 4096 x 11008 3.5 TB/s), else the launch and two trips to memory.  Two
// launches, the quantizer's 2.6 us first -> one, called from Python on 500 MB of weights in turn: 1 x 1024 x 1024 8.8 -> 5.1 us, 2 x 4096 x 4096 9.3 -> 6.7, 4 x 768 x 10800
// 11.1 -> 5.2, 4 x 4096 x 11008 13.6 -> 12.2, 8 x 1152 x 7200 9.4 -> 5.3, 8 x 4096 x 11008 15.2 -> 13.2, 16 x 2048 x 11008 11.8 -> 9.8.
#include "i8_gemm.h"

namespace rumus {

// Eight waves.  P of them share a row, or each takes R rows (P = 1): NV loads of 1 KB a lane and row, all in flight, then the largest
// magnitude, the digits into LDS.  The first column tiles' weights are on their way meanwhile.  1 << share waves then take a share of the K
// steps of 64 each, in chunks of eight, of one column tile of 16, 8 >> share tiles at a time; the workgroup walks over such groups of tiles
// (blockIdx.x, + gridDim.x, ...) as i8_resident_kernel does over tiles, the next chunk's weights in flight.  The partial tiles meet in LDS,
// two sets in turn, one barrier a group.
template <int P, int R, int NV>
__global__ __launch_bounds__(512) void i8_linear_kernel(const float* __restrict__ x, const int8_t* __restrict__ wq,
                                                        const float* __restrict__ sw, const float* __restrict__ bias,
                                                        float* __restrict__ y, uint32_t M, uint32_t K, uint32_t N, uint32_t share) {
    extern __shared__ __attribute__((aligned(16))) int8_t xs[];    // [row][pitch], zeros from K to a whole step
    __shared__ int32_t part[2][8][4][64];                          // [set][wave][register][lane]
    __shared__ float scale_of[16], top_of[8];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t c = lane & 15, q = lane >> 4;
    const uint32_t tiles = (N + 15) / 16, steps = (K + 63) / 64, pitch = steps * 64 + 16;
    const uint32_t waves = 1u << share, at_once = 8u >> share;     // of a tile; tiles of a group
    const uint32_t groups = (tiles + at_once - 1) >> (3 - share);
    const uint32_t ks = (steps + waves - 1) >> share, chunks = (ks + 7) / 8, first = (wave & (waves - 1)) * ks;
    const uint32_t mine = first < steps ? min(ks, steps - first) : 0;   // K steps of this wave
    auto buffer = [](const void* p, uint32_t bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
    };

    // ---- the rows (past the end of a row, and of the rows: zeros by the range check)
    const uint32_t row0 = P > 1 ? wave / P : wave, k0 = (wave % P) * (NV * 256);
    v4i raw[R][NV];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t row = row0 + 8 * r;
        const auto from = buffer(x + (uint64_t)min(row, M - 1) * K, row < M ? K * 4 : 0);
#pragma unroll
        for (int i = 0; i < NV; i++)
            raw[r][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(from, (int)((k0 + i * 256 + lane * 4) * 4), 0, 0));
    }
    __builtin_amdgcn_sched_barrier(0);                             // asked for first, wanted first

    // a lane's piece of 16 bytes; of a last step that K cuts short the last whole one (it meets zeros)
    const uint32_t b_at = c * K + 16 * q, b_last = c * K + min(16 * q, K - 64 * (steps - 1) - 16);
    v4i b[2][8];
    auto fetch = [&](auto buf, uint32_t group, uint32_t chunk) __attribute__((always_inline)) {
        const uint32_t tile = group * at_once + (wave >> share);
        // rows past N, and all of a tile past the last, are zeros that no load is made for
        const auto from = buffer(wq + (uint64_t)(16 * min(tile, tiles - 1)) * K, tile < tiles ? min(16u, N - 16 * tile) * K : 0);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t step = min(first + 8 * chunk + i, steps - 1);
            b[decltype(buf)::value][i] =
                __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(from, (int)(step + 1 == steps ? b_last : b_at), (int)(64 * step), 0));
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    fetch(B0{}, blockIdx.x, 0);                                    // blockIdx.x < groups
    __builtin_amdgcn_sched_barrier(0);

    float top[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        top[r] = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) top[r] = fmaxf(top[r], fabsf(__int_as_float(raw[r][i][j])));
        top[r] = wave_max(top[r]);
    }
    if constexpr (P > 1) {
        if (lane == 0) top_of[wave] = top[0];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < P; i++) top[0] = fmaxf(top[0], top_of[wave / P * P + i]);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t row = row0 + 8 * r;
        if (row >= M) continue;
        const float inv = top[r] == 0.0f ? 0.0f : __fdiv_rn(127.0f, top[r]);
        if (lane == 0) {
            scale_of[row] = top[r] == 0.0f ? 1.0f : __fdiv_rn(top[r], 127.0f);
            // zeros as such: in a row of 1e-37 `inv` is an infinity, and its product with a zero no number
            for (uint32_t kk = K; kk < steps * 64; kk += 16) *reinterpret_cast<v4i*>(xs + row * pitch + kk) = v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const uint32_t kk = k0 + i * 256 + lane * 4;
            const float4 v = make_float4(__int_as_float(raw[r][i][0]), __int_as_float(raw[r][i][1]), __int_as_float(raw[r][i][2]), __int_as_float(raw[r][i][3]));
            if (kk < K) *reinterpret_cast<uint32_t*>(xs + row * pitch + kk) = pack_i8x4(v, inv);
        }
    }
    __syncthreads();

    // ---- the product
    const int8_t* const a_at = xs + min(c, M - 1) * pitch + 16 * q;    // rows past M: the last one again, not stored
    v4i acc = {0, 0, 0, 0};
    uint32_t group = blockIdx.x, chunk = 0, set = 0;
    // after the barrier a wave adds up registers wave + 8 j of the group's 4 a tile: j = 0, and 1 and 1 to 3 for two and one waves a tile
    const auto scales = buffer(sw, N * 4), shifts = buffer(bias ? bias : sw, bias ? N * 4 : 0);
    float swc[4], bc[4];
    auto column = [&](uint32_t j) { return 16 * (group * at_once + ((wave + 8 * j) >> 2)) + c; };
    // the weights in `buf`; false when they were the last
    auto item = [&](auto buf, auto other) __attribute__((always_inline)) {
        const bool last = chunk + 1 == chunks;
        if (chunk == 0) {                                          // behind this group's weights, ahead of the next one's
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t col = 4 * column(j);                // (past N: 0)
                swc[j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(scales, (int)col, 0, 0));
                bc[j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(shifts, (int)col, 0, 0));
            }
        }
        fetch(other, last ? group + gridDim.x : group, last ? 0 : chunk + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (8 * chunk + i < mine)
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const v4i*>(a_at + 64 * (first + 8 * chunk + i)), b[decltype(buf)::value][i], acc, 0, 0, 0);
        if (!last) {
            chunk++;
            return true;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) part[set][wave][r][lane] = acc[r];
        __syncthreads();
        // register r of lane l: row 4 (l / 16) + r, column l % 16
        const uint32_t r = wave & 3, row = 4 * q + r;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint32_t t = (wave + 8 * j) >> 2, col = column(j);
            if (t >= at_once) break;
            if (row >= M || col >= N) continue;
            int32_t v = 0;
            for (uint32_t w = 0; w < waves; w++) v += part[set][t * waves + w][r][lane];
            float f = __fmul_rn(__fmul_rn((float)v, scale_of[row]), swc[j]);
            if (bias) f = __fadd_rn(f, bc[j]);
            y[(uint64_t)row * N + col] = f;
        }
        acc = v4i{0, 0, 0, 0};
        set ^= 1;
        chunk = 0;
        group += gridDim.x;
        return group < groups;
    };
    while (item(B0{}, B1{}) && item(B1{}, B0{})) {}
}

// One or two rows against more than 512 column tiles of more than 3072 k keep the two launches: two columns a wave fill the chip evenly
// where these groups of tiles leave up to a third of it idle (us there and in one launch: 1 x 11008 x 11008 25.3, 26.4; 1 x 4080 x 11008 10.9, 11.5; 2 x
// 4096 x 10000 10.5, 11.2; but 1 x 3072 x 11008 9.1, 9.0; 1 x 8192 x 8192 14.4, 13.4; 3 x 4096 x 11008 12.2, 12.1).
// What the rows of a workgroup cost it in registers (64 for the rows of a wave) and in reads out of the L2 (a row is K * 4 bytes, and all
// workgroups read all of them) limits K by the rows.
static uint32_t i8_linear_max_k(uint32_t m) { return m <= 2 ? 16384 : m <= 4 ? 8192 : m <= 8 ? 4096 : m <= 16 ? 2048 : 0; }

static bool i8_linear_one_launch(uint32_t m, uint32_t k, uint32_t n) {
    return m > 0 && n > 0 && k <= i8_linear_max_k(m) && !(m <= 2 && n > 8192 && k > 3072);
}

// Waves of a column tile (1 << share) and workgroups, one per compute unit at most.  A round of the workgroups takes its waves' chunks of eight steps
// and, as long as 0.6 of one, the meeting of its tiles.  Few waves a tile leave no chunk half empty where K is short and make fewer rounds; where
// the tiles are few, eight.  One row from HBM, us with 8, 4 and 2 waves a tile: 768 x 10800 8.0, 6.3, 5.1; 2048 x 5504 6.5, 5.6, 6.7; 2048 x
// 11008 9.2, 7.4, 7.4; 4096 x 11008 11.3, 11.5, 10.8; 8192 x 8192 13.9, 13.5, 18.3; 3456 x 2240 5.1, 6.1, 9.5.  Two workgroups a compute
// unit are slower everywhere (4096 x 11008 14.1).
struct I8LinearSplit { uint32_t share, grid; };
static I8LinearSplit i8_linear_split(uint32_t k, uint32_t n) {
    const uint32_t tiles = ceil_div(n, 16), steps = ceil_div(k, 64);
    I8LinearSplit best{3, 1};
    uint64_t least = ~uint64_t(0);
    for (uint32_t share = 4; share-- > 0;) {
        const uint32_t groups = ceil_div(tiles, 8u >> share), rounds = ceil_div(groups, 256), chunks = ceil_div(ceil_div(steps, 1u << share), 8);
        const uint64_t cost = (uint64_t)rounds * (5 * chunks + 3);
        if (cost < least) { least = cost; best = I8LinearSplit{share, ceil_div(groups, rounds)}; }
    }
    return best;
}

template <int P, int R, int NV>
static int launch_i8_linear(const float* x, const int8_t* wq, const float* sw, const float* bias, float* y, uint32_t m, uint32_t k,
                            uint32_t n, hipStream_t s) {
    const I8LinearSplit z = i8_linear_split(k, n);
    hipLaunchKernelGGL((i8_linear_kernel<P, R, NV>), dim3(z.grid), dim3(512), (size_t)m * (ceil_div(k, 64) * 64 + 16), s, x, wq, sw, bias,
                       y, m, k, n, z.share);
    return check_launch("i8_linear_kernel");
}

}  // namespace rumus

using namespace rumus;

extern "C" {

uint64_t rumus_hip_i8_linear_scratch_size(uint32_t m, uint32_t k, uint32_t n) {
    return i8_linear_one_launch(m, k, n) ? 0 : (((uint64_t)m * k + 255) & ~uint64_t(255)) + 4 * (uint64_t)m;
}

int rumus_hip_i8_linear(const float* x, const int8_t* wq, const float* sw, const float* bias, void* scratch, float* y, uint32_t m,
                        uint32_t k, uint32_t n, rumus_hip_stream_t stream) {
    RUMUS_REQUIRE(k > 0 && k % 16 == 0, "i8_linear: k must be a positive multiple of 16 (got %u)", k);
    if (m == 0 || n == 0) return RUMUS_HIP_OK;
    RUMUS_REQUIRE(x && wq && sw && y, "i8_linear: null operand");
    RUMUS_REQUIRE((reinterpret_cast<uintptr_t>(wq) & 15) == 0, "i8_linear: operands must be 16-byte aligned");
    hipStream_t s = as_stream(stream);
    if (!i8_linear_one_launch(m, k, n)) {
        RUMUS_REQUIRE(scratch, "i8_linear: null scratch");
        int8_t* const xq = static_cast<int8_t*>(scratch);
        float* const sx = reinterpret_cast<float*>(xq + (((uint64_t)m * k + 255) & ~uint64_t(255)));
        if (int rc = rumus_hip_i8_quantize_rows(x, xq, sx, m, k, stream)) return rc;
        return rumus_hip_i8_gemm(xq, wq, sx, sw, bias, nullptr, y, m, k, n, stream);
    }
#define RUMUS_I8_LINEAR(P, R, NV) return launch_i8_linear<P, R, NV>(x, wq, sw, bias, y, m, k, n, s)
    const uint32_t by2048 = ceil_div(k, 2048);
    if (m == 1) {
        if (by2048 <= 2) RUMUS_I8_LINEAR(8, 1, 2);
        if (by2048 <= 4) RUMUS_I8_LINEAR(8, 1, 4);
        RUMUS_I8_LINEAR(8, 1, 8);
    }
    if (m == 2) {
        if (by2048 <= 2) RUMUS_I8_LINEAR(4, 1, 4);
        if (by2048 <= 4) RUMUS_I8_LINEAR(4, 1, 8);
        RUMUS_I8_LINEAR(4, 1, 16);
    }
    if (m <= 4) {
        if (by2048 <= 1) RUMUS_I8_LINEAR(2, 1, 4);
        if (by2048 <= 2) RUMUS_I8_LINEAR(2, 1, 8);
        RUMUS_I8_LINEAR(2, 1, 16);
    }
    if (m <= 8) {
        if (k <= 1024) RUMUS_I8_LINEAR(1, 1, 4);
        if (by2048 <= 1) RUMUS_I8_LINEAR(1, 1, 8);
        RUMUS_I8_LINEAR(1, 1, 16);
    }
    if (k <= 1024) RUMUS_I8_LINEAR(1, 2, 4);
    RUMUS_I8_LINEAR(1, 2, 8);
#undef RUMUS_I8_LINEAR
}

}  // extern "C"
