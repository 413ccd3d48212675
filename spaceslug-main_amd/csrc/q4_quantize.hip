// fp32 -> int4 group-32 quantizer that writes the packed weight layout the
// GEMM/GEMV kernels read (q4gemm.comp:7-19: uint8[N][K/2], even k in the low
// nibble, two's-complement nibbles; float[N][K/32] scales).
//
// Rule, per column n and group g (32 consecutive k):
//   m     = the value of largest magnitude among w[32g .. 32g+31][n] (the first
//           one in k order when several share that magnitude);
//   scale = -m / 8                          (exact: a power-of-two division);
//   v_k   = clamp(rint(w_k / scale), -8, 7) (IEEE division, round to nearest
//           even), 0 for every k when scale == 0.
// The extreme value maps to -8 exactly; a value of the opposite sign and the
// same magnitude maps to +8 and is clamped to 7. A group holding a NaN or an
// infinity gets a NaN scale and zero nibbles (the host entry point rejects
// non-finite input before that).
//
// Bound by memory (4 bytes read and 0.625 written per weight) once these are out of the way:
//   - stores: a thread quantizes one (column, group), the 64 lanes of a wavefront 64 consecutive
//     columns of one group, so every read of w[k][n0 .. n0+63] is one coalesced 256-byte row
//     segment, but the 16 packed bytes and the scale it produces lie a column apart. A workgroup
//     takes GW consecutive groups of its columns, collects them in LDS and stores GW * 16 and GW * 4
//     contiguous bytes per column (whole 128-byte lines of packed weights at GW = 8);
//   - divisions: 32 IEEE divisions per thread were most of the kernel's VALU time (~30 us per SIMD of
//     the 60 us a 4096 x 14336 matrix took). rint(w / scale) equals rint(w * (1 / scale)) unless the
//     product lies within their errors of a tie, so a thread divides only if one of its values does
//     (quantize_group);
//   - rows read through several L2s: workgroups go to the XCDs in turn, so neighbouring column blocks,
//     which share lines when N is no multiple of 32, are put on one XCD (a run of blocks each).
// 4096 x 14336 (k x n) 68.5 -> 48.6 us (5.6 TB/s), 2880 x 11001 51.1 -> 29.2, 1024 x 1000 3.8 -> 3.7.
#include "q4_device.hpp"
#include "q4_kernels.hpp"

namespace spaceslug {
namespace {

// clamp(rint(v / scale), -8, 7) of 32 values as packed words, with IEEE division.
__device__ void quantize_group_divide(const float (&v)[32], float scale, uint32_t (&words)[4]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        words[w] = 0u;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float r = rintf(v[8 * w + t] / scale);
            const int q = static_cast<int>(fminf(fmaxf(r, -8.0f), 7.0f));
            words[w] |= (static_cast<uint32_t>(q) & 0xFu) << (4 * t);
        }
    }
}

// The same through one reciprocal. |v / scale| <= 8; inv = 1 / scale and v * inv carry a relative
// error of 2^-24 each, so the product is within 8 * 2^-23 of v / scale, as is the rounded quotient
// (2^-24): farther than 1.5e-6 from a tie both round to the same integer. Magnitudes whose scale or
// reciprocal would leave the normal range divide.
__device__ __forceinline__ void quantize_group(const float (&v)[32], float m, float scale, uint32_t (&words)[4]) {
    const float inv = 1.0f / scale;
    float frac = 0.0f;  // largest distance from an integer
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t half[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float sum = 0.0f;  // base-16 digits q + 8, most significant first: below 2^16, exact
#pragma unroll
            for (int t = 3; t >= 0; --t) {
                const float x = v[8 * w + 4 * h + t] * inv;
                const float r = rintf(x);
                frac = fmaxf(frac, fabsf(x - r));
                sum = fmaf(sum, 16.0f, __builtin_amdgcn_fmed3f(r, -8.0f, 7.0f) + 8.0f);
            }
            half[h] = static_cast<uint32_t>(sum);
        }
        words[w] = (half[0] | (half[1] << 16)) ^ 0x88888888u;  // (q + 8) xor 8 is q's two's-complement nibble
    }
    const float mag = fabsf(m);
    if (!(frac < 0.5f - 1.5e-6f) || mag < 0x1p-100f || mag > 0x1p100f) quantize_group_divide(v, scale, words);
}

// A workgroup of CW * GW wavefronts takes 64 CW columns of GW groups. STREAM: w is read past the caches.
template <int CW, int GW, bool STREAM>
__global__ __launch_bounds__(64 * CW * GW) void q4_quantize_kernel(const float* __restrict__ w, u32x4* __restrict__ packed,
                                                                   float* __restrict__ scales, int N, int K, int blocks_n,
                                                                   int blocks) {
    constexpr int kCols = 64 * CW;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int cw = wave % CW, gw = wave / CW;
    const int run = (blocks + 7) >> 3;
    const int lin = static_cast<int>(blockIdx.x & 7) * run + static_cast<int>(blockIdx.x >> 3);
    if (lin >= blocks) return;
    const int n0 = (lin % blocks_n) * kCols, g0 = (lin / blocks_n) * GW;
    const int G = K >> 5;
    const int col = n0 + 64 * cw + lane;
    const int n = min(col, N - 1);         // lanes past the last column repeat it and store nothing
    const int g = min(g0 + gw, G - 1);     // as do wavefronts past the last group
    const float* src = w + static_cast<size_t>(g) * 32 * N + n;
    float v[32];
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        const float* at = src + static_cast<size_t>(t) * N;
        v[t] = STREAM ? __builtin_nontemporal_load(at) : *at;
    }
    float m = v[0], probe = 0.0f * v[0];
#pragma unroll
    for (int t = 1; t < 32; ++t) {
        m = fabsf(v[t]) > fabsf(m) ? v[t] : m;
        probe = fmaf(v[t], 0.0f, probe);  // NaN if any value is not finite
    }
    float scale = -m * 0.125f;
    uint32_t words[4] = {0u, 0u, 0u, 0u};
    if (__builtin_isnan(probe)) {
        scale = __builtin_nanf("");
    } else if (scale == 0.0f) {
        scale = 0.0f;  // also turns -0 into +0
    } else {
        quantize_group(v, m, scale, words);
    }
    const u32x4 out = {words[0], words[1], words[2], words[3]};
    __shared__ u32x4 pk[GW][kCols + 1];  // one column of padding: a column's groups then lie in distinct banks
    __shared__ float sc[GW][kCols + 1];
    pk[gw][64 * cw + lane] = out;
    sc[gw][64 * cw + lane] = scale;
    __syncthreads();
    const int c = threadIdx.x / GW, gi = threadIdx.x % GW;
    if (n0 + c < N && g0 + gi < G) {
        const size_t at = static_cast<size_t>(n0 + c) * G + g0 + gi;
        packed[at] = pk[gi][c];
        scales[at] = sc[gi][c];
    }
}

}  // namespace

hipError_t launch_q4_quantize(const float* w, uint8_t* w_packed, float* w_scales, uint32_t n, uint32_t k,
                              hipStream_t stream) {
    const uint32_t groups = k / kGroup;
    auto go = [&](auto cw, auto gw, auto stream_c) {
        constexpr uint32_t CW = decltype(cw)::value, GW = decltype(gw)::value;
        const uint32_t blocks_n = (n + 64 * CW - 1) / (64 * CW), blocks = blocks_n * ((groups + GW - 1) / GW);
        hipLaunchKernelGGL((q4_quantize_kernel<CW, GW, decltype(stream_c)::value>), dim3((blocks + 7) / 8 * 8),
                           dim3(64 * CW * GW), 0, stream, w, reinterpret_cast<u32x4*>(w_packed), w_scales,
                           static_cast<int>(n), static_cast<int>(k), static_cast<int>(blocks_n),
                           static_cast<int>(blocks));
        return hipGetLastError();
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    using I8 = std::integral_constant<int, 8>;
    // More than half of the 256 MB last-level cache: such a matrix is not found there, and reading it past the
    // caches leaves them to the stores (4096 x 14336: 48.6 against 58.4 us; 2880 x 11001, 127 MB, 34.5 against 30.2).
    const bool stream_w = static_cast<uint64_t>(n) * k > (uint64_t{1} << 25);
    // Fewer than eight groups: no wavefronts for groups that are not there (and with two per workgroup the
    // largest grids stay below 2^32 threads).
    if (groups < 8) return stream_w ? go(I1{}, I2{}, std::true_type{}) : go(I1{}, I4{}, std::false_type{});
    if (stream_w) return go(I2{}, I8{}, std::true_type{});
    // Few wavefronts: smaller workgroups spread wider (1024 x 1000 3.7 against 3.9 us; 3008 x 3000 9.5 against 9.4).
    const uint64_t waves = static_cast<uint64_t>((n + 63) / 64) * groups;
    return waves < 3000 ? go(I1{}, I4{}, std::false_type{}) : go(I1{}, I8{}, std::false_type{});
}

}  // namespace spaceslug
