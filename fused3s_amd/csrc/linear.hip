// linear.hip -- Y = X W^T + b in binary16 with float32 sums, for the
// projections around the fused pass: many rows (nodes), few inputs and
// outputs per row.
//
// Such a product is bound by the rows it reads and writes, not by the matrix
// cores (128 inputs, 384 outputs: 96 flops per byte), so W is laid out once
// per workgroup in LDS, in the order the MFMA operands are read, and each wave
// streams blocks of 16 rows past it: a row block's operands are loaded straight
// into registers, one block ahead of the products.  W is the A operand, its
// rows dealt to the tiles so that a lane holds eight consecutive outputs of one
// row (two 16x16 tiles side by side): no transpose on the way out.  Two such
// pieces go through a small stage so that whole 128-byte lines are stored
// (500,000 x 128 -> 384: 138 us with 64-byte stores, 111 us so, 4.6 TB/s, and
// 193 us in the library; non-temporal stores 92 us, but the fused pass then
// finds nothing of its Q, K and V in the caches: layer 627 against 635 us).
// 32 rows per wave, halving the LDS reads, changed nothing: they do not bound it.
#include <algorithm>

#include "attn_common.hpp"

namespace f3s {

struct LinearParams {
    const _Float16* X;
    const _Float16* W;
    const _Float16* bias;   // NULL: none
    _Float16* Y;
    int64_t n;
    int32_t K, M;
    int32_t cols;           // outputs per workgroup (blockIdx.y), a multiple of 32
};

// KF: operand fragments of 32 inputs per row (K <= 32 KF).  NW waves share one
// copy of `cols` rows of W: cols * KF * 4 <= PIECES.
template <int KF, int NW, int PIECES>
__global__ void __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(4)))
linear_kernel(const LinearParams p)
{
    __shared__ __align__(16) h8 wl[PIECES];
    __shared__ __align__(16) _Float16 bl[PIECES / (4 * KF)];
    // (four waves: a stage would cost a workgroup per CU)
    constexpr bool kStaged = NW > 4;
    __shared__ __align__(16) _Float16 stage[kStaged ? NW : 1][kStaged ? 16 * kStageRow : 8];
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int g = lane >> 4, r = lane & 15;
    const int32_t m0 = blockIdx.y * p.cols;
    const int32_t mc = min(p.cols, p.M - m0);   // a multiple of 32
    const h8 zero = {};

    // W in operand order: piece (((pair * 2 + t) * KF + f) * 64 + l) is what
    // lane l supplies for fragment f of tile t of that pair of tiles
    for (int i = tid; i < mc * KF * 4; i += NW * kWave) {
        const int l = i & 63, f = (i >> 6) % KF, tile = (i >> 6) / KF;
        const int row = l & 15;
        const int col = (tile >> 1) * 32 + 8 * (row >> 2) + 4 * (tile & 1) + (row & 3);
        const int k = 32 * f + 8 * (l >> 4);
        wl[i] = k < p.K ? *reinterpret_cast<const h8*>(p.W + (int64_t)(m0 + col) * p.K + k) : zero;
    }
    for (int i = tid; i < mc; i += NW * kWave) bl[i] = p.bias ? p.bias[m0 + i] : (_Float16)0.f;
    __syncthreads();

    const int64_t blocks = (p.n + 15) >> 4, step = (int64_t)gridDim.x * NW;
    int64_t b = (int64_t)blockIdx.x * NW + wave;
    if (b >= blocks) return;
    auto load = [&](int64_t blk, h8 (&x)[KF]) __attribute__((always_inline)) {
        const int64_t row = min(blk * 16 + r, p.n - 1);   // (past the end: not stored)
        const _Float16* src = p.X + row * p.K + 8 * g;
#pragma unroll
        for (int f = 0; f < KF; ++f)
            x[f] = 32 * f + 8 * g < p.K ? *reinterpret_cast<const h8*>(src + 32 * f) : zero;
    };
    h8 x[KF], nx[KF];
    // outputs c + 8 g .. + 7 of row r of the block
    auto product = [&](int32_t c) __attribute__((always_inline)) -> h8 {
        const h8* w = wl + (c >> 5) * (2 * KF * 64) + lane;
        const h8 bias = *reinterpret_cast<const h8*>(&bl[c + 8 * g]);
        f4 a0 = {(float)bias[0], (float)bias[1], (float)bias[2], (float)bias[3]};
        f4 a1 = {(float)bias[4], (float)bias[5], (float)bias[6], (float)bias[7]};
#pragma unroll
        for (int f = 0; f < KF; ++f) {
            a0 = mfma16x16x32(w[f * 64], x[f], a0);
            a1 = mfma16x16x32(w[(KF + f) * 64], x[f], a1);
        }
        const h4 y0 = __builtin_convertvector(a0, h4), y1 = __builtin_convertvector(a1, h4);
        return h8{y0[0], y0[1], y0[2], y0[3], y1[0], y1[1], y1[2], y1[3]};
    };
    _Float16* out = stage[kStaged ? wave : 0];
    load(b, x);
    for (; b < blocks; b += step) {
        if (b + step < blocks) load(b + step, nx);
        int32_t c = 0;
        for (; kStaged && c + 64 <= mc; c += 64) {
            // 16 rows of 128 bytes through the stage, stored eight whole lines at a time
            *reinterpret_cast<h8*>(&out[r * kStageRow + 8 * g]) = product(c);
            *reinterpret_cast<h8*>(&out[r * kStageRow + 32 + 8 * g]) = product(c + 32);
            wave_lds_order();
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const int rr = 8 * v + (lane >> 3);
                const h8 y = *reinterpret_cast<const h8*>(&out[rr * kStageRow + 8 * (lane & 7)]);
                const int64_t row = b * 16 + rr;
                if (row < p.n)
                    *reinterpret_cast<h8*>(p.Y + row * p.M + m0 + c + 8 * (lane & 7)) = y;
            }
            wave_lds_order();
        }
        for (; c < mc; c += 32) {
            const h8 y = product(c);
            if (b * 16 + r < p.n)
                *reinterpret_cast<h8*>(p.Y + (b * 16 + r) * p.M + m0 + c + 8 * g) = y;
        }
#pragma unroll
        for (int f = 0; f < KF; ++f) x[f] = nx[f];
    }
}

// Many rows: 16 waves share up to 96 KB of W and read X once per 96 KB of it
// (64,000 x 128 -> 1,536: 43 us, 66 by fours, 63 in the library).
// Fewer: 4 waves and 32 KB, more workgroups (50,000 x 128 -> 384: 19 us, 26 in
// the library; 2,708 x 128 -> 192: 5.2 and 4.6, with half the host time).
constexpr int kBigPieces = 6144, kSmallPieces = 2048;
constexpr int64_t kBigRows = 48 * 1024;

template <int KF>
static f3s_status launch_linear(LinearParams p, int cus, hipStream_t st)
{
    const bool big = p.n >= kBigRows;
    const int32_t most = (big ? kBigPieces : kSmallPieces) / (4 * KF) / 32 * 32;
    const int32_t ny = (int32_t)ceil_div(p.M, most);
    const int32_t unit = p.M % 64 == 0 && most % 64 == 0 ? 64 : 32;   // whole lines where M allows
    p.cols = (int32_t)ceil_div(ceil_div(p.M, ny), unit) * unit;
    const int nw = big ? 16 : 4;
    const int64_t need = ceil_div(ceil_div(p.n, 16), nw);
    // as many workgroups as are resident at once (one per CU, or four)
    const int64_t nx = std::max<int64_t>(1, std::min<int64_t>(need, (big ? 1 : 4) * cus / ny));
    if (big)
        hipLaunchKernelGGL((linear_kernel<KF, 16, kBigPieces>), dim3((unsigned)nx, (unsigned)ny),
                           dim3(16 * kWave), 0, st, p);
    else
        hipLaunchKernelGGL((linear_kernel<KF, 4, kSmallPieces>), dim3((unsigned)nx, (unsigned)ny),
                           dim3(4 * kWave), 0, st, p);
    F3S_HIP(hipGetLastError());
    return F3S_OK;
}

__global__ void warm_linear_kernel() {}

hipError_t warm_linear(hipStream_t s)
{
    hipLaunchKernelGGL(warm_linear_kernel, dim3(1), dim3(64), 0, s);
    return hipGetLastError();
}

}  // namespace f3s

extern "C" f3s_status f3s_linear_f16(const uint16_t* X, const uint16_t* W, const uint16_t* bias,
                                     uint16_t* Y, int64_t n, int32_t K, int32_t M, void* stream)
{
    using namespace f3s;
    F3S_REQUIRE(n >= 0 && K >= 1 && M >= 1, "f3s_linear_f16: bad size");
    if (K % 8 != 0 || K > 256 || M % 32 != 0 || M > 32768 || n >= ((int64_t)1 << 35)) {
        set_error("f3s_linear_f16: needs K a multiple of 8 up to 256 and M a multiple of 32 up "
                  "to 32768");
        return F3S_EUNSUPPORTED;
    }
    if (n == 0) return F3S_OK;
    F3S_REQUIRE(X && W && Y, "f3s_linear_f16: NULL pointer");
    F3S_REQUIRE(((((uintptr_t)X) | ((uintptr_t)W) | ((uintptr_t)Y)) & 15) == 0,
                "f3s_linear_f16: X, W and Y must be 16-byte aligned");
    F3S_TRY(require_device());
    clear_error();
    int dev = 0, cus = 0;
    F3S_HIP(hipGetDevice(&dev));
    F3S_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    LinearParams p{reinterpret_cast<const _Float16*>(X), reinterpret_cast<const _Float16*>(W),
                   reinterpret_cast<const _Float16*>(bias), reinterpret_cast<_Float16*>(Y),
                   n, K, M, 0};
    hipStream_t st = as_stream(stream);
    if (K <= 64) return launch_linear<2>(p, cus, st);
    if (K <= 128) return launch_linear<4>(p, cus, st);
    return launch_linear<8>(p, cus, st);
}
