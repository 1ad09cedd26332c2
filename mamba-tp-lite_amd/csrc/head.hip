// The tied lm_head of a decode step at up to 16 rows (gfx950):
//   Y[m, n] = sum_k x[m, k] W[n, k],   m < M <= 16, n < N >> M
// (model.py:326, 353), fp32 or bf16.
//
// A [50280, 2048] fp32 embedding is 412 MB for a few rows of x: the product
// is a stream of W through the chip.  The library's GEMM tiles it at 4.4-4.9
// TB/s (84-94 us at 5 rows), and the skinny GEMM of linear.hip, which copies x
// through LDS beside every 16 rows of W, was slower (93-126 us).  Here nothing
// but W moves: one workgroup of 8 wavefronts per CU walks many 16-row tiles of
// W; wavefront w owns the w-th eighth of K and keeps x's part of it in
// registers as matrix operands for the whole launch, and streams W from
// global memory straight into registers, the next half tile in flight while
// the present one is multiplied.  Lane l = r + 16 kk takes the 16-byte chunk
// kk of row r of a 16-row, 64-byte-wide block: 4 v_mfma_f32_16x16x4_f32 (or
// one v_mfma_f32_16x16x32_bf16) per block.  The eight partial tiles are added
// in wavefront order through LDS (deterministic).  Tile t of workgroup b is
// t gridDim + b: the chip reads one contiguous stretch of W at a time.
//
// [50280, 2048], cold weights, 5 rows: fp32 84-87 -> 75 us (5.5 TB/s), bf16
// 45-50 -> 41 us.  With 32 rows of x (2 x 16) it was level with the library
// (98 / 92-99 us), with narrower rows of W behind it (768 columns fp32, 16
// rows: 38 / 32 us): mtl_lm_head_ok leaves those to it.  2 and 4 workgroups
// per CU were slower (77, 83 us).

#include "common.h"

namespace mtl {
namespace {

typedef __bf16 B8h __attribute__((ext_vector_type(8)));

constexpr int kHeadWaves = 8;

template <typename T>
struct HeadArgs {
    const T* x;        // [M, K] contiguous
    const T* W;        // [N, K] contiguous
    T* y;              // [M, N] contiguous
    int M, N;
};

// NC: 64-byte blocks of a wavefront's K range, K = 8 NC 64 bytes
template <typename T, int NC>
__global__ void __launch_bounds__(kHeadWaves * 64, 2) head_kernel(const HeadArgs<T> a) {
    constexpr int BC = 64 / (int)sizeof(T);              // columns of a block
    constexpr int K = kHeadWaves * NC * BC;
    constexpr int NA = (NC + 1) / 2, NB = NC - NA;       // blocks of the two halves of a tile
    __shared__ __align__(16) F4v s_part[2][kHeadWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, kk = lane >> 4;
    const int tiles = (a.N + 15) / 16, k0 = wave * NC * BC + kk * (BC / 4);

    F4v xv[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        xv[c] = *reinterpret_cast<const F4v*>(a.x + (int64_t)min(r, a.M - 1) * K + k0 + c * BC);

    auto load = [&](F4v* w, int tile, int c0, int n) __attribute__((always_inline)) {
        const T* p = a.W + (int64_t)min(tile * 16 + r, a.N - 1) * K + k0 + c0 * BC;
#pragma unroll
        for (int c = 0; c < n; ++c) w[c] = __builtin_nontemporal_load(reinterpret_cast<const F4v*>(p + c * BC));
    };
    F4v acc[2];                                          // two chains, added at the end of a tile
    auto mma = [&](const F4v* w, int c0, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < n; ++c) {
            if constexpr (sizeof(T) == 2) {
                acc[c & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(B8h, w[c]), __builtin_bit_cast(B8h, xv[c0 + c]), acc[c & 1], 0, 0, 0);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[c][q], xv[c0 + c][q], acc[q & 1], 0, 0, 0);
            }
        }
    };

    F4v wa[NA], wb[NB];
    int t = blockIdx.x, buf = 0;
    if (t < tiles) load(wa, t, 0, NA);
    for (; t < tiles; t += gridDim.x, buf ^= 1) {
        acc[0] = acc[1] = F4v{0.f, 0.f, 0.f, 0.f};
        load(wb, t, NA, NB);
        __builtin_amdgcn_sched_barrier(0);
        mma(wa, 0, NA);
        __builtin_amdgcn_sched_barrier(0);
        // (past the end it reads the last tile again rather than branch around the loads)
        load(wa, min(t + (int)gridDim.x, tiles - 1), 0, NA);
        __builtin_amdgcn_sched_barrier(0);
        mma(wb, NA, NB);
        s_part[buf][wave][lane] = acc[0] + acc[1];
        // one barrier per tile: the other buffer's reader is past it when its writers return to it
        __syncthreads();
        if (wave == 0) {
            F4v sum = s_part[buf][0][lane];
#pragma unroll
            for (int w = 1; w < kHeadWaves; ++w) sum += s_part[buf][w][lane];
            // D[i][j]: row j = lane % 16 of x, W rows 4 (lane / 16) .. + 3
            const int n = t * 16 + 4 * kk;
            if (r < a.M && n < a.N) st4(a.y + (int64_t)r * a.N + n, sum);
        }
    }
}

template <typename T>
int head(const void* x, const void* W, void* y, int64_t M, int64_t N, int nc, int grid, hipStream_t st) {
    const HeadArgs<T> a{static_cast<const T*>(x), static_cast<const T*>(W), static_cast<T*>(y), (int)M, (int)N};
    switch (nc) {
#define MTL_NC(V) case V: hipLaunchKernelGGL((head_kernel<T, V>), dim3(grid), dim3(kHeadWaves * 64), 0, st, a); break;
        MTL_NC(8) MTL_NC(9) MTL_NC(10) MTL_NC(11)
        MTL_NC(12) MTL_NC(13) MTL_NC(14) MTL_NC(15) MTL_NC(16)
#undef MTL_NC
    }
    return check_launch("lm_head");
}

}  // namespace
}  // namespace mtl

// 64-byte blocks of K per wavefront where the kernel takes the sizes, else 0
static int head_blocks(int64_t M, int64_t N, int64_t K, int32_t dtype) {
    if (dtype != MTL_F32 && dtype != MTL_BF16) return 0;
    const int64_t unit = mtl::kHeadWaves * 64 / (dtype == MTL_F32 ? 4 : 2);
    if (M < 1 || M > 16 || N < 4 || N % 4 != 0 || N >= (int64_t(1) << 27) || K % unit != 0 || K < 8 * unit ||
        K > 16 * unit)
        return 0;
    return (int)(K / unit);
}

extern "C" int mtl_lm_head_ok(int64_t M, int64_t N, int64_t K, int32_t dtype) {
    // (N: at least 8 tiles for each of 256 CUs)
    return N >= 32768 && head_blocks(M, N, K, dtype) ? 1 : 0;
}

extern "C" int mtl_lm_head(const void* x, const void* W, void* y, int64_t M, int64_t N, int64_t K, int32_t dtype,
                           mtl_stream_t stream) {
    using namespace mtl;
    clear_error();
    MTL_REQUIRE(dtype == MTL_F32 || dtype == MTL_BF16, "dtype must be MTL_F32 or MTL_BF16");
    const int nc = head_blocks(M, N, K, dtype);
    MTL_REQUIRE(nc > 0, "M in [1, 16], N a multiple of 4 below 2^27, K a multiple of 128 in [1024, 2048] (bf16: of "
                        "256 in [2048, 4096])");
    MTL_REQUIRE(x && W && y, "null pointer");
    MTL_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(y)) % 16 == 0,
                "x, W and y must be 16-byte aligned");
    hipStream_t st = as_stream(stream);
    int dev = 0, cus = 0;
    if (hipStreamGetDevice(st, &dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
        set_error("device query failed");
        return MTL_EHIP;
    }
    const int grid = (int)std::min<int64_t>((N + 15) / 16, cus);
    return dtype == MTL_F32 ? head<float>(x, W, y, M, N, nc, grid, st) : head<uint16_t>(x, W, y, M, N, nc, grid, st);
}
