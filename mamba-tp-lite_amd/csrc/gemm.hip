// fp32 GEMM for the projections of a long prompt on the f16 matrix cores
// (gfx950):   Y[m, n] = sum_k X[m, k] W[n, k] (+ bias[n]),   fp32 in and out.
//
// The projections of a prefill (in_proj, out_proj: model.py:197, 240; the
// tied lm_head: model.py:339) are compute-bound fp32 products, and the fp32
// matrix instructions run at 1/16 of the f16 ones (154 against 1470 TFLOP/s
// measured on 8192^3 library products).  Every fp32 value is therefore split
// into two f16 parts,
//   x 2^e = hi + lo,   hi = f16(x 2^e),  lo = f16(x 2^e - hi),
// with one power of two 2^e per row (of X and of W) that puts the row's
// largest magnitude in [2^14, 2^15).  hi + lo holds 22 significand bits of
// every element down to 2^-17 of its row's largest, and an absolute 2^-40 of
// that largest below it.  A product takes three MFMAs,
//   x w = lo_x hi_w + hi_x lo_w + hi_x hi_w   (lo lo, under 2^-22 of the product, is left out),
// all accumulated in fp32, and the epilogue multiplies by 2^-(e_x + e_w)
// (exact).  The dropped and rounded parts are ~2^-24 of each product, as
// fp32's own rounding is, and the fp32 accumulator is rounded 3 times per 16
// columns in place of 16, so the result is closer to the exact product than
// the fp32 matrix path's (tests/test_gpu_gemm.py).
//
// Operand layout (split_rows_kernel writes it): blocks of 64 rows, in them
// 16-column panels,
//   [rows / 64][K / 16][64][64 bytes],  a row's 64 bytes = hi of columns 0-7,
//   lo of 0-7, hi of 8-15, lo of 8-15 of the panel (K padded to 32 columns
//   with zeros; the rows past the last are never written and never used),
// so a stage of the GEMM -- a panel or two of a tile's rows -- is a few
// contiguous 4 KB runs, a tile's whole operand lies in one stretch of memory,
// and a split row takes exactly the bytes of its fp32 values.
//
// Three kinds of rows are not split (split_ok):
//   * a row that holds an infinity or NaN;
//   * a row of great spread, more than 1/16 of whose nonzero values lie under
//     2^-20 of its largest: those keep under 20 bits, and where the other
//     operand is zero or small at the large ones the product shows it (K 768,
//     one value 2^20 times the rest against a zero weight: 7.9e-7 split, 5.0e-7
//     fp32; at 2^17 and below 2.4e-7 split).  Gaussian rows have 1e-5 of their
//     values there, gated y rows up to a few percent;
//   * a row of fewer than 32 nonzero values, whose fp32 sums round so little
//     that 22 bits per operand would be the larger error (a row that selects
//     one column is exact in fp32).
// The exponent of such a row is marked, and the epilogue computes the outputs that touch it from the fp32
// operands on the fp32 matrix instructions, so infinities and NaN come out as
// an fp32 product gives them.  Measured, us, no row / one row of x / every row
// marked (library fp32 product): 4096 x 3072 x 768 72 / 128 / 362 (162), 1024 x
// 8192 x 2048 121 / 249 / 572 (265), 32768 x 3072 x 768 424 / 483 / 2610 (1107);
// a lane's own sum over K per output took hundreds of products' time.
//
// Measured (us; library fp32 GEMM -> this product, plus the splits of X and W):
//   32768 x 3072 x 768 (mamba-130m in_proj, 32 x 1024 tokens)   1246 -> 449 + 41
//   32768 x 768 x 1536 (its out_proj)                            554 -> 215 + 73
//   1024 x 8192 x 2048 (mamba-1.4b in_proj, 1024 tokens)         240 -> 94 + 34
//   1024 x 2048 x 4096 (its out_proj)                            119 -> 66 + 21
//   999 x 50280 x 768 (the tied lm_head)                         700 -> 224 + 52
// at 250 to 392 TFLOP/s of fp32 product, 3 MFMAs each: 0.75 to 1.18 PFLOP/s of
// the 1.47 that the library reaches on an 8192^3 f16 product.  The relative
// error against 64 bits (2-norm) falls from 5.0e-7 to 3.1e-7 at K = 768,
// 8.1e-7 to 5.0e-7 at 2048 and 1.15e-6 to 7.1e-7 at 4096.  With the
// conversion inside the product's loop (fp32 tiles in LDS, no split pass) the
// 1024 x 8192 x 2048 product took 147 us in place of 100 + 42.

#include <type_traits>

#include "common.h"
#include "gemm.h"

namespace mtl {
namespace {

typedef _Float16 H8 __attribute__((ext_vector_type(8)));
typedef float F16v __attribute__((ext_vector_type(16)));

constexpr int kPanel = 16;                 // columns of a panel
constexpr int kPanelBytes = 64;            // bytes of a row in it
constexpr int kRowBlock = 64;              // rows of a block
constexpr int kExpSpecial = 1 << 20;       // exponent mark of a row that cannot be split

// ------------------------------------------------------------------ splitting
// One workgroup takes 16 rows: lane = (row of 16, 8-column block of 4), so a
// wavefront reads whole 128-byte runs of 16 rows and writes 1 KB runs of two
// panels; the wavefronts take 32-column units in turn.  Each row's largest
// |x| is found first (bit patterns, so a NaN is the largest), then the parts
// are written.
constexpr int kSplitRows = 16;

__device__ __forceinline__ void load8(const float* p, int n, bool vec, float* v) {
    if (vec && n >= 8) {
        const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = j < n ? p[j] : 0.f;
    }
}

// Whether a row's split holds it as well as fp32 does, from its largest
// magnitude's bits and its counts over `cols` values: those that are not zero,
// and those under 2^-20 of the largest.
struct RowCount {
    float below;                           // 2^-20 of the largest (0 where that is no normal number: none is small)
    int nonzero = 0, small = 0;
    __device__ __forceinline__ explicit RowCount(uint32_t mx)
        : below(mx >= (21u << 23) ? __uint_as_float(mx - (20u << 23)) : 0.f) {}
    __device__ __forceinline__ void add(float v) {
        nonzero += v != 0.f;
        small += fabsf(v) < below;         // (zeros too)
    }
};
__device__ __forceinline__ bool split_ok(int nonzero, int small, int cols) {
    small -= small ? cols - nonzero : 0;   // without the zeros (all or none of them were counted)
    return (int64_t)small * 16 <= nonzero && (nonzero >= 32 || nonzero == 0);
}

// the power of two of a row whose largest magnitude has the bits `mx`
__device__ __forceinline__ int split_exp(uint32_t mx) {
    if (mx >= 0x7f800000u) return kExpSpecial;
    // (a zero or subnormal row takes the largest scale, 2^126)
    return min(14 - ((int)(mx >> 23) - 127), 126);
}

// 8 columns of a row into its hi and lo parts
__device__ __forceinline__ void split8(const float* v, float scale, H8& hi, H8& lo) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float s = v[j] * scale;
        hi[j] = (_Float16)s;
        lo[j] = (_Float16)(s - (float)hi[j]);
    }
}

// The 4 lanes of a row hold two panels' 64 bytes, two lanes a panel; they swap
// parts so that a store instruction writes one panel of 16 rows, 1 KB without
// gaps (hi and lo stored by their own lanes left every other 16 bytes to the
// next instruction).
__device__ __forceinline__ void store_panels(const H8& hi, const H8& lo, uint8_t* q0, uint8_t* q1, int blk) {
    typedef int I4 __attribute__((ext_vector_type(4)));
    const I4 h = __builtin_bit_cast(I4, hi), l = __builtin_bit_cast(I4, lo);
    I4 a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // quad_perm [0, 0, 1, 1] and [2, 2, 3, 3]
        const int h0 = __builtin_amdgcn_update_dpp(0, h[i], 0x50, 0xF, 0xF, false);
        const int l0 = __builtin_amdgcn_update_dpp(0, l[i], 0x50, 0xF, 0xF, false);
        const int h1 = __builtin_amdgcn_update_dpp(0, h[i], 0xFA, 0xF, 0xF, false);
        const int l1 = __builtin_amdgcn_update_dpp(0, l[i], 0xFA, 0xF, 0xF, false);
        a[i] = blk & 1 ? l0 : h0;
        b[i] = blk & 1 ? l1 : h1;
    }
    *reinterpret_cast<I4*>(q0 + blk * 16) = a;
    *reinterpret_cast<I4*>(q1 + blk * 16) = b;
}

struct SplitJob {
    const float* x;
    int64_t ld, rows;
    int K, vec;                            // vec: 16-byte aligned rows
    uint8_t* out;
    int* exps;                             // [rows rounded up to 64]
};

// U: 32-column units a wavefront holds in registers from one pass over the
// row, all loaded up front (8 wavefronts: K <= 256 U); 0: any K, the rows read
// a second time.  HBM is the bound.  Against two passes with one load in
// flight at a time (both operands of a product, us): in_proj + out_proj of 32768
// tokens at d_model 768 153 -> 114 (5.5 TB/s at K = 1536), of 1024 tokens at
// 2048 70 -> 55, the lm_head's 999 + 50280 rows of 768 74 -> 52.  16 units take
// 167 VGPRs (3 wavefronts a SIMD), 32 would spill.  Beside the norm (below)
// the weight's workgroups are few and keep two passes: 10.2 us either way at
// 999 + 3072 x 768, 11.0 since the rows' counts (split_ok) are taken.
template <int NT, int U>
__device__ __forceinline__ void split_block(const SplitJob& j, int64_t block) {
    constexpr int NW = NT / 64, UR = U > 0 ? U : 1;
    __shared__ uint32_t s_max[NW][kSplitRows];
    __shared__ int2 s_cnt[NW][kSplitRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane >> 2, blk = lane & 3, K = j.K;
    const bool vec = j.vec;
    const int64_t row = block * kSplitRows + r;
    const float* p = j.x + min(row, j.rows - 1) * j.ld;
    const int units = (K + 31) / 32;
    float held[UR][8];
    uint32_t mx = 0;
    if constexpr (U > 0) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int c = min(wave + i * NW, units - 1) * 32 + blk * 8;      // a unit past the end: the last again
            load8(p + c, K - c, vec, held[i]);
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int q = 0; q < 8; ++q) mx = max(mx, abs_bits(held[i][q]));
    } else {
        for (int u = wave; u < units; u += NW) {
            const int c = u * 32 + blk * 8;
            load8(p + c, K - c, vec, held[0]);
#pragma unroll
            for (int q = 0; q < 8; ++q) mx = max(mx, abs_bits(held[0][q]));
        }
    }
    mx = max(mx, dpp_mov_u<kDppXor1>(mx));
    mx = max(mx, dpp_mov_u<kDppXor2>(mx));
    if (blk == 0) s_max[wave][r] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = max(mx, s_max[w][r]);
    const int e = split_exp(mx);
    RowCount cnt(mx);
    // a marked row's parts are never used: zeros do
    const float scale = e >= kExpSpecial ? 0.f : __uint_as_float((uint32_t)(e + 127) << 23);
    const int np = 2 * units;
    uint8_t* const q = j.out + (row / kRowBlock * np) * (kRowBlock * kPanelBytes) + (row % kRowBlock) * kPanelBytes;
    auto put = [&](float* v, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) cnt.add(v[i]);
        if (e >= kExpSpecial) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = 0.f;
        }
        H8 hi, lo;
        split8(v, scale, hi, lo);
        uint8_t* qu = q + (int64_t)(2 * u) * (kRowBlock * kPanelBytes);
        if (row < j.rows) store_panels(hi, lo, qu, qu + kRowBlock * kPanelBytes, blk);   // whole quads of lanes
    };
    if constexpr (U > 0) {
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (wave + i * NW < units) put(held[i], wave + i * NW);
    } else {
        for (int u = wave; u < units; u += NW) {
            const int c = u * 32 + blk * 8;
            load8(p + c, K - c, vec, held[0]);
            put(held[0], u);
        }
    }
    auto quad_sum = [](int v) __attribute__((always_inline)) {
        v += (int)dpp_mov_u<kDppXor1>((uint32_t)v);
        return v + (int)dpp_mov_u<kDppXor2>((uint32_t)v);
    };
    const int2 c4 = make_int2(quad_sum(cnt.nonzero), quad_sum(cnt.small));
    if (blk == 0) s_cnt[wave][r] = c4;
    // (a barrier for the LDS writes only: __syncthreads would wait for the stores)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave == 0 && blk == 0) {                   // exps is padded to whole row blocks
        int2 c = c4;
#pragma unroll
        for (int w = 1; w < NW; ++w) { c.x += s_cnt[w][r].x; c.y += s_cnt[w][r].y; }
        j.exps[row] = row >= j.rows ? 0 : split_ok(c.x, c.y, 32 * units) ? e : kExpSpecial;
    }
}

// workgroups [0, nb0) take the first matrix, the others the second
template <int NT, int U>
__global__ void __launch_bounds__(NT) split_rows_kernel(const SplitJob j0, const SplitJob j1, int nb0) {
    const bool second = (int)blockIdx.x >= nb0;
    split_block<NT, U>(second ? j1 : j0, (int)blockIdx.x - (second ? nb0 : 0));
}

// The residual add and RMSNorm in front of an in_proj (model.py:306, 130-135)
// with the split of its output, and the split of the in_proj's weight, in one
// launch: the first nbn workgroups take 8 rows each (a wavefront a row, 8
// columns per lane and run, all loaded up front), the others 16 weight rows.
// Separate launches of the norm and the two splits took 5.5 + 6.8 + 7 us at
// 999 x 768, each of them mostly its launch and first round trip.
struct NormArgs {
    const float* x; const float* y;        // h, and the mixer output to add (null: none)
    float* x_out;                          // x + y (null: not stored)
    const float* w;
    float* normed;                         // the norm's output in fp32
    float eps;
};
constexpr int kNsThreads = 512, kNsRows = kNsThreads / 64;

template <int RU>                          // 512-column runs of a row
__global__ void __launch_bounds__(kNsThreads) norm_split_kernel(const NormArgs n, const SplitJob jx, const SplitJob jw,
                                                                int nbn) {
    if ((int)blockIdx.x >= nbn) {
        split_block<kNsThreads, 0>(jw, (int)blockIdx.x - nbn);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * kNsRows + (threadIdx.x >> 6);
    const int cols = jx.K;                 // a multiple of 32
    if (row >= jx.rows) {                  // whole wavefronts: the row block's padding
        if (lane == 0) jx.exps[row] = 0;
        return;
    }
    float v[RU][8], wv[RU][8];
#pragma unroll
    for (int u = 0; u < RU; ++u) {
        const int c = min(u * 512 + lane * 8, cols - 8);
        load8(n.x + row * cols + c, 8, true, v[u]);
        load8(n.w + c, 8, true, wv[u]);
    }
    if (n.y) {
        float yv[RU][8];
#pragma unroll
        for (int u = 0; u < RU; ++u) load8(n.y + row * cols + min(u * 512 + lane * 8, cols - 8), 8, true, yv[u]);
#pragma unroll
        for (int u = 0; u < RU; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) v[u][j] += yv[u][j];
    }
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < RU; ++u)
        if (u * 512 + lane * 8 < cols) {
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf(v[u][j], v[u][j], ss);
        }
    const float r = rsqrtf(group_sum<64>(ss) / (float)cols + n.eps);
    uint32_t mx = 0;
#pragma unroll
    for (int u = 0; u < RU; ++u) {
        const int c = u * 512 + lane * 8;
        if (c >= cols) continue;
        if (n.x_out) {
            float4* p = reinterpret_cast<float4*>(n.x_out + row * cols + c);
            p[0] = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
            p[1] = make_float4(v[u][4], v[u][5], v[u][6], v[u][7]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v[u][j] = wv[u][j] * (v[u][j] * r);
            mx = max(mx, abs_bits(v[u][j]));
        }
        float4* p = reinterpret_cast<float4*>(n.normed + row * cols + c);
        p[0] = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
        p[1] = make_float4(v[u][4], v[u][5], v[u][6], v[u][7]);
    }
    mx = group_umax<64>(mx);
    const int e = split_exp(mx);
    RowCount cnt(mx);
#pragma unroll
    for (int u = 0; u < RU; ++u)
        if (u * 512 + lane * 8 < cols) {
#pragma unroll
            for (int j = 0; j < 8; ++j) cnt.add(v[u][j]);
        }
    const bool ok = split_ok((int)group_sum<64>((float)cnt.nonzero), (int)group_sum<64>((float)cnt.small), cols);
    if (lane == 0) jx.exps[row] = ok ? e : kExpSpecial;
    if (e >= kExpSpecial) return;          // a marked row's parts are never used
    const float scale = __uint_as_float((uint32_t)(e + 127) << 23);
    const int np = cols / kPanel;
#pragma unroll
    for (int u = 0; u < RU; ++u) {
        const int c = u * 512 + lane * 8;
        if (c >= cols) continue;
        H8 hi, lo;
        split8(v[u], scale, hi, lo);
        uint8_t* q = jx.out + (row / kRowBlock * np + c / kPanel) * (kRowBlock * kPanelBytes) +
                     (row % kRowBlock) * kPanelBytes + (c / 8 % 2) * 32;
        *reinterpret_cast<H8*>(q) = hi;
        *reinterpret_cast<H8*>(q + 16) = lo;
    }
}

// ------------------------------------------------------------------ the product
struct GemmArgs {
    const uint8_t* xs; const int* ex;      // split X [M, K]
    const uint8_t* ws; const int* ew;      // split W [N, K]
    float* y0; float* y1;                  // columns [0, n_split) to y0, the others to y1
    int64_t ldy0, ldy1;
    const float* bias;
    const float* x32; const float* w32;    // the fp32 operands, for rows that cannot be split
    int64_t ldx, ldw;
    int M, N, K, n_split;
    int tm, tn;                            // tiles along M and N
    bool vec;                              // 16-byte aligned fp32 rows
};

// 4 consecutive columns of an fp32 row, zeros past the n there are
__device__ __forceinline__ F4v load4(const float* p, int n) {
    F4v v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = j < n ? p[j] : 0.f;
    return v;
}

// Mapping: a workgroup of 4 wavefronts takes a BM x BN tile of Y, each
// wavefront WM x WN of it as 32 x 32 MFMA tiles; the K loop walks stages of PK
// panels through an LDS ring of ST slots.
//   * The copies (global_load_lds_dwordx4, 16 rows x 64 bytes each) put 16-byte
//     chunk c of a row at position c ^ ((row >> 2) & 3): the fragment reads
//     (ds_read_b128, 32 rows of one chunk) then meet no bank conflict
//     (counted; with (row >> 1) & 3 half of the LDS cycles were conflicts).
//   * One barrier per stage.  The next panel's fragments are read into a
//     second register set, and the next stages' copies issued, between the
//     MFMAs of the present panel; issued in one piece after the barrier, the
//     copies held up the MFMAs behind them (32768 x 768 x 1536: 250 -> 218 us).
//   * The three products run tile by tile in turn, so an accumulator is used
//     again TI TJ MFMAs later.
template <int BM, int BN, int WM, int WN, int PK, int ST, int OCC>
__global__ void __launch_bounds__(BM / WM * (BN / WN) * 64, OCC) gemm_split_kernel(const GemmArgs a) {
    constexpr int NWM = BM / WM, NWN = BN / WN, NW = NWM * NWN;
    constexpr int TI = WM / 32, TJ = WN / 32;             // 32x32 MFMA tiles of a wavefront
    constexpr int SROWS = BM + BN, STAGE = PK * SROWS * kPanelBytes;
    constexpr int NI = PK * SROWS / 16 / NW;                   // 1 KB copies per wavefront and stage
    static_assert(SROWS % (16 * NW) == 0, "copies divide over the wavefronts");
    __shared__ __align__(1024) uint8_t ring[ST * STAGE];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / NWN, wn = wave % NWN;

    // XCD-aware tile order (workgroups are dealt to the 8 XCDs round robin):
    // each XCD takes a contiguous range of tiles, ordered 8 row tiles by all
    // column tiles, rows fastest, so the tiles resident on an XCD at one time
    // share their operand rows in its L2
    int t = blockIdx.x;
    const int total = a.tm * a.tn;
    {
        const int per = total / 8, rem = total % 8, x = t % 8, i = t / 8;
        t = x * per + min(x, rem) + i;
    }
    constexpr int GM = 8;
    const int group = t / (GM * a.tn), g0 = group * GM, gm = min(GM, a.tm - g0);
    const int in_g = t - group * GM * a.tn;
    // (uniform, but the divisions run on the VALU: back to SGPRs)
    const int m0 = __builtin_amdgcn_readfirstlane((g0 + in_g % gm) * BM);
    const int n0 = __builtin_amdgcn_readfirstlane(in_g / gm * BN);

    // copy lane: row 16 g + lane / 4 of the stage; position lane % 4 of a row
    // takes 16-byte chunk (lane % 4) ^ ((row >> 2) & 3) (above)
    const int np = (a.K + 31) / 32 * 2;                    // panels (K padded to 32)
    const uint8_t* base[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int g = (wave * NI + i) % (SROWS / 16), pk = (wave * NI + i) / (SROWS / 16);
        const int row = 16 * g + (lane >> 2);
        const int c = (lane & 3) ^ ((row >> 2) & 3);
        const bool isx = 16 * g < BM;                     // wavefront-uniform (BM a multiple of 16)
        const int rr = isx ? min(m0 + row, a.M - 1) : min(n0 + row - BM, a.N - 1);
        base[i] = (isx ? a.xs : a.ws) + ((int64_t)(rr / kRowBlock) * np + pk) * (kRowBlock * kPanelBytes) +
                  rr % kRowBlock * kPanelBytes + c * 16;
    }
    // stage s's panels; a last stage past the panels re-reads the last ones (its products are skipped)
    auto issue1 = [&](int i, int slot, int s) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
        const uint32_t so = (uint32_t)s * (PK * kRowBlock * kPanelBytes);
        __builtin_amdgcn_global_load_lds(base[i] + so, ring + slot * STAGE + (wave * NI + i) * 1024, 16, 0, 0);
#else
        (void)i; (void)slot; (void)s;
#endif
    };
    auto issue = [&](int slot, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NI; ++i) issue1(i, slot, s);
    };

    F16v acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

    const int r32 = lane & 31, g2 = lane >> 5;
    // byte offsets of this lane's hi chunk in rows 32 i + r32 of a tile (the
    // swizzle, of a period of 16 rows, depends on r32 only)
    const int sw = (r32 >> 2) & 3;
    const uint32_t o_hi = r32 * kPanelBytes + ((2 * g2) ^ sw) * 16, o_lo = r32 * kPanelBytes + ((2 * g2 + 1) ^ sw) * 16;
    struct Frag { H8 xh[TI], xl[TI], wh[TJ], wl[TJ]; };
    constexpr int NR = 2 * (TI + TJ);                     // LDS reads of a fragment set
    auto read1 = [&](Frag& f, int k, int slot, int pk) __attribute__((always_inline)) {
        const uint8_t* p = ring + slot * STAGE + pk * SROWS * kPanelBytes;
        const uint8_t* px = p + wm * WM * kPanelBytes;
        const uint8_t* pw = p + (BM + wn * WN) * kPanelBytes;
        // x lo and w hi first: the first product takes them
        if (k < TI) f.xl[k] = *reinterpret_cast<const H8*>(px + k * 32 * kPanelBytes + o_lo);
        else if (k < TI + TJ) f.wh[k - TI] = *reinterpret_cast<const H8*>(pw + (k - TI) * 32 * kPanelBytes + o_hi);
        else if (k < 2 * TI + TJ) f.xh[k - TI - TJ] = *reinterpret_cast<const H8*>(px + (k - TI - TJ) * 32 * kPanelBytes + o_hi);
        else f.wl[k - 2 * TI - TJ] = *reinterpret_cast<const H8*>(pw + (k - 2 * TI - TJ) * 32 * kPanelBytes + o_lo);
    };
    constexpr int MT = TI * TJ;                            // MFMAs of one of the three products
    // MFMA t of the 3 MT of a panel: product t / MT (lo hi, hi lo, hi hi) of
    // tile t % MT, so an accumulator is used again MT MFMAs later
    auto mma1 = [&](const Frag& f, int t) __attribute__((always_inline)) {
        const int p = t / MT, i = t % MT % TI, j = t % MT / TI;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(p == 0 ? f.xl[i] : f.xh[i], p == 1 ? f.wl[j] : f.wh[j],
                                                           acc[i][j], 0, 0, 0);
    };

    const int ns = (np + PK - 1) / PK;                      // stages
    int slot = 0;
    // stage s + 1 of the ring is read into nxt while stage s (in cur) is multiplied
    auto sync = [&](bool tail) __attribute__((always_inline)) {
        if (tail)
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * NI) : "memory");
    };
    auto body = [&](Frag& cur, Frag& nxt, int s, int pk) __attribute__((always_inline)) {
        int prev = slot;
        bool load = false, rd = true;
#pragma unroll
        for (int t = 0; t < MT; ++t) mma1(cur, t);
        __builtin_amdgcn_sched_barrier(0);
        if (pk + 1 == PK) {
            rd = s + 1 < ns;
            if (rd) {
                sync(s + ST > ns);
                slot = slot + 1 == ST ? 0 : slot + 1;
                load = s + ST < ns;
            }
        }
        const int npk = pk + 1 == PK ? 0 : pk + 1;
        // the reads and then the copies go between the MFMAs of the other two products
#pragma unroll
        for (int t = 0; t < 2 * MT; ++t) {
            mma1(cur, MT + t);
            if (rd) {
#pragma unroll
                for (int k = t * NR / MT; k < (t + 1) * NR / MT && k < NR; ++k) read1(nxt, k, slot, npk);
            }
            if (t >= MT && load) {
#pragma unroll
                for (int k = (t - MT) * NI / MT; k < (t - MT + 1) * NI / MT; ++k) issue1(k, prev, s + ST);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int s = 0; s < ST; ++s)
        if (s < ns) issue(s, s);
    Frag f0, f1;
    if (ns >= ST)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((ST - 1) * NI) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int k = 0; k < NR; ++k) read1(f0, k, 0, 0);
    int s = 0;
    if constexpr (PK == 1) {
        for (; s + 1 < ns; s += 2) {
            body(f0, f1, s, 0);
            body(f1, f0, s + 1, 0);
        }
        if (s < ns) body(f0, f1, s, 0);
    } else {
        for (; s < ns; ++s) {
            body(f0, f1, s, 0);
            body(f1, f0, s, 1);
        }
    }

    // D[i][j] of a tile: column j = lane % 32 (an output column n), row
    // 8 (q / 4) + 4 (lane / 32) + q % 4 in register q (an output row m).  The
    // stores go through buffer resources that end at this tile's last row of
    // y.  A lane past the last column, or in the last tile past the last row,
    // gets a VGPR offset past the end, so neither needs a branch; the SGPR
    // offset, which the range check need not cover, holds a row of y's only.
    const int mw = m0 + wm * WM, mpad = (a.M + kRowBlock - 1) / kRowBlock * kRowBlock;
    auto row_exps = [&](int mt, int* em) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int4 v = *reinterpret_cast<const int4*>(a.ex + min(mt + 8 * q + 4 * g2, mpad - 4));
            em[4 * q] = v.x; em[4 * q + 1] = v.y; em[4 * q + 2] = v.z; em[4 * q + 3] = v.w;
        }
    };
    int en[TJ];
    float bn[TJ];
    bool special = false;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const int n = n0 + wn * WN + 32 * j + r32, nc = min(n, a.N - 1);
        en[j] = a.ew[nc];
        bn[j] = a.bias ? a.bias[nc] : 0.f;
        special |= en[j] >= kExpSpecial;
    }
    auto store = [&](auto all_rows) __attribute__((always_inline)) {
        constexpr bool ALL = decltype(all_rows)::value;
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            int em[16], top = 0;
            row_exps(mw + 32 * i, em);
#pragma unroll
            for (int q = 0; q < 16; ++q) top = max(top, em[q]);
            special |= top >= kExpSpecial;
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                const int nt = n0 + wn * WN + 32 * j;        // n_split is a multiple of 32 (host-checked)
                const bool first = nt < a.n_split;
                const int64_t ldy = first ? a.ldy0 : a.ldy1;
                const int n = nt + r32, col = first ? n : n - a.n_split;
                float* yt = (first ? a.y0 : a.y1) + (int64_t)m0 * ldy;
                const auto ry = __builtin_amdgcn_make_buffer_rsrc(yt, (short)0, (int)(min(BM, a.M - m0) * ldy * 4), 0x00020000);
                const uint32_t vo = n < a.N ? (uint32_t)(col + 4 * g2 * ldy) * 4u : 0xfffffff0u;
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int ml = wm * WM + 32 * i + 8 * (q >> 2) + (q & 3);
                    const float v = __builtin_amdgcn_ldexpf(acc[i][j][q], -(em[q] + en[j])) + bn[j];
                    const uint32_t vq = ALL || m0 + ml + 4 * g2 < a.M ? vo : 0xfffffff0u;
                    const int so = ALL || m0 + ml < a.M ? (int)(ml * ldy * 4) : 0;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ry, (int)vq, so, 0);
                }
            }
        }
    };
    if (m0 + BM <= a.M) store(std::true_type{});
    else store(std::false_type{});
    // outputs of rows that could not be split, over the values stored above by
    // the same lanes: the 32 x 32 tiles that hold any, from the fp32 operands.
    // Lane half g2 takes 4 consecutive columns of its row; MFMA q of a group
    // of 8 columns sums columns q and q + 4.
    if (__any(special)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        for (int t = 0; t < TI * TJ; ++t) {
            const int mt = mw + 32 * (t / TJ), n = n0 + wn * WN + 32 * (t % TJ) + r32;
            const int m = min(mt + r32, a.M - 1), nc = min(n, a.N - 1);
            const bool ns_ = a.ew[nc] >= kExpSpecial;
            if (!__any(ns_ || a.ex[m] >= kExpSpecial)) continue;
            const float* x = a.x32 + m * a.ldx + 4 * g2;
            const float* w = a.w32 + nc * a.ldw + 4 * g2;
            F16v c, c2;                                      // two chains
#pragma unroll
            for (int q = 0; q < 16; ++q) c[q] = c2[q] = 0.f;
            constexpr int KG = 4;                            // groups of 8 columns loaded at a time
            struct Cols { F4v x[KG], w[KG]; } cur, nxt;
            auto load = [&](Cols& d, int k) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < KG; ++u) { d.x[u] = ld4(x + k + 8 * u); d.w[u] = ld4(w + k + 8 * u); }
            };
            auto mma = [&](const Cols& d) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < KG; ++u)
#pragma unroll
                    for (int q = 0; q < 4; q += 2) {
                        c = __builtin_amdgcn_mfma_f32_32x32x2f32(d.x[u][q], d.w[u][q], c, 0, 0, 0);
                        c2 = __builtin_amdgcn_mfma_f32_32x32x2f32(d.x[u][q + 1], d.w[u][q + 1], c2, 0, 0, 0);
                    }
            };
            const int whole_k = a.vec ? a.K & -(8 * KG) : 0;
            if (whole_k) load(cur, 0);
            for (int k = 0; k < whole_k; k += 8 * KG, cur = nxt) {
                load(nxt, min(k + 8 * KG, whole_k - 8 * KG));
                __builtin_amdgcn_sched_barrier(0);
                mma(cur);
            }
            for (int k = whole_k; k < a.K; k += 8 * KG) {    // the last columns, or all of unaligned rows
#pragma unroll
                for (int u = 0; u < KG; ++u) {
                    const int left = a.K - k - 8 * u - 4 * g2;
                    cur.x[u] = load4(x + k + 8 * u, left);
                    cur.w[u] = load4(w + k + 8 * u, left);
                }
                mma(cur);
            }
            c += c2;
            const float bias = a.bias ? a.bias[nc] : 0.f;
            int em[16];
            row_exps(mt, em);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int mq = mt + 8 * (q >> 2) + 4 * g2 + (q & 3);
                if (mq >= a.M || n >= a.N || (!ns_ && em[q] < kExpSpecial)) continue;
                if (n < a.n_split) a.y0[mq * a.ldy0 + n] = c[q] + bias;
                else a.y1[mq * a.ldy1 + n - a.n_split] = c[q] + bias;
            }
        }
    }
}

template <int BM, int BN, int WM, int WN, int PK, int ST, int OCC>
void launch_gemm(GemmArgs a, hipStream_t st) {
    a.tm = (a.M + BM - 1) / BM;
    a.tn = (a.N + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WM, WN, PK, ST, OCC>), dim3((unsigned)(a.tm * a.tn)),
                       dim3(BM / WM * (BN / WN) * 64), 0, st, a);
}

int64_t pad_to(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

SplitJob split_job(const float* x, int64_t ld, int64_t rows, int64_t K, void* buf) {
    SplitJob j{};
    j.x = x; j.ld = ld; j.rows = rows; j.K = (int)K;
    j.vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && ld % 4 == 0;
    j.exps = static_cast<int*>(buf);
    j.out = static_cast<uint8_t*>(buf) + pad_to(pad_to(rows, kRowBlock) * (int64_t)sizeof(int), 1024);
    return j;
}

}  // namespace

int64_t split_bytes(int64_t rows, int64_t K) {
    return pad_to(pad_to(rows, kRowBlock) * (int64_t)sizeof(int), 1024) + pad_to(rows, kRowBlock) * pad_to(K, 32) * 4;
}

int split_rows(const float* x, int64_t ldx, int64_t M, const float* w, int64_t ldw, int64_t N, int64_t K, void* xbuf,
               void* wbuf, hipStream_t st) {
    const SplitJob jx = split_job(x ? x : w, x ? ldx : ldw, x ? M : N, K, x ? xbuf : wbuf);
    const SplitJob jw = split_job(w ? w : x, w ? ldw : ldx, w ? N : M, K, w ? wbuf : xbuf);
    const int64_t bx = x ? pad_to(M, kRowBlock) / kSplitRows : 0, bw = w ? pad_to(N, kRowBlock) / kSplitRows : 0;
    const dim3 grid((unsigned)(bx + bw)), nt(512);
#define MTL_SPLIT(U) hipLaunchKernelGGL((split_rows_kernel<512, U>), grid, nt, 0, st, jx, jw, (int)bx)
    if (K <= 1024) MTL_SPLIT(4);
    else if (K <= 2048) MTL_SPLIT(8);
    else if (K <= 4096) MTL_SPLIT(16);
    else MTL_SPLIT(0);
#undef MTL_SPLIT
    return check_launch("split_rows");
}

int norm_split(const float* x, const float* y, float* x_out, const float* w, float eps, float* normed, int64_t M,
               int64_t K, const float* wmat, int64_t ldw, int64_t N, void* xbuf, void* wbuf, hipStream_t st) {
    const NormArgs n{x, y, x_out, w, normed, eps};
    const SplitJob jx = split_job(normed, K, M, K, xbuf), jw = split_job(wmat, ldw, N, K, wbuf);
    const int64_t bn = pad_to(M, kRowBlock) / kNsRows, bw = pad_to(N, kRowBlock) / kSplitRows;
    const dim3 grid((unsigned)(bn + bw)), nt(kNsThreads);
    if (K <= 512) hipLaunchKernelGGL((norm_split_kernel<1>), grid, nt, 0, st, n, jx, jw, (int)bn);
    else if (K <= 1024) hipLaunchKernelGGL((norm_split_kernel<2>), grid, nt, 0, st, n, jx, jw, (int)bn);
    else hipLaunchKernelGGL((norm_split_kernel<4>), grid, nt, 0, st, n, jx, jw, (int)bn);
    return check_launch("norm_split");
}

bool norm_split_ok(const float* x, const float* y, const float* w, const float* normed, int64_t K) {
    return K % 32 == 0 && K <= 2048 &&
           (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(w) |
            reinterpret_cast<uintptr_t>(normed)) % 16 == 0;
}

// Where the product with the splits of x and W beats the library's fp32 GEMM:
// the split of W is paid once per call, so the gain needs rows, and few tiles
// leave CUs idle.  Measured, us, library / split + product: 999 x 3072 x 768
// 45 / 40, 768 x 3072 x 768 36 / 39; 768 x 2048 x 4096 107 / 96, 512 x 2048 x
// 4096 69 / 86; 384 x 8192 x 2048 112 / 96, 256 x 8192 x 2048 74 / 81; 256 x
// 50280 x 768 171 / 156, 192 x 50280 x 768 146 / 150; 999 x 768 x 1536 24 / 38.
bool split_pays(int64_t M, int64_t N, int64_t K) {
    const double flops = 2.0 * (double)M * (double)N * (double)K;
    return N >= 256 && K >= 128 && ((M >= 256 && flops >= 1.2e10) || (M >= 896 && flops >= 4.5e9));
}

int gemm_split(const SplitGemm& g, hipStream_t st) {
    const SplitJob x = split_job(g.x, g.ldx, g.M, g.K, g.xbuf), w = split_job(g.w, g.ldw, g.N, g.K, g.wbuf);
    GemmArgs a{};
    a.xs = x.out; a.ex = x.exps; a.ws = w.out; a.ew = w.exps;
    a.y0 = g.y0; a.ldy0 = g.ldy0; a.y1 = g.y1 ? g.y1 : g.y0; a.ldy1 = g.y1 ? g.ldy1 : g.ldy0;
    a.n_split = (int)(g.y1 ? g.n_split : g.N);
    a.bias = g.bias;
    a.x32 = g.x; a.ldx = g.ldx; a.w32 = g.w; a.ldw = g.ldw;
    a.M = (int)g.M; a.N = (int)g.N; a.K = (int)g.K;
    a.vec = x.vec && w.vec;
    // Tile by the number of tiles each gives (us at M x N x K; 256 x 128, 128 x
    // 128, 64 x 64): 32768 x 3072 x 768 449 / 499 / 739, 512 x 50280 x 768 147 /
    // 158 / 234 (786 large tiles); 768 x 8192 x 2048 100 / 90 / 103, 512 x 8192 x
    // 2048 90 / 59 / 75 (256 middle tiles); 384 x 8192 x 2048 91 / 55 / 54, 999 x
    // 3072 x 768 44 / 28 / 26 (192), 1024 x 2048 x 4096 154 / 92 / 69 (128).  A
    // CU holds 2, 2 and 3 of these workgroups.
    const int64_t large = ((g.M + 255) / 256) * ((g.N + 127) / 128), middle = ((g.M + 127) / 128) * ((g.N + 127) / 128);
    if (large >= 512) launch_gemm<256, 128, 128, 64, 1, 3, 2>(a, st);
    else if (middle >= 224) launch_gemm<128, 128, 64, 64, 2, 2, 2>(a, st);
    else launch_gemm<64, 64, 32, 32, 2, 3, 3>(a, st);
    return check_launch("gemm_split");
}

}  // namespace mtl

extern "C" int mtl_linear_f32_pays(int64_t M, int64_t N, int64_t K) { return mtl::split_pays(M, N, K) ? 1 : 0; }

extern "C" int64_t mtl_linear_f32_ws_bytes(int64_t M, int64_t N, int64_t K) {
    if (M < 1 || N < 1 || K < 1) return 0;
    return mtl::pad_to(mtl::split_bytes(M, K), 1024) + mtl::split_bytes(N, K);
}

extern "C" int mtl_linear_f32(const mtl_linear_f32_args* g, mtl_stream_t stream) {
    using namespace mtl;
    clear_error();
    MTL_REQUIRE(g, "null args");
    MTL_REQUIRE(g->M >= 0 && g->N >= 0 && g->K >= 1, "M, N must be >= 0 and K >= 1");
    if (g->M == 0 || g->N == 0) return MTL_OK;
    MTL_REQUIRE(g->x && g->W && g->y0 && g->ws, "null x, W, y0 or ws");
    // 2^30: tile counts, exponent indexes and 256 output rows' byte offsets stay in 32 bits
    MTL_REQUIRE(g->M <= (int64_t(1) << 30) && g->N <= (int64_t(1) << 30) && g->K <= (int64_t(1) << 23),
                "M, N must be <= 2^30 and K <= 2^23");
    MTL_REQUIRE(((g->M + 63) / 64) * ((g->N + 63) / 64) < (int64_t(1) << 31), "too many output tiles");
    MTL_REQUIRE(g->ldx >= g->K && g->ldw >= g->K, "ldx and ldw must be >= K");
    const int64_t n0 = g->y1 ? g->n_split : g->N;
    MTL_REQUIRE(!g->y1 || (g->n_split > 0 && g->n_split < g->N && g->n_split % 32 == 0),
                "n_split must be a multiple of 32 inside (0, N)");
    MTL_REQUIRE(g->ldy0 >= n0 && g->ldy0 < (int64_t(1) << 21) &&
                (!g->y1 || (g->ldy1 >= g->N - n0 && g->ldy1 < (int64_t(1) << 21))),
                "ldy must cover the output's columns and be below 2^21");
    MTL_REQUIRE(g->ws_bytes >= mtl_linear_f32_ws_bytes(g->M, g->N, g->K), "ws is too small");
    MTL_REQUIRE(reinterpret_cast<uintptr_t>(g->ws) % 16 == 0, "ws must be 16-byte aligned");
    SplitGemm s{};
    s.x = g->x; s.ldx = g->ldx; s.w = g->W; s.ldw = g->ldw; s.bias = g->bias;
    s.y0 = g->y0; s.ldy0 = g->ldy0; s.y1 = g->y1; s.ldy1 = g->ldy1; s.n_split = g->n_split;
    s.M = g->M; s.N = g->N; s.K = g->K;
    s.xbuf = g->ws;
    s.wbuf = static_cast<uint8_t*>(g->ws) + pad_to(split_bytes(g->M, g->K), 1024);
    hipStream_t st = as_stream(stream);
    const int rc = split_rows(s.x, s.ldx, s.M, s.w, s.ldw, s.N, s.K, s.xbuf, s.wbuf, st);
    return rc ? rc : gemm_split(s, st);
}
