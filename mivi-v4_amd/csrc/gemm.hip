// quantized_matmul_rows (crates/mivi-quant/src/lib.rs:143-357) for gfx950.
//
// batch == 1 is exactly the matvec path (lib.rs:171-182). From kMfmaMinBatch
// rows on (rows_route below) the products run on the matrix cores:
//
//   gemm_prep_kernel   one wave per input row: the prologue, then the row
//                      split into 16-bit planes in MFMA operand order (fp16
//                      hi + lo under a power-of-two row scale; bf16 hi + mid
//                      + lo for bf16 weights);
//   gemm_rows_kernel   v_mfma_f32_32x32x16, one wave per 64 x 64 (32 x 64)
//                      outputs and share of the depth, the weights loaded
//                      straight from memory into registers, the inputs too
//                      or, in wide workgroups, shared through LDS.
//
// Every weight enters the products exactly (Q4_K: sc * q, an integer <= 945;
// Q6_K and Q8_0: the integer q, its scale applied to the f32 sums; F16 and
// BF16: the value itself), so the inputs' split and the f32 sums are the only
// roundings. Other formats and shapes, and fewer rows, run the batched GEMV
// (the inputs as its columns).
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "common.h"
#include "gemv.h"

namespace mivi {
bool format_sizes(int32_t t, size_t* bs, size_t* ts);
bool ggml_sizes(int32_t t, size_t* bs, size_t* ts);
}  // namespace mivi

using namespace mivi;

namespace {

constexpr int kMfmaMinBatch = 16;     // K-quants at the depths of the batched GEMVs
constexpr int kMfmaMinBatchRows = 4;  // shapes with one GEMV launch per input
constexpr int kTk = 64;  // k-tile of the packed copy: one Q4_K group (a sub-block pair)

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------- prep
// Row m of the activations, v = pro(X row m) with X row m at X + m * ldx
// (PRO_NONE v = x; PRO_RMSNORM v = (x * s) * w, s = 1/sqrt(mean(x^2) + eps)
// (norm.rs:38-72); PRO_SWIGLU v = silu(x) * x2 (math.rs:87-95), X2 row m at
// X2 + m * ldx), into the A operand of the row products.
//
// fp16 planes (P = 2): the row scaled by the power of two that puts its
// largest finite |v| in [2^14, 2^15) (so the lo part of a value within 2^-15
// of the largest is no denormal) and split v = hi + lo, each rounded to
// nearest: v to 2^-23 relative, from 2^-17 of the largest down to 2^-39 of the
// largest. bf16 planes (P = 3, bf16 weights, whose
// range fp16 does not cover): v = hi + mid + lo unscaled. An infinite value
// keeps its hi part only (no inf - inf).
// Operand order: per 32 rows and 16-value k-step, one 1 KB block per plane,
// lane l = m % 32 + 32 h holding the values 16 ks + 8 h .. + 7 (16 bytes) of
// row m, at ((m / 32) * (K / 16) + ks) * P + plane) KB. Rows >= M are zero.
// Q4_K also takes the 32-value sub-block sums of the scaled row, times 2^-5
// (a sum may reach 2^20, past fp16's range), as fp16 hi / lo: per 32 rows and
// super-block a 1 KB block, lane m % 32 the eight hi parts, lane m % 32 + 32
// the lo parts.
//
// One wave per row, eight rows per workgroup: an operand line of 128 bytes
// holds eight consecutive rows' chunks of eight values, so the workgroup
// writes whole lines (through LDS). One row per workgroup wrote every line in
// eight pieces from eight workgroups, each a partial write to memory: 18 us at
// 512 x 8192 against 6 here. Lane l owns the chunks l + 64 j; J > 0: at most J
// of them, held in registers through both reductions; J = 0: any K, the row
// re-read by each pass. vec: rows (and norm weights) 16-byte aligned.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kStepBytes = 1024;  // one operand block: 32 rows x 16 values of 16 bits
constexpr int kPrepRows = 8;

template <int J, int P>
__global__ void __launch_bounds__(512) gemm_prep_kernel(const float* __restrict__ X, const float* __restrict__ X2,
                                                        const float* __restrict__ norm_w, float eps, int pro,
                                                        int64_t ldx, int M, int K, int vec, uint8_t* __restrict__ xa,
                                                        uint8_t* __restrict__ xs, float* __restrict__ rowscale) {
    constexpr int C = 4;  // chunks of a lane per write pass
    __shared__ __attribute__((aligned(16))) uint8_t buf[C * P * 64 * kPrepRows * 16];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int m = kPrepRows * blockIdx.x + w;
    const bool live = m < M;
    const float* x = X + (live ? m : 0) * ldx;
    const float* x2 = pro == PRO_SWIGLU ? X2 + (live ? m : 0) * ldx : nullptr;
    auto load8 = [&](const float* p, int i, float (&v)[8]) {
        if (vec) {
            const f32x4 a = *(const f32x4*)(p + i), b = *(const f32x4*)(p + i + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = p[i + q];
        }
    };
    const int nj = J > 0 ? J : (K + 511) / 512;
    constexpr int JJ = J > 0 ? J : 1;
    float v[JJ][8];
    float scale = 1.0f;
    // chunk j of the prologue's input: x, or silu(x) * x2
    auto input = [&](int j, float (&o)[8]) {
        const int i = 8 * (lane + 64 * j);
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = 0.f;
        if (!live || i >= K) return;
        load8(x, i, o);
        if (pro == PRO_SWIGLU) {
            float u[8];
            load8(x2, i, u);
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = silu_f(o[q]) * u[q];
        }
    };
    auto normed = [&](int j, float (&o)[8]) {
        const int i = 8 * (lane + 64 * j);
        if (pro != PRO_RMSNORM || !live || i >= K) return;
        float g[8];
        load8(norm_w, i, g);
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = o[q] * scale * g[q];
    };
    if constexpr (J > 0) {
#pragma unroll
        for (int j = 0; j < J; j++) input(j, v[j]);
    }
    if (pro == PRO_RMSNORM) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < nj; j++) {
            float (&o)[8] = v[J > 0 ? j : 0];
            if (J == 0) input(j, o);
#pragma unroll
            for (int q = 0; q < 8; q++) ss = fmaf(o[q], o[q], ss);
        }
        ss = wave_sum(ss);
        scale = 1.0f / sqrtf(ss / (float)K + eps);
    }
    if constexpr (J > 0) {
#pragma unroll
        for (int j = 0; j < J; j++) normed(j, v[j]);
    }
    float inv = 1.0f;
    if constexpr (P == 2) {
        float mx = 0.f;
#pragma unroll
        for (int j = 0; j < nj; j++) {
            float (&o)[8] = v[J > 0 ? j : 0];
            if (J == 0) { input(j, o); normed(j, o); }
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float av = fabsf(o[q]);
                mx = av <= 3.40282347e38f ? fmaxf(mx, av) : mx;
            }
        }
        mx = wave_max(mx);
        // max * 2^-e in [2^14, 2^15); e >= -110 keeps 2^-e finite
        int e = 0;
        if (mx > 0.f) {
            frexpf(mx, &e);
            e = max(e - 15, -110);
        }
        inv = ldexpf(1.0f, -e);
        if (lane == 0) rowscale[m] = live ? ldexpf(1.0f, e) : 0.f;
    } else if (lane == 0) {
        rowscale[m] = live ? 1.0f : 0.f;
    }
    // chunk j as planes into buf: [chunk of the pass][plane][lane][row], the
    // rows of a lane permuted by the lane so that the writes of a wave hit
    // distinct banks
    auto split = [&](int j, int c, float (&o)[8]) {
        const int i = 8 * (lane + 64 * j);
        uint8_t* dst = buf + ((c * P * 64 + lane) * kPrepRows + (w ^ (lane & 7))) * 16;
        constexpr int PS = 64 * kPrepRows * 16;
        if constexpr (P == 2) {
            half8 hv, lv;
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float s = o[q] * inv;  // exact: power-of-two scaling
                hv[q] = (_Float16)s;
                const float rest = s - (float)hv[q];
                lv[q] = fabsf(s) <= 3.40282347e38f ? (_Float16)rest : (_Float16)0.0f;
                sum += s;
            }
            *(half8*)dst = hv;
            *(half8*)(dst + PS) = lv;
            if (xs) {
                // 4 consecutive lanes hold one 32-value sub-block
                sum += __shfl_xor(sum, 1, 64);
                sum += __shfl_xor(sum, 2, 64);
                if ((lane & 3) == 0 && i < K) {
                    sum *= 0.03125f;
                    const _Float16 h = (_Float16)sum;
                    uint8_t* sp = xs + ((size_t)(m >> 5) * (K / 256) + i / 256) * kStepBytes + 16 * (m & 31) + 2 * ((i / 32) & 7);
                    *(_Float16*)sp = h;
                    *(_Float16*)(sp + 512) = (_Float16)(sum - (float)h);
                }
            }
        } else {
            bf16x8 b[3];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                __bf16 b0, b1, b2;
                split_bf16(o[q], b0, b1, b2);
                b[0][q] = b0; b[1][q] = b1; b[2][q] = b2;
            }
#pragma unroll
            for (int p = 0; p < 3; p++) *(bf16x8*)(dst + p * PS) = b[p];
        }
    };
    const int r = threadIdx.x & 7, l8 = threadIdx.x >> 3;  // the thread's row and chunk lane when writing
    const int mw = kPrepRows * blockIdx.x + r;
    uint8_t* xrow = xa + ((size_t)(mw >> 5) * (K / 16) * P) * kStepBytes + 16 * (mw & 31);
#pragma unroll
    for (int j0 = 0; j0 < nj; j0 += C) {
        if (j0) __syncthreads();
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int j = j0 + c;
            if (J > 0 && j >= J) break;
            float (&o)[8] = v[J > 0 ? j : 0];
            if (J == 0) { input(j, o); normed(j, o); }
            split(j, c, o);
        }
        __syncthreads();
        const int k8 = l8 + 64 * j0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int k = k8 + 64 * c;
            if (8 * k >= K) break;
            uint8_t* d = xrow + (size_t)(k >> 1) * P * kStepBytes + (k & 1) * 512;
#pragma unroll
            for (int p = 0; p < P; p++)
                *(u32x4*)(d + p * kStepBytes) = *(const u32x4*)(buf + (((c * P + p) * 64 + l8) * kPrepRows + (r ^ (l8 & 7))) * 16);
        }
    }
}

// (scale, min) pair of sub-block j (0..7) from the 12 scale bytes held in
// hdr dwords 1..3 (get_scale_min_k4, q4_k_m.rs:11-22)
__device__ __forceinline__ void scale_min_k4(const uint8_t* q, int j, uint32_t& sc, uint32_t& m) {
    if (j < 4) {
        sc = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        sc = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// ------------------------------------------------ Q4_K B operand converted once
//
// launch_pack_q4k_gemm layout of a rows x cols Q4_K matrix (rows % 32 == 0,
// cols % 256 == 0), read by gemm_rows_kernel<RF_Q4P>:
//   B section: per 32-row tile nt and 64-value k-tile kt (Q4_K group g = kt %
//   4 of super-block kt / 4: sub-block 2g from the low nibbles of its 32 code
//   bytes, 2g + 1 from the high ones), per k-step s (values 16s .. 16s + 15
//   of the k-tile), the v_mfma_f32_32x32x16_f16 B operand: lane l (row 32 nt +
//   l % 32, values 16 s + 8 (l / 32) .. + 7) holds the 8 fp16 sc * q, exact
//   (<= 945), at byte ((nt * KT + kt) * 4 + s) * 1024 + 16 l (KT = cols / 64);
//   H section (after the rows * cols * 2 bytes of B): per (nt, super-block
//   sb), 640 bytes: the 32 rows' d | dmin << 16 (their header's first dword),
//   then their 8 sub-block mins as fp16 (16 bytes a row).
// The values are those gemm_rows_kernel<RF_Q4> forms in registers for every
// tile of input rows; here they are built once and every k-step's B is one
// contiguous 1 KB load.
constexpr int kGemmHBytes = 640;

__global__ void __launch_bounds__(256) pack_q4k_gemm_kernel(const uint8_t* __restrict__ src,
                                                            uint8_t* __restrict__ dst, int rows, int cols) {
    const int KT = cols / kTk, NB = cols / 256;
    const size_t rb = (size_t)NB * 144;
    const size_t nb16 = (size_t)rows / 32 * KT * 4 * 64;  // 16-byte B entries
    const size_t nh = (size_t)rows / 32 * NB * 32;        // (row, super-block) header entries
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nb16) {
        const int l = (int)(i & 63);
        size_t q = i >> 6;
        const int s = (int)(q & 3);
        q >>= 2;
        const int kt = (int)(q % KT);
        const size_t nt = q / KT;
        const int kk0 = 16 * s + 8 * (l >> 5), g = kt % 4;  // values kk0 .. kk0 + 7 of the group
        const uint8_t* blk = src + (32 * nt + (l & 31)) * rb + (size_t)(kt / 4) * 144;
        uint32_t sc, mn;
        scale_min_k4(blk + 4, 2 * g + (kk0 >= 32), sc, mn);
        half8 v;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t byte = blk[16 + 32 * g + ((kk0 + e) & 31)];
            v[e] = (_Float16)(float)((kk0 >= 32 ? byte >> 4 : byte & 15u) * sc);
        }
        *(half8*)(dst + i * 16) = v;
    } else if (i < nb16 + nh) {
        const size_t h = i - nb16, q = h >> 5;  // q = nt * NB + sb
        const int r = (int)(h & 31), sb = (int)(q % NB);
        const size_t nt = q / NB;
        const uint8_t* blk = src + (32 * nt + r) * rb + (size_t)sb * 144;
        uint8_t* H = dst + (size_t)rows * cols * 2 + q * kGemmHBytes;
        *(uint32_t*)(H + 4 * r) = *(const uint32_t*)blk;
        half8 mv;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            uint32_t sc, mn;
            scale_min_k4(blk + 4, j, sc, mn);
            mv[j] = (_Float16)(float)mn;
        }
        *(half8*)(H + 128 + 16 * r) = mv;
    }
}


// ------------------------------------------------------------ the product
// Weight formats of the row products: Q4_K in the operand layout of
// launch_pack_q4k_gemm (below), or rows as the file holds them.
enum RowsFmt : int { RF_Q4P, RF_Q4, RF_Q6, RF_Q8, RF_F16, RF_BF16 };

// f(std::integral_constant<int, I>) for I = I0 .. N - 1, unrolled at compile
// time (register arrays indexed by I stay in registers)
template <int I0, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I0 < N) {
        f(std::integral_constant<int, I0>{});
        static_for<I0 + 1, N>(f);
    }
}

struct RowsSeg {
    const uint8_t* W;  // weight rows (RF_Q4P: the operand copy)
    float* y;
    int n;             // rows
    int t0;            // its first column tile of the launch
};

struct RowsArgs {
    RowsSeg seg[3];
    int nseg, ntiles, mtiles;  // column tiles (all segments), row tiles
    int K, M;
    size_t rb;                 // bytes from a weight row to the next (the rows' own, also where K is a piece of them)
    const uint8_t* xa;         // gemm_prep_kernel's operands of the rows
    const uint8_t* xs;
    const float* rowscale;
    int64_t ldy;
    int accumulate;            // y += result
    int swiglu;                // seg[0] gate, seg[1] up, equal rows: seg[0].y = silu(gate) * up
};

// The 6-bit scale and min of sub-block j (compile time) from the 12 scale
// bytes (header dwords y, z, w), get_scale_min_k4 of q4_k_m.rs:11-22.
__device__ __forceinline__ uint32_t q4_scale(const u32x4& h, int j) {
    const int sh = 8 * (j & 3);
    return j < 4 ? (h.y >> sh) & 63u : ((h.w >> sh) & 0xFu) | (((h.y >> (sh + 6)) & 3u) << 4);
}
__device__ __forceinline__ uint32_t q4_min(const u32x4& h, int j) {
    const int sh = 8 * (j & 3);
    return j < 4 ? (h.z >> sh) & 63u : ((h.w >> (sh + 4)) & 0xFu) | (((h.z >> (sh + 6)) & 3u) << 4);
}
__device__ __forceinline__ _Float16 u2h(uint32_t v) { return (_Float16)(uint16_t)v; }

// Eight bytes c (each 0 .. 255) as fp16 1024 + c: the bits 0x6400 | c.
__device__ __forceinline__ void bytes_1024(uint32_t t0, uint32_t t1, half2v (&h)[4]) {
    h[0] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, t0, 0x07010700u));
    h[1] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, t0, 0x07030702u));
    h[2] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, t1, 0x07010700u));
    h[3] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, t1, 0x07030702u));
}
// c - off: the difference of two fp16 integers below 2048 is exact
__device__ __forceinline__ void bytes_to_half(uint32_t t0, uint32_t t1, float off, half2v (&h)[4]) {
    const half2v o = {(_Float16)(-1024.0f - off), (_Float16)(-1024.0f - off)};
    bytes_1024(t0, t1, h);
#pragma unroll
    for (int e = 0; e < 4; e++) h[e] += o;
}
__device__ __forceinline__ u32x4 pack_half(const half2v (&h)[4]) {
    return u32x4{__builtin_bit_cast(uint32_t, h[0]), __builtin_bit_cast(uint32_t, h[1]),
                 __builtin_bit_cast(uint32_t, h[2]), __builtin_bit_cast(uint32_t, h[3])};
}

// 16 bytes at byte v (per lane) + s (uniform) of a buffer: the address takes
// one register for all the loads of a wave. Past the buffer's end: zeros.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t buffer_of(const uint8_t* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ u32x4 buf16(rsrc_t r, int v, int s) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0);
}

template <bool BF>
__device__ __forceinline__ f32x16 mfma16(const u32x4& a, const u32x4& b, const f32x16& c) {
    if constexpr (BF)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

// value e of eight fp16 or bf16 ones
template <bool BF>
__device__ __forceinline__ float part16_f32(const u32x4& w, int e) {
    const uint32_t b = w[e >> 1] >> (16 * (e & 1));
    return BF ? bf16_bits_to_f32(b) : half_bits_to_f32(b);
}

typedef uint32_t u32x4_a2g __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_a2g __attribute__((ext_vector_type(2), aligned(2)));

template <int FMT, int WN, int KQ, int MT, bool MID>
__global__ void __launch_bounds__(256, 1) gemm_rows_kernel(const RowsArgs a) {
    static_assert(WN * KQ == 4 && (MT == 1 || MT == 2), "four waves");
    static_assert(WN == 1 || FMT == RF_Q4P || FMT == RF_Q4 || FMT == RF_Q6, "wide groups take K-quants");
    constexpr bool BF = FMT == RF_BF16, Q4 = FMT == RF_Q4P || FMT == RF_Q4;
    constexpr int P = BF ? 3 : 2;
    constexpr bool SH = WN > 1;            // the input planes of a k-tile shared through LDS
    constexpr bool CONV = FMT == RF_Q4 || FMT == RF_Q6 || FMT == RF_Q8;  // weights become fp16 in registers
    constexpr int AB = KQ * MT * 4 * P;    // their 1 KB blocks: [depth share][32 rows][k-step][plane]
    constexpr int ABUF = SH ? 4 : 1;
    constexpr int SMEM = SH ? ABUF * AB * kStepBytes : 16;
    constexpr int RED = KQ > 1 ? 4 * MT * 2 * 16 * 64 * 4 : 16;
    __shared__ __attribute__((aligned(16))) uint8_t smem[SMEM > RED ? SMEM : RED];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int wn = wave % WN, kq = wave / WN;
    // tile: with a multiple of eight column tiles, the row tiles of a column
    // tile follow each other on one XCD (workgroup id % 8), so its weights
    // come into one L2
    int tn, tm;
    if ((a.ntiles & 7) == 0) {
        const int slot = blockIdx.x >> 3;
        tn = (slot / a.mtiles) * 8 + (blockIdx.x & 7);
        tm = slot % a.mtiles;
    } else {
        tn = blockIdx.x % a.ntiles;
        tm = blockIdx.x / a.ntiles;
    }
    const int sg = a.nseg > 2 && tn >= a.seg[2].t0 ? 2 : a.nseg > 1 && tn >= a.seg[1].t0 ? 1 : 0;
    const int N = a.seg[sg].n;
    // the wave's two 32-column tiles: weight rows c0 + cj * j of Wj[j] (SwiGLU: the gate's rows and the up's)
    const int cj = a.swiglu ? 0 : 32;
    const int c0 = ((tn - a.seg[sg].t0) * WN + wn) * (32 + cj);
    const uint8_t* const Wj[2] = {a.seg[sg].W, a.swiglu ? a.seg[1].W : a.seg[sg].W};
    const int K = a.K, KS = K / 16, NB = K / 256;
    const int nsb = (NB - kq + KQ - 1) / KQ;  // the wave's super-blocks kq, kq + KQ, ...
    const int nbt = SH ? (NB + KQ - 1) / KQ : nsb;

    // the 64 (32) input rows: per 32 rows KS * P blocks
    const int a_mt = KS * P * kStepBytes;
    const rsrc_t Ar = buffer_of(a.xa + (size_t)(tm * MT) * a_mt, (size_t)MT * a_mt);
    const rsrc_t Sr = buffer_of(Q4 ? a.xs + (size_t)(tm * MT) * NB * kStepBytes : a.xa, (size_t)MT * NB * kStepBytes);
    const int l16 = 16 * lane;
    const uint8_t* Bb[2];   // the lane's row
    rsrc_t Br[2], Hr[2];    // RF_Q4P: the column tile's blocks, its headers
#pragma unroll
    for (int j = 0; j < 2; j++) {
        if constexpr (FMT == RF_Q4P) {
            const int nt = min((c0 + cj * j) / 32, N / 32 - 1);  // (past N: the last tile, computed and not stored)
            Br[j] = buffer_of(Wj[j] + (size_t)nt * KS * kStepBytes, (size_t)KS * kStepBytes);
            Hr[j] = buffer_of(Wj[j] + (size_t)N * K * 2 + (size_t)nt * NB * kGemmHBytes, (size_t)NB * kGemmHBytes);
        } else {
            Bb[j] = Wj[j] + (size_t)min(c0 + cj * j + li, N - 1) * a.rb;
        }
    }

    // Register rings. B (and A when each wave reads its own): slot s holds
    // k-step s of a unit of eight (128 values) and takes the next unit's
    // k-step s once it is used. Shared A: k-tile t + 4 loads while t computes,
    // t + 2 goes into LDS, the fragments are read a pair of k-steps ahead.
    u32x4 A[SH ? 4 : 8][MT][P];     // own: by slot; shared: fragments, two pairs of k-steps
    constexpr int SC = SH ? AB * kStepBytes / 4096 : 1;  // 16-byte chunks of a k-tile per thread
    u32x4 st[2][SC];
    u32x4 B[8][2];                  // operand blocks, F16 / BF16 values
    u32x2 C8[8][2];                 // Q8_0: the k-step's eight quants
    u32x2 Cq[2][2][FMT == RF_Q6 ? 6 : 4];  // Q4_K / Q6_K: code bytes of the unit (by its half)
    uint32_t Dq[2][2][4];           // Q8_0: block scales of the unit
    u32x4 hd[2], hdn[2];            // super-block headers: Q4_K header or mins, Q6_K scales; the next one's
    uint32_t dd[2], ddn[2];         // d | dmin << 16 (RF_Q4P), d (Q6_K)
    u32x4 sm[MT], smn[MT];          // Q4_K: sub-block sums
    f32x16 acc[MT][2], mid[MT][2], c[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x16{};

    // shared A: thread's chunks of k-tile g of the depth shares' super-blocks
    // b (share q: super-block q + KQ b, past the end a re-read of the last)
    auto stage_load = [&](int b, int g, u32x4 (&r)[SC]) {
#pragma unroll
        for (int k = 0; k < SC; k++) {
            // a chunk's block row (share, 32 rows) is uniform over the workgroup:
            // a k-tile of 32 rows is 4 P KB, P chunks of the 256 threads
            const int q = k / (MT * P), i = (k / P) % MT;
            const int sb = min(q + KQ * b, q + KQ * ((NB - q - 1) / KQ));
            r[k] = buf16(Ar, 16 * (int)threadIdx.x, i * a_mt + (16 * sb + 4 * g) * (P * kStepBytes) + (k % P) * 4096);
        }
    };
    auto stage_store = [&](const u32x4 (&r)[SC], int buf) {
#pragma unroll
        for (int k = 0; k < SC; k++) *(u32x4*)(smem + buf * (AB * kStepBytes) + k * 4096 + 16 * threadIdx.x) = r[k];
    };
    auto frag = [&](int buf, int s, int i, int p) {  // k-step s of the k-tile in buf
        return *(const u32x4*)(smem + (buf * AB + ((kq * MT + i) * 4 + s) * P + p) * kStepBytes + 16 * lane);
    };
    auto load_step = [&](int ks, auto S) {  // k-step ks (its unit's slot S)
        constexpr int s = decltype(S)::value;
        if constexpr (!SH) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int p = 0; p < P; p++)
                    A[s][i][p] = buf16(Ar, l16, i * a_mt + (ks * P + p) * kStepBytes);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (FMT == RF_Q4P) B[s][j] = buf16(Br[j], l16, ks * kStepBytes);
            else if constexpr (FMT == RF_F16 || BF) B[s][j] = *(const u32x4_a2g*)(Bb[j] + (size_t)ks * 32 + 16 * lh);
            else if constexpr (FMT == RF_Q8)
                C8[s][j] = *(const u32x2_a2g*)(Bb[j] + (size_t)(ks >> 1) * 34 + 2 + 16 * (ks & 1) + 8 * lh);
        }
    };
    // what a unit (half H of super-block sb) takes beside its k-steps
    auto load_unit = [&](int sb, auto H) {
        constexpr int h = decltype(H)::value;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (FMT == RF_Q4) {
                const uint8_t* q = Bb[j] + (size_t)sb * 144 + 16 + 64 * h + 8 * lh;
#pragma unroll
                for (int g = 0; g < 4; g++) Cq[h][j][g] = *(const u32x2_a2g*)(q + 16 * g);
            } else if constexpr (FMT == RF_Q6) {
                const uint8_t* q = Bb[j] + (size_t)sb * 210 + 8 * lh;
#pragma unroll
                for (int g = 0; g < 4; g++) Cq[h][j][g] = *(const u32x2_a2g*)(q + 64 * h + 16 * g);
#pragma unroll
                for (int g = 0; g < 2; g++) Cq[h][j][4 + g] = *(const u32x2_a2g*)(q + 128 + 32 * h + 16 * g);
            } else if constexpr (FMT == RF_Q8) {
#pragma unroll
                for (int g = 0; g < 4; g++) Dq[h][j][g] = ld_u16(Bb[j] + (size_t)(8 * sb + 4 * h + g) * 34);
            }
        }
    };
    auto load_head = [&](int sb) {
        if constexpr (FMT == RF_Q4P || FMT == RF_Q4 || FMT == RF_Q6) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (FMT == RF_Q4P) {
                    ddn[j] = __builtin_amdgcn_raw_buffer_load_b32(Hr[j], 4 * li, sb * kGemmHBytes, 0);
                    hdn[j] = buf16(Hr[j], 16 * li, sb * kGemmHBytes + 128);
                } else if constexpr (FMT == RF_Q4) {
                    hdn[j] = *(const u32x4_a2g*)(Bb[j] + (size_t)sb * 144);
                } else {
                    hdn[j] = *(const u32x4_a2g*)(Bb[j] + (size_t)sb * 210 + 192);
                    ddn[j] = ld_u16(Bb[j] + (size_t)sb * 210 + 208);
                }
            }
        }
        if constexpr (Q4) {
#pragma unroll
            for (int i = 0; i < MT; i++)
                smn[i] = buf16(Sr, l16, (i * NB + sb) * kStepBytes);
        }
    };
    auto take_head = [&]() {
#pragma unroll
        for (int j = 0; j < 2; j++) { hd[j] = hdn[j]; dd[j] = ddn[j]; }
#pragma unroll
        for (int i = 0; i < MT; i++) sm[i] = smn[i];
    };
    // the B operand of k-step S of half H, column tile j
    auto operand = [&](auto H, auto S, int j, const u32x4& head) -> u32x4 {
        constexpr int h = decltype(H)::value, s = decltype(S)::value;
        if constexpr (FMT == RF_Q4) {
            // group 2h + s / 4; sub-block 2 * group + (s / 2) % 2 (low or high nibbles)
            constexpr int sub = 2 * (2 * h + s / 4) + ((s >> 1) & 1);
            const u32x2 q = Cq[h][j][2 * (s / 4) + (s & 1)];
            const uint32_t t0 = (s >> 1) & 1 ? (q.x >> 4) & 0x0F0F0F0Fu : q.x & 0x0F0F0F0Fu;
            const uint32_t t1 = (s >> 1) & 1 ? (q.y >> 4) & 0x0F0F0F0Fu : q.y & 0x0F0F0F0Fu;
            // sc * q = sc * (1024 + q) - 1024 sc in one exact fma (sc * q <= 945)
            const _Float16 sc = u2h(q4_scale(head, sub));
            const half2v s2 = {sc, sc}, o2 = s2 * half2v{(_Float16)-1024.0f, (_Float16)-1024.0f};
            half2v v[4];
            bytes_1024(t0, t1, v);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = __builtin_elementwise_fma(v[e], s2, o2);
            return pack_half(v);
        } else if constexpr (FMT == RF_Q6) {
            // quarter s / 2 of the half: ql bytes 32 (quarter % 2) + 16 (s % 2), nibble quarter / 2, qh bits 2 quarter
            constexpr int qt = s >> 1;
            const u32x2 l = Cq[h][j][2 * (qt & 1) + (s & 1)], u = Cq[h][j][4 + (s & 1)];
            auto code = [&](uint32_t lo, uint32_t hi) {
                const uint32_t n = qt >= 2 ? (lo >> 4) & 0x0F0F0F0Fu : lo & 0x0F0F0F0Fu;
                const uint32_t b = qt == 0 ? hi << 4 : qt == 1 ? hi << 2 : qt == 2 ? hi : hi >> 2;
                return n | (b & 0x30303030u);
            };
            half2v v[4];
            bytes_to_half(code(l.x, u.x), code(l.y, u.y), 32.0f, v);
            return pack_half(v);
        } else if constexpr (FMT == RF_Q8) {
            half2v v[4];
            bytes_to_half(C8[s][j].x ^ 0x80808080u, C8[s][j].y ^ 0x80808080u, 128.0f, v);
            return pack_half(v);
        } else {
            return B[s][j];
        }
    };

    const int kql = min(kq, NB - 1);  // (a share without super-blocks loads the last one's)
    if (nbt > 0) {
        load_head(kql);
        load_unit(kql, std::integral_constant<int, 0>{});
        if constexpr (SH) {
            u32x4 s0[SC], s1[SC];
            stage_load(0, 0, s0);
            stage_load(0, 1, s1);
            stage_load(0, 2, st[0]);
            stage_load(0, 3, st[1]);
            static_for<0, 8>([&](auto S) { load_step(16 * kql + decltype(S)::value, S); });
            stage_store(s0, 0);
            stage_store(s1, 1);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int p = 0; p < P; p++) A[u][i][p] = frag(0, u, i, p);
        } else {
            static_for<0, 8>([&](auto S) { load_step(16 * kql + decltype(S)::value, S); });
        }
        take_head();
    }
    u32x4 bq[2][2];  // the pair's B operands; CONV: formed a pair ahead, beside the products
    if constexpr (CONV) {
        if (nbt > 0)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                bq[0][j] = operand(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, j, hd[j]);
                bq[1][j] = operand(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, j, hd[j]);
            }
    }
    for (int b = 0; b < nbt; b++) {
        const bool live = b < nsb;  // (wave-uniform; a share may have one super-block fewer)
        const int sb = live ? kq + KQ * b : kql, sbn = b + 1 < nsb ? sb + KQ : sb;  // (past the end: re-read)
        static_for<0, 4>([&](auto G) {
            constexpr int g = decltype(G)::value, h = g / 2;
            using Hc = std::integral_constant<int, h>;
            const int usb = h == 0 ? sb : sbn;  // the next unit: half 1 - h of super-block usb
            if constexpr (g % 2 == 0) {
                load_unit(usb, std::integral_constant<int, 1 - h>{});
                if constexpr (h == 1) load_head(sbn);
            }
            if constexpr (SH) {
                stage_store(st[g & 1], (g + 2) & 3);
                stage_load(b + 1, g, st[g & 1]);
            }
            static_for<0, 2>([&](auto R) {
                constexpr int pr = decltype(R)::value, s0 = 4 * (g & 1) + 2 * pr;  // slots s0, s0 + 1
                using S0 = std::integral_constant<int, s0>;
                using S1 = std::integral_constant<int, s0 + 1>;
                constexpr int f0 = SH ? 2 * pr : s0;  // where the pair's A is
                if constexpr (SH) {  // the next pair's fragments
#pragma unroll
                    for (int u = 0; u < 2; u++)
#pragma unroll
                        for (int i = 0; i < MT; i++)
#pragma unroll
                            for (int p = 0; p < P; p++)
                                A[2 * (1 - pr) + u][i][p] = frag((g + pr) & 3, pr == 0 ? 2 + u : u, i, p);
                }
                u32x4 bn[2][2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if constexpr (CONV) {
                        // the next pair (of the next super-block after the last)
                        constexpr int np = (2 * g + pr + 1) & 7;
                        using Hn = std::integral_constant<int, np / 4>;
                        const u32x4& head = np == 0 ? hdn[j] : hd[j];
                        bn[0][j] = operand(Hn{}, std::integral_constant<int, 2 * (np & 3)>{}, j, head);
                        bn[1][j] = operand(Hn{}, std::integral_constant<int, 2 * (np & 3) + 1>{}, j, head);
                    } else {
                        bq[0][j] = operand(Hc{}, S0{}, j, hd[j]);
                        bq[1][j] = operand(Hc{}, S1{}, j, hd[j]);
                    }
                }
                // Chains start from zero: every k-step for Q6_K (one
                // sub-block), every pair for Q8_0 (one block), otherwise
                // every k-tile, or every super-block without MID (Q4_K).
                // Within a pair the small parts come first, so only the hi
                // parts round at the chain's full size.
#pragma unroll
                for (int q = 0; q < 2 * P; q++) {
                        // (Q8_0, whose chain is one pair: k-step by k-step,
                        // hi then lo, measured closer to the 64-bit result)
                        const int p = FMT == RF_Q8 ? q % P : P - 1 - q / 2, u = FMT == RF_Q8 ? q / P : q % 2;
                        if (FMT == RF_Q6 && u == 1) continue;
                        const bool first = q == 0 && (FMT == RF_Q6 || FMT == RF_Q8 || (pr == 0 && (MID || g == 0)));
#pragma unroll
                        for (int i = 0; i < MT; i++)
#pragma unroll
                            for (int j = 0; j < 2; j++)
                                c[i][j] = mfma16<BF>(A[f0 + u][i][p], bq[u][j], first ? f32x16{} : c[i][j]);
                }
                f32x16 (&sum)[MT][2] = MID ? mid : acc;
                auto fold = [&](int u) {  // sum (+)= f * c
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        float f = 1.0f;
                        if constexpr (FMT == RF_Q6) {
                            const uint32_t w = g == 0 ? hd[j].x : g == 1 ? hd[j].y : g == 2 ? hd[j].z : hd[j].w;
                            f = half_bits_to_f32(dd[j]) * sbyte_f32(w, 2 * pr + u);
                        } else if constexpr (FMT == RF_Q8) {
                            f = half_bits_to_f32(Dq[h][j][s0 >> 1]);
                        }
                        const bool start = MID && g == 0 && u == 0 && (pr == 0 || !(FMT == RF_Q6 || FMT == RF_Q8));
#pragma unroll
                        for (int i = 0; i < MT; i++) {
                            if constexpr (FMT == RF_Q6 || FMT == RF_Q8) {
                                if (start) sum[i][j] = f * c[i][j];
                                else
#pragma unroll
                                    for (int r = 0; r < 16; r++) sum[i][j][r] = fmaf(f, c[i][j][r], sum[i][j][r]);
                            } else {
                                if (start) sum[i][j] = c[i][j];
                                else sum[i][j] += c[i][j];
                            }
                        }
                    }
                };
                if constexpr (FMT == RF_Q6) {
                    fold(0);
#pragma unroll
                    for (int p = P - 1; p >= 0; p--)
#pragma unroll
                        for (int i = 0; i < MT; i++)
#pragma unroll
                            for (int j = 0; j < 2; j++)
                                c[i][j] = mfma16<BF>(A[f0 + 1][i][p], bq[1][j], p == P - 1 ? f32x16{} : c[i][j]);
                    fold(1);
                } else if constexpr (FMT == RF_Q8) {
                    fold(0);
                } else if constexpr (MID && pr == 1) {
                    fold(0);
                }
                load_step(16 * usb + 8 * (1 - h) + s0, S0{});
                load_step(16 * usb + 8 * (1 - h) + s0 + 1, S1{});
                if constexpr (CONV)
#pragma unroll
                    for (int j = 0; j < 2; j++) { bq[0][j] = bn[0][j]; bq[1][j] = bn[1][j]; }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (SH) __syncthreads();
        });
        if (live) {
            if constexpr (Q4) {
                // end of the super-block: acc += d * sums, then the min term
                // dmin * sum_sub m_sub * X_sub as one product over K = 16: the
                // eight hi sums in the lower lane half, the lo sums in the upper
                // one, the mins in both
                u32x4 bm[2];
                float d[2], dm[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if constexpr (FMT == RF_Q4P) {
                        bm[j] = hd[j];
                        d[j] = half_bits_to_f32(dd[j]);
                        dm[j] = half_bits_to_f32(dd[j] >> 16);
                    } else {
                        half2v v[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = half2v{u2h(q4_min(hd[j], 2 * e)), u2h(q4_min(hd[j], 2 * e + 1))};
                        bm[j] = pack_half(v);
                        d[j] = half_bits_to_f32(hd[j].x);
                        dm[j] = half_bits_to_f32(hd[j].x >> 16);
                    }
                    dm[j] *= 32.0f;  // exact: the sums are times 2^-5
                }
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const f32x16 c2 = mfma16<false>(sm[i], bm[j], f32x16{});
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            const float cs = MID ? mid[i][j][r] : c[i][j][r];
                            acc[i][j][r] = fmaf(-dm[j], c2[r], fmaf(d[j], cs, acc[i][j][r]));
                        }
                    }
            } else if constexpr (MID) {
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[i][j] += mid[i][j];
            }
        }
        take_head();
    }

    // the KQ partial sums of the tile, added in a fixed order: wave kq takes
    // register groups [G0, G0 + 4 / KQ) of four rows
    constexpr int NG = 4 / KQ;
    const int g0 = kq * NG;
    float* red = (float*)smem;  // [wave][32 rows, column tile, register][lane]
    constexpr int RW = MT * 2 * 16 * 64;
    if constexpr (KQ > 1) {
        if constexpr (SH) __syncthreads();  // (the last k-tile's fragments are read)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[wave * RW + ((i * 2 + j) * 16 + r) * 64 + lane] = acc[i][j][r];
        __syncthreads();
    }
    // D[i][j] in lane j + 32 * ((i / 4) % 2), register 4 * (i / 8) + i % 4.
    // Every row scale and (with accumulate) every old value is loaded before
    // the first store: a store could alias a later load as far as the
    // compiler knows, which would make each element wait for its own trip.
    float* y = a.seg[sg].y;
    float v[MT][2][NG][4], old[MT][2][NG][4];
    f32x4 rs[MT][NG];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const int m = 32 * (tm * MT + i) + 8 * (g0 + g) + 4 * lh;
            rs[i][g] = *(const f32x4*)(a.rowscale + m);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int n = c0 + cj * j + li;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    old[i][j][g][e] = a.accumulate && m + e < a.M && n < N ? y[(m + e) * a.ldy + n] : 0.f;
                    if constexpr (KQ == 1) {
                        v[i][j][g][e] = acc[i][j][4 * g + e];
                    } else {
                        const int q = ((i * 2 + j) * 16 + 4 * (g0 + g) + e) * 64 + lane;
                        if constexpr (KQ == 2) v[i][j][g][e] = red[wn * RW + q] + red[(wn + WN) * RW + q];
                        else v[i][j][g][e] = (red[q] + red[RW + q]) + (red[2 * RW + q] + red[3 * RW + q]);
                    }
                }
            }
        }
    if constexpr (FMT == RF_F16 || BF) {
        // An infinite weight times a lo part (0, or of the other sign) is NaN
        // where the value itself gives an infinity: outputs that came out
        // infinite or NaN are summed again in f32 from whole weights and
        // inputs, one per lane at a time (ordinary data: none; the test costs
        // 0.2 us of 20).
        static_assert(KQ == 4, "four outputs per column tile and 32 rows");
        float z[4] = {0.f, 0.f, 0.f, 0.f};  // 0 * v summed: 0 unless a v is infinite or NaN
#pragma unroll
        for (int q = 0; q < MT * 8; q++) z[q % 4] = fmaf(v[q / 8][(q / 4) % 2][0][q % 4], 0.f, z[q % 4]);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64((z[0] + z[1]) + (z[2] + z[3]) != 0.f) != 0, 0)) {
            uint32_t again = 0;
#pragma unroll
            for (int q = 0; q < MT * 8; q++) {
                const int i = q / 8, j = (q / 4) % 2, e = q % 4;
                const bool in = 32 * (tm * MT + i) + 8 * g0 + 4 * lh + e < a.M && c0 + cj * j + li < N;
                if (in && !(fabsf(v[i][j][0][e]) <= 3.40282347e38f)) again |= 1u << q;
            }
            while (__builtin_amdgcn_ballot_w64(again != 0)) {
                const int q = again ? __builtin_ctz(again) : 0;
                const int m = 32 * (tm * MT + q / 8) + 8 * g0 + 4 * lh + q % 4;
                const uint8_t* const w = (q / 4) % 2 ? Bb[1] : Bb[0];
                const uint8_t* const x = a.xa + (size_t)(m >> 5) * a_mt + 16 * (m & 31);
                float sum = 0.f;
#pragma unroll 1
                for (int k = 0; k < K / 8; k++) {
                    const u32x4 wk = *(const u32x4_a2g*)(w + (size_t)16 * k);
                    u32x4 xk[P];
#pragma unroll
                    for (int p = 0; p < P; p++)
                        xk[p] = *(const u32x4*)(x + (size_t)((k >> 1) * P + p) * kStepBytes + 512 * (k & 1));
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        float xv = 0.f;
#pragma unroll
                        for (int p = P - 1; p >= 0; p--) xv += part16_f32<BF>(xk[p], e);
                        sum = fmaf(part16_f32<BF>(wk, e), xv, sum);
                    }
                }
#pragma unroll
                for (int k = 0; k < MT * 8; k++)
                    if (again && k == q) v[k / 8][(k / 4) % 2][0][k % 4] = sum;
                again &= again - 1;  // (0 stays 0)
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (a.swiglu && j == 1) continue;
            const int n = c0 + cj * j + li;
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int m = 32 * (tm * MT + i) + 8 * (g0 + g) + 4 * lh + e;
                    if (m < a.M && n < N) {
                        float r = v[i][j][g][e] * rs[i][g][e];
                        if (a.swiglu) r = silu_f(r) * (v[i][1][g][e] * rs[i][g][e]);  // ffn.rs:84-95
                        y[m * a.ldy + n] = a.accumulate ? old[i][j][g][e] + r : r;  // one writer per output
                    }
                }
        }
}

}  // namespace

// types.rs:188-235 validate_matmul_args after lib.rs:152-166
static int32_t validate_matmul(int32_t t, size_t out_len, size_t w_len, size_t in_len, size_t batch, size_t rows,
                               size_t cols) {
    size_t bs, ts, row_bytes, e;
    if (!ggml_sizes(t, &bs, &ts)) return err_unsupported(t);
    if (cols % bs != 0) return err_misaligned(cols, bs);
    if (__builtin_mul_overflow(cols / bs, ts, &row_bytes)) return err_overflow();
    if (__builtin_mul_overflow(batch, rows, &e)) return err_overflow();
    if (out_len < e) return err_buffer_too_small(e, out_len);
    if (__builtin_mul_overflow(batch, cols, &e)) return err_overflow();
    if (in_len < e) return err_buffer_too_small(e, in_len);
    if (__builtin_mul_overflow(rows, row_bytes, &e)) return err_overflow();
    if (w_len < e) return err_buffer_too_small(e, w_len);
    return MIVI_OK;
}

// Device workspaces of the MFMA path: up to kWsSlots grow-only buffers per
// device, one to a stream as far as they reach, so that products of different
// streams run side by side as their GEMVs do (two streams, Q4_K, 4 inputs x 512
// x 4608: 79.6 us a pair on one buffer). Each use waits for the event recorded
// after the buffer's last one, so uses never overlap, whichever stream a
// buffer passes to. They live until the process ends.
constexpr int kWsSlots = 4;
struct GemmWorkspace {
    void* ptr = nullptr;
    size_t bytes = 0;
    hipEvent_t done = nullptr;
    hipStream_t stream = nullptr;  // its last user
    uint64_t used = 0;             // when (0: never)
};
struct GemmWorkspaces {
    std::mutex mu;
    GemmWorkspace slot[kWsSlots];
    uint64_t clock = 0;
};

static GemmWorkspaces& gemm_workspaces(int dev) {
    static std::mutex mu;
    static std::vector<GemmWorkspaces*> all;
    std::lock_guard<std::mutex> lk(mu);
    if ((size_t)dev >= all.size()) all.resize(dev + 1, nullptr);
    if (!all[dev]) all[dev] = new GemmWorkspaces();  // lives until the process ends
    return *all[dev];
}

// The buffer that stream s used last, else one not used yet, else the one
// longest unused.
static GemmWorkspace& workspace_of(GemmWorkspaces& all, hipStream_t s) {
    GemmWorkspace* best = &all.slot[0];
    for (GemmWorkspace& w : all.slot) {
        if (w.used && w.stream == s) return w;
        if (w.used < best->used) best = &w;
    }
    return *best;
}

// 0: the GEMVs, one input or a few at a time; 1: the matrix cores; 2: the
// matrix cores where a workspace can be had. K-quants with K a multiple of
// 2048 from 16 rows on: below, the batched GEMVs read each weight row once
// for up to eight inputs. Other depths and Q8_0, F16 and BF16 rows have one
// GEMV launch per input, so the product pays from a few inputs on.
static int rows_route(int32_t t, const GemvArgs& a) {
    const bool kq = t == MIVI_GGML_Q4_K || t == MIVI_GGML_Q6_K;
    const bool fmt = kq || t == MIVI_GGML_Q8_0 || t == MIVI_GGML_F16 || t == MIVI_GGML_BF16;
    if (!fmt || a.K <= 0 || a.K % 256 || a.ncol > INT32_MAX - 64) return 0;
    if (kq && a.K % 2048 == 0) {
        auto a16 = [](const void* p) { return p == nullptr || (uintptr_t)p % 16 == 0; };
        const bool aligned = a16(a.x) && a16(a.x2) && a16(a.norm_w) && a.xs % 4 == 0;
        return a.ncol >= kMfmaMinBatch && aligned ? 1 : 0;
    }
    // Rows under 1024 columns (narrower than the loader's configurations) keep
    // the GEMVs and with them each matvec's own bits: over a Q8_0 cache one
    // flipped code shows in the logits of a small model. The product is the
    // faster side there too (512 x 512, Q4_K: 4 inputs 18.6 us against 12.5, 128
    // inputs 624 against 13). The GEMVs stage one input row in LDS: longer ones
    // than 12288 are refused there.
    if (a.K < 1024 || a.K > 12288 || a.ncol < kMfmaMinBatchRows) return 0;
    if (t == MIVI_GGML_Q4_K) return 2;  // (4 inputs: 14-32 us against 24-46)
    if (t == MIVI_GGML_Q6_K) {
        // Below 4096 rows a GEMV takes about 1.5 us and 5 for each 4096
        // columns begun, the product 6.5 and 7.6 for each 1024 begun: at four
        // inputs of 512 rows 16 us against 23 at 1024 columns and 41 against
        // 48 at 4608, but 61 against 47.5 at 6400 and 96 against 77 at 12032;
        // from six inputs on the product. More rows fill the GEMVs' CUs (8192
        // x 6400: 61 against 130).
        int64_t n = 0;
        for (int i = 0; i < a.nseg; i++) n += a.seg[i].n;
        return n >= 4096 || a.ncol * (1.5 + 5.0 * ((a.K + 4095) / 4096)) > 6.5 + 7.6 * ((a.K + 1023) / 1024) ? 2 : 0;
    }
    // Q8_0, F16, BF16: a GEMV is near its bytes' time, so few inputs stay
    // with it. Fitted to both sides at 1024 to 8192 rows of 1024 to 4608
    // columns (f16 2048 x 2048: 4 inputs 18 us against 22, 6 inputs 26 against
    // 23; Q8_0 1024 x 4608: 8 inputs 34 against 52, 12 inputs 50 against 52);
    // timed again at 1 to 8192 rows of 1024 to 12288 columns and 4 to 32
    // inputs, it takes the faster side or one within 9 % of it but for Q8_0
    // 4608 x 2048 at 6 inputs (29 us against 25).
    double bytes = 0;
    for (int i = 0; i < a.nseg; i++) bytes += (double)a.seg[i].n * a.K * (t == MIVI_GGML_Q8_0 ? 34.0 / 32 : 2.0);
    const double gemvs = a.ncol * (3.2 + bytes / 4.2e6);
    const double product = 10.0 + a.K * (t == MIVI_GGML_Q8_0 ? 0.0095 : 0.0072) + bytes / 5e6;
    return product < gemvs ? 2 : 0;
}

bool mivi::launch_rows_on_matrix_cores(int32_t t, size_t batch, size_t K) {
    GemvArgs a = {};
    a.seg[0].n = 1;
    a.nseg = 1;
    a.K = (int)std::min<size_t>(K, INT32_MAX);
    a.ncol = (int)std::min<size_t>(batch, INT32_MAX - 64);
    return rows_route(t, a) != 0;
}

// Workgroup shape of a product: WN column groups of 64 by KQ shares of the
// depth, WN * KQ = 4 waves. Wider groups read the inputs fewer times; more
// depth shares make more workgroups where the outputs alone would leave CUs
// idle. Picks the least rounds(workgroups / CUs) * (fixed + super-blocks per
// wave), one workgroup a CU. Against all three widths timed at seven shapes of
// 512 to 16384 rows, 2048 to 8192 columns and 16 to 2048 inputs, within 6 % of
// the fastest for 153 of 168; the rest up to 38 % over it, Q6_K, whose narrow
// groups of 64 rows do better than this says (2048 x 8192, 1024 inputs: 203 us
// wide, 147 narrow), and Q4_K at 512 rows and 2048 inputs (42 us, 31 at two
// column groups). The shares change the order of a row's sums with the number
// of inputs, so its last bits depend on the batch it is in.
struct RowsTile {
    int wn, ntiles;
};
static RowsTile rows_tile(int32_t t, const GemvArgs& a, int mtiles) {
    RowsTile best = {4, 0};
    double least = 0;
    const int wide = (t == MIVI_GGML_Q4_K || t == MIVI_GGML_Q6_K) && a.K % 2048 == 0 ? 4 : 1;
    for (int wn = wide; wn >= 1; wn /= 2) {
        int nt = 0;
        if (a.epilogue == EPI_SWIGLU) nt = (a.seg[0].n + 32 * wn - 1) / (32 * wn);
        else
            for (int i = 0; i < a.nseg; i++) nt += (a.seg[i].n + 64 * wn - 1) / (64 * wn);
        const int kq = 4 / wn, nsb = (a.K / 256 + kq - 1) / kq;
        const double rounds = (double)(((size_t)nt * mtiles + num_cus() - 1) / num_cus());
        const double cost = rounds * (3.0 + nsb * (wn == 4 ? 1.7 : wn == 2 ? 1.9 : 2.2));
        if (best.ntiles == 0 || cost < least) {
            least = cost;
            best = {wn, nt};
        }
    }
    return best;
}

template <int FMT>
static void launch_rows_kernel(const RowsArgs& r, int wn, int mt, hipStream_t s) {
    const dim3 grid((unsigned)(r.ntiles * r.mtiles));
#define LR(WN, MT, MID) hipLaunchKernelGGL((gemm_rows_kernel<FMT, WN, 4 / WN, MT, MID>), grid, dim3(256), 0, s, r)
    // Without MID a chain runs over a whole super-block (Q4_K) and its sums go
    // straight into the accumulators: the depths of the batched GEMVs, in
    // workgroups of any width. Other depths replace f32 GEMVs, which the longer
    // chains would not match (errors at 1024 to 12032 columns: Q4_K 3.7e-7 to
    // 4.0e-7 without MID, 2.7e-7 to 3.3e-7 with it, the matvecs 3.0e-7 to
    // 3.3e-7; Q6_K up to 3.3e-7, 2.4e-7, 2.7e-7), and with MID's sums wide
    // groups of 64 rows do not fit the registers (100 to 3340 bytes a lane
    // spilled).
    if constexpr (FMT == RF_Q4P || FMT == RF_Q4 || FMT == RF_Q6) {
        if (wn == 4) { if (mt == 1) LR(4, 1, false); else LR(4, 2, false); return; }
        if (wn == 2) { if (mt == 1) LR(2, 1, false); else LR(2, 2, false); return; }
        // (the operand copy exists at these depths only)
        if (FMT == RF_Q4P || r.K % 2048 == 0) { if (mt == 1) LR(1, 1, false); else LR(1, 2, false); return; }
    }
    if constexpr (FMT != RF_Q4P) { if (mt == 1) LR(1, 1, true); else LR(1, 2, true); }
#undef LR
}

// Most bytes of input planes one launch takes: longer batches run in slabs of
// rows, so that the workspace stays bounded.
constexpr size_t kRowsSlabBytes = 256u << 20;

// Deepest product of one launch: the kernel addresses the inputs of a tile
// (256 bytes a column) in 32 bits. Deeper rows run in pieces, summed in y.
constexpr size_t kRowsMaxDepth = 1u << 22;

static size_t row_bytes(int32_t t, size_t K) {
    size_t bs, ts;
    format_sizes(t, &bs, &ts);
    return K / bs * ts;
}

static size_t rows_slab(int32_t t, size_t K) {
    const size_t P = t == MIVI_GGML_BF16 ? 3 : 2;
    const size_t row_bytes = K * 2 * P + (t == MIVI_GGML_Q4_K ? K / 8 : 0) + 4;
    return std::max<size_t>(64, kRowsSlabBytes / row_bytes / 64 * 64);
}
size_t mivi::launch_rows_workspace(int32_t t, size_t batch, size_t K) {
    const size_t P = t == MIVI_GGML_BF16 ? 3 : 2;
    const size_t mp = (std::min(batch, rows_slab(t, K)) + 63) / 64 * 64;
    return mp * (K * 2 * P + (t == MIVI_GGML_Q4_K ? K / 8 : 0) + 4);
}

// The product with its workspace at hand; weight rows of Kw columns (Kw > K:
// a piece of them).
static int32_t rows_mfma_in(int32_t t, int pro, const GemvArgs& a, size_t Kw, void* ws, hipStream_t s) {
    const size_t K = (size_t)a.K, P = t == MIVI_GGML_BF16 ? 3 : 2;
    const bool q4 = t == MIVI_GGML_Q4_K, swiglu = a.epilogue == EPI_SWIGLU;
    const size_t slab = rows_slab(t, K);
    const size_t mp0 = (std::min((size_t)a.ncol, slab) + 63) / 64 * 64;
    const size_t bx = mp0 * K * 2 * P, bs = q4 ? mp0 * K / 8 : 0;
    auto a16 = [](const void* p) { return p == nullptr || (uintptr_t)p % 16 == 0; };
    const int vec = a16(a.x) && a16(a.x2) && a16(a.norm_w) && a.xs % 4 == 0;
    bool packed = q4;
    for (int i = 0; i < a.nseg; i++) packed = packed && a.seg[i].wg && a.seg[i].n % 32 == 0;
    for (size_t m0 = 0; m0 < (size_t)a.ncol; m0 += slab) {
        const int M = (int)std::min(slab, (size_t)a.ncol - m0);
        int mt = M <= 32 ? 1 : 2, mtiles = (M + 32 * mt - 1) / (32 * mt);
        RowsArgs r = {};
        r.xa = (const uint8_t*)ws;
        r.xs = q4 ? r.xa + bx : nullptr;
        float* rs = (float*)((uint8_t*)ws + bx + bs);
        r.rowscale = rs;
        r.K = (int)K;
        r.rb = row_bytes(t, Kw);
        r.M = M;
        r.ldy = a.ys;
        r.accumulate = a.accumulate;
        r.swiglu = swiglu;
#define LP(R, PL)                                                                                                    \
    hipLaunchKernelGGL((gemm_prep_kernel<R, PL>), dim3((unsigned)(mtiles * 32 * mt / kPrepRows)), dim3(512), 0, s, a.x + m0 * a.xs, \
                       a.x2 ? a.x2 + m0 * a.xs : nullptr, a.norm_w, a.eps, pro, a.xs, M, (int)K, vec,                \
                       (uint8_t*)ws, (uint8_t*)r.xs, rs)
#define LPR(PL)                                                                                                      \
    if (K <= 2048) LP(4, PL); else if (K <= 4096) LP(8, PL); else if (K <= 8192) LP(16, PL); \
    else LP(0, PL)
        if (P == 3) { LPR(3); } else { LPR(2); }
#undef LPR
#undef LP
        const RowsTile tile = rows_tile(t, a, mtiles);
        int t0 = 0;
        for (int i = 0; i < a.nseg; i++) {
            if (a.seg[i].n == 0) continue;  // (no tiles: left out of the table)
            r.seg[r.nseg++] = {packed ? a.seg[i].wg : a.seg[i].W, a.seg[i].y + m0 * a.ys, a.seg[i].n, t0};
            t0 += (a.seg[i].n + 64 * tile.wn - 1) / (64 * tile.wn);
        }
        if (swiglu) {
            t0 = (a.seg[0].n + 32 * tile.wn - 1) / (32 * tile.wn);  // tiles of 32 gate|up pairs a wave
            r.nseg = 1;  // (seg[1] stays in the table: the up rows)
        }
        r.ntiles = t0;
        if (t0 == 0) break;
        // Tiles of 32 input rows where those of 64 would leave half of the CUs
        // idle: twice the workgroups, each with half the products and sums
        // (Q8_0 128 x 2048 x 2048: 34.1 us on 64 workgroups, 30.3 on 128).
        if (mt == 2 && 2 * (size_t)t0 * mtiles <= (size_t)num_cus()) {
            mt = 1;
            mtiles = (M + 31) / 32;
        }
        r.mtiles = mtiles;
        if (t == MIVI_GGML_Q6_K) launch_rows_kernel<RF_Q6>(r, tile.wn, mt, s);
        else if (t == MIVI_GGML_Q8_0) launch_rows_kernel<RF_Q8>(r, tile.wn, mt, s);
        else if (t == MIVI_GGML_F16) launch_rows_kernel<RF_F16>(r, tile.wn, mt, s);
        else if (t == MIVI_GGML_BF16) launch_rows_kernel<RF_BF16>(r, tile.wn, mt, s);
        else if (packed) launch_rows_kernel<RF_Q4P>(r, tile.wn, mt, s);
        else launch_rows_kernel<RF_Q4>(r, tile.wn, mt, s);
    }
    MIVI_HIP_CHECK(hipGetLastError());
    return MIVI_OK;
}

// Y_s[m * ys + n] (=|+=) sum_k W_s[n, k] * pro(X)[m, k] for the segments s
// of a (K % 256 == 0): one activation split, one product over all segments.
// MIVI_ERR_UNSUPPORTED when the workspace cannot be had.
static int32_t rows_mfma(int32_t t, int pro, const GemvArgs& a, hipStream_t s, const RowsWorkspace& own,
                         size_t Kw = 0) {
    const size_t K = (size_t)a.K;
    if (!Kw) Kw = K;
    if (K > kRowsMaxDepth) {
        if (pro == PRO_RMSNORM || a.epilogue != EPI_STORE)  // (they need whole rows)
            return set_error(MIVI_ERR_UNSUPPORTED, "no row product of %d columns with a norm or SwiGLU", a.K);
        for (size_t k0 = 0; k0 < K; k0 += kRowsMaxDepth) {
            GemvArgs p = a;
            p.K = (int)std::min(kRowsMaxDepth, K - k0);
            p.x += k0;
            if (p.x2) p.x2 += k0;
            for (int i = 0; i < a.nseg; i++) {
                p.seg[i].W += row_bytes(t, k0);
                p.seg[i].wg = nullptr;
            }
            p.accumulate = a.accumulate || k0 > 0;
            if (int32_t rc = rows_mfma(t, pro, p, s, own, Kw)) return rc;
        }
        return MIVI_OK;
    }
    size_t bytes = launch_rows_workspace(t, (size_t)a.ncol, K);
    if (own.p && own.bytes >= bytes) return rows_mfma_in(t, pro, a, Kw, own.p, s);
    int dev = 0;
    MIVI_HIP_CHECK(hipGetDevice(&dev));
    GemmWorkspaces& all = gemm_workspaces(dev);
    std::lock_guard<std::mutex> lk(all.mu);
    GemmWorkspace* ws = &workspace_of(all, s);
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess) (void)hipGetLastError();
    if (cap != hipStreamCaptureStatusNone && (ws->bytes < bytes || ws->stream == s)) {
        // no allocation in a capture, and no wait for what the capturing
        // stream itself ran before it: another stream's buffer, if one will do
        for (GemmWorkspace& w : all.slot)
            if (w.bytes >= bytes && w.stream != s) ws = &w;
    }
    if (ws->bytes < bytes) {
        if (ws->ptr) {
            MIVI_HIP_CHECK(hipEventSynchronize(ws->done));
            MIVI_HIP_CHECK(hipFree(ws->ptr));
            ws->ptr = nullptr;
            ws->bytes = 0;
        }
        if (hipMalloc(&ws->ptr, bytes) == hipSuccess) {
            ws->bytes = bytes;
        } else {
            (void)hipGetLastError();
            ws->ptr = nullptr;
            for (GemmWorkspace& w : all.slot)  // another stream's, after its work
                if (w.bytes >= bytes) ws = &w;
            if (ws->bytes < bytes)
                return set_error(MIVI_ERR_UNSUPPORTED, "no workspace of %zu bytes for the row products", bytes);
        }
    }
    // (no system-scope release at the event: it orders work of this device, and the flush cost 6 us a call)
    if (!ws->done) MIVI_HIP_CHECK(hipEventCreateWithFlags(&ws->done, hipEventDisableTiming | hipEventDisableSystemFence));
    else MIVI_HIP_CHECK(hipStreamWaitEvent(s, ws->done, 0));  // the previous user is done with it
    ws->stream = s;
    ws->used = ++all.clock;
    const int32_t rc = rows_mfma_in(t, pro, a, Kw, ws->ptr, s);
    MIVI_HIP_CHECK(hipEventRecord(ws->done, s));  // (also after an error: some of it may run)
    return rc;
}
namespace mivi {
int32_t launch_pack_q4k_gemm(const uint8_t* src, uint8_t* dst, size_t rows, size_t cols, hipStream_t s) {
    if (rows % 32 || cols % 256 || rows > (size_t)INT32_MAX || cols > (size_t)INT32_MAX)
        return set_error(MIVI_ERR_UNSUPPORTED, "no row-product layout for %zu rows of %zu columns", rows, cols);
    const size_t n = rows / 32 * (cols / kTk) * 4 * 64 + rows / 32 * (cols / 256) * 32;
    if (n == 0) return MIVI_OK;
    hipLaunchKernelGGL(pack_q4k_gemm_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, dst, (int)rows,
                       (int)cols);
    MIVI_HIP_CHECK(hipGetLastError());
    return MIVI_OK;
}

int32_t launch_rows(int32_t t, int pro, const GemvArgs& a, hipStream_t s, const RowsWorkspace& ws) {
    const bool swiglu = a.epilogue == EPI_SWIGLU;
    if (pro == PRO_CONV || (a.epilogue != EPI_STORE && !swiglu))
        return set_error(MIVI_ERR_UNSUPPORTED, "row products take no conv prologue and no such epilogue");
    const int route = rows_route(t, a);
    if (swiglu) {
        // (the models' prefill, with a workspace of its own and never under capture)
        if (route == 0 || a.nseg != 2 || a.seg[1].n != a.seg[0].n || a.accumulate || !ws.p)
            return set_error(MIVI_ERR_UNSUPPORTED, "no SwiGLU row product for this shape");
        return rows_mfma(t, pro, a, s, ws);
    }
    if (route == 1) return rows_mfma(t, pro, a, s, ws);
    if (route == 2) {
        // shapes whose GEMVs need no workspace: those still run them where
        // none can be had (a capturing stream, no memory)
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone) {
            const int32_t rc = rows_mfma(t, pro, a, s, ws);
            if (rc != MIVI_ERR_UNSUPPORTED) return rc;
            clear_error();
        } else {
            (void)hipGetLastError();
        }
    }
    return launch_gemv_ex(t, pro, a, s);
}
}  // namespace mivi

static bool gemm_packable(int32_t t, size_t rows, size_t cols) {
    return t == MIVI_GGML_Q4_K && rows % 32 == 0 && cols % 2048 == 0;
}

extern "C" size_t mivi_hip_gemm_packed_size(int32_t t, size_t rows, size_t cols) {
    return gemm_packable(t, rows, cols) ? mivi::q4k_gemm_packed_bytes(rows, cols) : 0;
}

extern "C" int32_t mivi_hip_pack_weights_gemm(int32_t t, const uint8_t* src, size_t src_len, uint8_t* dst,
                                              size_t dst_len, size_t rows, size_t cols, void* stream) {
    size_t bs, ts, need;
    if (!format_sizes(t, &bs, &ts)) return err_unsupported(t);
    if (cols % bs != 0) return err_misaligned(cols, bs);
    if (!gemm_packable(t, rows, cols))
        return set_error(MIVI_ERR_UNSUPPORTED, "no row-product layout for type %d with %zu rows of %zu columns", t,
                         rows, cols);
    if (__builtin_mul_overflow(rows, (cols / bs) * ts, &need)) return err_overflow();
    if (src_len < need) return err_buffer_too_small(need, src_len);
    const size_t out = mivi::q4k_gemm_packed_bytes(rows, cols);
    if (dst_len < out) return err_buffer_too_small(out, dst_len);
    if (rows && (!src || !dst)) return set_error(MIVI_ERR_INVALID_ARGUMENT, "null buffer");
    if ((uintptr_t)src % 16 || (uintptr_t)dst % 16)
        return set_error(MIVI_ERR_INVALID_ARGUMENT, "weights and packed copy must be 16-byte aligned");
    if (rows && src < dst + out && dst < src + need)
        return set_error(MIVI_ERR_INVALID_ARGUMENT, "packing needs distinct buffers");
    clear_error();
    return mivi::launch_pack_q4k_gemm(src, dst, rows, cols, (hipStream_t)stream);
}

extern "C" int32_t mivi_hip_quantized_matmul_rows_gemm_packed(float* out, size_t out_len, int32_t t,
                                                              const uint8_t* w, size_t w_len, const uint8_t* wg,
                                                              size_t wg_len, const float* in, size_t in_len,
                                                              size_t batch, size_t rows, size_t cols, void* stream) {
    int32_t rc = validate_matmul(t, out_len, w_len, in_len, batch, rows, cols);
    if (rc) return rc;
    if (!gemm_packable(t, rows, cols))
        return set_error(MIVI_ERR_UNSUPPORTED, "no row-product layout for type %d with %zu rows of %zu columns", t,
                         rows, cols);
    const size_t need = mivi::q4k_gemm_packed_bytes(rows, cols);
    if (wg_len < need) return err_buffer_too_small(need, wg_len);
    if (batch == 0 || rows == 0) return clear_error();
    if (!out || !w || !wg || !in) return set_error(MIVI_ERR_INVALID_ARGUMENT, "null buffer");
    if ((uintptr_t)wg % 16) return set_error(MIVI_ERR_INVALID_ARGUMENT, "packed copy must be 16-byte aligned");
    if (rows > (size_t)INT32_MAX || cols > (size_t)INT32_MAX || batch > (size_t)INT32_MAX - 64) return err_overflow();
    clear_error();
    // batch >= kMfmaMinBatch: the matrix cores on the packed copy; fewer
    // rows: the GEMVs on the GGUF rows
    mivi::GemvArgs a = {};
    a.seg[0] = {w, out, (int)rows, wg};
    a.nseg = 1;
    a.K = (int)cols;
    a.x = in;
    a.ncol = (int)batch;
    a.xs = (int64_t)cols;
    a.ys = (int64_t)rows;
    return mivi::launch_rows(t, mivi::PRO_NONE, a, (hipStream_t)stream);
}

extern "C" int32_t mivi_hip_quantized_matmul_rows(float* out, size_t out_len, int32_t t, const uint8_t* w,
                                                  size_t w_len, const float* in, size_t in_len, size_t batch,
                                                  size_t rows, size_t cols, void* stream) {
    int32_t rc = validate_matmul(t, out_len, w_len, in_len, batch, rows, cols);
    if (rc) return rc;
    size_t bs, ts;
    // lib.rs:173-182 (matvec) and :273-277 (dequantize_slice) both reject
    // formats outside the supported set before writing anything.
    if (batch > 0 && rows > 0 && !format_sizes(t, &bs, &ts)) return err_unsupported(t);
    if (batch == 0 || rows == 0) return clear_error();
    if (!out || !w || !in) return set_error(MIVI_ERR_INVALID_ARGUMENT, "null buffer");
    clear_error();
    hipStream_t s = (hipStream_t)stream;
    if (rows > (size_t)INT32_MAX || cols > (size_t)INT32_MAX || batch > (size_t)INT32_MAX - 64) return err_overflow();
    // The matrix cores where rows_route says so; otherwise the GEMVs, the
    // batch's input rows as columns where the streaming kernels take several,
    // else one launch per input row, with the matvecs' own bits (lib.rs:404-457)
    // but on the Q4_K column kernels
    mivi::GemvArgs a = {};
    a.seg[0] = {w, out, (int)rows};
    a.nseg = 1;
    a.K = (int)cols;
    a.x = in;
    a.ncol = (int)batch;
    a.xs = (int64_t)cols;
    a.ys = (int64_t)rows;
    return mivi::launch_rows(t, mivi::PRO_NONE, a, s);
}
