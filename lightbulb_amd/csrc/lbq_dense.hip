// lbq_dense.hip -- QMatMul over dense F32 / F16 / BF16 weights.
//
// candle's QMatMul::from_qtensor does not keep F32 / F16 / BF16 tensors
// quantised: it dequantises them (F16 and BF16 widened exactly to f32) and forward is a
// plain f32 matmul, y = x . W^T (the dense variant; the reference reaches it for
// whatever type output.weight or a projection has, custom_transformer.rs:360-363,
// custom_attention.rs:195-206, mlp_wrapper.rs:127-135).  Here the weight stays
// in its file layout ([n][k], f16, bf16 or f32) and is widened on the fly:
//   m <= 8  k_dense_gemv: waves stream weight rows in 4096-column units with
//           the next unit's 16-byte loads in flight, x staged in LDS, f32 FMA
//           against up to 8 activation rows, DPP row sums -- HBM-bound like the
//           quantised decode GEMV;
//   m > 8   k_dense_mm (F16 / BF16), k_dense_mm32 (F32): x as three bf16 operands that add
//           up to it, an F16 weight as two and an F32 weight as three, on the 16-bit
//           matrix cores with f32 accumulation;
//           k_dense_gemm (calls without a workspace): 64 x 128
//           output tiles on v_mfma_f32_32x32x2_f32, operands staged through LDS.
// Every product is formed at f32 precision and summed in f32; only the
// summation order differs from candle's, so results agree to f32 rounding (~1e-6
// relative on a row).
#include <algorithm>

#include "lbq_device.hpp"
#include "lbq_internal.hpp"

namespace lbq {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// 8 consecutive weights of row `row` at column c (c % 8 == 0) widened to f32
template <bool F16, bool BF = false>
__device__ __forceinline__ void load_w8(const uint8_t *row, int64_t c, float w[8]) {
    if constexpr (F16) {
        const uint4 v = *reinterpret_cast<const uint4 *>(row + 2 * c);
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w[2 * i] = w16<BF>(d[i] & 0xffffu);
            w[2 * i + 1] = w16<BF>(d[i] >> 16);
        }
    } else {
        const float4 a = *reinterpret_cast<const float4 *>(row + 4 * c);
        const float4 b = *reinterpret_cast<const float4 *>(row + 4 * c + 16);
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
        w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
    }
}

// ---------------------------------------------------------------------------
// m <= 8.  Waves take rows gw, gw + nw, ...; a row is cut into units of 512 UN
// columns (a lane covers 8 consecutive columns per 512-column step; k % 8 == 0,
// a partial last step is masked), and each wave keeps the next unit's weight
// loads in flight while it computes the current one.  With XL the x rows are
// staged in LDS once per workgroup (m k f32 <= 64 KB), else every wave reads
// them through the caches.
// ---------------------------------------------------------------------------
// 8 consecutive values of x at c (vec: 16-byte aligned, else four-byte loads)
__device__ __forceinline__ void load_x8(const float *p, bool vec, float v[8]) {
    load4f(p, vec, v);
    load4f(p + 4, vec, v + 4);
}

constexpr int DENSE_XL_BYTES = 65536;  // x staged in LDS up to this size

template <bool F16>
struct DenseUnit {
    static constexpr int UN = 8;  // 4096 f16 / 4096 f32 weights of a row per unit and wave
    uint4 w[F16 ? UN : 2 * UN];
};

template <bool F16, int MR, bool XL, bool BF = false>
__global__ __launch_bounds__(256) void k_dense_gemv(const uint8_t *__restrict__ W, int64_t N, int64_t K,
                                                    const float *__restrict__ x, int m, float *__restrict__ y) {
    extern __shared__ __align__(16) float xs[];  // XL: x [m][K]
    const bool xv = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;  // K % 8 == 0: every row likewise
    constexpr int UN = DenseUnit<F16>::UN;
    constexpr int64_t WB = F16 ? 2 : 4, CH = 512 * UN;
    const int t = threadIdx.x, lane = t & 63;
    if constexpr (XL) {
        const int64_t total = (int64_t)m * K;
        if (xv) {
            for (int64_t i = 4 * t; i < total; i += 1024)
                *reinterpret_cast<float4 *>(xs + i) = *reinterpret_cast<const float4 *>(x + i);
        } else {
            for (int64_t i = t; i < total; i += 256) xs[i] = x[i];
        }
        __syncthreads();
    }
    const int64_t gw = (int64_t)blockIdx.x * 4 + (t >> 6), nw = (int64_t)gridDim.x * 4;
    const int64_t nch = (K + CH - 1) / CH;
    const int64_t rows = gw < N ? (N - gw + nw - 1) / nw : 0, units = rows * nch;
    auto load = [&](int64_t u, DenseUnit<F16> &d) {
        const uint8_t *row = W + (gw + (u / nch) * nw) * K * WB;
        const int64_t c0 = (u % nch) * CH;
#pragma unroll
        for (int v = 0; v < UN; v++) {
            const int64_t c = c0 + 512 * v + 8 * lane;
            if constexpr (F16) {
                d.w[v] = c < K ? *reinterpret_cast<const uint4 *>(row + 2 * c) : make_uint4(0, 0, 0, 0);
            } else {
                d.w[2 * v] = c < K ? *reinterpret_cast<const uint4 *>(row + 4 * c) : make_uint4(0, 0, 0, 0);
                d.w[2 * v + 1] = c < K ? *reinterpret_cast<const uint4 *>(row + 4 * c + 16) : make_uint4(0, 0, 0, 0);
            }
        }
    };
    float acc[MR];
#pragma unroll
    for (int i = 0; i < MR; i++) acc[i] = 0.f;
    auto compute = [&](int64_t u, const DenseUnit<F16> &d) {
        const int64_t c0 = (u % nch) * CH;
#pragma unroll
        for (int v = 0; v < UN; v++) {
            const int64_t c = c0 + 512 * v + 8 * lane;
            if (c >= K) continue;
            float w[8];
            if constexpr (F16) {
                const uint32_t dw[4] = {d.w[v].x, d.w[v].y, d.w[v].z, d.w[v].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    w[2 * e] = w16<BF>(dw[e] & 0xffffu);
                    w[2 * e + 1] = w16<BF>(dw[e] >> 16);
                }
            } else {
                const uint4 a = d.w[2 * v], b = d.w[2 * v + 1];
                w[0] = __uint_as_float(a.x); w[1] = __uint_as_float(a.y); w[2] = __uint_as_float(a.z); w[3] = __uint_as_float(a.w);
                w[4] = __uint_as_float(b.x); w[5] = __uint_as_float(b.y); w[6] = __uint_as_float(b.z); w[7] = __uint_as_float(b.w);
            }
#pragma unroll
            for (int i = 0; i < MR; i++) {
                if (i < m) {
                    float xv8[8];
                    if constexpr (XL) {
                        const float4 p = *reinterpret_cast<const float4 *>(xs + (int64_t)i * K + c);
                        const float4 q = *reinterpret_cast<const float4 *>(xs + (int64_t)i * K + c + 4);
                        xv8[0] = p.x; xv8[1] = p.y; xv8[2] = p.z; xv8[3] = p.w;
                        xv8[4] = q.x; xv8[5] = q.y; xv8[6] = q.z; xv8[7] = q.w;
                    } else {
                        load_x8(x + (int64_t)i * K + c, xv, xv8);
                    }
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[i] = fmaf(w[e], xv8[e], acc[i]);
                }
            }
        }
        if (u % nch == nch - 1) {  // the row's last unit: its sums
            const int64_t r = gw + (u / nch) * nw;
#pragma unroll
            for (int i = 0; i < MR; i++) {
                if (i < m) {
                    const float s = row_sum_f32(acc[i]);
                    const float tt = __int_as_float(rl(__float_as_uint(s), 0)) + __int_as_float(rl(__float_as_uint(s), 16)) +
                                     __int_as_float(rl(__float_as_uint(s), 32)) + __int_as_float(rl(__float_as_uint(s), 48));
                    if (lane == 0) y[(int64_t)i * N + r] = tt;
                }
                acc[i] = 0.f;
            }
        }
    };
    DenseUnit<F16> ring[2];
    if (units > 0) load(0, ring[0]);
    for (int64_t u = 0; u < units; u += 2) {
        if (u + 1 < units) load(u + 1, ring[1]);
        compute(u, ring[0]);
        if (u + 1 >= units) break;
        if (u + 2 < units) load(u + 2, ring[0]);
        compute(u + 1, ring[1]);
    }
}

// ---------------------------------------------------------------------------
// m > 8.  Workgroup tile 64 (m) x 128 (n), four waves; wave w owns columns
// 32w..32w+31 for all 64 rows (two 32 x 32 MFMA tiles that share the B operand).
// k advances in stages of 64: x [64][64] and W [128][64] (f16 widened) are stored
// k-major into LDS (row stride padded), then 32 k-steps of
// v_mfma_f32_32x32x2_f32: lane l supplies A[row l%32][k 2s + l/32] and
// B[k 2s + l/32][column l%32].  The next stage's global loads are issued into
// registers before the current stage's MFMAs, so their latency hides behind 64
// MFMAs (F16 4096^2 at M = 512: 276 -> 254 us against 32-deep stages loaded
// after the previous stage's MFMAs).  Out-of-range rows, columns and k read as
// zero.
// ---------------------------------------------------------------------------
constexpr int DBM = 64, DBN = 128, DBK = 64;

template <bool F16>
struct DenseStage {
    float4 x[4];                    // x rows (t / 16) + 16 j, k 4 (t % 16)
    uint4 w[F16 ? 4 : 8];           // W rows (t / 8) + 32 j, k 8 (t % 8): f16 x 8, or f32 x 8 as two
};

template <bool F16, bool BF = false>
__global__ __launch_bounds__(256) void k_dense_gemm(const uint8_t *__restrict__ W, int64_t N, int64_t K,
                                                    const float *__restrict__ x, int64_t M, float *__restrict__ y) {
    __shared__ float As[DBK][DBM + 4];
    __shared__ float Bs[DBK][DBN + 4];
    constexpr int64_t WB = F16 ? 2 : 4;
    const bool xv = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, h = lane >> 5, lr = lane & 31;
    const int64_t m0 = (int64_t)blockIdx.y * DBM, n0 = (int64_t)blockIdx.x * DBN;
    floatx16 acc[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[i][v] = 0.f;
    auto load = [&](int64_t k0, DenseStage<F16> &g) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = (t >> 4) + 16 * j, kk = 4 * (t & 15);
            float v[4] = {0.f, 0.f, 0.f, 0.f};
            if (m0 + r < M && k0 + kk < K) load4f(x + (m0 + r) * K + k0 + kk, xv, v);
            g.x[j] = make_float4(v[0], v[1], v[2], v[3]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = (t >> 3) + 32 * j, kk = 8 * (t & 7);
            const bool ok = n0 + r < N && k0 + kk < K;
            const uint8_t *src = W + (n0 + r) * K * WB + (k0 + kk) * WB;
            if constexpr (F16) {
                g.w[j] = ok ? *reinterpret_cast<const uint4 *>(src) : make_uint4(0, 0, 0, 0);
            } else {
                g.w[2 * j] = ok ? *reinterpret_cast<const uint4 *>(src) : make_uint4(0, 0, 0, 0);
                g.w[2 * j + 1] = ok ? *reinterpret_cast<const uint4 *>(src + 16) : make_uint4(0, 0, 0, 0);
            }
        }
    };
    auto store = [&](const DenseStage<F16> &g) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = (t >> 4) + 16 * j, kk = 4 * (t & 15);
            As[kk][r] = g.x[j].x; As[kk + 1][r] = g.x[j].y; As[kk + 2][r] = g.x[j].z; As[kk + 3][r] = g.x[j].w;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = (t >> 3) + 32 * j, kk = 8 * (t & 7);
            float w[8];
            if constexpr (F16) {
                const uint32_t d[4] = {g.w[j].x, g.w[j].y, g.w[j].z, g.w[j].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    w[2 * e] = w16<BF>(d[e] & 0xffffu);
                    w[2 * e + 1] = w16<BF>(d[e] >> 16);
                }
            } else {
                const uint4 a = g.w[2 * j], b = g.w[2 * j + 1];
                w[0] = __uint_as_float(a.x); w[1] = __uint_as_float(a.y); w[2] = __uint_as_float(a.z); w[3] = __uint_as_float(a.w);
                w[4] = __uint_as_float(b.x); w[5] = __uint_as_float(b.y); w[6] = __uint_as_float(b.z); w[7] = __uint_as_float(b.w);
            }
#pragma unroll
            for (int e = 0; e < 8; e++) Bs[kk + e][r] = w[e];
        }
    };
    DenseStage<F16> g;
    load(0, g);
    store(g);
    __syncthreads();
    for (int64_t k0 = 0; k0 < K; k0 += DBK) {
        const bool more = k0 + DBK < K;
        if (more) load(k0 + DBK, g);  // in flight during this stage's MFMAs
#pragma unroll
        for (int s = 0; s < DBK / 2; s++) {
            const float b = Bs[2 * s + h][32 * wave + lr];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float a = As[2 * s + h][32 * i + lr];
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
            }
        }
        __syncthreads();
        if (more) {
            store(g);
            __syncthreads();
        }
    }
    // D layout of a 32 x 32 tile: lane holds column l%32, rows 8(v/4) + 4h + v%4
    const int64_t n = n0 + 32 * wave + lr;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int64_t m = m0 + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m < M && n < N) y[m * N + n] = acc[i][v];
        }
}


// ---------------------------------------------------------------------------
// m > 8 with F16 / BF16 weights.  x enters as three bf16 operands (k_dense_pieces) whose
// sum is x; a BF16 weight is an operand as it lies in memory, and an F16 weight, 11 bits,
// is the sum of two bf16 values that a wave forms in registers (dense_split2).  All
// products, three or six of them, are taken, and each is exact in the f32 accumulator
// of v_mfma_f32_32x32x16_bf16, so only the f32 summation rounds: an output is as good as
// an f32 product's whatever the range of its row.  (Two fp16 operands for x at one
// exponent a row took a third of the MFMAs, but lose what lies 2^-17 and more below the
// row's largest |x|, which may well meet a zero weight.)
// Range.  x, and an F32 weight, is taken times 2^24 (DENSE_UP), results times 2^-24 for
// each: the last bit of the smallest f32, 2^-149, is then a normal bf16, so that nothing
// is too small for its operands to add up to it.  What is too large for the factor
// (2^104, results 2^80 with F32 weights) gives an infinity and is formed again (below).
// Bound by the matrix cores from M = 512 (1.0-1.5 PFLOP/s of operand products), by the
// launches below.  Against k_dense_gemm, us per call and relative error against 64 bits:
//   F16 4096^2    M = 9 / 64 / 512   236 / 240 / 243 -> 16.2 / 25.9 / 91.9, 1.2e-6 -> 1.2e-7 / 1.2e-7 / 2.7e-7
//   F16 8192^2    M = 2048           2976 -> 1144, 1.6e-6 -> 5.7e-7
//   BF16 4096^2   M = 32 / 512       238 / 245 -> 17.1 / 58.1, 1.2e-6 -> 1.2e-7 / 2.7e-7
//   BF16 8192^2   M = 2048           2980 -> 654,  1.6e-6 -> 5.7e-7
//   F16 512^2     M = 9              32.1 -> 12.6, 4.1e-7 -> 9.1e-8
//
// Tiles.  A workgroup of WM x WN waves owns BM = 32 WM TM rows of x and
// BN = 32 WN TN weight rows; a wave its TM x TN tiles of 32 x 32.  k advances in
// stages of 64: the 3 x BM x 64 pieces and the BN x 64 weights go into LDS by
// buffer loads to LDS (16 B a lane, 8 rows of 128 B an instruction), two buffers;
// row r's 16-byte chunk c sits in slot c ^ ((r >> 1) & 7), so the 32 rows of an
// operand read spread over the banks.  One barrier a stage, before its last k-step:
// there every wave has read the whole stage (and its own loads of the next one have
// landed), so the buffer is refilled, and the next stage's first operands are
// read, under the last k-step's MFMAs.  Rows past N and k past K read as zero
// (outside the buffer resource); rows past M are never stored.
// Few tiles: k is split over workgroups whose partial sums k_dense_sum adds in
// slice order.
//
// A result that is not finite is formed again from x and W on the f32 matrix cores
// (dense_tile): an infinity in x or W would otherwise meet the zero pieces.  A wave does
// that once for a 32 x 32 tile, so that a batch of nothing but NaN costs one such pass
// (F16 4096^2 M = 512 0.33 ms, k_dense_gemm 0.26), and a finite result keeps its bits whatever stands beside it.
// ---------------------------------------------------------------------------
constexpr int DK = 64;  // values of k per stage
constexpr float DENSE_UP = 0x1p24f;
template <bool W32>
constexpr float dense_down() { return W32 ? 0x1p-48f : 0x1p-24f; }

typedef __bf16 dbf8 __attribute__((ext_vector_type(8)));
typedef __bf16 dbf2 __attribute__((ext_vector_type(2)));
typedef float dfl2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ floatx16 dense_mfma(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(dbf8, a), __builtin_bit_cast(dbf8, b), c, 0, 0, 0);
}

// two values' bf16 (nearest), value 0 in the low half; v keeps what is left
__device__ __forceinline__ uint32_t dense_split2(float &v0, float &v1) {
    const dfl2 f = {v0, v1};
    const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, dbf2));
    v0 -= __uint_as_float(b << 16);
    v1 -= __uint_as_float(b & 0xffff0000u);
    return b;
}

__device__ __forceinline__ bool dense_finite(float v) { return fabsf(v) <= 3.4028234664e38f; }  // false for NaN

// The f32 products of x rows mt .. mt + 31 and this lane's weight row n (l % 32 of the
// tile), in the layout of the accumulators; the whole wave calls it.  A lane takes four
// values of k at a time, its half h those from 8 i + 4 h.
template <bool BF, bool W32>
__device__ __attribute__((noinline)) floatx16 dense_tile(const float *x, const uint8_t *W, int64_t K, int64_t M, int64_t N,
                                                         int64_t mt, int64_t n) {
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int64_t m = mt + (lane & 31);
    const uintptr_t xr = reinterpret_cast<uintptr_t>(x + (m < M ? m : M - 1) * K + 4 * h);
    const uint8_t *wr = W + ((n < N ? n : N - 1) * K + 4 * h) * (W32 ? 4 : 2);
    floatx16 acc = {};
    for (int64_t k0 = 0; k0 < K; k0 += 32) {  // four loads of each in flight
        float a[4][4], w[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t k = k0 + 8 * u < K ? k0 + 8 * u : 0;
            const u32x4a4 v = gld16(reinterpret_cast<gbytes_c>(xr + 4 * k));
            a[u][0] = __uint_as_float(v.x); a[u][1] = __uint_as_float(v.y);
            a[u][2] = __uint_as_float(v.z); a[u][3] = __uint_as_float(v.w);
            if constexpr (W32) {
                const float4 b = *reinterpret_cast<const float4 *>(wr + 4 * k);
                w[u][0] = b.x; w[u][1] = b.y; w[u][2] = b.z; w[u][3] = b.w;
            } else {
                const uint2 b = *reinterpret_cast<const uint2 *>(wr + 2 * k);
                w[u][0] = w16<BF>(b.x & 0xffffu); w[u][1] = w16<BF>(b.x >> 16);
                w[u][2] = w16<BF>(b.y & 0xffffu); w[u][3] = w16<BF>(b.y >> 16);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k0 + 8 * u < K)
#pragma unroll
                for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][i], w[u][i], acc, 0, 0, 0);
    }
    return acc;
}

// One 32 x 32 tile of results from row mt on: without the operands' factor, and those that
// are not finite formed again.  0 * r summed over the lane's sixteen is a NaN if any of
// them is not finite, of rows past M too.
template <bool BF, bool W32>
__device__ __forceinline__ void dense_results(floatx16 &acc, int64_t mt, int64_t M, int64_t N, int64_t n, int h, const float *x,
                                              const uint8_t *W, int64_t K) {
    acc *= dense_down<W32>();
    float z = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) z = fmaf(acc[v], 0.f, z);
    if (!__any(z != 0.f)) return;
    bool bad = false;
#pragma unroll
    for (int v = 0; v < 16; v++) bad = bad || (mt + 8 * (v >> 2) + 4 * h + (v & 3) < M && n < N && !dense_finite(acc[v]));
    if (!__any(bad)) return;
    const floatx16 f = dense_tile<BF, W32>(x, W, K, M, N, mt, n);
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] = dense_finite(acc[v]) ? acc[v] : f[v];
}

// x [M][K] -> pieces [3][rows][Kp] of 2^24 x (Kp = K up to a multiple of DK, zero filled);
// one workgroup per row of x
__global__ __launch_bounds__(256) void k_dense_pieces(const float *__restrict__ x, int64_t K, int64_t Kp, int64_t rows,
                                                      unsigned short *__restrict__ A) {
    const int64_t m = blockIdx.x;
    const bool xv = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    const float *xr = x + m * K;
    unsigned short *a = A + m * Kp;
    const int64_t ps = rows * Kp;
    for (int64_t c = 8 * threadIdx.x; c < Kp; c += 8 * blockDim.x) {
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (c < K) load_x8(xr + c, xv, v);
        uint32_t pc[3][4];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            uint32_t b[3];
            v[i] *= DENSE_UP;
            const uint32_t u0 = __float_as_uint(v[i]);
            const bool fin = dense_finite(v[i]);
            // a NaN keeps a mantissa bit in the upper half
            b[0] = (u0 >> 16) | (v[i] != v[i] ? 0x40u : 0u);
            const float r1 = v[i] - __uint_as_float(u0 & 0xffff0000u);
            const uint32_t u1 = fin ? __float_as_uint(r1) : 0u;
            b[1] = u1 >> 16;
            b[2] = fin ? __float_as_uint(r1 - __uint_as_float(u1 & 0xffff0000u)) >> 16 : 0u;
#pragma unroll
            for (int p = 0; p < 3; p++) {
                if (i & 1) pc[p][i >> 1] |= b[p] << 16;
                else pc[p][i >> 1] = b[p];
            }
        }
#pragma unroll
        for (int p = 0; p < 3; p++)
            *reinterpret_cast<uint4 *>(a + p * ps + c) = make_uint4(pc[p][0], pc[p][1], pc[p][2], pc[p][3]);
    }
}

// a buffer resource over [p, p + bytes), wave-uniform
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dense_rsrc(const void *p, int64_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
                       ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)) << 32);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(u), (short)0,
                                             __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}

struct DenseGrid {
    int tiles_m, tiles_n, splits, sps;  // sps: stages of k per split
    int64_t rows, Kp;                   // rows of a piece, its row length
    int64_t split_stride;               // partials apart (0: out is y)
};

template <bool BF, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void k_dense_mm(const uint8_t *__restrict__ W, int64_t N, int64_t K,
                                                           const unsigned short *__restrict__ A, const float *__restrict__ x,
                                                           int64_t M, float *__restrict__ out, DenseGrid g) {
    constexpr int P = 3;
    constexpr int NW = WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
    constexpr int RA = BM / 8 / NW, RB = BN / 8 / NW;  // staging instructions per wave: RA per piece, RB
    static_assert(RA * 8 * NW == BM && RB * 8 * NW == BN && NW % 2 == 0, "whole staging instructions per wave");
    __shared__ __align__(1024) uint8_t As0[P * BM * 128], As1[P * BM * 128];
    __shared__ __align__(1024) uint8_t Bs0[BN * 128], Bs1[BN * 128];
    // tiles that share weight rows on one XCD
    const int G = (int)gridDim.x, L = (int)blockIdx.x;
    const int T = (G & 7) == 0 ? (L & 7) * (G >> 3) + (L >> 3) : L;
    const int tm = T % g.tiles_m, tn = (T / g.tiles_m) % g.tiles_n, z = T / (g.tiles_m * g.tiles_n);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int s0 = z * g.sps, ns = min(g.sps, (int)(g.Kp / DK) - s0);  // ns >= 1
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, lr = lane & 31;
    const int wm = wave / WN, wn = wave % WN;

    const __amdgpu_buffer_rsrc_t a0 = dense_rsrc(A + m0 * g.Kp, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t a1 = dense_rsrc(A + (g.rows + m0) * g.Kp, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t a2 = dense_rsrc(A + (2 * g.rows + m0) * g.Kp, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t br = dense_rsrc(W + n0 * K * 2, (N - n0 < BN ? N - n0 : BN) * K * 2);
    // lane l of an instruction fills row l/8, slot l%8 of its 8 rows; the rows' number
    // / 8 has the wave's parity (NW is even)
    const int ch = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
    const uint32_t va = (uint32_t)((lane >> 3) * (int)g.Kp * 2 + 16 * ch);
    const uint32_t vb = (uint32_t)((lane >> 3) * (int)K * 2 + 16 * ch);
    // stage s (of the slice) into buffer `buf`; past the slice, zeros (no memory access).
    // Straight-line code with the buffers' names in it: a load to LDS that the compiler
    // cannot tell from a read's buffer makes it wait for the load before the read.
    auto stage_in = [&](int s, int buf) __attribute__((always_inline)) {
        const int k0 = (s0 + s) * DK;
        const uint32_t v0 = s < ns ? va : 0x80000000u;
#pragma unroll
        for (int p = 0; p < P; p++)
#pragma unroll
            for (int j = 0; j < RA; j++) {
                const int rb = wave + NW * j;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    p == 0 ? a0 : p == 1 ? a1 : a2, (__attribute__((address_space(3))) void *)((buf ? As1 : As0) + (p * BM + 8 * rb) * 128), 16, v0,
                    (8 * rb * (int)g.Kp + k0) * 2, 0, 0);
            }
        const uint32_t v1 = s < ns && k0 + 8 * ch < (int)K ? vb : 0x80000000u;  // past K: zero
#pragma unroll
        for (int j = 0; j < RB; j++) {
            const int rb = wave + NW * j;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                br, (__attribute__((address_space(3))) void *)((buf ? Bs1 : Bs0) + 8 * rb * 128), 16, v1,
                (8 * rb * (int)K + k0) * 2, 0, 0);
        }
    };
    // byte offsets of a lane's operands of k-step ks, kept as plain numbers (a chain of
    // pointer steps hides from the compiler which buffer it points into)
    int oa[4], ob[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
        const int o = lr * 128 + 16 * ((2 * ks + h) ^ ((lr >> 1) & 7));
        oa[ks] = o + wm * TM * 4096;
        ob[ks] = o + wn * TN * 4096;
        asm volatile("" : "+v"(oa[ks]), "+v"(ob[ks]));
    }

    // sums of the first pieces' products, and of the others, which are 2^-7 of them and
    // less: a rounding at the size of the result an MFMA step instead of three to eight
    floatx16 acc[TM][TN] = {}, low[TM][TN] = {};
    // operands of this k-step and the next: a weight's (BF) or its two pieces', x's pieces;
    // the next one's F16 weights
    constexpr int Q = BF ? 1 : 2, NA = P * TM, NM = P * Q * TM * TN;
    uint4 xa[2][NA], wb[2][TN][Q], raw[TN];
    auto read = [&](int buf, int ks, int r, int q) __attribute__((always_inline)) {
        if (q < TN) (BF ? wb[r][q][0] : raw[q]) = *reinterpret_cast<const uint4 *>((buf ? Bs1 : Bs0) + (ob[ks] + q * 4096));
        else
            xa[r][q - TN] = *reinterpret_cast<const uint4 *>((buf ? As1 : As0) +
                                                             (oa[ks] + (q - TN) / TM * (BM * 128) + (q - TN) % TM * 4096));
    };
    // pair c (two F16 weights) of raw -> wb[r]
    auto split = [&](int r, int c) __attribute__((always_inline)) {
        const int j = c >> 2, e = c & 3;
        const uint32_t u = e == 0 ? raw[j].x : e == 1 ? raw[j].y : e == 2 ? raw[j].z : raw[j].w;
        float v0 = w16<false>(u & 0xffffu), v1 = w16<false>(u >> 16);
#pragma unroll
        for (int p = 0; p < Q; p++) {
            const uint32_t b = dense_split2(v0, v1);
            if (e == 0) wb[r][j][p].x = b;
            else if (e == 1) wb[r][j][p].y = b;
            else if (e == 2) wb[r][j][p].z = b;
            else wb[r][j][p].w = b;
        }
    };
    // the MFMAs of the k-step in xa[r], wb[r], each followed by its share of the next one's
    // reads and, F16, after half of them of its splits
    auto step = [&](int r, int buf, int ks) __attribute__((always_inline)) {
        constexpr int H = BF ? NM : NM / 2, NR = TN + NA;
#pragma unroll
        for (int u = 0; u < NM; u++) {
            const int j = u % TN, i = u / TN % TM, p = u / TN / TM;
            floatx16 &to = p ? low[i][j] : acc[i][j];
            to = dense_mfma(xa[r][p / Q * TM + i], wb[r][j][p % Q], to);
            if (u < H) {
#pragma unroll
                for (int q = u * NR / H; q < (u + 1) * NR / H; q++) read(buf, ks, r ^ 1, q);
            } else {
#pragma unroll
                for (int c = (u - H) * 4 * TN / (NM - H + BF); c < (u - H + 1) * 4 * TN / (NM - H + BF); c++) split(r ^ 1, c);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    stage_in(0, 0);
    stage_in(1, 1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TN + NA; q++) read(0, 0, 0, q);
    if constexpr (!BF)
#pragma unroll
        for (int c = 0; c < 4 * TN; c++) split(0, c);
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < 3; ks++) step(ks & 1, buf, ks + 1);
        __builtin_amdgcn_s_waitcnt(0);  // this wave's operands, and its loads of stage s + 1
        __syncthreads();
        stage_in(s + 2, buf);
        __builtin_amdgcn_sched_barrier(0);
        step(1, buf ^ 1, 0);
    };
    for (int s = 0; s < ns; s += 2) {  // an odd count ends with a stage of zeros
        stage(s, 0);
        stage(s + 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0);  // the loads past the slice
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] += low[i][j];
    float *y = out + (int64_t)z * g.split_stride;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int64_t mt = m0 + 32 * (wm * TM + i), n = n0 + 32 * (wn * TN + j) + lr;
            if (g.split_stride == 0) dense_results<BF, false>(acc[i][j], mt, M, N, n, h, x, W, K);
            if constexpr (TM * TN >= 4) {
                store_tile(y + mt * N, M - mt, N, n, h, [&](int v) __attribute__((always_inline)) { return acc[i][j][v]; });
            } else {  // (few stores, and partial sums that are read back: plain ones)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int64_t m = mt + 8 * (v >> 2) + 4 * h + (v & 3);
                    if (m < M && n < N) y[m * N + n] = acc[i][j][v];
                }
            }
        }
}

// ---------------------------------------------------------------------------
// m > 8 with F32 weights: x as the three bf16 pieces of k_dense_pieces (their sum
// is x), and each weight as three bf16 pieces that a wave forms in registers from the
// f32 value in LDS: hi = bf16(w), mid = bf16(w - hi), lo = w - hi - mid, rounded to
// nearest, again exact.  Eight of the nine products, all exact in the accumulator; the
// ninth, lo lo, is below 2^-32 of |x w| (|lo| < 2^-15 |x|, <= 2^-17 |w|), a 256th of the
// rounding of one f32 product.  As k_dense_mm otherwise (tiles, two LDS buffers
// filled by loads to LDS, one barrier a stage), with stages of 32 values of k: a
// weight row is 128 B of a stage, its 16-byte chunk c in slot c ^ ((r >> 1) & 7); a
// piece's row is 64 B, two rows a line, chunk c of row r in slot
// (c ^ ((r >> 2) & 3)) + 4 (r & 1), so operand reads meet no bank twice.
// The split costs about 6.5 vector instructions a weight: under the MFMAs of TM tiles
// (256 TM clocks against 208), so waves take two row tiles where m has them.
// Bound by the matrix cores from M = 200 (1.0-1.4 PFLOP/s of operand products), by the
// weights' bytes and the launches below.  Against k_dense_gemm, us per call and relative
// error against 64 bits:
//   4096^2       M = 9 / 64 / 512  231 / 242 / 244 -> 20.3 / 29.7 / 121, 1.2e-6 -> 1.2e-7 / 1.2e-7 / 2.7e-7
//   1024 x 4096  M = 32            234 -> 15.4
//   8192^2       M = 2048          3016 -> 1650, 1.6e-6 -> 5.7e-7
//   512^2        M = 9 / 128       31.8 / 35.1 -> 12.5 / 18.9
// ---------------------------------------------------------------------------
constexpr int DK32 = 32;  // values of k per stage

template <int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void k_dense_mm32(const uint8_t *__restrict__ W, int64_t N, int64_t K,
                                                             const unsigned short *__restrict__ A,
                                                             const float *__restrict__ x, int64_t M,
                                                             float *__restrict__ out, DenseGrid g) {
    constexpr int NW = WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
    constexpr int RA = 3 * BM / 16, RB = BN / 8;  // staging instructions (1 KB): all pieces, the weights
    static_assert(RB % NW == 0 && NW % 2 == 0 && (BM / 16) % 2 == 0, "whole staging instructions per wave");
    constexpr int RAW = (RA + NW - 1) / NW;  // per wave, the last ones of them without a piece
    __shared__ __align__(1024) uint8_t As0[1024 * RAW * NW], As1[1024 * RAW * NW];
    __shared__ __align__(1024) uint8_t Bs0[BN * 128], Bs1[BN * 128];
    // tiles that share weight rows on one XCD
    const int G = (int)gridDim.x, L = (int)blockIdx.x;
    const int T = (G & 7) == 0 ? (L & 7) * (G >> 3) + (L >> 3) : L;
    const int tm = T % g.tiles_m, tn = (T / g.tiles_m) % g.tiles_n, z = T / (g.tiles_m * g.tiles_n);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int s0 = z * g.sps, ns = min(g.sps, (int)(g.Kp / DK32) - s0);  // ns >= 1
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, lr = lane & 31;
    const int wm = wave / WN, wn = wave % WN;

    // the piece that this wave's instruction j = 0, 1, 2 loads from
    const int64_t ps = g.rows * g.Kp;
    const unsigned short *Am = A + m0 * g.Kp;
    const __amdgpu_buffer_rsrc_t a0 = dense_rsrc(Am + wave / (BM / 16) * ps, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t a1 = dense_rsrc(Am + (wave + NW) / (BM / 16) * ps, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t a2 = dense_rsrc(Am + (wave + 2 * NW) / (BM / 16) * ps, BM * g.Kp * 2);
    const __amdgpu_buffer_rsrc_t br = dense_rsrc(W + n0 * K * 4, (N - n0 < BN ? N - n0 : BN) * K * 4);
    // pieces: lane l of an instruction fills line l/8 of 8, slot l%8: row 2 (l/8) + slot/4 of 16
    const uint32_t va = (uint32_t)((2 * (lane >> 3) + ((lane >> 2) & 1)) * (int)g.Kp * 2 + 16 * ((lane & 3) ^ (lane >> 4)));
    // weights: row l/8, slot l%8 of 8 rows whose number / 8 has the wave's parity
    const int ch = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
    const uint32_t vb = (uint32_t)((lane >> 3) * (int)K * 4 + 16 * ch);
    auto stage_in = [&](int s, int buf) __attribute__((always_inline)) {
        const int k0 = (s0 + s) * DK32;
        const uint32_t v0 = s < ns ? va : 0x80000000u;
#pragma unroll
        for (int j = 0; j < RAW; j++) {
            const int q = wave + NW * j;  // instruction q: piece q / (BM / 16), its rows 16 (q % (BM / 16)) on
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                j == 0 ? a0 : j == 1 ? a1 : a2, (__attribute__((address_space(3))) void *)((buf ? As1 : As0) + 1024 * q), 16,
                RA % NW == 0 || q < RA ? v0 : 0x80000000u, (16 * (q % (BM / 16)) * (int)g.Kp + k0) * 2, 0, 0);
        }
        const uint32_t v1 = s < ns && k0 + 4 * ch < (int)K ? vb : 0x80000000u;  // past K: zero
#pragma unroll
        for (int j = 0; j < RB / NW; j++) {
            const int rb = wave + NW * j;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                br, (__attribute__((address_space(3))) void *)((buf ? Bs1 : Bs0) + 1024 * rb), 16, v1,
                (8 * rb * (int)K + k0) * 4, 0, 0);
        }
    };
    int oa[2], ob[4];  // byte offsets of a lane's operands: pieces of k-step ks; weight chunks
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        oa[ks] = wm * TM * 2048 + (lr >> 1) * 128 + 16 * (((2 * ks + h) ^ ((lr >> 2) & 3)) + 4 * (lr & 1));
        asm volatile("" : "+v"(oa[ks]));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            ob[2 * ks + i] = wn * TN * 4096 + lr * 128 + 16 * ((4 * ks + 2 * h + i) ^ ((lr >> 1) & 7));
            asm volatile("" : "+v"(ob[2 * ks + i]));
        }
    }

    // sums of the first pieces' products, and of the others, which are 2^-7 of them and
    // less: a rounding at the size of the result an MFMA step instead of three to eight
    floatx16 acc[TM][TN] = {}, low[TM][TN] = {};
    // operands of this k-step and the next: x pieces, weight pieces; the next one's weights
    constexpr int NA = 3 * TM, NB = 2 * TN, NM = 8 * TM * TN;
    uint4 xa[2][NA], wb[2][TN][3], raw[NB];
    auto read = [&](int buf, int ks, int r, int q) __attribute__((always_inline)) {
        if (q < NB) raw[q] = *reinterpret_cast<const uint4 *>((buf ? Bs1 : Bs0) + (ob[2 * ks + (q & 1)] + (q >> 1) * 4096));
        else
            xa[r][q - NB] = *reinterpret_cast<const uint4 *>((buf ? As1 : As0) +
                                                             (oa[ks] + (q - NB) / TM * (BM * 64) + (q - NB) % TM * 2048));
    };
    // pair c (two weights) of raw -> wb[r]
    auto split = [&](int r, int c) __attribute__((always_inline)) {
        const int j = c >> 2, e = c & 3;
        const uint4 v = raw[2 * j + (e >> 1)];
        float v0 = __uint_as_float(e & 1 ? v.z : v.x) * DENSE_UP, v1 = __uint_as_float(e & 1 ? v.w : v.y) * DENSE_UP;
#pragma unroll
        for (int p = 0; p < 3; p++) {
            const uint32_t b = dense_split2(v0, v1);
            if (e == 0) wb[r][j][p].x = b;
            else if (e == 1) wb[r][j][p].y = b;
            else if (e == 2) wb[r][j][p].z = b;
            else wb[r][j][p].w = b;
        }
    };
    // the MFMAs of the k-step in xa[r], wb[r], each followed by its share of the next
    // one's reads (first half) or splits (second half)
    auto step = [&](int r, int buf, int ks) __attribute__((always_inline)) {
        constexpr int H = NM / 2, PR[8] = {0, 0, 1, 1, 0, 2, 1, 2}, PW[8] = {0, 1, 0, 1, 2, 0, 2, 1};
#pragma unroll
        for (int u = 0; u < NM; u++) {
            const int j = u % TN, i = u / TN % TM, p = u / TN / TM;
            floatx16 &to = p ? low[i][j] : acc[i][j];
            to = dense_mfma(xa[r][PR[p] * TM + i], wb[r][j][PW[p]], to);
            if (u < H) {
#pragma unroll
                for (int q = u * (NA + NB) / H; q < (u + 1) * (NA + NB) / H; q++) read(buf, ks, r ^ 1, q);
            } else {
#pragma unroll
                for (int c = (u - H) * 4 * TN / (NM - H); c < (u - H + 1) * 4 * TN / (NM - H); c++) split(r ^ 1, c);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    stage_in(0, 0);
    stage_in(1, 1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA + NB; q++) read(0, 0, 0, q);
#pragma unroll
    for (int c = 0; c < 4 * TN; c++) split(0, c);
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
        step(0, buf, 1);
        __builtin_amdgcn_s_waitcnt(0);  // this wave's operands, and its loads of stage s + 1
        __syncthreads();
        stage_in(s + 2, buf);
        __builtin_amdgcn_sched_barrier(0);
        step(1, buf ^ 1, 0);
    };
    for (int s = 0; s < ns; s += 2) {  // an odd count ends with a stage of zeros
        stage(s, 0);
        stage(s + 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0);  // the loads past the slice
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] += low[i][j];
    float *y = out + (int64_t)z * g.split_stride;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int64_t mt = m0 + 32 * (wm * TM + i), n = n0 + 32 * (wn * TN + j) + lr;
            if (g.split_stride == 0) dense_results<true, true>(acc[i][j], mt, M, N, n, h, x, W, K);
            if constexpr (TM * TN >= 4) {
                store_tile(y + mt * N, M - mt, N, n, h, [&](int v) __attribute__((always_inline)) { return acc[i][j][v]; });
            } else {  // (few stores, and partial sums that are read back: plain ones)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int64_t m = mt + 8 * (v >> 2) + 4 * h + (v & 3);
                    if (m < M && n < N) y[m * N + n] = acc[i][j][v];
                }
            }
        }
}

// y[m][n] = the slices' sums added in order, without the operands' factor; a workgroup
// takes 32 x 32 outputs, a wave eight rows of them, 16 bytes a lane.  What is not finite is
// formed again by the first wave.
template <bool BF, bool W32>
__global__ __launch_bounds__(256) void k_dense_sum(const float *__restrict__ part, int S, int64_t M, int64_t N,
                                                   const float *__restrict__ x, const uint8_t *__restrict__ W, int64_t K,
                                                   float *__restrict__ y) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t mt = 32 * (int64_t)blockIdx.y, nt = 32 * (int64_t)blockIdx.x, st = M * N;
    const int64_t m = mt + 8 * wave + (lane >> 3), n = nt + 4 * (lane & 7);
    bool bad = false;
    if (m < M && n < N) {
        const float *p = part + m * N + n;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        if ((N & 3) == 0) {
            for (int z0 = 0; z0 < S; z0 += 8) {
                float4 v[8];
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (z0 + j < S) v[j] = *reinterpret_cast<const float4 *>(p + (z0 + j) * st);
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (z0 + j < S) { s[0] += v[j].x; s[1] += v[j].y; s[2] += v[j].z; s[3] += v[j].w; }
            }
        } else {
            for (int i = 0; i < 4 && n + i < N; i++)
                for (int z = 0; z < S; z++) s[i] += p[z * st + i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] *= dense_down<W32>();
            bad = bad || !dense_finite(s[i]);
        }
        float *o = y + m * N + n;
        if ((N & 3) == 0 && !bad && (reinterpret_cast<uintptr_t>(y) & 15u) == 0) {
            *reinterpret_cast<float4 *>(o) = make_float4(s[0], s[1], s[2], s[3]);
        } else {
            for (int i = 0; i < 4 && n + i < N; i++)
                if (dense_finite(s[i])) o[i] = s[i];
        }
    }
    if (!__syncthreads_or(bad) || wave) return;
    const int64_t c = nt + (lane & 31);
    const floatx16 f = dense_tile<BF, W32>(x, W, K, M, N, mt, c);
#pragma unroll
    for (int v = 0; v < 16; v++) {
        const int64_t r = mt + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (r >= M || c >= N) continue;
        float s = 0.f;
        for (int z = 0; z < S; z++) s += part[z * st + r * N + c];
        if (!dense_finite(s * dense_down<W32>())) y[r * N + c] = f[v];
    }
}

namespace {
struct DensePlan {
    int bm, bn;
    DenseGrid g;
    size_t a_off, part_off, total;
};
// Tile by m (32, 64, 128 rows; 64 also where 128-row tiles would leave half the CUs idle and
// k is too short for slices: F16 512x256 M = 1000 15.4 -> 11.7 us, M = 4000 22.5 -> 18.5, F32
// 4096x256 M = 300 18.0 -> 13.6; 128 x 256 where such tiles fill the chip by themselves:
// BF16 8192^2 M = 2048 945 -> 622 us, 14336x4096 M = 512 158 -> 143), then k split until the
// resident workgroups (three of the 32-row tiles a CU, two of the 64-row, one of the
// 128-row) are there, at least 256 values of k a slice.
DensePlan dense_plan(int type, int64_t n, int64_t k, int64_t m) {
    DensePlan p;
    const bool w32 = type == TYPE_F32;
    const int64_t cus = num_cus();
    const bool idle = ((m + 127) / 128) * ((n + 127) / 128) * 2 <= cus && k < 8 * DK;
    p.bm = m <= 32 ? 32 : m <= 64 || idle ? 64 : 128;
    p.bn = 128;
    if (p.bm == 128 && ((m + 127) / 128) * ((n + 255) / 256) * 4 >= 3 * cus) p.bn = 256;
    p.g.tiles_m = (int)((m + p.bm - 1) / p.bm);
    p.g.tiles_n = (int)((n + p.bn - 1) / p.bn);
    p.g.rows = (int64_t)p.g.tiles_m * p.bm;
    p.g.Kp = (k + DK - 1) / DK * DK;
    const int64_t ns = p.g.Kp / (w32 ? DK32 : DK), tiles = (int64_t)p.g.tiles_m * p.g.tiles_n;
    const int64_t slots = cus * (p.bm == 32 ? 3 : p.bm == 64 ? 2 : 1);
    const int64_t s = std::max<int64_t>(1, std::min(slots / tiles, ns / (w32 ? 8 : 4)));
    p.g.sps = (int)((ns + s - 1) / s);
    p.g.splits = (int)((ns + p.g.sps - 1) / p.g.sps);
    p.g.split_stride = p.g.splits > 1 ? m * n : 0;
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    p.a_off = 0;
    p.part_off = up((size_t)3 * (size_t)p.g.rows * (size_t)p.g.Kp * 2);
    p.total = p.part_off + (p.g.splits > 1 ? up((size_t)p.g.splits * (size_t)(m * n) * 4) : 0);
    return p;
}
}  // namespace

size_t dense_workspace_bytes(int type, int64_t n, int64_t k, int64_t m) {
    // the buffer resources: 128 rows of pieces, 256 of f32 weights within 2^31 bytes
    if (m <= 8 || k % 8 || k > (type == TYPE_F32 ? 1 << 20 : 1 << 22) || m > 65535) return 0;
    // one stage and one launch of k_dense_gemm instead: 4096 x 64 M = 9 / 100 F16 8.9 / 10.2 -> 7.0 /
    // 7.7 us; with more outputs its rate counts (16384 x 64 M = 4000, F16 / BF16 / F32, 131 / 131 / 148
    // against 126 / 101 / 124)
    if (k <= DK && m * n < (int64_t)1 << 22) return 0;
    return dense_plan(type, n, k, m).total;
}

static hipError_t dense_pieces(int type, const uint8_t *w, int64_t n, int64_t k, const float *x, int64_t m, float *y,
                               uint8_t *ws, hipStream_t st) {
    const DensePlan p = dense_plan(type, n, k, m);
    unsigned short *a = reinterpret_cast<unsigned short *>(ws + p.a_off);
    float *out = p.g.splits > 1 ? reinterpret_cast<float *>(ws + p.part_off) : y;
    k_dense_pieces<<<(unsigned)m, p.g.Kp >= 2048 ? 256 : p.g.Kp > 512 ? 128 : 64, 0, st>>>(x, k, p.g.Kp, p.g.rows, a);
    const unsigned grid = (unsigned)(p.g.tiles_m * p.g.tiles_n * p.g.splits);
    auto go = [&](auto kern, int threads) { kern<<<grid, threads, 0, st>>>(w, n, k, a, x, m, out, p.g); };
    const dim3 sg((unsigned)((n + 31) / 32), (unsigned)((m + 31) / 32));
    if (type == TYPE_F32) {
        if (p.bm == 32) go(k_dense_mm32<1, 4, 1, 1>, 256);
        else if (p.bm == 64) go(k_dense_mm32<2, 4, 1, 1>, 512);
        else if (p.bn == 128) go(k_dense_mm32<2, 4, 2, 1>, 512);
        else go(k_dense_mm32<2, 4, 2, 2>, 512);
        if (p.g.splits > 1) k_dense_sum<true, true><<<sg, 256, 0, st>>>(out, p.g.splits, m, n, x, w, k, y);
    } else if (type == TYPE_F16) {
        if (p.bm == 32) go(k_dense_mm<false, 1, 4, 1, 1>, 256);
        else if (p.bm == 64) go(k_dense_mm<false, 2, 4, 1, 1>, 512);
        else if (p.bn == 128) go(k_dense_mm<false, 2, 4, 2, 1>, 512);
        else go(k_dense_mm<false, 2, 4, 2, 2>, 512);
        if (p.g.splits > 1) k_dense_sum<false, false><<<sg, 256, 0, st>>>(out, p.g.splits, m, n, x, w, k, y);
    } else {
        if (p.bm == 32) go(k_dense_mm<true, 1, 4, 1, 1>, 256);
        else if (p.bm == 64) go(k_dense_mm<true, 2, 4, 1, 1>, 512);
        else if (p.bn == 128) go(k_dense_mm<true, 4, 2, 1, 2>, 512);
        else go(k_dense_mm<true, 2, 4, 2, 2>, 512);
        if (p.g.splits > 1) k_dense_sum<true, false><<<sg, 256, 0, st>>>(out, p.g.splits, m, n, x, w, k, y);
    }
    return hipGetLastError();
}

template <bool F16, bool BF = false>
static hipError_t dense_typed(const uint8_t *w, int64_t n, int64_t k, const float *x, int64_t m, float *y,
                              hipStream_t st) {
    if (m <= 8) {
        const int64_t waves = std::min<int64_t>(n, (int64_t)num_cus() * 8);
        const unsigned grid = (unsigned)((waves + 3) / 4);
        const int mi = (int)m;
        const size_t xb = (size_t)m * (size_t)k * 4;
        const bool xl = xb <= DENSE_XL_BYTES;
        const size_t lds = xl ? xb : 0;
#define LBQ_DG(MR)                                                                    \
    {                                                                                 \
        if (xl) k_dense_gemv<F16, MR, true, BF><<<grid, 256, lds, st>>>(w, n, k, x, mi, y); \
        else k_dense_gemv<F16, MR, false, BF><<<grid, 256, 0, st>>>(w, n, k, x, mi, y);     \
    }
        if (m == 1) LBQ_DG(1) else if (m <= 2) LBQ_DG(2) else if (m <= 4) LBQ_DG(4) else LBQ_DG(8)
#undef LBQ_DG
        return hipGetLastError();
    }
    const dim3 grid((unsigned)((n + DBN - 1) / DBN), (unsigned)((m + DBM - 1) / DBM));
    k_dense_gemm<F16, BF><<<grid, 256, 0, st>>>(w, n, k, x, m, y);
    return hipGetLastError();
}

hipError_t launch_dense(int type, const uint8_t *w, int64_t n, int64_t k, const float *x, int64_t m, float *y,
                        void *ws, hipStream_t st) {
    if (k % 8 || m > 65535LL * DBM) return hipErrorInvalidValue;
    if (ws && dense_workspace_bytes(type, n, k, m))
        return dense_pieces(type, w, n, k, x, m, y, static_cast<uint8_t *>(ws), st);
    if (type == TYPE_F16) return dense_typed<true>(w, n, k, x, m, y, st);
    if (type == TYPE_F32) return dense_typed<false>(w, n, k, x, m, y, st);
    if (type == TYPE_BF16) return dense_typed<true, true>(w, n, k, x, m, y, st);
    return hipErrorInvalidValue;
}

}  // namespace lbq
