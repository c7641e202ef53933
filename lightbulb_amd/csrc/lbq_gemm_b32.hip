// lbq_gemm_b32.hip -- m > 8 for weights of 32-value blocks whose k is no multiple of
// 256 (Q8_0, Q4_0, Q4_1, Q5_0, Q5_1): the reference's block dot products on the fp16
// matrix cores, exact.
//
// y[m][n] = sum over blocks b of (sum_i c[n][i] q[m][i]) * (d_w[n][b] d_x[m][b]) (+ m_w[n][b] s_x[m][b])
// with the weight codes c and the activation codes q as the integers they are (fp16 holds
// them exactly): two v_mfma_f32_32x32x16_f16 give a 32 x 32 tile of block sums, exact in
// f32, and a third the tile of d_w d_x (fp16 values, one used k-slot: 22-bit products,
// exact), so an output takes one f32 FMA per block.  The offset types' m_w s_x of four
// blocks is one more MFMA straight into the sums.  The arithmetic is the reference's but
// for the f32 summation order: relative error against 64 bits as the integer decode
// kernel's (Q8_0 5760x2880, M = 200: 7.6e-8), infinite and NaN scales included.
//
// These shapes ran the decode GEMV over chunks of 8 rows before: the weights read, and
// a launch, per chunk.  Here a pre-pass (k_b32_ops) quantises x and writes the codes as
// MFMA operands, and a workgroup of eight waves owns 32 TM rows of y and 256 columns, wave
// w columns 32w..32w+31: a lane loads its half of its column's next four blocks (one
// stage ahead, in registers: 16 code bytes and the scales), turns the codes into the B
// operands, and every operand feeds TM MFMAs.  The A operands, 1 KB contiguous per
// (block, row tile, k-step), come through LDS by buffer loads to LDS, two stages.  Bound
// at large m by the matrix cores together with one LDS operand read per 1.4 MFMAs, at
// small m by the launches and the weight stream.  (With the activations as fp16 hi + lo
// operands scaled by d_x, four MFMAs and four reads per block and tile, the LDS reads
// held the kernel: 34.7 against 30.4 us at M = 200.)  Few tiles: k is split over
// workgroups, partials added in order by k_split_sum.
//
// us per call, row chunks -> now: Q8_0 5760x2880 M = 9 / 32 / 64 / 200 19.6 / 52 / 101 /
// 310 -> 17.4 / 18.3 / 22.5 / 36.0; Q5_0 4096x4128 M = 128 249 -> 35.3; Q4_0 8000x8160
// M = 1500 7242 -> 498.
#include <algorithm>

#include "lbq_device.hpp"
#include "lbq_internal.hpp"

namespace lbq {

typedef _Float16 bhalf8 __attribute__((ext_vector_type(8)));
typedef _Float16 bhalf4 __attribute__((ext_vector_type(4)));
typedef _Float16 bhalf2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int B32_WAVES = 8, B32_BN = 32 * B32_WAVES;
constexpr int NS = 4;  // blocks per stage

template <int TYPE>
constexpr int b32_bytes() {
    return TYPE == TYPE_Q4_0 ? 18 : TYPE == TYPE_Q4_1 ? 20 : TYPE == TYPE_Q5_0 ? 22 : TYPE == TYPE_Q5_1 ? 24 : 34;
}
template <int TYPE>
constexpr bool b32_ofs() { return TYPE == TYPE_Q4_1 || TYPE == TYPE_Q5_1; }

__device__ __forceinline__ uint32_t b32_ld2(const uint8_t *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) unsigned short *>(reinterpret_cast<uintptr_t>(p));
}

// The bytes of one block a lane of half h needs: the scale(s), the fifth bits, and 16
// code bytes (Q8_0: values 16h..16h+15; the others: all of qs, of which the lane uses
// nibble h).  Codes 2 past a dword are read as the aligned 16 bytes before them and
// the two bytes after, and shifted when used (mis).
template <int TYPE>
struct B32Raw {
    uint32_t w[4], tail, dm, qh;
    static constexpr bool AL4 = TYPE == TYPE_Q4_1 || TYPE == TYPE_Q5_1;  // every block dword aligned
    __device__ __forceinline__ void load(const uint8_t *blk, int h) {
        constexpr int QO = TYPE == TYPE_Q8_0 || TYPE == TYPE_Q4_0 ? 2 : TYPE == TYPE_Q4_1 ? 4 : TYPE == TYPE_Q5_0 ? 6 : 8;
        const uint8_t *q = blk + QO + (TYPE == TYPE_Q8_0 ? 16 * h : 0);
        const uintptr_t qa = reinterpret_cast<uintptr_t>(q);
        const u32x4a4 v = gld16(align4_global(qa));
        w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
        if constexpr (AL4) {
            dm = gld4(align4_global(reinterpret_cast<uintptr_t>(blk)));
            if constexpr (TYPE == TYPE_Q5_1) qh = gld4(align4_global(reinterpret_cast<uintptr_t>(blk + 4)));
        } else {
            tail = b32_ld2(q + 14);  // the codes' last two bytes
            dm = b32_ld2(blk);
            if constexpr (TYPE == TYPE_Q5_0) qh = b32_ld2(blk + 2) | (b32_ld2(blk + 4) << 16);
        }
    }
    // the B operands of the block's two k-steps: values 16h + 8 ks .. + 7
    __device__ __forceinline__ void codes(bool mis, int h, uint4 op[2]) const {
        uint32_t q[4] = {w[0], w[1], w[2], w[3]};
        if constexpr (!AL4) {
            const uint32_t sh = mis ? 16u : 0u;
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = __builtin_amdgcn_alignbit(i < 3 ? w[i + 1] : tail, w[i], sh);
        }
        uint32_t f[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t u;
            if constexpr (TYPE == TYPE_Q8_0) {
                u = q[i] ^ 0x80808080u;  // code + 128
            } else {
                u = (q[i] >> (4 * h)) & 0x0f0f0f0fu;
                if constexpr (TYPE == TYPE_Q5_0 || TYPE == TYPE_Q5_1) {
                    // bits 4i..4i+3 of the half's 16 fifth bits, one to bit 4 of each byte
                    const uint32_t b = (qh >> (16 * h + 4 * i)) & 0xfu;
                    u |= ((__umul24(b, 0x00204081u) & 0x01010101u) << 4);
                }
            }
            // a byte u under 0x64 is the fp16 1024 + u; minus 1024 and the code's offset, exact
            constexpr float off = -(1024.f + (TYPE == TYPE_Q8_0 ? 128.f : TYPE == TYPE_Q4_0 ? 8.f : TYPE == TYPE_Q5_0 ? 16.f : 0.f));
            const bhalf2 c = {(_Float16)off, (_Float16)off};
            const bhalf2 lo = __builtin_bit_cast(bhalf2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + c;
            const bhalf2 hi = __builtin_bit_cast(bhalf2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + c;
            f[2 * i] = __builtin_bit_cast(uint32_t, lo);
            f[2 * i + 1] = __builtin_bit_cast(uint32_t, hi);
        }
        op[0] = make_uint4(f[0], f[1], f[2], f[3]);
        op[1] = make_uint4(f[4], f[5], f[6], f[7]);
    }
};

struct B32Grid {
    int tiles_m, tiles_n, splits, sps;  // sps: stages per split
    int64_t split_stride;               // partials apart (0: out is y)
};

// Operand image, per row tile of 32 tm rows: codes [stage][block of the stage][k-step][32-row
// tile][lane][8 fp16], lane 32 h + row % 32 holding values 16 h + 8 ks .. + 7 of the block;
// scales (and the offset types' s) [stage][row][4 blocks] fp16.
//
// One wave: 8 rows by one stage; lane 8 hb + r the half-block hb of row r, so the rows'
// 16-byte chunks fill whole lines.  SRC_X: quantises f32 x (16-byte aligned) as candle's
// BlockQ8_0 / BlockQ8_1::from_float do; else from codes.
template <bool SRC_X, bool OFS>
__global__ __launch_bounds__(256) void k_b32_ops(const float *__restrict__ x, ActView act, int64_t M, int tm, int nst,
                                                 _Float16 *__restrict__ A, _Float16 *__restrict__ D,
                                                 _Float16 *__restrict__ S) {
    const int64_t wv = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, hb = lane >> 3, nb = act.nb;
    const int st = (int)(wv % nst), b = NS * st + (hb >> 1), h = hb & 1;
    const int64_t m = wv / nst * 8 + (lane & 7);
    const bool live = m < M && b < nb;  // blocks past k: zeros
    const int64_t mc = m < M ? m : M - 1;
    int8_t q[16];
    float d = 0.f, s = 0.f;
    if constexpr (SRC_X) {
        float v[16];
        const float4 *src = reinterpret_cast<const float4 *>(x + mc * act.k + 32 * (int64_t)(b < nb ? b : nb - 1) + 16 * h);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 f = src[i];
            v[4 * i] = f.x; v[4 * i + 1] = f.y; v[4 * i + 2] = f.z; v[4 * i + 3] = f.w;
        }
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) amax = fmaxf(amax, fabsf(v[i]));
        amax = fmaxf(amax, __shfl_xor(amax, 8));
        const float d0 = amax / 127.f, id = d0 != 0.f ? 1.f / d0 : 0.f;
        int sum = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float r = roundf(v[i] * id);
            const int c = (r != r) ? 0 : (int)fminf(fmaxf(r, -128.f), 127.f);
            q[i] = (int8_t)c;
            sum += c;
        }
        d = __half2float(__float2half_rn(d0));
        if constexpr (OFS) {
            sum += __shfl_xor(sum, 8);
            s = __half2float(__float2half_rn((float)sum)) * d;
        }
    } else if (live) {
        const uint4 c = *reinterpret_cast<const uint4 *>(act.xq + m * act.k + 32 * (int64_t)b + 16 * h);
        __builtin_memcpy(q, &c, 16);
        d = act.xd[m * nb + b];
        if constexpr (OFS) s = act.xs[m * nb + b];
    }
    if (m >= M) return;
    const int64_t tile = m / (32 * tm);
    const int row = (int)(m % (32 * tm));
    _Float16 *o = A + ((((tile * nst + st) * NS + (hb >> 1)) * 2 * tm + (row >> 5)) * 64 + 32 * h + (row & 31)) * 8;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        bhalf8 f;
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = (_Float16)(live ? (float)q[8 * ks + i] : 0.f);
        *reinterpret_cast<bhalf8 *>(o + ks * tm * 512) = f;
    }
    if (h == 0) {
        const int64_t at = ((tile * nst + st) * 32 * tm + row) * NS + (hb >> 1);
        D[at] = (_Float16)(live ? d : 0.f);
        if constexpr (OFS) S[at] = (_Float16)(live ? s : 0.f);
    }
}

// a buffer resource over [p, p + bytes), wave-uniform
__device__ __forceinline__ __amdgpu_buffer_rsrc_t b32_rsrc(const void *p, int bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
                       ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)) << 32);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(u), (short)0, __builtin_amdgcn_readfirstlane(bytes),
                                             0x00020000);
}

__device__ __forceinline__ floatx16 b32_mfma(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(bhalf8, a), __builtin_bit_cast(bhalf8, b), c, 0, 0, 0);
}

// products of four k-slots (eight per lane half and operand half the registers, the same rate)
__device__ __forceinline__ floatx16 b32_mfma8(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(bhalf4, make_uint2(a0, a1)),
                                                __builtin_bit_cast(bhalf4, make_uint2(b0, b1)), c, 0, 0, 0);
}

template <int TYPE, int TM>
__global__ __launch_bounds__(64 * B32_WAVES) void k_gemm_b32(const uint8_t *__restrict__ W, int64_t N, int64_t row_bytes,
                                                             const _Float16 *__restrict__ A, const _Float16 *__restrict__ D,
                                                             const _Float16 *__restrict__ S, int nb, int64_t M,
                                                             float *__restrict__ out, B32Grid g) {
    constexpr int BB = b32_bytes<TYPE>(), SB = 2 * TM * 1024;  // bytes of a weight block, of a block's A operands
    constexpr int NI = NS * SB / 1024 / B32_WAVES;             // staging instructions per wave and stage
    constexpr bool OFS = b32_ofs<TYPE>();
    constexpr int DB = 256 * TM;  // bytes of a stage's d (and s): loaded as 1 KB, the rest unused
    __shared__ __align__(1024) uint8_t As0[NS * SB], As1[NS * SB], Ds0[1024], Ds1[1024], Ss0[OFS ? 1024 : 16], Ss1[OFS ? 1024 : 16];
    const int G = (int)gridDim.x, L = (int)blockIdx.x;
    const int T = (G & 7) == 0 ? (L & 7) * (G >> 3) + (L >> 3) : L;  // tiles that share weights on one XCD
    const int tm = T % g.tiles_m, tn = (T / g.tiles_m) % g.tiles_n, z = T / (g.tiles_m * g.tiles_n);
    const int nst = (nb + NS - 1) / NS;
    const int s0 = z * g.sps, s1 = s0 + g.sps < nst ? s0 + g.sps : nst;  // this slice's stages, s0 < s1
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, lr = lane & 31;
    const int64_t m0 = (int64_t)tm * 32 * TM, n = (int64_t)tn * B32_BN + 32 * wave + lr;
    const uint8_t *wrow = W + (n < N ? n : N - 1) * row_bytes;
    // the tile's operands: stages past the last read as zero
    const __amdgpu_buffer_rsrc_t ar = b32_rsrc(A + (int64_t)tm * nst * NS * SB / 2, nst * NS * SB);
    const __amdgpu_buffer_rsrc_t dr = b32_rsrc(D + (int64_t)tm * nst * DB / 2, nst * DB);
    const __amdgpu_buffer_rsrc_t sr = b32_rsrc(S + (OFS ? (int64_t)tm * nst * DB / 2 : 0), OFS ? nst * DB : 0);
    auto stage_in = [&](int st, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const int c = wave + B32_WAVES * j;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (__attribute__((address_space(3))) void *)((buf ? As1 : As0) + c * 1024),
                                                     16, (uint32_t)lane * 16, st * NS * SB + c * 1024, 0, 0);
        }
        if (wave == 0)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(dr, (__attribute__((address_space(3))) void *)(buf ? Ds1 : Ds0), 16,
                                                     (uint32_t)lane * 16, st * DB, 0, 0);
        if constexpr (OFS)
            if (wave == 1)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (__attribute__((address_space(3))) void *)(buf ? Ss1 : Ss0), 16,
                                                         (uint32_t)lane * 16, st * DB, 0, 0);
    };
    B32Raw<TYPE> raw[NS];  // a lane's weights: this stage's until its operands are formed, then the next's
    auto load = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NS; j++) {
            const int b = NS * st + j;
            raw[j].load(wrow + (int64_t)(b < nb ? b : nb - 1) * BB, h);
        }
    };
    floatx16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[i][v] = 0.f;
    int lo = lane * 16, ld = lr * 8;
    asm volatile("" : "+v"(lo), "+v"(ld));
    const uint32_t half0 = h ? 0u : 0xffffffffu;
    // codes two bytes past a dword: blocks of 18, 22 or 34 bytes alternate
    const bool odd = (reinterpret_cast<uintptr_t>(wrow) & 2u) != 0;
    constexpr bool QMIS = TYPE == TYPE_Q8_0 || TYPE == TYPE_Q4_0 || TYPE == TYPE_Q5_0;  // the codes of a dword-aligned block
    // One stage, unit (row tile i, block j) after unit: its three MFMAs, each beside
    // a part of the next unit's operand reads and of the last unit's FMAs.  The four
    // blocks' values of an output are added to each other first: a quarter of the
    // roundings at the size of the running sum.  Blocks past k: zero scales.
    auto blocks = [&](int st, int buf) __attribute__((always_inline)) {
        uint4 op[NS][2];
        uint32_t dw[NS], mw[NS];  // f16 bits, in the lanes of half 0 (k-slot 0 of the scale MFMA)
#pragma unroll
        for (int j = 0; j < NS; j++) {
            raw[j].codes(((j & 1) != 0) != (odd != QMIS), h, op[j]);
            const bool in = NS * st + j < nb;
            dw[j] = in ? raw[j].dm & 0xffffu & half0 : 0u;
            mw[j] = OFS && in ? (raw[j].dm >> 16) & half0 : 0u;
        }
        __builtin_amdgcn_sched_barrier(0);
        load(st + 1);  // (past the slice: not used)
        uint4 a[2][2];
        uint2 dx[2], sx[2];  // the row's four d (and s) of tile i
        floatx16 c[2], sc;
        float u[16];
        auto read = [&](int un, int q) __attribute__((always_inline)) {  // k-step q of unit un; q = 2: its tile's scales
            const int i = un / NS, j = un % NS;
            if (q < 2) {
                a[un & 1][q] = *reinterpret_cast<const uint4 *>((buf ? As1 : As0) + (lo + j * SB + (q * TM + i) * 1024));
            } else if (j == 0) {
                const uint2 f = *reinterpret_cast<const uint2 *>((buf ? Ds1 : Ds0) + (ld + 256 * i));
                dx[i & 1] = make_uint2(f.x & half0, f.y & half0);
                if constexpr (OFS) {
                    const uint2 e = *reinterpret_cast<const uint2 *>((buf ? Ss1 : Ss0) + (ld + 256 * i));
                    sx[i & 1] = make_uint2(e.x & half0, e.y & half0);
                }
            }
        };
        auto sums = [&](int un, int v) __attribute__((always_inline)) {  // value v of unit un
            const int i = un / NS, j = un % NS;
            u[v] = j ? fmaf(c[un & 1][v], sc[v], u[v]) : c[un & 1][v] * sc[v];
            if (j == NS - 1) acc[i][v] += u[v];
        };
#pragma unroll
        for (int q = 0; q < 3; q++) read(0, q);
        const floatx16 zero = {};
#pragma unroll
        for (int un = 0; un < NS * TM; un++) {
            const int i = un / NS, j = un % NS;
            for (int q = 0; q < 3; q++) {
                if (q < 2) {
                    c[un & 1] = b32_mfma(a[un & 1][q], op[j][q], q == 0 ? zero : c[un & 1]);
                } else {  // the scales' product, once the last unit's FMAs are done with theirs
                    const uint32_t w = j < 2 ? dx[i & 1].x : dx[i & 1].y;
                    sc = b32_mfma8(j & 1 ? w >> 16 : w & 0xffffu, 0u, dw[j], 0u, zero);
                }
                // the last unit's FMAs after the first two MFMAs
                if (un && q < 2)
#pragma unroll
                    for (int v = 8 * q; v < 8 * q + 8; v++) sums(un - 1, v);
                if (un + 1 < NS * TM) read(un + 1, q);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (OFS)
                if (j == NS - 1)  // m_w s_x of the four blocks
                    acc[i] = b32_mfma8(sx[i & 1].x, sx[i & 1].y, mw[0] | mw[1] << 16, mw[2] | mw[3] << 16, acc[i]);
        }
#pragma unroll
        for (int v = 0; v < 16; v++) sums(NS * TM - 1, v);
    };
    stage_in(s0, 0);
    load(s0);
    __syncthreads();
    auto stage = [&](int st, int buf) __attribute__((always_inline)) {
        stage_in(st + 1, buf ^ 1);  // (past the slice: its next blocks, or zeros; not used)
        blocks(st, buf);
        __syncthreads();  // the compiler waits here for the loads to LDS, not for the weights after them
    };
    for (int st = s0; st < s1; st += 2) {
        stage(st, 0);
        if (st + 1 >= s1) break;
        stage(st + 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0);  // the loads past the slice
    float *y = out + (int64_t)z * g.split_stride;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int64_t m = m0 + 32 * i + 8 * (v >> 2) + 4 * h + (v & 3);
            if (m < M && n < N) y[m * N + n] = acc[i][v];
        }
}

namespace {
struct B32Plan {
    int tm, nst;  // row tiles of 32 per workgroup; stages of k
    B32Grid g;
    size_t a_off, d_off, s_off, part_off, total;
};
// Row tiles by m (32, 64 or 128 rows); k split until the resident workgroups (one a CU,
// two of 32 or 64 rows) are there, at least two stages a slice -- one where up to sixteen
// slices of one stage fit the CUs (Q8_0 4096x1056 M = 9 15.8 -> 12.7 us, 8192x544 14.4 ->
// 11.8), or more of them half the CUs; elsewhere more slices only add partials: 5760x2880
// M = 9 17.4 -> 21.0, 1024x8160 M = 40 20.0 -> 22.4.
B32Plan b32_plan(int type, int64_t n, int64_t k, int64_t m) {
    B32Plan p;
    p.tm = m <= 32 ? 1 : m <= 64 ? 2 : 4;
    p.nst = (int)((k / 32 + NS - 1) / NS);
    p.g.tiles_m = (int)((m + 32 * p.tm - 1) / (32 * p.tm));
    p.g.tiles_n = (int)((n + B32_BN - 1) / B32_BN);
    const int64_t tiles = (int64_t)p.g.tiles_m * p.g.tiles_n, slots = (int64_t)num_cus() * (p.tm == 4 ? 1 : 2);
    const int64_t most = (p.nst <= 16 ? 1 : 2) * tiles * p.nst <= num_cus() ? p.nst : p.nst / 2;
    const int64_t s = std::max<int64_t>(1, std::min(slots / tiles, most));
    p.g.sps = (int)((p.nst + s - 1) / s);
    p.g.splits = (p.nst + p.g.sps - 1) / p.g.sps;
    p.g.split_stride = p.g.splits > 1 ? m * n : 0;
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t rows = (size_t)p.g.tiles_m * 32 * p.tm;
    p.a_off = 0;
    p.d_off = rows * (size_t)p.nst * (NS * 32 * 2);
    p.s_off = p.d_off + rows * (size_t)p.nst * (NS * 2);
    p.part_off = p.s_off + (gemm_offset_step(type) ? rows * (size_t)p.nst * (NS * 2) : 0);
    p.total = p.part_off + (p.g.splits > 1 ? up((size_t)p.g.splits * (size_t)(m * n) * 4) : 0);
    return p;
}
}  // namespace

// (a row tile's operands, 256 bytes a row and stage, within 2^31)
bool gemm_b32_serves(int type, int64_t k, int64_t m) {
    return (is_legacy(type) || type == TYPE_Q8_0) && k % 32 == 0 && k % 256 != 0 && m > 8 && k <= (1 << 21);
}

size_t gemm_b32_workspace_bytes(int type, int64_t n, int64_t k, int64_t m) {
    return gemm_b32_serves(type, k, m) ? b32_plan(type, n, k, m).total : 0;
}

template <int TYPE>
static hipError_t b32_typed(const uint8_t *w, int64_t n, int64_t k, int64_t row_bytes, const ActView &act, const float *x,
                            int64_t m, float *y, uint8_t *ws, hipStream_t st) {
    constexpr bool OFS = b32_ofs<TYPE>();
    const B32Plan p = b32_plan(TYPE, n, k, m);
    _Float16 *a = reinterpret_cast<_Float16 *>(ws + p.a_off), *d = reinterpret_cast<_Float16 *>(ws + p.d_off),
             *s = reinterpret_cast<_Float16 *>(ws + p.s_off);
    float *out = p.g.splits > 1 ? reinterpret_cast<float *>(ws + p.part_off) : y;
    const unsigned og = (unsigned)(((m + 7) / 8 * p.nst + 3) / 4);
    if (x) {
        k_b32_ops<true, OFS><<<og, 256, 0, st>>>(x, act, m, p.tm, p.nst, a, d, s);
    } else {
        if (OFS && !act.xs) return hipErrorInvalidValue;
        k_b32_ops<false, OFS><<<og, 256, 0, st>>>(nullptr, act, m, p.tm, p.nst, a, d, s);
    }
    const unsigned grid = (unsigned)(p.g.tiles_m * p.g.tiles_n * p.g.splits);
    constexpr int NT = 64 * B32_WAVES;
    const int nb = (int)(k / 32);
    if (p.tm == 1) k_gemm_b32<TYPE, 1><<<grid, NT, 0, st>>>(w, n, row_bytes, a, d, s, nb, m, out, p.g);
    else if (p.tm == 2) k_gemm_b32<TYPE, 2><<<grid, NT, 0, st>>>(w, n, row_bytes, a, d, s, nb, m, out, p.g);
    else k_gemm_b32<TYPE, 4><<<grid, NT, 0, st>>>(w, n, row_bytes, a, d, s, nb, m, out, p.g);
    if (p.g.splits > 1) return launch_split_sum(out, p.g.splits, m * n, y, st);
    return hipGetLastError();
}

bool gemm_b32_quantises(const float *x) { return x && (reinterpret_cast<uintptr_t>(x) & 15u) == 0; }

hipError_t launch_gemm_b32(int type, const uint8_t *w, int64_t n, int64_t k, int64_t row_bytes, const ActView &act,
                           const float *x, int64_t m, float *y, void *ws, hipStream_t st) {
    if (!ws || !gemm_b32_serves(type, k, m) || (x && !gemm_b32_quantises(x))) return hipErrorInvalidValue;
    uint8_t *b = static_cast<uint8_t *>(ws);
    switch (type) {
    case TYPE_Q8_0: return b32_typed<TYPE_Q8_0>(w, n, k, row_bytes, act, x, m, y, b, st);
    case TYPE_Q4_0: return b32_typed<TYPE_Q4_0>(w, n, k, row_bytes, act, x, m, y, b, st);
    case TYPE_Q4_1: return b32_typed<TYPE_Q4_1>(w, n, k, row_bytes, act, x, m, y, b, st);
    case TYPE_Q5_0: return b32_typed<TYPE_Q5_0>(w, n, k, row_bytes, act, x, m, y, b, st);
    case TYPE_Q5_1: return b32_typed<TYPE_Q5_1>(w, n, k, row_bytes, act, x, m, y, b, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace lbq
