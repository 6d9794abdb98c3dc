// Matmuls on the int8 matrix cores, bit-identical to the serial double chain.
//
// Every output of the step's matmuls is f32(s), s the double chain sum over l ascending of a_l b_l. The FP64 matrix
// cores run that chain at 78.6 TFLOP/s; the int8 ones are 64 times faster per product. So the sums are formed twice
// over: here from integers, with a bound on how far the chain can lie from them, and by the chain itself only where
// that bound leaves the rounding open.
//
//   Split. Each row of an operand (A's i or B's j, over the reduction l of one window) is scaled by a power of two to
//   48-bit integers and cut into six signed base-256 digits, d_1 (high) to d_6. a = sum_p d_p 256^(6-p) exactly for floats
//   down to 2^-24 of the row's largest; below that a is rounded, by at most half a unit.
//   Products. sum_l a_l b_l is a sum over digit pairs (p, q), each a matrix product of int8. The 19 pairs of the first five
//   digits with p + q <= 7 are formed, exact in int32 (a window's length is limited so that 6 pairs x 2^14 x L < 2^31); pairs
//   of equal p + q share an accumulator. The sixth digit is nearly always zero; a tile for which its norm matters adds the
//   pairs (1, 6) and (6, 1).
//   Bound. With N = ||a||_2 of a row (and N_p of its digits, r of its rounding), Cauchy-Schwarz bounds what is left
//   out: 2^16 (N_3a N_5b + N_4a N_4b + N_5a N_3b) + 2^8 (N_4a N_5b + N_5a N_4b) + N_5a N_5b + r_a N_b + N_a r_b + r_a r_b.
//   The chain itself is off by at most 2^-53 sum_k |s_k| over its partial sums s_k; with the integer partial sum S_c
//   known at every 128th l, |s_k| <= |S_c| + (the norms over the 128 values in between), whose sum over all chunks is
//   at most 128 N_a N_b (Cauchy-Schwarz over the chunks).
//   Decision. When the integer sum plus and minus the bound round to the same float, the chain rounds to it too.
//   Otherwise the output goes to a list, and split_fix_kernel computes its chain: one output in 2500 on Gaussian operands
//   at L = 1536, one in 260 at 8192 with rows and columns of unequal size. A tile of which more than one in 64 would go
//   there (rows of very wide dynamic range, infinities, NaNs) is flagged and recomputed whole by the FP64 matmul.
//   Measured: 1023 x 8960 x 1536 in 269 us of 371 for the call, against 600 in FP64 (matrix cores 43% busy at 2.26 GHz: 4.4
//   rounds of workgroups and their epilogues); 8192 x 1536 x 8960 in 1.69 ms (133 TFLOP/s, 70% busy at 1.72 GHz: power
//   lowers the clock, and random digits on registers alone reach 181), with splitting and recomputation 2.5, against 3.5.
#include <algorithm>

#include "common.h"
#include "gemm_split.h"
#include "kernels.h"
#include "lds_copy.h"
#include "workspace.h"

namespace dllm_hip {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kDigits = 5;                       // of the 19 products; the sixth is kept apart
constexpr int kOrders = 6;                       // p + q = 2 .. 7
constexpr int kFragment = 1024;                  // 32 rows x 32 l of one digit: 16 bytes per lane
constexpr int kStageL = 64;                      // the digits' windows are padded to whole 64 l: two steps
constexpr int kStepBytes = kDigits * kFragment;  // 32 l of a 32-row block
constexpr int kStageBytes = 2 * kStepBytes;
constexpr int kPartL = 256;                      // l per workgroup of the split passes
constexpr int64_t kMaxWindow = 21824;            // l per window, or per leg of a long reduction (the int32 sums' range)
constexpr int kCheckSteps = 4;                   // partial sums enter the bound every 128 l
constexpr int kRing = 3;                         // LDS buffers of one step
constexpr float kUp = 1.01f;                     // covers the rounding of the bounds' own float arithmetic

// What the bounds need of one operand row over one window: the largest |value| (float bits), the sums of its digits'
// squares, and how many values six digits do not hold exactly.
struct RowMeta {
    uint32_t amax;
    float q1, q3, q4, q5, q6;
    float n6;
    int out_l;    // long reductions: the row's one value far above the others (out_a != 0), kept out of its digits
    float out_a;
    float pad[3];
};
static_assert(sizeof(RowMeta) % 16 == 0, "cleared in 16-byte pieces");

struct Operand {
    const float* src;
    int64_t ld;
    int rows_contiguous;  // src[l][row] (1) or src[row][l] (0)
    int64_t rows, blocks;
    int8_t* digits;  // [block of 32 rows][stage][2][digit][lane][16]
    int8_t* digits6; // [block][stage][2][lane][16]: the sixth digit
    RowMeta* meta;   // [window][padded rows]
    float* t;        // rows_contiguous: the values as [row][stage][64 l], zero past a window's end
};

struct SplitParams {
    Operand a, b;
    const float* out_b;  // long reductions: B[l][j], for the values kept apart
    int64_t ld_out_b;
    int64_t stages;      // stages of all windows together (the digits' stride per block)
    const int64_t* seg;  // device offsets of the windows, or null: one window [0, l1)
    int nseg;
    int64_t l1;
    float* C;
    int64_t ldc;
    int64_t I, J;
    const float* bias;
    const float* addsrc;
    int64_t ld_add;
    const float* seg_addend;
    const int* seg_addrow;
    int64_t ld_addrow;
    int64_t ld_seg_add;
    const float* seg_weight;
    const float* seg_rowscale;
    float* partial;
    uint8_t* tile_flags;
    uint32_t* count;  // [0] chains to compute, [1] flagged tiles, [2] outputs with an undecided window
    uint64_t* list;   // the chains: window << 48 | i * J + j; windows in sequence: window << 48 | output slot
    uint32_t list_cap;
    // windows in sequence: an undecided output's slot holds i * J + j | first undecided window << 48, the sum of the
    // windows before it, and each later window's result (decided ones from the tile, the others from their chains)
    uint64_t* slots;
    float* slot_values;  // [slot][1 + nseg]
    uint32_t slot_cap;
    uint32_t* stat;  // the caller's SplitDone (null: none kept)
};

struct Window {
    int64_t l0, l1, stage0;
};

// Window s: its l range and its first stage (each window's stages start on a boundary of their own).
__device__ __forceinline__ Window window_of(const SplitParams& p, int s) {
    if (p.seg == nullptr) return {0, p.l1, 0};
    int64_t st = 0, lo = p.seg[0];
    for (int k = 0; k < s; ++k) {
        const int64_t hi = p.seg[k + 1];
        st += (hi - lo + kStageL - 1) / kStageL;
        lo = hi;
    }
    return {lo, p.seg[s + 1], st};
}

__device__ __forceinline__ bool finite_bits(uint32_t amax) { return amax < 0x7f800000u; }

// The exponent e of a row: |a| <= 0.9901 x 2^e, so that |a| 2^(47 - e) fits six signed base-256 digits (at most
// 0.996 x 2^47).
__device__ __forceinline__ int row_exponent(uint32_t amax) {
    if (amax == 0 || !finite_bits(amax)) return 0;
    return ilogb(static_cast<double>(__uint_as_float(amax)) * 1.01) + 1;
}

__device__ __forceinline__ int64_t padded32(int64_t n) { return (n + 31) / 32 * 32; }

// Part k of the reduction (kPartL l of one window): the window and its range, or false past the last part.
__device__ __forceinline__ bool part_of(const SplitParams& p, int64_t k, int& s, int64_t& l0, int64_t& l1,
                                        int64_t& stage) {
    if (p.seg == nullptr) {
        s = 0;
        l0 = k * kPartL;
        l1 = p.l1;
        stage = k * (kPartL / kStageL);
        return l0 < l1;
    }
    int64_t st = 0, lo = p.seg[0];
    for (s = 0; s < p.nseg; ++s) {
        const int64_t hi = p.seg[s + 1], parts = (hi - lo + kPartL - 1) / kPartL;
        if (k < parts) {
            l0 = lo + k * kPartL;
            l1 = hi;
            stage = st + k * (kPartL / kStageL);
            return true;
        }
        k -= parts;
        st += (hi - lo + kStageL - 1) / kStageL;
        lo = hi;
    }
    return false;
}

__global__ __launch_bounds__(256) void split_clear_kernel(uint4* __restrict__ a, int64_t na, uint4* __restrict__ b,
                                                          int64_t nb, uint32_t* count) {
    for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < na + nb;
         e += static_cast<int64_t>(gridDim.x) * 256)
        (e < na ? a[e] : b[e - na]) = uint4{0, 0, 0, 0};
    if (blockIdx.x == 0 && threadIdx.x < 3) count[threadIdx.x] = 0;
}

constexpr int kSplitRows = 128;  // operand rows per workgroup of the split passes

// The largest |value| of each operand row over one part: 128 rows x kPartL l per workgroup.
__device__ __forceinline__ void amax_block(const SplitParams& p, const Operand& o, int64_t blk, int64_t part) {
    int s;
    int64_t l0, lend, stage;
    if (!part_of(p, part, s, l0, lend, stage)) return;
    const int64_t l1 = l0 + kPartL < lend ? l0 + kPartL : lend;
    const int64_t r0 = blk * kSplitRows;
    RowMeta* meta = o.meta + static_cast<int64_t>(s) * o.blocks * 32;
    const int tid = static_cast<int>(threadIdx.x);
    if (o.rows_contiguous) {  // thread: 4 rows (one 16-byte load) of every 8th l
        __shared__ uint32_t best[kSplitRows];
        if (tid < kSplitRows) best[tid] = 0;
        __syncthreads();
        const int64_t r = r0 + (tid & 31) * 4;
        if (r < o.rows) {  // rows is a multiple of 4
            uint32_t m[4] = {0, 0, 0, 0};
            for (int64_t l = l0 + (tid >> 5); l < l1; l += 8) {
                const uint4 v = *reinterpret_cast<const uint4*>(o.src + l * o.ld + r);
                m[0] = max(m[0], v.x & 0x7fffffffu);
                m[1] = max(m[1], v.y & 0x7fffffffu);
                m[2] = max(m[2], v.z & 0x7fffffffu);
                m[3] = max(m[3], v.w & 0x7fffffffu);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) atomicMax(&best[(tid & 31) * 4 + c], m[c]);
        }
        __syncthreads();
        if (tid < kSplitRows && r0 + tid < o.rows) atomicMax(&meta[r0 + tid].amax, best[tid]);
    } else {  // a wave per row: 4 l per lane, 32 rows each
        const int wave = tid >> 6, lane = tid & 63;
        for (int k = wave; k < kSplitRows; k += 4) {
            const int64_t r = r0 + k;
            if (r >= o.rows) break;
            uint32_t m = 0;
            const int64_t l = l0 + lane * 4;
            if (l < l1) {  // the reduction is a multiple of 4
                const uint4 v = *reinterpret_cast<const uint4*>(o.src + r * o.ld + l);
                m = max(max(v.x & 0x7fffffffu, v.y & 0x7fffffffu), max(v.z & 0x7fffffffu, v.w & 0x7fffffffu));
            }
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), d)));
            if (lane == 0) atomicMax(&meta[r].amax, m);
        }
    }
}

// Long reductions (the logits' gradient times the head, l over the vocabulary): a row is a softmax, tiny values and one
// near -1 at its target, and scaled by that one the others would keep too few bits. Each row's largest |value| is found
// with its place and the second largest; more than 64 times the second, it stays out of the digits, and the epilogue adds
// its product.
__global__ __launch_bounds__(256) void split_top_kernel(Operand o, int64_t l1) {
    const int64_t r = blockIdx.x;
    const float* src = o.src + r * o.ld;
    uint32_t best = 0, second = 0;
    int at = 0;
    auto take = [&](float x, int64_t l) {
        const uint32_t b = __float_as_uint(x) & 0x7fffffffu;
        if (b > best) {
            second = best;
            best = b;
            at = static_cast<int>(l);
        } else {
            second = max(second, b);
        }
    };
    for (int64_t l = static_cast<int64_t>(threadIdx.x) * 4; l < l1; l += 1024) {
        const float4 v = *reinterpret_cast<const float4*>(src + l);
        take(v.x, l);
        take(v.y, l + 1);
        take(v.z, l + 2);
        take(v.w, l + 3);
    }
    __shared__ uint32_t sb[256], ss[256];
    __shared__ int sa[256];
    sb[threadIdx.x] = best;
    ss[threadIdx.x] = second;
    sa[threadIdx.x] = at;
    for (int d = 128; d > 0; d >>= 1) {
        __syncthreads();
        if (threadIdx.x < static_cast<unsigned>(d)) {
            const uint32_t b1 = sb[threadIdx.x], b2 = sb[threadIdx.x + d];
            ss[threadIdx.x] = max(max(ss[threadIdx.x], ss[threadIdx.x + d]), min(b1, b2));
            if (b2 > b1) {
                sb[threadIdx.x] = b2;
                sa[threadIdx.x] = sa[threadIdx.x + d];
            }
        }
    }
    if (threadIdx.x != 0) return;
    RowMeta m{};
    m.amax = sb[0];
    if (finite_bits(sb[0]) && __uint_as_float(sb[0]) > 64.0f * __uint_as_float(ss[0])) {
        m.amax = ss[0];
        m.out_l = sa[0];
        m.out_a = src[sa[0]];
    }
    o.meta[r] = m;
}

__global__ __launch_bounds__(256) void split_amax_kernel(SplitParams p, int64_t a_blocks) {
    const bool a = blockIdx.x < a_blocks;
    const Operand o = a ? p.a : p.b;
    amax_block(p, o, a ? blockIdx.x : blockIdx.x - a_blocks, blockIdx.y);
}

// dot(x, x) of 16 signed bytes
__device__ __forceinline__ int square16(const uint32_t (&w)[4]) {
    int t = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        t = __builtin_amdgcn_sdot4(static_cast<int>(w[k]), static_cast<int>(w[k]), t, false);
    return t;
}

// One row's 16 consecutive l: the digits into the fragments, and the sums of squares. `inexact`: float bits below which
// a nonzero |value| loses bits below the sixth digit.
struct RowSums {
    int n1 = 0, n3 = 0, n4 = 0, n5 = 0, n6 = 0, inexact = 0;
};

__device__ __forceinline__ void digits16(const float (&x)[16], double scale, uint32_t inexact, int8_t* dst, int8_t* dst6,
                                         RowSums& sums) {
    uint32_t out[kDigits + 1][4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // rounds x 2^(47 - e) to an integer in the low mantissa bits of 1.5 x 2^52
            const double m = static_cast<double>(x[w * 4 + k]) * scale + 6755399441055744.0;
            sums.inexact += (__float_as_uint(x[w * 4 + k]) & 0x7fffffffu) - 1u < inexact ? 1 : 0;
            // + 128 in every byte turns the two's complement into digits + 128
            const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(m)) + 0x808080808080ull;
            lo[k] = static_cast<uint32_t>(bits) ^ 0x80808080u;
            hi[k] = static_cast<uint32_t>(bits >> 32) ^ 0x8080u;
        }
        // byte transposes: out[d][w] = the four elements' digit d
        const uint32_t a01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x05010400);  // bytes 0 of 0, 1, then bytes 1
        const uint32_t c01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x07030602);  // bytes 2, then bytes 3
        const uint32_t a23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x05010400);
        const uint32_t c23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x07030602);
        const uint32_t h01 = __builtin_amdgcn_perm(hi[1], hi[0], 0x05010400);
        const uint32_t h23 = __builtin_amdgcn_perm(hi[3], hi[2], 0x05010400);
        out[5][w] = __builtin_amdgcn_perm(a23, a01, 0x05040100);
        out[4][w] = __builtin_amdgcn_perm(a23, a01, 0x07060302);
        out[3][w] = __builtin_amdgcn_perm(c23, c01, 0x05040100);
        out[2][w] = __builtin_amdgcn_perm(c23, c01, 0x07060302);
        out[1][w] = __builtin_amdgcn_perm(h23, h01, 0x05040100);
        out[0][w] = __builtin_amdgcn_perm(h23, h01, 0x07060302);
        __builtin_amdgcn_sched_barrier(0);  // four elements at a time: all sixteen would spill
    }
    sums.n1 += square16(out[0]);
    sums.n3 += square16(out[2]);
    sums.n4 += square16(out[3]);
    sums.n5 += square16(out[4]);
    sums.n6 += square16(out[5]);
#pragma unroll
    for (int d = 0; d < kDigits; ++d)
        *reinterpret_cast<uint4*>(dst + d * kFragment) = uint4{out[d][0], out[d][1], out[d][2], out[d][3]};
    *reinterpret_cast<uint4*>(dst6) = uint4{out[5][0], out[5][1], out[5][2], out[5][3]};
}

// The digits of 128 operand rows over one part and the rows' sums of squares. A thread takes row tid % 128 and two
// groups of 16 l per 64-l stage: straight from memory where the row is contiguous (a row's 64 bytes are one thread's
// four loads), else through an LDS tile of the stage.
template <bool kOut>
__device__ __forceinline__ void digits_block(const SplitParams& p, const Operand& o, int64_t blk, int64_t part) {
    constexpr int kStride = kSplitRows + 4;  // 16-byte rows; a wave reads 64 consecutive floats of one
    __shared__ float tile[kStageL * kStride];
    int s;
    int64_t l0, lend, stage;
    if (!part_of(p, part, s, l0, lend, stage)) return;
    const int64_t r0 = blk * kSplitRows;
    RowMeta* meta = o.meta + static_cast<int64_t>(s) * o.blocks * 32;
    const int tid = static_cast<int>(threadIdx.x);
    const int row = tid & (kSplitRows - 1), g0 = (tid >> 7) * 2;
    const bool live = r0 + row < o.rows;
    const uint32_t amax = live ? meta[r0 + row].amax : 0;
    const bool fin = finite_bits(amax);
    const int e = row_exponent(amax);
    const double scale = ldexp(1.0, 47 - e);
    // values below 2^(e - 24) have bits below 2^(e - 47) (a float's last bit is 2^-149 at least)
    const uint32_t inexact = e > -102 ? (static_cast<uint32_t>(e - 24 + 127) << 23) - 1u : 0u;
    const int64_t b32 = (r0 + row) >> 5;
    RowSums sums;
    auto dst6_of = [&](int64_t st, int g) {
        return o.digits6 + ((b32 * p.stages + st) * 2 + (g >> 1)) * kFragment + ((g & 1) * 32 + (row & 31)) * 16;
    };
    auto dst_of = [&](int64_t st, int g) {
        return o.digits + ((b32 * p.stages + st) * 2 + (g >> 1)) * kStepBytes + ((g & 1) * 32 + (row & 31)) * 16;
    };
    const int64_t l_end = l0 + kPartL < lend ? l0 + kPartL : lend;
    if (!o.rows_contiguous) {
        const int64_t out_l = kOut && live && meta[r0 + row].out_a != 0.0f ? meta[r0 + row].out_l : -1;
        const float* src = o.src + (live ? r0 + row : 0) * o.ld;
        if (b32 >= o.blocks) return;
        const int64_t groups = (l_end - l0 + kStageL - 1) / kStageL * 2;  // this thread's, of 16 l
        float4 v[4];
        auto load = [&](int64_t k) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int64_t at = l0 + (k >> 1) * kStageL + (g0 + (k & 1)) * 16 + w * 4;
                v[w] = float4{0.0f, 0.0f, 0.0f, 0.0f};
                if (live && fin && at < lend) v[w] = *reinterpret_cast<const float4*>(src + at);
            }
        };
        load(0);
#pragma unroll 1
        for (int64_t k = 0; k < groups; ++k) {
            float x[16];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                x[4 * w] = v[w].x;
                x[4 * w + 1] = v[w].y;
                x[4 * w + 2] = v[w].z;
                x[4 * w + 3] = v[w].w;
            }
            if constexpr (kOut) {
                const int64_t rel = out_l - (l0 + (k >> 1) * kStageL + (g0 + (k & 1)) * 16);
                if (rel >= 0 && rel < 16) {
#pragma unroll
                    for (int q = 0; q < 16; ++q) x[q] = rel == q ? 0.0f : x[q];
                }
            }
            if (k + 1 < groups) load(k + 1);
            const int g = g0 + static_cast<int>(k & 1);
            digits16(x, scale, inexact, dst_of(stage + (k >> 1), g), dst6_of(stage + (k >> 1), g), sums);
        }
    } else {
        const int lr = tid >> 5, lc = (tid & 31) * 4;  // this thread's loads: l rows lr + 8 k, 4 operand rows from lc
        float4 v[8];
        auto load = [&](int64_t l) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[k] = float4{0.0f, 0.0f, 0.0f, 0.0f};
                if (l + lr + 8 * k < lend && r0 + lc < o.rows)
                    v[k] = *reinterpret_cast<const float4*>(o.src + (l + lr + 8 * k) * o.ld + r0 + lc);
            }
        };
        load(l0);
#pragma unroll 1
        for (int64_t l = l0; l < l_end; l += kStageL, ++stage) {
#pragma unroll
            for (int k = 0; k < 8; ++k) *reinterpret_cast<float4*>(tile + (lr + 8 * k) * kStride + lc) = v[k];
            lds_barrier();
            if (l + kStageL < l_end) load(l + kStageL);
#pragma unroll 1
            for (int u = 0; u < 2; ++u) {
                const int g = g0 + u;
                float x[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) x[k] = tile[(g * 16 + k) * kStride + row];
                if (live) {
                    float4* dst = reinterpret_cast<float4*>(o.t + ((r0 + row) * p.stages + stage) * kStageL + g * 16);
#pragma unroll
                    for (int w = 0; w < 4; ++w) dst[w] = float4{x[4 * w], x[4 * w + 1], x[4 * w + 2], x[4 * w + 3]};
                }
                if (!fin) {
#pragma unroll
                    for (int k = 0; k < 16; ++k) x[k] = 0.0f;
                }
                if (b32 < o.blocks) digits16(x, scale, inexact, dst_of(stage, g), dst6_of(stage, g), sums);
            }
            lds_barrier();
        }
    }
    if (!live) return;
    RowMeta* m = meta + r0 + row;
    atomicAdd(&m->q1, static_cast<float>(sums.n1));
    atomicAdd(&m->q3, static_cast<float>(sums.n3));
    atomicAdd(&m->q4, static_cast<float>(sums.n4));
    atomicAdd(&m->q5, static_cast<float>(sums.n5));
    if (sums.n6) atomicAdd(&m->q6, static_cast<float>(sums.n6));
    if (sums.inexact) atomicAdd(&m->n6, static_cast<float>(sums.inexact));
}

template <bool kOut>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void split_digits_kernel(SplitParams p, int64_t a_blocks) {
    const bool a = blockIdx.x < a_blocks;
    const Operand o = a ? p.a : p.b;
    digits_block<kOut>(p, o, a ? blockIdx.x : blockIdx.x - a_blocks, blockIdx.y);
}

// The bound's factors of one operand row, in units of the fifth digit: the bound on |chain - integer sum| of (i, j),
// less the checked partial sums, is P_i n5_j + n5_i P_j + r_i N_j + N_i r_j + X_i X_j, with r = r5 where five digits are
// multiplied; with the sixth times the first added, r = r6 and another n6 (N_2 256^2 + ...) of each row.
struct RowBound {
    float P, n5, r5, r6, N, X;
    float wide;  // what the sixth digit's products leave out
    int e;
    float out, out_a;  // long reductions: the value kept apart, and in the row's integer units
    int out_l;
};

__device__ __forceinline__ RowBound row_bound(const RowMeta& m, float len) {
    RowBound b;
    const float root = sqrtf(len);
    const float n3 = sqrtf(m.q3) * kUp, n4 = sqrtf(m.q4) * kUp, n6 = sqrtf(m.q6) * kUp;
    b.n5 = sqrtf(m.q5) * kUp;
    b.P = 65536.0f * n3 + 256.0f * n4 + b.n5;
    b.r6 = sqrtf(m.n6) * (0.5f / 256.0f * kUp);
    b.r5 = n6 * (1.0f / 256.0f) + b.r6;
    b.wide = n6 * 65536.0f * 129.0f * root * kUp;
    // ||a||: the first digit's, and the rest at most 0.502 of its unit each
    b.N = m.amax == 0 ? 0.0f : 4294967296.0f * kUp * (sqrtf(m.q1) + 0.502f * root);
    // the chain's 2^-53 x 128 N N (the partial sums between two checked ones)
    const float chain = 128.0f * 1.1102230246251565e-16f * kUp;
    b.X = sqrtf(65536.0f * n4 * n4 * kUp + chain * b.N * b.N);
    if (!finite_bits(m.amax)) b.N = b.P = __builtin_inff();
    b.e = row_exponent(m.amax);
    b.out_a = m.out_a;
    b.out_l = m.out_l;
    b.out = ldexpf(fabsf(m.out_a), 39 - b.e);
    return b;
}

// A workgroup: 64 x 64 outputs by 2 x 2 waves of 32 x 32 (96 accumulator registers each), two workgroups on a CU, so that
// one's epilogue and barriers run beside the other's matrix instructions (128 x 64 outputs by eight waves, the same
// registers and a quarter less traffic, measured 3% to 24% slower).
constexpr int kTile = 64;
constexpr int kCopies = 4 * kDigits;    // 1 KB copies per 32-l step
constexpr int kCopiesPerWave = kCopies / 4;

__device__ __forceinline__ int64_t split_xcd_contiguous(int64_t hw, int64_t n) {
    constexpr int64_t kXcds = 8;
    const int64_t q = n / kXcds, r = n % kXcds, x = hw % kXcds, k = hw / kXcds;
    return x < r ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
}

__device__ __forceinline__ v16i mfma_i8(v4i a, v4i b, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

constexpr int64_t kSplitGroupRows = 4;

// One window or reduction of at most kMaxWindow; several windows (in sequence or in parallel); a longer reduction in
// legs of kMaxWindow, whose sums are added in double.
enum SplitMode { kOne = 0, kWindows = 1, kLong = 2 };

template <int kMode>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void split_gemm_kernel(
    SplitParams p, int64_t gx, int64_t gy) {
    constexpr bool kSeg = kMode == kWindows;
    __shared__ __attribute__((aligned(16))) int8_t ring[kRing][kCopies * kFragment];
    __shared__ RowBound rows_i[kTile];
    __shared__ RowBound rows_j[kTile];
    __shared__ float predicted[2];
    __shared__ uint32_t undecided, base_slot, full;
    const int tid = static_cast<int>(threadIdx.x);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int wi = wave >> 1, wj = wave & 1;
    const int64_t id = split_xcd_contiguous(blockIdx.x, gx * gy);
    const int64_t first = id / (kSplitGroupRows * gx) * kSplitGroupRows;
    const int64_t rows_in_group = gy - first < kSplitGroupRows ? gy - first : kSplitGroupRows;
    const int64_t by = first + (id % (kSplitGroupRows * gx)) % rows_in_group;
    const int64_t bx = (id % (kSplitGroupRows * gx)) / rows_in_group;
    const int64_t i_blk = by * kTile, j_blk = bx * kTile;
    const int s_begin = p.partial ? static_cast<int>(blockIdx.y) : 0;
    const int s_end = kMode == kLong ? static_cast<int>((p.l1 + kMaxWindow - 1) / kMaxWindow)
                      : p.partial    ? s_begin + 1
                                     : p.nseg;
    const bool sequence = kSeg && !p.partial;
    uint8_t* flag = p.tile_flags + (static_cast<int64_t>(blockIdx.y) * gy + by) * gx + bx;

    // A step's 1 KB copies, dealt over the waves: copy c is digit c % 5 of block c / 5 of the tile (A's two, then B's). Copies
    // past the last step repeat it, so every wave always has the same number in flight.
    const uint32_t voff = static_cast<uint32_t>(lane) * 16;
    const int8_t* src[kCopiesPerWave];
    int dst[kCopiesPerWave];
#pragma unroll
    for (int t = 0; t < kCopiesPerWave; ++t) {
        const int c = wave + t * 4, blk = c / kDigits;
        const bool isa = blk < 2;
        const int64_t last = (isa ? p.a.blocks : p.b.blocks) - 1;
        const int64_t want = isa ? i_blk / 32 + blk : j_blk / 32 + blk - 2;
        src[t] = (isa ? p.a.digits : p.b.digits) + (want < last ? want : last) * p.stages * kStageBytes +
                 (c % kDigits) * kFragment;
        dst[t] = c * kFragment;
    }
    auto issue = [&](int buf, int64_t step) {
#pragma unroll
        for (int t = 0; t < kCopiesPerWave; ++t)
            copy16_to_lds_s(src[t] + step * kStepBytes, voff, &ring[buf][dst[t]]);
    };
    const int fa = wi * kStepBytes + lane * 16, fb = (2 + wj) * kStepBytes + lane * 16;

    const int jl = wj * 32 + (lane & 31);  // this lane's column in the tile
    const int64_t j = j_blk + jl;
    // the tile row of this lane's output r
    auto row_of = [&](int r) { return wi * 32 + 8 * (r / 4) + 4 * (lane >> 5) + r % 4; };
    float run[16];
    uint32_t open = 0;  // outputs left undecided by some window
#pragma unroll
    for (int r = 0; r < 16; ++r) run[r] = 0.0f;
    bool heavy = false, use6 = false;  // use6: this window adds the sixth digit's products
    if (tid == 0) undecided = full = 0;
    double sum[kMode == kLong ? 16 : 1];  // the legs before, and the bound on them
    float bound[kMode == kLong ? 16 : 1];
    if constexpr (kMode == kLong) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = 0.0, bound[r] = 0.0f;
    }

    for (int s = s_begin; s < s_end; ++s) {
        const Window w = kMode == kLong ? Window{s * kMaxWindow, p.l1 < (s + 1) * kMaxWindow ? p.l1 : (s + 1) * kMaxWindow,
                                                 s * (kMaxWindow / kStageL)}
                                        : window_of(p, s);
        const int64_t len = w.l1 - w.l0, nst = (len + kStageL - 1) / kStageL;
        const float lenf = static_cast<float>(kMode == kLong ? p.l1 : len);
        if (tid == 0) predicted[0] = predicted[1] = 0.0f;
        const int64_t steps = 2 * nst, step0 = 2 * w.stage0;
        if (nst > 0) {
            issue(0, step0);
            issue(1, step0 + 1);
            issue(2, step0 + (steps > 2 ? 2 : 1));
        }
        for (int k = tid; k < 2 * kTile && (kMode != kLong || s == 0); k += 256) {
            const bool isa = k < kTile;
            const Operand& o = isa ? p.a : p.b;
            const int64_t r = isa ? i_blk + k : j_blk + k - kTile;
            RowMeta m{};
            if (r < o.rows) m = o.meta[static_cast<int64_t>(kSeg ? s : 0) * o.blocks * 32 + r];
            (isa ? rows_i[k] : rows_j[k - kTile]) = row_bound(m, lenf);
        }
        __syncthreads();
        const RowBound bj = rows_j[jl];
        // The expected number of undecided outputs, from the bound against the typical size N_i N_j / sqrt(len) of a
        // sum (a result is undecided when a rounding boundary, one in every 2^-23 of its size, lies within the bound; 8
        // stands for the small results; within 30% of what Gaussian, product and lognormal operands measure). With
        // more than 1 in 160 the tile adds the sixth digit's products (a third of its time, against the recomputation's
        // 1e12 l per second); a tile of which more than 1 in 64 would be undecided even so is not begun.
        if (kMode != kLong || s == 0) {
            float q5 = 0.0f, q6 = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const RowBound& bi = rows_i[row_of(r)];
                const float e = bi.P * bj.n5 + bi.n5 * bj.P + bi.X * bj.X;
                const float e5 = e + bi.r5 * bj.N + bi.N * bj.r5;
                const float e6 = e + bi.r6 * bj.N + bi.N * bj.r6 + bi.wide + bj.wide;
                const float size = kMode == kLong ? bi.N * bj.N + bi.out * bj.N : bi.N * bj.N;
                const float per = 8.0f * 16777216.0f * __builtin_amdgcn_sqrtf(lenf) / size;
                q5 += size == 0.0f ? 0.0f : fminf(1.0f, e5 * per);
                q6 += size == 0.0f ? 0.0f : fminf(1.0f, e6 * per);
                if (!(e5 < __builtin_inff())) q5 = q6 += 64.0f;
            }
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) {
                q5 += __shfl_xor(q5, d);
                q6 += __shfl_xor(q6, d);
            }
            if (lane == 0) {
                atomicAdd(&predicted[0], q5);
                atomicAdd(&predicted[1], q6);
            }
        }
        __syncthreads();
        if (kMode != kLong || s == 0) {
            use6 = kMode != kLong && predicted[0] > kTile * kTile / 160.0f;
            if (!(predicted[use6 ? 1 : 0] <= kTile * kTile / 64.0f)) heavy = true;
        }
        if (heavy) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first stage's copies have landed
            break;
        }

        v16i acc[kOrders];
#pragma unroll
        for (int m = 0; m < kOrders; ++m) acc[m] = v16i{};
        float sabs[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) sabs[r] = 0.0f;
        // Step c: its fragments are in registers; while its MFMAs run, those of step c + 1 are read from LDS, and steps
        // c + 2 and c + 3 are on their way to it. The wait: this wave's copies of step c + 1 have landed (the ones after
        // it may still fly) and its reads of step c are done; after the barrier everyone's are, so step c's buffer is
        // free for step c + 3.
        v4i a0[kDigits], b0[kDigits], a1[kDigits], b1[kDigits];
        int buf = 0;
        auto next = [&](int k) { return buf + k < kRing ? buf + k : buf + k - kRing; };
        auto fragment = [&](const int8_t* from, int n, v4i (&a)[kDigits], v4i (&b)[kDigits]) {
            a[n] = *reinterpret_cast<const v4i*>(from + fa + n * kFragment);
            b[n] = *reinterpret_cast<const v4i*>(from + fb + n * kFragment);
        };
        auto check_sums = [&](int r) {
            sabs[r] += __builtin_fabsf(
                __builtin_fmaf(static_cast<float>(acc[0][r]), 256.0f, static_cast<float>(acc[1][r])));
        };
        // The wave's MFMAs of a step, the orders round-robin and the two checked orders last, with the next step's reads and
        // copies in their shadows: the matrix core waits for nothing but the barrier (all of them ahead of the MFMAs left
        // it idle for an eighth of the step). check: the partial sums as the step before left them.
        auto step = [&](int64_t c, bool check, const v4i (&a)[kDigits], const v4i (&b)[kDigits], v4i (&an)[kDigits],
                        v4i (&bn)[kDigits]) {
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kCopiesPerWave) : "memory");
            const int64_t ahead = step0 + (c + 3 < steps ? c + 3 : steps - 1);
            const int8_t* from = ring[next(1)];  // after the last step: bytes that are never used
            constexpr int kPairs[19][2] = {{0, 4}, {1, 4}, {0, 3}, {0, 2}, {1, 3}, {2, 3}, {1, 2}, {1, 1}, {2, 2}, {3, 2},
                                           {2, 1}, {2, 0}, {3, 1}, {4, 1}, {3, 0}, {4, 0}, {0, 1}, {1, 0}, {0, 0}};
#pragma unroll
            for (int n = 0; n < 19; ++n) {
                const int d = kPairs[n][0], q = kPairs[n][1];
                acc[d + q] = mfma_i8(a[d], b[q], acc[d + q]);
                if (n < kDigits) fragment(from, n, an, bn);
                if (n >= kDigits && n < kDigits + kCopiesPerWave)
                    copy16_to_lds_s(src[n - kDigits] + ahead * kStepBytes, voff, &ring[buf][dst[n - kDigits]]);
                if (n >= 11 && n < 15 && check) {
#pragma unroll
                    for (int r = (n - 11) * 4; r < (n - 10) * 4; ++r) check_sums(r);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            buf = next(1);
        };
        if (steps > 0) {
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * kCopiesPerWave) : "memory");
#pragma unroll
            for (int n = 0; n < kDigits; ++n) fragment(ring[0], n, a0, b0);
        }
        for (int64_t c = 0; c < steps; c += 2) {  // an even number of steps
            step(c, c % kCheckSteps == 0, a0, b0, a1, b1);
            step(c + 1, false, a1, b1, a0, b0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) check_sums(r);
        // the surplus copies have landed everywhere before the ring is used again
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

        if (use6) {
            // The sixth digit's products with the first, (1, 6) and (6, 1), into the last accumulator: two digits of each
            // block, kBatch steps to a barrier, the next ones on their way to the other half of the ring.
            constexpr int kBatch = 3;
            static_assert(2 * kBatch * 8 <= kRing * kCopies, "two batches of 8 KB steps in the ring");
            int8_t* const half0 = &ring[0][0];
            auto issue6 = [&](int64_t c) {  // past the last step: the last one again, never used
                const bool isa = wave < 2;  // this wave's block: A's two, then B's
                const int64_t last = (isa ? p.a.blocks : p.b.blocks) - 1;
                const int64_t want = isa ? i_blk / 32 + wave : j_blk / 32 + wave - 2;
                const int64_t row = (want < last ? want : last) * p.stages * 2 + step0;
#pragma unroll
                for (int t = 0; t < 2 * kBatch; ++t) {
                    const int64_t at = row + (c + t / 2 < steps ? c + t / 2 : steps - 1);
                    const int8_t* from = t % 2 == 0 ? (isa ? p.a.digits : p.b.digits) + at * kStepBytes
                                                    : (isa ? p.a.digits6 : p.b.digits6) + at * kFragment;
                    copy16_to_lds_s(from, voff, half0 + (c / kBatch % 2 * kBatch * 8 + t / 2 * 8 + 2 * wave + t % 2) *
                                                            kFragment);
                }
            };
            if (steps > 0) issue6(0);
            for (int64_t c = 0; c < steps; c += kBatch) {
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                if (c + kBatch < steps) issue6(c + kBatch);
#pragma unroll
                for (int t = 0; t < kBatch; ++t) {
                    if (c + t >= steps) break;
                    const int8_t* mem = half0 + (c / kBatch % 2 * kBatch * 8 + t * 8) * kFragment + lane * 16;
                    const v4i a1 = *reinterpret_cast<const v4i*>(mem + wi * 2 * kFragment);
                    const v4i a6 = *reinterpret_cast<const v4i*>(mem + (wi * 2 + 1) * kFragment);
                    const v4i b1 = *reinterpret_cast<const v4i*>(mem + (2 + wj) * 2 * kFragment);
                    const v4i b6 = *reinterpret_cast<const v4i*>(mem + ((2 + wj) * 2 + 1) * kFragment);
                    acc[kOrders - 1] = mfma_i8(a1, b6, acc[kOrders - 1]);
                    acc[kOrders - 1] = mfma_i8(a6, b1, acc[kOrders - 1]);
                }
            }
        }

        // the window's results
        // 2^-53 x 128 x (the checked sums, in units of 256^7), and len 2^-53 x (what the checked sums leave out: the
        // digits below the second, at most 2^23.02 sqrt(len) (N_i + N_j), and d_2 d_2, at most 2^62 len)
        const float kChain = 128.0f * 1.1102230246251565e-16f * kUp * 72057594037927936.0f;
        const float below = lenf * 1.1102230246251565e-16f * 8700000.0f * kUp * __builtin_amdgcn_sqrtf(lenf);
        const float below2 = lenf * 1.1102230246251565e-16f * 4611686018427387904.0f * kUp * lenf;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int il = row_of(r);
            const RowBound& bi = rows_i[il];
            const int64_t i = i_blk + il;
            double v = static_cast<double>(acc[0][r]);
#pragma unroll
            for (int m = 1; m < kOrders; ++m) v = __builtin_fma(v, 256.0, static_cast<double>(acc[m][r]));
            const int ex = bi.e + bj.e - 78;
            float ef = sabs[r] * kChain;
            if constexpr (kMode == kLong) {
                // the partial sums of this leg start from the legs before; the rest of the bound is of the whole row
                ef += static_cast<float>(__builtin_fabs(sum[r])) * (16777216.0f * 1.1102230246251565e-16f * kUp) *
                      static_cast<float>(len);
                ef += (static_cast<float>(__builtin_fabs(v)) + static_cast<float>(__builtin_fabs(sum[r]))) *
                      (16777216.0f * 8.9e-16f);  // the leg's Horner steps and the sum of the legs
                bound[r] += ef;
                sum[r] += v;
                if (s + 1 < s_end) continue;
                v = sum[r];
                ef = bound[r];
            }
            v = ldexp(v, ex + 24);
            ef += bi.P * bj.n5 + bi.n5 * bj.P + bi.X * bj.X;
            ef += use6 ? bi.r6 * bj.N + bi.N * bj.r6 + bi.wide + bj.wide : bi.r5 * bj.N + bi.N * bj.r5;
            ef += below * (bi.N + bj.N) + below2;
            if (bi.N * bj.N == 0.0f) ef = 0.0f;  // a zero row: every partial sum is exactly 0
            double e = ldexp(static_cast<double>(ef) * 1.01, ex);
            e += __builtin_fabs(v) * 8.8817841970012523e-16;  // 2^-50: the Horner steps' own rounding
            if constexpr (kMode == kLong) {
                if (bi.out_a != 0.0f && i < p.I && j < p.J) {
                    const double o = static_cast<double>(bi.out_a) * static_cast<double>(p.out_b[bi.out_l * p.ld_out_b + j]);
                    v += o;
                    // every partial sum after it holds it
                    e += __builtin_fabs(o) * (static_cast<double>(p.l1) * 1.13e-16) + __builtin_fabs(v) * 2.3e-16;
                }
            }
            if (!kSeg && p.bias && j < p.J && i < p.I) {
                const double b = static_cast<double>(p.bias[j]);
                v += b;
                e += __builtin_fabs(v) * 8.8817841970012523e-16;
            }
            const float lo = static_cast<float>(v - e), hi = static_cast<float>(v + e);
            const bool inside = i < p.I && j < p.J;
            const bool undec = inside && (!(__float_as_uint(lo) == __float_as_uint(hi)) || !(e < __builtin_inf()));
            float x = lo;
            if constexpr (kSeg) {
                if (inside) {
                    if (p.seg_addrow) {
                        const int ar = p.seg_addrow[static_cast<int64_t>(s) * p.ld_addrow + i];
                        x = x + (ar >= 0 ? p.seg_addend[ar * p.ld_seg_add + j] : 0.0f);
                    }
                    if (p.seg_rowscale) x = x * p.seg_rowscale[i];
                    if (p.seg_weight) x = x * p.seg_weight[s];
                }
                if (sequence) {
                    const bool was = open >> r & 1;
                    if (undec) {
                        uint32_t slot = was ? __float_as_uint(run[r]) : atomicAdd(&p.count[2], 1u);
                        const uint32_t item = atomicAdd(&p.count[0], 1u);
                        atomicAdd(&undecided, 1u);
                        if (slot >= p.slot_cap || item >= p.list_cap) full = 1;  // the tile goes to the FP64 matmul
                        if (item < p.list_cap)
                            p.list[item] = slot < p.slot_cap ? (static_cast<uint64_t>(s) << 48) | slot : ~uint64_t{0};
                        if (!was && slot < p.slot_cap) {
                            p.slots[slot] = (static_cast<uint64_t>(s) << 48) | static_cast<uint64_t>(i * p.J + j);
                            p.slot_values[static_cast<int64_t>(slot) * (1 + p.nseg)] = run[r];
                        }
                        run[r] = __uint_as_float(slot);
                        open |= 1u << r;
                    } else if (was) {
                        const uint32_t slot = __float_as_uint(run[r]);
                        if (slot < p.slot_cap) p.slot_values[static_cast<int64_t>(slot) * (1 + p.nseg) + 1 + s] = x;
                    } else {
                        run[r] = s == s_begin ? x : run[r] + x;
                    }
                    continue;
                }
            }
            run[r] = x;
            if (undec) open |= 1u << r;
        }
        __syncthreads();  // rows_i and rows_j are read before the next window's are written
    }

    const uint32_t mine = heavy || sequence ? 0 : static_cast<uint32_t>(__popc(open));
    uint32_t slot = 0;
    if (mine) slot = atomicAdd(&undecided, mine);
    __syncthreads();
    const uint32_t total = undecided;
    if (total > kTile * kTile / 32 * (sequence ? static_cast<uint32_t>(p.nseg) : 1u) || full) heavy = true;
    if (!sequence && !heavy && total > 0) {
        if (tid == 0) base_slot = atomicAdd(p.count, total);
        __syncthreads();
        if (base_slot + total > p.list_cap) {  // the list is full: the tile goes to the FP64 matmul, its slots stay empty
            for (uint32_t k = tid; k < total; k += 256)
                if (base_slot + k < p.list_cap) p.list[base_slot + k] = ~uint64_t{0};
            heavy = true;
        }
    }
    if (tid == 0) {
        *flag = heavy ? 1 : 0;
        if (heavy) {
            atomicAdd(&p.count[1], 1u);
            if (p.stat) atomicAdd(p.stat, 1u);
        }
    }
    if (heavy) return;
    float* out = p.partial ? p.partial + static_cast<int64_t>(blockIdx.y) * p.I * p.J : p.C;
    const int64_t ld = p.partial ? p.J : p.ldc;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t i = i_blk + row_of(r);
        if (i >= p.I || j >= p.J) continue;
        if (open >> r & 1) {
            if (!sequence) p.list[base_slot + slot++] = (static_cast<uint64_t>(blockIdx.y) << 48) | static_cast<uint64_t>(i * p.J + j);
        } else {
            float x = run[r];
            if (!kSeg && p.addsrc) x = p.addsrc[i * p.ld_add + j] + x;
            out[i * ld + j] = x;
        }
    }
}

// The undecided outputs, by their chains in the reference's order. A workgroup takes kFixRows (output, window) pairs.
// Four waves form the products of kFixL l of every pair (exact in double, so multiply-then-add rounds like the fused
// form) from 16-byte loads along l, two chunks ahead; a fifth adds the chunk before in order, one lane per pair, so the
// chain waits for nothing but its adds. Few pairs are in flight, so the time is the chain's: 128 l took 1.2 us with one
// chunk in flight and the adds between two barriers.
constexpr int kFixRows = 32;
constexpr int kFixL = 128;

struct ChainBuffers {
    // products of l 4 k, 4 k + 1 at 2 k, those of 4 k + 2, 4 k + 3 at kFixL / 2 + 2 k: 16-byte writes of consecutive
    // lanes are adjacent
    __attribute__((aligned(16))) double prod[2][kFixRows][kFixL + 2];
    const float* a[kFixRows];
    const float* b[kFixRows];
    int len[kFixRows];
};

// The serial double sums of a[q][l] b[q][l], l ascending, of the workgroup's kFixRows pairs: the result of pair q in
// thread 256 + q. Called by all 320 threads once the buffers' pointers and lengths are visible. Loads are 16 bytes: those
// past a pair's length must read zeros or, for lengths that are multiples of 4, do not happen.
__device__ __forceinline__ double chains(ChainBuffers& s, int tid) {
    int longest = 0;
#pragma unroll 8
    for (int q = 0; q < kFixRows; ++q) longest = max(longest, s.len[q]);
    const int chunks = (longest + kFixL - 1) / kFixL;
    double acc = 0.0;
    if (tid < 256) {  // wave-uniform
        constexpr int kN = kFixRows / 8;
        const int q0 = tid >> 5, lq = (tid & 31) * 4;  // this thread's pairs q0 + 8 k, and its l in a chunk
        const float *ga[kN], *gb[kN];
        int len[kN];
#pragma unroll
        for (int q = 0; q < kN; ++q) {
            ga[q] = s.a[q0 + 8 * q] + lq;
            gb[q] = s.b[q0 + 8 * q] + lq;
            len[q] = s.len[q0 + 8 * q] - lq;
        }
        float4 x0[kN], y0[kN], x1[kN], y1[kN];
        auto load = [&](float4 (&x)[kN], float4 (&y)[kN], int l) {
#pragma unroll
            for (int q = 0; q < kN; ++q) {
                const bool in = l < len[q];
                const float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
                x[q] = in ? *reinterpret_cast<const float4*>(ga[q] + l) : zero;
                y[q] = in ? *reinterpret_cast<const float4*>(gb[q] + l) : zero;
            }
        };
        auto form = [&](const float4 (&x)[kN], const float4 (&y)[kN], int c) {
#pragma unroll
            for (int q = 0; q < kN; ++q) {
                double* d = &s.prod[c & 1][q0 + 8 * q][lq / 2];
                *reinterpret_cast<double2*>(d) = double2{static_cast<double>(x[q].x) * static_cast<double>(y[q].x),
                                                         static_cast<double>(x[q].y) * static_cast<double>(y[q].y)};
                *reinterpret_cast<double2*>(d + kFixL / 2) =
                    double2{static_cast<double>(x[q].z) * static_cast<double>(y[q].z),
                            static_cast<double>(x[q].w) * static_cast<double>(y[q].w)};
            }
        };
        load(x0, y0, 0);
        load(x1, y1, kFixL);
        for (int c = 0; c < chunks; c += 2) {
            form(x0, y0, c);
            load(x0, y0, (c + 2) * kFixL);
            lds_barrier();
            if (c + 1 >= chunks) break;
            form(x1, y1, c + 1);
            load(x1, y1, (c + 3) * kFixL);
            lds_barrier();
        }
        return acc;
    }
    for (int c = 0; c < chunks; ++c) {
        lds_barrier();  // chunk c is formed; the producers go on to chunk c + 1
        if (tid - 256 < kFixRows) {  // past a pair's length the products are +0, which change no sum
            const double2* lo = reinterpret_cast<const double2*>(s.prod[c & 1][tid - 256]);
            const double2* hi = lo + kFixL / 4;
            double2 t[8];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[2 * u] = lo[u], t[2 * u + 1] = hi[u];
#pragma unroll
            for (int e = 0; e < kFixL / 4; e += 4) {  // 16 l
                double2 tn[8];
                const int en = e + 4 < kFixL / 4 ? e + 4 : 0;
#pragma unroll
                for (int u = 0; u < 4; ++u) tn[2 * u] = lo[en + u], tn[2 * u + 1] = hi[en + u];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    acc = acc + t[u].x;
                    acc = acc + t[u].y;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 8; ++u) t[u] = tn[u];
            }
        }
    }
    return acc;
}

template <bool kSeg>
__global__ __launch_bounds__(320) __attribute__((amdgpu_waves_per_eu(2))) void split_fix_kernel(SplitParams p) {
    __shared__ ChainBuffers s_mem;
    const uint32_t n = *p.count < p.list_cap ? *p.count : p.list_cap;
    const int tid = static_cast<int>(threadIdx.x);
    const bool owner = tid >= 256 && tid - 256 < kFixRows;  // the lanes that add
    const int row = owner ? tid - 256 : 0;
    const bool sequence = kSeg && !p.partial;
    if (p.stat && blockIdx.x == 0 && tid == 0) atomicAdd(p.stat + 1, n);
    for (uint32_t k0 = blockIdx.x * kFixRows; k0 < n; k0 += gridDim.x * kFixRows) {
        const uint32_t k = k0 + static_cast<uint32_t>(row);
        const uint64_t item = k < n ? p.list[k] : ~uint64_t{0};
        const bool valid = item != ~uint64_t{0};
        const int s = kSeg && valid ? static_cast<int>(item >> 48) : 0;
        const int64_t low = static_cast<int64_t>(item & ((uint64_t{1} << 48) - 1));
        const int64_t at = !valid ? 0
                           : sequence ? static_cast<int64_t>(p.slots[low] & ((uint64_t{1} << 48) - 1))
                                      : low;
        const int64_t i = at / p.J, j = at % p.J;
        __syncthreads();  // the pairs before are done
        if (owner) {
            const Window w = window_of(p, s);
            s_mem.a[row] = p.a.rows_contiguous ? p.a.t + (i * p.stages + w.stage0) * kStageL : p.a.src + i * p.a.ld;
            s_mem.b[row] = p.b.rows_contiguous ? p.b.t + (j * p.stages + w.stage0) * kStageL : p.b.src + j * p.b.ld;
            s_mem.len[row] = valid ? static_cast<int>(w.l1 - w.l0) : 0;
        }
        __syncthreads();
        // past a window's end the transposed copy holds zeros; a row-major operand's reduction is a multiple of 4
        double acc = chains(s_mem, tid);
        if (!owner || !valid) continue;
        if constexpr (!kSeg) {
            if (p.bias) acc += static_cast<double>(p.bias[j]);
            float v = static_cast<float>(acc);
            if (p.addsrc) v = p.addsrc[i * p.ld_add + j] + v;
            p.C[i * p.ldc + j] = v;
        } else {
            float v = static_cast<float>(acc);
            if (p.seg_addrow) {
                const int ar = p.seg_addrow[static_cast<int64_t>(s) * p.ld_addrow + i];
                v = v + (ar >= 0 ? p.seg_addend[ar * p.ld_seg_add + j] : 0.0f);
            }
            if (p.seg_rowscale) v = v * p.seg_rowscale[i];
            if (p.seg_weight) v = v * p.seg_weight[s];
            if (sequence)
                p.slot_values[low * (1 + p.nseg) + 1 + s] = v;
            else
                p.partial[(static_cast<int64_t>(s) * p.I + i) * p.J + j] = v;
        }
    }
}

// A forward matmul of few outputs (a token or a few through a projection): every output's chain as above, straight from
// x and the weight's rows, 32 outputs per workgroup (rows of a token side by side, so a weight row is read once from
// memory). The time is a read of the weight and one chain. 1 x 896 x 4864: the transpose of the weight and 32 x 32 tiles
// took 22.8 us, this takes 11.8.
__global__ __launch_bounds__(320) __attribute__((amdgpu_waves_per_eu(2))) void chain_linear_kernel(
    const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw, const float* __restrict__ bias,
    const float* __restrict__ addsrc, int64_t ld_add, float* __restrict__ out, int64_t ldc, int64_t rows, int64_t outs,
    int len) {
    __shared__ ChainBuffers s_mem;
    const int tid = static_cast<int>(threadIdx.x);
    const bool owner = tid >= 256 && tid - 256 < kFixRows;
    const int q = owner ? tid - 256 : 0;
    const int64_t k = static_cast<int64_t>(blockIdx.x) * kFixRows + q;
    const bool valid = k < rows * outs;
    const int64_t i = valid ? k % rows : 0, j = valid ? k / rows : 0;
    if (owner) {
        s_mem.a[q] = x + i * ldx;
        s_mem.b[q] = w + j * ldw;
        s_mem.len[q] = valid ? len : 0;
    }
    __syncthreads();
    double acc = chains(s_mem, tid);
    if (!owner || !valid) return;
    if (bias) acc += static_cast<double>(bias[j]);
    float v = static_cast<float>(acc);
    if (addsrc) v = addsrc[i * ld_add + j] + v;
    out[i * ldc + j] = v;
}

// Windows in sequence: each slot's output from the sum before its first undecided window and the results after it.
__global__ __launch_bounds__(256) void split_sum_kernel(SplitParams p, int64_t gx) {
    const uint32_t n = p.count[2] < p.slot_cap ? p.count[2] : p.slot_cap;
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
        const uint64_t slot = p.slots[k];
        const int first = static_cast<int>(slot >> 48);
        const int64_t at = static_cast<int64_t>(slot & ((uint64_t{1} << 48) - 1));
        const int64_t i = at / p.J, j = at % p.J;
        if (p.tile_flags[i / kTile * gx + j / kTile]) continue;  // the FP64 matmul's
        const float* v = p.slot_values + static_cast<int64_t>(k) * (1 + p.nseg);
        float run = first == 0 ? v[1] : v[0] + v[1 + first];
        for (int s = first + 1; s < p.nseg; ++s) run = run + v[1 + s];
        p.C[i * p.ldc + j] = run;
    }
}

// The scratch of one call (or row block): the shared operand's part first, at the same place for every call that shares
// it, then the other's, then the tile flags and the list of undecided outputs.
struct SplitLayout {
    int64_t a_blocks, b_blocks, nseg, stages, parts, tiles, at_rows, bt_rows;
    uint32_t list_cap, slot_cap;  // slot_cap 0: no windows in sequence
    bool b_first;
    size_t bytes;
};

void add_operand(Layout& y, int64_t blocks, int64_t t_rows, const SplitLayout& l) {
    y.add<int8_t>(static_cast<size_t>(blocks * l.stages) * kStageBytes);
    y.add<int8_t>(static_cast<size_t>(blocks * l.stages) * 2 * kFragment);
    y.add<RowMeta>(static_cast<size_t>(blocks * 32 * l.nseg));
    y.add<float>(static_cast<size_t>(t_rows * l.stages) * kStageL);
}

SplitLayout split_layout(const GemmCall& g, int64_t z) {
    SplitLayout l{};
    l.a_blocks = ceil_div(g.I, 32);
    l.b_blocks = ceil_div(g.J, 32);
    l.nseg = g.seg ? g.nseg : 1;
    l.stages = g.l1 / kStageL + l.nseg;
    l.parts = g.l1 / kPartL + l.nseg;
    l.tiles = ceil_div(g.I, kTile) * ceil_div(g.J, kTile) * z;
    l.at_rows = g.a_kind == 2 ? 0 : g.I;
    l.bt_rows = g.Bt ? 0 : g.J;
    l.b_first = g.split_share == 2;
    l.list_cap = static_cast<uint32_t>(std::min<int64_t>(std::max<int64_t>(g.I * g.J * z / 64, 1 << 16), 1 << 25));
    if (g.seg && z == 1) {  // room for 1 in 160 undecided chains per window, in outputs of their own and in all
        const int64_t outs = std::max<int64_t>(g.I * g.J * std::min<int64_t>(l.nseg, 16) / 160, 1 << 14);
        l.slot_cap = static_cast<uint32_t>(std::min<int64_t>(outs, 1 << 24));
        l.list_cap = l.slot_cap + l.slot_cap / 2;
    }
    Layout y;
    for (int k = 0; k < 2; ++k) {
        if ((k == 0) == l.b_first) add_operand(y, l.b_blocks, l.bt_rows, l);
        else add_operand(y, l.a_blocks, l.at_rows, l);
    }
    y.add<uint8_t>(static_cast<size_t>(l.tiles));
    y.add<uint32_t>(3);
    y.add<uint64_t>(l.list_cap);
    y.add<uint64_t>(l.slot_cap);
    y.add<float>(static_cast<size_t>(l.slot_cap) * static_cast<size_t>(1 + l.nseg));
    l.bytes = y.bytes + kAlign;
    return l;
}

// The windows' results go to memory of their own where the tiles in sequence are few.
bool split_parallel(const GemmCall& g) {
    return g.seg && g.nseg > 1 && g.seg_partial && g.nseg * g.I * g.J <= g.seg_partial_cap &&
           static_cast<int64_t>(ceil_div(g.I, kTile) * ceil_div(g.J, kTile)) < 2048;
}

// Where the int8 path pays, by the times both paths measure. Its passes (five launches, the recomputation) take about 50
// us, splitting 4 ps per operand value, and a round of the 512 workgroups that the chip holds 1.14 us per 32-l step (118
// TFLOP/s) and 10 us of epilogue per window. FP64's round of 512 tiles of 128 x 128 takes 0.247 us per l, a last round of
// at most one tile per CU 0.55 of that; launches of fewer tiles run at about 55 TFLOP/s. At 1023 x 8960 x 1536 the two
// measure 370 and 600 us, at 2048 x 896 x 4864 285 and 310, at 1024 x 576 x 49152 (144 workgroups) 1.8 and 1.2 ms.
// In blocks of `rows` rows B is split once, and every block has its own passes and rounds.
SplitCost split_cost(const GemmCall& g, int64_t rows) {
    const double I = static_cast<double>(g.I), J = static_cast<double>(g.J), L = static_cast<double>(g.l1);
    const int64_t z = split_parallel(g) ? g.nseg : 1;
    const int64_t windows = g.seg ? g.nseg / z : 1;
    const auto block = [&](int64_t n) {
        const double r = static_cast<double>(ceil_div(n, kTile) * ceil_div(g.J, kTile) * z) / 512.0;
        return 50e-6 + (r <= 1.0 ? 1.0 : r + 0.25) *
                           (L / static_cast<double>(z) / 32.0 * 1.14e-6 + static_cast<double>(windows) * 10e-6);
    };
    const int64_t rest = g.I % rows;
    const double split = (I + J) * L * 4e-12 + static_cast<double>(g.I / rows) * block(rows) + (rest ? block(rest) : 0.0);
    const int64_t big = ceil_div(g.I, 128) * ceil_div(g.J, 128) * z;
    const int64_t last = big % 512;
    const double fp64 = big >= 512 ? (static_cast<double>(big / 512) + (last == 0 ? 0.0 : last <= 256 ? 0.55 : 1.0)) *
                                         (L / static_cast<double>(z)) * 0.247e-6
                                   : 2.0 * I * J * L / 55e12;
    return {fp64, split, g.seg ? L / static_cast<double>(g.nseg) : L, L * static_cast<double>(ceil_div(g.I, rows)),
            g.seg != nullptr && z == 1};
}

bool split_pays(const GemmCall& g, int64_t rows) {
    const SplitCost c = split_cost(g, rows);
    return c.split < 0.95 * c.fp64;
}

// Whether the path takes the call's operands and reduction at all.
bool split_takes(const GemmCall& g) {
    if (g.a_kind == 0 || g.l0 != 0 || g.l1 < 256 || g.I <= 0 || g.J <= 0) return false;
    if (g.seg == nullptr ? g.l1 > kMaxWindow && (g.a_kind != 2 || g.Bt == nullptr || g.bt_transpose != nullptr || g.l1 >= (1 << 30)) : g.seg_max <= 0 || g.seg_max > kMaxWindow || g.nseg > 64) return false;
    return g.l1 / kPartL + (g.seg ? g.nseg : 1) <= 65535;
}

}  // namespace

size_t split_gemm_bytes(const GemmCall& g) {
    return split_takes(g) && split_pays(g, g.I) ? split_layout(g, split_parallel(g) ? g.nseg : 1).bytes : 0;
}

SplitCost gemm_split_cost(const GemmCall& g) { return split_cost(g, gemm_split_rows(g)); }

// Every 256 workgroups' worth of 32 chains take 9.6 ns per l (1030 x 1792 x 4320: 83 us for two rounds, 1792 x 1504 x 4320: 124
// us for three); the first round is in split_cost's estimate. Handed-back tiles, however few, take a tile's whole reduction
// in FP64, 70 to 130 ns per l: fewer than 160 of 476 tiles of 1030 x 1792 x 36000 took 2.53 ms (all of them in FP64 2.61),
// some of 4096 x 1536 x 151936 took 19.6 ms (29). In a sequence of windows an open output also costs its slot, 2 ns and
// more: the logits' gradient of 8192 rows and 151936 words times hidden 1536, 8 windows, takes 47.8 ms with 0.7 million
// chains (flat logits), 53.1 with 2.4 (logits of deviation 0.78), 73.6 with 3.4 (1.2), 113 with 4.4 (2), and 55.5 in FP64.
// A gain below an eighth of the FP64 time is within what the two estimates are off by and counts as that eighth.
bool gemm_split_lost(const SplitCost& c, const SplitDone& d) {
    const int64_t rounds = ceil_div(static_cast<int64_t>(d.chains), 256 * kFixRows);
    double t = static_cast<double>(rounds > 1 ? rounds - 1 : 0) * c.chain_l * 9.6e-9;
    if (c.sequence) t += static_cast<double>(d.chains) * 2.5e-9;
    if (d.tiles > 0) t += std::min(c.fp64, c.tile_l * std::max(130e-9, static_cast<double>(d.tiles) * 0.18e-9));
    return t > std::max(c.fp64 - c.split, c.fp64 / 8.0);
}

SplitPlan split_plan(const GemmCall& g) {
    SplitPlan plan;
    if (g.split_scratch == nullptr || !split_takes(g)) return plan;
    if (g.split_block) {  // decided with the whole call
        plan.rows = g.I;
        return plan;
    }
    if (!split_pays(g, g.I)) return plan;
    plan.parallel = split_parallel(g);
    if (split_layout(g, plan.parallel ? g.nseg : 1).bytes <= g.split_cap) {
        plan.rows = g.I;
        return plan;
    }
    if (plan.parallel) return plan;
    // the largest halving of the rows whose block fits: all blocks run here, or none
    GemmCall b = g;
    b.split_share = 2;
    for (b.I = (g.I / 2 + 127) / 128 * 128; b.I >= 1024; b.I = (b.I / 2 + 127) / 128 * 128)
        if (split_layout(b, 1).bytes <= g.split_cap) {
            if (split_pays(g, b.I)) plan.rows = b.I;
            return plan;
        }
    return plan;
}

// Few outputs: 256 workgroups (8192 outputs) side by side take 10.7 ns per l and 2 us, the tiled matmul 13.6 ns per l and,
// where it has to be made, the weight's transpose at about 2.5 TB/s. 1 x 896 x 4864: 11.8 us against 22.8; 2 x 896 x 4864:
// 20.9 against 22.8; 4 x 896 x 4864: 30.1 against 22.9 (not taken); 4 x 8960 x 1536: 78 against 122; 1 x 2048 x 50304:
// 160 against 476.
bool chain_linear_fits(const GemmCall& g) {
    if (g.a_kind != 2 || g.Bt == nullptr || g.seg != nullptr || g.l0 != 0 || g.l1 <= 0 || g.l1 >= (1 << 30)) return false;
    if (g.I > 64) return false;
    const double L = static_cast<double>(g.l1);
    const double transpose = g.bt_transpose ? 8.0 * L * static_cast<double>(g.J) / 2.5e12 : 0.0;
    return static_cast<double>(ceil_div(g.I * g.J, 256 * kFixRows)) * L * 10.7e-9 + 2e-6 < L * 13.6e-9 + transpose;
}

int launch_chain_linear(const GemmCall& g, hipStream_t stream) {
    const int64_t pairs = g.I * g.J;
    hipLaunchKernelGGL(chain_linear_kernel, dim3(static_cast<unsigned>(ceil_div(pairs, kFixRows))), dim3(320), 0, stream,
                       g.Af, g.lda, g.Bt, g.ldbt, g.bias, g.addsrc, g.ld_add, g.C, g.ldc, g.I, g.J,
                       static_cast<int>(g.l1));
    return check_launch("chain linear");
}

int launch_split_gemm(const GemmCall& g, float* partial, hipStream_t stream, SplitRedo* redo) {
    const int64_t z = partial ? g.nseg : 1;
    const SplitLayout l = split_layout(g, z);
    Carve c(g.split_scratch, g.split_cap);
    SplitParams p{};
    const bool bt = g.Bt != nullptr;
    p.a = {g.Af, g.lda, g.a_kind == 1, g.I, l.a_blocks, nullptr, nullptr, nullptr, nullptr};
    p.b = {bt ? g.Bt : g.B, bt ? g.ldbt : g.ldb, bt ? 0 : 1, g.J, l.b_blocks, nullptr, nullptr, nullptr, nullptr};
    for (int k = 0; k < 2; ++k) {
        const bool isb = (k == 0) == l.b_first;
        Operand& o = isb ? p.b : p.a;
        o.digits = c.take<int8_t>(static_cast<size_t>(o.blocks * l.stages) * kStageBytes);
        o.digits6 = c.take<int8_t>(static_cast<size_t>(o.blocks * l.stages) * 2 * kFragment);
        o.meta = c.take<RowMeta>(static_cast<size_t>(o.blocks * 32 * l.nseg));
        o.t = c.take<float>(static_cast<size_t>((isb ? l.bt_rows : l.at_rows) * l.stages) * kStageL);
    }
    p.tile_flags = c.take<uint8_t>(static_cast<size_t>(l.tiles));
    p.count = c.take<uint32_t>(3);
    p.list = c.take<uint64_t>(l.list_cap);
    p.slots = c.take<uint64_t>(l.slot_cap);
    p.slot_values = c.take<float>(static_cast<size_t>(l.slot_cap) * static_cast<size_t>(1 + l.nseg));
    p.slot_cap = l.slot_cap;
    DLLM_REQUIRE(!c.overflow, "split matmul scratch too small");
    p.list_cap = l.list_cap;
    p.out_b = g.B;
    p.ld_out_b = g.ldb;
    p.stages = l.stages;
    p.seg = g.seg;
    p.nseg = static_cast<int>(l.nseg);
    p.l1 = g.l1;
    p.C = g.C;
    p.ldc = g.ldc;
    p.I = g.I;
    p.J = g.J;
    p.bias = g.bias;
    p.addsrc = g.addsrc;
    p.ld_add = g.ld_add;
    p.seg_addend = g.seg_addend;
    p.seg_addrow = g.seg_addrow;
    p.ld_addrow = g.ld_addrow ? g.ld_addrow : g.I;
    p.ld_seg_add = g.ld_seg_add;
    p.seg_weight = g.seg_weight;
    p.seg_rowscale = g.seg_rowscale;
    p.partial = partial;
    p.stat = g.split_stat;
    // a shared operand that the call before left in the scratch is not split again
    const bool a_ready = g.split_ready && g.split_share == 1, b_ready = g.split_ready && g.split_share == 2;
    const int64_t per = 32 * l.nseg * static_cast<int64_t>(sizeof(RowMeta) / 16);
    const int64_t na = a_ready ? 0 : l.a_blocks * per, nb = b_ready ? 0 : l.b_blocks * per;
    hipLaunchKernelGGL(split_clear_kernel,
                       dim3(static_cast<unsigned>(std::min<int64_t>(ceil_div(na + nb + 1, 256), 1024))), dim3(256), 0,
                       stream, reinterpret_cast<uint4*>(p.a.meta), na, reinterpret_cast<uint4*>(p.b.meta), nb, p.count);
    DLLM_TRY(check_launch("split clear"));
    const int64_t pa = a_ready ? 0 : ceil_div(g.I, kSplitRows), pb = b_ready ? 0 : ceil_div(g.J, kSplitRows);
    const bool is_long = g.seg == nullptr && g.l1 > kMaxWindow;
    if (pa + pb > 0) {
        const dim3 pgrid(static_cast<unsigned>(pa + pb), static_cast<unsigned>(l.parts));
        const int64_t ma = is_long ? 0 : pa;  // a long reduction's A rows: their largest two values
        if (pa > ma) {
            hipLaunchKernelGGL(split_top_kernel, dim3(static_cast<unsigned>(g.I)), dim3(256), 0, stream, p.a, g.l1);
            DLLM_TRY(check_launch("split top"));
        }
        if (ma + pb > 0) {
            hipLaunchKernelGGL(split_amax_kernel, dim3(static_cast<unsigned>(ma + pb), pgrid.y), dim3(256), 0, stream, p,
                               ma);
            DLLM_TRY(check_launch("split amax"));
        }
        if (is_long) hipLaunchKernelGGL(split_digits_kernel<true>, pgrid, dim3(256), 0, stream, p, pa);
        else hipLaunchKernelGGL(split_digits_kernel<false>, pgrid, dim3(256), 0, stream, p, pa);
        DLLM_TRY(check_launch("split digits"));
    }
    const int64_t gx = ceil_div(g.J, kTile), gy = ceil_div(g.I, kTile);
    const dim3 grid(static_cast<unsigned>(gx * gy), static_cast<unsigned>(z));
    if (g.seg) hipLaunchKernelGGL(split_gemm_kernel<kWindows>, grid, dim3(256), 0, stream, p, gx, gy);
    else if (is_long) hipLaunchKernelGGL(split_gemm_kernel<kLong>, grid, dim3(256), 0, stream, p, gx, gy);
    else hipLaunchKernelGGL(split_gemm_kernel<kOne>, grid, dim3(256), 0, stream, p, gx, gy);
    DLLM_TRY(check_launch("split gemm"));
    if (g.seg) hipLaunchKernelGGL(split_fix_kernel<true>, dim3(512), dim3(320), 0, stream, p);
    else hipLaunchKernelGGL(split_fix_kernel<false>, dim3(512), dim3(320), 0, stream, p);
    DLLM_TRY(check_launch("split fix"));
    if (l.slot_cap > 0) {
        hipLaunchKernelGGL(split_sum_kernel, dim3(std::min<unsigned>(256, l.slot_cap / 256)), dim3(256), 0, stream, p, gx);
        DLLM_TRY(check_launch("split sum"));
    }
    redo->tiles = p.count + 1;
    redo->tile_flags = p.tile_flags;
    redo->tile = kTile;
    return kOk;
}

}  // namespace dllm_hip
