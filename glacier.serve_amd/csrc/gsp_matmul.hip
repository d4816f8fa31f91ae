// Batched projection GEMM of the engine step, gfx950:
//   y[b][o] = sum_i W[o][i] * x[b][i]
// the product QuantKernels.MatMulBatch(type, W, x, y, inDim, outDim, batch)
// computes around the attention step (PagedTransformerRunner.cs:601-603,659).
// W holds out_dim rows of in_dim weights (the GGUF [in, out] layout) as F32,
// Q8_0 (blocks of 32 int8 with an fp16 scale d: w = d * q), or the K-quant
// super-blocks Q4_K and Q6_K (256 weights each, decoded further down).
//
// Three forms.  The tile form (matmul_tile_kernel, described further down) takes
// every product with enough work.  The fp32 form (matmul_batch_kernel, smaller
// F32 products and the quantized ones too small for the fp16 forms): every weight is exact in fp32
// (Q8_0's d * q has at most 19 significant bits), and the products run on
// v_mfma_f32_16x16x4f32 with fp32 accumulation, so no operand is rounded below
// fp32.  The fp16 forms
// (matmul_f16_kernel and the small-batch variants for at most 64 batch rows,
// described further down) run Q8_0, Q4_K and Q6_K blocks on fp16 matrix steps
// with the quants exact in fp16 and x as a scaled fp16 pair.
//
// fp32 form:
// A workgroup (four waves) owns 64 weight rows (16 per wave, MFMA M) and 64
// batch rows (four 16-column MFMA tiles, N) over a range of K, in 64-wide
// chunks.  Each chunk of x is staged once in LDS and serves all four waves;
// lane group g = lane / 16 supplies k = k0 + 16 g + s at step s of the chunk
// in both operands, so each lane reads 16 contiguous weights of its row from
// memory and 16 contiguous inputs of a batch row from LDS.  The next chunk's
// weights and x load while the current chunk computes.  When the host splits
// K over grid.z workgroups, each writes its sums to a partial buffer and a
// second kernel adds the partials in order, so results do not depend on
// timing.
#include <cfloat>
#include <type_traits>

#include "gsp_epilogue.h"
#include "gsp_internal.h"

namespace gsp {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kMmThreads = 256;
constexpr int kMmRowsWg = 64;  // weight rows per workgroup, 16 per wave

// The lane's 16 weights of row o at columns k0 + 16 g .. + 15, in two steps:
// load_raw issues the loads into registers, expand turns them into floats.
// A chunk's raw words are loaded one chunk ahead and expanded only when the
// chunk is computed, so the loads have a whole chunk of products to arrive.
template <int WT>
struct WRaw;

template <>
struct WRaw<kWeightF32> {
    f4 v[4];
};

// Q8_0: five dwords holding the lane's 16 bytes, and the dword holding its scale.
template <>
struct WRaw<kWeightQ8_0> {
    uint32_t dw[5];
    uint32_t sw;
};

__device__ __forceinline__ void load_raw(WRaw<kWeightF32>& r, const MatmulArgs& a, int o, int k0, int g) {
    const f4* p = reinterpret_cast<const f4*>(static_cast<const float*>(a.w) + (int64_t)o * a.in_dim + k0 + 16 * g);
#pragma unroll
    for (int j = 0; j < 4; ++j) r.v[j] = p[j];
}

__device__ __forceinline__ void expand(float (&w)[16], const WRaw<kWeightF32>& r, int) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * j + e] = r.v[j][e];
}

// Q8_0: a 64-wide chunk of a row is two 34-byte blocks, 68 bytes starting at a
// multiple of 4 (in_dim is a multiple of 64).  Lane group g's 16 values sit at
// bytes 2 + 16 g (g < 2, first block) or 36 + 16 (g - 2) (second block): the
// lane reads the five dwords from (byte 0, 16, 36, 52) and shifts out the
// first 2 (g < 2) or 0 bytes.  Its block's scale is the low half of dword 0
// or the high half of dword 8.  Every dword read lies inside the chunk.
__device__ __forceinline__ void load_raw(WRaw<kWeightQ8_0>& r, const MatmulArgs& a, int o, int k0, int g) {
    const int64_t row_bytes = (int64_t)(a.in_dim / 32) * 34;
    const uint32_t* cw = reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)o * row_bytes +
                                                           (int64_t)(k0 / 64) * 68);
    const int first = g < 2 ? 4 * g : 9 + 4 * (g - 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.dw[i] = cw[first + i];
    r.dw[4] = cw[g < 2 ? first + 4 : first + 3];  // only read as the high half of a 2-byte shift
    r.sw = cw[g < 2 ? 0 : 8];
}

__device__ __forceinline__ void expand(float (&w)[16], const WRaw<kWeightQ8_0>& r, int g) {
    const int shift = g < 2 ? 2 : 0;
    const _Float16 dh = __builtin_bit_cast(_Float16, (uint16_t)(g < 2 ? (r.sw & 0xFFFFu) : (r.sw >> 16)));
    const float d = (float)dh;
    const float bias = -128.0f * d;  // w = d * (u - 128) for the byte u = q ^ 0x80, exact in one fma
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t qd = __builtin_amdgcn_alignbyte(r.dw[i + 1], r.dw[i], shift) ^ 0x80808080u;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * i + e] = fmaf((float)((qd >> (8 * e)) & 0xFFu), d, bias);
    }
}

// K-quants: super-blocks of 256 weights in the public GGML layouts.  A
// 64-wide chunk lies inside one super-block; lane group g's 16 weights are
// columns 16 g .. 16 g + 15 of the chunk.  Every weight is decoded to the
// float32 value the layout defines, in its own order of operations, so the
// products stay exact fp32 products as for F32 weights.
//
// Q4_K (144 bytes: fp16 d, fp16 dmin, 12 bytes of 6-bit scales and mins, 128
// bytes of 4-bit quants): chunk p of the super-block is sub-blocks 2 p (the low
// nibbles of quant bytes 32 p .. 32 p + 31) and 2 p + 1 (their high nibbles),
// weight = (d * sc) * q - dmin * m with one rounding.  The lane reads the
// header dword, the three scale dwords and the four dwords of its 16 quant
// bytes (32 p + 16 (g % 2)); super-blocks are 4-byte aligned.
template <>
struct WRaw<kWeightQ4_K> {
    uint32_t hdr;    // d | dmin << 16
    uint32_t sc[3];  // the 12 packed scale/min bytes
    uint32_t q[4];   // the lane's 16 quant bytes
    int j;           // the lane's sub-block, 0..7
};

__device__ __forceinline__ void load_raw(WRaw<kWeightQ4_K>& r, const MatmulArgs& a, int o, int k0, int g) {
    const int64_t row_bytes = (int64_t)(a.in_dim / 256) * 144;
    const uint32_t* bw = reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)o * row_bytes +
                                                           (int64_t)(k0 / 256) * 144);
    const int p = (k0 & 255) >> 6;
    r.hdr = bw[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) r.sc[i] = bw[1 + i];
    const int qw = 4 + 8 * p + 4 * (g & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.q[i] = bw[qw + i];
    r.j = 2 * p + (g >> 1);
}

__device__ __forceinline__ uint32_t sc_byte(const uint32_t (&sc)[3], int k) {
    const uint32_t w = k < 4 ? sc[0] : k < 8 ? sc[1] : sc[2];
    return (w >> (8 * (k & 3))) & 0xFFu;
}

// The six-bit scale and min of sub-block j: bytes j and j + 4 for j < 4;
// else the nibbles of byte j + 4 with the top two bits of bytes j - 4
// (scale) and j (min).
__device__ __forceinline__ void q4k_scale_min(const uint32_t (&sc)[3], int j, uint32_t& scv, uint32_t& mv) {
    if (j < 4) {
        scv = sc_byte(sc, j) & 63u;
        mv = sc_byte(sc, j + 4) & 63u;
    } else {
        scv = (sc_byte(sc, j + 4) & 0xFu) | ((sc_byte(sc, j - 4) >> 6) << 4);
        mv = (sc_byte(sc, j + 4) >> 4) | ((sc_byte(sc, j) >> 6) << 4);
    }
}

__device__ __forceinline__ void expand(float (&w)[16], const WRaw<kWeightQ4_K>& r, int g) {
    const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.hdr & 0xFFFFu));
    const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.hdr >> 16));
    uint32_t scv, mv;
    q4k_scale_min(r.sc, r.j, scv, mv);
    const float d1 = d * (float)scv;   // exact
    const float m1 = dmin * (float)mv;  // exact
    const int shift = 4 * (g >> 1);     // low nibbles for sub-block 2 p, high for 2 p + 1
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * i + e] = fmaf(d1, (float)((r.q[i] >> (8 * e + shift)) & 0xFu), -m1);
}

// Q6_K (210 bytes: 128 bytes of the quants' low 4 bits, 64 bytes of their
// high 2 bits, 16 int8 scales, fp16 d): chunk cc of the super-block is half
// n = cc / 2, and lane group g takes quarter c = 2 (cc % 2) + g / 2, weights
// l0 .. l0 + 15 of it (l0 = 16 (g % 2)): low bytes 64 n + 32 (c % 2) + l
// (low nibble for c < 2, high for c >= 2), bits 2 c .. 2 c + 1 of high bytes
// 32 n + l, scale 8 n + l / 16 + 2 c; weight = (d * scale) * (q - 32).
// Super-blocks are only 2-byte aligned (210 bytes), so the lane reads 16-bit
// words.
template <>
struct WRaw<kWeightQ6_K> {
    uint32_t lo[4];  // the 16 low-nibble bytes (pairs of 16-bit words)
    uint32_t hi[4];  // the 16 high-bit bytes
    uint32_t sd;     // the scale byte | d << 16
    int c;           // the lane's quarter, 0..3
};

__device__ __forceinline__ void load_raw(WRaw<kWeightQ6_K>& r, const MatmulArgs& a, int o, int k0, int g) {
    const int64_t row_bytes = (int64_t)(a.in_dim / 256) * 210;
    const uint8_t* blk = static_cast<const uint8_t*>(a.w) + (int64_t)o * row_bytes + (int64_t)(k0 / 256) * 210;
    const uint16_t* bh = reinterpret_cast<const uint16_t*>(blk);
    const int cc = (k0 & 255) >> 6;
    const int n = cc >> 1;
    const int c = 2 * (cc & 1) + (g >> 1);
    const int l0 = 16 * (g & 1);
    const int lo_h = (64 * n + 32 * (c & 1) + l0) >> 1;  // in 16-bit words
    const int hi_h = (128 + 32 * n + l0) >> 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r.lo[i] = (uint32_t)bh[lo_h + 2 * i] | ((uint32_t)bh[lo_h + 2 * i + 1] << 16);
        r.hi[i] = (uint32_t)bh[hi_h + 2 * i] | ((uint32_t)bh[hi_h + 2 * i + 1] << 16);
    }
    r.sd = (uint32_t)blk[192 + 8 * n + (l0 >> 4) + 2 * c] | ((uint32_t)bh[104] << 16);
    r.c = c;
}

__device__ __forceinline__ void expand(float (&w)[16], const WRaw<kWeightQ6_K>& r, int) {
    const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.sd >> 16));
    const float ds = d * (float)(int8_t)(r.sd & 0xFFu);  // exact
    const int nib = 4 * (r.c >> 1);
    const int hb = 2 * r.c;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int q = (int)(((r.lo[i] >> (8 * e + nib)) & 0xFu) | (((r.hi[i] >> (8 * e + hb)) & 3u) << 4)) - 32;
            w[4 * i + e] = ds * (float)q;
        }
}

template <int WT>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_batch_kernel(MatmulArgs a) {
    // The chunk of x (64 batch rows x 64 k), two buffers; rows padded by one
    // 16-byte word so that the 16 lanes of one read hit distinct banks.
    __shared__ f4 xs[2][64][17];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int m = lane & 15;  // weight row of the wave's tile (A) and batch row within a tile (B)
    const int g = lane >> 4;  // K group
    const int o0 = blockIdx.x * kMmRowsWg + 16 * wave;
    const int b0 = blockIdx.y * 64;
    const int nt = min(4, (a.batch - b0 + 15) >> 4);  // batch tiles in use
    const int o = min(o0 + m, a.out_dim - 1);          // rows past out_dim load row out_dim - 1, never stored
    const int chunks = a.in_dim / 64;
    const int c_begin = blockIdx.z * a.chunks_per_split;
    const int c_end = min(chunks, c_begin + a.chunks_per_split);

    // x staging: thread tid moves batch row tid / 4, columns 16 (tid % 4) .. + 15.
    const int xr = tid >> 2;
    const int xq = tid & 3;
    const f4* xsrc = reinterpret_cast<const f4*>(a.x + (int64_t)min(b0 + xr, a.batch - 1) * a.in_dim + 16 * xq);
    f4 xreg[4];
    WRaw<WT> wraw;
    auto load_chunk = [&](int c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) xreg[j] = xsrc[16 * c + j];
        load_raw(wraw, a, o, 64 * c, g);
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[buf][xr][4 * xq + j] = xreg[j];
    };

    f4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    if (c_begin < c_end) {
        load_chunk(c_begin);
        store_x(0);
    }
    __syncthreads();
    for (int c = c_begin; c < c_end; ++c) {
        const int buf = (c - c_begin) & 1;
        float w[16];
        expand(w, wraw, g);
        const bool more = c + 1 < c_end;
        if (more) load_chunk(c + 1);  // the next chunk loads while this one computes
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t < nt) {
                float xv[16];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f4 v = xs[buf][16 * t + m][4 * g + j];
#pragma unroll
                    for (int e = 0; e < 4; ++e) xv[4 * j + e] = v[e];
                }
#pragma unroll
                for (int s2 = 0; s2 < 16; ++s2)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s2], xv[s2], acc[t], 0, 0, 0);
            }
        }
        if (more) store_x(buf ^ 1);  // the other buffer's last readers passed the previous barrier
        __syncthreads();
    }

    // Lane holds weight rows o0 + 4 g + r of batch row b0 + 16 t + m.
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int b = b0 + 16 * t + m;
        if (t >= nt || b >= a.batch) continue;
        float* dst = a.split_out ? a.split_out + ((int64_t)blockIdx.z * a.batch + b) * a.out_dim
                                 : a.y + (int64_t)b * a.out_dim;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int oo = o0 + 4 * g + r;
            if (oo < a.out_dim) dst[oo] = acc[t][r];
        }
    }
}

// ---- Q8_0 weights on the fp16 matrix cores ----------------------------------
//
// One Q8_0 block (32 weights of a row) is one K step of v_mfma_f32_16x16x32_f16:
// its int8 values are exact in fp16, and x enters as a pair x = 2^e (x_hi +
// x_lo) of fp16 halves, scaled per batch row so that the row's largest |x|
// lies in [2^12, 2^13) (the pair then carries ~22 significant bits and x_lo
// stays a normal fp16 number).  A block's two products go into a fresh
// accumulator, which the block's scale d then adds into the running sum;
// 2^e multiplies the finished row.  The products are exact in fp32, so the
// result differs from the fp32 kernel's only by summation order and the
// ~2^-22 relative truncation of x.
//
// Tile layout (M = batch rows, N = weight rows): A lane l holds
// x[batch 16 t + l % 16][k0 + 8 (l / 16) .. + 7], B lane l holds
// q[row l % 16][the same k], and the result lane holds
// y[batch 16 t + 4 (l / 16) + r][row l % 16]: the lane's own weight row, so
// its block scale is its own.

// x of one batch row as scaled fp16 pairs: one workgroup per row, four
// elements per access (in_dim is a multiple of 64, rows 16-byte aligned).
// With kSums (Q4_K weights) it also writes each 32-wide block's sum of the
// scaled x, xsum[b * (in_dim / 32) + block], for the weights' min term.
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
template <bool kSums>
__global__ __launch_bounds__(kMmThreads) void matmul_split_x_kernel(MatmulArgs a) {
    __shared__ float red[kMmThreads / 64];
    const int b = blockIdx.x;
    const int n4 = a.in_dim / 4;
    const f4* xr = reinterpret_cast<const f4*>(a.x + (int64_t)b * a.in_dim);
    // Rows of up to 16384 values stay in registers between the two passes
    // (every load issued at once, indexes clamped); longer rows are read twice.
    constexpr int kHeld = 16;
    const bool held = n4 <= kHeld * kMmThreads;
    f4 hv[kHeld];
    float mx = 0.f;
    if (held) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (kMmThreads * j < n4) hv[j] = xr[min((int)threadIdx.x + kMmThreads * j, n4 - 1)];
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (kMmThreads * j < n4)
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(hv[j][0]), fabsf(hv[j][1])), fmaxf(fabsf(hv[j][2]), fabsf(hv[j][3]))));
    } else {
#pragma unroll 4
        for (int i = threadIdx.x; i < n4; i += kMmThreads) {
            const f4 v = xr[i];
            mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // e with mx * 2^-e in [2^12, 2^13), clamped to [-126, 115] so that 2^-e
    // and 2^e stay normal floats.  The ceiling covers every finite row (ex is
    // at most 128), so no finite x overflows fp16; rows below 2^-113 keep
    // their absolute fp16 rounding only.
    int ex = 0;
    if (mx > 0.f && mx <= FLT_MAX) (void)frexpf(mx, &ex);
    const int e = mx > 0.f ? (mx <= FLT_MAX ? min(115, max(-126, ex - 13)) : 115) : 0;
    const float down = ldexpf(1.0f, -e);
    h4v* xh = reinterpret_cast<h4v*>(static_cast<_Float16*>(a.xh) + (int64_t)b * a.in_dim);
    h4v* xl = reinterpret_cast<h4v*>(static_cast<_Float16*>(a.xl) + (int64_t)b * a.in_dim);
    auto put = [&](int i, f4 raw) {
        const f4 v = raw * down;
        const h4v h = __builtin_convertvector(v, h4v);
        // An infinite element rides on its hi half alone (Inf - Inf would make
        // the lo half NaN), as it would through the fp32 form.
        f4 l = v - __builtin_convertvector(h, f4);
#pragma unroll
        for (int c = 0; c < 4; ++c) l[c] = __builtin_isinf(v[c]) ? 0.f : l[c];
        const h4v lh = __builtin_convertvector(l, h4v);
        xh[i] = h;
        xl[i] = lh;
        if constexpr (kSums) {
            // Eight consecutive threads hold a block's 32 values (n4 is a multiple
            // of 16, so a group is active or inactive as a whole): a tree over it.
            float sm = (v[0] + v[1]) + (v[2] + v[3]);
            sm += __shfl_xor(sm, 1);
            sm += __shfl_xor(sm, 2);
            sm += __shfl_xor(sm, 4);
            if ((i & 7) == 0) a.xsum[(int64_t)b * (a.in_dim / 32) + (i >> 3)] = sm;
        }
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const int i = threadIdx.x + kMmThreads * j;
            if (i < n4) put(i, hv[j]);
        }
    } else if constexpr (kSums) {
        // The block sums' lane exchanges keep this loop rolled.
        for (int i = threadIdx.x; i < n4; i += kMmThreads) put(i, xr[i]);
    } else {
#pragma unroll 4
        for (int i = threadIdx.x; i < n4; i += kMmThreads) put(i, xr[i]);
    }
    if (threadIdx.x == 0) a.xexp[b] = e;
}

// The small-batch form's pre-pass: workgroup (b, z) turns batch row b's K
// range z (the product kernel's range, chunks_per_split chunks of 64) into
// scaled fp16 pairs in the order the product kernel's A operands are read,
// tile by tile: for M tile t (batch rows 16 t ..) and chunk c, 4096 bytes as
// [block][hi, lo][lane g * 16 + m][8 halves], the halves
// x[16 t + m][64 c + 32 block + 8 g ..], so that a wave loads one operand of
// one block as 1 KB in one instruction.  Each range has an exponent of its
// own, xexp[z][b]
// (the product kernel scales each range's partial by it).  A range's largest
// |x| is at most its row's, so every element keeps at least the per-row
// form's precision.  One f4 per thread and a single load round trip: for
// Qwen2.5-7B's 3584-wide rows at 64 batch rows that is 448 workgroups of 128
// elements' worth each instead of 64 workgroups walking whole rows.
// With kSums (Q4_K weights) it also writes each 32-wide block's sum of the
// scaled x, xsum[(z * 2 chunks_per_split + block of the range) * 64 + b], for
// the weights' min term.
// kSlots f4 per thread: ranges of up to 16 kSlots chunks.
template <bool kSums, int kSlots>
__global__ __launch_bounds__(kMmThreads) void matmul_split_x_range_kernel(MatmulArgs a) {
    __shared__ float red[kMmThreads / 64];
    const int b = blockIdx.x;
    const int z = blockIdx.y;
    const int i0 = z * a.chunks_per_split * 16;  // first f4 of the range
    const int n4 = min(a.in_dim / 4, i0 + a.chunks_per_split * 16) - i0;  // host: at most kSlots * kMmThreads
    const int t = threadIdx.x;
    const f4* xr = reinterpret_cast<const f4*>(a.x + (int64_t)b * a.in_dim) + i0;
    f4 raw[kSlots];
    float mx = 0.f;
#pragma unroll
    for (int sl = 0; sl < kSlots; ++sl) {
        const int tt = t + sl * kMmThreads;
        raw[sl] = tt < n4 ? xr[tt] : f4{0.f, 0.f, 0.f, 0.f};
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(raw[sl][0]), fabsf(raw[sl][1])), fmaxf(fabsf(raw[sl][2]), fabsf(raw[sl][3]))));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // As in matmul_split_x_kernel: mx * 2^-e in [2^12, 2^13), e clamped to [-126, 115].
    int ex = 0;
    if (mx > 0.f && mx <= FLT_MAX) (void)frexpf(mx, &ex);
    const int e = mx > 0.f ? (mx <= FLT_MAX ? min(115, max(-126, ex - 13)) : 115) : 0;
#pragma unroll
    for (int sl = 0; sl < kSlots; ++sl) {
        if (sl * kMmThreads >= n4) break;  // the same for every thread
        const int tt = t + sl * kMmThreads;
        const f4 v = raw[sl] * ldexpf(1.0f, -e);
        if constexpr (kSums) {
            // Eight threads hold a block's 32 values: a tree over the group.
            float s = (v[0] + v[1]) + (v[2] + v[3]);
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) s += __shfl_xor(s, off);
            if (tt < n4 && (tt & 7) == 0) a.xsum[((int64_t)z * 2 * a.chunks_per_split + (tt >> 3)) * 64 + b] = s;
        }
        if (tt < n4) {
            const h4v h = __builtin_convertvector(v, h4v);
            f4 l = v - __builtin_convertvector(h, f4);
#pragma unroll
            for (int c = 0; c < 4; ++c) l[c] = __builtin_isinf(v[c]) ? 0.f : l[c];
            const h4v lh = __builtin_convertvector(l, h4v);
            _Float16* xt = static_cast<_Float16*>(a.xh);
            const int k = 4 * (i0 + tt);
            const int64_t tile0 = (int64_t)(b >> 4) * (a.in_dim / 64);
            const int64_t base = ((tile0 + (k >> 6)) * 2 + ((k >> 5) & 1)) * 2 * 512 +
                                 (((k >> 3) & 3) * 16 + (b & 15)) * 8 + (k & 7);
            *reinterpret_cast<h4v*>(xt + base) = h;
            *reinterpret_cast<h4v*>(xt + base + 512) = lh;
        }
    }
    if (t == 0) a.xexp[z * a.batch + b] = e;
}

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// Eight int8 (two dwords) as fp16: with u = q ^ 0x80, the half 0x6400 | u is
// 1024 + u, so subtracting 1152 leaves q exactly.  v_perm_b32 pairs each byte
// of u with a 0x64 byte from the constant operand.
__device__ __forceinline__ h8 q8_to_h8(uint32_t d0, uint32_t d1) {
    h8 r;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t u = (k ? d1 : d0) ^ 0x80808080u;
        const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);  // bytes u0, 64, u1, 64
        const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);  // bytes u2, 64, u3, 64
        const h2 a0 = __builtin_bit_cast(h2, p0) - h2{(_Float16)1152.0f, (_Float16)1152.0f};
        const h2 a1 = __builtin_bit_cast(h2, p1) - h2{(_Float16)1152.0f, (_Float16)1152.0f};
        r[4 * k + 0] = a0[0];
        r[4 * k + 1] = a0[1];
        r[4 * k + 2] = a1[0];
        r[4 * k + 3] = a1[1];
    }
    return r;
}

// Four nibbles per dword (one per byte, 0..15) as fp16: the half 0x6400 | q is
// 1024 + q, so subtracting 1024 leaves q exactly.
__device__ __forceinline__ h8 nib_to_h8(uint32_t d0, uint32_t d1) {
    h8 r;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t u = k ? d1 : d0;
        const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);  // bytes u0, 64, u1, 64
        const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);  // bytes u2, 64, u3, 64
        const h2 a0 = __builtin_bit_cast(h2, p0) - h2{(_Float16)1024.0f, (_Float16)1024.0f};
        const h2 a1 = __builtin_bit_cast(h2, p1) - h2{(_Float16)1024.0f, (_Float16)1024.0f};
        r[4 * k + 0] = a0[0];
        r[4 * k + 1] = a0[1];
        r[4 * k + 2] = a1[0];
        r[4 * k + 3] = a1[1];
    }
    return r;
}

// Four six-bit values (one per byte, 0..63) as fp16 minus 32: the half
// 0x6400 | u is 1024 + u, so subtracting 1056 leaves u - 32 exactly.
__device__ __forceinline__ void six_to_h4(uint32_t u, h2& lo, h2& hi) {
    lo = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - h2{(_Float16)1056.0f, (_Float16)1056.0f};
    hi = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - h2{(_Float16)1056.0f, (_Float16)1056.0f};
}

// The lane's raw words of one 64-wide chunk of its weight row (68 bytes at a
// multiple of 4): block 0's eight values at bytes 2 + 8 g (dwords 2g .. 2g + 2,
// shifted by 2), block 1's at 36 + 8 g (dwords 9 + 2g, 10 + 2g), and the two
// scales (low half of dword 0, high half of dword 8).  All inside the chunk.
struct Q8Raw {
    uint32_t b0[3];
    uint32_t b1[2];
    uint32_t s0, s8;
};

__device__ __forceinline__ void load_q8_raw(Q8Raw& r, const MatmulArgs& a, int o, int c, int g) {
    const int64_t row_bytes = (int64_t)(a.in_dim / 32) * 34;
    const uint32_t* cw =
        reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)o * row_bytes + (int64_t)c * 68);
#pragma unroll
    for (int i = 0; i < 3; ++i) r.b0[i] = cw[2 * g + i];
    r.b1[0] = cw[9 + 2 * g];
    r.b1[1] = cw[10 + 2 * g];
    r.s0 = cw[0];
    r.s8 = cw[8];
}

// Q4_K: the lane's words of chunk c of its weight row: the super-block head
// (d | dmin << 16 and the three scale words) and the two quant dwords at bytes
// 32 p + 8 g of the chunk's quarter p, whose low nibbles are block 0's values
// 8 g .. 8 g + 7 (sub-block 2 p) and high nibbles block 1's (sub-block 2 p + 1).
struct Q4KRaw {
    uint32_t hdr;
    uint32_t sc[3];
    uint32_t q[2];
};

__device__ __forceinline__ void load_q4k_raw(Q4KRaw& r, const MatmulArgs& a, int o, int c, int g) {
    const int64_t row_bytes = (int64_t)(a.in_dim / 256) * 144;
    const uint32_t* bw = reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)o * row_bytes +
                                                           (int64_t)(c >> 2) * 144);
    r.hdr = bw[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) r.sc[i] = bw[1 + i];
    r.q[0] = bw[4 + 8 * (c & 3) + 2 * g];
    r.q[1] = bw[5 + 8 * (c & 3) + 2 * g];
}

// Q6_K: the lane's words of chunk c of its weight row (quarters 2 e and 2 e + 1
// of half hn of the super-block, e = c % 2, hn = c % 4 / 2): the low-bit bytes
// 64 hn + 8 g .. and 64 hn + 32 + 8 g .. (nibble e), the high-bit bytes
// 32 hn + 8 g .. (bits 4 e .. 4 e + 3), the four scales 8 hn + 4 e .. and d.
// Super-blocks are 210 bytes, so these are raw buffer loads at 2-byte aligned
// offsets (gfx950 runs with unaligned buffer access), inside the super-block.
struct Q6KRaw {
    uint32_t l0[2], l1[2], h[2];
    uint32_t sc;
    uint16_t d;
};

__device__ __forceinline__ void load_q6k_raw(Q6KRaw& r, __amdgpu_buffer_rsrc_t wr, int row_off, int c, int g) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    const int hn = (c >> 1) & 1;
    const int off = row_off + (c >> 2) * 210;
    const u2 l0 = __builtin_amdgcn_raw_buffer_load_b64(wr, off + 64 * hn + 8 * g, 0, 0);
    const u2 l1 = __builtin_amdgcn_raw_buffer_load_b64(wr, off + 64 * hn + 32 + 8 * g, 0, 0);
    const u2 h = __builtin_amdgcn_raw_buffer_load_b64(wr, off + 128 + 32 * hn + 8 * g, 0, 0);
    r.l0[0] = l0[0];
    r.l0[1] = l0[1];
    r.l1[0] = l1[0];
    r.l1[1] = l1[1];
    r.h[0] = h[0];
    r.h[1] = h[1];
    r.sc = __builtin_amdgcn_raw_buffer_load_b32(wr, off + 192 + 8 * hn + 4 * (c & 1), 0, 0);
    r.d = __builtin_amdgcn_raw_buffer_load_b16(wr, off + 208, 0, 0);
}

// matmul_f16_kernel<WT>: Q8_0, Q4_K or Q6_K weights.  For Q4_K a block's values are
// its quants q (exact in fp16) and its scale d1 = d * sc, and the min term
// m1 * sum_k x_k of each block comes from the pre-pass's block sums: per chunk
// and M tile one v_mfma_f32_16x16x4f32 of the sums (A: batch rows x the
// chunk's two blocks, zero in lane groups 2-3) against the lane's m1 values
// (B), into a second accumulator subtracted before the scaling.  For Q6_K a
// block's values are q - 32 (exact in fp16) with a scale d * sc per 16: the
// block runs as two masked pairs of matrix steps (B zero outside lane groups
// 0-1 or 2-3), each half's sum scaled by its own d * sc.
template <int WT>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_f16_kernel(MatmulArgs a) {
    static_assert(WT == kWeightQ8_0 || WT == kWeightQ4_K || WT == kWeightQ6_K, "Q8_0, Q4_K or Q6_K weights");
    constexpr bool kQ4K = WT == kWeightQ4_K;
    constexpr bool kQ6K = WT == kWeightQ6_K;
    // The chunk of x as fp16 pairs: [buffer][hi, lo][64 batch rows][64 halves + 8 padding].
    __shared__ _Float16 xs[2][2][64][72];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int n = lane & 15;  // weight row within the wave's 16 (B column, result column)
    const int g = lane >> 4;
    const int o0 = blockIdx.x * kMmRowsWg + 16 * wave;
    const int b0 = blockIdx.y * 64;
    const int nt = min(4, (a.batch - b0 + 15) >> 4);
    const int o = min(o0 + n, a.out_dim - 1);
    const int chunks = a.in_dim / 64;
    const int c_begin = blockIdx.z * a.chunks_per_split;
    const int c_end = min(chunks, c_begin + a.chunks_per_split);

    // x staging: thread tid moves batch row tid / 4, halves 16 (tid % 4) .. + 15 of hi and lo.
    const int xr = tid >> 2;
    const int xq = tid & 3;
    const int64_t xoff = (int64_t)min(b0 + xr, a.batch - 1) * a.in_dim + 16 * xq;
    const u4* xh_src = reinterpret_cast<const u4*>(static_cast<const _Float16*>(a.xh) + xoff);
    const u4* xl_src = reinterpret_cast<const u4*>(static_cast<const _Float16*>(a.xl) + xoff);
    u4 xreg[4];
    std::conditional_t<kQ4K, Q4KRaw, std::conditional_t<kQ6K, Q6KRaw, Q8Raw>> wraw;
    // Q6_K: the workgroup's weight rows through one descriptor (the lane's row
    // is clamped to out_dim - 1, as for the other types, so it stays inside).
    const int q6_row_bytes = (a.in_dim / 256) * 210;
    const __amdgpu_buffer_rsrc_t q6w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)blockIdx.x * kMmRowsWg * q6_row_bytes),
        (short)0, min(kMmRowsWg, a.out_dim - (int)blockIdx.x * kMmRowsWg) * q6_row_bytes, 0x00020000);
    float xsr[4];  // Q4_K: block sums of the lane's A operands for the min term
    auto load_chunk = [&](int c) {
        xreg[0] = xh_src[8 * c];
        xreg[1] = xh_src[8 * c + 1];
        xreg[2] = xl_src[8 * c];
        xreg[3] = xl_src[8 * c + 1];
        if constexpr (kQ4K) {
            load_q4k_raw(wraw, a, o, c, g);
            // Lane (n, g < 2): batch row b0 + 16 t + n, block 2 c + g.
#pragma unroll
            for (int t = 0; t < 4; ++t)
                xsr[t] = g < 2 && t < nt ? a.xsum[(int64_t)min(b0 + 16 * t + n, a.batch - 1) * (a.in_dim / 32) + 2 * c + g]
                                         : 0.f;
        } else if constexpr (kQ6K) {
            load_q6k_raw(wraw, q6w, (o - (int)blockIdx.x * kMmRowsWg) * q6_row_bytes, c, g);
        } else {
            load_q8_raw(wraw, a, o, c, g);
        }
    };
    auto store_x = [&](int buf) {
        *reinterpret_cast<u4*>(&xs[buf][0][xr][16 * xq]) = xreg[0];
        *reinterpret_cast<u4*>(&xs[buf][0][xr][16 * xq + 8]) = xreg[1];
        *reinterpret_cast<u4*>(&xs[buf][1][xr][16 * xq]) = xreg[2];
        *reinterpret_cast<u4*>(&xs[buf][1][xr][16 * xq + 8]) = xreg[3];
    };

    f4 acc[4], accm[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = accm[t] = f4{0.f, 0.f, 0.f, 0.f};
    if (c_begin < c_end) {
        load_chunk(c_begin);
        store_x(0);
    }
    __syncthreads();
    for (int c = c_begin; c < c_end; ++c) {
        const int buf = (c - c_begin) & 1;
        // This chunk's two blocks of the lane's row: values and scales.
        h8 wq0, wq1;
        float d0, d1, mb = 0.f, xsc[4];
        float e0 = 0.f, e1 = 0.f;  // Q6_K: the blocks' scales for k >= 16 (d0, d1 for k < 16)
        if constexpr (kQ6K) {
            const int e = c & 1;
            const float d = (float)__builtin_bit_cast(_Float16, wraw.d);
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) {
                const uint32_t u0 = ((wraw.l0[t2] >> (4 * e)) & 0x0F0F0F0Fu) | (((wraw.h[t2] >> (4 * e)) & 0x03030303u) << 4);
                const uint32_t u1 =
                    ((wraw.l1[t2] >> (4 * e)) & 0x0F0F0F0Fu) | (((wraw.h[t2] >> (4 * e + 2)) & 0x03030303u) << 4);
                h2 lo, hi;
                six_to_h4(u0, lo, hi);
                wq0[4 * t2 + 0] = lo[0];
                wq0[4 * t2 + 1] = lo[1];
                wq0[4 * t2 + 2] = hi[0];
                wq0[4 * t2 + 3] = hi[1];
                six_to_h4(u1, lo, hi);
                wq1[4 * t2 + 0] = lo[0];
                wq1[4 * t2 + 1] = lo[1];
                wq1[4 * t2 + 2] = hi[0];
                wq1[4 * t2 + 3] = hi[1];
            }
            d0 = d * (float)(int8_t)(wraw.sc & 0xFFu);  // exact
            e0 = d * (float)(int8_t)((wraw.sc >> 8) & 0xFFu);
            d1 = d * (float)(int8_t)((wraw.sc >> 16) & 0xFFu);
            e1 = d * (float)(int8_t)(wraw.sc >> 24);
        } else if constexpr (kQ4K) {
            const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(wraw.hdr & 0xFFFFu));
            const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(wraw.hdr >> 16));
            uint32_t sc0, m0, sc1, m1;
            q4k_scale_min(wraw.sc, 2 * (c & 3), sc0, m0);
            q4k_scale_min(wraw.sc, 2 * (c & 3) + 1, sc1, m1);
            d0 = d * (float)sc0;  // exact
            d1 = d * (float)sc1;
            mb = g == 0 ? dmin * (float)m0 : g == 1 ? dmin * (float)m1 : 0.f;  // B of the min term
            wq0 = nib_to_h8(wraw.q[0] & 0x0F0F0F0Fu, wraw.q[1] & 0x0F0F0F0Fu);
            wq1 = nib_to_h8((wraw.q[0] >> 4) & 0x0F0F0F0Fu, (wraw.q[1] >> 4) & 0x0F0F0F0Fu);
#pragma unroll
            for (int t = 0; t < 4; ++t) xsc[t] = xsr[t];
        } else {
            wq0 = q8_to_h8(__builtin_amdgcn_alignbyte(wraw.b0[1], wraw.b0[0], 2),
                           __builtin_amdgcn_alignbyte(wraw.b0[2], wraw.b0[1], 2));
            wq1 = q8_to_h8(wraw.b1[0], wraw.b1[1]);
            d0 = (float)__builtin_bit_cast(_Float16, (uint16_t)(wraw.s0 & 0xFFFFu));
            d1 = (float)__builtin_bit_cast(_Float16, (uint16_t)(wraw.s8 >> 16));
        }
        const bool more = c + 1 < c_end;
        if (more) load_chunk(c + 1);  // the next chunk loads while this one computes
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t < nt) {
                const int row = 16 * t + n;  // A row: batch row of this lane
#pragma unroll
                for (int blk = 0; blk < 2; ++blk) {
                    const h8 ah = *reinterpret_cast<const h8*>(&xs[buf][0][row][32 * blk + 8 * g]);
                    const h8 al = *reinterpret_cast<const h8*>(&xs[buf][1][row][32 * blk + 8 * g]);
                    const h8 wq = blk ? wq1 : wq0;
                    const float d = blk ? d1 : d0;
                    if constexpr (kQ6K) {
                        const h8 wa = g < 2 ? wq : h8{};  // k < 16 of the block
                        const h8 wb = g < 2 ? h8{} : wq;
                        f4 pa = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, wa, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        pa = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, wa, pa, 0, 0, 0);
                        f4 pb = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, wb, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        pb = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, wb, pb, 0, 0, 0);
                        const float de = blk ? e1 : e0;
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[t][r] = fmaf(de, pb[r], fmaf(d, pa[r], acc[t][r]));
                    } else {
                        f4 part = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, wq, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        part = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, wq, part, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[t][r] = fmaf(d, part[r], acc[t][r]);
                    }
                }
                if constexpr (kQ4K) accm[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xsc[t], mb, accm[t], 0, 0, 0);
            }
        }
        if (more) store_x(buf ^ 1);  // the other buffer's last readers passed the previous barrier
        __syncthreads();
    }

    // Lane holds batch rows b0 + 16 t + 4 g + r of weight row o0 + n.
    const int oo = o0 + n;
    if (oo >= a.out_dim) return;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int b = b0 + 16 * t + 4 * g + r;
            if (t >= nt || b >= a.batch) continue;
            const float v = ldexpf(kQ4K ? acc[t][r] - accm[t][r] : acc[t][r], a.xexp[b]);
            float* dst = a.split_out ? a.split_out + ((int64_t)blockIdx.z * a.batch + b) * a.out_dim
                                     : a.y + (int64_t)b * a.out_dim;
            dst[oo] = v;
        }
    }
}

// ---- Q8_0 weights, batches of up to 64 rows ---------------------------------
//
// matmul_q8_f16_small_kernel<NT, CH, kPasses> is the fp16 form for batches of
// at most 64 rows (NT M tiles of 16), laid out so that nothing waits in line:
//   - x comes from the pre-pass in tile order (matmul_split_x_range_kernel):
//     a wave loads the A operands of its M tile straight into registers, one
//     KB per instruction, every chunk of its range at once, with no LDS and no
//     barrier between chunks;
//   - the workgroup's 64 weight rows over its range of at most CH chunks are
//     expanded to fp16 once, into LDS, with their block scales as floats;
//   - a longer range (kPasses: the merge holds too few ranges for chunks of
//     CH, as for an 18944-wide K at 64 rows) is walked CH chunks at a time
//     through the same LDS, with a barrier between passes;
//   - wave w takes M tile w NT / 4 and NT of the four N tiles (16 weight rows
//     each), so every staged operand serves several matrix steps;
//   - two workgroups fit on a CU;
//   - with K split over grid.z, each workgroup stores its tile coherently,
//     waits for the stores and counts itself on the output tile's counter; the
//     last one adds the ranges' tiles in z order (its own from registers),
//     every load issued before the first add, and resets the counter.  No
//     reduce launch, and results do not depend on timing.
constexpr int kSmMaxPartials = 32;  // K ranges x tiles per lane the merge holds at most
constexpr int kSmRowHalves = 8 * 64 + 8;  // an LDS weight row: 8 chunks of 64 halves, +16 bytes

// The small forms' shared steps.  Wave w of a workgroup takes M tile
// mt = w NT / 4 (batch rows 16 mt ..) against N tiles nt0 .. nt0 + NT - 1
// (weight rows 64 blockIdx.x + 16 nt0 ..); lane (g = lane / 16, n = lane % 16).

// A operands of the wave's M tile, every chunk of the range at once:
// [chunk][block][hi, lo], one KB per load from the pre-pass's tile order.
template <int CH>
__device__ __forceinline__ void small_load_x(h8 (&ax)[CH][2][2], const MatmulArgs& a, int mt, int chunks, int c_begin,
                                             int nc, int lane) {
    const h8* xt = reinterpret_cast<const h8*>(static_cast<const _Float16*>(a.xh)) +
                   ((int64_t)mt * chunks + c_begin) * 256 + lane;
#pragma unroll
    for (int i = 0; i < CH; ++i)
        if (i < nc)
#pragma unroll
            for (int blk = 0; blk < 2; ++blk)
#pragma unroll
                for (int part = 0; part < 2; ++part) ax[i][blk][part] = xt[i * 256 + (blk * 2 + part) * 64];
}

// One pass's products: per block, hi and lo into a fresh accumulator, which
// the block's scale (wd: [weight row][2 chunk + block]) adds into acc.
template <int NT, int CH>
__device__ __forceinline__ void small_products(f4 (&acc)[NT], const h8 (&ax)[CH][2][2], const _Float16* wh,
                                               const float (*wd)[2 * CH + 1], int nc, int nt0, int n, int g) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if (i < nc) {
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int r = 16 * (nt0 + j) + n;  // B column: the lane's weight row
                    const h8 wq = *reinterpret_cast<const h8*>(&wh[r * kSmRowHalves + i * 64 + blk * 32 + g * 8]);
                    const float d = wd[r][2 * i + blk];
                    f4 part = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][0], wq, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    part = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][1], wq, part, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[j][q] = fmaf(d, part[q], acc[j][q]);
                }
            }
        }
    }
}

// The tile's end: scale by 2^xexp of each batch row's K range, then either
// store y (one range) or store the partial coherently, count the tile and, in
// the last workgroup of the tile, add the ranges in z order (every load issued
// before the first add) and reset the counter.
template <int NT>
__device__ __forceinline__ void small_finish(const MatmulArgs& a, const f4 (&acc)[NT], int mt, int nt0, int n, int g,
                                             int tid, int& last) {
    // Lane holds batch rows 16 mt + 4 g + q of weight rows 64 x + 16 (nt0 + j) + n,
    // scaled by 2^-xexp of the batch row's K range.
    float v[NT][4];
    int bq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bq[q] = 16 * mt + 4 * g + q;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = a.xexp[blockIdx.z * a.batch + min(bq[q], a.batch - 1)];
#pragma unroll
        for (int j = 0; j < NT; ++j) v[j][q] = ldexpf(acc[j][q], e);
    }
    const int obase = blockIdx.x * kMmRowsWg + 16 * nt0 + n;
    if (a.splits == 1) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (obase + 16 * j < a.out_dim && bq[q] < a.batch) a.y[(int64_t)bq[q] * a.out_dim + obase + 16 * j] = v[j][q];
        return;
    }
    const int z = blockIdx.z;
    const int64_t plane = (int64_t)a.batch * a.out_dim;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (obase + 16 * j < a.out_dim && bq[q] < a.batch)
                coherent_store(a.split_out + z * plane + (int64_t)bq[q] * a.out_dim + obase + 16 * j, v[j][q]);
    wait_vm_complete();
    __syncthreads();
    if (tid == 0)
        last = __hip_atomic_fetch_add(a.counters + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               a.splits - 1;
    __syncthreads();
    if (!last) return;
    constexpr int kZ = kSmMaxPartials / NT;
    float p[NT][4][kZ];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float* pb = a.split_out + (int64_t)min(bq[q], a.batch - 1) * a.out_dim + min(obase + 16 * j, a.out_dim - 1);
#pragma unroll
            for (int zz = 0; zz < kZ; ++zz) p[j][q][zz] = coherent_load(pb + min(zz, a.splits - 1) * plane);
        }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float s = z == 0 ? v[j][q] : p[j][q][0];
#pragma unroll
            for (int zz = 1; zz < kZ; ++zz)
                if (zz < a.splits) s += zz == z ? v[j][q] : p[j][q][zz];
            if (obase + 16 * j < a.out_dim && bq[q] < a.batch) a.y[(int64_t)bq[q] * a.out_dim + obase + 16 * j] = s;
        }
    if (tid == 0) __hip_atomic_store(a.counters + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int NT, int CH, bool kPasses>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_q8_f16_small_kernel(MatmulArgs a) {
    static_assert(CH <= 8, "an LDS weight row holds 8 chunks");
    __shared__ _Float16 wh[kMmRowsWg * kSmRowHalves];  // [weight row][chunk][64 halves]
    __shared__ float wd[kMmRowsWg][2 * CH + 1];        // block scales [weight row][2 chunk + block]
    __shared__ int last;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int n = lane & 15;
    const int g = lane >> 4;
    const int chunks = a.in_dim / 64;
    const int c_begin = blockIdx.z * a.chunks_per_split;
    const int nc_range = min(chunks, c_begin + a.chunks_per_split) - c_begin;  // 1..CH, or more with kPasses (host)
    constexpr int kWavesPerM = 4 / NT;
    const int mt = wave / kWavesPerM;           // the wave's M tile
    const int nt0 = (wave % kWavesPerM) * NT;   // its first N tile

    f4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
    // With kPasses the range is walked CH chunks at a time through the same LDS.
    for (int c0 = 0;;) {
        const int nc = kPasses ? min(CH, nc_range - c0) : nc_range;
        const int cb = c_begin + c0;
        h8 ax[CH][2][2];
        small_load_x<CH>(ax, a, mt, chunks, cb, nc, lane);

        // Weights to fp16: unit u = 64 r + 8 i + 4 block + gg (row r, chunk i, lane
        // group gg) is eight values; thread tid takes units tid + 256 k, that is
        // one fixed (chunk, block, lane group) of rows tid / 64 + 4 k.  A wave's
        // units are one row's chunks, so its loads cover whole 68-byte windows.
        // Every unit's three dwords load first, one 12-byte raw buffer load each
        // (dword aligned; one lane offset per thread): block 0's values sit at
        // dwords 2 gg .. 2 gg + 2 shifted by 2 bytes, block 1's at 9 + 2 gg,
        // 10 + 2 gg (the load covers 8 + 2 gg .. 10 + 2 gg), and the scale is the
        // low half of dword 0 or the high half of dword 8, both in lane group 0's
        // load.
        // Units of chunks past the range load the range's last chunk and store
        // nothing; rows past out_dim read as zero (past the buffer's end).
        {
            constexpr int kU = (kMmRowsWg * 64) / kMmThreads;
            const int row_bytes = chunks * 68;
            const int rows_here = min(kMmRowsWg, a.out_dim - (int)blockIdx.x * kMmRowsWg);
            typedef uint32_t u3 __attribute__((ext_vector_type(3)));
            const int r0 = tid >> 6;
            const int i = (tid >> 3) & 7;
            const int blk = (tid >> 2) & 1;
            const int gg = tid & 3;
            const int s0 = blk ? 8 + 2 * gg : 2 * gg;  // the unit's three dwords: s0 .. s0 + 2, inside the chunk
            const int voff = r0 * row_bytes + (cb + min(i, nc - 1)) * 68 + 4 * s0;
            u3 wdw[kU];
#pragma unroll
            for (int k = 0; k < kU; ++k) {
                // Rows r0 + 4 k: the row step goes into the descriptor (base and
                // record count), so one lane offset serves every load and the
                // range check, which covers the lane offset, still stops at out_dim.
                const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<uint8_t*>(static_cast<const uint8_t*>(a.w) + ((int64_t)blockIdx.x * kMmRowsWg + 4 * k) * row_bytes),
                    (short)0, max(0, rows_here - 4 * k) * row_bytes, 0x00020000);
                wdw[k] = __builtin_amdgcn_raw_buffer_load_b96(wr, voff, 0, 0);
            }
            const int sh = blk ? 0 : 2;
            _Float16* wdst = &wh[r0 * kSmRowHalves + i * 64 + blk * 32 + gg * 8];
            float* ddst = &wd[r0][2 * i + blk];
            if (i < nc) {
#pragma unroll
                for (int k = 0; k < kU; ++k) {
                    const uint32_t d0 = blk ? wdw[k][1] : wdw[k][0];
                    const uint32_t d1 = blk ? wdw[k][2] : wdw[k][1];
                    const h8 q = q8_to_h8(__builtin_amdgcn_alignbyte(d1, d0, sh), __builtin_amdgcn_alignbyte(wdw[k][2], d1, sh));
                    *reinterpret_cast<h8*>(wdst + 4 * k * kSmRowHalves) = q;
                    // Lane group 0 holds the block's scale: dword 0 (low half) or 8 (high half).
                    const uint32_t sw = blk ? wdw[k][0] >> 16 : wdw[k][0];
                    if (gg == 0) ddst[4 * k * (2 * CH + 1)] = (float)__builtin_bit_cast(_Float16, (uint16_t)(sw & 0xFFFFu));
                }
            }
        }
        __syncthreads();

        small_products<NT, CH>(acc, ax, wh, wd, nc, nt0, n, g);
        if constexpr (!kPasses) break;
        c0 += CH;
        if (c0 >= nc_range) break;
        __syncthreads();  // every wave is done with this pass's weights
    }
    small_finish<NT>(a, acc, mt, nt0, n, g, tid, last);
}

// ---- Q4_K weights, batches of up to 64 rows ---------------------------------
//
// matmul_q4k_f16_small_kernel<NT, kPasses> is the Q8_0 small form with Q4_K weights.
// A weight is w = d1 q - m1 per 32-wide sub-block (d1 = d * sc and
// m1 = dmin * m, both exact in fp32; q = 0..15, exact in fp16), so
//   y[b][o] = sum over blocks of  d1 * sum_k q_k x_k  -  m1 * sum_k x_k.
// The first term is the Q8_0 form's: the quants go to LDS as fp16 and each
// block is one hi/lo pair of 16x16x32 fp16 matrix steps scaled by d1.  The
// second needs only the blocks' sums of x, which the pre-pass writes (of the
// scaled x, so both terms carry the range's 2^-xexp): per four blocks one
// v_mfma_f32_16x16x4f32 of the x sums (A: batch rows x blocks) against the
// m1 values (B: blocks x weight rows) into a second accumulator, subtracted
// before the scaling.  A chunk of 64 weights is one quarter p of a 256-weight
// super-block: sub-blocks 2 p (low nibbles of quant bytes 32 p ..) and 2 p + 1
// (their high nibbles), so ranges need not start on a super-block.
template <int NT, bool kPasses>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_q4k_f16_small_kernel(MatmulArgs a) {
    constexpr int CH = 8;
    __shared__ _Float16 wh[kMmRowsWg * kSmRowHalves];  // quants [weight row][chunk][64 halves]
    __shared__ float wd[kMmRowsWg][2 * CH + 1];        // d1 = d * sc [weight row][2 chunk + block]
    __shared__ float wm[kMmRowsWg][2 * CH + 1];        // m1 = dmin * m, the same way
    __shared__ __attribute__((aligned(16))) float xs[2 * CH][64];  // block sums of scaled x [block][batch row]
    __shared__ int last;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int n = lane & 15;
    const int g = lane >> 4;
    const int chunks = a.in_dim / 64;
    const int c_begin = blockIdx.z * a.chunks_per_split;
    const int nc_range = min(chunks, c_begin + a.chunks_per_split) - c_begin;  // 1..CH, or more with kPasses (host)
    constexpr int kWavesPerM = 4 / NT;
    const int mt = wave / kWavesPerM;
    const int nt0 = (wave % kWavesPerM) * NT;

    f4 acc[NT], accm[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = accm[j] = f4{0.f, 0.f, 0.f, 0.f};
    // With kPasses the range is walked CH chunks at a time through the same LDS.
    for (int c0 = 0;;) {
        const int nc = kPasses ? min(CH, nc_range - c0) : nc_range;
        const int cb = c_begin + c0;
        h8 ax[CH][2][2];
        small_load_x<CH>(ax, a, mt, chunks, cb, nc, lane);

        // Weights: unit (row r, chunk i) is one super-block quarter, 64 quants in 32
        // bytes plus the super-block's 16-byte head (d, dmin, the 12 scale bytes);
        // thread tid takes chunk tid % 8 of rows tid / 8 and tid / 8 + 32, three
        // 16-byte raw buffer loads each (super-blocks are 144 bytes, so every load
        // is dword aligned), all issued before the first is used.  Units of chunks
        // past the range load the range's last chunk and store zero scales; rows
        // past out_dim read as zero (past the buffer's end).
        {
            const int row_bytes = (a.in_dim / 256) * 144;
            const int rows_here = min(kMmRowsWg, a.out_dim - (int)blockIdx.x * kMmRowsWg);
            const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<uint8_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)blockIdx.x * kMmRowsWg * row_bytes),
                (short)0, rows_here * row_bytes, 0x00020000);
            const int i = tid & 7;
            const int r0 = tid >> 3;
            const int c = cb + min(i, nc - 1);
            const int p = c & 3;
            const int voff = r0 * row_bytes + (c >> 2) * 144;
            u4 hd[2], qa[2], qb[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int off = voff + 32 * k * row_bytes;
                hd[k] = __builtin_amdgcn_raw_buffer_load_b128(wr, off, 0, 0);
                qa[k] = __builtin_amdgcn_raw_buffer_load_b128(wr, off + 16 + 32 * p, 0, 0);
                qb[k] = __builtin_amdgcn_raw_buffer_load_b128(wr, off + 32 + 32 * p, 0, 0);
            }
            // The range's block sums, loaded after the weights (the memory counter
            // drains in order, so the weights need not wait for them) and stored
            // after the expansion: thread tid takes block tid / 16, batch rows
            // 4 (tid % 16) .. + 3; blocks past the range and rows past the batch are 0.
            const int sblk = tid >> 4;
            const int b4 = 4 * (tid & 15);
            f4 xsv = f4{0.f, 0.f, 0.f, 0.f};
            if (sblk < 2 * nc)
                xsv = *reinterpret_cast<const f4*>(a.xsum + ((int64_t)blockIdx.z * 2 * a.chunks_per_split + 2 * c0 + sblk) * 64 + b4);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int r = r0 + 32 * k;
                float d1[2] = {0.f, 0.f}, m1[2] = {0.f, 0.f};
                if (i < nc) {
                    const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[k][0] & 0xFFFFu));
                    const float dmin = (float)__builtin_bit_cast(_Float16, (uint16_t)(hd[k][0] >> 16));
                    const uint32_t sc[3] = {hd[k][1], hd[k][2], hd[k][3]};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        uint32_t scv, mv;
                        q4k_scale_min(sc, 2 * p + h, scv, mv);
                        d1[h] = d * (float)scv;   // exact
                        m1[h] = dmin * (float)mv;  // exact
                    }
                    const uint32_t q[8] = {qa[k][0], qa[k][1], qa[k][2], qa[k][3], qb[k][0], qb[k][1], qb[k][2], qb[k][3]};
                    _Float16* dst = &wh[r * kSmRowHalves + i * 64];
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        *reinterpret_cast<h8*>(dst + 8 * s) = nib_to_h8(q[2 * s] & 0x0F0F0F0Fu, q[2 * s + 1] & 0x0F0F0F0Fu);
                        *reinterpret_cast<h8*>(dst + 32 + 8 * s) =
                            nib_to_h8((q[2 * s] >> 4) & 0x0F0F0F0Fu, (q[2 * s + 1] >> 4) & 0x0F0F0F0Fu);
                    }
                }
                wd[r][2 * i] = d1[0];
                wd[r][2 * i + 1] = d1[1];
                wm[r][2 * i] = m1[0];
                wm[r][2 * i + 1] = m1[1];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (b4 + c >= a.batch) xsv[c] = 0.f;
            *reinterpret_cast<f4*>(&xs[sblk][b4]) = xsv;
        }
        __syncthreads();

        small_products<NT, CH>(acc, ax, wh, wd, nc, nt0, n, g);
        // The min term, four blocks per matrix step: lane (g, n) supplies block
        // 4 s + g of batch row 16 mt + n (A) and of weight row 16 (nt0 + j) + n (B).
#pragma unroll
        for (int s = 0; s < CH / 2; ++s) {
            if (2 * s < nc) {
                const float xa = xs[4 * s + g][16 * mt + n];
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    accm[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, wm[16 * (nt0 + j) + n][4 * s + g], accm[j], 0, 0, 0);
            }
        }
        if constexpr (!kPasses) break;
        c0 += CH;
        if (c0 >= nc_range) break;
        __syncthreads();  // every wave is done with this pass's weights and sums
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] -= accm[j];
    small_finish<NT>(a, acc, mt, nt0, n, g, tid, last);
}

// ---- Q6_K weights, batches of up to 64 rows ---------------------------------
//
// matmul_q6k_f16_small_kernel<NT, kPasses> is the Q8_0 small form with Q6_K
// weights.  A weight is w = (d * sc) * (q - 32) with the int8 scale sc per 16
// weights: q - 32 is exact in fp16 and d * sc exact in fp32, but the scale
// changes inside a 32-wide matrix step.  So each block runs as two masked
// pairs of 16x16x32 fp16 steps (B operand zero outside the lanes of one
// 16-wide half: lane groups 0-1 hold k < 16, 2-3 the rest), each half's sum
// scaled by its own d * sc.  The unit of staging is one 128-weight half n of a
// super-block (chunks 2 n' and 2 n' + 1 of the range, so ranges start on even
// chunks): quant bytes 64 n .. (low 4 bits, the chunk's nibble), high-bit
// bytes 128 + 32 n .., scales 192 + 8 n .. and d at 208.  Super-blocks are
// 210 bytes, so the loads are only 2-byte aligned; gfx950 runs with unaligned
// buffer access, and every load stays inside its super-block.
template <int NT, int CH>
__device__ __forceinline__ void small_products_q6k(f4 (&acc)[NT], const h8 (&ax)[CH][2][2], const _Float16* wh,
                                                   const float (*ws)[4 * CH + 1], int nc, int nt0, int n, int g) {
    const h8 zero = h8{};
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if (i < nc) {
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int r = 16 * (nt0 + j) + n;
                    const h8 wq = *reinterpret_cast<const h8*>(&wh[r * kSmRowHalves + i * 64 + blk * 32 + g * 8]);
                    const h8 wa = g < 2 ? wq : zero;  // k < 16: the block's first scale
                    const h8 wb = g < 2 ? zero : wq;
                    const float sa = ws[r][4 * i + 2 * blk];
                    const float sb = ws[r][4 * i + 2 * blk + 1];
                    f4 pa = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][0], wa, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    pa = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][1], wa, pa, 0, 0, 0);
                    f4 pb = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][0], wb, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    pb = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[i][blk][1], wb, pb, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[j][q] = fmaf(sb, pb[q], fmaf(sa, pa[q], acc[j][q]));
                }
            }
        }
    }
}

template <int NT, bool kPasses>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_q6k_f16_small_kernel(MatmulArgs a) {
    constexpr int CH = 8;
    __shared__ _Float16 wh[kMmRowsWg * kSmRowHalves];  // q - 32 [weight row][chunk][64 halves]
    __shared__ float ws[kMmRowsWg][4 * CH + 1];        // d * sc [weight row][4 chunk + 16-wide part]
    __shared__ int last;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int n = lane & 15;
    const int g = lane >> 4;
    const int chunks = a.in_dim / 64;
    const int c_begin = blockIdx.z * a.chunks_per_split;  // even (host)
    const int nc_range = min(chunks, c_begin + a.chunks_per_split) - c_begin;  // 1..CH, or more with kPasses (host)
    constexpr int kWavesPerM = 4 / NT;
    const int mt = wave / kWavesPerM;
    const int nt0 = (wave % kWavesPerM) * NT;

    // Staging: thread tid takes row tid / 4 and the range's half tid % 4 (its
    // chunks 2 (tid % 4) and 2 (tid % 4) + 1); a wave's loads cover 16 rows.
    const int row_bytes = (a.in_dim / 256) * 210;
    const int rows_here = min(kMmRowsWg, a.out_dim - (int)blockIdx.x * kMmRowsWg);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(static_cast<const uint8_t*>(a.w) + (int64_t)blockIdx.x * kMmRowsWg * row_bytes), (short)0,
        rows_here * row_bytes, 0x00020000);
    const int r = tid >> 2;
    const int hh = tid & 3;

    f4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0;;) {
        const int nc = kPasses ? min(CH, nc_range - c0) : nc_range;
        const int cb = c_begin + c0;
        h8 ax[CH][2][2];
        small_load_x<CH>(ax, a, mt, chunks, cb, nc, lane);
        {
            // The unit's half of the super-block (the range's last when past it).
            const int hl = min(2 * hh, nc - 1) >> 1;
            const int half = (cb >> 1) + hl;
            const int hn = half & 1;
            const int off = r * row_bytes + (half >> 1) * 210;
            u4 ql[4], qh[2];
#pragma unroll
            for (int t = 0; t < 4; ++t) ql[t] = __builtin_amdgcn_raw_buffer_load_b128(wr, off + 64 * hn + 16 * t, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) qh[t] = __builtin_amdgcn_raw_buffer_load_b128(wr, off + 128 + 32 * hn + 16 * t, 0, 0);
            typedef uint32_t u2 __attribute__((ext_vector_type(2)));
            const u2 sc = __builtin_amdgcn_raw_buffer_load_b64(wr, off + 192 + 8 * hn, 0, 0);
            const uint16_t dh = __builtin_amdgcn_raw_buffer_load_b16(wr, off + 208, 0, 0);
            const float d = (float)__builtin_bit_cast(_Float16, dh);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int i = 2 * hh + e;  // the chunk in this pass
                if (i < nc) {
                    _Float16* dst = &wh[r * kSmRowHalves + i * 64];
#pragma unroll
                    for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                        for (int s = 0; s < 4; ++s) {
                            h8 v;
#pragma unroll
                            for (int t2 = 0; t2 < 2; ++t2) {
                                const int t = 2 * s + t2;  // dword of the block: its weights 4 t .. 4 t + 3
                                const uint32_t qlw = ql[(8 * blk + t) >> 2][(8 * blk + t) & 3];
                                const uint32_t qhw = qh[t >> 2][t & 3];
                                const uint32_t u = ((qlw >> (4 * e)) & 0x0F0F0F0Fu) |
                                                   (((qhw >> (4 * e + 2 * blk)) & 0x03030303u) << 4);
                                h2 lo, hi;
                                six_to_h4(u, lo, hi);
                                v[4 * t2 + 0] = lo[0];
                                v[4 * t2 + 1] = lo[1];
                                v[4 * t2 + 2] = hi[0];
                                v[4 * t2 + 3] = hi[1];
                            }
                            *reinterpret_cast<h8*>(dst + blk * 32 + 8 * s) = v;
                        }
                    }
                    // Scales 8 hn + 4 e + 2 blk + part: byte 2 blk + part of scale dword e.
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        ws[r][4 * i + p] = d * (float)(int8_t)((sc[e] >> (8 * p)) & 0xFFu);  // exact
                }
            }
        }
        __syncthreads();
        small_products_q6k<NT, CH>(acc, ax, wh, ws, nc, nt0, n, g);
        if constexpr (!kPasses) break;
        c0 += CH;
        if (c0 >= nc_range) break;
        __syncthreads();  // every wave is done with this pass's weights
    }
    small_finish<NT>(a, acc, mt, nt0, n, g, tid, last);
}

// ---- The tile form: products with enough work to fill the chip -----------------
//
// matmul_tile_kernel<WT>.  matmul_f16_kernel and matmul_batch_kernel expand (or
// load) a weight for every 64 rows x 16 weight rows of a wave and read each x
// operand for one matrix step; instruction issue and LDS, not the matrix cores,
// bound them.  Here a workgroup owns 64 batch rows (four M tiles of 16) and 128
// weight rows, wave w the two N tiles (32 weight rows) from 32 w: an x operand
// staged in LDS serves all four waves and two N tiles, and a wave expands its
// own rows' words to fp16 operands in registers once per chunk of 64 k and uses
// each for four M tiles.  Measured at 1024 rows of 4096 x 4096 (us): Q8_0 177 ->
// 107, Q4_K 185 -> 101, Q6_K 194 -> 136, F32 279 -> 168, about 700 TFLOP/s of
// fp16 matrix steps.  Matrix cores busy 22 to 36%, vector issue 35 to 41%, waves
// waiting on memory or barriers 26 to 28%, but 45% for Q6_K, whose loop over four M
// tiles reloads spilled registers (a chunk of Q6_K is 48 matrix steps and 130 vector
// instructions a wave).
//
// x comes from matmul_split_x_tile_kernel as scaled fp16 pairs in the order the
// operands are read, so a chunk of the workgroup's 64 rows is 16 KB in one
// piece and goes to LDS with direct loads, a ring of four chunks with one barrier each.
//
// The k order inside a chunk is free as long as both operands agree, so each
// weight type takes the order in which a lane's words are contiguous (KOrder):
//   Q8_0: chunk c, block blk, lane group g: k = 64 c + 32 blk + 8 g ..; the
//     block's int8 values are exact in fp16, its sum goes to a fresh
//     accumulator that its scale adds to the running one.
//   Q4_K: lane group g owns quarter g of the super-block (sub-blocks 2 g and
//     2 g + 1, 32 contiguous quant bytes).  sc * (q - 8) is exact in fp16, so
//     only d remains outside, one fma per chunk.  The min term dmin m - 8 d sc
//     is two matrix steps per super-block: the 8 sub-block sums of x, each in
//     three halves that hold its fp32 value (from the pre-pass, times 2^-6),
//     against the 6-bit mins and scales.
//   Q6_K: lane group g owns l = 16 (g % 2) .. + 15 of each quarter of half
//     g / 2.  m = sc * (q - 32), at most 4096, takes two halves: its fp16
//     rounding and the rest (0 or +-1), three matrix steps instead of the four
//     that scaling each 16 weights apart takes.
//   F32: as Q8_0, but a lane's eight values are k = 32 blk + 4 g .. + 3 and 16
//     further on, so that one load instruction covers 64 contiguous bytes of
//     each row.  They enter as an fp16 pair scaled by the row's largest |w| of
//     the chunk (2^e, applied with the chunk's sum).  A pair keeps 22 bits of an
//     element, or 2^-38 of the scale's largest where that is more, and the lo x
//     lo product (at most 2^-22, typically 2^-25 of the term) is left out;
//     operands whose range is too wide for that, or that leave fp16's, go to
//     plain_products (kWideLog2, kXPlain).  Against float64 the products are closer than the fp32 form's
//     (4096 x 4096 at 256 rows: 8.4e-7 -> 1.6e-7): a running sum rounds once a
//     chunk instead of once per four k.
// K is split over ranges only where the tiles leave CUs idle; the ranges' sums
// are then added in order by matmul_reduce_kernel.
template <int WT>
struct KOrder {
    // Where the eight values from k (a multiple of 8) go: chunk, block and lane group
    // (F32: see matmul_split_x_tile_kernel).
    static __device__ __forceinline__ void place(int k, int& c, int& blk, int& g) {
        if constexpr (WT == kWeightQ4_K) {
            c = 4 * (k >> 8) + 2 * ((k >> 4) & 1) + ((k >> 5) & 1);
            g = (k >> 6) & 3;
            blk = (k >> 3) & 1;
        } else if constexpr (WT == kWeightQ6_K) {
            c = 4 * (k >> 8) + ((k >> 5) & 3);
            g = 2 * ((k >> 7) & 1) + ((k >> 4) & 1);
            blk = (k >> 3) & 1;
        } else {
            c = k >> 6;
            blk = (k >> 5) & 1;
            g = (k >> 3) & 3;
        }
    }
};

// Added to a row's exponent when the fp16 pairs cannot stand for the row (F32
// products: an infinite element, a row whose largest |x| is below 2^-113, or one
// of a wide range): its outputs are summed in plain fp32 instead.
constexpr int kXPlain = 1 << 16;
// A scaled pair holds an element to 2^-23 of itself or 2^-38 of the scale's
// largest, whichever is more (the matrix cores keep fp16 subnormals).  F32
// operands are wide, and summed in plain fp32, when a group of neighbours (four of
// a row of x; of weights the eight of a 64-wide chunk that one lane has from each
// 32) lies below 2^-kWideLog2 of the largest and is not all zero: otherwise every
// group keeps 22 bits of its own largest.  (Among 4096 normal values beside a
// channel 12 times as loud that happens once in 10^9 rows.)
constexpr int kWideLog2 = 16;
// `low`: the least, over the groups, of the bits of a group's largest magnitude minus one (zero groups wrap to the top).
__device__ __forceinline__ bool wide_row(uint32_t low, float mx) {
    return low + 1 < __float_as_uint(mx * (1.0f / (1 << kWideLog2))) && low != ~0u;
}
constexpr int kTileHalves = 2048;   // one M tile of a chunk: [block][hi, lo][lane][8 halves]
constexpr int kXBlockSumLog2 = 6;   // Q4_K's sub-block sums of x enter times 2^-6 (32 values below 2^13 each)
// The second and third halves of a sum are stored over these factors, which the
// weights' side carries (6-bit values times them are exact, normal halves).
constexpr float kSumScale1 = 1.0f / (1 << 11), kSumScale2 = 1.0f / (1 << 14);

// x of batch row b over K range z as scaled fp16 pairs in tile order,
// [64-row group][chunk][M tile][block][hi, lo][lane g * 16 + m][8 halves], with
// the exponent xexp[z][b]: as matmul_split_x_kernel, mx * 2^-e in [2^12, 2^13).
template <int WT>
__global__ __launch_bounds__(kMmThreads) void matmul_split_x_tile_kernel(MatmulArgs a) {
    __shared__ float red[kMmThreads / 64];
    __shared__ uint32_t red_low[kMmThreads / 64];
    const int b = blockIdx.x;
    const int z = blockIdx.y;
    const int t = threadIdx.x;
    const int p0 = z * a.chunks_per_split * 8;  // pieces of eight values
    const int np = min(a.in_dim / 8, p0 + a.chunks_per_split * 8) - p0;
    const f4* xr = reinterpret_cast<const f4*>(a.x + (int64_t)b * a.in_dim) + 2 * (int64_t)p0;
    // Ranges of up to 8192 values stay in registers between the two passes; longer ones are read twice.
    constexpr int kHeld = 4;
    const bool held = np <= kHeld * kMmThreads;
    f4 hv[kHeld][2];
    float mx = 0.f;
    uint32_t low = ~0u;  // F32: see kWideRow
    auto max8 = [&](const f4& u, const f4& v) {
        const float mu = fmaxf(fmaxf(fabsf(u[0]), fabsf(u[1])), fmaxf(fabsf(u[2]), fabsf(u[3])));
        const float mv = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
        mx = fmaxf(mx, fmaxf(mu, mv));
        if constexpr (WT == kWeightF32) low = min(low, min(__float_as_uint(mu) - 1, __float_as_uint(mv) - 1));
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (kMmThreads * j < np) {
                const int i = min(t + kMmThreads * j, np - 1);
                hv[j][0] = xr[2 * i];
                hv[j][1] = xr[2 * i + 1];
            }
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (kMmThreads * j < np) max8(hv[j][0], hv[j][1]);
    } else {
#pragma unroll 4
        for (int i = t; i < np; i += kMmThreads) max8(xr[2 * i], xr[2 * i + 1]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((t & 63) == 0) red[t >> 6] = mx;
    if constexpr (WT == kWeightF32) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) low = min(low, (uint32_t)__shfl_xor((int)low, off));
        if ((t & 63) == 0) red_low[t >> 6] = low;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int ex = 0;
    if (mx > 0.f && mx <= FLT_MAX) (void)frexpf(mx, &ex);
    const int e = mx > 0.f ? (mx <= FLT_MAX ? min(115, max(-126, ex - 13)) : 115) : 0;
    const float down = ldexpf(1.0f, -e);
    _Float16* xt = static_cast<_Float16*>(a.xh);
    const int64_t chunks = a.in_dim / 64;
    const int64_t row0 = (int64_t)(b >> 6) * chunks;  // chunks before the row's group
    const int tile = (b >> 4) & 3;
    const int m = b & 15;
    auto put = [&](int i, const f4& r0, const f4& r1) {
        h8 hi, lo;
        float sm = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float v = (q < 4 ? r0[q & 3] : r1[q & 3]) * down;
            hi[q] = (_Float16)v;
            // An infinite element rides on its hi half alone (Inf - Inf would be NaN).
            lo[q] = (_Float16)(__builtin_isinf(v) ? 0.f : v - (float)hi[q]);
            sm += v;
        }
        const int k = 8 * (p0 + i);
        int c, blk, g;
        KOrder<WT>::place(k, c, blk, g);
        _Float16* dst = xt + ((row0 + c) * 4 + tile) * kTileHalves + blk * 1024;
        if constexpr (WT == kWeightF32) {
            // The two fours from k and k + 4 go to lane groups (k / 4) % 4 and the next, first or second half.
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                _Float16* d4 = dst + ((((k >> 2) + q) & 3) * 16 + m) * 8 + 4 * ((k >> 4) & 1);
                *reinterpret_cast<h4v*>(d4) = q ? __builtin_shufflevector(hi, hi, 4, 5, 6, 7) : __builtin_shufflevector(hi, hi, 0, 1, 2, 3);
                *reinterpret_cast<h4v*>(d4 + 512) = q ? __builtin_shufflevector(lo, lo, 4, 5, 6, 7) : __builtin_shufflevector(lo, lo, 0, 1, 2, 3);
            }
        } else {
            *reinterpret_cast<h8*>(dst + (g * 16 + m) * 8) = hi;
            *reinterpret_cast<h8*>(dst + (g * 16 + m) * 8 + 512) = lo;
        }
        if constexpr (WT == kWeightQ4_K) {
            // Four consecutive threads hold a sub-block's 32 values, eight the two of a lane group
            // (ranges are whole super-blocks).  A sum's fp32 value is three halves (11 + 11 + 2
            // bits); the lane group's operand is both sums' first halves, then their second and
            // third ones and zeros, [64-row group][super-block][M tile][lane][8 halves].
            sm += __shfl_xor(sm, 1);
            sm += __shfl_xor(sm, 2);
            const float other = __shfl_xor(sm, 4);
            if ((i & 7) == 0) {
                h8 ops = {};
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const float v = (q ? other : sm) * (1.0f / (1 << kXBlockSumLog2));
                    const bool inf = __builtin_isinf(v);  // rides on its first half alone
                    ops[q] = (_Float16)v;
                    const float r1 = inf ? 0.f : (v - (float)ops[q]) * (1.0f / kSumScale1);
                    ops[2 + q] = (_Float16)r1;
                    ops[4 + q] = (_Float16)((r1 - (float)ops[2 + q]) * (kSumScale1 / kSumScale2));
                }
                _Float16* sd = reinterpret_cast<_Float16*>(a.xsum) + (((row0 >> 2) + (k >> 8)) * 4 + tile) * 512 +
                               (((k >> 6) & 3) * 16 + m) * 8;
                *reinterpret_cast<h8*>(sd) = ops;
            }
        }
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const int i = t + kMmThreads * j;
            if (i < np) put(i, hv[j][0], hv[j][1]);
        }
    } else {
        for (int i = t; i < np; i += kMmThreads) put(i, xr[2 * i], xr[2 * i + 1]);
    }
    if (t == 0) {
        bool plain = WT == kWeightF32 && (mx > FLT_MAX || (mx > 0.f && ex - 13 < -126));
        if constexpr (WT == kWeightF32)
            plain |= wide_row(min(min(red_low[0], red_low[1]), min(red_low[2], red_low[3])), mx);
        a.xexp[z * a.batch + b] = e + (plain ? kXPlain : 0);
    }
}

// The wave's weights, by units of kUnit chunks (F32 one, Q8_0 two, the K-quants a
// super-block).  fetch(c) loads the unit that holds chunk c, turn() makes the
// fetched unit the one in hand, expand<CC>() its chunk CC's operands.
//
// Quantized types: read straight into the operand layout (16 rows x 4 lane
// groups a few words each) one load instruction touches 16 rows' lines and the
// L1's line rate, not the matrix cores, bounds the product (Q8_0 512 x 4096 x
// 4096 was 46 cycles of L1 per load).  So a fetch loads a tile's 16 rows in
// 16-byte (Q8_0 8-byte) pieces in row order, and turn() passes them through a
// few KB of LDS that belong to the wave alone: no barrier, LDS serves a wave's
// accesses in order.
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ h2 splat2(_Float16 v) { return h2{v, v}; }

// The weights' side of Q4_K's sums operand: the 6-bit values of two sub-blocks against three halves each.
__device__ __forceinline__ h8 sums_operand(h2 q) {
    const h2 q1 = q * splat2((_Float16)kSumScale1);
    const h2 q2 = q * splat2((_Float16)kSumScale2);
    return h8{q[0], q[1], q1[0], q1[1], q2[0], q2[1], 0, 0};
}

template <int WT>
struct TileW;

constexpr int kTileNT = 2;       // N tiles of a wave
constexpr int kTurnBytes = 3456;  // LDS of one wave's turn(), the largest type's

struct TileWBase {
    __amdgpu_buffer_rsrc_t rsrc;
    int rows;              // rows of the wave inside out_dim (at least one)
    int n, g, lane;
    uint32_t* lds;         // the wave's kTurnBytes
    h8 w[kTileNT][2];      // [N tile][block of the chunk]
    float d[kTileNT];      // the chunk's scale

    // Rows past out_dim read row out_dim - 1; their sums are never stored.  The
    // descriptor starts and ends at dwords (Q6_K rows need not): the up to two
    // bytes this adds at either end share a dword with bytes of the rows.
    __device__ __forceinline__ int base_init(const MatmulArgs& a, int o0, int64_t row_bytes, int lane_, uint32_t* lds_) {
        const int first = min(o0, a.out_dim - 1);
        rows = min(16 * kTileNT, a.out_dim - first);
        const uintptr_t at = reinterpret_cast<uintptr_t>(a.w) + first * row_bytes;
        const int skew = (int)(at & 3);
        rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at - skew), (short)0,
                                                 ((int)(rows * row_bytes) + skew + 3) & ~3, 0x00020000);
        lane = lane_;
        n = lane & 15;
        g = lane >> 4;
        lds = lds_;
        return skew;
    }
    // Piece q of 16 rows of P pieces each, for the lane's i-th load (past the last: the last again).
    template <int P>
    __device__ __forceinline__ void piece(int i, int& q, int& row, int& at) const {
        q = min(lane + 64 * i, 16 * P - 1);
        row = q / P;
        at = q - row * P;
    }
};

// A unit is two chunks, 136 contiguous bytes of a row (17 pieces of 8).  When
// the row ends inside it the rest belongs to the next row and is not used.
template <>
struct TileW<kWeightQ8_0> : TileWBase {
    static constexpr bool kLo = false;
    static constexpr int kUnit = 2, kPieces = 5, kLoads = kPieces * kTileNT;
    u2v next[kTileNT][kPieces];
    int off[kTileNT][kPieces], dst[kPieces];
    struct Raw {
        uint32_t r0[3], r1[2], s0, s1;
    } raw[kTileNT][kUnit];
    float d1[kTileNT];  // block 1's scale (d: block 0's)

    __device__ __forceinline__ void init(const MatmulArgs& a, int o0, int lane_, uint32_t* lds_) {
        const int row_bytes = (a.in_dim / 32) * 34;
        base_init(a, o0, row_bytes, lane_, lds_);
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            int q, row, at;
            piece<17>(i, q, row, at);
            dst[i] = 2 * q;
#pragma unroll
            for (int j = 0; j < kTileNT; ++j) off[j][i] = min(16 * j + row, rows - 1) * row_bytes + 8 * at;
        }
    }
    __device__ __forceinline__ void fetch(int c) {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j)
#pragma unroll
            for (int i = 0; i < kPieces; ++i) next[j][i] = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off[j][i], c * 68, 0);
    }
    // Chunk h of the unit: dwords 17 h .. of the row; block 0's values from byte 2
    // of dword 2 g on, block 1's at dwords 9 + 2 g and 10 + 2 g, the scales the low half of dword
    // 0 and the high half of dword 8.
    __device__ __forceinline__ void turn() {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u2v*>(lds + dst[i]) = next[j][i];
#pragma unroll
            for (int h = 0; h < kUnit; ++h) {
                const uint32_t* row = lds + 34 * n + 17 * h;
                Raw& r = raw[j][h];
#pragma unroll
                for (int i = 0; i < 3; ++i) r.r0[i] = row[2 * g + i];
#pragma unroll
                for (int i = 0; i < 2; ++i) r.r1[i] = row[9 + 2 * g + i];
                r.s0 = row[0];
                r.s1 = row[8];
            }
        }
    }
    template <int CC>
    __device__ __forceinline__ void expand() {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
            const Raw& q = raw[j][CC];
            w[j][0] = q8_to_h8(__builtin_amdgcn_alignbyte(q.r0[1], q.r0[0], 2), __builtin_amdgcn_alignbyte(q.r0[2], q.r0[1], 2));
            w[j][1] = q8_to_h8(q.r1[0], q.r1[1]);
            d[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(q.s0 & 0xFFFFu));
            d1[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(q.s1 >> 16));
        }
    }
};

template <>
struct TileW<kWeightQ4_K> : TileWBase {
    static constexpr bool kLo = false;
    static constexpr int kUnit = 4, kPieces = 3, kLoads = kPieces * kTileNT;
    u4 next[kTileNT][kPieces];
    int off[kTileNT][kPieces], dst[kPieces];
    struct Raw {
        u4 hd, q[2];
    } raw[kTileNT];
    h2 sp[kTileNT];     // the quarter's two scales
    h2 mp[kTileNT];     // and mins
    float dm[kTileNT];  // dmin, times 2^6 for the sums' scale

    __device__ __forceinline__ void init(const MatmulArgs& a, int o0, int lane_, uint32_t* lds_) {
        const int row_bytes = (a.in_dim / 256) * 144;
        base_init(a, o0, row_bytes, lane_, lds_);
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            int q, row, at;
            piece<9>(i, q, row, at);
            dst[i] = 4 * q;
#pragma unroll
            for (int j = 0; j < kTileNT; ++j) off[j][i] = min(16 * j + row, rows - 1) * row_bytes + 16 * at;
        }
    }
    __device__ __forceinline__ void fetch(int c) {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j)
#pragma unroll
            for (int i = 0; i < kPieces; ++i)
                next[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[j][i], (c >> 2) * 144, 0);
    }
    __device__ __forceinline__ void turn() {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u4*>(lds + dst[i]) = next[j][i];
            const u4* row = reinterpret_cast<const u4*>(lds) + 9 * n;
            raw[j].hd = row[0];
            raw[j].q[0] = row[1 + 2 * g];
            raw[j].q[1] = row[2 + 2 * g];
        }
    }
    // Chunk CC: sub-block 2 g + CC % 2 (the low or the high nibbles), quant bytes 16 (CC / 2) .. of the quarter.
    // The operand is sc (q - 8): half the size of sc q, and so is the error of its sums; the 8 sc joins the min term.
    template <int CC>
    __device__ __forceinline__ void expand() {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
            const Raw& q = raw[j];
            if constexpr (CC == 0) {
                // Sub-blocks 2 g and 2 g + 1: bytes j and j + 4 of the packed scales for g < 2,
                // else nibbles of byte j + 4 under the top bits of bytes j - 4 and j.
                const int sh = 16 * (g & 1);
                const uint32_t b0 = q.hd[1] >> sh, b1 = q.hd[2] >> sh, b2 = q.hd[3] >> sh;
                const bool low = g < 2;
                const uint32_t s = low ? b0 & 0x3F3Fu : (b2 & 0x0F0Fu) | ((b0 >> 2) & 0x3030u);
                const uint32_t m = low ? b1 & 0x3F3Fu : ((b2 >> 4) & 0x0F0Fu) | ((b1 >> 2) & 0x3030u);
                sp[j] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, s, 0x04010400u)) - splat2((_Float16)1024.0f);
                mp[j] = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, m, 0x04010400u)) - splat2((_Float16)1024.0f);
                d[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(q.hd[0] & 0xFFFFu));
                dm[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(q.hd[0] >> 16)) * (float)(1 << kXBlockSumLog2);
            }
            const h2 s2 = splat2(sp[j][CC & 1]);
            const h2 off8 = s2 * splat2((_Float16)-136.0f);  // exact: a multiple of 8 below 2^14
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                h8 r;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    // The half 0x5800 | 8 q is 128 + q.
                    const uint32_t qw = q.q[CC >> 1][2 * blk + t];
                    const uint32_t u = (CC & 1 ? qw >> 1 : qw << 3) & 0x78787878u;
                    const h2 p0 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x58585858u, u, 0x04010400u));
                    const h2 p1 = __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x58585858u, u, 0x04030402u));
                    const h2 w0 = __builtin_elementwise_fma(p0, s2, off8);  // (128 + q) sc - 136 sc, exact
                    const h2 w1 = __builtin_elementwise_fma(p1, s2, off8);
                    r[4 * t + 0] = w0[0];
                    r[4 * t + 1] = w0[1];
                    r[4 * t + 2] = w1[0];
                    r[4 * t + 3] = w1[1];
                }
                w[j][blk] = r;
            }
        }
    }
};

// Super-blocks are 210 bytes, so a row's may start in the middle of a dword: the
// 53 dwords that hold it are fetched as 13 pieces of 16 bytes and a tail dword,
// and turn() shifts the lane's words into place.
template <>
struct TileW<kWeightQ6_K> : TileWBase {
    static constexpr bool kLo = true;
    static constexpr int kUnit = 4, kPieces = 4, kLoads = (kPieces + 1) * kTileNT;
    u4 next[kTileNT][kPieces];
    uint32_t tail[kTileNT];
    int sb_bytes = 0;  // byte offset of the fetched super-block in a row
    int off[kTileNT][kPieces], dst[kPieces], at16[kPieces];
    int row_off[kTileNT];  // of row n
    struct Raw {
        uint32_t l[2][4], h[4], sc[2], dh;
    } raw[kTileNT];
    h8 lo[kTileNT][2];

    __device__ __forceinline__ void init(const MatmulArgs& a, int o0, int lane_, uint32_t* lds_) {
        const int row_bytes = (a.in_dim / 256) * 210;
        const int skew = base_init(a, o0, row_bytes, lane_, lds_);
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            int q, row;
            piece<13>(i, q, row, at16[i]);
            dst[i] = 4 * q;
#pragma unroll
            for (int j = 0; j < kTileNT; ++j) off[j][i] = skew + min(16 * j + row, rows - 1) * row_bytes;
        }
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) row_off[j] = skew + min(16 * j + n, rows - 1) * row_bytes;
    }
    __device__ __forceinline__ void fetch(int c) {
        const int sb = (c >> 2) * 210;
        sb_bytes = sb;
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i)
                next[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, ((off[j][i] + sb) & ~3) + 16 * at16[i], 0, 0);
            tail[j] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, ((row_off[j] + sb) & ~3) + 208, 0, 0);
        }
    }
    __device__ __forceinline__ void turn() {
        const int hn = g >> 1, l = 4 * (g & 1);  // half of the super-block, the lane's dwords in a quarter
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
#pragma unroll
            for (int i = 0; i < kPieces; ++i) *reinterpret_cast<u4*>(lds + dst[i]) = next[j][i];
            const uint32_t* row = lds + 52 * n;
            const int s = (row_off[j] + sb_bytes) & 2;
            auto window = [&](int at, uint32_t (&out)[4]) {
                const u4 v = *reinterpret_cast<const u4*>(row + at);
                const uint32_t e = row[at + 4];
                out[0] = __builtin_amdgcn_alignbyte(v[1], v[0], s);
                out[1] = __builtin_amdgcn_alignbyte(v[2], v[1], s);
                out[2] = __builtin_amdgcn_alignbyte(v[3], v[2], s);
                out[3] = __builtin_amdgcn_alignbyte(e, v[3], s);
            };
            Raw& r = raw[j];
            window(16 * hn + l, r.l[0]);
            window(16 * hn + l + 8, r.l[1]);
            window(32 + 8 * hn + l, r.h);
            const uint32_t s0 = row[48 + 2 * hn], s1 = row[49 + 2 * hn];
            const uint32_t s2 = hn ? tail[j] : row[50];
            r.sc[0] = __builtin_amdgcn_alignbyte(s1, s0, s);
            r.sc[1] = __builtin_amdgcn_alignbyte(s2, s1, s);
            r.dh = tail[j] >> (8 * s);  // d in the low half
        }
    }
    // Chunk CC is quarter CC of the half: its 16 values of the lane share the scale 8 n + g % 2 + 2 CC.
    template <int CC>
    __device__ __forceinline__ void expand() {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
            const Raw& r = raw[j];
            if constexpr (CC == 0) d[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.dh & 0xFFFFu));
            const int sv = (int)(int8_t)((r.sc[CC >> 1] >> (8 * (g & 1) + 16 * (CC & 1))) & 0xFFu);
            const h2 s2 = splat2((_Float16)(float)sv);
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                h8 hi, lw;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint32_t u = ((r.l[CC & 1][2 * blk + t] >> (4 * (CC >> 1))) & 0x0F0F0F0Fu) |
                                       (((r.h[2 * blk + t] >> (2 * CC)) & 0x03030303u) << 4);
                    h2 q[2];
                    six_to_h4(u, q[0], q[1]);
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const h2 m = q[v] * s2;
                        const h2 rest = __builtin_elementwise_fma(q[v], s2, -m);  // exact: 0 or +-1
                        hi[4 * t + 2 * v] = m[0];
                        hi[4 * t + 2 * v + 1] = m[1];
                        lw[4 * t + 2 * v] = rest[0];
                        lw[4 * t + 2 * v + 1] = rest[1];
                    }
                }
                w[j][blk] = hi;
                lo[j][blk] = lw;
            }
        }
    }
};

// Max of x over lanes l, l ^ 16, l ^ 32 and l ^ 48.
__device__ __forceinline__ float lane_group_max(float x) {
    const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
    const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}

// One chunk per unit, fetched two ahead straight into the operand layout (a load
// covers 64 contiguous bytes of each row).
template <>
struct TileW<kWeightF32> : TileWBase {
    static constexpr bool kLo = true;
    static constexpr int kUnit = 1, kLoads = 4 * kTileNT;
    struct Raw {
        f4 v[4];
    } next[2][kTileNT];
    int row_off[kTileNT];
    h8 lo[kTileNT][2];
    uint32_t range[kTileNT] = {};  // see expand; each lane group of the row has its part

    __device__ __forceinline__ void init(const MatmulArgs& a, int o0, int lane_, uint32_t* lds_) {
        base_init(a, o0, (int64_t)a.in_dim * 4, lane_, lds_);
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) row_off[j] = min(16 * j + n, rows - 1) * a.in_dim * 4 + 16 * g;
    }
    __device__ __forceinline__ void fetch(int slot, int c) {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                next[slot][j].v[i] =
                    __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, row_off[j] + 64 * i, c * 256, 0));
    }
    // The row's largest |w| of the chunk goes to [2^12, 2^13).  d is 2^(e - 13), the
    // other 2^13 joining the batch row's exponent at the end, so that the running
    // sum stays about |w| times the scaled x.  Chunks that reach 2^100 (or hold an infinity), or
    // with weights below 2^-100, leave fp16's or that sum's range, and a chunk of a wide range
    // (kWideLog2) leaves the pairs': their row is summed in plain fp32.  The check is in whole
    // numbers on purpose: as compares and a mask it cost 4.5 of 62 us (256 rows of 4096 x 4096),
    // with groups of four weights 2.5; as it is, nothing.
    template <int CC>
    __device__ __forceinline__ void expand(int slot) {
#pragma unroll
        for (int j = 0; j < kTileNT; ++j) {
            const f4 (&r)[4] = next[slot][j].v;
            float mx = 0.f;
            uint32_t low = ~0u;  // see wide_row; the groups are the lane's halves of the chunk
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float m8 = 0.f;
#pragma unroll
                for (int q = 0; q < 8; ++q) m8 = fmaxf(m8, fabsf(r[2 * i + (q >> 2)][q & 3]));
                mx = fmaxf(mx, m8);
                low = min(low, __float_as_uint(m8) - 1);
            }
            mx = lane_group_max(mx);
            const int field = (int)(__float_as_uint(mx) >> 23);
            const int e = min(87, max(-113, field - 139));  // field 126 + ex, mx = f * 2^ex with f in [0.5, 1)
            // The distance, as bits, from the chunk's largest (at least 2^-84) to its least group, or
            // from 2^84 to its largest: 2^16 apart or more and the pairs cannot stand for the row.
            const uint32_t m = __float_as_uint(mx);
            range[j] = max(range[j], max(__builtin_elementwise_sub_sat(max(m, (127u - 84) << 23), low),
                                         __builtin_elementwise_sub_sat(m, (127u + 84) << 23)));
            const float down = __uint_as_float((uint32_t)(127 - e) << 23);
            d[j] = __uint_as_float((uint32_t)(127 + e - 13) << 23);
#pragma unroll
            for (int blk = 0; blk < 2; ++blk)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float v = r[2 * blk + (q >> 2)][q & 3] * down;
                    const _Float16 hi = (_Float16)v;
                    w[j][blk][q] = hi;
                    lo[j][blk][q] = (_Float16)(v - (float)hi);
                }
        }
    }
};

// x in LDS: a ring of four chunks, each an array of its own so that the
// compiler sees which direct loads a read depends on.
struct TileLds {
    u4 *x0, *x1, *x2, *x3;
    template <int S>
    __device__ __forceinline__ u4* slot() const {
        return S == 0 ? x0 : S == 1 ? x1 : S == 2 ? x2 : x3;
    }
};

// The workgroup's K loop over MT M tiles (16 MT batch rows from 64 by).
//
// Per chunk c the direct loads of x chunk c + 3 go out, and at a unit's start the
// fetch of the next unit (F32: of chunk c + 2), then chunk c's products run.  A
// wave waits for its part of chunk c + 1 before the barrier that ends chunk c.
// Memory loads count in order, so it waits until only the loads issued after
// that part are left: the 2 MT direct loads of chunks c + 2 and c + 3, and those
// of the fetches in chunks c - 2 .. c (the compiler may not move loads over the
// asm).  Past the range's end the last chunk is loaded again (into a slot nobody
// reads any more), so that the count holds to the end.
template <int WT, int MT>
__device__ __forceinline__ void tile_products(const MatmulArgs& a, TileW<WT>& w, f4 (&acc)[4][kTileNT], const TileLds& xs,
                                              int by, int c_begin, int c_end) {
    constexpr int NT = kTileNT;
    constexpr int kUnit = TileW<WT>::kUnit;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int chunks = a.in_dim / 64;

    // The 4 MT KB of a chunk's M tiles: wave w moves kilobytes w MT .. + MT - 1.
    const _Float16* xg = static_cast<const _Float16*>(a.xh) + (int64_t)by * chunks * 4 * kTileHalves;
    auto stage_x = [&](auto s_t, int c) {
        u4* dst = xs.slot<decltype(s_t)::value>();
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<_Float16*>(xg + (int64_t)min(c, c_end - 1) * 4 * kTileHalves), (short)0, 4 * kTileHalves * 2, 0x00020000);
#pragma unroll
        for (int i = 0; i < MT; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                r, (__attribute__((address_space(3))) void*)(dst + 64 * (wave * MT + i)), 16, 16 * lane,
                1024 * (wave * MT + i), 0, 0);
    };
    // Q4_K: the M tiles' sub-block sums of a super-block.
    const h8* sg = reinterpret_cast<const h8*>(a.xsum) + (int64_t)by * (chunks / 4) * 256 + lane;
    h8 sx[MT];
    auto load_sums = [&](int c) {
#pragma unroll
        for (int t = 0; t < MT; ++t) sx[t] = sg[(c >> 2) * 256 + 64 * t];
    };

    // Chunk c = c_begin + S (mod 4).
    auto chunk = [&](auto s_t, int c) {
        constexpr int S = decltype(s_t)::value;
        constexpr int CC = S % kUnit;
        stage_x(std::integral_constant<int, (S + 3) % 4>{}, c + 3);
        __builtin_amdgcn_sched_barrier(0x78F);  // no vector memory access crosses: kLater counts the fetches below as later
        if constexpr (WT == kWeightF32) {
            w.template expand<CC>(S % 2);
            w.fetch(S % 2, min(c + 2, c_end - 1));
        } else {
            // The last unit once more at the range's end, unused.
            if constexpr (CC == 0) w.fetch(c + kUnit < c_end ? c + kUnit : c);
            w.template expand<CC>();
        }
        if constexpr (WT == kWeightQ4_K) {
            if constexpr (CC == 0) {  // the super-block's min term, dmin m - 8 d sc against the sums of x
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const h8 mb = sums_operand(w.mp[j]);
                    const h8 sb = sums_operand(w.sp[j]);
                    const float d8 = w.d[j] * (float)(8 << kXBlockSumLog2);
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const f4 pm = __builtin_amdgcn_mfma_f32_16x16x32_f16(sx[t], mb, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        const f4 ps = __builtin_amdgcn_mfma_f32_16x16x32_f16(sx[t], sb, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[t][j][r] = fmaf(-w.dm[j], pm[r], fmaf(d8, ps[r], acc[t][j][r]));
                    }
                }
                load_sums(min(c + 4, c_end - 1));
            }
        }
        const h8* xb = reinterpret_cast<const h8*>(xs.slot<S>()) + lane;
        // M tiles in pairs: 2 NT independent accumulator chains keep the matrix
        // cores busy through each other's latency.
        constexpr int kPair = MT < 2 ? 1 : 2;
#pragma unroll
        for (int t0 = 0; t0 < MT; t0 += kPair) {
            h8 ax[kPair][2][2];
#pragma unroll
            for (int p = 0; p < kPair; ++p)
#pragma unroll
                for (int blk = 0; blk < 2; ++blk)
#pragma unroll
                    for (int h = 0; h < 2; ++h) ax[p][blk][h] = xb[(t0 + p) * (kTileHalves / 8) + (blk * 2 + h) * 64];
            f4 part[kPair][NT], sum[kPair][NT];
            auto zero = [&] {
#pragma unroll
                for (int p = 0; p < kPair; ++p)
#pragma unroll
                    for (int j = 0; j < NT; ++j) part[p][j] = f4{0.f, 0.f, 0.f, 0.f};
            };
            auto step = [&](int blk, int h, const h8 (&wv)[NT][2]) {
#pragma unroll
                for (int p = 0; p < kPair; ++p)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        part[p][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ax[p][blk][h], wv[j][blk], part[p][j], 0, 0, 0);
            };
            auto add = [&](const float (&sc)[NT]) {
#pragma unroll
                for (int p = 0; p < kPair; ++p)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[t0 + p][j][r] = fmaf(sc[j], part[p][j][r], acc[t0 + p][j][r]);
            };
            zero();
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                step(blk, 1, w.w);
                if constexpr (TileW<WT>::kLo) step(blk, 0, w.lo);
                step(blk, 0, w.w);
                if constexpr (WT == kWeightQ8_0) {
                    // Each block its own scale; the chunk's two sums join before the running
                    // one, which then rounds once a chunk as for the other types.
#pragma unroll
                    for (int p = 0; p < kPair; ++p)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                if (blk == 0) sum[p][j][r] = w.d[j] * part[p][j][r];
                                else acc[t0 + p][j][r] += fmaf(w.d1[j], part[p][j][r], sum[p][j][r]);
                            }
                    zero();
                }
            }
            if constexpr (WT != kWeightQ8_0) add(w.d);
        }
        if constexpr (WT != kWeightF32) {
            if constexpr (CC == kUnit - 1) w.turn();
        }
        // lgkmcnt(0): this wave's reads of the slot are done, and the next chunk's direct loads may overwrite it.
        constexpr int kFetches = (S % kUnit == 0) + ((S + 3) % kUnit == 0) + ((S + 2) % kUnit == 0);
        constexpr int kLater = 2 * MT + kFetches * (TileW<WT>::kLoads + (WT == kWeightQ4_K ? MT : 0));
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLater) : "memory");
        __builtin_amdgcn_s_barrier();
    };

    if constexpr (WT == kWeightF32) {
        w.fetch(0, c_begin);
        w.fetch(1, min(c_begin + 1, c_end - 1));
    } else {
        w.fetch(c_begin);
    }
    if constexpr (WT == kWeightQ4_K) load_sums(c_begin);
    stage_x(std::integral_constant<int, 0>{}, c_begin);
    stage_x(std::integral_constant<int, 1>{}, c_begin + 1);
    stage_x(std::integral_constant<int, 2>{}, c_begin + 2);
    if constexpr (WT != kWeightF32) w.turn();
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // chunks c_begin .. + 2 have landed
    __builtin_amdgcn_s_barrier();
    for (int c = c_begin; c < c_end; c += 4) {  // super-block types: ranges are whole super-blocks (host)
        chunk(std::integral_constant<int, 0>{}, c);
        if (kUnit < 4 && c + 1 >= c_end) break;
        chunk(std::integral_constant<int, 1>{}, c + 1);
        if (kUnit < 4 && c + 2 >= c_end) break;
        chunk(std::integral_constant<int, 2>{}, c + 2);
        if (kUnit < 4 && c + 3 >= c_end) break;
        chunk(std::integral_constant<int, 3>{}, c + 3);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load outlives the loop
}

// MB x NB blocks of 16 x 16 outputs (M tiles from batch row b, N tiles from weight
// row o) over k0 .. k1 on the fp32 matrix cores.  Operand order as
// in the fp32 form: lane (n, g) brings k = 16 i + 4 g + s to step s; the next 64 k
// load while these are multiplied.
template <int MB, int NB>
__device__ __forceinline__ void plain_block(const MatmulArgs& a, int b, int o, int n, int g, int k0, int k1, f4 (&acc)[MB][NB]) {
    const float *xr[MB], *wr[NB];
#pragma unroll
    for (int p = 0; p < MB; ++p) xr[p] = a.x + (int64_t)min(b + 16 * p + n, a.batch - 1) * a.in_dim + 4 * g;
#pragma unroll
    for (int j = 0; j < NB; ++j)
        wr[j] = static_cast<const float*>(a.w) + (int64_t)min(o + 16 * j + n, a.out_dim - 1) * a.in_dim + 4 * g;
    f4 xv[2][MB][4], wv[2][NB][4];
    auto load = [&](int slot, int k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int p = 0; p < MB; ++p) xv[slot][p][i] = *reinterpret_cast<const f4*>(xr[p] + k + 16 * i);
#pragma unroll
            for (int j = 0; j < NB; ++j) wv[slot][j][i] = *reinterpret_cast<const f4*>(wr[j] + k + 16 * i);
        }
    };
#pragma unroll
    for (int p = 0; p < MB; ++p)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[p][j] = f4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int p = 0; p < MB; ++p)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        acc[p][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[slot][p][i][s], wv[slot][j][i][s], acc[p][j], 0, 0, 0);
    };
    load(0, k0);
    for (int k = k0; k < k1; k += 128) {  // ranges are whole chunks
        if (k + 64 < k1) load(1, k + 64);
        products(0);
        if (k + 64 >= k1) break;
        if (k + 128 < k1) load(0, k + 128);
        products(1);
    }
}

// F32 outputs that the fp16 pairs cannot stand for: bit m of `xm` marks batch row b0
// + m, bit i of wm[w] weight row o0 + 32 w + i.  The workgroup sums the blocks with
// such a row in plain fp32, 2 x 2 blocks to each wave in turn, and those outputs
// replace what was stored.  256 rows of 4096 x 4096: one such weight row 84 us (58
// without), one such row of x 102, all of them 174 (the fp32 form 87): the loads'
// address work bounds it, 16 rows a load.
__device__ __forceinline__ void plain_products(const MatmulArgs& a, uint64_t xm, const uint32_t (&wm)[4], int b0, int mt,
                                               int o0, int lane, int wave, int k0, int k1, float* dst) {
    const int n = lane & 15, g = lane >> 4;
    int turn = 0;
    for (int at = 0; at < 8; ++at) {
        const int t = 2 * (at >> 2), pair = at & 3;  // M tiles t, t + 1 and N tiles 2 pair, 2 pair + 1
        if (t >= mt) break;
        const uint32_t xb = (uint32_t)(xm >> (16 * t)), wb = wm[pair];  // 32 rows each
        if (!(xb | wb) || (turn++ & 3) != wave) continue;
        const int b = b0 + 16 * t, o = o0 + 32 * pair;
        auto store = [&](int p, int j, const f4& sum) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = 16 * p + 4 * g + r, i = 16 * j + n;
                if (b + m < a.batch && o + i < a.out_dim && (((xb >> m) | (wb >> i)) & 1))
                    dst[(int64_t)(b + m) * a.out_dim + o + i] = sum[r];
            }
        };
        // Rows of one M (N) tile only: half the block.
        if (!wb && (!(xb >> 16) || !(xb & 0xFFFFu))) {
            const int p = xb >> 16 ? 1 : 0;
            f4 acc[1][2];
            plain_block(a, b + 16 * p, o, n, g, k0, k1, acc);
            store(p, 0, acc[0][0]);
            store(p, 1, acc[0][1]);
        } else if (!xb && (!(wb >> 16) || !(wb & 0xFFFFu))) {
            const int j = wb >> 16 ? 1 : 0;
            f4 acc[2][1];
            plain_block(a, b, o + 16 * j, n, g, k0, k1, acc);
            store(0, j, acc[0][0]);
            store(1, j, acc[1][0]);
        } else {
            f4 acc[2][2];
            plain_block(a, b, o, n, g, k0, k1, acc);
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int j = 0; j < 2; ++j) store(p, j, acc[p][j]);
        }
    }
}

template <int WT>
__global__ __launch_bounds__(kMmThreads, 2) void matmul_tile_kernel(MatmulArgs a) {
    constexpr int NT = kTileNT;
    __shared__ u4 xs0[4 * kTileHalves / 8], xs1[4 * kTileHalves / 8], xs2[4 * kTileHalves / 8], xs3[4 * kTileHalves / 8];
    __shared__ u4 turn[4][kTurnBytes / 16];
    const TileLds xs{xs0, xs1, xs2, xs3};

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int g = lane >> 4;
    const int chunks = a.in_dim / 64;

    // Workgroups go to the eight XCDs in turn; each XCD takes a contiguous run of
    // (range, weight tile, batch group), batch groups fastest, so that the
    // workgroups that share a weight tile share an L2.
    const int wtiles = (a.out_dim + 64 * NT - 1) / (64 * NT);
    const int groups = (a.batch + 63) / 64;
    const int total = wtiles * groups * a.splits;
    const int xcd = blockIdx.x % 8, per_xcd = total / 8, extra = total % 8;
    const int id = xcd * per_xcd + min(xcd, extra) + blockIdx.x / 8;
    const int by = id % groups;
    const int bx = (id / groups) % wtiles;
    const int z = id / (groups * wtiles);

    const int b0 = by * 64;
    const int mt = min(4, (a.batch - b0 + 15) >> 4);  // M tiles in use
    const int o0 = (bx * 4 + wave) * 16 * NT;
    const int c_begin = z * a.chunks_per_split;
    const int c_end = min(chunks, c_begin + a.chunks_per_split);

    TileW<WT> w;
    w.init(a, o0, lane, reinterpret_cast<uint32_t*>(turn[wave]));
    f4 acc[4][NT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[t][j] = f4{0.f, 0.f, 0.f, 0.f};
    if (mt > 2) tile_products<WT, 4>(a, w, acc, xs, by, c_begin, c_end);
    else if (mt == 2) tile_products<WT, 2>(a, w, acc, xs, by, c_begin, c_end);
    else tile_products<WT, 1>(a, w, acc, xs, by, c_begin, c_end);

    // Lane holds batch rows b0 + 16 t + 4 g + r of weight rows o0 + 16 j + n.
    float* dst = a.split_out ? a.split_out + (int64_t)z * a.batch * a.out_dim : a.y;
    constexpr int kExtra = WT == kWeightF32 ? 13 : 0;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int b = b0 + 16 * t + 4 * g + r;
            if (b >= a.batch) continue;
            const int e = a.xexp[z * a.batch + b];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int o = o0 + 16 * j + n;
                if (o < a.out_dim) dst[(int64_t)b * a.out_dim + o] = ldexpf(acc[t][j][r], e + kExtra);
            }
        }
    if constexpr (WT == kWeightF32) {
        // Rows the fp16 pairs cannot stand for, as masks: the batch group's 64 and each wave's 32.
        uint32_t rows = 0;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            uint32_t m = w.range[j];
            m = max(m, (uint32_t)__shfl_xor((int)m, 16));
            m = max(m, (uint32_t)__shfl_xor((int)m, 32));
            rows |= ((uint32_t)__ballot(m >= ((uint32_t)kWideLog2 << 23)) & 0xFFFFu) << (16 * j);
        }
        const uint64_t xm = __ballot(b0 + lane < a.batch && a.xexp[z * a.batch + b0 + lane] > kXPlain / 2);
        // Words of their own: other waves' last direct loads of x may still be landing.  The barrier also
        // orders a wave's stores above before another's below.
        __shared__ uint32_t wide_rows[4];
        if (lane == 0) wide_rows[wave] = rows;
        __syncthreads();
        const uint32_t wm[4] = {wide_rows[0], wide_rows[1], wide_rows[2], wide_rows[3]};
        if (xm || wm[0] | wm[1] | wm[2] | wm[3])
            plain_products(a, xm, wm, b0, mt, bx * 64 * NT, lane, wave, 64 * c_begin, 64 * c_end, dst);
    }
}

// y = the sum over z of the split partials, in z order; four elements per
// thread and step when y and the partials are 16-byte aligned, else one.
__global__ __launch_bounds__(kMmThreads) void matmul_reduce_kernel(MatmulArgs a) {
    const int64_t n = (int64_t)a.batch * a.out_dim;
    const int64_t stride = (int64_t)gridDim.x * kMmThreads;
    const int64_t first = (int64_t)blockIdx.x * kMmThreads + threadIdx.x;
    if (n % 4 == 0 && reinterpret_cast<uintptr_t>(a.y) % 16 == 0) {
        const f4* src = reinterpret_cast<const f4*>(a.split_out);
        f4* dst = reinterpret_cast<f4*>(a.y);
        const int64_t n4 = n / 4;
        for (int64_t i = first; i < n4; i += stride) {
            f4 s = src[i];
            for (int z = 1; z < a.splits; ++z) s += src[(int64_t)z * n4 + i];
            dst[i] = s;
        }
        return;
    }
    for (int64_t i = first; i < n; i += stride) {
        float s = a.split_out[i];
        for (int z = 1; z < a.splits; ++z) s += a.split_out[(int64_t)z * n + i];
        a.y[i] = s;
    }
}

}  // namespace

int matmul_small_chunks(int) { return 8; }

int matmul_small_range_chunks_max() { return 4 * kMmThreads / 16; }  // the pre-pass: four f4 per thread

int64_t matmul_small_x_halves(int batch, int in_dim) {
    return (int64_t)(batch <= 16 ? 1 : batch <= 32 ? 2 : 4) * 16 * in_dim * 2;  // NT whole M tiles, hi and lo
}

int matmul_small_max_splits(int batch) { return kSmMaxPartials / (batch <= 16 ? 1 : batch <= 32 ? 2 : 4); }

namespace {

template <int NT, bool kPasses>
void launch_small_product(const MatmulArgs& a, dim3 grid, hipStream_t stream) {
    if (a.w_type == kWeightQ4_K)
        hipLaunchKernelGGL((matmul_q4k_f16_small_kernel<NT, kPasses>), grid, dim3(kMmThreads), 0, stream, a);
    else if (a.w_type == kWeightQ6_K)
        hipLaunchKernelGGL((matmul_q6k_f16_small_kernel<NT, kPasses>), grid, dim3(kMmThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((matmul_q8_f16_small_kernel<NT, 8, kPasses>), grid, dim3(kMmThreads), 0, stream, a);
}

template <bool kPasses>
void launch_small_product(const MatmulArgs& a, dim3 grid, hipStream_t stream) {
    if (a.batch <= 16)
        launch_small_product<1, kPasses>(a, grid, stream);
    else if (a.batch <= 32)
        launch_small_product<2, kPasses>(a, grid, stream);
    else
        launch_small_product<4, kPasses>(a, grid, stream);
}

}  // namespace

hipError_t launch_matmul_small(const MatmulArgs& a, hipStream_t stream) {
    if (a.batch <= 0 || a.out_dim <= 0) return hipSuccess;
    const bool q4k = a.w_type == kWeightQ4_K;
    const bool q6k = a.w_type == kWeightQ6_K;
    if (a.batch > 64 || (a.w_type != kWeightQ8_0 && !q4k && !q6k) || !a.xh || !a.xl || !a.xexp ||
        a.chunks_per_split < 1 || a.chunks_per_split > matmul_small_range_chunks_max() ||
        a.splits > matmul_small_max_splits(a.batch) || (a.splits > 1 && (!a.split_out || !a.counters)) ||
        (q4k && (!a.xsum || a.in_dim % 256 != 0)) || (q6k && (a.in_dim % 256 != 0 || a.chunks_per_split % 2 != 0)))
        return hipErrorInvalidValue;
    const dim3 pre(a.batch, a.splits);
    if (a.chunks_per_split * 16 <= kMmThreads) {
        if (q4k)
            hipLaunchKernelGGL((matmul_split_x_range_kernel<true, 1>), pre, dim3(kMmThreads), 0, stream, a);
        else
            hipLaunchKernelGGL((matmul_split_x_range_kernel<false, 1>), pre, dim3(kMmThreads), 0, stream, a);
    } else {
        if (q4k)
            hipLaunchKernelGGL((matmul_split_x_range_kernel<true, 4>), pre, dim3(kMmThreads), 0, stream, a);
        else
            hipLaunchKernelGGL((matmul_split_x_range_kernel<false, 4>), pre, dim3(kMmThreads), 0, stream, a);
    }
    const dim3 grid((a.out_dim + kMmRowsWg - 1) / kMmRowsWg, 1, a.splits);
    if (a.chunks_per_split <= matmul_small_chunks(a.batch))
        launch_small_product<false>(a, grid, stream);
    else
        launch_small_product<true>(a, grid, stream);
    return hipGetLastError();
}

int matmul_tile_rows() { return 64 * kTileNT; }

static void launch_reduce(const MatmulArgs& a, hipStream_t stream) {
    const int64_t n = (int64_t)a.batch * a.out_dim;
    const int blocks = (int)std::min<int64_t>((n / 4 + kMmThreads - 1) / kMmThreads + 1, 2048);
    hipLaunchKernelGGL(matmul_reduce_kernel, dim3(blocks), dim3(kMmThreads), 0, stream, a);
}

// The tile form: the x pre-pass, then matmul_tile_kernel.
hipError_t launch_matmul_tile(const MatmulArgs& a, hipStream_t stream) {
    if (a.batch <= 0 || a.out_dim <= 0) return hipSuccess;
    const bool kquant = a.w_type == kWeightQ4_K || a.w_type == kWeightQ6_K;
    if (!a.xh || !a.xexp || a.chunks_per_split < 1 || (a.splits > 1) != (a.split_out != nullptr) ||
        (kquant && (a.in_dim % 256 != 0 || a.chunks_per_split % 4 != 0)) || (a.w_type == kWeightQ4_K && !a.xsum))
        return hipErrorInvalidValue;
    const int64_t total = (int64_t)((a.out_dim + 64 * kTileNT - 1) / (64 * kTileNT)) * ((a.batch + 63) / 64) * a.splits;
    if (total > INT32_MAX) return hipErrorInvalidValue;
    auto go = [&](auto wt) {
        constexpr int WT = decltype(wt)::value;
        hipLaunchKernelGGL(matmul_split_x_tile_kernel<WT>, dim3(a.batch, a.splits), dim3(kMmThreads), 0, stream, a);
        hipLaunchKernelGGL(matmul_tile_kernel<WT>, dim3((unsigned)total), dim3(kMmThreads), 0, stream, a);
        if (a.splits > 1) launch_reduce(a, stream);
        return hipGetLastError();
    };
    switch (a.w_type) {
        case kWeightF32: return go(std::integral_constant<int, kWeightF32>{});
        case kWeightQ8_0: return go(std::integral_constant<int, kWeightQ8_0>{});
        case kWeightQ4_K: return go(std::integral_constant<int, kWeightQ4_K>{});
        case kWeightQ6_K: return go(std::integral_constant<int, kWeightQ6_K>{});
    }
    return hipErrorInvalidValue;
}

hipError_t launch_matmul(const MatmulArgs& a, hipStream_t stream) {
    if (a.batch <= 0 || a.out_dim <= 0) return hipSuccess;
    const dim3 grid((a.out_dim + kMmRowsWg - 1) / kMmRowsWg, (a.batch + 63) / 64, a.splits);
    if (a.w_type == kWeightF32)
        hipLaunchKernelGGL(matmul_batch_kernel<kWeightF32>, grid, dim3(kMmThreads), 0, stream, a);
    else if (a.w_type == kWeightQ8_0 && a.xh) {
        hipLaunchKernelGGL(matmul_split_x_kernel<false>, dim3(a.batch), dim3(kMmThreads), 0, stream, a);
        hipLaunchKernelGGL(matmul_f16_kernel<kWeightQ8_0>, grid, dim3(kMmThreads), 0, stream, a);
    } else if (a.w_type == kWeightQ4_K && a.xh && a.xsum && a.in_dim % 256 == 0) {
        hipLaunchKernelGGL(matmul_split_x_kernel<true>, dim3(a.batch), dim3(kMmThreads), 0, stream, a);
        hipLaunchKernelGGL(matmul_f16_kernel<kWeightQ4_K>, grid, dim3(kMmThreads), 0, stream, a);
    } else if (a.w_type == kWeightQ6_K && a.xh && a.in_dim % 256 == 0) {
        hipLaunchKernelGGL(matmul_split_x_kernel<false>, dim3(a.batch), dim3(kMmThreads), 0, stream, a);
        hipLaunchKernelGGL(matmul_f16_kernel<kWeightQ6_K>, grid, dim3(kMmThreads), 0, stream, a);
    } else if (a.w_type == kWeightQ8_0)
        hipLaunchKernelGGL(matmul_batch_kernel<kWeightQ8_0>, grid, dim3(kMmThreads), 0, stream, a);
    else if (a.w_type == kWeightQ4_K && a.in_dim % 256 == 0)
        hipLaunchKernelGGL(matmul_batch_kernel<kWeightQ4_K>, grid, dim3(kMmThreads), 0, stream, a);
    else if (a.w_type == kWeightQ6_K && a.in_dim % 256 == 0)
        hipLaunchKernelGGL(matmul_batch_kernel<kWeightQ6_K>, grid, dim3(kMmThreads), 0, stream, a);
    else
        return hipErrorInvalidValue;
    if (a.splits > 1) launch_reduce(a, stream);
    return hipGetLastError();
}

}  // namespace gsp
