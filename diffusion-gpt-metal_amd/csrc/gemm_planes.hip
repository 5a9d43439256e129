// Large GEMMs on 16-bit MFMA over operands split into planes (gfx950):
//
//   out[i,j] = sum_c A[i,c] * B[j,c]  (+ bias[j], or += out)
//
// The forward (A = X, B = deq(W)), dX (A = dY, B = deq(W)^T) and
// dW (A = dY^T, B = X^T) of the linears are all this product; only where
// element (row, c) of an operand lies differs (struct Src).
//
// Every operand row is scaled by a power of two that brings its largest
// element into [2^14, 2^15), and split into two f16 pieces x = h + 2^-12 l with
// h = f16(x), l = f16(2^12 (x - h)): 22 bits and a sign, an error of at most
// 2^-23 |x| for elements down to 2^-27 of the row's largest, 2^-20 |x| down to
// 2^-31, and 2^-51 of the largest below that (l unscaled: 2^-39 of the largest below
// 2^-15). Rows of which more than one nonzero element in 16 lies below 2^-31 of
// the largest are flagged: their outputs are computed from the original
// operands in fp32. So a row keeps fp32's error where one huge element meets
// zeros, or where the factors of the other operand grow as the row's elements
// fall. What is left out: a row with few such elements against one that is zero
// at nearly all others; its sum, below 2^-31 of what the row can give, then has
// their error. (Every such element counted, the products of three
// normal values that a SwiGLU backward returns would flag a row in most calls, at
// 130 us each.)
// The product is hh + hl + lh on v_mfma_f32_32x32x16_f16 with
// fp32 accumulation; the omitted ll is below 2^-22 of the product. Products of
// f16 pieces are exact, and the matrix unit rounds its sum once per 8 of them
// (measured: 4.0e-7 in the 2-norm over 4096 random products, the figure of a
// CPU chain rounded every 8), so hh, summed by itself, has half the roundings
// of v_mfma_f32_16x16x4_f32; hl and lh go to a second accumulator whose
// roundings are 2^-11 of those. Against 64 bits, the fp32 MFMA kernels first:
// 2048 x 14336 x 4096 5.3e-7, 4.0e-7; dX and dW of 2048 x 4096 x 4096 5.7e-7
// and 4.2e-7, 4.1e-7 and 3.1e-7; dW over 12288 rows 1.0e-6, 2.8e-7.
// A forward whose codes come in groups of whole 32-c stages keeps them as one
// plane (integers of 8 bits, exact in f16): h and l of x against the codes,
// summed per group, and the sum goes to the accumulator times the group's
// scale. Two products instead of three, and no rounding of code * scale: 1.4e-7
// for the first case above.
// There l stays against the codes times 2^-12 (exact in f16).
// Rows with an infinity or NaN are flagged too (an infinity times a low piece
// of the other sign would be NaN).
//
// What it gains: v_mfma_f32_16x16x4_f32 peaks at 157 TFLOP/s and its kernels
// here ran at 50-57; three f16 products per fp32 product at 2.5 PFLOP/s peak at
// 833, two at 1250. Measured, those kernels first: 2048 x 14336 x 4096 int4
// 4816 and 466 us (517 TFLOP/s), 517 x 4100 x 4128 int8 320 and 80, dX + dW of 2048 x
// 4096 x 4096 2416 and 418, forward + dX + dW of fp32 12288 x 1536 x 384 779 and 302.
// (l unscaled, 2^-39 of a row's largest: 451, 76, 417 and 300; the codes' packed
// multiplies are the difference. The figures beside the rules below are of that form.)
// What bounds it: the power the matrix unit draws. With zeros for data the
// GEMM of 4096 x 4096 x 4096 takes 225 us instead of 320 (the clock stays up);
// interleaving the LDS reads with the MFMAs, raising their priority, one wave
// per SIMD with twice the tile (64 instead of 85 LDS bytes per clock), all
// within 3% of this form.
//
// Three launches: the rows' largest elements, the split into planes, the
// GEMM; a fourth adds the parts of tiles that are cut along c (struct Plan).
// dX and dW of one linear share them (struct Pair).
//
// Plane layout: 32 rows x 16 c of a plane are one fragment of the MFMA, 1 KB
// in lane order (lane l: row l % 32, c = 8 (l / 32) .. + 7), and a 32-row
// block's h and l fragments of the same 16 c are neighbours. So every
// direct-to-LDS load and every LDS read is 1 KB contiguous (whole cache lines,
// no bank conflicts, no swizzle), the rows are padded to whole tiles and c to
// whole stages with zeros, and the GEMM has no bounds checks before its stores.
//
// GEMM: WM x WN waves, each MT x NT tiles of 32 x 32. A ring of three or four
// stages of 16 or 32 c; a step waits for the next stage by count, meets the other waves,
// issues the loads of the stage two or three ahead and reads the next stage's
// fragments into registers while the MFMAs of the current one run, so the
// load latency, the LDS latency and the barrier are off the MFMAs' path.
#include "common.hpp"

#include <algorithm>

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kFlag = 1 << 30;      // an exponent: the row's elements do not fit the pieces
constexpr float kLow = 1.0f / 4096.0f;   // of l
constexpr int kMaxParts = 16;       // row chunks of a column-maximum pass

// One operand: element (r, c) of R x C.
struct Src {
    const void* p;
    const float* scale;   // codes: per (weight row, group)
    int64_t ld;           // elements from one stored row to the next
    int R, C;
    int bits;             // 32, 8, 4
    int col;              // 0: p[r * ld + c], 1: p[c * ld + r] (codes: the weight row is c)
    int G, groups;        // codes
    int vec;              // 8 consecutive stored elements can be loaded at once
};

struct Operand {
    Src s;
    uint8_t* planes;
    uint32_t* part;       // largest |element| (its bits) of each row: parts x width
    int parts, width;
    int* exps;            // row scale 2^e, or kFlag; then (each [32 rb]) how many of the row's elements
                          // lie below 2^-31 of its largest but are not zero, and how many are zero (of codes, none counts)
    int rb, kb;           // 32-row blocks and 16-c blocks written (padded)
    float* scales;        // codes kept as one plane: their scales 2^e, [group][32 rb]
    int gpad;             // groups written there (padded)
    int blocks;           // workgroups of its split
};

__device__ __forceinline__ float code_at(const void* p, int bits, int64_t i) {
    if (bits == 8) return float(static_cast<const int8_t*>(p)[i]);
    const uint8_t b = static_cast<const uint8_t*>(p)[i >> 1];
    return float(int8_t((i & 1) ? b : uint8_t(b << 4)) >> 4);
}

__device__ __forceinline__ float elem(const Src& s, int r, int c) {
    const int64_t i = s.col ? int64_t(c) * s.ld + r : int64_t(r) * s.ld + c;
    if (s.bits == 32) return static_cast<const float*>(s.p)[i];
    const int64_t si = s.col ? int64_t(c) * s.groups + r / s.G : int64_t(r) * s.groups + c / s.G;
    return code_at(s.p, s.bits, i) * s.scale[si];
}

// ---- launch 1: largest |element| of each row ---------------------------------------
// One pass over fp32 data (X, dY, W, or the scales that bound the codes'
// weights). Rows stored contiguously: lpr lanes per row. Rows stored across:
// a block takes 64 of them and one of `parts` chunks of c.
struct MaxArg {
    const float* p;
    int64_t ld;
    int R, C, col, lpr, parts, blocks;
    uint32_t* out;
    int* counts;     // of the split, cleared: n_counts of them
    int n_counts;
};

__device__ __forceinline__ void max_part(const MaxArg& a, int block) {
    const int t = threadIdx.x;
    for (int i = block * 256 + t; i < a.n_counts; i += a.blocks * 256) a.counts[i] = 0;
    if (!a.col) {
        const int per = 256 / a.lpr;
        const int r = block * per + t / a.lpr, l = t % a.lpr;
        uint32_t m = 0;
        if (r < a.R) {
            const float* row = a.p + int64_t(r) * a.ld;
            const bool vec = (a.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(a.p) & 15) == 0;
            int c = 0;
            if (vec) {
                const int n4 = a.C >> 2;
#pragma unroll 4
                for (int i = l; i < n4; i += a.lpr) {
                    const u32x4 v = reinterpret_cast<const u32x4*>(row)[i] & 0x7fffffffu;
                    m = max(max(m, max(v[0], v[1])), max(v[2], v[3]));
                }
                c = n4 << 2;
            }
            for (int i = c + l; i < a.C; i += a.lpr) m = max(m, __float_as_uint(row[i]) & 0x7fffffffu);
        }
        for (int off = a.lpr >> 1; off >= 1; off >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), off)));
        if (r < a.R && l == 0) a.out[r] = m;
        return;
    }
    __shared__ uint32_t sh[4][64];
    const int nb = (a.R + 63) / 64;
    const int r = (block % nb) * 64 + (t & 63), part = block / nb;
    const int64_t chunk = (int64_t(a.C) + a.parts - 1) / a.parts;
    const int64_t c1 = min(int64_t(a.C), (part + 1) * chunk);
    uint32_t m = 0;
    if (r < a.R) {
#pragma unroll 8
        for (int64_t c = part * chunk + (t >> 6); c < c1; c += 4)
            m = max(m, __float_as_uint(a.p[c * a.ld + r]) & 0x7fffffffu);
    }
    sh[t >> 6][t & 63] = m;
    __syncthreads();
    if (t < 64 && r < a.R) a.out[int64_t(part) * a.R + r] = max(max(sh[0][t], sh[1][t]), max(sh[2][t], sh[3][t]));
}

// The operands of up to two products.
struct MaxArgs {
    MaxArg m[4];
};

__global__ __launch_bounds__(256) void row_max_kernel(MaxArgs a) {
    int b = int(blockIdx.x);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (b < a.m[i].blocks) {
            max_part(a.m[i], b);
            return;
        }
        b -= a.m[i].blocks;
    }
}

// ---- launch 2: the split ---------------------------------------------------------------
// Elements (r, c .. c + 7), zero outside R x C.
template <int BITS, int COL>
__device__ __forceinline__ void load8(const Src& s, int r, int c, float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.0f;
    if (r >= s.R || c >= s.C) return;
    if constexpr (COL) {
        const int n = min(8, s.C - c);
        if constexpr (BITS == 32) {
            const float* p = static_cast<const float*>(s.p) + int64_t(c) * s.ld + r;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j < n) v[j] = p[j * s.ld];
        } else {
            const float* sp = s.scale + int64_t(c) * s.groups + r / s.G;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j < n) v[j] = code_at(s.p, BITS, int64_t(c + j) * s.ld + r) * sp[j * s.groups];
        }
    } else if (s.vec && c + 8 <= s.C) {
        const int64_t i = int64_t(r) * s.ld + c;
        if constexpr (BITS == 32) {
            const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(s.p) + i);
            const float4 x = p[0], y = p[1];
            v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
            v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
        } else {
            const float sc = s.scale[int64_t(r) * s.groups + c / s.G];   // G % 8 == 0
            if constexpr (BITS == 8) {
                const int2 q = *reinterpret_cast<const int2*>(static_cast<const int8_t*>(s.p) + i);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[j] = float((q.x << (24 - 8 * j)) >> 24) * sc;
                    v[4 + j] = float((q.y << (24 - 8 * j)) >> 24) * sc;
                }
            } else {
                const int q = *reinterpret_cast<const int*>(static_cast<const uint8_t*>(s.p) + (i >> 1));
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = float((q << (28 - 4 * j)) >> 28) * sc;
            }
        }
    } else {
        const int n = min(8, s.C - c);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j < n) v[j] = elem(s, r, c + j);
    }
}

// 8 codes as f16 (exact), zero outside R x C.
template <int BITS>
__device__ __forceinline__ f16x8 codes8(const Src& s, int r, int c) {
    f16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (r >= s.R || c >= s.C) return v;   // C is a multiple of 32
    const int64_t i = int64_t(r) * s.ld + c;
    if (!s.vec) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = _Float16(code_at(s.p, BITS, i + j));
    } else if constexpr (BITS == 8) {
        const int2 q = *reinterpret_cast<const int2*>(static_cast<const int8_t*>(s.p) + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = _Float16((q.x << (24 - 8 * j)) >> 24);
            v[4 + j] = _Float16((q.y << (24 - 8 * j)) >> 24);
        }
    } else {
        const int q = *reinterpret_cast<const int*>(static_cast<const uint8_t*>(s.p) + (i >> 1));
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = _Float16((q << (28 - 4 * j)) >> 28);
    }
    return v;
}

// 2^e brings a row of largest magnitude `bits` below 2^15 (extra: the codes'
// bits above the scale); e <= 126 keeps the factor a normal number.
__device__ __forceinline__ int row_exp(uint32_t bits, int extra) {
    if (bits >= 0x7f800000u) return kFlag;
    return bits == 0 ? 0 : min(126, 14 + 127 - int(bits >> 23) - extra);
}

__device__ __forceinline__ float exp_factor(int e) {
    return __uint_as_float(uint32_t((e == kFlag ? 0 : e) + 127) << 23);
}

template <int BITS>
__device__ __forceinline__ void codes_part(const Operand& o, int block) {
    const int chunks = (o.kb + 15) / 16;
    const int rb = block / chunks, chunk = block % chunks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = rb * 32 + (lane & 31), h = lane >> 5;
    f16x8 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = codes8<BITS>(o.s, r, (chunk * 16 + u * 4 + wave) * 16 + 8 * h);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int kb = chunk * 16 + u * 4 + wave;
        if (kb < o.kb) *reinterpret_cast<f16x8*>(o.planes + (int64_t(rb) * o.kb + kb) * 1024 + lane * 16) = v[u];
    }
    if (chunk != 0) return;
    const int e = row_exp(r < o.s.R ? o.part[r] : 0u, BITS == 8 ? 7 : 3);
    if (wave == 0 && h == 0) o.exps[r] = e;   // its counts stay at 0: codes are exact
    const float f = exp_factor(e);
    for (int g = threadIdx.x >> 5; g < o.gpad; g += 8)
        o.scales[int64_t(g) * (o.rb * 32) + r] =
            r < o.s.R && g < o.s.groups ? o.s.scale[int64_t(r) * o.s.groups + g] * f : 0.0f;
}

template <int BITS, int COL>
__device__ __forceinline__ void split_part(const Operand& o, int block) {
    const int chunks = (o.kb + 15) / 16;
    const int rb = block / chunks, chunk = block % chunks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = rb * 32 + (lane & 31), h = lane >> 5;
    float v[4][8];
#pragma unroll
    for (int u = 0; u < 4; ++u) load8<BITS, COL>(o.s, r, (chunk * 16 + u * 4 + wave) * 16 + 8 * h, v[u]);
    const int at = BITS != 32 && COL ? r / o.s.G : r;
    uint32_t m = 0;
    if (r < o.s.R) {
        if constexpr (COL) {
            uint32_t p[kMaxParts];   // all in flight together
#pragma unroll
            for (int i = 0; i < kMaxParts; ++i) p[i] = o.part[int64_t(min(i, o.parts - 1)) * o.width + at];
#pragma unroll
            for (int i = 0; i < kMaxParts; ++i) m = max(m, p[i]);
        } else {
            m = o.part[r];
        }
    }
    const int e = row_exp(m, BITS == 32 ? 0 : (BITS == 8 ? 7 : 3));
    if (chunk == 0 && wave == 0 && h == 0) o.exps[r] = e;
    const float f = exp_factor(e);
    int far = 0, zeros = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int kb = chunk * 16 + u * 4 + wave;
        if (kb >= o.kb) continue;
        f16x8 hi, lo;
        uint32_t least = ~0u, most = 0;   // of |x| minus one: a zero is the largest
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = v[u][j] * f;
            const uint32_t k = (__float_as_uint(x) << 1) - 1;
            least = min(least, k);
            most = max(most, k);
            hi[j] = _Float16(x);
            lo[j] = _Float16((x - float(hi[j])) * (1.0f / kLow));
        }
        uint8_t* out = o.planes + (int64_t(rb) * o.kb + kb) * 2048 + lane * 16;
        *reinterpret_cast<f16x8*>(out) = hi;
        *reinterpret_cast<f16x8*>(out + 1024) = lo;
        if (least < 2 * 0x37000000u - 1 || (BITS == 32 && most == ~0u)) {   // below 2^-17, or zero
            const int n = min(8, o.s.C - kb * 16 - 8 * h);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                zeros += BITS == 32 && j < n && v[u][j] == 0.0f;
                far += v[u][j] != 0.0f && fabsf(v[u][j] * f) < 0x1p-17f;
            }
        }
    }
    // From e = 114 on, fp32's own last bit (2^-149) is a multiple of l's (2^-36).
    if (far && e < 114) atomicAdd(o.exps + 32 * o.rb + r, far);
    if (zeros && r < o.s.R) atomicAdd(o.exps + 64 * o.rb + r, zeros);
}

__device__ __forceinline__ void split_any(const Operand& o, int block) {
    if (o.scales) {
        if (o.s.bits == 8) codes_part<8>(o, block);
        else codes_part<4>(o, block);
    } else if (o.s.col) {
        if (o.s.bits == 32) split_part<32, 1>(o, block);
        else if (o.s.bits == 8) split_part<8, 1>(o, block);
        else split_part<4, 1>(o, block);
    } else {
        if (o.s.bits == 32) split_part<32, 0>(o, block);
        else if (o.s.bits == 8) split_part<8, 0>(o, block);
        else split_part<4, 0>(o, block);
    }
}

struct Operands {
    Operand o[4];
};

__global__ __launch_bounds__(256) void split_kernel(Operands a) {
    int b = int(blockIdx.x), i = 0;
    while (i < 3 && b >= a.o[i].blocks) b -= a.o[i++].blocks;
    const Operand o = i == 0 ? a.o[0] : i == 1 ? a.o[1] : i == 2 ? a.o[2] : a.o[3];
    split_any(o, b);
}

// ---- launch 3: the GEMM ----------------------------------------------------------------
struct PlaneArgs {
    const uint8_t *A, *B;
    const int *ea, *eb;   // as Operand::exps, of rows_a and rows_b rows
    int rows_a, rows_b;
    Src sa, sb;           // the original operands, for flagged rows
    const float* bias;
    float *out, *out2;    // columns from cols1 on go to out2; rows of ldo floats
    int ldo, cols1;
    int M, N;             // rows of A, rows of B
    int stages, chunk;    // parts are whole chunks of stages
    const float* scales;  // CODE: [group][scale_ld]
    int scale_ld, gps;    // stages of a group
    int tiles_m, tiles_n;
    int full, per_full;   // tiles computed whole, and how many of them an XCD takes
    int splits, per_part; // the other tiles: c in `splits` parts, and an XCD's share of the parts
    float* part;          // their sums: [tile - full][part][wave][float4 of the accumulators][lane]
    int accumulate;
};

constexpr int GROUP_M = 8;   // tile rows of the order inside an XCD

// CODE: B is one plane of codes. A stage is KB blocks of 16 c, in LDS per
// 32-row block of A its KB h and l fragments, of B its KB fragments (one or
// two planes), then (CODE) the tile's scales of the stage's group.
template <int WM_, int WN_, int MT_, int NT_, bool CODE_, int RING_>
struct Geo {
    static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_, RING = RING_;
    static constexpr bool CODE = CODE_;
    static constexpr int WAVES = WM * WN;
    static constexpr int TM = WM * MT * 32, TN = WN * NT * 32;
    static constexpr int KB = CODE ? 2 : 1;
    static constexpr int AU = 2 * KB, BU = 2;   // 1 KB units of a 32-row block (BU: 2 planes, or 2 blocks of c)
    static constexpr int UNITS = TM / 32 * AU + TN / 32 * BU;
    static constexpr int UPW = UNITS / WAVES;
    static constexpr int LOADS = UPW + (CODE ? 1 : 0);   // loads a wave issues for a stage
    static constexpr int STAGE = UNITS * 1024 + (CODE ? TN * 4 : 0);
    static constexpr int LDS = RING * STAGE + (TM + TN) * 4;
    static_assert(UNITS % WAVES == 0 && LDS <= 160 * 1024, "");
};

__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// Codes times kLow.
__device__ __forceinline__ u32x4 lowered(u32x4 b) {
    return __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, b) * _Float16(kLow));
}

// Up to two products in one launch: the workgroups of the first, then those
// of the second, which fill what the first leaves idle.
struct PlaneGroup {
    PlaneArgs p[2];
    int first;   // workgroups of p[0]
};

// p[second] of the kernel's one argument, read where it is used (a copy of the
// chosen one would keep 50 more scalar registers than there are).
__device__ __forceinline__ const PlaneArgs& args_of(bool second) {
    return ((const PlaneArgs*)__builtin_amdgcn_kernarg_segment_ptr())[second ? 1 : 0];
}

// The exponent of row r of C elements, or kFlag.
__device__ __forceinline__ int row_scale(const int* exps, int rows, int r, int C) {
    return exps[rows + r] > (C - exps[2 * rows + r]) / 16 ? kFlag : exps[r];
}

// Tile L of the order: groups of GROUP_M tile rows, column after column, so
// that the tiles an XCD runs at once share their strips in its L2.
__device__ __forceinline__ void tile_at(const PlaneArgs& a, int L, int& ti, int& tj) {
    const int group = L / (GROUP_M * a.tiles_n);
    const int gm = min(GROUP_M, a.tiles_m - group * GROUP_M);
    const int within = L - group * GROUP_M * a.tiles_n;
    ti = group * GROUP_M + within % gm;
    tj = within / gm;
}

// Stores one 32 x 32 tile of sums at (r0, c0), but for the elements of flagged
// rows and columns; true where there are any. Lane l holds column l % 32,
// rows 8 (e / 4) + 4 (l / 32) + e % 4. ea: the rows' exponents from r0.
__device__ __forceinline__ bool store_tile(const PlaneArgs& a, f32x16 acc, int r0, int c0, const int* ea, int eb) {
    const int lane = threadIdx.x & 63, q = lane >> 5;
    const int M = a.M, N = a.N, ld = a.ldo, c = c0 + (lane & 31);
    float* const base = c0 < a.cols1 ? a.out : a.out2 - a.cols1;   // cols1 is a multiple of 32, or N
    const float bv = a.bias ? a.bias[min(c, N - 1)] : 0.0f;
    int er[16];
    bool odd = eb == kFlag;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        er[e] = ea[8 * (e >> 2) + 4 * q + (e & 3)];
        odd = odd || er[e] == kFlag;
        acc[e] = ldexpf(acc[e], -(er[e] + eb));
    }
    if (a.bias) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] += bv;
    }
    float* o = base + int64_t(r0 + 4 * q) * ld + c;
    if (r0 + 32 <= M && c0 + 32 <= N && !__any(odd)) {
        if (a.accumulate) {
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] += o[int64_t(8 * (e >> 2) + (e & 3)) * ld];
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) o[int64_t(8 * (e >> 2) + (e & 3)) * ld] = acc[e];
        return false;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int r = r0 + 8 * (e >> 2) + 4 * q + (e & 3);
        if (r < M && c < N && er[e] != kFlag && eb != kFlag) {
            float* at = o + int64_t(8 * (e >> 2) + (e & 3)) * ld;
            *at = a.accumulate ? *at + acc[e] : acc[e];
        }
    }
    return __any(odd);
}

__device__ __forceinline__ void load_any(const Src& s, int r, int c, float (&v)[8]) {
    if (s.col) {
        if (s.bits == 32) load8<32, 1>(s, r, c, v);
        else if (s.bits == 8) load8<8, 1>(s, r, c, v);
        else load8<4, 1>(s, r, c, v);
    } else {
        if (s.bits == 32) load8<32, 0>(s, r, c, v);
        else if (s.bits == 8) load8<8, 0>(s, r, c, v);
        else load8<4, 0>(s, r, c, v);
    }
}

// The flagged elements of one 32 x 32 tile, from the operands in fp32
// (v_mfma_f32_32x32x2_f32, a lane 8 consecutive c of its row and column). One
// token of NaN gradients flags every row of dW, so this has to run at about the
// rate of the fp32 MFMA kernels: dX + dW of 2048 x 2048 x 2048 with such a token
// 859 us, those kernels 659, a chain of scalar fmas per element 42810.
__device__ __forceinline__ void exact_tile(const PlaneArgs& a, int r0, int c0, const int* ea, int eb) {
    const int lane = threadIdx.x & 63, q = lane >> 5;
    f32x16 acc = {};
    for (int k = 0; k < a.sa.C; k += 32) {
        float x[2][8], y[2][8];
        // Kept opaque: the addresses of every form that load_any has would
        // otherwise be computed before the loop, in registers that the
        // kernel's other waves then go without.
        int rx = r0 + (lane & 31), ry = c0 + (lane & 31);
        asm volatile("" : "+v"(rx), "+v"(ry));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            load_any(a.sa, rx, k + 16 * u + 8 * q, x[u]);
            load_any(a.sb, ry, k + 16 * u + 8 * q, y[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[u][j], y[u][j], acc, 0, 0, 0);
    }
    const int c = c0 + (lane & 31);
    if (c >= a.N) return;
    float* const o = (c0 < a.cols1 ? a.out : a.out2 - a.cols1) + c;
    const float bv = a.bias ? a.bias[c] : 0.0f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int lr = 8 * (e >> 2) + 4 * q + (e & 3), r = r0 + lr;
        if (r >= a.M || (ea[lr] != kFlag && eb != kFlag)) continue;
        float* at = o + int64_t(r) * a.ldo;
        const float v = acc[e] + bv;
        *at = a.accumulate ? *at + v : v;
    }
}

template <typename T>   // two waves to a SIMD: the 8 of a workgroup, or two workgroups of 4
__global__ __launch_bounds__(64 * T::WAVES, 2) void plane_gemm_kernel(PlaneGroup g) {
    const bool second = int(blockIdx.x) >= g.first;
    const PlaneArgs& a = args_of(second);
    constexpr int MT = T::MT, NT = T::NT, RING = T::RING;
    constexpr bool CODE = T::CODE;
    extern __shared__ __align__(16) uint8_t smem[];
    int* exps = reinterpret_cast<int*>(smem + RING * T::STAGE);
    const int t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / T::WN, wn = wave % T::WN;

    // XCD x (workgroups x, x + 8, ...) takes a run of the whole tiles, then a
    // run of the parts.
    const int b = int(blockIdx.x) - (second ? g.first : 0), nfull = a.per_full * 8;
    const bool whole = b < nfull;
    int L, part = 0;
    if (whole) {
        L = (b & 7) * a.per_full + (b >> 3);
        if (L >= a.full) return;
    } else {
        const int u = ((b - nfull) & 7) * a.per_part + ((b - nfull) >> 3);
        L = a.full + u / a.splits;
        part = u % a.splits;
        if (L >= a.tiles_m * a.tiles_n) return;
    }
    const int chunks = a.stages / a.chunk;
    const int first = whole ? 0 : a.chunk * (part * chunks / a.splits);
    const int end = whole ? a.stages : a.chunk * ((part + 1) * chunks / a.splits);
    int ti, tj;
    tile_at(a, L, ti, tj);
    const int m0 = ti * T::TM, n0 = tj * T::TN;

    for (int i = t; i < T::TM + T::TN; i += 64 * T::WAVES)
        exps[i] = i < T::TM ? row_scale(a.ea, a.rows_a, m0 + i, a.sa.C)
                                : row_scale(a.eb, a.rows_b, n0 + i - T::TM, a.sa.C);

    // This wave's loads of a stage: units wave * UPW ..; first A's (AU to a
    // 32-row block), then B's. A stage further is AU or BU KB further.
    const uint8_t* src[T::UPW];
    uint32_t step_bytes[T::UPW];
    const int64_t strip_a = int64_t(a.stages) * T::AU * 1024, strip_b = int64_t(a.stages) * T::BU * 1024;
#pragma unroll
    for (int i = 0; i < T::UPW; ++i) {
        const int u = wave * T::UPW + i, v = u - T::TM / 32 * T::AU;
        const bool isa = v < 0;
        src[i] = isa ? a.A + (m0 / 32 + u / T::AU) * strip_a + (u % T::AU) * 1024
                     : a.B + (n0 / 32 + v / T::BU) * strip_b + (v % T::BU) * 1024;
        step_bytes[i] = (isa ? T::AU : T::BU) * 1024u;
    }
    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(smem));
    const uint32_t scol = uint32_t((n0 + (t & (T::TN - 1))) * 4);   // CODE: this lane's column of the scales
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    auto issue = [&](int s, int slot) {   // past the last stage: the last one again, never read
        const uint32_t at = uint32_t(min(s, end - 1));
        const uint32_t lds = lds0 + uint32_t(slot) * T::STAGE + uint32_t(wave * T::UPW) * 1024u;
#pragma unroll
        for (int i = 0; i < T::UPW; ++i)
            asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds + i * 1024),
                         "v"(at * (T::AU == T::BU ? T::AU * 1024u : step_bytes[i]) + uint32_t(lane) * 16u), "s"(src[i])
                         : "memory", "m0");
        if constexpr (CODE)   // waves past the tile's columns load them again
            asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(
                             lds0 + uint32_t(slot) * T::STAGE + T::UNITS * 1024u +
                             uint32_t(wave % (T::TN / 64)) * 256u),
                         "v"(at / uint32_t(a.gps) * uint32_t(a.scale_ld) * 4u + scol), "s"(a.scales)
                         : "memory", "m0");
    };
#pragma clang diagnostic pop

    // Fragments of 16 c: A's h and l; B's h and l, or (CODE) its codes.
    struct Frags {
        u32x4 a[MT][2], b[NT][CODE ? 1 : 2];
    };
    auto fetch = [&](int slot, int kb, Frags& f) {
        const uint8_t* st = smem + slot * T::STAGE + lane * 16;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                f.a[i][p] = *reinterpret_cast<const u32x4*>(st + ((wm * MT + i) * T::AU + 2 * kb + p) * 1024);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int p = 0; p < (CODE ? 1 : 2); ++p)
                f.b[j][p] = *reinterpret_cast<const u32x4*>(
                    st + (T::TM / 32 * T::AU + (wn * NT + j) * T::BU + kb + p) * 1024);
    };
    // The matrix unit rounds once per 8 products. Two planes: hh is summed
    // apart from hl + lh (2^12 too large), whose roundings are then 2^-11 of
    // those of the sum.
    // CODE: `low` is the sum of the group, x as h and l against the codes, and
    // goes to acc times the group's scale.
    f32x16 acc[MT][NT], low[MT][NT];
    const f32x16 zero = {};
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = low[i][j] = zero;
    auto multiply = [&](const Frags& f, bool fresh) {
        if constexpr (CODE) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        low[i][j] = mfma(f.a[i][p], p == 0 ? f.b[j][0] : lowered(f.b[j][0]),
                                         fresh && p == 0 ? zero : low[i][j]);
        } else {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma(f.a[i][0], f.b[j][0], acc[i][j]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) low[i][j] = mfma(f.a[i][0], f.b[j][CODE ? 0 : 1], low[i][j]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) low[i][j] = mfma(f.a[i][1], f.b[j][0], low[i][j]);
        }
    };

    __syncthreads();   // exps; and no plain load is in flight when the counted ones start
#pragma unroll
    for (int i = 0; i < RING - 1; ++i) issue(first + i, i);
    Frags f0, f1;
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((RING - 2) * T::LOADS) : "memory");
    fetch(0, 0, f0);
    // Start of step s: its first fragments are in registers. Stage s + 1 has
    // landed once at most the loads of the stages after it are in flight, and
    // this wave's reads of stage s - 1 are done once at most those of stage s are
    // (two planes: the 2 (MT + NT) 16-byte reads since the last step; CODE reads
    // both stages in a step, in an order that is the compiler's). Waited for here:
    // the MFMAs that use them may be scheduled past the barrier. Past it both
    // hold for every wave, and the ring slot of stage s - 1 is free. Two planes with
    // no read left open: 1 to 1.6% slower.
    int slot = 0;   // of stage s
    auto start = [&](int s) {
        constexpr int reads = CODE ? 0 : 2 * (MT + NT);
        static_assert(reads < 16, "lgkmcnt has four bits");
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)\n\ts_barrier" ::"n"((RING - 3) * T::LOADS), "n"(reads)
                     : "memory");
        issue(s + RING - 1, slot == 0 ? RING - 1 : slot - 1);
    };
    auto next = [&](int v) { return v == RING - 1 ? 0 : v + 1; };
    if constexpr (CODE) {
        float sc[NT];   // of the stage's group
        auto step = [&](int s, bool fresh) {
            start(s);
            fetch(slot, 1, f1);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                sc[j] = *reinterpret_cast<const float*>(smem + slot * T::STAGE + T::UNITS * 1024 +
                                                        ((wn * NT + j) * 32 + (lane & 31)) * 4);
            multiply(f0, fresh);
            slot = next(slot);
            fetch(slot, 0, f0);
            multiply(f1, false);
        };
        auto fold = [&] {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = __builtin_fmaf(sc[j], low[i][j][e], acc[i][j][e]);
        };
        if (a.gps == 1) {
            for (int s = first; s < end; ++s) {
                step(s, true);
                fold();
            }
        } else {
            for (int s = first; s < end;) {
                const int stop = s + a.gps;
                step(s, true);
                for (++s; s < stop; ++s) step(s, false);
                fold();
            }
        }
    } else {
        auto step = [&](int s, const Frags& cur, Frags& nxt) {
            start(s);
            slot = next(slot);
            fetch(slot, 0, nxt);
            multiply(cur, false);
        };
        for (int s = first; s < end; s += 2) {
            step(s, f0, f1);
            step(s + 1, f1, f0);
        }
    }
    // No direct-to-LDS load may outlive the workgroup's LDS.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    uint32_t odd = 0;   // tiles with flagged elements
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if constexpr (!CODE) {
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = __builtin_fmaf(low[i][j][e], kLow, acc[i][j][e]);
            }
            if (whole) {
                const int lr = (wm * MT + i) * 32, lc = (wn * NT + j) * 32;
                if (store_tile(a, acc[i][j], m0 + lr, n0 + lc, exps + lr, exps[T::TM + lc + (lane & 31)]))
                    odd |= 1u << (i * NT + j);
            } else {
                f32x4* o = reinterpret_cast<f32x4*>(a.part) +
                           ((int64_t(L - a.full) * a.splits + part) * T::WAVES + wave) * (MT * NT * 4 * 64) +
                           (i * NT + j) * 4 * 64 + lane;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e * 64] = f32x4{acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2],
                                      acc[i][j][4 * e + 3]};
            }
        }
    for (; odd; odd &= odd - 1) {
        const int k = __builtin_ctz(odd), lr = (wm * MT + k / NT) * 32, lc = (wn * NT + k % NT) * 32;
        exact_tile(a, m0 + lr, n0 + lc, exps + lr, exps[T::TM + lc + (lane & 31)]);
    }
}

// The parts of the split tiles, added in order: one wave per 32 x 32 tile.
template <typename T>
__global__ __launch_bounds__(256, 7) void part_sum_kernel(PlaneGroup g) {
    constexpr int SUB = T::MT * T::NT;
    const bool second = int(blockIdx.x) >= g.first;
    const PlaneArgs& a = args_of(second);
    const int lane = threadIdx.x & 63;
    const int u = (int(blockIdx.x) - (second ? g.first : 0)) * 4 + (threadIdx.x >> 6);   // (tile, wave, subtile)
    const int sub = u % SUB, wave = u / SUB % T::WAVES, tile = u / (SUB * T::WAVES);
    int ti, tj;
    tile_at(a, a.full + tile, ti, tj);
    const int r0 = ti * T::TM + (wave / T::WN * T::MT + sub / T::NT) * 32;
    const int c0 = tj * T::TN + (wave % T::WN * T::NT + sub % T::NT) * 32;
    if (r0 >= a.M || c0 >= a.N) return;
    const int row_e = row_scale(a.ea, a.rows_a, r0 + (lane & 31), a.sa.C);   // used after the sums
    const int eb = row_scale(a.eb, a.rows_b, c0 + (lane & 31), a.sa.C);
    f32x16 acc;
    for (int p = 0; p < a.splits; ++p) {
        const f32x4* o = reinterpret_cast<const f32x4*>(a.part) +
                         ((int64_t(tile) * a.splits + p) * T::WAVES + wave) * (SUB * 4 * 64) + sub * 4 * 64 + lane;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const f32x4 v = o[e * 64];
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[4 * e + k] = p == 0 ? v[k] : acc[4 * e + k] + v[k];
        }
    }
    __shared__ int exps[4][32];   // a wave's own
    int* const ea = exps[threadIdx.x >> 6];
    if (lane < 32) ea[lane] = row_e;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (store_tile(a, acc, r0, c0, ea, eb)) exact_tile(a, r0, c0, ea, eb);
}

template <typename T>
int launch_gemm(dgm_gpu* g, const PlaneArgs* p, int n) {
    auto kern = plane_gemm_kernel<T>;
    if (T::LDS > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
        if (e != hipSuccess)
            return dgm::fail(g, DGM_ERR_HIP, "plane gemm: cannot reserve %d bytes of LDS: %s", T::LDS,
                             hipGetErrorString(e));
    }
    PlaneGroup grp{};
    unsigned wgs[2] = {}, sums[2] = {};
    for (int i = 0; i < n; ++i) {
        grp.p[i] = p[i];
        wgs[i] = unsigned(p[i].per_full + p[i].per_part) * 8u;
        sums[i] = unsigned(p[i].tiles_m * p[i].tiles_n - p[i].full) * unsigned(T::MT * T::NT * T::WAVES / 4);
    }
    grp.first = int(wgs[0]);
    hipLaunchKernelGGL(kern, dim3(wgs[0] + wgs[1]), dim3(64 * T::WAVES), T::LDS, g->stream, grp);
    if (sums[0] + sums[1] > 0) {
        grp.first = int(sums[0]);
        hipLaunchKernelGGL(part_sum_kernel<T>, dim3(sums[0] + sums[1]), dim3(256), 0, g->stream, grp);
    }
    return DGM_OK;
}

// Tiles of 8 waves (128 x 256, 256 x 128: one workgroup per CU) and of 4
// (128 x 128: two).
using Wide = Geo<2, 4, 2, 2, false, 4>;
using Tall = Geo<4, 2, 2, 2, false, 4>;
using Small = Geo<2, 2, 2, 2, false, 4>;
using CodeWide = Geo<2, 4, 2, 2, true, 4>;
using CodeTall = Geo<4, 2, 2, 2, true, 3>;
using CodeSmall = Geo<2, 2, 2, 2, true, 3>;

struct Tile {
    int tm, tn, slots;   // slots: workgroups a CU holds (build.py checks the registers for it)
};
constexpr Tile kTiles[] = {{128, 256, 1}, {256, 128, 1}, {128, 128, 2}};

int64_t round_up(int64_t v, int64_t to) { return (v + to - 1) / to * to; }

// How a product is cut into tiles and parts, and its time in microseconds.
// Fitted to runs on 256 CUs, one 16-c block in every busy slot: 128 x 256 tiles
// of two planes take 0.36 us with few CUs busy and 0.62 us with all (the clock
// falls under the matrix load), 128 x 128 tiles 0.26 us alone on a CU and 0.70
// us for the two of a CU; codes two thirds of that, and 0.10 us where the
// block's stage ends a group. A round also fills and drains (4 us). Where the
// tiles leave the last round partly empty, that round's tiles are cut along c:
// the sums of the parts cost a launch and their traffic, mostly in the
// Infinity Cache. Whole against cut, same run, the better tile of each: int8
// 517 x 4100 x 4128 104 and 76 us, int4 256 x 4096 x 4096 89 and 48, fp32 512
// x 4096 x 4096 105 and 94, fp32 1536 x 384 x 12288 226 and 98; whole is better
// at fp32 2048 x 2048 x 2048 (70 against 81).
struct Plan {
    int tile;
    int64_t tiles, full;   // all; computed whole (the others in `splits` parts)
    int splits;
    double us;
};

// One round of `units` workgroups, each `blocks` of 16 c long. fold: codes, the
// share of a block that ends a group's stage (0: two planes).
double round_us(int tile, int64_t units, int cus, double blocks, double fold) {
    const double busy = std::min(1.0, double(units) / cus);
    const bool pair = units > cus;   // two 128 x 128 tiles to a CU
    double block;
    if (fold > 0.0) block = (tile < 2 ? 0.24 + 0.17 * busy : pair ? 0.47 : 0.24) + 0.10 * fold;
    else block = tile < 2 ? 0.36 + 0.26 * busy : pair ? 0.70 : 0.26 + 0.10 * busy;
    return 4.0 + block * blocks;
}

double rounds_us(int tile, int64_t units, int cus, double blocks, double fold) {
    const int64_t slots = int64_t(cus) * kTiles[tile].slots;
    const int64_t rest = units % slots;
    return double(units / slots) * round_us(tile, slots, cus, blocks, fold) +
           (rest ? round_us(tile, rest, cus, blocks, fold) : 0.0);
}

// uniform: all tiles whole or all of them cut.
Plan plan_for(int64_t M, int64_t N, int64_t blocks, int chunk, double fold, bool uniform, int cus) {
    Plan best{0, 0, 0, 1, 1e30};
    for (int tile = 0; tile < 3; ++tile) {
        const Tile& t = kTiles[tile];
        const int64_t tiles = int64_t(dgm::ceil_div(M, t.tm)) * dgm::ceil_div(N, t.tn);
        const double us = rounds_us(tile, tiles, cus, double(blocks), fold);
        if (us < best.us) best = Plan{tile, tiles, tiles, 1, us};
        const int64_t slots = int64_t(cus) * t.slots, full = uniform ? 0 : tiles / slots * slots,
                      cut = tiles - full;
        for (int s = 2; s <= 8 && cut > 0 && blocks / s >= std::max(16, chunk); ++s) {
            const double part = double(dgm::ceil_div(blocks / chunk, s)) * chunk;
            const double cut_us = (full ? rounds_us(tile, full, cus, double(blocks), fold) : 0.0) +
                                  rounds_us(tile, cut * s, cus, part, fold) + 4.0 +
                                  double(cut) * s * t.tm * t.tn * 8.0 / 8e6;
            if (cut_us < best.us) best = Plan{tile, tiles, full, s, cut_us};
        }
    }
    return best;
}

// The tile for two products of two planes in one launch, each cut (or not) as
// it would be by itself, so that each element is the same sums either way.
// Units are dealt in order to `slots` workgroups: the first product's fill
// whole rounds and part of one, the second's start where a slot is free.
int pair_tile(const int64_t (&M)[2], const int64_t (&N)[2], const int64_t (&blocks)[2], const int (&splits)[2],
              int cus) {
    int best = 0;
    double best_us = 1e30;
    for (int tile = 0; tile < 3; ++tile) {
        const Tile& t = kTiles[tile];
        const int64_t slots = int64_t(cus) * t.slots;
        int64_t n[2];
        for (int i = 0; i < 2; ++i)
            n[i] = int64_t(dgm::ceil_div(M[i], t.tm)) * dgm::ceil_div(N[i], t.tn) * splits[i];
        const int64_t all = std::min(n[0] + n[1], slots);
        const double a = round_us(tile, all, cus, double(blocks[0]) / splits[0], 0.0);
        const double b = round_us(tile, all, cus, double(blocks[1]) / splits[1], 0.0);
        const int64_t rest = n[0] % slots;
        double early = double(n[0] / slots) * a, late = early + a, us = rest ? late : early;
        if (n[1] > 64 * slots) {   // many rounds: the throughput
            us = early + (double(rest) * a + double(n[1]) * b) / double(slots);
        } else {
            for (int64_t left = n[1]; left > 0;) {
                const bool e = early <= late || rest == 0;
                double& clock = e ? early : late;
                clock += b;
                us = std::max(us, clock);
                left -= e ? slots - rest : rest;
            }
        }
        for (int i = 0; i < 2; ++i)
            if (splits[i] > 1) us += double(n[i]) * t.tm * t.tn * 8.0 / 8e6;
        if (us < best_us) {
            best_us = us;
            best = tile;
        }
    }
    return best;
}

Operand operand(const Src& s, int tile, int64_t blocks) {
    Operand o{};
    o.s = s;
    o.rb = int(round_up(s.R, tile) / 32);
    o.kb = int(blocks);
    o.parts = s.col ? int(std::min<int64_t>(kMaxParts, std::max<int64_t>(1, s.C / 64))) : 1;
    o.width = s.col && s.bits != 32 ? s.groups : s.R;
    o.blocks = o.rb * int(dgm::ceil_div(o.kb, 16));
    return o;
}

MaxArg max_arg(const Operand& o) {
    MaxArg m{};
    const Src& s = o.s;
    const bool codes = s.bits != 32;
    m.p = codes ? s.scale : static_cast<const float*>(s.p);
    m.ld = codes ? s.groups : s.ld;
    m.col = s.col;
    m.parts = o.parts;
    m.out = o.part;
    m.counts = o.exps + 32 * o.rb;
    m.n_counts = 64 * o.rb;
    m.R = o.width;
    m.C = codes && !s.col ? s.groups : s.C;
    m.lpr = m.C >= 512 ? 64 : m.C >= 128 ? 16 : 8;
    m.blocks = s.col ? int(dgm::ceil_div(m.R, 64)) * o.parts : int(dgm::ceil_div(m.R, 256 / m.lpr));
    return m;
}

// The forward keeps the codes as one plane where a stage of 32 c lies in one
// group: 2 products instead of 3, and half the bytes of B's planes. Same run, three
// products first: 2048 x 14336 x 4096 in groups of 128 669 -> 457 us, 4096 x
// 4096 x 4096 380 -> 263, in groups of 32 (a fold every stage) 388 -> 302, 517
// x 4100 x 4128 in groups of 32 94 -> 77.
bool one_plane(const Src& b) { return b.bits != 32 && !b.col && b.G % 32 == 0; }

// out[M, N] (+)= A B^T (+ bias), columns from cols1 on in out2.
struct Product {
    Src a, b;
    const float* bias;
    float *out, *out2;
    int ldo, cols1;
    bool accumulate;
};

// How one product, or two of two planes, are cut, and where their pieces lie
// in the plane buffer.
struct Layout {
    bool code;             // one product, its B one plane
    int gps, chunk, t;     // t: of kTiles
    int64_t M[2], N[2], blocks[2], tiles[2], full[2];
    int splits[2];
    Operands op;
    size_t bytes, at[4][4], parts[2];
};

// False: not for these kernels.
bool layout(const Product* q, int n, int cus, Layout& l) {
    l = Layout{};
    const bool code = l.code = n == 1 && one_plane(q[0].b);
    l.gps = code ? q[0].b.G / 32 : 1;
    l.chunk = code ? l.gps : 2;
    for (int i = 0; i < n; ++i) {
        l.M[i] = q[i].a.R;
        l.N[i] = q[i].b.R;
        l.blocks[i] = code ? q[i].a.C / 16 : round_up(dgm::ceil_div(q[i].a.C, 16), 2);
    }
    // The backward's products are cut alike in one call and in two.
    const bool uniform = n == 2 || q[0].a.col || q[0].b.col;
    for (int i = 0; i < n; ++i) {
        const Plan plan = plan_for(l.M[i], l.N[i], l.blocks[i], code ? l.chunk * 2 : l.chunk, code ? 1.0 / l.gps : 0.0,
                                   uniform, cus);
        l.t = plan.tile;
        l.full[i] = plan.full;
        l.splits[i] = plan.splits;
    }
    if (n == 2) l.t = pair_tile(l.M, l.N, l.blocks, l.splits, cus);
    const Tile& tile = kTiles[l.t];
    auto take = [&](int64_t size) {
        const size_t here = l.bytes;
        l.bytes += size_t(round_up(size, 256));
        return here;
    };
    for (int i = 0; i < n; ++i) {
        l.tiles[i] = int64_t(dgm::ceil_div(l.M[i], tile.tm)) * dgm::ceil_div(l.N[i], tile.tn);
        if (l.tiles[i] > (1 << 24)) return false;   // 32-bit tile numbers
        if (n == 2) l.full[i] = l.splits[i] == 1 ? l.tiles[i] : 0;
        l.op.o[2 * i] = operand(q[i].a, tile.tm, l.blocks[i]);
        l.op.o[2 * i + 1] = operand(q[i].b, tile.tn, l.blocks[i]);
        if (code) l.op.o[1].gpad = int(l.blocks[0] / 2 / l.gps);
        for (int k = 2 * i; k < 2 * i + 2; ++k) {
            const Operand& o = l.op.o[k];
            // The GEMM's 32-bit offsets of a stage (of two planes, 2 KB to a
            // 16-c block) and of a group's scales.
            if (int64_t(o.kb) * 2048 > (int64_t(1) << 32) || int64_t(o.gpad) * o.rb * 128 > (int64_t(1) << 32))
                return false;
            l.at[k][0] = take(int64_t(o.rb) * o.kb * (o.gpad ? 1024 : 2048));
            l.at[k][1] = take(int64_t(o.rb) * 3 * 128);
            l.at[k][2] = take(int64_t(o.parts) * o.width * 4);
            l.at[k][3] = take(int64_t(o.gpad) * o.rb * 128);
        }
        l.parts[i] = take((l.tiles[i] - l.full[i]) * l.splits[i] * tile.tm * tile.tn * 4);
    }
    return true;
}

// kNotFused, launching nothing, without a plane buffer. dry: only whether
// there is one.
int run(dgm_gpu* g, const Product* q, int n, bool dry = false) {
    Layout l;
    if (!layout(q, n, g->num_cus, l)) return dgm::kNotFused;
    uint8_t* ws = dgm::planes_buffer(g, l.bytes);
    if (!ws) return dgm::kNotFused;
    if (dry) return DGM_OK;
    const Tile& tile = kTiles[l.t];
    Operands& op = l.op;
    MaxArgs mx{};
    PlaneArgs p[2] = {};
    unsigned max_blocks = 0, split_blocks = 0;
    for (int k = 0; k < 2 * n; ++k) {
        Operand& o = op.o[k];
        o.planes = ws + l.at[k][0];
        o.exps = reinterpret_cast<int*>(ws + l.at[k][1]);
        o.part = reinterpret_cast<uint32_t*>(ws + l.at[k][2]);
        if (o.gpad) o.scales = reinterpret_cast<float*>(ws + l.at[k][3]);
        mx.m[k] = max_arg(o);
        max_blocks += unsigned(mx.m[k].blocks);
        split_blocks += unsigned(o.blocks);
    }
    hipLaunchKernelGGL(row_max_kernel, dim3(max_blocks), dim3(256), 0, g->stream, mx);
    hipLaunchKernelGGL(split_kernel, dim3(split_blocks), dim3(256), 0, g->stream, op);
    for (int i = 0; i < n; ++i) {
        const Operand &a = op.o[2 * i], &b = op.o[2 * i + 1];
        PlaneArgs& r = p[i];
        r.A = a.planes;
        r.B = b.planes;
        r.ea = a.exps;
        r.eb = b.exps;
        r.rows_a = a.rb * 32;
        r.rows_b = b.rb * 32;
        r.sa = q[i].a;
        r.sb = q[i].b;
        r.bias = q[i].bias;
        r.out = q[i].out;
        r.out2 = q[i].out2;
        r.ldo = q[i].ldo;
        r.cols1 = q[i].cols1;
        r.M = int(l.M[i]);
        r.N = int(l.N[i]);
        r.stages = int(l.code ? l.blocks[i] / 2 : l.blocks[i]);
        r.chunk = l.chunk;
        r.scales = b.scales;
        r.scale_ld = b.rb * 32;
        r.gps = l.gps;
        r.tiles_m = a.rb * 32 / tile.tm;
        r.tiles_n = b.rb * 32 / tile.tn;
        r.full = int(l.full[i]);
        r.per_full = (r.full + 7) / 8;
        r.splits = l.splits[i];
        r.per_part = (int(l.tiles[i] - l.full[i]) * l.splits[i] + 7) / 8;
        r.part = reinterpret_cast<float*>(ws + l.parts[i]);
        r.accumulate = q[i].accumulate;
    }
    if (l.code) {
        if (l.t == 0) return launch_gemm<CodeWide>(g, p, n);
        if (l.t == 1) return launch_gemm<CodeTall>(g, p, n);
        return launch_gemm<CodeSmall>(g, p, n);
    }
    if (l.t == 0) return launch_gemm<Wide>(g, p, n);
    if (l.t == 1) return launch_gemm<Tall>(g, p, n);
    return launch_gemm<Small>(g, p, n);
}

Src dense(const float* p, int R, int C, int64_t ld, int col) {
    Src s{};
    s.p = p;
    s.ld = ld;
    s.R = R;
    s.C = C;
    s.bits = 32;
    s.col = col;
    s.G = 1;
    s.vec = (ld & 3) == 0 && dgm::aligned(p, 16);
    return s;
}

// The weights [N, K]: rows n over k (col 0), or rows k over n (col 1).
Src weights(int bits, const void* W, const float* scale, const dgm_GemmP* p, int col) {
    const int N = int(p->N), K = int(p->K);
    if (bits == 32) return dense(static_cast<const float*>(W), col ? K : N, col ? N : K, K, col);
    Src s{};
    s.p = W;
    s.scale = scale;
    s.ld = K;
    s.R = col ? K : N;
    s.C = col ? N : K;
    s.bits = bits;
    s.col = col;
    s.G = int(p->qGroup);
    s.groups = K / s.G;
    s.vec = K % 8 == 0 && s.G % 8 == 0 && dgm::aligned(W, 8);
    return s;
}

}  // namespace

namespace dgm {

// Where three or four launches and the planes' traffic cost less than they
// save: the planes take 20 us and more before the last sum. Measured on int8
// in groups of 32, us on the fp32 MFMA kernels and on these (G = 2^30 products):
//   forward, K below 1280: 1024 x 768 x 768 (0.56 G) 24.7 and 27.7, 1100 x 1100 x
//     576 (0.65 G) 27.8 and 31.7, 8192 x 192 x 480 (0.70 G) 34.8 and 33.4 (int4
//     29.9 and 33.4), 256 x 4096 x 1024 (1 G) 45.5 and 30.6 (int4 38.4 and 29.1);
//   forward, longer K, where those have few tiles: 256 x 512 x 2240 (0.27 G) 22.0
//     and 28.8, 256 x 1024 x 2048 (0.5 G) 40.6 and 29.3 but fp32 24.9 and 27.5,
//     128 x 2304 x 2048 (0.56 G) 58.0 and 30.9, fp32 35.2 and 31.3;
//   up to 64 rows are the decode's; 70 x 4096 x 4096 110.6 and 55.7.
bool planes_pay_fwd(int64_t M, int64_t N, int64_t K) {
    return M > 64 && N >= 128 && K >= 128 &&
           double(M) * double(N) * double(K) >= double(K >= 1280 ? int64_t(9) << 26 : int64_t(3) << 28);
}

// One line for dX, dW and both, which give the same bits (gemmBwd's promise),
// where neither alone loses (in groups of 32, us as above: both, dX, dW):
//   512 x 1024 x 1024 (0.5 G) 41.4 and 40.1, 21.6 and 33.7, 18.5 and 25.3;
//   1024 x 768 x 768 (0.56 G) 48.8 and 39.3, 23.2 and 33.5, 24.7 and 26.0;
//   640 x 1536 x 768 (0.70 G) 68.4 and 44.9, 35.6 and 35.1, 30.7 and 29.6;
//   70 x 4096 x 4096 (1.09 G) 138 and 83, 70 and 58, 56 and 32.
bool planes_pay_bwd(int64_t M, int64_t N, int64_t K) {
    return M > 64 && N >= 128 && K >= 128 && double(M) * double(N) * double(K) >= double(int64_t(11) << 26);
}

namespace {

// Y [M, N], or Y and Y2 [M, N / 2].
Product forward_of(int bits, const void* W, const float* scale, const float* X, const float* bias, float* Y,
                   const dgm_GemmP* p, float* Y2) {
    const int N = int(p->N), cols1 = Y2 ? N / 2 : N;
    return Product{dense(X, int(p->M), int(p->K), p->K, 0), weights(bits, W, scale, p, 0), p->hasBias ? bias : nullptr,
                   Y, Y2, cols1, cols1, false};
}

int backward_of(Product* q, int bits, const void* W, const float* scale, const float* dY, const float* X, float* dX,
                float* dW, const dgm_GemmP* p, bool accumulate) {
    const int M = int(p->M), N = int(p->N), K = int(p->K);
    int n = 0;
    if (dX) q[n++] = Product{dense(dY, M, N, N, 0), weights(bits, W, scale, p, 1), nullptr, dX, nullptr, K, K, false};
    if (dW) q[n++] = Product{dense(dY, N, M, N, 1), dense(X, K, M, K, 1), nullptr, dW, nullptr, K, K, accumulate};
    return n;
}

size_t layout_bytes(const Product* q, int n, int cus) {
    Layout l;
    return layout(q, n, cus, l) ? l.bytes : 0;
}

}  // namespace

size_t planes_bytes(int64_t M, int64_t N, int64_t K, int cus, bool forward, bool backward) {
    const dgm_GemmP p{uint32_t(M), uint32_t(N), uint32_t(K), 0u, 1u, 0u, 0u, 0u};
    size_t b = 0;
    forward = forward && K <= (int64_t(1) << 25);   // longer ones layout() refuses
    Product q[2];
    if (forward && planes_pay_fwd(M, N, K)) {
        q[0] = forward_of(32, nullptr, nullptr, nullptr, nullptr, nullptr, &p, nullptr);   // two planes of any weights
        b = layout_bytes(q, 1, cus);
        for (int64_t stages = K / 32, gps = 1; K % 32 == 0 && gps <= stages; ++gps) {   // one plane, every group
            if (stages % gps != 0) continue;
            dgm_GemmP pg = p;
            pg.qGroup = uint32_t(32 * gps);
            q[0] = forward_of(8, nullptr, nullptr, nullptr, nullptr, nullptr, &pg, nullptr);
            b = std::max(b, layout_bytes(q, 1, cus));
        }
    }
    if (backward && planes_pay_bwd(M, N, K)) {
        float* const some = reinterpret_cast<float*>(16);   // asked for, never read
        for (int both = 0; both < 3; ++both) {
            const int n = backward_of(q, 32, nullptr, nullptr, nullptr, nullptr, both != 1 ? some : nullptr,
                                      both != 0 ? some : nullptr, &p, false);
            b = std::max(b, layout_bytes(q, n, cus));
        }
    }
    return b;
}

int planes_fwd(dgm_gpu* g, int bits, const void* W, const float* scale, const float* X, const float* bias,
               float* Y, const dgm_GemmP* p, float* Y2) {
    const Product q = forward_of(bits, W, scale, X, bias, Y, p, Y2);
    return run(g, &q, 1, X == nullptr);
}

int planes_bwd(dgm_gpu* g, int bits, const void* W, const float* scale, const float* dY, const float* X, float* dX,
               float* dW, const dgm_GemmP* p, bool accumulate) {
    Product q[2];
    const int n = backward_of(q, bits, W, scale, dY, X, dX, dW, p, accumulate);
    return run(g, q, n, dY == nullptr);
}

}  // namespace dgm
