// The half pipe of the product kernels: fp32 operands as two fp16 numbers each, three matrix instructions per product.
//
// An operand x is scaled by a power of two s (exact) that puts the largest element of its matrix into [2^14, 2^15) and
// written as x s = h + r / 2^11 with h = fp16(x s) and r = fp16((x s - h) 2^11): 22 to 23 significant bits as long as
// x s >= 2^-14, that is for elements down to 2^-28 of the matrix's largest, and an error of at most 2^-51 of that largest
// element below.  A product is then  h_a h_b + (r_a h_b + h_a r_b) 2^-11  (r_a r_b is below 2^-24 of it), the leading
// terms and the rests summed in fp32 accumulators of their own by v_mfma_f32_32x32x16_f16.
//
// Against the split of the bf16 pipe (three bf16 numbers, six matrix instructions, one accumulator): half of the matrix
// instructions, two thirds of the LDS traffic and less split arithmetic, and a third of the roundings in the accumulators;
// but one bit less of every fourth element.  Relative 2-norm error against float64, bf16 split and this: Gaussian
// matrices k = 128 1.6e-7 and 1.1e-7, 1024 4.9e-7 and 2.2e-7, 3072 8.7e-7 and 3.6e-7; I + 1e-3 noise, where one element makes
// most of a sum, k = 256 1.5e-7 and 1.6e-7, 512 2.2e-7 both, 1024 3.1e-7 both; inverse fourth roots of condition 20, order
// 128 5.3e-7 and 6.1e-7, 256 5.9e-7 and 5.8e-7, 768 9.1e-7 and 7.4e-7: hence kHalfLeastK.  Rates: 99 x 1024^3 1.05 -> 0.76 ms
// (203 -> 279 TFLOP/s), 24 x 2304^3 2.81 -> 1.98 ms (296).
//
// The scale needs the largest element beforehand (qtensor_gemm_ranges): a bound that the caller knows, what the launch
// that wrote the matrix found (amax_out), or a pass over it.  It only has to be near: while the tiles are split the
// kernel keeps the largest element of every tile row it reads, and a tile with a row that overflows its scale, is not finite,
// or is small against the scale (below 2^-24 of the largest element) is multiplied out again by the bf16 split.
//
// That does not see small elements in a row that holds large ones as well -- a small row of B or column of A, all rows of
// which are fine: with a diagonal A a row of B at 2^-40 of the others is a row of the result with 11 bits, at 2^-52 it is
// zero.  So the launches that look for the largest element look for the smallest *piece* too: four elements of a row or
// up to eight of a column next to each other (of the result of a product: four, eight rows apart), of which the largest
// counts, and only pieces that are not zero.  Where every piece is at least 2^-28 of the bound an element is kept to 2^-23
// of the largest next to it, in its row and in its column; a matrix with a smaller one is left to the bf16 split as a
// whole (half_scale).  A piece, not an element, because some element of a matrix of noise is always that small: of a
// Gaussian one of 768 x 3072 every eighth has one, of one with elements of 1e-6 of its diagonal all do.  Launches hand the
// reciprocal on, the largest over the pieces ("fineness"), so that vectors of zeroes are what to begin with.  A caller that
// gives bounds alone vouches for the pieces.
#pragma once
#include "qt_common.h"
#include "qt_offsets.h"

namespace qt {
namespace {

typedef _Float16 qt_f16x8 __attribute__((ext_vector_type(8)));
constexpr int HK = 32;                                 // k per LDS tile: a 128-byte line of a row whose k is contiguous
constexpr int kHalfLeastK = 256;
constexpr float kRestScale = 2048.0f;

// An operand tile of ROWS rows in LDS: [h, r][16 k][8 k][row][8 fp16].  A lane's fragment (8 consecutive k of one row) is
// one 16-byte read, 32 rows read 512 contiguous bytes.  The paddings put the four groups of 8 k of a row 32 bytes apart
// in the banks, so that the 8-byte stores of eight lanes that hold one row (HalfKContig) do not meet (with 64 bytes they
// did: 146 cycles more per operand tile, 804 -> 750 us for 99 x 1024^3).
template <int ROWS> struct HalfLayout {
    static constexpr int kEight = ROWS * 16 + 32, kSub = 2 * kEight, kPlane = 2 * kSub, kOperand = 2 * kPlane;      // bytes
};

// Two elements: scaled, split, and folded into `top` (NaN is not seen there, but makes its row of the result NaN).
// Written out because the compiler's own form of the subtraction converts h once more, with an instruction of half rate.
__device__ __forceinline__ void halve_pair(float a, float b, float s, uint32_t &h, uint32_t &r, float &top) {
    const float x = a * s, y = b * s;
    float u, v;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(h) : "v"(x), "v"(y));
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[0,0,1]" : "=v"(u) : "v"(x), "v"(h));
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(v) : "v"(y), "v"(h));
    u *= kRestScale;
    v *= kRestScale;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(u), "v"(v));
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(top) : "v"(x), "v"(y), "v"(top));
}

// Loaders.  `prepare` fixes a thread's place; `fetch` issues part q of four of a k tile's loads into one of SETS register
// sets; `pair` splits two elements of a set and stores to LDS whenever a store's worth is together (`ahead` starts the table
// look-ups of a pair of codes); `tops` folds the largest (scaled) elements seen into one word per tile row.  Rows beyond
// the matrix are clamped into it.
// Source of a k tile: base addresses in scalar registers.
struct DenseSource { __amdgpu_buffer_rsrc_t at; };
struct QuantSource { __amdgpu_buffer_rsrc_t codes, absmax; };

// k contiguous (element (row, k) at base[row * ld + k], rows 16-byte aligned): eight lanes take the 128 bytes of a row,
// a thread the rows t / 8 + 32 i.
template <int ROWS, int SETS>
struct HalfKContig {
    static constexpr int VEC = ROWS / 32, kPairs = 2 * VEC;
    float v[SETS][4 * VEC];
    float top[VEC];
    uint32_t off[VEC];
    uint32_t h[2], r[2];
    __device__ __forceinline__ void prepare(int ld, int row0, int rows) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            off[i] = (uint32_t)((min(row0 + (int)(threadIdx.x >> 3) + 32 * i, rows - 1) - row0) * ld + (threadIdx.x & 7) * 4) * 4u;
            top[i] = 0.0f;
        }
    }
    __device__ __forceinline__ void ahead(int, int) {}
    __device__ __forceinline__ void patch(unsigned char *, int, float) const {}
    __device__ __forceinline__ void fetch(const DenseSource &src, int set, int q) {
#pragma unroll
        for (int i = q * VEC / 4; i < (q + 1) * VEC / 4; ++i) {
            const qt_u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(src.at, (int)off[i], 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[set][4 * i + e] = __uint_as_float(x[e]);
        }
    }
    __device__ __forceinline__ void pair(unsigned char *operand, int set, float s, int p) {
        using L = HalfLayout<ROWS>;
        halve_pair(v[set][2 * p], v[set][2 * p + 1], s, h[p & 1], r[p & 1], top[p >> 1]);
        if (p & 1) {
            const int c = threadIdx.x & 7;
            unsigned char *at = operand + (c >> 2) * L::kSub + ((c >> 1) & 1) * L::kEight + (threadIdx.x >> 3) * 16 + (c & 1) * 8 + (p >> 1) * 32 * 16;
            *reinterpret_cast<uint2 *>(at) = make_uint2(h[0], h[1]);
            *reinterpret_cast<uint2 *>(at + L::kPlane) = make_uint2(r[0], r[1]);
        }
    }
    __device__ __forceinline__ void tops(uint32_t *s_top) const {
#pragma unroll
        for (int i = 0; i < VEC; ++i) atomicMax(s_top + (threadIdx.x >> 3) + 32 * i, __float_as_uint(top[i]));
    }
};

// Row index contiguous (element (row, k) at base[k * ld + row]): a thread takes row t % ROWS and the k of part t / ROWS,
// one word per load, a wave's load covers 64 consecutive words.
template <int ROWS, int SETS>
struct HalfRowContig {
    static constexpr int PER = ROWS * HK / 256, kPairs = PER / 2;
    float v[SETS][PER];
    float top;
    uint32_t off, step;                                // this thread's first word, and one k further (the same for all)
    uint32_t h[4], r[4];
    __device__ __forceinline__ void prepare(int ld, int row0, int rows) {
        const int row = threadIdx.x & (ROWS - 1), part = threadIdx.x / ROWS;
        off = (uint32_t)(part * PER * ld + (min(row0 + row, rows - 1) - row0)) * 4u;
        step = (uint32_t)ld * 4u;
        top = 0.0f;
    }
    __device__ __forceinline__ void ahead(int, int) {}
    __device__ __forceinline__ void patch(unsigned char *, int, float) const {}
    __device__ __forceinline__ void fetch(const DenseSource &src, int set, int q) {
#pragma unroll
        for (int j = q * PER / 4; j < (q + 1) * PER / 4; ++j)
            v[set][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(src.at, (int)off, (int)(j * step), 0));
    }
    __device__ __forceinline__ void pair(unsigned char *operand, int set, float s, int p) {
        using L = HalfLayout<ROWS>;
        halve_pair(v[set][2 * p], v[set][2 * p + 1], s, h[p & 3], r[p & 3], top);
        if ((p & 3) == 3) {
            const int row = threadIdx.x & (ROWS - 1), eight = threadIdx.x / ROWS * (PER / 8) + (p >> 2);
            unsigned char *at = operand + (eight >> 1) * L::kSub + (eight & 1) * L::kEight + row * 16;
            *reinterpret_cast<qt_u32x4 *>(at) = qt_u32x4{h[0], h[1], h[2], h[3]};
            *reinterpret_cast<qt_u32x4 *>(at + L::kPlane) = qt_u32x4{r[0], r[1], r[2], r[3]};
        }
    }
    __device__ __forceinline__ void tops(uint32_t *s_top) const { atomicMax(s_top + (threadIdx.x & (ROWS - 1)), __float_as_uint(top)); }
};

// Quantized square matrices (order x order, flat layout), expanded while they are split.  A pair costs the look-ups of two
// codes (issued one pair ahead: their latency lies behind a matrix instruction) and two products besides its split.
// `patch` writes the exact diagonal over what the codes gave, on the few k tiles that hold a part of it: by the thread that
// wrote those elements, behind all its pairs (a branch that touches neither loads nor accumulators; a loop body of its own
// for those tiles had the compiler spill the accumulators).
__device__ __forceinline__ void patch_element(unsigned char *at, int plane, float x) {
    const _Float16 h = (_Float16)x;
    *reinterpret_cast<_Float16 *>(at) = h;
    *reinterpret_cast<_Float16 *>(at + plane) = (_Float16)((x - (float)h) * kRestScale);
}

// Left factor, k along the matrix rows: a thread takes 16 (128 tile rows) or 8 consecutive codes of one row.
template <int ROWS, int BITS, int SETS>
struct HalfQuantLeft {
    static constexpr int PER = ROWS * HK / 256, PARTS = HK / PER, kPairs = PER / 2, WORDS = PER * BITS / 32;
    uint32_t w[SETS][WORDS];
    float amax[SETS];
    float dval, top;
    uint32_t code_off, amax_off;
    int row;                                           // the tile row's matrix row less this thread's first k
    const float *table;
    float c[2][2];
    uint32_t h[4], r[4];
    __device__ __forceinline__ void prepare(const float *code, const float *diag, int order, int bs_shift, int row0, float s) {
        const int part = threadIdx.x % PARTS;
        table = code;
        row = min(row0 + (int)(threadIdx.x / PARTS), order - 1);
        code_off = code_offset<BITS>(row, part * PER, order);
        amax_off = absmax_offset(row, order, bs_shift);
        dval = diag != nullptr ? diag[row] : 0.0f;
        row -= part * PER;
        top = fabsf(dval) * s;
    }
    __device__ __forceinline__ void fetch(const QuantSource &src, int set, int q) {
        if (q == 0) {
            if constexpr (WORDS == 1) w[set][0] = __builtin_amdgcn_raw_buffer_load_b32(src.codes, (int)code_off, 0, 0);
            else if constexpr (WORDS == 2) {
                const qt_u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(src.codes, (int)code_off, 0, 0);
                w[set][0] = x.x; w[set][1] = x.y;
            } else {
                const qt_u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(src.codes, (int)code_off, 0, 0);
                w[set][0] = x.x; w[set][1] = x.y; w[set][2] = x.z; w[set][3] = x.w;
            }
            amax[set] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(src.absmax, (int)amax_off, 0, 0));
        }
    }
    __device__ __forceinline__ void ahead(int set, int p) {
        if (p >= kPairs) return;
        if constexpr (BITS == 4) {
            const uint32_t byte = w[set][p >> 2] >> (8 * (p & 3));
            c[p & 1][0] = table[(byte >> 4) & 15u];
            c[p & 1][1] = table[byte & 15u];
        } else {
            const uint32_t two = w[set][p >> 1] >> (16 * (p & 1));
            c[p & 1][0] = table[two & 255u];
            c[p & 1][1] = table[(two >> 8) & 255u];
        }
    }
    __device__ __forceinline__ void pair(unsigned char *operand, int set, float s, int p) {
        using L = HalfLayout<ROWS>;
        float a = c[p & 1][0] * amax[set], b = c[p & 1][1] * amax[set];
        ahead(set, p + 1);
        halve_pair(a, b, s, h[p & 3], r[p & 3], top);
        if ((p & 3) == 3) {
            const int eight = threadIdx.x % PARTS * (PER / 8) + (p >> 2);
            unsigned char *at = operand + (eight >> 1) * L::kSub + (eight & 1) * L::kEight + threadIdx.x / PARTS * 16;
            *reinterpret_cast<qt_u32x4 *>(at) = qt_u32x4{h[0], h[1], h[2], h[3]};
            *reinterpret_cast<qt_u32x4 *>(at + L::kPlane) = qt_u32x4{r[0], r[1], r[2], r[3]};
        }
    }
    __device__ __forceinline__ void patch(unsigned char *operand, int k0, float s) const {
        using L = HalfLayout<ROWS>;
        const int d = row - k0;                        // the element on the diagonal, if in 0 .. PER - 1
        if ((unsigned)d < (unsigned)PER) {
            const int eight = threadIdx.x % PARTS * (PER / 8) + (d >> 3);
            patch_element(operand + (eight >> 1) * L::kSub + (eight & 1) * L::kEight + threadIdx.x / PARTS * 16 + (d & 7) * 2, L::kPlane, dval * s);
        }
    }
    __device__ __forceinline__ void tops(uint32_t *s_top) const { atomicMax(s_top + threadIdx.x / PARTS, __float_as_uint(top)); }
};

// Right factor, k along the matrix columns: a thread takes the codes of two neighbouring columns (one byte, or two) of 8
// (128 tile rows) or 4 consecutive matrix rows, so that nothing has to be turned around.  (It reads the whole word they lie
// in, as two or four lanes do: what a byte load returns the compiler masks again, at once, and waits for it.)  Of every eight lanes four begin with the even column and four with the odd one: their 16-byte stores then
// fall into different banks.
template <int ROWS, int BITS, int SETS>
struct HalfQuantRight {
    static constexpr int LANES = ROWS / 2, GROUPS = 256 / LANES, PER = HK / GROUPS, kPairs = PER;      // k per thread; pairs: first column's, then the second's
    uint32_t w[SETS][PER];
    float amax[SETS][PER];
    float dval[2], top[2];
    uint32_t code_off, amax_off, code_step, amax_step, at[2];
    int column, way;                                   // the first column less this thread's first k, and how far the second is (1 or -1)
    const float *table;
    float c[2][2];
    uint32_t h[4], r[4];
    __device__ __forceinline__ void prepare(const float *code, const float *diag, int order, int bs_shift, int row0, float s) {
        const int lane = threadIdx.x % LANES, group = threadIdx.x / LANES;
        const int even = min(row0 + 2 * lane, order - 2);
        table = code;
        way = (lane >> 2) & 1 ? -1 : 1;
        column = even + (way < 0 ? 1 : 0);
        code_step = code_offset<BITS>(1, 0, order);
        amax_step = absmax_offset(1, order, bs_shift);
        code_off = (uint32_t)(group * PER) * code_step + ((uint32_t)(even * BITS / 8) & ~3u);
        // a column's place in the word: 4 bits: the even column in the high half of its byte
        const uint32_t first = ((uint32_t)(even * BITS / 8) & 3u) * 8;
        at[0] = first + (BITS == 4 ? (way > 0 ? 4 : 0) : (way > 0 ? 0 : 8));
        at[1] = first + (BITS == 4 ? (way > 0 ? 0 : 4) : (way > 0 ? 8 : 0));
        amax_off = (uint32_t)(group * PER) * amax_step + (uint32_t)(even >> bs_shift) * 4u;
        dval[0] = diag != nullptr ? diag[column] : 0.0f;
        dval[1] = diag != nullptr ? diag[column + way] : 0.0f;
        column -= group * PER;
        top[0] = fabsf(dval[0]) * s;
        top[1] = fabsf(dval[1]) * s;
    }
    __device__ __forceinline__ void fetch(const QuantSource &src, int set, int q) {
#pragma unroll
        for (int j = q * PER / 4; j < (q + 1) * PER / 4; ++j) {
            w[set][j] = __builtin_amdgcn_raw_buffer_load_b32(src.codes, (int)code_off, (int)(j * code_step), 0);
            amax[set][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(src.absmax, (int)amax_off, (int)(j * amax_step), 0));
        }
    }
    __device__ __forceinline__ void ahead(int set, int p) {
        if (p >= kPairs) return;
        const int second = p / (PER / 2), j = p % (PER / 2) * 2;
        c[p & 1][0] = table[(w[set][j] >> at[second]) & ((1u << BITS) - 1)];
        c[p & 1][1] = table[(w[set][j + 1] >> at[second]) & ((1u << BITS) - 1)];
    }
    __device__ __forceinline__ void pair(unsigned char *operand, int set, float s, int p) {
        using L = HalfLayout<ROWS>;
        constexpr int HALF = PER / 2, WORDS = PER / 2;                       // packed words per column
        const int second = p / HALF, j = p % HALF * 2;
        float a = c[p & 1][0] * amax[set][j], b = c[p & 1][1] * amax[set][j + 1];
        ahead(set, p + 1);
        halve_pair(a, b, s, h[p % WORDS], r[p % WORDS], top[second]);
        if (p % WORDS == WORDS - 1) {
            const int lane = threadIdx.x % LANES, group = threadIdx.x / LANES, k8 = group * PER / 8;
            const int tile_row = 2 * lane + ((way < 0) != (second != 0) ? 1 : 0);
            unsigned char *at = operand + (k8 >> 1) * L::kSub + (k8 & 1) * L::kEight + tile_row * 16 + (PER == 4 ? (group & 1) * 8 : 0);
            if constexpr (WORDS == 4) {
                *reinterpret_cast<qt_u32x4 *>(at) = qt_u32x4{h[0], h[1], h[2], h[3]};
                *reinterpret_cast<qt_u32x4 *>(at + L::kPlane) = qt_u32x4{r[0], r[1], r[2], r[3]};
            } else {
                *reinterpret_cast<uint2 *>(at) = make_uint2(h[0], h[1]);
                *reinterpret_cast<uint2 *>(at + L::kPlane) = make_uint2(r[0], r[1]);
            }
        }
    }
    // (What this needs is hidden from the compiler until it is needed: left to itself it carries the split diagonal elements and
    // their places through the loop in ten registers, and spills others.  A reload from scratch at the top of a tile waits
    // for all loads in flight, those of the next tile too: 99 x 1024^3 931 -> 907 us)
    __device__ __forceinline__ void patch(unsigned char *operand, int k0, float s) const {
        using L = HalfLayout<ROWS>;
        int thread = threadIdx.x, first = column;
        asm volatile("" : "+v"(thread), "+v"(first), "+v"(k0));
        const int lane = thread % LANES, group = thread / LANES, k8 = group * PER / 8;
#pragma unroll
        for (int second = 0; second < 2; ++second) {
            const int d = first + (second ? way : 0) - k0;
            float x = dval[second];
            asm volatile("" : "+v"(x));
            if ((unsigned)d < (unsigned)PER)
                patch_element(operand + (k8 >> 1) * L::kSub + (k8 & 1) * L::kEight + (2 * lane + ((way < 0) != (second != 0) ? 1 : 0)) * 16 +
                              ((PER == 4 ? (group & 1) * 4 : 0) + d) * 2, L::kPlane, x * s);
        }
    }
    __device__ __forceinline__ void tops(uint32_t *s_top) const {
        const int lane = threadIdx.x % LANES;
        atomicMax(s_top + 2 * lane + (way < 0 ? 1 : 0), __float_as_uint(top[0]));
        atomicMax(s_top + 2 * lane + (way < 0 ? 0 : 1), __float_as_uint(top[1]));
    }
};

// The scale of an operand whose largest element has the bits amax[b], and its inverse.  False where a scale, its inverse or
// the product of two could leave the fp32 range (an infinite or zero bound too), and where the smallest piece of the
// operand, scaled, lies below 2^-13: the bf16 split takes such a product.  (Nothing but two words and their comparison here:
// with a look at the code table as well the compiler spilled inside the loops with a quantized operand, 84 -> 96 us for
// a product by a quantized 3072 x 3072.)
__device__ __forceinline__ bool half_scale(const uint32_t *amax, const float *fine, int b, float &s, float &inverse) {
    const uint32_t e = amax[b] >> 23;                  // the largest element lies in [2^(e - 127), 2^(e - 126))
    if (e < 67 || e > 187) return false;
    s = __uint_as_float((127 + 14 + 127 - e) << 23);
    inverse = __uint_as_float((e - 14) << 23);
    return fine == nullptr || fine[b] * 0x1p-13f <= s;
}

// The smallest piece of what is shown to it, four elements of a row at a time (minus one, as bits: zero counts as the largest).
struct Pieces {
    uint32_t low = 0xffffffffu;
    float column[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    __device__ __forceinline__ void see(float piece) { low = min(low, __float_as_uint(piece) - 1u); }
    __device__ __forceinline__ void row(const float y[4]) {
        see(fmaxf(fmaxf(fabsf(y[0]), fabsf(y[1])), fmaxf(fabsf(y[2]), fabsf(y[3]))));
#pragma unroll
        for (int e = 0; e < 4; ++e) column[e] = fmaxf(column[e], fabsf(y[e]));
    }
    __device__ __forceinline__ void end() {              // of a run of rows: their columns' pieces
#pragma unroll
        for (int e = 0; e < 4; ++e) { see(column[e]); column[e] = 0.0f; }
    }
};
// *word = max(*word, value) for a word that only ever rises.  Atomics on one line come one after the other, 10 ns each, so a
// look at the word first leaves out those that change nothing, all but a few.
__device__ __forceinline__ void raise_word(uint32_t *word, uint32_t value) {
    if (value > __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(word, value);
}
__device__ __forceinline__ void raise_fineness(uint32_t *fine, uint32_t low) {
    if (low != 0xffffffffu) raise_word(fine, __float_as_uint(1.0f / __uint_as_float(low + 1u)));
}

// A tile row is fine if its largest scaled element is zero or in [2^-10, 2^15).
__device__ __forceinline__ bool half_row_fine(uint32_t top) {
    const int up = (int)(top >> 23) - 127;
    return top == 0 || (up >= -10 && up < 15);
}

// Main loop: 4 waves in a 2 x 2 grid multiply the `tiles` k tiles of a BM x BN tile.  src_a(t), src_b(t): where k tile t
// of an operand lies, in scalar registers.  Work that one tile needs is laid between the matrix instructions of another by
// hand, one piece behind each (the fences keep the compiler from gathering it): a matrix instruction takes 32 cycles of
// its pipe and a split pair 28 of the vector units, and both run at once.  Tile t is multiplied out of one LDS stage
// while tile t + 1, loaded SETS tiles before, is split into the other and tile t + 1 + SETS is asked for.  (99 x 1024^3:
// left to the compiler 830 us, matrix pipes busy 0.43; this 775, 0.50.  What bounds it from there on is power: the same
// launch on zeros takes 500 us, at 2.3 instead of 1.6 GHz.)  Loads past the last tile repeat it instead of being left
// out: a branch around a load makes the next wait one for all loads in flight.
// k_begin: the first k; diag_k, diag_rows: the exact diagonal of a quantized operand is met by k in diag_k .. diag_k + diag_rows - 1.
template <int BM, int BN, int SETS, bool DIAG, typename LA, typename LB, typename SrcA, typename SrcB, typename Acc>
__device__ __forceinline__ void half_main_loop(unsigned char *mem, LA &la, LB &lb, SrcA src_a, SrcB src_b, int tiles, int k_begin, int diag_k,
                                               int diag_rows, float sa, float sb, Acc &acc, Acc &rest) {
    using HA = HalfLayout<BM>;
    using HB = HalfLayout<BN>;
    constexpr int MI = BM / 64, NI = BN / 64, STAGE = HA::kOperand + HB::kOperand;
    constexpr int BLOCKS = MI * NI, STEPS = 6 * BLOCKS;                    // matrix instructions per k tile
    constexpr int WORK = LA::kPairs + 4 + LB::kPairs + 4;                  // pieces to lay between them
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row_a = (wave >> 1) * (BM / 2) + (lane & 31), row_b = (wave & 1) * (BN / 2) + (lane & 31), eight = lane >> 5;
    // (First all loads of one operand, then those of the other, as in the loop: a wait inside the loop counts the loads that may
    // be behind its own on either way into it, and interleaved here it waited for most of the other operand's, just issued:
    // 99 x 1024^3 by a quantized right factor 907 -> 892 us, dense 782 -> 771, 36 x 1024 x 768 by 768 178 -> 168)
    auto fetch_tile = [&](int t, int s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) la.fetch(src_a(t), s, q);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q) lb.fetch(src_b(t), s, q);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < SETS; ++s) fetch_tile(s, s);
    la.ahead(0, 0);
    lb.ahead(0, 0);
#pragma unroll
    for (int p = 0; p < LA::kPairs; ++p) la.pair(mem, 0, sa, p);
#pragma unroll
    for (int p = 0; p < LB::kPairs; ++p) lb.pair(mem + HA::kOperand, 0, sb, p);
    fetch_tile(SETS, 0);
    auto patch = [&](unsigned char *stage, int t) {
        if constexpr (DIAG) {
            const int k0 = k_begin + t * HK;
            if (k0 + HK > diag_k && k0 < diag_k + diag_rows) {
                la.patch(stage, k0, sa);
                lb.patch(stage + HA::kOperand, k0, sb);
            }
        }
    };
    patch(mem, 0);
    __syncthreads();
    auto tile = [&](int t, int cur, int set) {          // multiplies tile t; `set` holds tile t + 1
        const unsigned char *pa = mem + cur * STAGE + eight * HA::kEight + row_a * 16;
        const unsigned char *pb = mem + cur * STAGE + HA::kOperand + eight * HB::kEight + row_b * 16;
        unsigned char *next = mem + (cur ^ 1) * STAGE;
        qt_f16x8 fa[2][2][MI], fb[2][2][NI];
        // fragments of one half of k, in the order in which the products use them: h h, r h, h r
        auto read = [&](int u, int n) {
            if (n < MI) fa[u][0][n] = *reinterpret_cast<const qt_f16x8 *>(pa + u * HA::kSub + n * 32 * 16);
            else if (n < MI + NI) fb[u][0][n - MI] = *reinterpret_cast<const qt_f16x8 *>(pb + u * HB::kSub + (n - MI) * 32 * 16);
            else if (n < 2 * MI + NI) fa[u][1][n - MI - NI] = *reinterpret_cast<const qt_f16x8 *>(pa + u * HA::kSub + HA::kPlane + (n - MI - NI) * 32 * 16);
            else fb[u][1][n - 2 * MI - NI] = *reinterpret_cast<const qt_f16x8 *>(pb + u * HB::kSub + HB::kPlane + (n - 2 * MI - NI) * 32 * 16);
        };
        constexpr int READS = 2 * (MI + NI);
        const auto from_a = src_a(t + 1 + SETS);
        const auto from_b = src_b(t + 1 + SETS);
#pragma unroll
        for (int n = 0; n < READS; ++n) read(0, n);
        la.ahead(set, 0);
#pragma unroll
        for (int g = 0; g < STEPS; ++g) {
            const int u = g / (3 * BLOCKS), c = g % (3 * BLOCKS) / BLOCKS, i = g % BLOCKS / NI, j = g % NI;
            auto &to = c == 0 ? acc[i][j] : rest[i][j];
            to = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[u][c == 1][i], fb[u][c == 2][j], to, 0, 0, 0);
#pragma unroll
            for (int w = g * WORK / STEPS; w < (g + 1) * WORK / STEPS; ++w) {
                if (w < LA::kPairs) la.pair(next, set, sa, w);
                else if (w < LA::kPairs + 4) {
                    la.fetch(from_a, set, w - LA::kPairs);
                    if (w == LA::kPairs + 3) lb.ahead(set, 0);
                } else if (w < LA::kPairs + 4 + LB::kPairs) lb.pair(next + HA::kOperand, set, sb, w - LA::kPairs - 4);
                else lb.fetch(from_b, set, w - LA::kPairs - 4 - LB::kPairs);
            }
            // the other half's fragments, from the middle of this half's products on
#pragma unroll
            for (int n = 0; n < READS; ++n)
                if (g == 2 * BLOCKS + n * BLOCKS / READS - (BLOCKS == 1 ? 1 : 0)) read(1, n);
            __builtin_amdgcn_sched_barrier(0);
        }
        patch(next, t + 1);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int ROUND = SETS % 2 == 0 ? SETS : 2 * SETS;     // stages and sets come round together
    for (int t = 0; t < tiles; t += ROUND) {
#pragma unroll
        for (int u = 0; u < ROUND; ++u) {
            if (t + u >= tiles) break;
            tile(t + u, u & 1, (u + 1) % SETS);
        }
    }
}

}  // namespace
}  // namespace qt
