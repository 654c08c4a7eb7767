// Blockwise quantize kernels for gfx950 (wave64) and their launchers.
//
// Two paths:
//  * flat path -- blocksize divides order.  The matrix is then a flat stream of whole segments
//    (segment s = elements [s*BS, (s+1)*BS), absmax index s).  A wave takes 2048 elements per
//    step as 8 coalesced 16-byte loads per lane, the segment maximum is a DPP butterfly, the
//    quotient is a correctly rounded fp32 division (one exact reciprocal per segment, then the
//    multiply / residual-fma / correction-fma sequence), and the index is a threshold count
//    done through a bucket table in LDS.
//  * general path -- any order/blocksize (ragged last segment, odd order with nibble pairs that
//    straddle rows), and whatever is small: chunks of segments, each read once by a group of lanes; the
//    threshold count through the bucket table in 8 bits, by a search in LDS in 4.
//
// Arithmetic follows qtensor/functional.py:526-615 and :703-735 of the reference.
#include "qt_common.h"
#include "qt_tables.h"
#include "qt_divide.h"

namespace qt {
namespace {

#ifndef QT_Q_THREADS
#define QT_Q_THREADS 256
#endif
#ifndef QT_Q_BLOCKS_PER_CU
#define QT_Q_BLOCKS_PER_CU 3
#endif
constexpr int kThreads = 256;            // general-path kernels
constexpr int kFlatThreads = QT_Q_THREADS;
static_assert(kFlatThreads == 256, "build_code_tables");
constexpr int kFlatBlocksPerCU = QT_Q_BLOCKS_PER_CU;
constexpr int kStep = 2048;              // elements a wave takes per step on the flat path

template <typename T> struct ElementLoader;
template <> struct ElementLoader<float> {
    template <bool STREAM>
    static __device__ __forceinline__ float4 load4(const float *base, uint32_t k) {
        return load_f32x4<STREAM>(base + k);
    }
    static __device__ __forceinline__ float load1(const float *base, size_t k) { return base[k]; }
};
template <> struct ElementLoader<uint16_t> {
    template <bool STREAM>
    static __device__ __forceinline__ float4 load4(const uint16_t *base, uint32_t k) {
        const uint2 w = load_u32x2<STREAM>(base + k);
        return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                           __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u));
    }
    static __device__ __forceinline__ float load1(const uint16_t *base, size_t k) { return bf16_bits_to_float(base[k]); }
};

// Per-wave staging area: packed codes of one step in element order, and its segment maxima.
template <int BITS>
struct WaveStage {
    uint4 codes[BITS == 4 ? 64 : 128];
    float maxima[32];
};

// One step of a wave = 2048 consecutive elements, fetched as J = 8 fully coalesced 16-byte
// loads per lane (vector j of lane L covers elements 256 j + 4 L .. +3).  A segment is G = BS/4
// lanes of one vector for BS <= 256, and JS = BS/256 whole vectors of the wave above that.  The
// packed codes and the maxima are parked in LDS so that they leave as one contiguous 1 KiB
// (4-bit) or 2 KiB (8-bit) run and one run of 2048/BS floats per step.
template <typename T, int BITS, int BS, bool DIAG, bool STREAM>
struct FlatQuantizer {
    static constexpr int NCODE = 1 << BITS;
    static constexpr int J = 8;
    static constexpr int JS = BS > 256 ? BS / 256 : 1;
    static constexpr int G = BS >= 256 ? 64 : BS / 4;
    static constexpr int SEGS = kStep / BS;

    const T *__restrict__ A;
    float *__restrict__ absmax;
    float *__restrict__ diag;
    uint8_t *__restrict__ out;
    const CodeTables<NCODE> &tab;
    const uint2 *lut;
    WaveStage<BITS> &stage;
    FastDiv row_div;                                        // by order/4
    FastDiv order_div;                                      // by order (rows of a stack -> row inside its matrix)
    bool fast_ok, ascending;
    uint32_t lane;

    struct Step {
        float4 v[J];
    };

    static __device__ __forceinline__ void load_step(const T *A, Step &s, uint32_t step) {
        const uint32_t k0 = step * (uint32_t)kStep + (threadIdx.x & 63u) * 4u;
#pragma unroll
        for (int j = 0; j < J; ++j) s.v[j] = ElementLoader<T>::template load4<STREAM>(A, k0 + (uint32_t)j * 256u);
    }

    __device__ __forceinline__ void load(Step &s, uint32_t step) const { load_step(A, s, step); }

    __device__ __forceinline__ void process(Step &s, uint32_t step) const {
        if (DIAG) {
            const uint32_t k4 = step * (uint32_t)(kStep / 4) + lane;
            uint32_t row = fastdiv(k4, row_div);            // row of the stack of matrices
            uint32_t col4 = k4 - row * row_div.divisor;
            uint32_t lrow = row - fastdiv(row, order_div) * order_div.divisor;   // row inside its matrix
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if ((lrow >> 2) == col4) {                  // this vector holds a diagonal element
                    const uint32_t e = lrow & 3u;
                    float4 &v = s.v[j];
                    diag[row] = e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w;
                    if (e == 0) v.x = 0.0f; else if (e == 1) v.y = 0.0f; else if (e == 2) v.z = 0.0f; else v.w = 0.0f;
                }
                col4 += 64u;
                while (col4 >= row_div.divisor) {
                    col4 -= row_div.divisor;
                    ++row;
                    if (++lrow == order_div.divisor) lrow = 0;
                }
            }
        }

        uint16_t *stage16 = reinterpret_cast<uint16_t *>(stage.codes);
        uint32_t *stage32 = reinterpret_cast<uint32_t *>(stage.codes);
#pragma unroll
        for (int jg = 0; jg < J; jg += JS) {
            uint32_t m = 0;
#pragma unroll
            for (int jj = 0; jj < JS; ++jj) {
                const float4 v = s.v[jg + jj];
                m = max(max(m, max(abs_bits(v.x), abs_bits(v.y))), max(abs_bits(v.z), abs_bits(v.w)));
            }
            m = group_max_u32<G>(m);

            // 2^-60 <= amax <= 2^60, else (zero, huge, tiny, inf, NaN) take the exact route
            const bool special = !fast_ok || (m - kFastDivLo) > (kFastDivHi - kFastDivLo);
            uint32_t idx[JS][4];
            if (__any(special)) {
                if (m > 0x7f800000u) m = 0x7fc00000u;       // any NaN in the segment -> canonical NaN
#pragma unroll
                for (int jj = 0; jj < JS; ++jj) {
                    const float4 v = s.v[jg + jj];
                    idx[jj][0] = exact_index<NCODE>(v.x, m, tab);
                    idx[jj][1] = exact_index<NCODE>(v.y, m, tab);
                    idx[jj][2] = exact_index<NCODE>(v.z, m, tab);
                    idx[jj][3] = exact_index<NCODE>(v.w, m, tab);
                }
            } else {
                const float amax = __uint_as_float(m);
                const float r = exact_reciprocal(amax);
#pragma unroll
                for (int jj = 0; jj < JS; ++jj) {
                    const float4 v = s.v[jg + jj];
                    const float x[4] = {v.x, v.y, v.z, v.w};
                    fast_four(x, amax, r, lut, idx[jj]);
                }
                if (!ascending) {
#pragma unroll
                    for (int jj = 0; jj < JS; ++jj)
#pragma unroll
                        for (int e = 0; e < 4; ++e) idx[jj][e] = tab.perm[idx[jj][e]];
                }
            }
            if ((lane & (G - 1)) == 0) stage.maxima[(jg * 256 + (int)lane * 4) / BS] = __uint_as_float(m);
#pragma unroll
            for (int jj = 0; jj < JS; ++jj) {
                const uint32_t *i = idx[jj];
                if (BITS == 4)
                    stage16[(jg + jj) * 64 + lane] = (uint16_t)(((i[0] << 4) | i[1]) | (((i[2] << 4) | i[3]) << 8));
                else
                    stage32[(jg + jj) * 64 + lane] = i[0] | (i[1] << 8) | (i[2] << 16) | (i[3] << 24);
            }
        }
        wave_lds_sync();
        uint4 *dst = reinterpret_cast<uint4 *>(out + (size_t)step * (kStep * BITS / 8));
        dst[lane] = stage.codes[lane];
        if (BITS == 8) dst[64 + lane] = stage.codes[64 + lane];
        if (lane < SEGS) absmax[step * (uint32_t)SEGS + lane] = stage.maxima[lane];
        wave_lds_sync();                                    // the next step rewrites the staging area
    }
};

template <typename T, int BITS, int BS, bool DIAG, bool STREAM>
__global__ __launch_bounds__(kFlatThreads) void quantize_flat_kernel(
    const T *__restrict__ A, const float *__restrict__ code, uint32_t n_steps, FastDiv row_div, FastDiv order_div,
    float *__restrict__ absmax, float *__restrict__ diag, uint8_t *__restrict__ out) {
    using Q = FlatQuantizer<T, BITS, BS, DIAG, STREAM>;
    constexpr int NCODE = Q::NCODE;
    constexpr int kWaves = kFlatThreads / 64;

    __shared__ CodeTables<NCODE> tab;
    __shared__ uint2 lut[kLutEntries];
    __shared__ WaveStage<BITS> stages[kWaves];
    const uint32_t w = threadIdx.x >> 6;
    typename Q::Step a, b;
    // the first step's loads are on their way while the tables are set up
    Q::load_step(A, a, min(blockIdx.x * kWaves + w, n_steps - 1));
    build_code_tables<NCODE>(code, tab, lut);
    const int flags = tab.flags;

    const Q q{A, absmax, diag, out, tab, lut, stages[w], row_div, order_div, (flags & kFlagLut) != 0,
              (flags & kFlagAscending) != 0, threadIdx.x & 63u};
    const uint32_t n_waves = gridDim.x * kWaves;
    uint32_t step = blockIdx.x * kWaves + w;
    if (step >= n_steps) return;
    // Two register buffers in ping-pong: the loads of the next step are in flight while the
    // current one is processed.  Look-ahead indices are clamped so every load is unconditional.
    const uint32_t last = n_steps - 1;
    while (true) {
        q.load(b, min(step + n_waves, last));
        q.process(a, step);
        step += n_waves;
        if (step >= n_steps) break;
        q.load(a, min(step + n_waves, last));
        q.process(b, step);
        step += n_waves;
        if (step >= n_steps) break;
    }
}

// ---- general path ----------------------------------------------------------------------
// Any order and alignment, one launch for a whole stack: every matrix has its own run of maxima, diagonal entries and
// code bytes, the codes of an odd order padded to a whole byte per matrix.  Bound by memory like the flat path, but its
// segments are ragged and start anywhere, so the unit of work is a chunk of consecutive segments per workgroup (places for
// 2048 elements, or four segments of 512 places and more): min(64, bs / 4) lanes hold a segment, four consecutive elements each per round, so that maximum and
// codes come out of one read (the rounds after the first of a segment longer than 256 elements are read twice, from the
// cache the second time).  WHOLE: the order is a multiple of four, every lane's four codes are whole bytes of the result
// and leave as one 2-byte (4-bit) or 4-byte store, 128 bytes or more per wave.  Otherwise a code byte can straddle lanes,
// segments and rows: the codes are parked in LDS as bytes and packed from there into aligned words; the byte that a
// chunk shares with the next one belongs to the chunk with its first element, which encodes that one segment further.
// Back to back, 4 bits, exact diagonal, against a launch for the maxima and one with a thread per code byte: one 1200 x
// 1200 matrix in segments of 64 5.8 us against 11.5, one 257 x 257 7.8 against 7.7, 100 of 27 x 27 7.5 against 8.9, 30
// of 576 x 576 in segments of 128 16.6 against 71.
template <typename T>
__device__ __forceinline__ void load_upto_four(const T *p, uint32_t n, float x[4]) {
    // (element alignment is all that is known; the hardware takes wide loads at any dword, bf16 at any two bytes)
    if (n >= 4u) {
        if constexpr (sizeof(T) == 4) {
            typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
            const f32x4_any v = *reinterpret_cast<const f32x4_any *>(p);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        } else {
            typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
            const u32x2_any v = *reinterpret_cast<const u32x2_any *>(p);
            x[0] = __uint_as_float(v.x << 16); x[1] = __uint_as_float(v.x & 0xffff0000u);
            x[2] = __uint_as_float(v.y << 16); x[3] = __uint_as_float(v.y & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) x[e] = e < n ? ElementLoader<T>::load1(p, e) : 0.0f;
    }
}

constexpr uint32_t kChunkIds = 8192;     // codes of the largest chunk (four segments of 2048)
// Segments of a chunk: places for 2048 elements (for 8192, where there are chunks enough all the same, is no faster).
inline uint32_t chunk_segments(uint32_t bs_shift) { return bs_shift < 9 ? 2048u >> bs_shift : 4u; }

template <typename T, int BITS, bool DIAG, bool WHOLE>
__global__ __launch_bounds__(kThreads) void quantize_general_kernel(
    const T *__restrict__ A, const float *__restrict__ code, uint32_t order, uint32_t bs_shift, uint32_t nb, FastDiv nb_div,
    uint32_t n_segments, uint32_t per_chunk, uint32_t chunks_per_matrix, uint32_t n_chunks, float *__restrict__ absmax,
    float *__restrict__ diag, uint8_t *__restrict__ out) {
    constexpr int NCODE = 1 << BITS;
    constexpr uint32_t EPB = 8 / BITS;
    __shared__ CodeTables<NCODE> tab;
    __shared__ uint8_t ids[WHOLE ? 1 : kChunkIds + 1];               // (the shared byte's second code behind them)
    __shared__ uint2 lut_mem[BITS == 8 ? kLutEntries : 1];
    uint2 *lut = BITS == 8 ? lut_mem : nullptr;
    const uint32_t bs = 1u << bs_shift;
    const uint32_t g_shift = min(bs_shift - 2u, 6u);                  // log2 of the lanes per segment
    const uint32_t in_group = (threadIdx.x & ((1u << g_shift) - 1u)) * 4u, group = threadIdx.x >> g_shift;
    const uint32_t n_groups = (uint32_t)kThreads >> g_shift;
    const uint32_t total = order * order, n_bytes = (total + EPB - 1) / EPB;
    // the first segment's first loads are on their way while the tables are set up
    float ahead[4] = {};
    uint32_t ahead_of = 0xffffffffu;                                  // the segment (of chunk blockIdx.x) that they are of
    {
        const uint32_t b = blockIdx.x / chunks_per_matrix, s = (blockIdx.x - b * chunks_per_matrix) * per_chunk + group;
        if (s < n_segments) {
            const uint32_t r = fastdiv(s, nb_div), c = ((s - r * nb) << bs_shift) + in_group, c1 = min(c - in_group + bs, order);
            load_upto_four<T>(A + (size_t)b * total + (size_t)r * order + c, c < c1 ? c1 - c : 0u, ahead);
            ahead_of = s;
        }
    }
    build_code_tables<NCODE>(code, tab, lut);
    const bool fast_ok = (tab.flags & kFlagLut) != 0, ascending = (tab.flags & kFlagAscending) != 0;

    for (uint32_t chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
        const uint32_t b = chunk / chunks_per_matrix;
        const T *src = A + (size_t)b * total;
        float *am = absmax + (size_t)b * n_segments;
        float *dg = DIAG ? diag + (size_t)b * order : nullptr;
        uint8_t *dst = out + (size_t)b * n_bytes;
        const uint32_t s0 = (chunk - b * chunks_per_matrix) * per_chunk, s1 = min(s0 + per_chunk, n_segments);
        uint32_t k0 = 0, k1 = 0;
        if (!WHOLE) {
            const uint32_t r0 = fastdiv(s0, nb_div), r1 = fastdiv(s1, nb_div);
            k0 = r0 * order + ((s0 - r0 * nb) << bs_shift);
            k1 = r1 * order + ((s1 - r1 * nb) << bs_shift);           // (s1 == n_segments: row `order`, column 0)
        }
        const bool shared_byte = !WHOLE && EPB == 2 && (k1 & 1u) != 0u && s1 < n_segments;
        const uint32_t s_end = s1 + (shared_byte ? 1u : 0u);
        for (uint32_t s = s0 + group; s < s_end; s += n_groups) {
            const uint32_t r = fastdiv(s, nb_div), c0 = (s - r * nb) << bs_shift;
            const uint32_t c1 = min(c0 + bs, order);
            const T *row = src + (size_t)r * order;
            const bool own = s < s1;                                  // the shared byte's other segment is not
            auto four = [&](uint32_t c, float x[4], bool first, bool loaded = false) {
                if (!loaded) load_upto_four<T>(row + c, c < c1 ? c1 - c : 0u, x);
                if (DIAG && r - c < 4u && r < c1) {
                    const uint32_t e = r - c;
                    const float d = e == 0 ? x[0] : e == 1 ? x[1] : e == 2 ? x[2] : x[3];
                    if (first && own) dg[r] = d;
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) x[i] = i == e ? 0.0f : x[i];
                }
            };
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = ahead[e];
            four(c0 + in_group, x, true, s == ahead_of);
            ahead_of = 0xffffffffu;
            uint32_t m = max(max(abs_bits(x[0]), abs_bits(x[1])), max(abs_bits(x[2]), abs_bits(x[3])));
            for (uint32_t c = c0 + 256u; c < c1; c += 256u) {                 // (c1 is the same for all lanes of a segment)
                float y[4];
                four(c + in_group, y, true);
                m = max(m, max(max(abs_bits(y[0]), abs_bits(y[1])), max(abs_bits(y[2]), abs_bits(y[3]))));
            }
            m = group_max_u32<16>(m);
            if (g_shift >= 5) m = max(m, (uint32_t)__shfl_xor((int)m, 16, 64));
            if (g_shift >= 6) m = max(m, (uint32_t)__shfl_xor((int)m, 32, 64));
            const bool exact = !fast_ok || (m - kFastDivLo) > (kFastDivHi - kFastDivLo);
            if (m > 0x7f800000u) m = 0x7fc00000u;
            if (own && in_group == 0u) am[s] = __uint_as_float(m);
            const float a = __uint_as_float(m), recip = exact ? 0.0f : exact_reciprocal(a);

            for (uint32_t c = c0; c < c1; c += 256u) {
                if (c != c0) four(c + in_group, x, false);
                const uint32_t at = c + in_group;
                if (at >= c1) continue;
                uint32_t idx[4];
                if (exact) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) idx[e] = exact_index<NCODE>(x[e], m, tab);
                } else {
                    if constexpr (BITS == 8) fast_four(x, a, recip, lut, idx);
                    else
#pragma unroll
                        for (int e = 0; e < 4; ++e) idx[e] = fast_index<NCODE>(x[e], a, recip, tab);
                    if (!ascending)
#pragma unroll
                        for (int e = 0; e < 4; ++e) idx[e] = tab.perm[idx[e]];
                }
                const uint32_t k = r * order + at;
                if (WHOLE) {
                    if (BITS == 4)
                        *reinterpret_cast<uint16_t *>(dst + (k >> 1)) = (uint16_t)(((idx[0] << 4) | idx[1]) | (((idx[2] << 4) | idx[3]) << 8));
                    else
                        *reinterpret_cast<uint32_t *>(dst + k) = idx[0] | (idx[1] << 8) | (idx[2] << 16) | (idx[3] << 24);
                } else {
#pragma unroll
                    for (uint32_t e = 0; e < 4u; ++e)
                        if (own ? at + e < c1 : (e == 0u && at == c0)) ids[k + e - k0] = (uint8_t)idx[e];
                }
            }
        }
        ahead_of = 0xffffffffu;                                       // (a group without a segment in the first chunk)
        if (!WHOLE) {
            __syncthreads();
            const uint32_t j0 = (k0 + EPB - 1) / EPB, j1 = (k1 + EPB - 1) / EPB;
            auto packed = [&](uint32_t j) -> uint32_t {
                if (EPB == 1) return ids[j - k0];
                const uint32_t k = 2u * j - k0;
                return ((uint32_t)ids[k] << 4) | (2u * j + 1u < total ? (uint32_t)ids[k + 1u] : 0u);
            };
            const uint32_t skew = (uint32_t)(reinterpret_cast<uintptr_t>(dst + j0) & 3u);    // bytes before j0 in its word
            const uint32_t n_words = (j1 - j0 + skew + 3u) / 4u;
            for (uint32_t w = threadIdx.x; w < n_words; w += (uint32_t)kThreads) {
                const int32_t j = (int32_t)(j0 + 4u * w) - (int32_t)skew;
                if (j >= (int32_t)j0 && j + 4 <= (int32_t)j1) {
                    *reinterpret_cast<uint32_t *>(dst + j) =
                        packed(j) | (packed(j + 1) << 8) | (packed(j + 2) << 16) | (packed(j + 3) << 24);
                } else {
                    for (int32_t i = max(j, (int32_t)j0); i < min(j + 4, (int32_t)j1); ++i) dst[i] = (uint8_t)packed((uint32_t)i);
                }
            }
            __syncthreads();                                          // the next chunk rewrites the codes
        }
    }
}

// ---- transposed source -----------------------------------------------------------------
// Quantizes the transpose of every matrix of a stack without writing the transpose out (the
// reference transposes first: V.T.contiguous() at qtensor/utils.py:169, then the plain quantizer).
// A workgroup takes BS input rows x 64 input columns, turns the tile around in LDS (row stride
// BS + 1: the scalar writes and reads below hit distinct banks for BS = 64), and every group of
// BS/4 lanes encodes one segment of an output row with the arithmetic of the flat path.
template <int BITS, int BS>
__global__ __launch_bounds__(kThreads) void quantize_transposed_kernel(
    const float *__restrict__ A, const float *__restrict__ code, uint32_t order, uint32_t n_tiles, uint32_t tiles_r, uint32_t tiles_c,
    float *__restrict__ absmax, uint8_t *__restrict__ out) {
    constexpr int NCODE = 1 << BITS;
    constexpr int LD = BS + 1;
    constexpr int G = BS / 4;                    // lanes per segment
    constexpr int SEGS = 64 / G;                 // segments a wave encodes at a time
    static_assert(BS == 64 || BS == 128 || BS == 256, "segment of 64, 128 or 256 elements");
    __shared__ CodeTables<NCODE> tab;
    __shared__ float tile[64 * LD];
    build_code_tables<NCODE>(code, tab, nullptr);
    const bool fast_ok = (tab.flags & kFlagLut) != 0, ascending = (tab.flags & kFlagAscending) != 0;
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t per_matrix = tiles_r * tiles_c;
    for (uint32_t id = blockIdx.x; id < n_tiles; id += gridDim.x) {
        const uint32_t b = id / per_matrix, rem = id - b * per_matrix;
        const uint32_t rb = rem / tiles_c, cb = rem - rb * tiles_c;
        const float *src = A + ((size_t)b * order + (size_t)rb * BS) * order + cb * 64u;
        const uint32_t c4 = (t & 15u) * 4u;
#pragma unroll
        for (int p = 0; p < BS / 16; ++p) {
            const uint32_t r = (uint32_t)p * 16u + (t >> 4);
            const float4 v = *reinterpret_cast<const float4 *>(src + (size_t)r * order + c4);
            tile[(c4 + 0) * LD + r] = v.x;
            tile[(c4 + 1) * LD + r] = v.y;
            tile[(c4 + 2) * LD + r] = v.z;
            tile[(c4 + 3) * LD + r] = v.w;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16 / SEGS; ++q) {
            const uint32_t cl = w * 16u + (uint32_t)q * SEGS + lane / G;       // output row inside the tile
            const uint32_t e0 = (lane % G) * 4u;                               // first of this lane's four elements
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = tile[cl * LD + e0 + e];
            uint32_t m = max(max(abs_bits(x[0]), abs_bits(x[1])), max(abs_bits(x[2]), abs_bits(x[3])));
            m = group_max_u32<G>(m);
            const bool special = !fast_ok || (m - kFastDivLo) > (kFastDivHi - kFastDivLo);
            uint32_t idx[4];
            if (__any(special)) {
                if (m > 0x7f800000u) m = 0x7fc00000u;
#pragma unroll
                for (int e = 0; e < 4; ++e) idx[e] = exact_index<NCODE>(x[e], m, tab);
            } else {
                const float amax = __uint_as_float(m);
                const float r = exact_reciprocal(amax);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    idx[e] = fast_index<NCODE>(x[e], amax, r, tab);
                    if (!ascending) idx[e] = tab.perm[idx[e]];
                }
            }
            const size_t orow = (size_t)b * order + cb * 64u + cl;            // row of the stack of transposes
            if (lane % G == 0) absmax[orow * tiles_r + rb] = __uint_as_float(m);
            const size_t k = orow * order + (size_t)rb * BS + e0;             // flat element index of x[0]
            if (BITS == 4)
                *reinterpret_cast<uint16_t *>(out + (k >> 1)) = (uint16_t)(((idx[0] << 4) | idx[1]) | (((idx[2] << 4) | idx[3]) << 8));
            else
                *reinterpret_cast<uint32_t *>(out + k) = idx[0] | (idx[1] << 8) | (idx[2] << 16) | (idx[3] << 24);
        }
        __syncthreads();                                                       // the next tile rewrites the LDS copy
    }
}

int grid_for(uint32_t work_items_per_block_unit, int blocks_per_cu) {
    const int cap = compute_units() * blocks_per_cu;
    const int need = (int)work_items_per_block_unit;
    return need < 1 ? 1 : (need < cap ? need : cap);
}

template <typename T, int BITS, int BS, bool DIAG>
void launch_flat(const T *A, const float *code, uint32_t order, uint32_t batch, float *absmax, float *diag, uint8_t *out, hipStream_t stream) {
    constexpr uint32_t kWaves = kFlatThreads / 64;
    const uint32_t total = order * order * batch;
    const uint32_t n_steps = total / kStep;
    const FastDiv rd = make_fastdiv(order / 4), od = make_fastdiv(order);
    const uint32_t blocks_needed = (n_steps + kWaves - 1) / kWaves;
    // Inputs far beyond the 256 MB last-level cache are read with the streaming hint, by the fewest workgroups that keep the
    // loads coming.  Below that 4-bit codes do better with five: us with three, four, five, fp32 with its diagonal 3072 x
    // 3072 13.7 12.8 12.8, 4096 x 4096 19.2 19.4 18.4, bf16 4096 x 4096 15.3 14.6 13.5; 8 bits, bf16 4096 x 4096 15.9 16.3 17.7.  Not
    // where a segment is several vectors of a wave, whose registers leave room for four, and a fifth comes after them: fp32 in
    // segments of 512 3072 x 3072 12.3 12.2 14.8, 4096 x 4096 17.9 17.8 19.0, of 2048 4096 x 4096 16.6 16.7 18.1; bf16 4096 x 4096 in
    // segments of 1024 12.0 12.1 11.3, of 2048 11.7 11.8 14.3.
    const bool streams = total >= (1u << 25), five_fit = BS <= (sizeof(T) == 4 ? 256 : 1024);
    const int grid = grid_for(blocks_needed, BITS == 4 && !streams && five_fit ? 5 : kFlatBlocksPerCU);
    if (streams)
        hipLaunchKernelGGL((quantize_flat_kernel<T, BITS, BS, DIAG, true>), dim3(grid), dim3(kFlatThreads), 0, stream,
                           A, code, n_steps, rd, od, absmax, diag, out);
    else
        hipLaunchKernelGGL((quantize_flat_kernel<T, BITS, BS, DIAG, false>), dim3(grid), dim3(kFlatThreads), 0, stream,
                           A, code, n_steps, rd, od, absmax, diag, out);
}

template <typename T, int BITS, bool DIAG>
void launch_general(const T *A, const float *code, uint32_t order, uint32_t bs, uint32_t batch, float *absmax, float *diag, uint8_t *out,
                    hipStream_t stream) {
    // A segment longer than the row is the row: the next power of two gives the same segments, as many of them to a chunk as
    // their real length allows.  Order 100 in 4 bits with a blocksize of 2048, 300 matrices: 29.3 us without, 9.0 with.
    while (bs > 64 && bs / 2 >= order) bs /= 2;
    const uint32_t bs_shift = (uint32_t)__builtin_ctz(bs);
    const uint32_t nb = (order + bs - 1) / bs;
    const uint32_t n_segments = order * nb;
    // 8 bits: the index from the bucket table instead of a search of eight dependent LDS reads, and no more workgroups than
    // share its set-up.  us with the search, and with the table and four or eight workgroups a unit: 1024 x 1024 bf16 6.6, 6.0 and
    // 6.7; 2048 x 2048 13.4, 9.2 and 15.0; 5001 x 5001 fp32 in segments of 128 75.9 with the search and 42.6.  (4-bit codes,
    // whose search is one dependent read, gain nothing: 5001 x 5001 39.9 with the search, 46.8 with the table.)
    const uint32_t per_chunk = chunk_segments(bs_shift), per_matrix = (n_segments + per_chunk - 1) / per_chunk;
    const uint32_t n_chunks = per_matrix * batch;      // (batch * order * order < 2^31 and batch <= 65535: fits)
    const FastDiv nbd = make_fastdiv(nb);
    const dim3 grid(grid_for(n_chunks, BITS == 8 ? 4 : 8));
    const bool whole = order % 4 == 0 && is_aligned(out, BITS == 4 ? 2 : 4);
#define QT_QUANT_GENERAL(WHOLE)                                                                                               \
    hipLaunchKernelGGL((quantize_general_kernel<T, BITS, DIAG, WHOLE>), grid, dim3(kThreads), 0, stream, A, code, order, bs_shift, \
                       nb, nbd, n_segments, per_chunk, per_matrix, n_chunks, absmax, diag, out)
    if (whole) QT_QUANT_GENERAL(true);
    else QT_QUANT_GENERAL(false);
#undef QT_QUANT_GENERAL
}

template <typename T, int BITS, bool DIAG>
void quantize_dispatch(const T *A, const float *code, int order_i, float *absmax, float *diag, uint8_t *out, int blocksize, hipStream_t stream,
                       int batch = 1) {
    clear_error();
    if (!(blocksize == 64 || blocksize == 128 || blocksize == 256 || blocksize == 512 || blocksize == 1024 || blocksize == 2048)) {
        set_error(kBadBlocksize, "quantize_blockwise: blocksize %d is not one of 64,128,256,512,1024,2048", blocksize);
        return;
    }
    if (order_i < 1 || batch < 1 || (int64_t)order_i * order_i * batch >= (int64_t(1) << 31)) {
        set_error(kBadOrder, "quantize_blockwise: order %d (batch %d) out of range (need order >= 1 and batch*order*order < 2^31)",
                  order_i, batch);
        return;
    }
    if (!A || !code || !absmax || !out || (DIAG && !diag)) {
        set_error(kNullPointer, "quantize_blockwise: null device pointer");
        return;
    }
    const uint32_t order = (uint32_t)order_i, bs = (uint32_t)blocksize;
    bool flat = order % bs == 0 && is_aligned(A, 4 * sizeof(T)) && is_aligned(out, 16) && is_aligned(absmax, 4);
    if (batch > 65535 && !flat) {
        set_error(kBadArgument, "quantize_blockwise: a stack whose order the blocksize does not divide (or with unaligned buffers) "
                                "takes at most 65535 matrices per launch");
        return;
    }
    // Small inputs are bound by latency: the general kernel, which takes eight elements a thread and not thirty-two, and in 4 bits
    // searches instead of setting up a bucket table, is the faster one.  us, flat and general, one matrix: 4 bits fp32 with its
    // diagonal 256 x 256 8.3 and 4.6, 1024 x 1024 7.6 and 5.0, 2048 x 2048 8.1 and 7.6, 2560 x 2560 9.3 and 8.8, 4096 x 4096 18.4
    // and 20.4; bf16 2560 x 2560 9.2 and 8.8, 3072 x 3072 10.3 and 11.5; 8 bits bf16 256 x 256 6.8 and 5.5, 1024 x 1024 7.1 and 6.0,
    // 1280 x 1280 7.2 and 7.0 (fp32 6.7 and 6.7), 2048 x 2048 7.9 and 9.2.  Segments of more than 512 it takes in rounds one
    // after the other, and reads twice: 4 bits 1024 x 1024 in segments of 1024 5.8 and 5.3, 2048 x 2048 6.9 and 7.1 (with its diagonal
    // 7.2 and 7.4, bf16 6.9 and 7.2), in segments of 2048 6.5 and 8.8; 8 bits 1024 x 1024 in segments of 1024 5.6 and 6.5.
    const bool long_segments = bs > 512;
    const uint32_t flat_from = BITS == 4 ? (long_segments ? 2u << 20 : 7u << 20) : long_segments ? 0u : 3u << 19;
    if ((uint64_t)order * order * batch < flat_from) flat = false;
    if (flat) {
        switch (blocksize) {
            case 64: launch_flat<T, BITS, 64, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
            case 128: launch_flat<T, BITS, 128, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
            case 256: launch_flat<T, BITS, 256, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
            case 512: launch_flat<T, BITS, 512, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
            case 1024: launch_flat<T, BITS, 1024, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
            default: launch_flat<T, BITS, 2048, DIAG>(A, code, order, (uint32_t)batch, absmax, diag, out, stream); break;
        }
    } else {
        launch_general<T, BITS, DIAG>(A, code, order, bs, (uint32_t)batch, absmax, diag, out, stream);
    }
    launch_ok("quantize_blockwise");
}

}  // namespace
}  // namespace qt

#define QT_DEFINE_QUANT(NAME, T, BITS)                                                                                   \
    extern "C" void cquantize_blockwise_##NAME##_stream(T *A, float *code, int order, float *absmax, unsigned char *out, \
                                                        int blocksize, void *stream) {                                   \
        qt::quantize_dispatch<T, BITS, false>(A, code, order, absmax, nullptr, out, blocksize, (hipStream_t)stream);     \
    }                                                                                                                    \
    extern "C" void cquantize_blockwise_##NAME(T *A, float *code, int order, float *absmax, unsigned char *out,          \
                                               int blocksize) {                                                          \
        qt::quantize_dispatch<T, BITS, false>(A, code, order, absmax, nullptr, out, blocksize, nullptr);                 \
    }                                                                                                                    \
    extern "C" void cquantize_blockwise_diagreal_##NAME##_stream(T *A, float *code, int order, float *absmax,            \
                                                                 float *diag, unsigned char *out, int blocksize,         \
                                                                 void *stream) {                                         \
        qt::quantize_dispatch<T, BITS, true>(A, code, order, absmax, diag, out, blocksize, (hipStream_t)stream);         \
    }                                                                                                                    \
    extern "C" void cquantize_blockwise_diagreal_##NAME(T *A, float *code, int order, float *absmax, float *diag,        \
                                                        unsigned char *out, int blocksize) {                             \
        qt::quantize_dispatch<T, BITS, true>(A, code, order, absmax, diag, out, blocksize, nullptr);                     \
    }

QT_DEFINE_QUANT(8bit_fp32, float, 8)
QT_DEFINE_QUANT(8bit_bf16, uint16_t, 8)
QT_DEFINE_QUANT(4bit_fp32, float, 4)
QT_DEFINE_QUANT(4bit_bf16, uint16_t, 4)

extern "C" void qtensor_hip_quantize_batched(const void *A, int a_is_bf16, const float *code, int bits, int order, int batch,
                                             float *absmax, float *diag, unsigned char *out, int blocksize, void *stream) {
    using namespace qt;
    hipStream_t st = (hipStream_t)stream;
    float *c = const_cast<float *>(code);
    (void)c;
    if (bits != 4 && bits != 8) { clear_error(); set_error(kBadArgument, "quantize_batched: bits must be 4 or 8"); return; }
#define QT_QB(T, BITS)                                                                                        \
    (diag ? quantize_dispatch<T, BITS, true>((const T *)A, code, order, absmax, diag, out, blocksize, st, batch)    \
          : quantize_dispatch<T, BITS, false>((const T *)A, code, order, absmax, nullptr, out, blocksize, st, batch))
    if (a_is_bf16) { if (bits == 4) QT_QB(uint16_t, 4); else QT_QB(uint16_t, 8); }
    else { if (bits == 4) QT_QB(float, 4); else QT_QB(float, 8); }
#undef QT_QB
}

extern "C" void qtensor_hip_quantize_transposed_batched(const float *A, const float *code, int bits, int order, int batch,
                                                        float *absmax, unsigned char *out, int blocksize, void *stream) {
    using namespace qt;
    clear_error();
    if (bits != 4 && bits != 8) { set_error(kBadArgument, "quantize_transposed: bits must be 4 or 8"); return; }
    if (blocksize != 64 && blocksize != 128 && blocksize != 256) {
        set_error(kBadBlocksize, "quantize_transposed: blocksize %d is not one of 64,128,256", blocksize);
        return;
    }
    if (order < 1 || batch < 1 || (int64_t)order * order * batch >= (int64_t(1) << 31) || order % blocksize != 0 || order % 64 != 0) {
        set_error(kBadOrder, "quantize_transposed: order %d (batch %d) must be a multiple of 64 and of the blocksize, batch*order*order < 2^31",
                  order, batch);
        return;
    }
    if (!A || !code || !absmax || !out) { set_error(kNullPointer, "quantize_transposed: null device pointer"); return; }
    if (!is_aligned(A, 16) || !is_aligned(out, 4) || !is_aligned(absmax, 4)) {
        set_error(kBadArgument, "quantize_transposed: A needs 16-byte, out and absmax 4-byte alignment");
        return;
    }
    const uint32_t tiles_r = (uint32_t)(order / blocksize), tiles_c = (uint32_t)(order / 64);
    const uint32_t n_tiles = tiles_r * tiles_c * (uint32_t)batch;
    const int grid = grid_for(n_tiles, blocksize == 256 ? 2 : 4);
#define QT_QT(BITS, BS)                                                                                                  \
    hipLaunchKernelGGL((quantize_transposed_kernel<BITS, BS>), dim3(grid), dim3(kThreads), 0, (hipStream_t)stream, A, code, \
                       (uint32_t)order, n_tiles, tiles_r, tiles_c, absmax, out)
    if (bits == 4) { if (blocksize == 64) QT_QT(4, 64); else if (blocksize == 128) QT_QT(4, 128); else QT_QT(4, 256); }
    else { if (blocksize == 64) QT_QT(8, 64); else if (blocksize == 128) QT_QT(8, 128); else QT_QT(8, 256); }
#undef QT_QT
    launch_ok("quantize_transposed");
}
