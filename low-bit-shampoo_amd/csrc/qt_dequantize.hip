// Blockwise dequantize kernels for gfx950 and their launchers.
//
// out[r,c] = fl32(code[idx] * absmax[segment]) -- except +0.0 for a zero-maximum segment --
// then rounded to the output type; the diagreal form overwrites the diagonal with diag[]
// (qtensor/functional.py:618-688 and :738-746 of the reference).
//
// flat path (blocksize divides order): codes are fetched 16 bytes per lane, turned around in
// LDS, and written out as fully coalesced 16-byte (fp32) or 8-byte (bf16) stores per lane -- the
// store stream is eight ninths of the traffic.  general path: four or eight consecutive elements per thread.
#include "qt_common.h"

namespace qt {
namespace {

#ifndef QT_D_THREADS
#define QT_D_THREADS 128
#endif
#ifndef QT_D_CHUNKED
#define QT_D_CHUNKED 0
#endif
constexpr int kThreads = 256;             // general-path kernel
constexpr int kFlatThreads = QT_D_THREADS;
constexpr int kSuper = 2048;              // elements a wave turns around per step

template <typename T> struct Vec4Store;
template <> struct Vec4Store<float> {
    template <bool STREAM>
    static __device__ __forceinline__ void store(float *base, uint32_t k, float4 y) {
        store_f32x4<STREAM>(base + k, y);
    }
    static __device__ __forceinline__ void store1(float *base, size_t k, float y) { base[k] = y; }
};
template <> struct Vec4Store<uint16_t> {
    template <bool STREAM>
    static __device__ __forceinline__ void store(uint16_t *base, uint32_t k, float4 y) {
        uint2 w;
        w.x = floats_to_bf16_pair(y.x, y.y);
        w.y = floats_to_bf16_pair(y.z, y.w);
        store_u32x2<STREAM>(base + k, w);
    }
    static __device__ __forceinline__ void store1(uint16_t *base, size_t k, float y) { base[k] = float_to_bf16_bits(y); }
};

// Flat path.  Per step a wave takes 2048 consecutive elements: their packed codes arrive with
// one 16-byte (4-bit) or two 16-byte (8-bit) loads per lane and the segment maxima with one
// 4-byte load on the first lanes; both are parked in the wave's private LDS area and read back
// in the order that makes every one of the 8 output stores a fully coalesced 1 KiB (fp32) run.
// The loads of the next step are issued before the stores of the current one.  Big outputs are written
// with the streaming hint, but the codes are always read with plain loads: on an MI355X the hint on this
// thin read stream beside the wide write stream costs a tenth of the bandwidth (0.224 -> 0.199 ms for the
// 16384^2 tensor), and six waves per compute unit in workgroups of two do better there than twelve in
// workgroups of four (0.199 -> 0.185 ms).
//
// The exact diagonal.  kDiagFew: orders of 2048 and more, where a step's elements lie in two rows at most: the places of
// their diagonal entries are the same for the whole wave and cost a scalar comparison per store.  kDiagAny: every lane
// walks along rows and columns, work that waits beside the loads: 8192 x 8192 with codes that come from memory, 4 bits to
// fp32 97 us, few 61 (without a diagonal 58), to bf16 54 us at best, few 34.  With codes that the last-level cache still
// holds, as right behind their quantizer, the walk of kDiagAny costs nothing (see the launch).
enum DiagKind : int { kDiagNone = 0, kDiagAny = 1, kDiagFew = 2 };
template <typename T, int BITS, int DIAG, bool STREAM, int THREADS = kFlatThreads>
__global__ __launch_bounds__(THREADS) void dequantize_flat_kernel(
    const uint8_t *__restrict__ q, const float *__restrict__ code, uint32_t n_super, uint32_t bs_shift,
    FastDiv row_div, FastDiv order_div, const float *__restrict__ absmax, const float *__restrict__ diag, T *__restrict__ out) {
    constexpr int NCODE = 1 << BITS;
    constexpr int kWaves = THREADS / 64;
    constexpr int CODE_VECS = BITS == 4 ? 1 : 2;            // uint4 loads per lane per step
    __shared__ float s_code[NCODE];
    __shared__ uint4 s_stage[kWaves][CODE_VECS * 64];
    __shared__ float s_scale[kWaves][32];
    for (int i = threadIdx.x; i < NCODE; i += THREADS) s_code[i] = code[i];
    __syncthreads();

    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    const uint32_t wave = blockIdx.x * kWaves + w;
    const uint32_t n_waves = gridDim.x * kWaves;
#if QT_D_CHUNKED
    const uint32_t per = (n_super + n_waves - 1) / n_waves;
    uint32_t st = wave * per;
    const uint32_t end = min(st + per, n_super);
    const uint32_t step = 1;
#else
    uint32_t st = wave;
    const uint32_t end = n_super;
    const uint32_t step = n_waves;
#endif
    if (st >= end) return;
    const uint32_t last = end - 1;
    const uint32_t seg_per_super = (uint32_t)kSuper >> bs_shift;   // 32 .. 1
    const uint4 *q16 = reinterpret_cast<const uint4 *>(q);

    uint4 c[CODE_VECS];
    float a = 0.0f;
    auto fetch = [&](uint32_t s) {
#pragma unroll
        for (int v = 0; v < CODE_VECS; ++v) c[v] = load_u32x4<false>(q16 + (size_t)s * (CODE_VECS * 64) + v * 64 + lane);
        if (lane < seg_per_super) a = absmax[s * seg_per_super + lane];
    };
    fetch(st);
    const uint16_t *stage16 = reinterpret_cast<const uint16_t *>(&s_stage[w][0]);
    const uint32_t *stage32 = reinterpret_cast<const uint32_t *>(&s_stage[w][0]);

    for (; st < end; st += step) {
#pragma unroll
        for (int v = 0; v < CODE_VECS; ++v) s_stage[w][v * 64 + lane] = c[v];
        if (lane < seg_per_super) s_scale[w][lane] = a;
        fetch(min(st + step, last));
        wave_lds_sync();

        const uint32_t k4_0 = st * (uint32_t)(kSuper / 4) + lane;   // index of this lane's first 4-vector
        uint32_t row = 0, col4 = 0, lrow = 0;                        // row of the stack, and inside its matrix
        // kDiagFew: where the two rows' diagonal entries lie, counted from the step's first element (beyond the step: none)
        uint32_t at0 = 0xffffffffu, at1 = 0xffffffffu;
        float d0 = 0.0f, d1 = 0.0f;
        if (DIAG == kDiagFew) {
            const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)st) * (uint32_t)kSuper, order = order_div.divisor;
            const uint32_t r = fastdiv(first >> 2, row_div), in = r - fastdiv(r, order_div) * order, next = in + 1u == order ? 0u : in + 1u;
            at0 = r * order + in - first;                            // (wraps around where the entry lies before the step)
            at1 = (r + 1u) * order + next - first;
            if (at0 < (uint32_t)kSuper) d0 = diag[r];
            if (at1 < (uint32_t)kSuper) d1 = diag[r + 1u];
        }
        if (DIAG == kDiagAny) {
            row = fastdiv(k4_0, row_div);
            col4 = k4_0 - row * row_div.divisor;
            lrow = row - fastdiv(row, order_div) * order_div.divisor;
        }
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t v4 = j * 64u + lane;                 // 4-vector inside the step
            uint32_t id0, id1, id2, id3;
            if (BITS == 4) {
                const uint32_t p = stage16[v4];
                id0 = (p >> 4) & 15u; id1 = p & 15u; id2 = (p >> 12) & 15u; id3 = (p >> 8) & 15u;
            } else {
                const uint32_t p = stage32[v4];
                id0 = p & 255u; id1 = (p >> 8) & 255u; id2 = (p >> 16) & 255u; id3 = p >> 24;
            }
            const float scale = s_scale[w][(v4 << 2) >> bs_shift];
            float4 y;
            if (scale == 0.0f) {
                y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            } else {
                y = make_float4(s_code[id0] * scale, s_code[id1] * scale, s_code[id2] * scale, s_code[id3] * scale);
            }
            if (DIAG == kDiagFew) {
                if (at0 >> 8 == j && (at0 >> 2 & 63u) == lane) {
                    const uint32_t e = at0 & 3u;
                    if (e == 0) y.x = d0; else if (e == 1) y.y = d0; else if (e == 2) y.z = d0; else y.w = d0;
                }
                if (at1 >> 8 == j && (at1 >> 2 & 63u) == lane) {
                    const uint32_t e = at1 & 3u;
                    if (e == 0) y.x = d1; else if (e == 1) y.y = d1; else if (e == 2) y.z = d1; else y.w = d1;
                }
            }
            if (DIAG == kDiagAny) {
                if ((lrow >> 2) == col4) {
                    const float d = diag[row];
                    const uint32_t e = lrow & 3u;
                    if (e == 0) y.x = d; else if (e == 1) y.y = d; else if (e == 2) y.z = d; else y.w = d;
                }
                col4 += 64u;
                while (col4 >= row_div.divisor) {
                    col4 -= row_div.divisor;
                    ++row;
                    if (++lrow == order_div.divisor) lrow = 0;
                }
            }
            Vec4Store<T>::template store<STREAM>(out, (k4_0 + j * 64u) << 2, y);
        }
        wave_lds_sync();   // the staging area is rewritten at the top of the next step
    }
}

// General path: any order and alignment, a stack of matrices with a run of code bytes, maxima and diagonal entries each.
// Few elements (the line is drawn in dequantize_dispatch): bound by the latency of a thread's chain of loads and integer
// divisions, not by memory, so a thread takes one code byte and the launch has as many threads as it can.
template <typename T, int BITS, bool DIAG>
__global__ __launch_bounds__(kThreads) void dequantize_bytes_kernel(
    const uint8_t *__restrict__ q, const float *__restrict__ code, uint32_t order, uint32_t bs_shift, uint32_t nb, uint32_t total,
    const float *__restrict__ absmax, const float *__restrict__ diag, T *__restrict__ out) {
    constexpr int NCODE = 1 << BITS;
    constexpr uint32_t EPB = 8 / BITS;
    __shared__ float s_code[NCODE];
    for (int i = threadIdx.x; i < NCODE; i += kThreads) s_code[i] = code[i];
    __syncthreads();
    const uint32_t n_bytes = (total + EPB - 1) / EPB;
    // blockIdx.y = matrix of a stack
    q += (size_t)blockIdx.y * n_bytes;
    absmax += (size_t)blockIdx.y * order * nb;
    if (DIAG) diag += (size_t)blockIdx.y * order;
    out += (size_t)blockIdx.y * total;
    for (uint32_t j = blockIdx.x * kThreads + threadIdx.x; j < n_bytes; j += gridDim.x * kThreads) {
        const uint32_t byte = q[j];
#pragma unroll
        for (uint32_t e = 0; e < EPB; ++e) {
            const uint32_t k = j * EPB + e;
            if (k >= total) break;
            const uint32_t id = BITS == 8 ? byte : (e == 0 ? byte >> 4 : byte & 15u);
            const uint32_t r = k / order, c = k - r * order;
            const float a = absmax[r * nb + (c >> bs_shift)];
            float y = a == 0.0f ? 0.0f : s_code[id] * a;
            if (DIAG && r == c) y = diag[r];
            Vec4Store<T>::store1(out, k, y);
        }
    }
}

// More elements: bound by the store stream.  A thread turns E consecutive elements of the flat matrix into 16-byte (bf16: 8-byte) stores,
// one division by the order and one or two maxima per E.  WHOLE: the order is a multiple of four, E = 4 elements lie in
// one segment of one row and their codes are whole, aligned bytes.  Otherwise E = 8 (whole bytes again) and the thread
// walks over the ends of segments and rows.
// One 1200 x 1200 matrix: 3.6 us against 4.8 with a thread per code byte; 1301 x 1301: 5.0 against 5.7; 30 x 576 x 576: 11.8
// against 21.5 (4-bit codes, back to back).
template <typename T> struct AnyAligned4;                  // four elements at any address of an element
template <> struct AnyAligned4<float> {
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    static __device__ __forceinline__ void store(float *p, const float y[4]) {
        const f32x4_any v = {y[0], y[1], y[2], y[3]};
        *reinterpret_cast<f32x4_any *>(p) = v;
    }
};
template <> struct AnyAligned4<uint16_t> {
    typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(2)));
    static __device__ __forceinline__ void store(uint16_t *p, const float y[4]) {
        const u32x2_any v = {floats_to_bf16_pair(y[0], y[1]), floats_to_bf16_pair(y[2], y[3])};
        *reinterpret_cast<u32x2_any *>(p) = v;
    }
};

template <typename T, int BITS, bool DIAG, bool WHOLE>
__global__ __launch_bounds__(kThreads) void dequantize_general_kernel(
    const uint8_t *__restrict__ q, const float *__restrict__ code, uint32_t order, uint32_t bs_shift, uint32_t nb, FastDiv quad_div,
    uint32_t total, const float *__restrict__ absmax, const float *__restrict__ diag, T *__restrict__ out) {
    constexpr int NCODE = 1 << BITS;
    constexpr uint32_t EPB = 8 / BITS, E = WHOLE ? 4 : 8;
    __shared__ float s_code[NCODE];
    for (int i = threadIdx.x; i < NCODE; i += kThreads) s_code[i] = code[i];
    __syncthreads();
    const uint32_t n_bytes = (total + EPB - 1) / EPB;
    // blockIdx.y = matrix of a stack
    q += (size_t)blockIdx.y * n_bytes;
    absmax += (size_t)blockIdx.y * order * nb;
    if (DIAG) diag += (size_t)blockIdx.y * order;
    out += (size_t)blockIdx.y * total;
    const uint32_t n_units = (total + E - 1) / E;
    for (uint32_t u = blockIdx.x * kThreads + threadIdx.x; u < n_units; u += gridDim.x * kThreads) {
        const uint32_t k = u * E;
        if (WHOLE) {
            uint32_t id[4];
            if (BITS == 4) {
                const uint32_t p = *reinterpret_cast<const uint16_t *>(q + (k >> 1));
                id[0] = (p >> 4) & 15u; id[1] = p & 15u; id[2] = p >> 12; id[3] = (p >> 8) & 15u;
            } else {
                const uint32_t p = *reinterpret_cast<const uint32_t *>(q + k);
                id[0] = p & 255u; id[1] = (p >> 8) & 255u; id[2] = (p >> 16) & 255u; id[3] = p >> 24;
            }
            const uint32_t r = fastdiv(u, quad_div), c = (u - r * quad_div.divisor) * 4u;
            const float a = absmax[r * nb + (c >> bs_shift)];
            float y[4];
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) y[e] = a == 0.0f ? 0.0f : s_code[id[e]] * a;
            if (DIAG && r - c < 4u) {
                const float d = diag[r];
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) y[e] = r - c == e ? d : y[e];
            }
            AnyAligned4<T>::store(out + k, y);
        } else {
            uint32_t r = k / order, c = k - r * order;
            const uint32_t left = min(E, total - k);
            const uint8_t *src = q + k / EPB;
            uint32_t word[BITS == 4 ? 1 : 2] = {};
            if (left == E) {
                typedef uint32_t u32_any __attribute__((aligned(1)));
                word[0] = *reinterpret_cast<const u32_any *>(src);
                if (BITS == 8) word[BITS == 4 ? 0 : 1] = *reinterpret_cast<const u32_any *>(src + 4);
            } else {
                for (uint32_t i = 0; i < (left + EPB - 1) / EPB; ++i) word[i / 4] |= (uint32_t)src[i] << (8u * (i & 3u));
            }
            const uint32_t in_segment = (1u << bs_shift) - 1u;
            float a = absmax[r * nb + (c >> bs_shift)];
            float y[8];
#pragma unroll
            for (uint32_t e = 0; e < E; ++e) {
                const uint32_t id = BITS == 8 ? (word[(BITS == 4 ? 0 : e / 4)] >> (8u * (e & 3u))) & 255u
                                              : (word[0] >> (8u * (e >> 1) + ((e & 1u) ? 0u : 4u))) & 15u;
                y[e] = a == 0.0f ? 0.0f : s_code[id] * a;
                if (DIAG && r == c && e < left) y[e] = diag[r];
                ++c;
                if (c == order) { c = 0; ++r; }
                if ((c & in_segment) == 0u && e + 1u < left) a = absmax[r * nb + (c >> bs_shift)];
            }
            if (left == E) {
                AnyAligned4<T>::store(out + k, y);
                AnyAligned4<T>::store(out + k + 4, y + 4);
            } else {
#pragma unroll
                for (uint32_t e = 0; e < E; ++e)
                    if (e < left) Vec4Store<T>::store1(out, k + e, y[e]);
            }
        }
    }
}

int capped_grid(uint32_t blocks_needed, int blocks_per_cu) {
    const uint32_t cap = (uint32_t)(compute_units() * blocks_per_cu);
    return (int)(blocks_needed < 1 ? 1 : (blocks_needed < cap ? blocks_needed : cap));
}

template <typename T, int BITS, bool DIAG>
void dequantize_dispatch(const uint8_t *q, const float *code, int order_i, const float *absmax, const float *diag,
                         T *out, int blocksize, hipStream_t stream, int batch = 1) {
    clear_error();
    int bs_shift = 0;
    switch (blocksize) {
        case 64: bs_shift = 6; break;
        case 128: bs_shift = 7; break;
        case 256: bs_shift = 8; break;
        case 512: bs_shift = 9; break;
        case 1024: bs_shift = 10; break;
        case 2048: bs_shift = 11; break;
        default:
            set_error(kBadBlocksize, "dequantize_blockwise: blocksize %d is not one of 64,128,256,512,1024,2048", blocksize);
            return;
    }
    if (order_i < 1 || batch < 1 || (int64_t)order_i * order_i * batch >= (int64_t(1) << 31)) {
        set_error(kBadOrder, "dequantize_blockwise: order %d (batch %d) out of range (need order >= 1 and batch*order*order < 2^31)",
                  order_i, batch);
        return;
    }
    if (!q || !code || !absmax || !out || (DIAG && !diag)) {
        set_error(kNullPointer, "dequantize_blockwise: null device pointer");
        return;
    }
    const uint32_t order = (uint32_t)order_i, bs = (uint32_t)blocksize;
    const uint32_t total = order * order * (uint32_t)batch;
    bool flat = order % bs == 0 && is_aligned(out, 4 * sizeof(T)) && is_aligned(q, 16) && is_aligned(absmax, 4);
    if (batch > 65535 && !flat) {
        set_error(kBadArgument, "dequantize_blockwise: a stack whose order the blocksize does not divide (or with unaligned buffers) "
                                "takes at most 65535 matrices per launch");
        return;
    }
    // Small outputs are bound by latency: a thread of the general kernel writes four elements and not thirty-two, and finds
    // the diagonal without a walk.  us, flat and general, one matrix in 4 bits (8 bits the same to 0.1): fp32 256 x 256 3.0 and
    // 2.4, with its diagonal 4.1 and 2.5; 1280 x 1280 3.9 and 3.7, 4.5 and 3.8; 1536 x 1536 4.3 and 4.5, 4.9 and 4.6; 1792 x 1792
    // 4.8 and 5.4, 5.4 and 5.5; bf16 1536 x 1536 4.2 and 3.9, 4.9 and 4.1; 1792 x 1792 4.4 and 4.4, 5.0 and 4.7; 2048 x 2048 4.6 and
    // 5.1, 5.0 and 5.4.
    if (total < (DIAG || sizeof(T) == 2 ? 3u << 20 : 1u << 21)) flat = false;
    if (flat) {
        constexpr uint32_t kWaves = kFlatThreads / 64;
        const uint32_t n_super = total / kSuper;
        const uint32_t blocks = (n_super + kWaves - 1) / kWaves;
        // Workgroups of two waves per unit.  An fp32 output that streams to memory is bound by its stores and takes the fewest
        // that keep them coming (8192 x 8192: 47 us with three, 49.5 with six); one that the last-level cache takes, and
        // bf16, whose look-ups per byte written are twice as many, want more waves to hide them behind: 4096 x 4096 fp32
        // with its diagonal 15.4 us with three, 13.9 with six; bf16 8 bits 14.6 with three, 11.0 with six and with ten, 4
        // bits 14.6, 10.2, 9.5; 12032 x 12032 bf16 80, 59, 61.
        // With the exact diagonal by wave-uniform places (kDiagFew) 4-bit codes do best with five waves per unit, each a workgroup
        // of its own.  us for codes from memory and right behind their quantizer, any place with 3 x 2 waves, few with 3 x 2, few
        // with 5 x 1: 8192 x 8192 104 70 68 and 48 50 47, 10240 x 10240 157 106 108 and 70 74 70, 12032 x 12032 217 147 141 and 95 100
        // 93.  8 bits the same to the noise for both of few, 8192 x 8192 114 81 82 and 51 54 54, 10240 x 10240 169 126 132 and 76 81 80,
        // 12032 x 12032 233 174 178 and 180 117 115: two to seven percent lost where 64 to 110 MB of codes have just been written.
        const bool streams = total >= (1u << 25);
        const dim3 grid(capped_grid(blocks, sizeof(T) == 2 ? (streams ? 6 : 10) : streams ? 3 : 6));
        constexpr int ANY = DIAG ? kDiagAny : kDiagNone, FEW = DIAG ? kDiagFew : kDiagNone;
        // Outputs far beyond the 256 MB last-level cache are written with the streaming hint.
#define QT_DEQUANT_FLAT(KIND, STREAM)                                                                                                   \
        hipLaunchKernelGGL((dequantize_flat_kernel<T, BITS, KIND, STREAM>), grid, dim3(kFlatThreads), 0, stream, q, code, n_super,       \
                           (uint32_t)bs_shift, make_fastdiv(order / 4), make_fastdiv(order), absmax, diag, out)
        constexpr bool ONE = DIAG && BITS == 4 && sizeof(T) == 4;
        if (order >= (uint32_t)kSuper) {
            if (streams)
                hipLaunchKernelGGL((dequantize_flat_kernel<T, BITS, FEW, true, ONE ? 64 : kFlatThreads>), ONE ? dim3(capped_grid(n_super, 5)) : grid,
                                   dim3(ONE ? 64 : kFlatThreads), 0, stream, q, code, n_super, (uint32_t)bs_shift, make_fastdiv(order / 4),
                                   make_fastdiv(order), absmax, diag, out);
            else QT_DEQUANT_FLAT(FEW, false);
        } else if (streams) QT_DEQUANT_FLAT(ANY, true);
        else QT_DEQUANT_FLAT(ANY, false);
#undef QT_DEQUANT_FLAT
    } else {
        const uint32_t nb = (order + bs - 1) / bs;
        const uint32_t one = order * order;
        const bool whole = order % 4 == 0 && is_aligned(q, BITS == 4 ? 2 : 4);
        // A thread per code byte where that is the faster one, back to back: walking over eight elements costs it 3.3 us
        // against 2.6 for 261 x 261, 3.7 against 2.6 for 100 x 27 x 27, 3.8 against 3.7 for 801 x 801, 4.1 against 4.2 for
        // 1001 x 1001; four whole elements 2.6 against 2.5 for 260 x 260 in 8 bits, the same from 340 x 340, and never
        // more in 4 bits.
        const bool bytes = total < (whole ? (BITS == 8 ? 1u << 17 : 0u) : 1000000u);
        const uint32_t n_units = bytes ? (one * BITS + 7) / 8 : whole ? one / 4 : (one + 7) / 8;
        const FastDiv quad_div = make_fastdiv(whole ? order / 4 : 1);
        const dim3 grid(capped_grid((n_units + kThreads - 1) / kThreads, 16), batch);
        if (bytes)
            hipLaunchKernelGGL((dequantize_bytes_kernel<T, BITS, DIAG>), grid, dim3(kThreads), 0, stream,
                               q, code, order, (uint32_t)bs_shift, nb, one, absmax, diag, out);
        else if (whole)
            hipLaunchKernelGGL((dequantize_general_kernel<T, BITS, DIAG, true>), grid, dim3(kThreads), 0, stream,
                               q, code, order, (uint32_t)bs_shift, nb, quad_div, one, absmax, diag, out);
        else
            hipLaunchKernelGGL((dequantize_general_kernel<T, BITS, DIAG, false>), grid, dim3(kThreads), 0, stream,
                               q, code, order, (uint32_t)bs_shift, nb, quad_div, one, absmax, diag, out);
    }
    launch_ok("dequantize_blockwise");
}

}  // namespace
}  // namespace qt

#define QT_DEFINE_DEQUANT(NAME, T, BITS)                                                                                  \
    extern "C" void cdequantize_blockwise_##NAME##_stream(unsigned char *A, float *code, int order, float *absmax,       \
                                                          T *out, int blocksize, void *stream) {                         \
        qt::dequantize_dispatch<T, BITS, false>(A, code, order, absmax, nullptr, out, blocksize, (hipStream_t)stream);   \
    }                                                                                                                    \
    extern "C" void cdequantize_blockwise_##NAME(unsigned char *A, float *code, int order, float *absmax, T *out,        \
                                                 int blocksize) {                                                        \
        qt::dequantize_dispatch<T, BITS, false>(A, code, order, absmax, nullptr, out, blocksize, nullptr);               \
    }                                                                                                                    \
    extern "C" void cdequantize_blockwise_diagreal_##NAME##_stream(unsigned char *A, float *code, int order,             \
                                                                   float *absmax, float *diag, T *out, int blocksize,    \
                                                                   void *stream) {                                       \
        qt::dequantize_dispatch<T, BITS, true>(A, code, order, absmax, diag, out, blocksize, (hipStream_t)stream);       \
    }                                                                                                                    \
    extern "C" void cdequantize_blockwise_diagreal_##NAME(unsigned char *A, float *code, int order, float *absmax,       \
                                                          float *diag, T *out, int blocksize) {                          \
        qt::dequantize_dispatch<T, BITS, true>(A, code, order, absmax, diag, out, blocksize, nullptr);                   \
    }

QT_DEFINE_DEQUANT(8bit_fp32, float, 8)
QT_DEFINE_DEQUANT(8bit_bf16, uint16_t, 8)
QT_DEFINE_DEQUANT(4bit_fp32, float, 4)
QT_DEFINE_DEQUANT(4bit_bf16, uint16_t, 4)

extern "C" void qtensor_hip_dequantize_batched(const unsigned char *q, const float *code, int bits, int order, int batch,
                                               const float *absmax, const float *diag, void *out, int out_is_bf16,
                                               int blocksize, void *stream) {
    using namespace qt;
    hipStream_t st = (hipStream_t)stream;
    if (bits != 4 && bits != 8) { clear_error(); set_error(kBadArgument, "dequantize_batched: bits must be 4 or 8"); return; }
#define QT_DB(T, BITS)                                                                                           \
    (diag ? dequantize_dispatch<T, BITS, true>(q, code, order, absmax, diag, (T *)out, blocksize, st, batch)       \
          : dequantize_dispatch<T, BITS, false>(q, code, order, absmax, nullptr, (T *)out, blocksize, st, batch))
    if (out_is_bf16) { if (bits == 4) QT_DB(uint16_t, 4); else QT_DB(uint16_t, 8); }
    else { if (bits == 4) QT_DB(float, 4); else QT_DB(float, 8); }
#undef QT_DB
}
