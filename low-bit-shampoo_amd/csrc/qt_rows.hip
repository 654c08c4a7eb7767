// Chosen rows of every matrix of a stack, as fp32: from codes, without the other rows, or from an fp32 stack, and if wanted
// each also times its weight (the reference: dequantize, index, multiply per matrix, qtensor/utils.py:200-203 and 205-215).
//
// Bound by the bytes that are written.  A thread takes four neighbouring elements of four runs, all loads ahead of the first
// store; a wave writes a kilobyte at a time.  us, against dequantizing all rows and torch's index: half of the rows from 4 bits
// of 36 x 1024 x 1024 87 -> 18 (4.7 TB/s), 60 x 768 x 768 85 -> 18, 30 x 1200 x 1200 106 -> 19; from fp32 with weights, against index and
// multiply: 72 -> 38, 66 -> 35, 93 -> 50.
#include "qt_common.h"

#include "qtensor_hip.h"

namespace qt {
namespace {

constexpr int kRowThreads = 256, kRuns = 4;

struct RowsArgs {
    const void *from;                                  // codes (BITS 4, 8) or fp32 (32), one matrix after the other
    const float *code, *absmax;
    const long long *rows;                             // [batch][count]
    const float *weight;                               // [batch][count]
    float *out, *scaled;                               // [batch][count][order]
    uint32_t order, bs_shift, nb, count, units;        // units: fours of elements per matrix of the result
    FastDiv quads;                                     // by order / 4
};

template <int BITS, bool SCALED>
__global__ __launch_bounds__(kRowThreads) void rows_kernel(const RowsArgs args) {
    constexpr int NCODE = BITS == 32 ? 1 : 1 << BITS;
    __shared__ float s_code[NCODE];
    const size_t b = blockIdx.y, matrix = (size_t)args.order * args.order;
    float4 y[kRuns];
    float a[kRuns], w[kRuns];
    uint32_t word[kRuns], at[kRuns];
    bool there[kRuns];
#pragma unroll
    for (int i = 0; i < kRuns; ++i) {
        const uint32_t u = min((blockIdx.x * kRuns + i) * kRowThreads + threadIdx.x, args.units - 1);    // (past the end: the last four again)
        const uint32_t r = fastdiv(u, args.quads), c = (u - r * args.quads.divisor) * 4u;
        const long long row = args.rows[b * args.count + r];
        there[i] = (unsigned long long)row < args.order;
        const uint32_t k = (there[i] ? (uint32_t)row : 0u) * args.order + c;
        at[i] = u;
        if (SCALED) w[i] = args.weight[b * args.count + r];
        if (BITS == 32) {
            y[i] = load_f32x4<false>(static_cast<const float *>(args.from) + b * matrix + k);
        } else {
            const uint8_t *codes = static_cast<const uint8_t *>(args.from) + b * (matrix * BITS / 8);
            word[i] = BITS == 4 ? *reinterpret_cast<const uint16_t *>(codes + (k >> 1)) : *reinterpret_cast<const uint32_t *>(codes + k);
            a[i] = args.absmax[b * args.order * args.nb + (there[i] ? (uint32_t)row : 0u) * args.nb + (c >> args.bs_shift)];
        }
    }
    if (BITS != 32) {
        for (int i = threadIdx.x; i < NCODE; i += kRowThreads) s_code[i] = args.code[i];
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < kRuns; ++i) {
        if (BITS != 32) {
            uint32_t id[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) id[e] = BITS == 4 ? word[i] >> (8 * (e >> 1) + ((e & 1) ? 0 : 4)) & 15u : word[i] >> (8 * e) & 255u;
            y[i] = a[i] == 0.0f ? make_float4(0.0f, 0.0f, 0.0f, 0.0f)
                                : make_float4(s_code[id[0] % NCODE] * a[i], s_code[id[1] % NCODE] * a[i], s_code[id[2] % NCODE] * a[i], s_code[id[3] % NCODE] * a[i]);
        }
        const float nan = __uint_as_float(0x7fc00000u);
        if (!there[i]) y[i] = make_float4(nan, nan, nan, nan);       // a row that no matrix has
        const size_t to = (b * args.units + at[i]) * 4;
        store_f32x4<false>(args.out + to, y[i]);
        if (SCALED) store_f32x4<false>(args.scaled + to, make_float4(y[i].x * w[i], y[i].y * w[i], y[i].z * w[i], y[i].w * w[i]));
    }
}

template <int BITS>
void launch_rows(const RowsArgs &args, int batch, hipStream_t stream) {
    const dim3 grid((args.units + kRowThreads * kRuns - 1) / (kRowThreads * kRuns), batch);
    if (args.scaled) hipLaunchKernelGGL((rows_kernel<BITS, true>), grid, dim3(kRowThreads), 0, stream, args);
    else hipLaunchKernelGGL((rows_kernel<BITS, false>), grid, dim3(kRowThreads), 0, stream, args);
}

}  // namespace
}  // namespace qt

extern "C" void qtensor_hip_rows_batched(const void *from, int bits, const float *code, const float *absmax, int blocksize, int order, int batch,
                                         const long long *rows, int count, const float *weight, float *out, float *scaled, void *stream_v) {
    using namespace qt;
    clear_error();
    const bool codes = bits == 4 || bits == 8;
    if (!from || !rows || !out || (codes && (!code || !absmax)) || (scaled && !weight)) { set_error(kNullPointer, "rows_batched: null device pointer"); return; }
    if ((!codes && bits != 32) || order < 4 || order % 4 || (long long)order * order >= (1LL << 31) || batch < 1 || batch > 65535 || count < 1 ||
        count > order) {
        set_error(kBadArgument, "rows_batched: needs 4, 8 or 32 bits, an order that is a multiple of four, 1 to 65535 matrices and 1 to order rows of each "
                                "(got %d bits, order %d, %d matrices, %d rows)", bits, order, batch, count);
        return;
    }
    if (codes && (blocksize < 64 || blocksize > 2048 || (blocksize & (blocksize - 1)))) {
        set_error(kBadBlocksize, "rows_batched: blocksize %d is not one of 64,128,256,512,1024,2048", blocksize);
        return;
    }
    if (!is_aligned(out, 16) || (scaled && !is_aligned(scaled, 16)) || !is_aligned(from, bits == 32 ? 16 : bits == 8 ? 4 : 2)) {
        set_error(kBadArgument, "rows_batched: unaligned buffer");
        return;
    }
    const RowsArgs args = {from, code, absmax, rows, weight, out, scaled, (uint32_t)order, codes ? (uint32_t)__builtin_ctz((unsigned)blocksize) : 0u,
                           codes ? (uint32_t)((order + blocksize - 1) / blocksize) : 0u, (uint32_t)count, (uint32_t)count * (uint32_t)(order / 4),
                           make_fastdiv((uint32_t)order / 4)};
    if (bits == 4) launch_rows<4>(args, batch, (hipStream_t)stream_v);
    else if (bits == 8) launch_rows<8>(args, batch, (hipStream_t)stream_v);
    else launch_rows<32>(args, batch, (hipStream_t)stream_v);
    launch_ok("rows_batched");
}
