// What the coupled Newton iteration does between its products, for a whole stack of matrices: the start (ridge, norm,
// first iterates), the power iteration's normalised vectors, the stopping rules and the choice of buffers, the result.
// The reference does these per matrix on the host (optimizers/matrix_functions.py:30-48, 100-141).
//
// Every one of them is a small kernel or one pass over the stack, and what they cost is launches: as torch operations a
// round took 22 of them beside its four products and a power iteration's step 11, most of 3 to 5 us in a chain.  One
// launch each here.  Inverse roots over a ViT-B/32's weights (248 matrices, seven parts): 3409 -> 591 launches.
#include "qt_common.h"
#include "qt_half.h"

namespace qt {
namespace {

constexpr int kBand = 8;                       // rows that a workgroup of the passes over a stack takes: the pieces of qt_half.h
                                               // are up to eight elements of a column

// Sum over the workgroup's 256 threads, delivered to all of them; the order is fixed.
__device__ __forceinline__ double block_sum(double x, double *s_wave) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    __syncthreads();                           // the last sum may still be read
    if ((threadIdx.x & 63) == 0) s_wave[threadIdx.x >> 6] = x;
    __syncthreads();
    return (s_wave[0] + s_wave[1]) + (s_wave[2] + s_wave[3]);
}

// u = v / |v| of every vector, v = what the product with u gave (`product`) or a start vector, unless its Rayleigh quotient
// has settled.  Sums in double precision: their rounding does not depend on the order.  A workgroup per matrix.
__global__ __launch_bounds__(256) void power_step_kernel(const float *product, float *u, float *value, float *change, int n, float tolerance, int first) {
    __shared__ double s_wave[4];
    const long long b = blockIdx.x;
    const float *v = product + b * n;
    float *at = u + b * n;
    if (first) {
        if (threadIdx.x == 0) { value[b] = 0.0f; change[b] = 1.0f; }
    } else {
        if (!(change[b] > tolerance)) return;                          // (the same for the whole workgroup)
        double dot = 0.0;
        for (int i = threadIdx.x; i < n; i += 256) dot += (double)(at[i] * v[i]);
        const float quotient = (float)block_sum(dot, s_wave);          // (and every thread has read change[b])
        if (threadIdx.x == 0) { change[b] = fabsf(quotient - value[b]); value[b] = quotient; }
    }
    double square = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) square += (double)v[i] * (double)v[i];
    const float norm = (float)sqrt(block_sum(square, s_wave));
    for (int i = threadIdx.x; i < n; i += 256) at[i] = v[i] / norm;
}

// Four elements of a stack that need not begin on a 16-byte boundary (wide: it does).
__device__ __forceinline__ float4 load_four(const float *p, bool wide) {
    return wide ? load_f32x4<false>(p) : make_float4(p[0], p[1], p[2], p[3]);
}

// The ridge onto the diagonal, and the sum of squares of every band of rows.
__global__ __launch_bounds__(256) void newton_norm_kernel(float *mats, const float *top, float ridge, int n, int bands, double *partial) {
    __shared__ double s_wave[4];
    const long long b = blockIdx.x / (unsigned)bands;
    const int r0 = (int)(blockIdx.x % (unsigned)bands) * kBand, rows = min(kBand, n - r0);
    float *base = mats + (b * n + r0) * n;
    const float add = ridge * top[b];
    if ((int)threadIdx.x < rows) base[(long long)threadIdx.x * n + r0 + threadIdx.x] += add;
    __syncthreads();
    double sum = 0.0;
    if ((n & 3) == 0) {
        const bool wide = is_aligned16(mats);
        for (int i = threadIdx.x; i < rows * (n >> 2); i += 256) {
            const float4 x = load_four(base + 4ll * i, wide);
            sum += ((double)x.x * x.x + (double)x.y * x.y) + ((double)x.z * x.z + (double)x.w * x.w);
        }
    } else {
        for (int i = threadIdx.x; i < rows * n; i += 256) sum += (double)base[i] * base[i];
    }
    sum = block_sum(sum, s_wave);
    if (threadIdx.x == 0) partial[blockIdx.x] = sum;
}

// First iterates: M = z A with z = (1 + p) / (2 |A|), E = M - I, the candidate root of the first round c (I + w E) with
// c = z^(1/p), w = -1/p; err = max |E|; fine (optional): raised to the fineness of E and M.  A thread takes squares of 8 rows by
// 4 columns, so that the pieces lie inside one thread.  Where M, E or R do not lie on 16-byte boundaries, nobody looks at the pieces
// and the fineness is that of pieces of any size, infinity, as behind a product whose output does not.
__global__ __launch_bounds__(256) void newton_first_kernel(const float *mats, const double *partial, int p, int n, int bands, float *M, float *E,
                                                           float *R, float *first_root, float *err, float *fine) {
    __shared__ double s_wave[4];
    const long long b = blockIdx.x / (unsigned)bands;
    const int r0 = (int)(blockIdx.x % (unsigned)bands) * kBand, rows = min(kBand, n - r0);
    double sum = 0.0;
    for (int i = threadIdx.x; i < bands; i += 256) sum += partial[b * bands + i];
    const float z = (float)(1 + p) / (2.0f * (float)sqrt(block_sum(sum, s_wave)));
    const float c = powf(z, 1.0f / (float)p), step = -1.0f / (float)p * c;
    if (r0 == 0 && threadIdx.x == 0) first_root[b] = c;
    const long long base = (b * n + r0) * n;
    uint32_t top = 0;
    Pieces seen;
    if ((n & 3) == 0 && is_aligned16(M) && is_aligned16(E) && is_aligned16(R)) {
        const bool wide = is_aligned16(mats);
        for (int q = threadIdx.x; q < n >> 2; q += 256) {
            const int c0 = q * 4;
            Pieces seen_m;                                             // (a run of rows of each)
            float4 x[kBand];
#pragma unroll
            for (int r = 0; r < kBand; ++r) x[r] = load_four(mats + base + (long long)min(r, rows - 1) * n + c0, wide);
#pragma unroll
            for (int r = 0; r < kBand; ++r) {
                if (r >= rows) break;
                const float a[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
                float m[4], e[4], t[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool diagonal = c0 + i == r0 + r;
                    m[i] = a[i] * z;
                    e[i] = diagonal ? m[i] - 1.0f : m[i];
                    t[i] = e[i] * step;
                    if (diagonal) t[i] += c;
                    top = max(top, __float_as_uint(e[i]) & 0x7fffffffu);
                }
                seen_m.row(m);
                seen.row(e);
                const long long at = base + (long long)r * n + c0;
                store_f32x4<false>(M + at, make_float4(m[0], m[1], m[2], m[3]));
                store_f32x4<false>(E + at, make_float4(e[0], e[1], e[2], e[3]));
                store_f32x4<false>(R + at, make_float4(t[0], t[1], t[2], t[3]));
            }
            seen_m.end();
            seen.end();
            seen.low = min(seen.low, seen_m.low);
        }
    } else {
        seen.low = 0;
        for (int i = threadIdx.x; i < rows * n; i += 256) {
            const bool diagonal = i % n == r0 + i / n;
            const float m = mats[base + i] * z, e = diagonal ? m - 1.0f : m;
            top = max(top, __float_as_uint(e) & 0x7fffffffu);
            M[base + i] = m;
            E[base + i] = e;
            R[base + i] = diagonal ? e * step + c : e * step;
        }
    }
    top = group_max_u32<64>(top);                                      // (NaN above everything finite)
    const uint32_t low = group_max_u32<64>(~seen.low);
    if ((threadIdx.x & 63) == 0) {
        raise_word(reinterpret_cast<uint32_t *>(err) + b, top);
        if (fine != nullptr) raise_fineness(reinterpret_cast<uint32_t *>(fine) + b, ~low);
    }
}

}  // namespace
}  // namespace qt

// include/qtensor_hip.h: qtensor_newton_state
struct qtensor_newton_state {
    int batch, iterations;
    float tolerance, step;
    float *err;
    int *done, *side, *rounds;
    const float *first_root, *first_fine;
    float *root_bound, *root_fine;
    long long *tables;
    long long buffers[6], stride;
};

namespace qt {
namespace {

// Whether the round that has just been multiplied out is accepted, which matrices go on, and where their iterates lie.
// new_err == nullptr: before the first round.  A thread per matrix.
__global__ __launch_bounds__(256) void newton_decide_kernel(const qtensor_newton_state s, const float *new_err, float *bound_m) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= s.batch) return;
    float err = s.err[b];
    int side = 0, rounds = 0, done = 0;
    if (new_err != nullptr) {
        const float next = new_err[b];
        side = s.side[b]; rounds = s.rounds[b]; done = s.done[b];
        const bool accept = !done && !(next > err * 1.2f);
        if (accept) { side ^= 1; ++rounds; err = next; s.err[b] = next; }
        else done = 1;
        if (bound_m != nullptr) bound_m[b] = 1.0f + next;
    } else {
        if (bound_m != nullptr) bound_m[b] = 1.0f + err;
        if (s.root_bound != nullptr) {         // of the root after the first round, c (I + w E): small pieces are c w times those of E
            const float c = s.first_root[b], w = fabsf(s.step);
            s.root_bound[b] = c * (1.0f + w * err);
            s.root_fine[b] = s.first_fine[b] / (w * c);
        }
    }
    if (err <= s.tolerance || rounds >= s.iterations) done = 1;
    s.done[b] = done; s.side[b] = side; s.rounds[b] = rounds;
#pragma unroll
    for (int which = 0; which < 3; ++which)
#pragma unroll
        for (int other = 0; other < 2; ++other)
            s.tables[(long long)(2 * which + other) * s.batch + b] = s.buffers[2 * which + (side ^ other)] + b * s.stride;
}

// out[b] = the accepted root: c I before the first round, else what lies in the buffer of `side` (out may be either buffer:
// what is there already is left alone).
__global__ __launch_bounds__(256) void newton_result_kernel(const float *r0, const float *r1, const int *side, const int *rounds,
                                                            const float *first_root, float *out, int n, unsigned groups) {
    const long long b = blockIdx.x / groups, size = (long long)n * n;
    const float *from = (side[b] ? r1 : r0) + b * size;
    float *to = out + b * size;
    const bool none = rounds[b] == 0;
    if (!none && from == to) return;
    const float c = first_root[b];
    const long long first = (long long)(blockIdx.x % groups) * 4096, last = min(size, first + 4096);
    if ((n & 3) == 0 && is_aligned16(from) && is_aligned16(to) && !none) {
        for (long long i = first + 4 * threadIdx.x; i < last; i += 1024) store_f32x4<false>(to + i, load_f32x4<false>(from + i));
        return;
    }
    for (long long i = first + threadIdx.x; i < last; i += 256) to[i] = !none ? from[i] : i / n == i % n ? c : 0.0f;
}

bool sizes_ok(const char *what, int n, int batch, long long blocks) {
    if (n >= 1 && batch >= 1 && n <= 46340 && blocks <= 0x7fffffffLL) return true;
    set_error(kBadArgument, "%s: need 1 <= n <= 46340 and 1 <= batch, not too many of them (got %d, %d)", what, n, batch);
    return false;
}

}  // namespace
}  // namespace qt

extern "C" void qtensor_hip_power_step_batched(const float *product, float *u, float *value, float *change, int n, int batch, float tolerance,
                                               int first, void *stream) {
    using namespace qt;
    clear_error();
    if (!product || !u || !value || !change) { set_error(kNullPointer, "power_step_batched: null pointer"); return; }
    if (!sizes_ok("power_step_batched", n, batch, batch)) return;
    hipLaunchKernelGGL(power_step_kernel, dim3((unsigned)batch), dim3(256), 0, (hipStream_t)stream, product, u, value, change, n, tolerance, first);
    launch_ok("power_step_batched");
}

extern "C" void qtensor_hip_newton_first_batched(float *mats, const float *top, float ridge, int p, int n, int batch, double *partial, float *M,
                                                 float *E, float *R, float *first_root, float *err, float *fine, void *stream) {
    using namespace qt;
    clear_error();
    if (!mats || !top || !partial || !M || !E || !R || !first_root || !err) { set_error(kNullPointer, "newton_first_batched: null pointer"); return; }
    const int bands = n < 1 ? 0 : (n + kBand - 1) / kBand;
    if (!sizes_ok("newton_first_batched", n, batch, (long long)bands * batch)) return;
    if (p < 1) { set_error(kBadArgument, "newton_first_batched: need p >= 1 (got %d)", p); return; }
    if (fine && (n & 3)) { set_error(kBadArgument, "newton_first_batched: finenesses of orders in multiples of 4 (got %d)", n); return; }
    const dim3 grid((unsigned)bands * (unsigned)batch);
    hipLaunchKernelGGL(newton_norm_kernel, grid, dim3(256), 0, (hipStream_t)stream, mats, top, ridge, n, bands, partial);
    hipLaunchKernelGGL(newton_first_kernel, grid, dim3(256), 0, (hipStream_t)stream, mats, partial, p, n, bands, M, E, R, first_root, err, fine);
    launch_ok("newton_first_batched");
}

extern "C" void qtensor_hip_newton_decide(const qtensor_newton_state *s, const float *new_err, float *bound_m, void *stream) {
    using namespace qt;
    clear_error();
    if (!s || !s->err || !s->done || !s->side || !s->rounds || !s->tables) { set_error(kNullPointer, "newton_decide: null pointer"); return; }
    if (s->root_bound && (!s->root_fine || !s->first_root || !s->first_fine)) { set_error(kNullPointer, "newton_decide: null pointer"); return; }
    if (s->batch < 1) { set_error(kBadArgument, "newton_decide: need batch >= 1 (got %d)", s->batch); return; }
    hipLaunchKernelGGL(newton_decide_kernel, dim3(((unsigned)s->batch + 255) / 256), dim3(256), 0, (hipStream_t)stream, *s, new_err, bound_m);
    launch_ok("newton_decide");
}

extern "C" void qtensor_hip_newton_result_batched(const float *r0, const float *r1, const int *side, const int *rounds, const float *first_root,
                                                  float *out, int n, int batch, void *stream) {
    using namespace qt;
    clear_error();
    if (!r0 || !r1 || !side || !rounds || !first_root || !out) { set_error(kNullPointer, "newton_result_batched: null pointer"); return; }
    const long long groups = n < 1 ? 0 : ((long long)n * n + 4095) / 4096;
    if (!sizes_ok("newton_result_batched", n, batch, groups * batch)) return;
    hipLaunchKernelGGL(newton_result_kernel, dim3((unsigned)(groups * batch)), dim3(256), 0, (hipStream_t)stream, r0, r1, side, rounds, first_root,
                       out, n, (unsigned)groups);
    launch_ok("newton_result_batched");
}
