// The elementwise end of a Shampoo optimizer step for all parameters in two launches:
//   1. per tensor, |grad|^2 and |direction|^2 (deterministic two-level sums);
//   2. direction *= |grad| / (|direction| + 1e-12)   (layer-wise grafting, optimizers/shampoo1.py:421
//      and shampoo2.py:453 of the reference), followed by the AdamW update (shampoo1.py:405-427,
//      shampoo2.py:446-468) or the SGD-with-momentum update (shampoo1.py:310-331, shampoo2.py:346-367).
// The reference does this with a dozen small torch kernels per parameter.
//
// Work is cut into chunks of kChunk consecutive elements of one tensor, one workgroup each;
// the table of tensors and the chunk -> tensor map live in device memory and are written by
// the caller once (they only change when a buffer moves).
#include "qt_common.h"

namespace qt {

struct TailTensor {            // one row of the device table: 8 x 64 bit
    float *param;
    const float *dir;          // preconditioned gradient (or the gradient itself)
    const float *grad;         // only read when the row is grafted
    float *m;                  // AdamW: exp_avg, SGD: momentum buffer
    float *v;                  // AdamW: exp_avg_sq, SGD: unused
    long long n;               // elements
    long long first_chunk;     // index of this tensor's first chunk
    long long flags;           // bit 0: rescale dir to the norm of grad; bit 1: stream past the caches
};

namespace {

constexpr int kChunk = 16384;  // elements per workgroup: sixteen float4 per thread
constexpr int kThreads = 256;

#define QT_GLOBAL __attribute__((address_space(1)))
template <bool STREAM = false>
__device__ __forceinline__ float4 g4(const float *p) {
    const qt_f32x4 v = STREAM ? __builtin_nontemporal_load((const QT_GLOBAL qt_f32x4 *)p) : *(const QT_GLOBAL qt_f32x4 *)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
template <bool STREAM = false>
__device__ __forceinline__ void s4(float *p, float4 y) {
    qt_f32x4 v;
    v.x = y.x; v.y = y.y; v.z = y.z; v.w = y.w;
    if (STREAM) __builtin_nontemporal_store(v, (QT_GLOBAL qt_f32x4 *)p);
    else *(QT_GLOBAL qt_f32x4 *)p = v;
}
__device__ __forceinline__ float g1(const float *p) { return *(const QT_GLOBAL float *)p; }
__device__ __forceinline__ void s1(float *p, float y) { *(QT_GLOBAL float *)p = y; }

__device__ __forceinline__ float block_sum(float x, float *s_part) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) s_part[wave] = x;
    __syncthreads();
    const float total = (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
    __syncthreads();
    return total;
}

// partial[2c] = sum grad^2, partial[2c+1] = sum dir^2 over chunk c (rows without graft: untouched)
template <bool STREAM>
__device__ __forceinline__ void norms_of_chunk(const TailTensor &t, int c, float *partial, float *s_part) {
    const long long start = ((long long)c - t.first_chunk) * kChunk;
    const long long left = t.n - start;
    const int len = left < kChunk ? (int)left : kChunk;
    const float *g = t.grad + start, *d = t.dir + start;
    float sg = 0.f, sd = 0.f;
    if (is_aligned16(g) && is_aligned16(d)) {
#pragma unroll 4
        for (int i = threadIdx.x * 4; i < len; i += kThreads * 4) {
            if (i + 3 < len) {
                const float4 a = g4<STREAM>(g + i), b = g4(d + i);
                sg += (a.x * a.x + a.y * a.y) + (a.z * a.z + a.w * a.w);
                sd += (b.x * b.x + b.y * b.y) + (b.z * b.z + b.w * b.w);
            } else {
                for (int e = i; e < len; ++e) { const float a = g1(g + e), b = g1(d + e); sg += a * a; sd += b * b; }
            }
        }
    } else {
        for (int i = threadIdx.x; i < len; i += kThreads) { const float a = g1(g + i), b = g1(d + i); sg += a * a; sd += b * b; }
    }
    sg = block_sum(sg, s_part);
    sd = block_sum(sd, s_part);
    if (threadIdx.x == 0) { s1(partial + 2 * c, sg); s1(partial + 2 * c + 1, sd); }
}

__global__ __launch_bounds__(kThreads) void tail_norms_kernel(const TailTensor *table, const int *chunk_tensor,
                                                              float *partial) {
    __shared__ float s_part[4];
    const TailTensor t = table[chunk_tensor[blockIdx.x]];
    if (!(t.flags & 1)) return;
    if (t.flags & 2) norms_of_chunk<true>(t, blockIdx.x, partial, s_part);
    else norms_of_chunk<false>(t, blockIdx.x, partial, s_part);
}

// |grad| / (|dir| + 1e-12) of the tensor that owns this chunk, summed in an order of its own number of chunks alone (the same
// value in every workgroup of the tensor).  By a wave: one thread that walked over the 144 chunks of a 768 x 3072 tensor
// kept its workgroup waiting.
__device__ __forceinline__ float graft_scale(const TailTensor &t, const float *partial, float *s_scale) {
    if (!(t.flags & 1)) return 1.0f;
    if (threadIdx.x < 64) {
        const long long chunks = (t.n + kChunk - 1) / kChunk;
        double sg = 0.0, sd = 0.0;
        for (long long c = threadIdx.x; c < chunks; c += 64) {
            const float *at = partial + 2 * (t.first_chunk + c);
            sg += (double)g1(at);
            sd += (double)g1(at + 1);
        }
        if (chunks > 1)                                          // (a small tensor's are on lane 0)
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) { sg += __shfl_xor(sg, off, 64); sd += __shfl_xor(sd, off, 64); }
        if (threadIdx.x == 0) {
            const float gn = (float)sqrt(sg), dn = (float)sqrt(sd);
            *s_scale = gn / (dn + 1e-12f);
        }
    }
    __syncthreads();
    return *s_scale;
}

struct AdamW {
    float decay, beta1, alpha1, beta2, alpha2, sqrt_c2, eps, neg_step;
    const float *row_corrections;      // optional: {sqrt(1 - beta2^t), -lr / (1 - beta1^t)} per table row (its own step count t)
    __device__ __forceinline__ void bind(int row) {
        if (row_corrections != nullptr) { sqrt_c2 = g1(row_corrections + 2 * row); neg_step = g1(row_corrections + 2 * row + 1); }
    }
    __device__ __forceinline__ void operator()(float &p, float &m, float &v, float d) const {
        p = p * decay;
        m = m * beta1 + alpha1 * d;
        v = v * beta2 + (alpha2 * d) * d;
        const float denom = sqrtf(v) / sqrt_c2 + eps;
        p = p + neg_step * (m / denom);
    }
};

struct Sgd {
    float momentum, weight_decay, neg_lr;
    int nesterov;
    __device__ __forceinline__ void bind(int) {}
    __device__ __forceinline__ void operator()(float &p, float &m, float &v, float d) const {
        (void)v;
        if (weight_decay != 0.0f) d = d + weight_decay * p;
        m = m * momentum + d;
        const float u = nesterov ? d + momentum * m : m;
        p = p + neg_lr * u;
    }
};

// A thread's first elements are on their way while the scale is summed up, the next ones while it works on the ones before.
// STREAM: every buffer is touched once a step, and the buffers of a step are more than the last-level cache holds.  Whether they are
// is in the table (bit 1 of a row's flags, the same in all), whose writer knows how many elements there are: from 2^24 on, of
// which they (20 to 28 bytes each) no longer fit its 256 MB.  The number of chunks does not say: a thousand small tensors have as
// many.  Bound by memory: AdamW over the 87.4 M elements of a ViT-B/32 460 -> 422 us, 5.8 TB/s.
template <typename RULE, bool HAS_V, bool STREAM>
__device__ __forceinline__ void update_chunk(const TailTensor &t, int c, const float *partial, const RULE &rule, float *s_scale) {
    const bool graft = (t.flags & 1) != 0;
    const long long start = ((long long)c - t.first_chunk) * kChunk;
    const long long left = t.n - start;
    const int len = left < kChunk ? (int)left : kChunk;
    float *p = t.param + start, *m = t.m + start, *v = HAS_V ? t.v + start : nullptr;
    const float *d = t.dir + start;
    const bool vec = is_aligned16(p) && is_aligned16(m) && is_aligned16(d) && (!HAS_V || is_aligned16(v));
    if (vec) {
        struct Four { float4 p, m, d, v; };
        const int whole = len & ~3;
        auto load = [&](int i) {
            Four x;
            x.p = g4<STREAM>(p + i);
            x.m = g4<STREAM>(m + i);
            x.d = g4<STREAM>(d + i);
            x.v = HAS_V ? g4<STREAM>(v + i) : make_float4(0.f, 0.f, 0.f, 0.f);
            return x;
        };
        int i = threadIdx.x * 4;
        Four x = {}, y = {};
        if (i < whole) x = load(i);
        const float scale = graft_scale(t, partial, s_scale);
        for (; i < whole; i += kThreads * 4) {
            if (i + kThreads * 4 < whole) y = load(i + kThreads * 4);
            if (graft) { x.d.x *= scale; x.d.y *= scale; x.d.z *= scale; x.d.w *= scale; }
            rule(x.p.x, x.m.x, x.v.x, x.d.x);
            rule(x.p.y, x.m.y, x.v.y, x.d.y);
            rule(x.p.z, x.m.z, x.v.z, x.d.z);
            rule(x.p.w, x.m.w, x.v.w, x.d.w);
            s4<STREAM>(p + i, x.p);
            s4<STREAM>(m + i, x.m);
            if (HAS_V) s4<STREAM>(v + i, x.v);
            x = y;
        }
        if ((int)threadIdx.x < len - whole) {
            const int e = whole + threadIdx.x;
            float P = g1(p + e), M = g1(m + e), V = HAS_V ? g1(v + e) : 0.f, D = g1(d + e);
            if (graft) D *= scale;
            rule(P, M, V, D);
            s1(p + e, P); s1(m + e, M);
            if (HAS_V) s1(v + e, V);
        }
    } else {
        const float scale = graft_scale(t, partial, s_scale);
        for (int e = threadIdx.x; e < len; e += kThreads) {
            float P = g1(p + e), M = g1(m + e), V = HAS_V ? g1(v + e) : 0.f, D = g1(d + e);
            if (graft) D *= scale;
            rule(P, M, V, D);
            s1(p + e, P); s1(m + e, M);
            if (HAS_V) s1(v + e, V);
        }
    }
}

template <typename RULE, bool HAS_V>
__global__ __launch_bounds__(kThreads) void tail_update_kernel(const TailTensor *table, const int *chunk_tensor,
                                                               const float *partial, const RULE launch_rule) {
    __shared__ float s_scale;
    const TailTensor t = table[chunk_tensor[blockIdx.x]];
    RULE rule = launch_rule;
    rule.bind(chunk_tensor[blockIdx.x]);
    if (t.flags & 2) update_chunk<RULE, HAS_V, true>(t, blockIdx.x, partial, rule, &s_scale);
    else update_chunk<RULE, HAS_V, false>(t, blockIdx.x, partial, rule, &s_scale);
}

bool tail_args_ok(const void *table, const void *chunk_tensor, int n_chunks, const void *partial, int graft, const char *what) {
    if (!table || !chunk_tensor || (graft && !partial)) { set_error(kNullPointer, "%s: null table, chunk map or partial-sum buffer", what); return false; }
    if (n_chunks < 0) { set_error(kBadArgument, "%s: negative chunk count", what); return false; }
    return true;
}

}  // namespace
}  // namespace qt

extern "C" int qtensor_hip_tail_chunk(void) { return qt::kChunk; }

namespace qt {
namespace {
void adamw_tail(const void *table, const int *chunk_tensor, int n_chunks, float *partial, int graft, double lr, double beta1,
                double beta2, double eps, double weight_decay, long long step, const float *row_corrections, void *stream) {
    clear_error();
    if (!tail_args_ok(table, chunk_tensor, n_chunks, partial, graft, "adamw_tail")) return;
    if (row_corrections == nullptr && step < 1) { set_error(kBadArgument, "adamw_tail: step counts from 1"); return; }
    if (n_chunks == 0) return;
    const TailTensor *tab = static_cast<const TailTensor *>(table);
    if (graft) {
        hipLaunchKernelGGL(tail_norms_kernel, dim3(n_chunks), dim3(kThreads), 0, (hipStream_t)stream, tab, chunk_tensor, partial);
        if (!launch_ok("adamw_tail (norms)")) return;
    }
    AdamW rule;
    rule.decay = (float)(1.0 - lr * weight_decay);
    rule.beta1 = (float)beta1;
    rule.alpha1 = (float)(1.0 - beta1);
    rule.beta2 = (float)beta2;
    rule.alpha2 = (float)(1.0 - beta2);
    rule.sqrt_c2 = row_corrections != nullptr ? 1.0f : (float)sqrt(1.0 - pow(beta2, (double)step));
    rule.eps = (float)eps;
    rule.neg_step = row_corrections != nullptr ? 0.0f : (float)(-lr / (1.0 - pow(beta1, (double)step)));
    rule.row_corrections = row_corrections;
    hipLaunchKernelGGL((tail_update_kernel<AdamW, true>), dim3(n_chunks), dim3(kThreads), 0, (hipStream_t)stream, tab,
                       chunk_tensor, partial, rule);
    launch_ok("adamw_tail");
}
}  // namespace
}  // namespace qt

extern "C" void qtensor_hip_adamw_tail(const void *table, const int *chunk_tensor, int n_chunks, float *partial, int graft,
                                       double lr, double beta1, double beta2, double eps, double weight_decay,
                                       long long step, void *stream) {
    qt::adamw_tail(table, chunk_tensor, n_chunks, partial, graft, lr, beta1, beta2, eps, weight_decay, step, nullptr, stream);
}

extern "C" void qtensor_hip_adamw_tail_rows(const void *table, const int *chunk_tensor, int n_chunks, float *partial, int graft,
                                            double lr, double beta1, double beta2, double eps, double weight_decay,
                                            const float *row_corrections, void *stream) {
    if (row_corrections == nullptr) {
        qt::clear_error();
        qt::set_error(qt::kNullPointer, "adamw_tail_rows: null row_corrections");
        return;
    }
    qt::adamw_tail(table, chunk_tensor, n_chunks, partial, graft, lr, beta1, beta2, eps, weight_decay, 0, row_corrections, stream);
}

extern "C" void qtensor_hip_sgd_tail(const void *table, const int *chunk_tensor, int n_chunks, float *partial, int graft,
                                     double lr, double momentum, double weight_decay, int nesterov, void *stream) {
    using namespace qt;
    clear_error();
    if (!tail_args_ok(table, chunk_tensor, n_chunks, partial, graft, "sgd_tail")) return;
    if (n_chunks == 0) return;
    const TailTensor *tab = static_cast<const TailTensor *>(table);
    if (graft) {
        hipLaunchKernelGGL(tail_norms_kernel, dim3(n_chunks), dim3(kThreads), 0, (hipStream_t)stream, tab, chunk_tensor, partial);
        if (!launch_ok("sgd_tail (norms)")) return;
    }
    Sgd rule;
    rule.momentum = (float)momentum;
    rule.weight_decay = (float)weight_decay;
    rule.neg_lr = (float)(-lr);
    rule.nesterov = nesterov != 0;
    hipLaunchKernelGGL((tail_update_kernel<Sgd, false>), dim3(n_chunks), dim3(kThreads), 0, (hipStream_t)stream, tab,
                       chunk_tensor, partial, rule);
    launch_ok("sgd_tail");
}
