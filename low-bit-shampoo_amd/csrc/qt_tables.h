// Device-side code-table preparation shared by the quantize kernels.
//
// The reference picks a table entry for v = x / absmax as follows (qtensor/functional.py:703-715):
// ins = #{entries <= v}; lo = max(ins-1,0); hi = min(ins,n-1); take hi iff
// |fl(v - code[lo])| > |fl(code[hi] - v)|, else lo.  Inside one gap [code[i], code[i+1]] both
// rounded distances are monotone in v, so the rule flips exactly once: there is a smallest
// fp32 value thr[i] from which entry i+1 is taken.  The chosen index is therefore
// #{i : !(v < thr[i])} -- which also gives 0 below the table, n-1 above it and n-1 for NaN,
// the values the reference's clamp + searchsorted produce.  thr[] is found per workgroup by
// bisection over fp32 bit patterns with the reference's own predicate, so it is exact for any
// table, not just the two shipped ones.
#pragma once

#include "qt_common.h"
#include "qt_divide.h"

namespace qt {

constexpr int kFlagAscending = 1;  // caller's table was already non-decreasing (perm = identity)
constexpr int kFlagLut = 2;        // bucket table usable (at most one threshold per bucket, none near 0)

// Bucket table geometry: a bucket is what an fp16 number with six mantissa bits is, v rounded towards zero (sign, exponent
// and six bits of the twelve that are left of v's conversion: one instruction for two values, then a shift and a mask).
// |v| reaches up to 1; below 2^-14, where fp16 has no exponents left, the buckets are 2^-20 wide.
constexpr int kLutTop = 0x3c0;             // 1.0; what lies beyond shares its bucket
constexpr int kLutNegative = 0x800;
constexpr int kLutEntries = kLutNegative + kLutTop + 1;
constexpr int kLutPlaces = 2 * (kLutTop + 1);      // buckets that are used, in ascending order of their values: lut_place

#if defined(__HIPCC__)

template <int NCODE>
struct alignas(16) CodeTables {
    float code[NCODE];     // ascending
    float thr[NCODE];      // thr[i], i < NCODE-1; last slot = +inf
    float raw[NCODE];      // caller's order
    uint8_t perm[NCODE];   // ascending position -> caller's index
    int flags;
    uint32_t wave_sum[4];
};

__device__ __forceinline__ bool takes_upper(float v, float clo, float chi) {
    if (v >= chi) return true;
    float dlo = v - clo;   // compiled with -ffp-contract=off: two separate fp32 roundings
    float dhi = chi - v;
    return fabsf(dlo) > fabsf(dhi);
}

// Two values as packed fp16, towards zero.
__device__ __forceinline__ uint32_t lut_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}
__device__ __forceinline__ int lut_bucket(float v) {
    const uint32_t p = lut_pair(v, 0.0f) >> 4;
    return (int)((p & kLutNegative) | min(p & 0x7ffu, (uint32_t)kLutTop));
}
__device__ __forceinline__ int lut_place(int p) { return p <= kLutTop ? kLutNegative + kLutTop - p : p - kLutTop - 1; }

// #{i < NCODE-1 : !(v < thr[i])}; thr ascending.  NaN counts everything -> NCODE-1.
template <int NCODE>
__device__ __forceinline__ int count_thresholds(float v, const float *thr) {
    if constexpr (NCODE == 16) {
        // two levels of four: the quarter from three fixed thresholds (reads that do not depend on v), then the
        // three thresholds inside it in one 16-byte read -- one dependent LDS access instead of four
        const int quarter = (int)!(v < thr[3]) + (int)!(v < thr[7]) + (int)!(v < thr[11]);
        const float4 t = *reinterpret_cast<const float4 *>(thr + 4 * quarter);
        return 4 * quarter + (int)!(v < t.x) + (int)!(v < t.y) + (int)!(v < t.z);
    } else {
        int pos = 0;
#pragma unroll
        for (int step = NCODE / 2; step >= 1; step >>= 1)
            if (!(v < thr[pos + step - 1])) pos += step;
        return pos;
    }
}

// The smallest value from which the upper of two neighbouring entries is taken.
__device__ __forceinline__ float entry_threshold(float clo, float chi) {
    if (takes_upper(clo, clo, chi)) return clo;      // repeated entry
    // the flip lies a few values from the middle of the gap: bracket it there, by the predicate itself, so
    // that three halvings remain of up to thirty-two
    uint32_t lo = float_to_key(clo), hi = float_to_key(chi);
    const uint32_t centre = float_to_key(0.5f * clo + 0.5f * chi);
    if (centre > lo && centre < hi) {
        const uint32_t below = centre - lo > 4u ? centre - 4u : lo, above = hi - centre > 4u ? centre + 4u : hi;
        if (takes_upper(key_to_float(below), clo, chi)) hi = below; else lo = below;
        if (lo < above && above < hi) {
            if (takes_upper(key_to_float(above), clo, chi)) hi = above; else lo = above;
        }
    }
    for (int it = 0; it < 32; ++it) {
        if (hi - lo <= 1u) break;
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (takes_upper(key_to_float(mid), clo, chi)) hi = mid; else lo = mid;
    }
    return key_to_float(hi);
}

// Sum over the lanes up to and with this one.
__device__ __forceinline__ uint32_t wave_running_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);       // row_shr:1, 2, 4, 8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);       // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);       // row_bcast:31 into rows 2 and 3
    return v;
}

// All 256 threads of the workgroup call this; ends with a barrier.  lut may be nullptr.
// Bound by latency: a chain that every workgroup runs before its first element, so what shortens it shows in every launch.
// A thread finds the threshold behind its entry from the two entries as they come from memory, as if the table ascended --
// one that does not is found out on the way and takes the longer way below -- with one barrier behind it; the clearing
// of the bucket table and the first barrier lie in the shadow of that load.  The bucket table's counts are a running sum over
// marks, nine buckets a thread.  Against five barriers, the entries through LDS between them, and a binary search per bucket,
// us: 4 bits, no bucket table, 256 x 256 5.1 -> 4.2; 8 bits 1024 x 1024 9.9 -> 7.1, bf16 4096 x 4096 19.9 -> 15.9.
template <int NCODE>
__device__ void build_code_tables(const float *__restrict__ code, CodeTables<NCODE> &t, uint2 *lut) {
    static_assert(NCODE <= 256, "a thread per entry");
    const int tid = threadIdx.x, i = min(tid, NCODE - 1);
    const float own = code[i], next = code[min(i + 1, NCODE - 1)];
    auto clear = [&]() {
        if (lut != nullptr)
            for (int b = tid; b < kLutEntries; b += 256) lut[b] = make_uint2(0x7f800000u, 0u);
    };
    // threshold i: into the table, and a mark on its bucket
    auto place = [&](float th) {
        // The fast quotient is only exact for |v| >= 2^-40; below that the chosen index
        // must not depend on v, so no threshold may sit that close to zero.
        if ((__float_as_uint(th) & 0x7fffffffu) < 0x2c800000u) atomicAnd(&t.flags, ~kFlagLut);
        t.thr[i] = th;
        if (lut != nullptr) {
            uint2 *at = lut + lut_bucket(th);
            at->x = __float_as_uint(th);
            atomicAdd(&at->y, 1u);
        }
    };
    if (tid == 0) { t.flags = kFlagAscending | kFlagLut; t.thr[NCODE - 1] = __uint_as_float(0x7f800000u); }
    clear();
    __syncthreads();
    if (tid < NCODE) {
        t.raw[i] = own;
        t.code[i] = own;
        t.perm[i] = (uint8_t)i;
        if (i < NCODE - 1) {
            if (!(own <= next)) atomicAnd(&t.flags, ~kFlagAscending);          // (a NaN, too)
            place(entry_threshold(own, next));
        }
    }
    __syncthreads();
    if ((t.flags & kFlagAscending) == 0) {           // (the same for the whole workgroup)
        // rank sort, ties by position
        int rank = 0;
        if (tid < NCODE)
            for (int j = 0; j < NCODE; ++j) {
                const float d = t.raw[j];
                rank += (d < own) || (d == own && j < i);
            }
        __syncthreads();
        if (tid == 0) t.flags = kFlagLut;
        if (tid < NCODE) {
            t.code[rank] = own;
            t.perm[rank] = (uint8_t)i;
        }
        clear();
        __syncthreads();
        if (tid < NCODE - 1) place(entry_threshold(t.code[i], t.code[i + 1]));
        __syncthreads();
    }
    if (lut != nullptr) {
        constexpr int kEach = 9;                                               // (odd: with eight, lanes 64 bytes apart meet in the banks)
        static_assert(256 * kEach >= kLutPlaces, "");
        const int p0 = tid * kEach;
        uint32_t marks[kEach], sum = 0;
#pragma unroll
        for (int u = 0; u < kEach; ++u) marks[u] = p0 + u < kLutPlaces ? lut[lut_place(p0 + u)].y : 0u;
#pragma unroll
        for (int u = 0; u < kEach; ++u) {
            if (marks[u] > 1u) atomicAnd(&t.flags, ~kFlagLut);                 // two thresholds in a bucket
            sum += marks[u];
        }
        const uint32_t upto = wave_running_sum(sum);
        if ((tid & 63) == 63) t.wave_sum[tid >> 6] = upto;
        __syncthreads();
        uint32_t base = upto - sum;
#pragma unroll
        for (int w = 0; w < 3; ++w) base += w < tid >> 6 ? t.wave_sum[w] : 0u;
#pragma unroll
        for (int u = 0; u < kEach; ++u) {
            if (p0 + u < kLutPlaces) lut[lut_place(p0 + u)].y = base;
            base += marks[u];
        }
        __syncthreads();
    }
}

// ---- from one value to its table index -------------------------------------------------------
__device__ __forceinline__ uint32_t abs_bits(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// Index by the exact route: IEEE division, then the threshold count.  amax_bits == 0 -> 0.
template <int NCODE>
__device__ __forceinline__ uint32_t exact_index(float x, uint32_t amax_bits, const CodeTables<NCODE> &t) {
    if (amax_bits == 0u) return 0u;
    const float q = x / __uint_as_float(amax_bits);
    return t.perm[count_thresholds<NCODE>(q, t.thr)];
}

template <int NCODE>
__device__ __forceinline__ uint32_t fast_index(float x, float a, float r, const CodeTables<NCODE> &t) {
    return (uint32_t)count_thresholds<NCODE>(quotient(x, a, r), t.thr);
}

// Four of them through the bucket table (quotients of magnitude 1 at most).
__device__ __forceinline__ void fast_four(const float x[4], float a, float r, const uint2 *lut, uint32_t idx[4]) {
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = quotient(x[e], a, r);
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
        const uint32_t p = lut_pair(q[e], q[e + 1]);
        const uint2 lo = lut[(p >> 4) & 0xfffu], hi = lut[p >> 20];
        idx[e] = lo.y + (uint32_t)!(q[e] < __uint_as_float(lo.x));
        idx[e + 1] = hi.y + (uint32_t)!(q[e + 1] < __uint_as_float(hi.x));
    }
}

// Four consecutive elements per lane, G lanes per segment: the segment maximum (as bits; a NaN
// becomes the canonical one) and the four table indices, by the arithmetic of the flat quantizer.
template <int NCODE, int G>
__device__ __forceinline__ uint32_t encode_four(const float x[4], const CodeTables<NCODE> &tab, bool fast_ok, bool ascending,
                                                uint32_t idx[4]) {
    uint32_t m = max(max(abs_bits(x[0]), abs_bits(x[1])), max(abs_bits(x[2]), abs_bits(x[3])));
    m = group_max_u32<G>(m);
    // 2^-60 <= maximum <= 2^60, else (zero, huge, tiny, inf, NaN) the exact route
    if (!fast_ok || (m - kFastDivLo) > (kFastDivHi - kFastDivLo)) {
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
    return m;
}

#endif  // __HIPCC__
}  // namespace qt
