// Device-side helpers shared by the gfx950 kernels: element types, bf16
// conversion and the fixed-sequence exp/log the router uses.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace rbmoe {

constexpr int kWave = 64;

// Raw bf16 storage.  Values are converted explicitly so that the rounding rule
// (nearest even on the bit pattern) is visible and identical everywhere.
struct bf16_t {
    uint16_t bits;
};

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return __uint_as_float((uint32_t)v.bits << 16); }
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
    uint32_t b = __float_as_uint(f);
    if ((b & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((b >> 16) | 0x0040u);
    b += 0x7fffu + ((b >> 16) & 1u);
    return (uint16_t)(b >> 16);
}

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) {
    return v;
}
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) {
    return bf16_t{f32_to_bf16_bits(v)};
}

// ---------------------------------------------------------------------------
// exp and log as fixed sequences of binary32 operations (Cephes expf/logf).
// Every step is either one fused multiply-add (__fmaf_rn) or one correctly
// rounded multiply/add (__fmul_rn/__fadd_rn), so the compiler cannot reorder
// or contract them and the result is the same on any IEEE-754 machine that
// runs the same sequence.  Softmax probabilities and the log-sum-exp depend on
// these bit for bit, and routing depends on the probabilities.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float rb_expf(float x) {
    if (x != x) return x;
    if (x > 88.72283935546875f) return __uint_as_float(0x7f800000u);
    if (x < -103.97208404541015625f) return 0.0f;
    const float t = __fmul_rn(x, 1.44269502162933349609375f);
    const float kf = rintf(t);
    float r = __fmaf_rn(kf, -0.693145751953125f, x);
    r = __fmaf_rn(kf, -1.428606765330187045037746429443359375e-6f, r);
    float p = 1.9875691500e-4f;
    p = __fmaf_rn(p, r, 1.3981999507e-3f);
    p = __fmaf_rn(p, r, 8.3334519073e-3f);
    p = __fmaf_rn(p, r, 4.1665795894e-2f);
    p = __fmaf_rn(p, r, 1.6666665459e-1f);
    p = __fmaf_rn(p, r, 5.0000001201e-1f);
    const float r2 = __fmul_rn(r, r);
    p = __fmaf_rn(p, r2, r);
    p = __fadd_rn(p, 1.0f);
    const int k = (int)kf;
    const int k1 = k / 2;
    const int k2 = k - k1;
    const float s1 = __uint_as_float((uint32_t)(k1 + 127) << 23);
    const float s2 = __uint_as_float((uint32_t)(k2 + 127) << 23);
    return __fmul_rn(__fmul_rn(p, s1), s2);
}

__device__ __forceinline__ float rb_logf(float x) {
    if (x != x) return x;
    if (x < 0.0f) return __uint_as_float(0x7fc00000u);
    if (x == 0.0f) return __uint_as_float(0xff800000u);
    if (__float_as_uint(x) == 0x7f800000u) return x;
    int e = 0;
    uint32_t b = __float_as_uint(x);
    if (b < 0x00800000u) {
        x = __fmul_rn(x, 8388608.0f);
        b = __float_as_uint(x);
        e = -23;
    }
    e += (int)(b >> 23) - 126;
    float m = __uint_as_float((b & 0x007fffffu) | 0x3f000000u);
    if (m < 0.707106769084930419921875f) {
        e -= 1;
        m = __fadd_rn(__fadd_rn(m, m), -1.0f);
    } else {
        m = __fadd_rn(m, -1.0f);
    }
    const float z = __fmul_rn(m, m);
    float y = 7.0376836292e-2f;
    y = __fmaf_rn(y, m, -1.1514610310e-1f);
    y = __fmaf_rn(y, m, 1.1676998740e-1f);
    y = __fmaf_rn(y, m, -1.2420140846e-1f);
    y = __fmaf_rn(y, m, 1.4249322787e-1f);
    y = __fmaf_rn(y, m, -1.6668057665e-1f);
    y = __fmaf_rn(y, m, 2.0000714765e-1f);
    y = __fmaf_rn(y, m, -2.4999993993e-1f);
    y = __fmaf_rn(y, m, 3.3333331174e-1f);
    y = __fmul_rn(__fmul_rn(y, m), z);
    const float fe = (float)e;
    y = __fmaf_rn(-2.12194440e-4f, fe, y);
    y = __fmaf_rn(-0.5f, z, y);
    float r = __fadd_rn(m, y);
    r = __fmaf_rn(0.693359375f, fe, r);
    return r;
}

__device__ __forceinline__ float inverse_rms_of(float sum, int d, float eps) {
    const float mean_square = __fdiv_rn(sum, (float)d);
    // The root must be the correctly rounded one (the reference's f32::sqrt): taken in double and rounded once,
    // which is exact for a square root; the single-precision root instruction alone is not.
    const float root = (float)sqrt((double)__fadd_rn(mean_square, eps));
    return __fdiv_rn(1.0f, root);
}

// LDS reads of 16 bytes each that stay where they are written.
template <typename V>
__device__ __forceinline__ V lds_load_ahead(const unsigned char* p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    static_assert(sizeof(V) % 16 == 0, "16-byte pieces");
    struct Raw {
        u32x4 v[sizeof(V) / 16];
    } raw;
#pragma unroll
    for (size_t i = 0; i < sizeof(V) / 16; ++i)
        raw.v[i] = *(const volatile __attribute__((address_space(3))) u32x4*)(const __attribute__((address_space(3))) void*)(p + 16 * i);
    return __builtin_bit_cast(V, raw);
}

// The sum, in index order, of the d squares that lie at `row_f` in LDS (d a multiple of 8, the row on a 16-byte boundary,
// at least 256 readable bytes behind it): what RmsNorm::forward adds up element by element (src/norm.rs:128-131).  One
// dependent chain of rounded adds, eight cycles each - the length of a row's norm where the width does not divide among a
// wave's lanes (ordered_sum_wave), or where one wave adds up more rows than it could take in turn.  So nothing else is
// on it: the squares are taken beforehand by every thread of the workgroup, and the reads go out 48 elements ahead in
// registers of their own, in an order the compiler does not change (left to itself it moves every read down to its use).
__device__ __forceinline__ float ordered_sum(const float* row_f, int d) {
    const unsigned char* row = reinterpret_cast<const unsigned char*>(row_f);
    struct Part {
        float4 q[4];
    };
    auto read = [&](Part& p, int at) {  // 16 elements
#pragma unroll
        for (int u = 0; u < 4; ++u) p.q[u] = lds_load_ahead<float4>(row + 64 * at + 16 * u);
        __builtin_amdgcn_sched_barrier(0);
    };
    float sum = 0.0f;
    auto add4 = [&](const float4& q) {
        sum = __fadd_rn(sum, q.x);
        sum = __fadd_rn(sum, q.y);
        sum = __fadd_rn(sum, q.z);
        sum = __fadd_rn(sum, q.w);
    };
    auto add = [&](const Part& p) {
#pragma unroll
        for (int u = 0; u < 4; ++u) add4(p.q[u]);
        __builtin_amdgcn_sched_barrier(0);
    };
    Part p0, p1, p2, p3;
    read(p0, 0);
    read(p1, 1);
    read(p2, 2);
    int left = d;
    for (; left >= 64; left -= 64) {
        read(p3, 3);
        add(p0);
        read(p0, 4);
        add(p1);
        read(p1, 5);
        add(p2);
        read(p2, 6);
        add(p3);
        row += 256;
    }
    // up to 56 elements are left
    read(p3, 3);
    auto rest = [&](const Part& p) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (left > 0) add4(p.q[u]);
            left -= 4;
        }
    };
    rest(p0);
    rest(p1);
    rest(p2);
    rest(p3);
    return sum;
}

// silu(x) = x * (1 / (1 + exp(-x))), the reference's operation order
// (src/ffn.rs:223-229).  Tolerance-checked, so the fast exponential is used.
__device__ __forceinline__ float silu_f32(float x) { return x * (1.0f / (1.0f + __expf(-x))); }

// The same with the hardware's 1-ulp reciprocal and base-2 exponential, for results that are
// rounded to bf16 anyway: 2 transcendental and 4 plain operations per value instead of a
// full IEEE division.
__device__ __forceinline__ float silu_bf16_grade(float x) {
    const float e = __builtin_amdgcn_exp2f(x * -1.44269504088896340736f);
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// ---- matrix-core operand helpers ------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
    bf16x2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// two int8 values of `word` (bytes shift/8 and shift/8 + 1) as a pair of bf16
__device__ __forceinline__ uint32_t widen2(uint32_t word, int shift) {
    const float lo = (float)(int)(int8_t)(word >> shift);
    const float hi = (float)(int)(int8_t)(word >> (shift + 8));
    return pack2(lo, hi);  // small integers are exact in bf16; one packed conversion instead of shift + and-or
}

__device__ __forceinline__ bf16x8 widen_i8(uint2 q) {
    const uint4 w = make_uint4(widen2(q.x, 0), widen2(q.x, 16), widen2(q.y, 0), widen2(q.y, 16));
    return __builtin_bit_cast(bf16x8, w);
}

// ---- 16-byte pieces of an activation row: 4 f32 or 8 bf16 --------------------------
template <typename T>
struct Vec16;
template <>
struct Vec16<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ uint4 load_raw(const float* p) { return *reinterpret_cast<const uint4*>(p); }
    static __device__ __forceinline__ void widen(const uint4& a, float (&v)[4]) {
        v[0] = __uint_as_float(a.x); v[1] = __uint_as_float(a.y); v[2] = __uint_as_float(a.z); v[3] = __uint_as_float(a.w);
    }
    static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
        const float4 a = *reinterpret_cast<const float4*>(p);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    }
    static __device__ __forceinline__ void store(float* p, const float (&v)[4]) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
};
template <>
struct Vec16<bf16_t> {
    static constexpr int N = 8;
    static __device__ __forceinline__ uint4 load_raw(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }
    static __device__ __forceinline__ void widen(const uint4& a, float (&v)[8]) {
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
        v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xffff0000u);
        v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xffff0000u);
    }
    static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[8]) {
        const uint4 a = *reinterpret_cast<const uint4*>(p);
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
        v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xffff0000u);
        v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xffff0000u);
    }
    static __device__ __forceinline__ void store(bf16_t* p, const float (&v)[8]) {
        uint4 o;
        o.x = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
        o.y = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
        o.z = f32_to_bf16_bits(v[4]) | ((uint32_t)f32_to_bf16_bits(v[5]) << 16);
        o.w = f32_to_bf16_bits(v[6]) | ((uint32_t)f32_to_bf16_bits(v[7]) << 16);
        *reinterpret_cast<uint4*>(p) = o;
    }
};

// Reductions over the G neighbouring lanes of a group (G a power of two up to 64, the same for the whole wave)
// without LDS: inside a row of 16 lanes through the lane-permuting operand of the instruction itself (every lane of
// the row ends with the result), across rows by handing a row's last lane to the next rows and one or two scalar reads.
template <int CTRL>
__device__ __forceinline__ uint32_t lanes_from(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <typename Op>
__device__ __forceinline__ uint32_t group_reduce(uint32_t v, int G, Op op) {
    if (G >= 2) v = op(v, lanes_from<0xB1>(v));   // quad_perm [1,0,3,2]
    if (G >= 4) v = op(v, lanes_from<0x4E>(v));   // quad_perm [2,3,0,1]
    if (G >= 8) v = op(v, lanes_from<0x141>(v));  // row_half_mirror
    if (G >= 16) v = op(v, lanes_from<0x140>(v)); // row_mirror
    if (G >= 32) {  // (rows 1 and 3, then rows 2 and 3; the others keep what they have)
        v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
        if (G == 64) {
            v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
            v = __builtin_amdgcn_readlane(v, 63);
        } else {
            const uint32_t lo = __builtin_amdgcn_readlane(v, 31), hi = __builtin_amdgcn_readlane(v, 63);
            v = (threadIdx.x & 32) ? hi : lo;
        }
    }
    return v;
}
__device__ __forceinline__ uint32_t group_umax(uint32_t v, int G) {
    return group_reduce(v, G, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
__device__ __forceinline__ uint32_t group_umin(uint32_t v, int G) {
    return group_reduce(v, G, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
// (no NaN among the operands; which zero wins among zeros of both signs does not matter to the callers)
__device__ __forceinline__ float group_fmax(float v, int G) {
    return __uint_as_float(group_reduce(__float_as_uint(v), G, [](uint32_t a, uint32_t b) {
        return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
}

// The sum, in index order, of the 32 L squares of a row, bit for bit ordered_sum's, by one wave: lane l holds the squares
// (l % 32) L .. + L - 1, both halves of the wave the same.
//
// Within a binade the sums are whole multiples n of one unit, and adding q rounds to n + a or n + a + 1 whatever n is, but
// for its parity where q lies halfway.  So what a stretch of additions adds to n depends on the parity of n alone, and
// stretches can be added up side by side from starts that are merely near: the lower half of the wave takes its L squares
// from an even start, the upper half from an odd one, and the differences are composed across the lanes (a scan) until one
// addition takes the sum over as many stretches as lie within a binade.  A stretch is "clean" if a plain prefix sum, which
// is within 2^-13 of the ordered one for rows of up to a thousand, keeps it inside a binade by twice that; the others - some
// five of 32, where the sum passes a power of two, and all of a row with infinities or NaN - are added from their true
// start one after the other.  2118 cycles at 768 columns, where the plain chain of dependent additions (eight cycles each)
// takes 6263; 1828 / 4279 at 512, 2298 / 8188 at 1024, 1678 / 2321 at 256.
template <int L>
__device__ __forceinline__ float ordered_sum_wave(const float (&q)[L]) {
    auto from = [](auto ctrl, float v) { return __uint_as_float(lanes_from<decltype(ctrl)::value>(__float_as_uint(v))); };
    typedef std::integral_constant<int, 0x111> Shr1;  // row_shr within rows of 16 lanes, zeros shifted in
    typedef std::integral_constant<int, 0x112> Shr2;
    typedef std::integral_constant<int, 0x114> Shr4;
    typedef std::integral_constant<int, 0x118> Shr8;
    const int lane = threadIdx.x & 63, stretch = lane & 31, in_row = lane & 15;
    const uint32_t parity = lane >> 5;
    // where the stretch starts and ends, about
    float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < L; ++i) part[i & 3] += q[i];
    const float own = (part[0] + part[1]) + (part[2] + part[3]);
    float upto = own;
    upto += from(Shr1{}, upto);
    upto += from(Shr2{}, upto);
    upto += from(Shr4{}, upto);
    upto += from(Shr8{}, upto);
    const float first_row = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(upto), 15));
    const float start = from(Shr1{}, upto) + ((lane & 16) ? first_row : 0.0f), end = start + own;
    const float lo = start * (1.0f - 0x1p-12f), hi = end * (1.0f + 0x1p-12f);
    const bool clean = stretch != 0 && lo >= 0x1p-100f && hi <= 0x1p126f &&
                       ((__float_as_uint(lo) ^ __float_as_uint(hi)) & 0x7f800000u) == 0;
    uint32_t dirty = ~(uint32_t)__ballot(clean);
    // the stretch from a start of this half's parity (the first: from zero, which is its true one)
    const uint32_t from_bits = stretch == 0 ? 0u : (__float_as_uint(start) & ~1u) | parity;
    float sum = __uint_as_float(from_bits);
#pragma unroll
    for (int i = 0; i < L; ++i) sum = __fadd_rn(sum, q[i]);
    uint32_t add = __float_as_uint(sum) - from_bits;  // units that the clean stretches from the run's first to this one add
    const int behind = stretch - (32 - __clz((int)(dirty & ((1u << stretch) - 1u))));  // clean ones in front, in its run
    auto compose = [&](uint32_t before, int reach) {  // `before` adds the same from the same parity, `reach` stretches earlier
        const auto both = __builtin_amdgcn_permlane32_swap(add, add, false, false);  // this stretch's from even and from odd
        const uint32_t n = before + (((parity ^ before) & 1u) ? both[1] : both[0]);
        add = behind >= reach ? n : add;
    };
    compose(lanes_from<0x111>(add), in_row >= 1 ? 1 : 64);
    compose(lanes_from<0x112>(add), in_row >= 2 ? 2 : 64);
    compose(lanes_from<0x114>(add), in_row >= 4 ? 4 : 64);
    compose(lanes_from<0x118>(add), in_row >= 8 ? 8 : 64);
    compose((uint32_t)__builtin_amdgcn_update_dpp(0, (int)add, 0x142, 0xa, 0xf, true), (lane & 16) ? in_row + 1 : 64);  // row_bcast:15
    // one clean run and the dirty stretch behind it a turn
    uint32_t s = __builtin_amdgcn_readlane(__float_as_uint(sum), 0);
    dirty &= ~1u;
    int at = 1;
    for (;;) {
        const int next = dirty ? (int)__builtin_ctz(dirty) : 32;
        const uint32_t jump = __builtin_amdgcn_readlane(add, next - 1 + 32 * (int)(s & 1));
        s += next > at ? jump : 0u;
        if (next == 32) break;
        float f = __uint_as_float(s);
#pragma unroll
        for (int i = 0; i < L; ++i) f = __fadd_rn(f, q[i]);
        s = __builtin_amdgcn_readlane(__float_as_uint(f), next);
        at = next + 1;
        dirty &= dirty - 1;
    }
    return __uint_as_float(s);
}
// Rows whose norm a wave takes by itself: 8 to 32 elements a lane, whole 16-byte pieces of either type.
__host__ __device__ static bool wave_norms(int d) { return d % 256 == 0 && d <= 1024; }
// f(integral_constant<int, d / 32>) for such a width
template <typename F>
__device__ __forceinline__ void with_lane_elements(int d, F&& f) {
    if (d <= 256) f(std::integral_constant<int, 8>{});
    else if (d <= 512) f(std::integral_constant<int, 16>{});
    else if (d <= 768) f(std::integral_constant<int, 24>{});
    else f(std::integral_constant<int, 32>{});
}
// This lane's L elements of a row, as they lie in memory and widened.
template <typename XT, int L>
struct LaneRow {
    static constexpr int N = Vec16<XT>::N, P = L / N;
    uint4 raw[P];
    __device__ __forceinline__ void load(const XT* row) {
#pragma unroll
        for (int p = 0; p < P; ++p) raw[p] = Vec16<XT>::load_raw(row + (threadIdx.x & 31) * L + p * N);
    }
    __device__ __forceinline__ void widen(float (&v)[L]) const {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            float w[N];
            Vec16<XT>::widen(raw[p], w);
#pragma unroll
            for (int i = 0; i < N; ++i) v[p * N + i] = w[i];
        }
    }
    // RmsNorm's factor of the row (src/norm.rs:128-131)
    __device__ __forceinline__ float inverse_rms(float eps) const {
        float q[L];
        widen(q);
#pragma unroll
        for (int i = 0; i < L; ++i) q[i] = __fmul_rn(q[i], q[i]);
        return inverse_rms_of(ordered_sum_wave<L>(q), 32 * L, eps);
    }
};

}  // namespace rbmoe
