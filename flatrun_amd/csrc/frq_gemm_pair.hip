// Batched matvec with the fp32 contract, x as pairs of fp16 values:
//   Y[M, N] (fp32) = X[M, K] (fp32) . W[N, K]^T, W = raw Q4_K, Q5_K, Q6_K or
//   Q1_0 blocks.
//
// The reference's batched entry points (matmul_<q>_batched, _C.cpp:154-283)
// run one fp32 matvec per row of X. Here the products run on
// v_mfma_f32_32x32x16_f16, two per product:
//   * x enters as hi + lo 2^-12, hi = f16(x 2^e), lo = f16((x 2^e - hi) 2^12),
//     with 2^e a power of two per row that puts the row's largest |x| in
//     [2^14, 2^15). The pair carries every element down to 2^-28 of the row's
//     largest to within 2^-23 of itself, smaller ones to within 2^-51 of the
//     largest: its own 2^-19 down to 2^-32.
//   * W enters as integers that f16 holds exactly (times 2^-14 for the products
//     with lo, 2^-2 for those with hi: one v_pk_mul_f16 per two codes apart):
//     Q4_K / Q5_K sc q - R with R the integer nearest dmin m / d, Q6_K q - 32,
//     Q1_0 +-1 (2^-12 and 1). A nibble masked in place is the f16 subnormal
//     q 2^-24 (or 16 q 2^-24), so one v_pk_fma_f16 turns two of them into
//     codes, scale and centre included.
//   * the matrix cores sum 64 elements (Q6_K 16, one sub-block) in fp32, then
//     acc += scale * sum in fp32 (the scale of a Q4_K / Q5_K block alone, since
//     sc is in the code). With up to 64 rows a wave, Q5_K, Q1_0 and 32 rows of
//     Q4_K keep acc in fp64, and the others add it to the result's accumulator
//     every 256 elements, so that the sums round less often at full size.
//     Q4_K / Q5_K add -(dmin m - d R) sum(x) per 32-element sub-block
//     on the matrix cores as well: three bf16 pieces of each factor, the six
//     products down to 2^-24 of their product.
//   With R the nearest integer, |d (sc q - R)| + |dmin m - d R| <= 3 |w|, so a
//   large x on a weight that is exactly zero leaves the others their bits.
//
// split_kernel writes the pairs once per call in the order the matrix cores
// take them, with the scale per row. A row whose largest |x| is outside
// [2^-100, 2^101) and one with an inf or NaN are computed weight by weight in
// fp64 instead (finish_kernel), as gemm_f32's are. What the pairs miss of
// elements by more than 2^-19 of the element itself (SwiGLU makes some: 1e-20
// beside 1e2) is added up per row; times the largest weight of a row of W that
// bounds what an output lost. It only counts where the weights of all the larger
// x are zero or nearly so, that is in an output that small itself: an output
// below 2^19 of that bound, and one that is not finite (a scale of W may not
// be), is computed weight by weight in fp64 too.
//
// Tiling: BM x BN of Y per workgroup; a wave owns 32 MT x 32 NT. W goes from
// memory to registers to the matrix cores (lane = one row of W; both halves
// of the wave read consecutive 16-byte parts), decoded once per workgroup
// where WM = 1; x goes through LDS, 32 KB per barrier, four buffers, as every
// wave reads all of it. K is split over S workgroups where the tiles
// do not fill the GPU; finish_kernel adds the partial planes in split order.
// Measured (whole calls, us, W cold; gemm_f32 / here): 333 rows, Q4_K 18944 x 3584
// 224 / 132 (800 TFLOP/s of matrix work on rows padded to 384 in the kernel, about
// 1300 in a large library product), Q6_K 3584 x 18944 322 / 168 (its scale per 16
// elements: eight times the vector work); 97 rows of Q5_K 14336 x 4096 1390 (a GEMV
// per row) / 58; 16 rows of Q4_K 4096 x 14336 36 / 32 (few_kernel 25). 128-row
// tiles are bound by the matrix cores' issue and power, few rows by the chain of
// decode and products per wave (3.7 us per 256 of k) and the three launches. The
// range of lo costs a vector instruction per two codes, or per sum with 128 rows:
// 127 -> 132 us, 97 rows of Q5_K (with fp64 sums) 55 -> 58.
// MFMA operand layouts (32x32x16, 8 values per lane): A lane l holds row l%32,
// k = 8*(l/32) .. +7; B lane l column l%32, same k; D register r of lane l is
// row 8*(r/4) + 4*(l/32) + r%4, column l%32. The order of k is free as long as
// A and B agree: it is chosen so that masked fields of a dword land in place.
#include "frq_common.h"
#include "frq_kernels.h"
#include "frq_weight_at.h"

#include <type_traits>

namespace frq {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
// dword-aligned parts of rows, and the 2-byte aligned dwords of Q1_0 blocks
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
typedef u32x3 u32x3_a4 __attribute__((aligned(4)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));

constexpr int kUnit = 256;               // K per unit (4 stages of 64)
constexpr int kStageBytes = 8192;        // 32 rows x 64 k x 2 pieces x 2 bytes

template <int QT>
constexpr bool kK4 = QT == kTypeQ4K || QT == kTypeQ5K;

constexpr uint32_t kSignCode = 0x0C000C00u;   // +2^-12 twice
// The largest |code| under a scale d: an output's limit is a row's `lim` (2^19 of
// what its pairs miss) times this and the largest |d| of a row of W.
template <int QT>
constexpr float kMaxCode = QT == kTypeQ4K ? 63.0f * 15.0f : QT == kTypeQ5K ? 63.0f * 31.0f : QT == kTypeQ6K ? 4096.0f : 1.0f;
// Whether an output stands as computed, |y| not below its limit and finite.
__device__ __forceinline__ bool stands(float y, float limit) { return !(fabsf(y) < limit) && fabsf(y) < __builtin_inff(); }

__device__ __forceinline__ f16x2 as_f16x2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t as_u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ uint32_t fma2(uint32_t a, f16x2 b, f16x2 c) {
    return as_u32(__builtin_elementwise_fma(as_f16x2(a), b, c));
}
__device__ __forceinline__ f16x2 pair_of(float v) {   // v exact in f16
    return __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(v, v));
}
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// Codes for hi from those for lo (exact).
__device__ __forceinline__ f16x8 for_hi(f16x8 c) { return c * (_Float16)4096.0f; }
__device__ __forceinline__ float add_scaled(float s, float t, float acc) { return __builtin_fmaf(s, t, acc); }
__device__ __forceinline__ double add_scaled(float s, float t, double acc) {
    return __builtin_fma((double)s, (double)t, acc);
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }
template <int S>
__device__ __forceinline__ uint32_t shl(uint32_t v) {   // left by S, right by -S
    if constexpr (S >= 0) return v << S;
    else return v >> -S;
}

// A pointer in scalar registers, from here on opaque to the optimiser: loads
// through it take the lane's part of the address as a 32-bit offset, instead of
// a 64-bit address per lane and load that is advanced every unit.
typedef const __attribute__((address_space(1))) uint8_t* gptr;
__device__ __forceinline__ gptr scalar_base(const uint8_t* p) {
    gptr g = (gptr)p;
    asm("" : "+s"(g));
    return g;
}
template <typename V>
__device__ __forceinline__ auto ld(gptr base, uint32_t off) {
    asm("" : "+v"(off));     // its extension to 64 bits stays beside the load, which folds it
    return *(const __attribute__((address_space(1))) V*)(base + off);
}

// 16 bytes per lane from memory straight to LDS, lane l's to dst + 16 l.
__device__ __forceinline__ void lds_copy(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off, uint8_t* dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, (int)lane_off, (int)off,
                                             0, 0);
}

// The 2-byte aligned fields of Q6_K blocks are read by dword-aligned loads and
// shifted when they are used: wide loads off dword boundaries run at a fraction
// of the rate (4096 x 14336, 16 rows: 54 us against 39). A window starts at
// the dword that holds the field's first byte and has one dword more than the
// field: up to two bytes before the first block of W (on a base that is 2 past a
// dword) or after its last one (on a dword) are read, in dwords that hold bytes of
// W, and used for nothing.
struct Window {
    gptr base;
    uint32_t off;           // of the dword that holds the byte at base + off
    __device__ __forceinline__ Window(gptr p, uint32_t o) {
        const uint64_t a = (uint64_t)p;
        base = (gptr)(a & ~(uint64_t)3);
        off = (o + ((uint32_t)a & 3u)) & ~3u;
    }
};
__device__ __forceinline__ uint32_t misaligned(gptr p, uint32_t o) {   // 16 where p + o is 2 past a dword, else 0
    return (((uint32_t)(uint64_t)p + o) & 2u) * 8u;
}
__device__ __forceinline__ uint32_t shifted(uint32_t lo, uint32_t hi, uint32_t sh) {
    return __builtin_amdgcn_alignbit(hi, lo, sh);
}

// One row's fields of one 256-element unit, as the lane (half h of its row)
// needs them: Head<QT> those used all through the unit, Body<QT> the codes,
// load<T> those of stage T (`unit` = the unit in the first of the
// workgroup's rows, `row` the lane's row from there, `left` = blocks of Q1_0
// from the unit on). frag<T, I>: the eight codes of slice
// I of stage T; scale<T, I>: what the sum of the group that ends with that
// slice is multiplied by. Stage / slice / element orders are those of
// Order<QT> below.
template <int QT>
struct Head;
template <int QT>
struct Body;

// Q4_K: stage t = qs bytes 32t .. 32t+31 (sub-blocks 2t low, 2t+1 high
// nibbles; gguf.py:209-219), half h the 16 bytes 32t + 16h; slice i = dword i.
template <>
struct Head<kTypeQ4K> {
    u32x4 hd;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int) { hd = ld<u32x4>(unit, row); }
};
template <>
struct Body<kTypeQ4K> {
    static constexpr int kLoads = 1, kHeadLoads = 1;   // vector loads of every load<T> / of the head, at least
    u32x4 q[4];
    template <int T>
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int h, int) {
        q[T] = ld<u32x4>(unit + 16 + 32 * T, row + 16 * h);
    }
    template <int T, int I>
    __device__ __forceinline__ u32x4 fields(const Head<kTypeQ4K>&) const {   // (low b0 b2, high b0 b2, low b1 b3, high b1 b3)
        const uint32_t v = q[T][I], v8 = v >> 8;
        return u32x4{v & 0x000F000Fu, v & 0x00F000F0u, v8 & 0x000F000Fu, v8 & 0x00F000F0u};
    }
};

// Q5_K: as Q4_K, bit 2t (2t + 1) of qh byte l is the fifth bit of element l of
// sub-block 2t (2t + 1) (gguf.py:258-275).
template <>
struct Head<kTypeQ5K> {
    u32x4 hd, qh;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int h) {
        hd = ld<u32x4>(unit, row);
        qh = ld<u32x4>(unit + 16, row + 16 * h);
    }
};
template <>
struct Body<kTypeQ5K> {
    static constexpr int kLoads = 1, kHeadLoads = 2;   // vector loads of every load<T> / of the head, at least
    u32x4 q[4];
    template <int T>
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int h, int) {
        q[T] = ld<u32x4>(unit + 48 + 32 * T, row + 16 * h);
    }
    template <int T, int I>
    __device__ __forceinline__ u32x4 fields(const Head<kTypeQ5K>& hh) const {
        const uint32_t v = q[T][I], v8 = v >> 8, b = hh.qh[I];
        return u32x4{(v & 0x000F000Fu) | (shl<4 - 2 * T>(b) & 0x00100010u),
                     (v & 0x00F000F0u) | (shl<7 - 2 * T>(b) & 0x01000100u),
                     (v8 & 0x000F000Fu) | (shl<-4 - 2 * T>(b) & 0x00100010u),
                     (v8 & 0x00F000F0u) | (shl<-1 - 2 * T>(b) & 0x01000100u)};
    }
};

// Q6_K: stage (h', p) = 2h' + p: ql bytes 64h' + 32p + l; slices (nibble c,
// l / 16 = u) = 2c + u are the 16-element groups of ks = p + 2c, half h their
// bytes 8h .. 8h+7 (gguf.py:401-419).
template <>
struct Head<kTypeQ6K> {
    uint32_t d, sh;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int) {
        d = ld<uint16_t>(unit + 208, row);
        sh = misaligned(unit, row);
    }
};
template <>
struct Body<kTypeQ6K> {
    static constexpr int kLoads = 2, kHeadLoads = 1;   // vector loads of every load<T> / of the head, at least
    u32x3 ql[4][2], qh[2][2], sc[2];                    // windows of eight bytes
    template <int T>
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int h, int) {
        const Window f(unit, row + 8 * h), f0(unit, row);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            ql[T][g] = ld<u32x3_a4>(f.base + 32 * T + 16 * g, f.off);
            if constexpr (T % 2 == 0) qh[T / 2][g] = ld<u32x3_a4>(f.base + 128 + 16 * T + 16 * g, f.off);
        }
        if constexpr (T % 2 == 0) sc[T / 2] = ld<u32x3_a4>(f0.base + 192 + 4 * T, f0.off);
    }
    template <int T, int I>
    __device__ __forceinline__ u32x4 frag(const Head<kTypeQ6K>& hh) const {
        constexpr int p = T & 1, c = I >> 1, g = I & 1;
        u32x4 r;
        const f16x2 m = c ? pair_of(64.0f) : pair_of(1024.0f), o = pair_of(-32.0f * 0x1p-14f);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t v = shifted(ql[T][g][e], ql[T][g][e + 1], hh.sh), v8 = v >> 8;
            const uint32_t b = shifted(qh[T >> 1][g][e], qh[T >> 1][g][e + 1], hh.sh);
            const uint32_t b0 = shl<4 - 2 * p>(b), b1 = shl<-4 - 2 * p>(b);
            const uint32_t f0 = c ? (v & 0x00F000F0u) | (b0 & 0x03000300u) : (v & 0x000F000Fu) | (b0 & 0x00300030u);
            const uint32_t f1 = c ? (v8 & 0x00F000F0u) | (b1 & 0x03000300u) : (v8 & 0x000F000Fu) | (b1 & 0x00300030u);
            r[2 * e] = fma2(f0, m, o);
            r[2 * e + 1] = fma2(f1, m, o);
        }
        return r;
    }
    // d * sc[8h' + u + 2 (p + 2c)]
    template <int T, int I>
    __device__ __forceinline__ float scale(const Head<kTypeQ6K>& hh) const {
        constexpr int j = (I & 1) + 2 * ((T & 1) + 2 * (I >> 1)), e = j >> 2;
        const uint32_t v = shifted(sc[T >> 1][e], sc[T >> 1][e + 1], hh.sh);
        return f16_bits_to_f32(hh.d) * 4.0f * (float)(int)(int8_t)(v >> (8 * (j & 3)));
    }
};

// Q1_0: stage t = bytes 8 (t & 1) .. of block t / 2, half h a dword of them;
// slice i register r = the signs of bits 4i + r and 16 + 4i + r (1 = +).
// The codes are negated (bit 1 -> -1), the scale with them.
template <>
struct Head<kTypeQ10> {
    __device__ __forceinline__ void load(gptr, uint32_t, int) {}
};
template <>
struct Body<kTypeQ10> {
    static constexpr int kLoads = 1, kHeadLoads = 0;   // vector loads of every load<T> / of the head, at least
    uint32_t q[4];
    uint32_t d[2];                       // of the two blocks
    template <int T>
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int h, int left) {
        const gptr bp = unit + (T / 2 < left ? T / 2 : left - 1) * kQ10Bytes;
        if constexpr (T % 2 == 0) {
            const uint32_t dv = ld<uint16_t>(bp, row);
            d[T / 2] = T / 2 < left ? dv : 0u;
        }
        q[T] = ld<u32_a2>(bp + 2 + 8 * (T % 2), row + 4 * h);
    }
    template <int T, int I>
    __device__ __forceinline__ u32x4 frag(const Head<kTypeQ10>&) const {
        u32x4 r;
        static_for<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            r[j] = ((q[T] << (15 - 4 * I - j)) & 0x80008000u) | kSignCode;
        });
        return r;
    }
    template <int T, int I>
    __device__ __forceinline__ float scale(const Head<kTypeQ10>&) const {
        return -f16_bits_to_f32(d[T >> 1]);
    }
};

// Where the eight x of (stage st, slice i, half h) are in the row: two runs
// of four from a and b, and the order they take in the fragment.
template <int QT>
struct Order {
    __device__ __forceinline__ static void runs(int st, int i, int h, int& a, int& b) {
        if constexpr (kK4<QT>) {
            a = 64 * st + 16 * h + 4 * i;
            b = a + 32;
        } else if constexpr (QT == kTypeQ6K) {
            a = 128 * (st >> 1) + 32 * ((st & 1) + (i & 2)) + 16 * (i & 1) + 8 * h;
            b = a + 4;
        } else {
            a = 64 * st + 32 * h + 4 * i;
            b = a + 16;
        }
    }
    __device__ __forceinline__ static void order(const f32x4 a, const f32x4 b, float (&v)[8]) {
        if constexpr (kK4<QT>) {
            v[0] = a[0], v[1] = a[2], v[2] = b[0], v[3] = b[2], v[4] = a[1], v[5] = a[3], v[6] = b[1], v[7] = b[3];
        } else if constexpr (QT == kTypeQ10) {
            v[0] = a[0], v[1] = b[0], v[2] = a[1], v[3] = b[1], v[4] = a[2], v[5] = b[2], v[6] = a[3], v[7] = b[3];
        } else {
            v[0] = a[0], v[1] = a[2], v[2] = a[1], v[3] = a[3], v[4] = b[0], v[5] = b[2], v[6] = b[1], v[7] = b[3];
        }
    }
};

// Workgroup-wide sum / max over the TPR threads of a row (LDS, fixed order).
template <int TPR, typename T, typename Op>
__device__ __forceinline__ T row_reduce(T v, T* lds, int tr, Op op) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) v = op(v, __shfl_xor(v, s, 64));
    if constexpr (TPR == 64) return v;
    __syncthreads();
    if ((tr & 63) == 0) lds[tr >> 6] = v;
    __syncthreads();
    T t = lds[0];
#pragma unroll
    for (int i = 1; i < TPR / 64; ++i) t = op(t, lds[i]);
    return t;
}

// Eight scaled values as pairs.
__device__ __forceinline__ void split8(const float (&v)[8], u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const f16x2 hv = {(_Float16)v[2 * p], (_Float16)v[2 * p + 1]};
        const f16x2 lv = {(_Float16)((v[2 * p] - (float)hv[0]) * 4096.0f), (_Float16)((v[2 * p + 1] - (float)hv[1]) * 4096.0f)};
        hi[p] = as_u32(hv);
        lo[p] = as_u32(lv);
    }
}
// What the pairs of four values x, scaled by s, miss of those that they miss by
// more than 2^-19 of the value. Only values below 2^-18 can be (the error is at
// most 2^-37 there and 2^-23 of the value above): those `least` finds. A value that
// the scale takes to zero counts as 2^-60.
__device__ __forceinline__ float lost4(const f32x4 x, float s) {
    float lost = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = x[i] * s, r = v - (float)(_Float16)v;
        const float e = fabsf(r - (float)(_Float16)(r * 4096.0f) * 0x1p-12f);
        lost += v == 0.0f ? (x[i] != 0.0f ? 0x1p-60f : 0.0f) : e > 0x1p-19f * fabsf(v) ? e : 0.0f;
    }
    return lost;
}
// The least nonzero |x| of v and `small`, as bits doubled less one.
__device__ __forceinline__ uint32_t least(uint32_t small, const f32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) small = min(small, (__float_as_uint(v[e]) << 1) - 1u);
    return small;
}
__device__ __forceinline__ bool below(uint32_t small, int e) {   // least's value under a scale 2^e: below 2^-18
    return small < (__float_as_uint(ldexpf(1.0f, -18 - e)) << 1) - 1u;
}

// The largest |x| of v and `big`, as bits (a NaN above inf).
__device__ __forceinline__ uint32_t largest(uint32_t big, const f32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) big = max(big, __float_as_uint(v[e]) & 0x7FFFFFFFu);
    return big;
}

// The power of two that takes values of at most `big` (bits) to [2^14, 2^15):
// false where 2^-100 <= big < 2^101 does not hold (exponent fields 27 .. 227).
__device__ __forceinline__ bool row_scale(uint32_t big, int& e) {
    const int ef = (int)(big >> 23);
    const bool ok = big == 0 || (ef >= 27 && ef <= 227);
    e = big == 0 || !ok ? 0 : 127 + 14 - ef;
    return ok;
}

// The two A fragments' parts of a row's sums s0, s1 over two neighbouring
// sub-blocks: x1 x2 x1 x2 and x3 x1 0 0 (see K4Stage).
__device__ __forceinline__ void sum_pieces(float s0, float s1, u32x4& f0, u32x4& f1) {
    const uint32_t p1 = bf16_pair(s0, s1);
    const float r0 = s0 - bf16_lo(p1), r1 = s1 - bf16_hi(p1);
    const uint32_t p2 = bf16_pair(r0, r1), p3 = bf16_pair(r0 - bf16_lo(p2), r1 - bf16_hi(p2));
    f0 = u32x4{p1, p2, p1, p2};
    f1 = u32x4{p3, p1, 0u, 0u};
}
__device__ __forceinline__ float sum8(float v) {       // over eight neighbouring lanes
    v += dpp_mov<0xB1>(v);
    v += dpp_mov<0x4E>(v);
    v += dpp_mov<0x141>(v);
    return v;
}

// The pairs of every row of x, the sub-block sums' pieces (Q4_K / Q5_K) and
// the factor that undoes the row's scale (0 = row computed weight by weight),
// and lim, 2^19 of what the row's pairs miss.
// RW rows per workgroup, TPR threads each, NC pieces of eight elements per
// thread: x is read once, into registers (NC = 0: rows too long for that are
// read twice). Eight neighbouring rows, whose 16-byte parts share lines of
// the output, go to workgroups of one XCD, where their writes meet in L2.
template <int QT, int RW, int TPR, int NC>
__global__ void __launch_bounds__(RW * TPR) split_kernel(const float* __restrict__ x, int M, int K, int units,
                                                         uint8_t* __restrict__ xf, uint8_t* __restrict__ xsum,
                                                         float* __restrict__ inv, float* __restrict__ lim) {
    __shared__ float red[RW][TPR / 64];
    static_assert(RW <= 8, "rows of a workgroup share an XCD's eight");
    constexpr int WR = 8 / RW;                         // workgroups of eight rows
    const int rr = threadIdx.x / TPR, tr = threadIdx.x % TPR, slot = (int)blockIdx.x >> 3;
    const int m = 64 * (slot / WR) + 8 * ((int)blockIdx.x & 7) + RW * (slot % WR) + rr;
    if (m - rr >= M) return;                           // none of this workgroup's rows
    const bool live = m < M;
    const float* xr = x + (int64_t)(live ? m : M - 1) * K;
    const int chunks = units * 32;                     // (stage, slice, half) triples
    auto load = [&](int c, f32x4& a, f32x4& b) __attribute__((always_inline)) {
        int ra, rb;
        Order<QT>::runs(c >> 3, (c >> 1) & 3, c & 1, ra, rb);
        const bool in = c < chunks;
        a = in && ra < K ? *reinterpret_cast<const f32x4*>(xr + ra) : f32x4{};
        b = in && rb < K ? *reinterpret_cast<const f32x4*>(xr + rb) : f32x4{};
    };
    f32x4 xa[NC ? NC : 1], xb[NC ? NC : 1];
    uint32_t big = 0;
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NC; ++j) load(tr + j * TPR, xa[j], xb[j]);
#pragma unroll
        for (int j = 0; j < NC; ++j) big = largest(largest(big, xa[j]), xb[j]);
    } else {
        for (int c = tr; c < K / 4; c += TPR) big = largest(big, *reinterpret_cast<const f32x4*>(xr + 4 * c));
    }
    big = row_reduce<TPR>(big, reinterpret_cast<uint32_t*>(red[rr]), tr,
                          [](uint32_t a, uint32_t b) { return a > b ? a : b; });
    int e;
    bool ok = row_scale(big, e);                         // max |x| 2^e in [2^14, 2^15)
    const float scale = ok ? ldexpf(1.0f, e) : 0.0f;
    const int64_t mt = m >> 5;
    const int nst = units * 4;
    auto split = [&](int c, f32x4 a, f32x4 b) __attribute__((always_inline)) {
        const int st = c >> 3, i = (c >> 1) & 3, h = c & 1;
        if (!ok) a = b = f32x4{};                        // inf * 0 would be NaN
        a *= scale;
        b *= scale;
        float v[8];
        Order<QT>::order(a, b, v);
        u32x4 hi, lo;
        split8(v, hi, lo);
        const bool out = live && c < chunks;
        if (out) {
            uint8_t* fp = xf + ((mt * nst + st) * 8 + 2 * i) * 1024 + ((m & 31) + 32 * h) * 16;
            *reinterpret_cast<u32x4*>(fp) = hi;
            *reinterpret_cast<u32x4*>(fp + 1024) = lo;
        }
        if constexpr (kK4<QT>) {                         // a, b: four elements of each sub-block, eight lanes
            const float s0 = sum8((a[0] + a[1]) + (a[2] + a[3])), s1 = sum8((b[0] + b[1]) + (b[2] + b[3]));
            if ((c & 7) == 0 && out) {
                u32x4 f0, f1;
                sum_pieces(s0, s1, f0, f1);
                uint8_t* sp = xsum + (mt * nst + st) * 1024 + (m & 31) * 16;
                *reinterpret_cast<u32x4*>(sp) = f0;
                *reinterpret_cast<u32x4*>(sp + 512) = f1;
            }
        }
    };
    if constexpr (NC > 0) {
#pragma unroll
        for (int j = 0; j < NC; ++j) split(tr + j * TPR, xa[j], xb[j]);
    } else {
        for (int c = tr; c < chunks; c += TPR) {
            f32x4 a, b;
            load(c, a, b);
            split(c, a, b);
        }
    }
    float lost = 0.0f;
    if (ok) {                                            // (a row decides alike in all its threads)
        if constexpr (NC > 0) {
            uint32_t small = ~0u;
#pragma unroll
            for (int j = 0; j < NC; ++j) small = least(least(small, xa[j]), xb[j]);
            if (below(small, e)) {
#pragma unroll
                for (int j = 0; j < NC; ++j) lost += lost4(xa[j], scale) + lost4(xb[j], scale);
            }
        } else {
            for (int c = tr; c < K / 4; c += TPR) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(xr + 4 * c);
                if (below(least(~0u, v), e)) lost += lost4(v, scale);
            }
        }
    }
    lost = row_reduce<TPR>(lost, red[rr], tr, [](float a, float b) { return a + b; });
    if (tr == 0 && live) {
        inv[m] = ok ? ldexpf(1.0f, -e) : 0.0f;
        lim[m] = ldexpf(lost, 19 - e);
    }
}

// The largest |d| of a unit (of its second half's block too: Q1_0).
template <int QT>
__device__ __forceinline__ float largest_scale(const Head<QT>& h, const Body<QT>& b) {
    if constexpr (QT == kTypeQ10) return fmaxf(fabsf(f16_bits_to_f32(b.d[0])), fabsf(f16_bits_to_f32(b.d[1])));
    else if constexpr (QT == kTypeQ6K) return fabsf(f16_bits_to_f32(h.d));
    else return fabsf(f16_bits_to_f32(h.hd[0]));
}

template <int QT>
__device__ __forceinline__ u32x4 head_words(const Head<QT>& h) {   // d, dmin and the scales
    if constexpr (kK4<QT>) return h.hd;
    else return u32x4{};
}

// A value of each of two lanes that share a pair of sub-blocks (ROW16: 16 lanes
// apart, else 32), to both: [0] from the lane of the even one, [1] of the odd one.
template <bool ROW16>
__device__ __forceinline__ u32x2 both(uint32_t v) {
    if constexpr (ROW16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return u32x2{r[0], r[1]};
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return u32x2{r[0], r[1]};
    }
}

// What Q4_K / Q5_K add to a stage: its two sub-blocks' code constants and the
// B fragment of (R - dmin m / d) 2^-E, to be multiplied by sum(x) (the pieces
// of split_kernel's fragment: w1 x1, w1 x2, w2 x1, w2 x2 | w1 x3, w3 x1). Each of
// the two lanes of a row that share the sub-blocks works out one of them (sc,
// mn; odd: which). 2^-E is the unit of the codes that meet hi.
template <int E>
struct K4Stage {
    static constexpr float kUnit = 1.0f / (1 << E), kInv = 1 << E;
    f16x2 mul[2], off[2];
    u32x4 uf;
    template <int QT, bool ROW16>
    __device__ __forceinline__ void set(const u32x4 hd, uint32_t sc, uint32_t mn, int odd) {
        const float d = f16_bits_to_f32(hd[0]), dm = f16_bits_to_f32(hd[0] >> 16);
        // d = 0: the codes are 0 and the whole weight, -dmin m, is the second term
        const bool z = d == 0.0f;
        const float rd = z ? 1.0f : __builtin_amdgcn_rcpf(d);
        const float s = z ? 0.0f : (float)sc, tm = dm * (float)mn;          // exact
        // d non-finite: fmaxf drops a NaN, so R lands in range anyway
        const float R = fminf(fmaxf(__builtin_rintf(tm * rd), 0.0f), (QT == kTypeQ4K ? 15.0f : 31.0f) * s);
        const float u = __builtin_fmaf(d, R, -tm) * (rd * kUnit);          // d R - tm in one rounding
        const u32x2 m = both<ROW16>(as_u32(pair_of(s * (odd ? 64.0f : 1024.0f))));
        const u32x2 o = both<ROW16>(as_u32(pair_of(R * -0x1p-14f)));
        mul[0] = as_f16x2(m[0]), mul[1] = as_f16x2(m[1]);
        off[0] = as_f16x2(o[0]), off[1] = as_f16x2(o[1]);
        const uint32_t u1 = bf16_pair(u, 0.0f);
        const float r1 = u - bf16_lo(u1);
        const uint32_t u2 = bf16_pair(r1, 0.0f);
        const u32x2 p = both<ROW16>(u1 | (u2 << 16)), p3 = both<ROW16>(bf16_pair(r1 - bf16_lo(u2), 0.0f));
        const uint32_t w1 = __builtin_amdgcn_perm(p[1], p[0], 0x05040100u), w2 = __builtin_amdgcn_perm(p[1], p[0], 0x07060302u);
        uf = u32x4{w1, odd ? p3[0] | (p3[1] << 16) : w1, odd ? 0u : w2, odd ? 0u : w2};
    }
    __device__ static __forceinline__ float scale(const u32x4 hd) {
        const float d = f16_bits_to_f32(hd[0]);
        return d == 0.0f ? kInv : d * kInv;
    }
};

// Scheduling of one chain: after each of its N matrix instructions, V of the
// vector instructions that run beside it and an LDS read.
template <int N, int V>
__device__ __forceinline__ void interleave() {
    static_for<0, N>([&](auto) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, V, 0);   // VALU
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
    });
}

// WM x WN = 8 waves of 32 MT x 32 NT; LS stages of x per barrier (32 KB), four
// buffers: period p + 3 is written while p is computed, into the buffer that
// p - 1 was read from; the barrier at the end of p - 1 completed the copies of
// p + 1 (kCopies below), so its first fragments are read before the next one.
// A wave's work is a sequence of chains of matrix instructions, one tile and
// scale group each: the small lo products before the hi ones (their sums round
// at their own size), into one of two register sets, while the other one is
// scaled into its tile's accumulator and the codes to come are made. Where the
// registers hold codes for lo and hi, the latter are made beside the products
// (VALU 16 per chain); else (128 rows of Q4_K) the sums of lo are scaled.
// DEPTH > 1: as many register sets of W, each loaded DEPTH units ahead (few
// rows of x: the kernel waits for W); else one, whose stages are loaded again,
// for the next unit, two stages ahead (128 rows: registers).
template <int QT, int WM, int WN, int MT, int NT, int DEPTH>
__global__ void __launch_bounds__(512) gemm_pair_kernel(
    const uint8_t* __restrict__ w, const uint8_t* __restrict__ xf, const uint8_t* __restrict__ xsum,
    const float* __restrict__ inv, const float* __restrict__ lim, float* __restrict__ y, int M, int N, int K, int units,
    int64_t ldy, int S, float* __restrict__ part, uint32_t* __restrict__ aux) {
    static_assert(WM * WN == 8, "eight waves");
    constexpr bool DB = DEPTH > 1;
    constexpr int BT = WM * MT, BM = 32 * BT, BN = 32 * WN * NT;
    constexpr int LS = 4 / BT;                         // stages per barrier
    static_assert(BT == 1 || BT == 2 || BT == 4, "32 KB of x per barrier");
    // slices summed before the scale
    constexpr int GS = QT == kTypeQ6K ? 1 : 4;
    // vector memory instructions of one period's copies; at least, of W's
    // loads per stage and per unit
    constexpr int kCopies = kK4<QT> ? 5 : 4, kStageLoads = NT * Body<QT>::kLoads;
    constexpr int kUnitLoads = NT * Body<QT>::kHeadLoads + 4 * kStageLoads;
    constexpr int kTileBytes = LS * kStageBytes, kSumOff = 32768, kBuf = kSumOff + (kK4<QT> ? 4096 : 0);
    __shared__ __attribute__((aligned(16))) uint8_t xs[4 * kBuf];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM, h = lane >> 5;
    // consecutive tiles on one XCD (workgroups go round the eight XCDs):
    // its L2 then serves a range of W to all tiles of x, and one split's x
    const int G = (int)gridDim.x, xcd = (int)blockIdx.x & 7, gq = G >> 3, gr = G & 7;
    const int id = (xcd < gr ? xcd * (gq + 1) : gr * (gq + 1) + (xcd - gr) * gq) + ((int)blockIdx.x >> 3);
    const int mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    const int mt0 = (id % mtiles) * BT, rest = id / mtiles, n0 = (rest % ntiles) * BN, split = rest / ntiles;
    const int u0 = (int)((int64_t)split * units / S), u1 = (int)((int64_t)(split + 1) * units / S);

    constexpr int kUnitBytes = (int)weight_row_bytes<QT>(kUnit), kUnitBlocks = 2;   // Q1_0 blocks
    const uint8_t* wtile = w + (int64_t)n0 * weight_row_bytes<QT>(K);
    uint32_t wrow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int n = 32 * (NT * wn + nt) + (lane & 31);
        wrow[nt] = (uint32_t)(n0 + n < N ? n : N - 1 - n0) * (uint32_t)weight_row_bytes<QT>(K);
    }
    // LDS order of x: [32-row tile][stage][slice][piece][lane], then
    // [tile][stage][lane] of the sums; a thread moves 16 bytes of each of the
    // period's four 8 KB parts and 8 of the sums
    const int tile_units = units * (4 * kStageBytes);  // from one 32-row tile to the next
    const auto xrs = buffer_rsrc(xf + (int64_t)mt0 * tile_units, (uint32_t)(BT * tile_units));
    const auto srs = buffer_rsrc(xsum + (int64_t)mt0 * units * 4096, (uint32_t)(BT * units * 4096));
    const uint32_t sl = 16 * (tid & 255), soff = sl / (LS * 1024) * (uint32_t)units * 4096u + sl % (LS * 1024);
    const int periods = (u1 - u0) * (4 / LS);          // barriers
    auto copy_x = [&](int p, int buf) __attribute__((always_inline)) {
        const int pp = (p < periods ? p : periods - 1) + u0 * (4 / LS);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            lds_copy(xrs, 16 * tid, (uint32_t)(pp * kTileBytes + (j / LS) * tile_units + (j % LS) * kStageBytes),
                     &xs[buf + kStageBytes * j + 1024 * wave]);
        if constexpr (kK4<QT>) lds_copy(srs, soff, (uint32_t)(pp * (LS * 1024)), &xs[buf + kSumOff + 1024 * (wave & 3)]);
    };
    // fragments of (stage `st` of its period) in the buffer at `buf`
    auto afrag = [&](int buf, int st, int mt, int i, int pc) __attribute__((always_inline)) {
        return *reinterpret_cast<const f16x8*>(
            &xs[buf + (MT * wm + mt) * kTileBytes + st * kStageBytes + (2 * i + pc) * 1024 + lane * 16]);
    };
    auto sfrag = [&](int buf, int st, int mt) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8*>(&xs[buf + kSumOff + (MT * wm + mt) * (LS * 1024) + st * 1024 + lane * 16]);
    };

    constexpr int kE = MT * NT > 2 ? 14 : 2;
    constexpr bool kScaleT = kK4<QT> && MT * NT > 2;
    // With up to 64 rows a wave there is room for two registers per sum: a second
    // level in fp32, every 256 elements, or one sum in fp64 for Q5_K and Q1_0, whose
    // rows one GEMV each would give: 97 rows of Q5_K 14336 x 4096, error against 64
    // bits 1.12e-7 and 0.89e-7 (one GEMV per row 1.05e-7), 58 and 61 us.
    // The 32-row tile of Q4_K, which may run through many units, as well: 16 rows of
    // 8192 x 18944 1.31e-7 and 1.11e-7, 53.1 and 54.5 us.
    constexpr bool kF64 = QT == kTypeQ5K || QT == kTypeQ10 || (QT == kTypeQ4K && MT * NT == 1);
    constexpr bool kTwo = !kF64 && MT * NT <= 2;
    typedef typename std::conditional<kF64, double, float>::type Sum;
    Sum acc[MT][NT][16];
    f32x16 tot[kTwo ? MT : 1][NT], t[2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[mt][nt][r] = 0.0f;
                if (kTwo) tot[kTwo ? mt : 0][nt][r] = 0.0f;
            }
#pragma unroll
    for (int r = 0; r < 16; ++r) t[1][r] = 0.0f;
    float tsc = 0.0f;                                  // the scale of the set not yet in acc

    // one set of heads is enough where the last stage's codes are made before
    // its second chain and the scale is kept apart (K4)
    constexpr int HS = DB ? DEPTH : kK4<QT> ? 1 : 2, UR = DB ? DEPTH : 2;   // sets, units per round of the loop
    Head<QT> hd[HS][NT];
    Body<QT> bd[DEPTH][NT];
    float d4[NT] = {}, dmax = 0.0f;                    // dmax: the largest |d| of the lane's rows of W
    auto load_head = [&](Head<QT> (&hh)[NT], int u) __attribute__((always_inline)) {
        const gptr up = scalar_base(wtile + (int64_t)(u < u1 ? u : u1 - 1) * kUnitBytes);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) hh[nt].load(up, wrow[nt], h);
    };
    auto load_body = [&](auto pc, Body<QT> (&bb)[NT], int u) __attribute__((always_inline)) {
        const int uu = u < u1 ? u : u1 - 1;
        const gptr up = scalar_base(wtile + (int64_t)uu * kUnitBytes);
        const int left = K / kQ10Elems - uu * kUnitBlocks;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) bb[nt].template load<decltype(pc)::value>(up, wrow[nt], h, left);
    };

    const uint32_t sh8 = 8u * (uint32_t)h;
    // a stage's codes of one 32-row tile of W
    struct Codes {
        f16x8 s[GS];
        bf16x8 u;
    };
    // the codes of stage T's slices from group `gc` of GS on
    auto decode = [&](auto tc, auto gc, const Head<QT>& hh, const Body<QT>& bb) __attribute__((always_inline)) {
        constexpr int T = decltype(tc)::value, I0 = decltype(gc)::value * GS;
        Codes c;
        K4Stage<kE> ks;
        if constexpr (kK4<QT>) {
            // (sc, m) of sub-block 2T + h (get_scale_min_k4, gguf.py:135-163)
            const u32x4 hw = head_words(hh);
            const uint32_t s0 = hw[1] >> sh8, s1 = hw[2] >> sh8, s2 = hw[3] >> sh8;
            constexpr int B = 16 * (T & 1);
            if constexpr (T < 2)
                ks.template set<QT, false>(hw, (s0 >> B) & 63u, (s1 >> B) & 63u, h);
            else
                ks.template set<QT, false>(hw, ((s2 >> B) & 15u) | (((s0 >> (B + 6)) & 3u) << 4),
                                           ((s2 >> (B + 4)) & 15u) | (((s1 >> (B + 6)) & 3u) << 4), h);
            c.u = __builtin_bit_cast(bf16x8, ks.uf);
        }
        static_for<0, GS>([&](auto ic) {
            constexpr int I = I0 + decltype(ic)::value;
            u32x4 f;
            if constexpr (kK4<QT>) {
                f = bb.template fields<T, I>(hh);
                f[0] = fma2(f[0], ks.mul[0], ks.off[0]);
                f[1] = fma2(f[1], ks.mul[1], ks.off[1]);
                f[2] = fma2(f[2], ks.mul[0], ks.off[0]);
                f[3] = fma2(f[3], ks.mul[1], ks.off[1]);
            } else {
                f = bb.template frag<T, I>(hh);
            }
            c.s[I - I0] = __builtin_bit_cast(f16x8, f);
        });
        return c;
    };

    // carried from chain to chain: a group's x fragments of one 32-row tile,
    // its codes and scales
    f16x8 a[GS][2];
    float gsc[NT] = {};
    bf16x8 sx;
    Codes b[NT];
    int cur = 0, nxt = kBuf, nx2 = 2 * kBuf, wr3 = 3 * kBuf;   // buffers of periods p .. p + 3

    // one unit: four stages of 64 k; (hn, bn) = the next unit's fields (none in
    // the tail, whose loads of them are dropped)
    auto unit = [&](auto tail, Head<QT> (&hh)[NT], Body<QT> (&bb)[NT], Head<QT> (&hn)[NT], Body<QT> (&bn)[NT], int u)
        __attribute__((always_inline)) {
        static_for<0, 4>([&](auto tc) {
            constexpr int T = decltype(tc)::value, TN = (T + 1) & 3;
            constexpr bool turn = T % LS == LS - 1;    // last stage of its period
            if constexpr (T % LS == 0) {
                const int p = (u - u0) * (4 / LS) + T / LS;
                copy_x(p + 3, wr3);
                asm volatile("" ::: "memory");         // loads of W stay behind the copies
            }
            if constexpr (kK4<QT> && T == 0) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) d4[nt] = K4Stage<kE>::scale(head_words(hh[nt]));
            }
            if constexpr (T == 2) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) dmax = fmaxf(dmax, largest_scale(hh[nt], bb[nt]));
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (GS == 4) {
                static_for<0, MT * NT>([&](auto pc) {
                    constexpr int PH = decltype(pc)::value, mt = PH / NT, nt = PH % NT;
                    constexpr bool lastnt = nt == NT - 1, last = PH == MT * NT - 1;
                    if constexpr (NT == 2 && PH == 0) b[1] = decode(tc, Int<0>{}, hh[1], bb[1]);
                    Codes b0;
                    if constexpr (last) {
                        if constexpr (T < 3) b0 = decode(Int<TN>{}, Int<0>{}, hh[0], bb[0]);
                        else b0 = decode(Int<0>{}, Int<0>{}, hn[0], bn[0]);
                    }
                    // next x fragments: the next tile's, or the next stage's first
                    f16x8 an[4][2];
                    bf16x8 sn = sx;
                    if constexpr (lastnt) {
                        constexpr int mn = last ? 0 : mt + 1, sn_ = last ? (turn ? 0 : T % LS + 1) : T % LS;
                        const int buf = last && turn ? nxt : cur;
                        if constexpr (kK4<QT>) sn = sfrag(buf, sn_, mn);
#pragma unroll
                        for (int q = 1; q >= 0; --q)
#pragma unroll
                            for (int i = 0; i < 4; ++i) an[i][q] = afrag(buf, sn_, mn, i, q);
                    }
                    constexpr int C = (T * MT * NT + PH) & 1;          // this chain's set
                    const f32x16 zero = {};
                    if constexpr (kK4<QT> && !kScaleT) t[C] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sx, b[nt].u, zero, 0, 0, 0);
#pragma unroll
                    for (int q = 1; q >= 0; --q) {                      // lo, then hi
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            t[C] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                a[i][q], q || kScaleT ? b[nt].s[i] : for_hi(b[nt].s[i]),
                                (!kK4<QT> || kScaleT) && q == 1 && i == 0 ? zero : t[C], 0, 0, 0);
                        if constexpr (kScaleT) {
                            if (q) {
#pragma unroll
                                for (int r = 0; r < 16; ++r) t[C][r] *= 0x1p-12f;
                                t[C] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(sx, b[nt].u, t[C], 0, 0, 0);
                            }
                        }
                    }
                    constexpr int PP = (PH + MT * NT - 1) % (MT * NT);  // the chain before this one
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[PP / NT][PP % NT][r] = add_scaled(tsc, t[C ^ 1][r], acc[PP / NT][PP % NT][r]);
                    if constexpr (kK4<QT>) tsc = d4[nt];
                    else tsc = bb[nt].template scale<T, 3>(hh[nt]);
                    if constexpr (last) b[0] = b0;
                    if constexpr (lastnt) {
#pragma unroll
                        for (int q = 0; q < 2; ++q)
#pragma unroll
                            for (int i = 0; i < 4; ++i) a[i][q] = an[i][q];
                        sx = sn;
                    }
                    if constexpr (kScaleT) {
                        constexpr int V = 2 + (NT == 2 && PH == 0 ? 8 : 0) + (last ? 8 : 0);
                        interleave<4, V>();
                        // the scaling, and the chain before into its sums while the last lo product ends
                        // (333 rows of Q4_K 18944 x 3584: 131.4 us, with the scaling alone 132.9)
                        __builtin_amdgcn_sched_group_barrier(0x002, 32, 0);
                        interleave<5, V>();
                    } else {
                        interleave<8 + (kK4<QT> ? 1 : 0), 4 + (NT == 2 && PH == 0 ? 8 : 0) + (last ? 8 : 0)>();
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (!DB && PH == (QT == kTypeQ5K && MT * NT > 2 ? 1 : 0)) {
                        if constexpr (T == (HS == 1 ? 3 : 2)) load_head(hn, u + 1);
                        load_body(Int<(T + 2) & 3>{}, bb, T < 2 ? u : u + 1);
                    }
                });
            } else {
                static_for<0, 4 / GS * MT>([&](auto pc) {
                    constexpr int G_ = decltype(pc)::value / MT, mt = decltype(pc)::value % MT;
                    constexpr bool lastmt = mt == MT - 1, last = lastmt && G_ == 4 / GS - 1;
                    // next x fragments: the next tile's, or the next group's first
                    constexpr int mn = lastmt ? 0 : mt + 1, gn = (G_ + lastmt) % (4 / GS);
                    constexpr int sn_ = last ? (turn ? 0 : T % LS + 1) : T % LS;
                    const int buf = last && turn ? nxt : cur;
                    f16x8 an[GS][2];
#pragma unroll
                    for (int q = 1; q >= 0; --q)
#pragma unroll
                        for (int i = 0; i < GS; ++i) an[i][q] = afrag(buf, sn_, mn, gn * GS + i, q);
                    Codes bx[NT];
                    if constexpr (lastmt) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) {
                            if constexpr (!last) bx[nt] = decode(tc, Int<gn>{}, hh[nt], bb[nt]);
                            else if constexpr (T < 3) bx[nt] = decode(Int<TN>{}, Int<0>{}, hh[nt], bb[nt]);
                            else bx[nt] = decode(Int<0>{}, Int<0>{}, hn[nt], bn[nt]);
                        }
                    }
                    static_for<0, NT>([&](auto nc) {
                        constexpr int nt = decltype(nc)::value;
                        constexpr int C = (((T * (4 / GS) + G_) * MT + mt) * NT + nt) & 1;
                        const f32x16 zero = {};
#pragma unroll
                        for (int q = 1; q >= 0; --q)
#pragma unroll
                            for (int i = 0; i < GS; ++i)
                                t[C] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i][q], q ? b[nt].s[i] : for_hi(b[nt].s[i]),
                                                                              q == 1 && i == 0 ? zero : t[C], 0, 0, 0);
                        constexpr int PP = (mt * NT + nt + MT * NT - 1) % (MT * NT);
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            acc[PP / NT][PP % NT][r] = add_scaled(tsc, t[C ^ 1][r], acc[PP / NT][PP % NT][r]);
                        if constexpr (mt == 0) gsc[nt] = bb[nt].template scale<T, G_ * GS>(hh[nt]);
                        tsc = gsc[nt];
                    });
                    if constexpr (lastmt) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) b[nt] = bx[nt];
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int i = 0; i < GS; ++i) a[i][q] = an[i][q];
                    interleave<2 * GS * NT, (GS == 1 ? 11 : 7) + (lastmt ? (GS == 1 ? 9 : 7) : 0)>();
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (!DB && G_ == 0 && mt == 0) {
                        if constexpr (T == 2) load_head(hn, u + 1);
                        load_body(Int<(T + 2) & 3>{}, bb, T < 2 ? u : u + 1);
                    }
                });
            }
            if constexpr (turn) {
                // Vector memory instructions finish in order: the copies of two
                // periods ahead are done when all but this period's copies and
                // the loads of W issued after the former are. Every wave has
                // then used its fragments of this period.
                constexpr int loads = decltype(tail)::value ? 0 : !DB ? LS * kStageLoads : T < LS ? kUnitLoads : 0;
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kCopies + loads) : "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const int tmp = cur;
                cur = nxt;
                nxt = nx2;
                nx2 = wr3;
                wr3 = tmp;
            }
        });
    };

    auto load_unit = [&](Head<QT> (&hh)[NT], Body<QT> (&bb)[NT], int u) __attribute__((always_inline)) {
        load_head(hh, u);
        static_for<0, 4>([&](auto tc) { load_body(tc, bb, u); });
    };

    copy_x(0, 0);
    copy_x(1, kBuf);
    copy_x(2, 2 * kBuf);
    asm volatile("" ::: "memory");
    if constexpr (DB) {
        static_for<0, DEPTH>([&](auto jc) {
            constexpr int J = decltype(jc)::value;
            load_unit(hd[J], bd[J], u0 + J);
        });
    } else {
        load_head(hd[0], u0);
        load_body(Int<0>{}, bd[0], u0);
        load_body(Int<1>{}, bd[0], u0);
    }
    // the first two periods' copies, as above
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kCopies + (DB ? DEPTH * kUnitLoads : NT * Body<QT>::kHeadLoads + 2 * kStageLoads))
                 : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < GS; ++i) a[i][q] = afrag(0, 0, 0, i, q);
    if constexpr (kK4<QT>) sx = sfrag(0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < (GS == 4 ? 1 : NT); ++nt) b[nt] = decode(Int<0>{}, Int<0>{}, hd[0][nt], bd[0][nt]);
    // a unit's sums into the result's (the one still in t joins the next unit's)
    auto flush = [&]() __attribute__((always_inline)) {
        if constexpr (kTwo) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        tot[mt][nt][r] += acc[mt][nt][r];
                        acc[mt][nt][r] = 0.0f;
                    }
                }
        }
    };
    int u = u0;
    for (; u + UR <= u1; u += UR) {
        static_for<0, UR>([&](auto jc) {
            constexpr int J = decltype(jc)::value, JN = (J + 1) % UR;
            unit(Int<0>{}, hd[J % HS], bd[J % DEPTH], hd[JN % HS], bd[JN % DEPTH], u + J);
            flush();
            if constexpr (DB) {
                load_unit(hd[J], bd[J], u + J + DEPTH);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    }
    static_for<0, UR - 1>([&](auto jc) {               // the last, incomplete round
        constexpr int J = decltype(jc)::value, JN = (J + 1) % UR;
        if (u + J < u1) {
            unit(Int<1>{}, hd[J % HS], bd[J % DEPTH], hd[JN % HS], bd[JN % DEPTH], u + J);
            flush();
        }
    });
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[MT - 1][NT - 1][r] = add_scaled(tsc, t[1][r], acc[MT - 1][NT - 1][r]);
    if constexpr (kTwo) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[mt][nt][r] += tot[mt][nt][r];
    }

    if (S > 1) {
        float* out = part + (int64_t)split * M * N;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int n = n0 + 32 * (NT * wn + nt) + (lane & 31);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = 32 * (mt0 + MT * wm + mt) + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (m < M && n < N) out[(int64_t)m * N + n] = (float)acc[mt][nt][r];
                }
            }
        if (mt0 == 0 && wm == 0 && h == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int n = n0 + 32 * (NT * wn + nt) + lane;
                if (n < N) aux[split * N + n] = __float_as_uint(dmax * kMaxCode<QT>);
            }
        }
        return;
    }
    // S = 1: outputs that do not stand leave as NaN, and the wave's word of aux tells finish_kernel
    uint32_t redo = 0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = 32 * (mt0 + MT * wm + mt) + 8 * i + 4 * h;
            const f32x4 f = *reinterpret_cast<const f32x4*>(inv + m);   // (padded to whole tiles, as lim)
            const f32x4 g = *reinterpret_cast<const f32x4*>(lim + m);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int n = n0 + 32 * (NT * wn + nt) + (lane & 31);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = (float)acc[mt][nt][4 * i + r] * f[r];
                    if (!stands(v, g[r] * (dmax * kMaxCode<QT>))) {
                        v = __builtin_nanf("");
                        redo |= m + r < M && n < N;
                    }
                    if (m + r < M && n < N) y[(int64_t)(m + r) * ldy + n] = v;
                }
            }
        }
    const bool any = __ballot(redo) != 0;
    if (lane == 0) aux[(mt0 / MT + wm) * (ntiles * WN) + n0 / (32 * NT) + wn] = any;
}

// Weights j .. j + 7 (j a multiple of eight) of a row, weight_at's bits.
template <int QT>
__device__ __forceinline__ void weights8(const uint8_t* __restrict__ wrow, int j, float (&v)[8]) {
    if constexpr (kK4<QT>) {
        const uint8_t* bp = wrow + (int64_t)(j >> 8) * (QT == kTypeQ4K ? kQ4KBytes : kQ5KBytes);
        const int sb = (j >> 5) & 7, l = j & 31;
        const uint4 h = *reinterpret_cast<const uint4*>(bp);
        const u32x2 q = *reinterpret_cast<const u32x2*>(bp + (QT == kTypeQ4K ? 16 : 48) + 32 * (sb >> 1) + l);
        u32x2 qh = {};
        if constexpr (QT == kTypeQ5K) qh = *reinterpret_cast<const u32x2*>(bp + 16 + l);
        uint32_t sc, mn;
        k4_scale_min(h.y, h.z, h.w, sb, sc, mn);
        const float s = f16_bits_to_f32(h.x) * (float)sc, t = f16_bits_to_f32(h.x >> 16) * (float)mn;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t c = (q[i >> 2] >> (8 * (i & 3) + 4 * (sb & 1))) & 15u;
            if constexpr (QT == kTypeQ5K) c |= ((qh[i >> 2] >> (8 * (i & 3) + sb)) & 1u) << 4;
            v[i] = s * (float)c - t;
        }
    } else if constexpr (QT == kTypeQ6K) {
        const uint8_t* bp = wrow + (int64_t)(j >> 8) * kQ6KBytes;
        const int e = j & 255, hh = e >> 7, ks = (e >> 5) & 3, l = e & 31;
        const float s = f16_bits_to_f32(ld_u16(bp + 208)) * (float)(int)(int8_t)bp[192 + 8 * hh + (l >> 4) + 2 * ks];
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            const uint32_t ql = ld_u16(bp + 64 * hh + 32 * (ks & 1) + l + i) >> (ks >= 2 ? 4 : 0);
            const uint32_t qh = ld_u16(bp + 128 + 32 * hh + l + i) >> (2 * ks);
#pragma unroll
            for (int b = 0; b < 2; ++b)
                v[i + b] = s * (float)((int)(((ql >> (8 * b)) & 15u) | (((qh >> (8 * b)) & 3u) << 4)) - 32);
        }
    } else {
        const uint8_t* bp = wrow + (int64_t)(j >> 7) * kQ10Bytes;
        const float d = f16_bits_to_f32(ld_u16(bp));
        const uint32_t bits = bp[2 + ((j & 127) >> 3)];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (bits >> i) & 1u ? d : -d;
    }
}

// R rows of x times one row of W by a wave in fp64, the sums in every lane.
template <int QT, int R>
__device__ __forceinline__ void exact_dots(const uint8_t* __restrict__ wr, const float* const (&xr)[R], int K, int lane,
                                           double (&s)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) s[r] = 0.0;
#pragma unroll 1
    for (int j = 8 * lane; j < K; j += 512) {
        float v[8];
        weights8<QT>(wr, j, v);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(xr[r] + j), b = *reinterpret_cast<const f32x4*>(xr[r] + j + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[r] = __builtin_fma((double)v[i], (double)a[i], s[r]);
                s[r] = __builtin_fma((double)v[4 + i], (double)b[i], s[r]);
            }
            // one row of x at a time: 92 registers, so that a batch's workgroups are one
            // round (333 rows of Q4_K 3584 x 3584, split: 42.9 -> 40.7 us)
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) s[r] += __shfl_xor(s[r], o, 64);
}

// S > 1: y = inv * (the planes added in split order, in fp64: free here, and
// one rounding instead of S). Then, S = 1 too, what the pairs do not carry,
// weight by weight in fp64, a wave per row of W over the whole grid:
//   * rows with inv = 0, or, where every split judged its part of x itself
//     (few_kernel; inv null, the planes in units of y, at most 32 rows, lim [S][32]),
//     an infinite lim of any split; up to four at a time, W decoded once;
//   * single outputs that do not stand, marked as NaN: with S > 1 by the planes'
//     sum and the largest scales that aux [S][N] holds, with S = 1 those in the
//     tiles of tm x tn outputs (one wave's) that aux marks.
template <int QT>
__global__ void __launch_bounds__(256) finish_kernel(const float* __restrict__ part, float* __restrict__ y, int S,
                                                     int M, int N, int64_t ldy, const float* __restrict__ inv,
                                                     const float* __restrict__ lim, const uint32_t* __restrict__ aux,
                                                     int tm, int tn, const uint8_t* __restrict__ w,
                                                     const float* __restrict__ x, int K) {
    const int lane = threadIdx.x & 63, wv = (int)blockIdx.x * 4 + (threadIdx.x >> 6), waves = (int)gridDim.x * 4;
    uint32_t bad = 0;                                    // few_kernel's rows, of any split
    float few_lim = 0.0f;                                // of row lane % 32
    if (!inv) {
        for (int i = lane; i < 32 * S; i += 64) few_lim += (i & 31) < M ? lim[i] : 0.0f;
        few_lim += __shfl_xor(few_lim, 32, 64);
        bad = (uint32_t)__ballot(few_lim == __builtin_inff());
    }
    const int64_t row_bytes = weight_row_bytes<QT>(K);
    // the lane's output (m, n), where it is a NaN and `in`
    auto redo_nans = [&](bool in, int m, int n) __attribute__((always_inline)) {
        const float v = in ? y[(int64_t)m * ldy + n] : 0.0f;
        for (uint64_t redo = __ballot(v != v); redo; redo &= redo - 1) {
            const int l = __builtin_ctzll(redo), ml = __builtin_amdgcn_readlane(m, l), nl = __builtin_amdgcn_readlane(n, l);
            const float* xr[1] = {x + (int64_t)ml * K};
            double s[1];
            exact_dots<QT, 1>(w + (int64_t)nl * row_bytes, xr, K, lane, s);
            if (lane == l) y[(int64_t)m * ldy + n] = (float)s[0];
        }
    };
    if (S > 1) {
        // V neighbouring outputs per lane; rows computed below are left alone
        auto add = [&](auto vc) __attribute__((always_inline)) {
            constexpr int V = decltype(vc)::value;
            typedef float fv __attribute__((ext_vector_type(V)));
            typedef double dv __attribute__((ext_vector_type(V)));
            const int64_t plane = (int64_t)M * N, total = plane / V, step = (int64_t)gridDim.x * 256;
            const int nq = N / V;
            bool again = false;
            for (int64_t e0 = (int64_t)wv * 64; e0 < total; e0 += step) {
                const int64_t e = e0 + lane < total ? e0 + lane : total - 1;
                const int m = (int)(e / nq), n = V * (int)(e - (int64_t)m * nq);
                const float* p = part + (int64_t)m * N + n;
                dv v = {};
                for (int q0 = 0; q0 < S; q0 += 8) {      // eight loads in flight
                    fv t[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) t[q] = *reinterpret_cast<const fv*>(p + (q0 + q < S ? q0 + q : 0) * plane);
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        if (q0 + q < S) v += __builtin_convertvector(t[q], dv);
                }
                const float f = inv ? inv[m] : (bad >> m) & 1u ? 0.0f : 1.0f;
                const float g = inv ? lim[m] : __shfl(few_lim, m, 64);
                fv r = __builtin_convertvector(v * (double)f, fv);
                const bool in = e0 + lane < total && f != 0.0f;
                fv c = {};                                // the largest scales, where the limit is not zero
                if (__ballot(g != 0.0f)) {
                    const float* a = reinterpret_cast<const float*>(aux) + n;
#pragma unroll 1
                    for (int q0 = 0; q0 < S; q0 += 8) {
                        fv t[8];
#pragma unroll
                        for (int q = 0; q < 8; ++q) t[q] = *reinterpret_cast<const fv*>(a + (int64_t)(q0 + q < S ? q0 + q : 0) * N);
#pragma unroll
                        for (int q = 0; q < 8; ++q)
#pragma unroll
                            for (int i = 0; i < V; ++i) c[i] = fmaxf(c[i], t[q][i]);
                    }
                }
#pragma unroll
                for (int i = 0; i < V; ++i)
                    if (!stands(r[i], g * c[i])) {
                        r[i] = __builtin_nanf("");
                        again |= in;
                    }
                if (in) *reinterpret_cast<fv*>(y + (int64_t)m * ldy + n) = r;
            }
            if (!__ballot(again)) return;
            for (int64_t e0 = (int64_t)wv * 64; e0 < total; e0 += step) {   // every lane its own outputs again
                const int64_t e = e0 + lane < total ? e0 + lane : total - 1;
                const int m = (int)(e / nq), n = V * (int)(e - (int64_t)m * nq);
                const bool in = e0 + lane < total && (inv ? inv[m] != 0.0f : !((bad >> m) & 1u));
#pragma unroll 1
                for (int i = 0; i < V; ++i) redo_nans(in, m, n + i);
            }
        };
        if (((N | ldy) & 3) == 0 && !(reinterpret_cast<uintptr_t>(y) & 15)) add(Int<4>{});
        else add(Int<1>{});
    } else {
        const int ct = (N + tn - 1) / tn, tiles = (M + tm - 1) / tm * ct, pitch = (N + 255) / 256 * (256 / tn);
        for (int i = wv; i < tiles; i += waves) {
            const int rt = i / ct, n0 = (i - rt * ct) * tn;
            if (!aux[rt * pitch + n0 / tn]) continue;
            for (int e0 = 0; e0 < tm * tn; e0 += 64) {   // a tile's width divides 64
                const int m = rt * tm + (e0 + lane) / tn, n = n0 + (e0 + lane) % tn;
                const bool in = m < M && n < N && (inv ? inv[m] != 0.0f : !((bad >> m) & 1u));
                redo_nans(in, m, n);
            }
        }
    }
    for (int m0 = 0; m0 < M; m0 += 64) {                // every wave scans all rows
        uint64_t hit = inv ? __ballot(m0 + lane < M && inv[m0 + lane < M ? m0 + lane : 0] == 0.0f) : bad;
        while (hit) {
            int m[4];
            const float* xr[4];
            int count = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {                // past the last one: it again
                m[r] = hit ? m0 + __builtin_ctzll(hit) : m[r ? r - 1 : 0];
                count += hit != 0;
                hit &= hit - 1;
                xr[r] = x + (int64_t)m[r] * K;
            }
            for (int n = wv; n < N; n += waves) {
                double s[4];
                exact_dots<QT, 4>(w + (int64_t)n * row_bytes, xr, K, lane, s);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (lane == 0 && r < count) y[(int64_t)m[r] * ldy + n] = (float)s[r];
            }
        }
    }
}

// ------------------------------------------------------------ up to 32 rows
// The same arithmetic for few rows of x, where launches and latency count: one
// launch splits x and multiplies. A workgroup owns 256 rows of W and a range of
// at most kFewUnits / MT units of k; its 16 waves are eight of 32 rows of W by two
// halves (128 elements) of every unit, on v_mfma_f32_16x16x32_f16 (MT tiles of
// 16 rows of x: half the matrix work and LDS of a padded 32-row tile). All loads
// of x and the first of W go out at once; wave r splits row r (and r + 16) of the
// range of x into LDS, scaled by the range's own largest |x|; one barrier; then
// every wave runs through its halves without another. Lane (c, q) of a tile holds row c of W and the
// 16 qs bytes (a dword of Q1_0) of k group q: every 64-byte part of a row in one
// load. The two halves are added through LDS, the splits of k by finish_kernel.
// 16 waves (four per SIMD) hide each other's chains of decode and products,
// which bound the 32-row tile of gemm_pair_kernel at two waves per SIMD. Measured
// (whole call, us, three launches with that tile / here): 16 rows of Q4_K
// 4096 x 14336 31.9 / 24.6 (1.4 TB/s of W; bound by vector work, about five
// instructions per weight), Q1_0 8192 x 1024 15.5 / 12.2, Q5_K 1024 x 1024 15.3 / 13.1.
constexpr int kFewUnits = 8;
constexpr int kFewAside = 256, kFewHead = kFewAside + 2048;   // LDS: factors and limits of the rows, a place for unused writes, x

template <int QT>
struct FewRaw;                                           // one tile's fields of half a unit
template <>
struct FewRaw<kTypeQ4K> {
    u32x4 hd, v;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int kh, int q, int) {
        hd = ld<u32x4>(unit, row);
        v = ld<u32x4>(unit + 16 + 64 * kh, row + 16 * q);
    }
};
template <>
struct FewRaw<kTypeQ5K> {
    u32x4 hd, qh, v;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int kh, int q, int) {
        hd = ld<u32x4>(unit, row);
        qh = ld<u32x4>(unit + 16, row + 16 * (q & 1));
        v = ld<u32x4>(unit + 48 + 64 * kh, row + 16 * q);
    }
};
template <>
struct FewRaw<kTypeQ10> {
    uint32_t d, v;
    __device__ __forceinline__ void load(gptr unit, uint32_t row, int kh, int q, int left) {
        const gptr bp = unit + (kh < left ? kh : left - 1) * kQ10Bytes;
        const uint32_t dv = ld<uint16_t>(bp, row);
        d = kh < left ? dv : 0u;
        v = ld<u32_a2>(bp + 2, row + 4 * q);
    }
};

template <int QT>
__device__ __forceinline__ uint32_t few_scale(const FewRaw<QT>& r) {
    if constexpr (kK4<QT>) return r.hd[0];
    else return r.d;
}

template <int QT, int MT>
__global__ void __launch_bounds__(1024) few_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                   float* __restrict__ y, int M, int N, int K, int units, int64_t ldy,
                                                   int S, float* __restrict__ part, float* __restrict__ lim,
                                                   uint32_t* __restrict__ aux) {
    constexpr int kHalf = 8192 + (kK4<QT> ? 1024 : 0);   // pairs and sums of 16 rows x 128 k
    constexpr int kUnitBytes = (int)weight_row_bytes<QT>(kUnit);
    // units of W in flight (registers; two tiles of Q5_K have at most four in all:
    // 24 rows of 14336 x 4096 29.0 us, with two 29.9 and sums in fp32)
    constexpr int DEPTH = QT == kTypeQ5K ? (MT == 2 ? 1 : 2) : 3;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 7, kh = wave >> 3, c = lane & 15, q = lane >> 4;
    const int G = (int)gridDim.x, xcd = (int)blockIdx.x & 7, gq = G >> 3, gr = G & 7;
    const int id = (xcd < gr ? xcd * (gq + 1) : gr * (gq + 1) + (xcd - gr) * gq) + ((int)blockIdx.x >> 3);
    const int ntiles = (N + 255) / 256, n0 = id % ntiles * 256, split = id / ntiles;
    const int u0 = (int)((int64_t)split * units / S), u1 = (int)((int64_t)(split + 1) * units / S), U = u1 - u0;
    float *inv = reinterpret_cast<float*>(lds), *row_lim = inv + 32;   // of the 16 MT rows
    uint8_t* xl = lds + kFewHead;

    const uint8_t* wtile = w + (int64_t)n0 * weight_row_bytes<QT>(K);
    uint32_t wrow[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int n = 32 * wn + 16 * nt + c;
        wrow[nt] = (uint32_t)(n0 + n < N ? n : N - 1 - n0) * (uint32_t)weight_row_bytes<QT>(K);
    }
    FewRaw<QT> raw[DEPTH][2];
    auto load_w = [&](FewRaw<QT> (&r)[2], int u) __attribute__((always_inline)) {
        const int uu = u < u1 ? u : u1 - 1;
        const gptr up = scalar_base(wtile + (int64_t)uu * kUnitBytes);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) r[nt].load(up, wrow[nt], kh, q, K / kQ10Elems - 2 * uu);
    };
    // x first (memory returns in order): wave r's rows r and (MT = 2) r + 16, lane
    // l's pieces l, l + 64, ...; past the range or the row its last elements,
    // made zeros below
    constexpr int NC = kFewUnits / MT / 2;               // 32 pieces of eight per unit
    const int kleft = K - u0 * kUnit, last = (U * kUnit < kleft ? U * kUnit : kleft) - 4;
    f32x4 xva[MT][NC], xvb[MT][NC];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = 16 * mt + wave < M ? 16 * mt + wave : M - 1;
        const gptr xr = scalar_base(reinterpret_cast<const uint8_t*>(x + (int64_t)m * K + (int64_t)u0 * kUnit));
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int p = lane + 64 * j;
            int ra, rb;
            Order<QT>::runs(p >> 3, (p >> 1) & 3, p & 1, ra, rb);
            xva[mt][j] = ld<f32x4>(xr, 4u * (uint32_t)(ra < last ? ra : last));
            xvb[mt][j] = ld<f32x4>(xr, 4u * (uint32_t)(rb < last ? rb : last));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, DEPTH>([&](auto jc) { load_w(raw[decltype(jc)::value], u0 + decltype(jc)::value); });
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = 16 * mt + wave;
        if (m < M) {                                     // wave-uniform
            f32x4 (&xa)[NC] = xva[mt], (&xb)[NC] = xvb[mt];
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                const int p = lane + 64 * j;
                int ra, rb;
                Order<QT>::runs(p >> 3, (p >> 1) & 3, p & 1, ra, rb);
                if (ra > last) xa[j] = f32x4{};
                if (rb > last) xb[j] = f32x4{};
            }
            uint32_t big = 0;
#pragma unroll
            for (int j = 0; j < NC; ++j) big = largest(largest(big, xa[j]), xb[j]);
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) big = max(big, (uint32_t)__shfl_xor((int)big, o, 64));
            __builtin_amdgcn_sched_barrier(0);
            int e;
            bool ok = row_scale(big, e);
            const float scale = ok ? ldexpf(1.0f, e) : 0.0f;
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                if (2 * j >= U) break;                   // uniform; an odd last unit's pair writes zeros beyond it
                const int p = lane + 64 * j, st = p >> 3, i = (p >> 1) & 3, h = p & 1, qq = (st & 1) * 2 + h;
                f32x4 a = xa[j], b = xb[j];
                if (!ok) a = b = f32x4{};                // inf * 0 would be NaN
                a *= scale;
                b *= scale;
                float v[8];
                Order<QT>::order(a, b, v);
                u32x4 hi, lo;
                split8(v, hi, lo);
                uint8_t* half = xl + (size_t)((st >> 1) * MT + mt) * kHalf;
                uint8_t* fp = half + 2 * i * 1024 + (wave + 16 * qq) * 16;
                *reinterpret_cast<u32x4*>(fp) = hi;
                *reinterpret_cast<u32x4*>(fp + 1024) = lo;
                if constexpr (kK4<QT>) {                 // one lane of eight writes the sums, the others aside
                    u32x4 f0, f1;
                    sum_pieces(sum8((a[0] + a[1]) + (a[2] + a[3])), sum8((b[0] + b[1]) + (b[2] + b[3])), f0, f1);
                    uint8_t* sp = (p & 7) == 0 ? half + 8192 + (wave + 16 * qq) * 16 : lds + kFewAside + lane * 32;
                    *reinterpret_cast<u32x4*>(sp) = f0;
                    *reinterpret_cast<u32x4*>(sp + ((p & 7) == 0 ? 256 : 16)) = f1;
                }
                __builtin_amdgcn_sched_barrier(0);       // one piece at a time: registers
            }
            uint32_t small = ~0u;
#pragma unroll
            for (int j = 0; j < NC; ++j) small = least(least(small, xa[j]), xb[j]);
            float lost = 0.0f;
            if (ok && __ballot(below(small, e))) {       // wave-uniform
#pragma unroll
                for (int j = 0; j < NC; ++j) lost += lost4(xa[j], scale) + lost4(xb[j], scale);
                lost = wave_sum(lost);
            }
            if (lane == 0) {
                inv[m] = ok ? ldexpf(1.0f, -e) : 0.0f;
                row_lim[m] = ok ? ldexpf(lost, 19 - e) : __builtin_inff();
                if (n0 == 0) lim[32 * split + m] = row_lim[m];
            }
        }
    }
    __syncthreads();

    // sums in fp64 for Q5_K and Q1_0, as in gemm_pair_kernel
    typedef typename std::conditional<QT == kTypeQ5K || QT == kTypeQ10, f64x4, f32x4>::type Sum;
    Sum acc[MT][2] = {};
    float dmax = 0.0f;                                   // the largest |d| of the lane's rows of W
    const PairDecode dec(4 * kh + q);                    // this lane's sub-block
    const int qs = 2 * (2 * kh + (q >> 1));              // the fifth bits of its pair
    auto compute = [&](const FewRaw<QT> (&r)[2], int u) __attribute__((always_inline)) {
        const uint8_t* xb = xl + (size_t)(2 * (u - u0) + kh) * MT * kHalf + lane * 16;
        f16x8 b[2][4];
        bf16x8 bu[2];
        float sc[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            dmax = fmaxf(dmax, fabsf(f16_bits_to_f32(few_scale(r[nt]))));
            if constexpr (kK4<QT>) {
                uint32_t s, mn;
                dec(r[nt].hd[1], r[nt].hd[2], r[nt].hd[3], s, mn);
                K4Stage<14> ks;
                ks.template set<QT, true>(r[nt].hd, s, mn, q & 1);
                bu[nt] = __builtin_bit_cast(bf16x8, ks.uf);
                sc[nt] = K4Stage<14>::scale(r[nt].hd);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t v = r[nt].v[i], v8 = v >> 8;
                    u32x4 f = {v & 0x000F000Fu, v & 0x00F000F0u, v8 & 0x000F000Fu, v8 & 0x00F000F0u};
                    if constexpr (QT == kTypeQ5K) {
                        const uint32_t g = r[nt].qh[i] >> qs;
                        f |= u32x4{(g << 4) & 0x00100010u, (g << 7) & 0x01000100u, (g >> 4) & 0x00100010u,
                                   (g >> 1) & 0x01000100u};
                    }
                    f[0] = fma2(f[0], ks.mul[0], ks.off[0]);
                    f[1] = fma2(f[1], ks.mul[1], ks.off[1]);
                    f[2] = fma2(f[2], ks.mul[0], ks.off[0]);
                    f[3] = fma2(f[3], ks.mul[1], ks.off[1]);
                    b[nt][i] = __builtin_bit_cast(f16x8, f);
                }
            } else {
                sc[nt] = f16_bits_to_f32(r[nt].d) * -4096.0f;   // codes negated and 2^-12, as in Body<kTypeQ10>
                static_for<0, 4>([&](auto ic) {
                    constexpr int I = decltype(ic)::value;
                    u32x4 f;
                    static_for<0, 4>([&](auto jc) {
                        constexpr int j = decltype(jc)::value;
                        f[j] = ((r[nt].v << (15 - 4 * I - j)) & 0x80008000u) | kSignCode;
                    });
                    b[nt][I] = __builtin_bit_cast(f16x8, f);
                });
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const uint8_t* xm = xb + mt * kHalf;
            f32x4 t[2] = {};
#pragma unroll
            for (int pc = 1; pc >= 0; --pc) {            // lo, then hi
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f16x8 a = *reinterpret_cast<const f16x8*>(xm + (2 * i + pc) * 1024);
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt)
                        t[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[nt][i], t[nt], 0, 0, 0);
                }
                if (pc) {                                // the same codes for both here: eight sums, 32 pairs of codes
#pragma unroll
                    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                        for (int r4 = 0; r4 < 4; ++r4) t[nt][r4] *= 0x1p-12f;
                    if constexpr (kK4<QT>) {
                        const bf16x8 a = *reinterpret_cast<const bf16x8*>(xm + 8192);
#pragma unroll
                        for (int nt = 0; nt < 2; ++nt) t[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bu[nt], t[nt], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) acc[mt][nt][r4] = add_scaled(sc[nt], t[nt][r4], acc[mt][nt][r4]);
        }
    };
    int u = u0;
    for (; u + DEPTH <= u1; u += DEPTH)
        static_for<0, DEPTH>([&](auto jc) {
            constexpr int J = decltype(jc)::value;
            compute(raw[J], u + J);
            load_w(raw[J], u + J + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
        });
    static_for<0, DEPTH - 1>([&](auto jc) {
        constexpr int J = decltype(jc)::value;
        if (u + J < u1) compute(raw[J], u + J);
    });

    // the second half's sums through LDS (x is done with), then out
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(xl) + wn * MT * 2 * 64 + lane;
    float* dred = reinterpret_cast<float*>(lds + kFewAside) + wn * 16 + c;
    if (kh == 1) {
        if (q == 0) *dred = dmax;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) red[(2 * mt + nt) * 64] = __builtin_convertvector(acc[mt][nt], f32x4);
        }
    }
    __syncthreads();
    if (kh == 1) return;
    float* out = S == 1 ? y : part + (int64_t)split * M * N;
    const int64_t ldo = S == 1 ? ldy : N;
    const float dm = fmaxf(dmax, *dred) * kMaxCode<QT>;
    uint32_t redo = 0;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int n = n0 + 32 * wn + 16 * nt + c;
        if (S > 1 && q == 0 && n < N) aux[split * N + n] = __float_as_uint(dm);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const f32x4 v = __builtin_convertvector(acc[mt][nt] + __builtin_convertvector(red[(2 * mt + nt) * 64], Sum), f32x4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = 16 * mt + 4 * q + r;
                float o = v[r] * inv[m];
                if (S == 1 && !stands(o, row_lim[m] * dm)) {   // as in gemm_pair_kernel
                    o = __builtin_nanf("");
                    redo |= m < M && n < N;
                }
                if (m < M && n < N) out[(int64_t)m * ldo + n] = o;
            }
        }
    }
    if (S == 1) {
        const bool any = __ballot(redo) != 0;
        if (lane == 0) aux[n0 / 32 + wn] = any;
    }
}

template <int QT>
void finish_go(const PairPlan& p, const float* part, const float* inv, const float* lim, const uint32_t* aux, int tm,
               int tn, const uint8_t* w, const float* x, float* y, int64_t ldy, hipStream_t s) {
    // at least 1024 workgroups, for rows computed weight by weight (eight rows of
    // Q5_K 14336 x 4096: 128 us, with 256 workgroups 266)
    const int64_t work = p.splits > 1 ? (p.m * p.n + 1023) / 1024 : 0;
    finish_kernel<QT><<<dim3((unsigned)(work < 1024 ? 1024 : work > 2048 ? 2048 : work)), dim3(256), 0, s>>>(
        part, y, p.splits, (int)p.m, (int)p.n, ldy, inv, lim, aux, tm, tn, w, x, (int)p.k);
}

template <int QT, int WM, int WN, int MT, int NT, int DEPTH>
void pair_go(const PairPlan& p, const uint8_t* w, const float* x, float* y, int64_t ldy, hipStream_t s,
             uint8_t* scratch) {
    const int64_t ntiles = (p.n + 32 * WN * NT - 1) / (32 * WN * NT), mtiles = (p.m + 32 * WM * MT - 1) / (32 * WM * MT);
    const float *inv = reinterpret_cast<const float*>(scratch), *lim = reinterpret_cast<const float*>(scratch + p.lim_off);
    float* part = reinterpret_cast<float*>(scratch + p.part_off);
    uint32_t* aux = reinterpret_cast<uint32_t*>(scratch + p.aux_off);
    gemm_pair_kernel<QT, WM, WN, MT, NT, DEPTH><<<dim3((unsigned)(ntiles * mtiles * p.splits)), dim3(512), 0, s>>>(
        w, scratch + p.x_off, scratch + p.sum_off, inv, lim, y, (int)p.m, (int)p.n, (int)p.k, (int)p.units, ldy, p.splits,
        part, aux);
    finish_go<QT>(p, part, inv, lim, aux, 32 * MT, 32 * NT, w, x, y, ldy, s);
}

// Few rows: 1024 threads each, for latency; more: enough threads that every
// one holds two to five pieces of the row in registers.
template <int QT, int RW, int TPR, int NC>
void split_launch(const PairPlan& p, const float* x, hipStream_t s, uint8_t* xf, uint8_t* xsum, float* inv, float* lim) {
    const unsigned grid = (unsigned)((p.m + 63) / 64 * 64 / RW);
    split_kernel<QT, RW, TPR, NC><<<dim3(grid), dim3(RW * TPR), 0, s>>>(x, (int)p.m, (int)p.k, (int)p.units, xf, xsum, inv,
                                                                                lim);
}
template <int QT>
void split_go(const PairPlan& p, const float* x, hipStream_t s, uint8_t* xf, uint8_t* xsum, float* inv, float* lim) {
    const int64_t chunks = p.units * 32;
    if (p.m <= 64 && chunks > 512) {
        if (chunks <= 1024) return split_launch<QT, 1, 1024, 1>(p, x, s, xf, xsum, inv, lim);
        if (chunks <= 2048) return split_launch<QT, 1, 1024, 2>(p, x, s, xf, xsum, inv, lim);
        if (chunks <= 3072) return split_launch<QT, 1, 1024, 3>(p, x, s, xf, xsum, inv, lim);
    }
    if (chunks <= 256) return split_launch<QT, 4, 128, 2>(p, x, s, xf, xsum, inv, lim);
    if (chunks <= 512) return split_launch<QT, 2, 256, 2>(p, x, s, xf, xsum, inv, lim);
    if (chunks <= 1024) return split_launch<QT, 2, 256, 4>(p, x, s, xf, xsum, inv, lim);
    if (chunks <= 2560) return split_launch<QT, 1, 512, 5>(p, x, s, xf, xsum, inv, lim);
    split_launch<QT, 1, 1024, 0>(p, x, s, xf, xsum, inv, lim);
}

template <int QT>
void pair_run(const PairPlan& p, const uint8_t* w, const float* x, float* y, int64_t ldy, hipStream_t s,
              uint8_t* scratch, bool x_ready) {
    float *inv = reinterpret_cast<float*>(scratch), *lim = reinterpret_cast<float*>(scratch + p.lim_off);
    if constexpr (QT != kTypeQ6K) {
        if (p.few) {
            uint32_t* aux = reinterpret_cast<uint32_t*>(scratch + p.aux_off);
            float* part = reinterpret_cast<float*>(scratch + p.part_off);
            const unsigned grid = (unsigned)((p.n + 255) / 256 * p.splits);
            const int mt = p.m <= 16 ? 1 : 2;
            const int64_t u = (p.units + p.splits - 1) / p.splits;
            const unsigned bytes = (unsigned)((u + 1) / 2 * 4 * mt * (8192 + (kK4<QT> ? 1024 : 0)));
            const unsigned red = (unsigned)(8 * mt * 2 * 64 * 16);
            const unsigned ldsb = kFewHead + (bytes > red ? bytes : red);
            if (mt == 1)
                few_kernel<QT, 1><<<dim3(grid), dim3(1024), ldsb, s>>>(w, x, y, (int)p.m, (int)p.n, (int)p.k,
                                                                       (int)p.units, ldy, p.splits, part, lim, aux);
            else
                few_kernel<QT, 2><<<dim3(grid), dim3(1024), ldsb, s>>>(w, x, y, (int)p.m, (int)p.n, (int)p.k,
                                                                       (int)p.units, ldy, p.splits, part, lim, aux);
            return finish_go<QT>(p, part, nullptr, lim, aux, 16 * mt, 32, w, x, y, ldy, s);
        }
    }
    if (!x_ready) split_go<QT>(p, x, s, scratch + p.x_off, scratch + p.sum_off, inv, lim);
    if (p.bm == 32)
        pair_go<QT, 1, 8, 1, 1, 2>(p, w, x, y, ldy, s, scratch);
    else if (p.bm == 64)
        pair_go<QT, 1, 8, 2, 1, QT == kTypeQ10 ? 2 : 1>(p, w, x, y, ldy, s, scratch);
    else if constexpr (QT == kTypeQ4K)
        pair_go<QT, 2, 4, 2, 2, 1>(p, w, x, y, ldy, s, scratch);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// A call's estimated time (us): its launches + rounds of 256 workgroups (one per
// CU), each a start and a workgroup's units of k, + the planes of a split k,
// written and read (8 bytes of each output and split, in 3.1 MB). With few CUs
// busy a unit takes up to 15 % less. The numbers fit 90000 measured calls: every
// tile of each format at 1 to 64 splits for 9900 random shapes of 3 to 512 rows (k
// 512 to 24576, n 400 to 65536, W cold in the caches). The plans chosen take 0.7 %
// (up to 32 rows) and 0.3 % more than the fastest measured ones on average; one
// unit time for all formats, and few_kernel wherever within 6 us of the tile, took
// 2.5 and 0.6 %. Some (us, both sides measured): 64- / 128-row tile, Q4_K 18944 x
// 3584 at 200 rows 119 / 113, at 333 149 / 140, 4096 x 4096 at 333 54 / 56;
// few_kernel / 32-row tile, Q4_K 4096 x 14336 at 16 rows 25 / 32, 24 rows 29 / 32,
// Q5_K 1024 x 1024 at 12 13 / 15, Q1_0 8192 x 1024 at 8 12 / 15, 1024 x 4096 at 32
// 19 / 17.
struct PairCost {
    double launches, start, unit, plane;
    double us(int64_t workgroups, int64_t units, int64_t splits, double plane_us) const {
        const double busy = workgroups < 256 ? (double)workgroups / 256 : 1.0;
        return launches + (double)((workgroups + 255) / 256) * (start + (double)units * unit * (0.85 + 0.15 * busy)) +
               (splits > 1 ? (double)splits * plane_us * plane : 0.0);
    }
};
// bm 16: few_kernel with up to 16 rows, 17: with more
PairCost pair_cost(int qtype, int bm) {
    const int f = qtype == kTypeQ4K ? 0 : qtype == kTypeQ5K ? 1 : qtype == kTypeQ10 ? 2 : 3;
    static constexpr double unit[5][4] = {
        {2.35, 3.2, 1.4, 0.0}, {3.05, 3.5, 2.2, 0.0}, {3.7, 4.4, 2.75, 5.6}, {4.6, 5.6, 4.3, 5.7}, {8.4, 0.0, 0.0, 0.0}};
    switch (bm) {
        case 16: return {5.5, 5.6, unit[0][f], 1.15};
        case 17: return {8.6, 3.8, unit[1][f], 1.1};
        case 32: return {8.5, 4.0, unit[2][f], 0.8};
        case 64: return {12.0, 0.6, unit[3][f], 0.9};
        default: return {12.0, 2.6, unit[4][f], 0.7};
    }
}

}  // namespace

bool plan_gemm_pair(int qtype, int64_t m, int64_t n, int64_t k, size_t cap, PairPlan* p) {
    const int64_t kq = qtype == kTypeQ10 ? kQ10Elems
                       : (qtype == kTypeQ4K || qtype == kTypeQ5K || qtype == kTypeQ6K) ? kQKElems
                                                                                      : 0;
    if (kq == 0 || m <= 0 || n <= 0 || k <= 0 || k % kq || m > kPairRows || n > 0x3FFFFFFF || k > (1 << 22))
        return false;
    const bool k4 = qtype == kTypeQ4K || qtype == kTypeQ5K;
    p->few = false;
    p->m = m;
    p->n = n;
    p->k = k;
    p->units = (k + kUnit - 1) / kUnit;
    p->bn = 256;
    p->layout = k4 ? kTypeQ4K : qtype;
    const int64_t ntiles = (n + p->bn - 1) / p->bn;
    // The row tile and the split of k with the least estimated time.
    const double plane_us = (double)m * (double)n * 8.0 / 3.1e6;
    // Only Q4_K has a 128-row tile. It adds all of a split's sums in one fp32 level:
    // Q5_K and Q1_0, whose rows otherwise run one GEMV each, keep to the tiles with
    // fp64 sums, which match a GEMV's error. For Q6_K it decoded W half as often but
    // is bound by the scaling of its 16-element sums (us, error against 64 bits, 64- /
    // 128-row tile: 18944 x 3584 at 200 rows 141 / 138; 62765 x 1024 at 383 191 and
    // 0.98e-7 / 177 and 1.34e-7; 65000 x 1536 at 120 93 and 1.12e-7 / 90 and 2.06e-7;
    // 14336 x 4096 at 128 61 / 68).
    const bool wide = qtype == kTypeQ4K;
    const int bms[2] = {m <= 32 ? 32 : 64, m <= 32 ? 32 : m <= 64 || !wide ? 64 : 128};
    double best = 0.0;
    bool found = false;
    for (int c = 0; c < 2; ++c) {
        const int bm = bms[c];
        const int64_t mtiles = (m + bm - 1) / bm, mpad = mtiles * bm;
        const size_t lim_off = (size_t)mpad * 4, sum_off = align256(2 * lim_off);
        const size_t x_off = sum_off + (k4 ? (size_t)(mpad / 32 * p->units) * 4096 : 0);
        const size_t part_off = x_off + (size_t)mpad * (size_t)p->units * kUnit * 4;
        if (part_off > cap) continue;
        const PairCost cost = pair_cost(qtype, bm);
        for (int64_t s = 1; s <= 64 && s <= p->units; ++s) {
            // the planes and the largest scales [s][n], or a word per wave of every tile
            const size_t planes = s > 1 ? align256((size_t)s * (size_t)m * (size_t)n * 4) : 0;
            const size_t aux = s > 1 ? (size_t)s * (size_t)n * 4 : (size_t)(mtiles * ntiles) * 8 * 4;
            if (part_off + planes + aux > cap) break;
            const double us = cost.us(mtiles * ntiles * s, (p->units + s - 1) / s, s, plane_us);
            if (!found || us < best) {
                found = true;
                best = us;
                p->bm = bm;
                p->splits = (int)s;
                p->lim_off = lim_off;
                p->sum_off = sum_off;
                p->x_off = x_off;
                p->part_off = part_off;
                p->aux_off = part_off + planes;
                p->bytes = p->aux_off + aux;
            }
        }
    }
    if (m <= 32 && qtype != kTypeQ6K) {
        // few_kernel: one round of 256 workgroups where its LDS lets it, every
        // split at least two units
        const int64_t most = kFewUnits / (m <= 16 ? 1 : 2), need = (p->units + most - 1) / most;
        int64_t fs = 256 / ntiles < 64 ? 256 / ntiles : 64;
        if (fs > (p->units + 1) / 2) fs = (p->units + 1) / 2;
        if (fs < need) fs = need;
        if (fs < 1) fs = 1;
        const int64_t share = (p->units + fs - 1) / fs;
        fs = (p->units + share - 1) / share;             // as few splits as give that share
        const double few_us = pair_cost(qtype, m <= 16 ? 16 : 17).us(ntiles * fs, share, fs, plane_us);
        const size_t part_off = align256((size_t)fs * 32 * 4);
        const size_t aux_off = part_off + (fs > 1 ? align256((size_t)fs * (size_t)m * (size_t)n * 4) : 0);
        const size_t bytes = aux_off + (fs > 1 ? (size_t)fs * (size_t)n * 4 : (size_t)ntiles * 8 * 4);
        if (bytes <= cap && fs * ntiles <= 0x7FFFFFFF && (!found || few_us < best)) {
            p->few = true;
            p->splits = (int)fs;
            p->bm = 32;
            p->layout = 0;                               // nothing that another launch could use
            p->lim_off = p->sum_off = p->x_off = 0;
            p->part_off = part_off;
            p->aux_off = aux_off;
            p->bytes = bytes;
            return true;
        }
    }
    return found;
}

hipError_t launch_gemm_pair(int qtype, const uint8_t* w, const float* x, float* y, int64_t ldy, const PairPlan& p,
                            hipStream_t stream, uint8_t* scratch, bool x_ready) {
    if (ldy < p.n || (reinterpret_cast<uintptr_t>(x) & 15) || !scratch) return hipErrorInvalidValue;
    const uintptr_t wa = reinterpret_cast<uintptr_t>(w);
    if (qtype == kTypeQ4K || qtype == kTypeQ5K ? (wa & 15) : (wa & 1)) return hipErrorInvalidValue;
    switch (qtype) {
        case kTypeQ4K: pair_run<kTypeQ4K>(p, w, x, y, ldy, stream, scratch, x_ready); break;
        case kTypeQ5K: pair_run<kTypeQ5K>(p, w, x, y, ldy, stream, scratch, x_ready); break;
        case kTypeQ6K: pair_run<kTypeQ6K>(p, w, x, y, ldy, stream, scratch, x_ready); break;
        case kTypeQ10: pair_run<kTypeQ10>(p, w, x, y, ldy, stream, scratch, x_ready); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace frq
