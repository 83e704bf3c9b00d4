// float32 values as three bfloat16 parts, for products on the bfloat16 MFMAs (gemm_mfma.h with SPLIT, conv_stem.h, conv_stem_wgrad.h).
//
// x = h + m + l, each the rest so far rounded to nearest: 3 x 8 bits, all 24 of x.  Six of the nine products of two such values are summed,
// l h + h l + m m + m h + h m into one accumulator and h h into another; what is left out, m l + l m + l l, is below 2^-26 of the product.
// A bfloat16 MFMA rounds once per 16 products where the float32 one rounds per product, so the result is closer to 64 bits (relative error,
// normal operands, K = 64 / 1024 / 4096: 1.4e-7 / 5.7e-7 / 1.15e-6 with float32 MFMAs, 5e-8 / 1.9e-7 / 4.0e-7 so; also for positive operands and for
// ones over 9 decades).
//
// The bfloat16 MFMAs take values below the normal range, 2^-126, for zero, and a part can be 2^-23 of its value.  Every value is therefore
// split as 2^24 x, and a sum comes out as 2^48 of itself: then the last bit of the smallest float32, 2^-149, is a normal bfloat16, and a
// product that is lost is below 2^-174, a quarter of 2^-149 even for 2^23 of them.  Powers of two change no bit of a result.  (Without them,
// tiles that held a value below 2^-100, such as the tail of a softmax, had to be multiplied again by float32 MFMAs, and every value was
// compared: us, ordinary operands / with such values among them, then / ordinary / with such values, so: a b^T 4096 x 4096 x 1024 196 / 266 / 192 / 188;
// 64 x 256 x 14 x 14 3x3 -> 256 123 / 303 / 116 / 116, its weight gradient 105 / 148 / 102 / 102; 32 x 3 x 224 x 224 7x7 stride 2 -> 64 60 / 326 / 59 / 60, its weight
// gradient 67 / 333 / 61 / 60.)
// Values from 2^104 on, sums from 2^80 on, infinities and NaN leave sums that are not finite: the kernels throw those away and use float32 MFMAs.

typedef float mjt_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 mjt_b16x2 __attribute__((ext_vector_type(2)));
#define MJT_SPLIT_UP 0x1p24f
#define MJT_SPLIT_DOWN 0x1p-48f          // of a sum of products of two such values

__device__ __forceinline__ unsigned mjt_bf16_pair(float x, float y) {      // both rounded to nearest even
    return __builtin_bit_cast(unsigned, __builtin_convertvector((mjt_f32x2){x, y}, mjt_b16x2));
}
__device__ __forceinline__ float mjt_low(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float mjt_high(unsigned p) { return __uint_as_float(p & 0xffff0000u); }
// two values (their bits) as pairs of parts
__device__ __forceinline__ void mjt_split(unsigned a, unsigned b, unsigned& h, unsigned& m, unsigned& l) {
    const float x = __uint_as_float(a) * MJT_SPLIT_UP, y = __uint_as_float(b) * MJT_SPLIT_UP;
    h = mjt_bf16_pair(x, y);
    const float x1 = x - mjt_low(h), y1 = y - mjt_high(h);
    m = mjt_bf16_pair(x1, y1);
    l = mjt_bf16_pair(x1 - mjt_low(m), y1 - mjt_high(m));
}
