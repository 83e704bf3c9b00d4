// The float32 results of a sum's slices added up: y[i] = sum over s of part[s][i], narrowed once to y's type, or handed to the element-wise
// group behind the product (epilogue.h).
//
// Supplied by the host: SLICES (at most 16), VS (adjacent results a lane takes: 4, 2 or 1), OUT (0 bfloat16 by truncation, 1 float16 rounded
// to nearest even, 2 float32).  a[0] part, a[1] y, a[2] vectors of VS.
//
// Bound by the trip to memory: the parts lie in the caches that the product has just written them to.  All of a lane's loads are under way
// together; the slices are added in their order.  us, the general reduce (and the group by itself) / this: 9 slices of 4 x 64 x 14 x 14 3.3 /
// 2.4, 12 of 3 x 256 x 14 x 14 with relu 4.0 + 2.2 / 4.0, 11 of 43 x 1136 with a bias 3.8 + 2.1 / 2.6.
#ifndef EPI
#define EPI 0
#define EPI_WORDS 0
#endif
struct Params { void* a[3 + EPI_WORDS]; };

extern "C" __global__ __launch_bounds__(256) void ENTRY(Params p) {
    struct alignas(VS * 4) vec { float v[VS]; };
    const long long n = (long long)p.a[2], i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const vec* __restrict__ part = (const vec*)p.a[0] + i;
    vec in[SLICES];
#pragma unroll
    for (int s = 0; s < SLICES; s++) in[s] = part[s * n];
#if EPI
    mjt_epi_in<VS> read;
    mjt_epi_load(p, read, (MJT_EPI_INDEX)(i * VS));
#endif
    vec sum = in[0];
#pragma unroll
    for (int s = 1; s < SLICES; s++)
#pragma unroll
        for (int k = 0; k < VS; k++) sum.v[k] += in[s].v[k];
#if EPI
    mjt_epi_finish(p, read, (MJT_EPI_INDEX)(i * VS), sum.v);
#elif OUT == 2
    *((vec*)p.a[1] + i) = sum;
#else
    struct alignas(VS * 2) { unsigned short v[VS]; } o;
#pragma unroll
    for (int k = 0; k < VS; k++)
#if OUT == 0
        o.v[k] = (unsigned short)(__float_as_uint(sum.v[k]) >> 16);                    // truncation (type/fp16_compute.h:238-241)
#else
        o.v[k] = __builtin_bit_cast(unsigned short, (_Float16)sum.v[k]);                // nearest even (type/fp16_compute.h:147-198)
#endif
    *((decltype(o)*)p.a[1] + i) = o;
#endif
}
