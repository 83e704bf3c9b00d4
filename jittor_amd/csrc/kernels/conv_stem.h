// Convolution of images with few channels, the first layer of a network, from windows that lie in LDS:
//   y[n][k][oh][ow] = sum_{c,r,s} w[k][c][r][s] * x[n][c][oh*SH-PH+r*DH][ow*2-PW+s]
// (python/jittor/nn.py:1251-1262, recognised by opt/tuner/conv_tuner.cc:218-411) with horizontal stride 2 and rows of up to 8 taps.  bfloat16 and
// float16 operands as they are, float32 ones as three bfloat16 parts each (split.h has the reasoning and the error), float32 sums.
//
// What it replaces, the product that gathers x (gemm_mfma.h, CONV 1), loads every element of x once for each tap that sees it, works out
// where it lies and multiplies float32 with float32 MFMAs.  Here a row of taps is 8 consecutive values of a row of x, taps beyond S zero, so
// a step of v_mfma_f32_32x32x16 is two rows (c, r), and a lane's operand, 8 values from column 2*ow on, is 16 bytes of LDS at a
// 4-byte aligned place: neighbouring lanes read neighbouring dwords.  A wave keeps the weights of 32 channels in registers for all its
// pixels.  Four waves; a workgroup walks `per` tiles of TR output rows and loads the next tile's rows of x behind the MFMAs of the current.
//
// us, product that gathers / this: 32 x 3 x 224 x 224 7x7 -> 64 float32 105.8 / 58.7, bfloat16 57.4 / 27.2; -> 16 float32
// 102 / 31; 32 x 3 x 190 x 190 -> 51 float32 78.3 / 45; 32 x 3 x 125 x 125 -> 64 bfloat16 24.2 / 16.5.  What bounds it: float32 the MFMAs, 54 GFLOP of parts and padding (43 at
// the rate of a large bfloat16 product); bfloat16 the stores, 51 MB.
//
// float32: sums that are not finite are thrown away, and the wave's 32 x 32 results come from float32 MFMAs over memory.
//
// Supplied by the host: IN (0 bfloat16, 1 float16, 2 float32), Y_16 (result in the operands' 16-bit type, else float32), C_, H_, W_, K_, R_, S_, OH_, OW_,
// SH, PH, PW, DH, TR (output rows of a tile).

typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
typedef unsigned mjt_u32x2v __attribute__((ext_vector_type(2)));
#if IN == 1
typedef _Float16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mjt_h8, a), __builtin_bit_cast(mjt_h8, b), c, 0, 0, 0)
#else
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mjt_h8, a), __builtin_bit_cast(mjt_h8, b), c, 0, 0, 0)
#endif
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros

template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

#ifndef EPI
#define EPI 0
#define EPI_WORDS 0
#endif
struct Params { void* a[6 + EPI_WORDS]; };       // x, w, y, images, tiles a workgroup, bytes of x

constexpr int ESZ = IN == 2 ? 4 : 2, PARTS = IN == 2 ? 3 : 1;
constexpr int CRS = C_ * R_ * S_, ROWS = C_ * R_, STEPS = (ROWS + 1) / 2;
constexpr int KH = K_ > 32 ? 2 : 1, KBLOCKS = (K_ + 32 * KH - 1) / (32 * KH), PW_ = 4 / KH;      // channel halves, blocks of channels, waves along the pixels
constexpr int SHIFT = PW & 1;                                          // a window begins at an even place: its first tap is value SHIFT of the 8
constexpr int LP = (PW + SHIFT + 3) / 4 * 4, FIRST = LP - PW - SHIFT;   // zeros left of a row; where the first window begins
constexpr int XR = (TR - 1) * SH + (R_ - 1) * DH + 1;
constexpr int WIDTH = LP + W_ > FIRST + 2 * OW_ + 6 ? LP + W_ : FIRST + 2 * OW_ + 6, PITCH = (WIDTH + 3) / 4 * 4;
constexpr int PARTB = C_ * XR * PITCH * 2, WPITCH = CRS | 1;           // bytes of a part; the weights' rows on their way: an odd pitch
constexpr int LDSB = PARTS * PARTB > 32 * KH * WPITCH * 4 ? PARTS * PARTB : 32 * KH * WPITCH * 4;
constexpr int NPX = TR * OW_, PT = (NPX + 31) / 32, TPI = (OH_ + TR - 1) / TR;
constexpr int G = W_ % 4 == 0 ? 4 : W_ % 2 == 0 ? 2 : 1;               // values of one load
constexpr int UNITS = C_ * XR * (W_ / G), NI = (UNITS + 255) / 256, GD = G * ESZ < 4 ? 1 : G * ESZ / 4;
static_assert(S_ + SHIFT <= 8 && LDSB <= 160 * 1024, "layout");

constexpr int row_at(int row) { return (row / R_ * XR + row % R_ * DH) * PITCH * 2; }             // bytes from an output row's first row of x
constexpr unsigned mask_of(int d) {                                    // values of dword d of a window that are taps
    return (2 * d >= SHIFT && 2 * d < SHIFT + S_ ? 0xffffu : 0u) | (2 * d + 1 >= SHIFT && 2 * d + 1 < SHIFT + S_ ? 0xffff0000u : 0u);
}

extern "C" __global__ __launch_bounds__(256, 2) void ENTRY(Params p) {
    const int N = (int)(long long)p.a[3], per = (int)(long long)p.a[4], tiles = N * TPI;
    const int kb = blockIdx.x % KBLOCKS, first = blockIdx.x / KBLOCKS * per, last = first + per < tiles ? first + per : tiles;
    if (first >= tiles) return;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDSB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5, wk = wave % KH, wp = wave / KH;
    const int k0 = (kb * KH + wk) * 32;
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[0], 0, (int)(long long)p.a[5], 0x00020000);

    unsigned xv[NI][GD];
    auto fetch = [&](int tile) {
        const int n = tile / TPI, ih0 = (tile - n * TPI) * TR * SH - PH;
        unsigned t = tid;
        asm volatile("" : "+v"(t));                    // (worked out anew for every tile: kept, the offsets would push the weights out)
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int u = (int)t + i * 256, row = u / (W_ / G), q = u - row * (W_ / G), c = row / XR, ih = ih0 + row - c * XR;
            const bool in = (i * 256 + 255 < UNITS || u < UNITS) && ih >= 0 && ih < H_;
            const unsigned off = in ? (unsigned)(((n * C_ + c) * H_ + ih) * W_ + q * G) * (unsigned)ESZ : MJT_NONE;
            if constexpr (G * ESZ == 2) {
                xv[i][0] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(x_rsrc, (int)off, 0, 0);
            } else if constexpr (G * ESZ == 4) {
                xv[i][0] = __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)off, 0, 0);
            } else if constexpr (G * ESZ == 8) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(x_rsrc, (int)off, 0, 0);
                xv[i][0] = v[0]; xv[i][GD - 1] = v[1];
            } else {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, (int)off, 0, 0);
                mjt_static_for<0, GD>([&](auto ec) { xv[i][decltype(ec)::v] = v[decltype(ec)::v]; });
            }
        });
    };
    auto commit = [&]() {                              // to LDS
        unsigned t = tid;
        asm volatile("" : "+v"(t));
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int u = (int)t + i * 256, row = u / (W_ / G), q = u - row * (W_ / G);
            if (i * 256 + 255 < UNITS || u < UNITS) {
                unsigned char* const to = lds + (row * PITCH + LP + q * G) * 2;
#if IN == 2
                unsigned a[2][3];
                mjt_split(xv[i][0], G > 1 ? xv[i][G > 1 ? 1 : 0] : 0u, a[0][0], a[0][1], a[0][2]);
                if constexpr (G == 4) mjt_split(xv[i][GD - 2], xv[i][GD - 1], a[1][0], a[1][1], a[1][2]);
                mjt_static_for<0, 3>([&](auto pc) {
                    constexpr int part = decltype(pc)::v;
                    if constexpr (G == 4) *(mjt_u32x2v*)(to + part * PARTB) = (mjt_u32x2v){a[0][part], a[1][part]};
                    else if constexpr (G == 2) *(unsigned*)(to + part * PARTB) = a[0][part];
                    else *(unsigned short*)(to + part * PARTB) = (unsigned short)a[0][part];
                });
#else
                if constexpr (G == 4) *(mjt_u32x2v*)to = (mjt_u32x2v){xv[i][0], xv[i][GD - 1]};
                else if constexpr (G == 2) *(unsigned*)to = xv[i][0];
                else *(unsigned short*)to = (unsigned short)xv[i][0];
#endif
            }
        });
    };

    // the weights of the wave's channels, by way of LDS: lane (l32, half) holds channel l32 and row 2 * step + half of taps
    fetch(first);
    mjt_u32x4v wf[STEPS][PARTS];
    for (int i = tid; i < 32 * KH * CRS; i += 256) {
        const int k = i / CRS, e = i - k * CRS, ko = kb * KH * 32 + k;
#if IN == 2
        ((unsigned*)lds)[k * WPITCH + e] = ko < K_ ? ((const unsigned*)p.a[1])[(long long)ko * CRS + e] : 0u;
#else
        ((unsigned*)lds)[k * WPITCH + e] = ko < K_ ? (unsigned)((const unsigned short*)p.a[1])[(long long)ko * CRS + e] : 0u;
#endif
    }
    __syncthreads();
    {
        const unsigned* const from = (const unsigned*)lds + (wk * 32 + l32) * WPITCH;
        mjt_static_for<0, STEPS>([&](auto sc) {
            constexpr int step = decltype(sc)::v;
            const bool none = 2 * step + 1 >= ROWS && half == 1;
            const int row = none ? 2 * step : 2 * step + half;
            unsigned v[8];
            mjt_static_for<0, 8>([&](auto ec) {
                constexpr int e = decltype(ec)::v;
                v[e] = 0u;
                if constexpr (e >= SHIFT && e < SHIFT + S_) v[e] = none ? 0u : from[row * S_ + e - SHIFT];
            });
            mjt_static_for<0, 4>([&](auto dc) {
                constexpr int d = decltype(dc)::v;
#if IN == 2
                unsigned a[3];
                mjt_split(v[2 * d], v[2 * d + 1], a[0], a[1], a[2]);
                mjt_static_for<0, 3>([&](auto pc) { wf[step][decltype(pc)::v][d] = a[decltype(pc)::v]; });
#else
                wf[step][0][d] = v[2 * d] | v[2 * d + 1] << 16;
#endif
            });
        });
    }
    __syncthreads();
    for (int i = tid * 16; i < LDSB / 16 * 16; i += 256 * 16) *(mjt_u32x4v*)(lds + i) = (mjt_u32x4v)(0u);      // (margins stay zero)
    for (int i = LDSB / 16 * 16 + tid; i < LDSB; i += 256) lds[i] = 0;

#pragma unroll 1
    for (int tile = first; tile < last; tile++) {
        __syncthreads();
        commit();
        __syncthreads();
        if (tile + 1 < last) fetch(tile + 1);
        const int n = tile / TPI, oh0 = (tile - n * TPI) * TR;
#pragma unroll 1
        for (int pt = wp; pt < PT; pt += PW_) {
            int q = pt * 32 + l32;
            q = q < NPX ? q : NPX - 1;
            const int row = q / OW_, col = q - row * OW_;
            const unsigned char* const from = lds + (row * SH * PITCH + FIRST + 2 * col) * 2;
            mjt_f32x16 acc = (mjt_f32x16)(0.0f), acc2 = (mjt_f32x16)(0.0f);
            // operand f: part 2, 1 or 0 (16 bits: the only one) of step f / PARTS, asked for three operands ahead of its MFMAs
            mjt_u32x4v ring[4];
            auto request = [&](auto fc) {
                constexpr int f = decltype(fc)::v, step = f / PARTS, part = PARTS - 1 - f % PARTS, r0 = 2 * step, r1 = 2 * step + 1 < ROWS ? 2 * step + 1 : 2 * step;
                const unsigned char* const at = from + (half ? row_at(r1) : row_at(r0)) + part * PARTB;
                mjt_static_for<0, 4>([&](auto dc) { ring[f % 4][decltype(dc)::v] = *(const unsigned*)(at + decltype(dc)::v * 4); });
            };
            mjt_static_for<0, (STEPS * PARTS < 3 ? STEPS * PARTS : 3)>(request);
            mjt_static_for<0, STEPS * PARTS>([&](auto fc) {
                constexpr int f = decltype(fc)::v, step = f / PARTS, part = PARTS - 1 - f % PARTS;
                __builtin_amdgcn_sched_barrier(0);     // (left to itself the compiler asks for an operand where it is needed)
                if constexpr (f + 3 < STEPS * PARTS) request(mjt_ic<f + 3>());
                mjt_u32x4v b = ring[f % 4];
                if constexpr (IN != 2)                 // (what is no tap may be infinite; float32 sums are looked at)
                    mjt_static_for<0, 4>([&](auto dc) {
                        constexpr int d = decltype(dc)::v;
                        if constexpr (mask_of(d) != ~0u) b[d] &= mask_of(d);
                        if constexpr (2 * step + 1 >= ROWS) b[d] = half ? 0u : b[d];
                    });
                if constexpr (PARTS == 1) {
                    acc = MJT_MFMA(wf[step][0], b, acc);
                } else if constexpr (part == 2) {
                    acc2 = MJT_MFMA(wf[step][0], b, acc2);
                } else if constexpr (part == 1) {
                    acc2 = MJT_MFMA(wf[step][1 % PARTS], b, acc2);
                    acc2 = MJT_MFMA(wf[step][0], b, acc2);
                } else {
                    acc2 = MJT_MFMA(wf[step][2 % PARTS], b, acc2);
                    acc = MJT_MFMA(wf[step][0], b, acc);
                    acc2 = MJT_MFMA(wf[step][1 % PARTS], b, acc2);
                }
            });
            const int oh = oh0 + row;
#if IN == 2
            acc += acc2;
            float z = 0.0f;                        // not zero if any sum is not finite
            mjt_static_for<0, 16>([&](auto ec) { z += acc[decltype(ec)::v] * 0.0f; });
            const bool again = __any(!(z == 0.0f));
            acc *= MJT_SPLIT_DOWN;
            if (again) {
                acc = (mjt_f32x16)(0.0f);
                const int ih0 = oh * SH - PH, iw0 = col * 2 - PW, ko = k0 + l32 < K_ ? k0 + l32 : K_ - 1;
                const float* const w = (const float*)p.a[1] + (long long)ko * CRS;
#pragma unroll 1
                for (int t0 = 0; t0 < CRS; t0 += 2) {  // (lanes of the upper half: the next tap)
                    const int t = t0 + half < CRS ? t0 + half : t0, c = t / (R_ * S_), r = t / S_ % R_, s = t % S_;
                    const int ih = ih0 + r * DH, iw = iw0 + s;
                    const bool in = ih >= 0 && ih < H_ && iw >= 0 && iw < W_ && t == t0 + half;
                    const float b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(x_rsrc, in ? (int)((unsigned)(((n * C_ + c) * H_ + ih) * W_ + iw) * 4u) : (int)MJT_NONE, 0, 0));
                    const float a = t == t0 + half ? w[t] : 0.0f;
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
                }
            }
#endif
            // D: lane holds column (pixel) lane % 32, rows (k) 8 * (e / 4) + 4 * (lane / 32) + e % 4
            if (pt * 32 + l32 < NPX && oh < OH_) {
                const long long base = ((long long)(n * K_ + k0 + 4 * half) * OH_ + oh) * OW_ + col;
#if EPI
                mjt_static_for<0, 4>([&](auto qc) {    // (what the group reads, four places at a time: sixteen would push the weights out)
                    constexpr int q = decltype(qc)::v;
                    mjt_epi_in<1> read[4];
                    mjt_static_for<0, 4>([&](auto ec) {
                        constexpr int e = decltype(ec)::v, k = 8 * q + e;
                        mjt_epi_load(p, read[e], (MJT_EPI_INDEX)(K_ % 32 == 0 || k0 + 4 * half + k < K_ ? base + k * (OH_ * OW_) : 0));
                    });
                    mjt_static_for<0, 4>([&](auto ec) {
                        constexpr int e = decltype(ec)::v, k = 8 * q + e;
                        if (K_ % 32 == 0 || k0 + 4 * half + k < K_) mjt_epi_finish(p, read[e], (MJT_EPI_INDEX)(base + k * (OH_ * OW_)), {acc[4 * q + e]});
                    });
                });
#else
                mjt_static_for<0, 16>([&](auto ec) {
                    constexpr int e = decltype(ec)::v, k = 8 * (e / 4) + e % 4;
                    if (K_ % 32 == 0 || k0 + 4 * half + k < K_) {
#if Y_16 && IN == 1
                        ((_Float16*)p.a[2])[base + k * (OH_ * OW_)] = (_Float16)acc[e];
#elif Y_16
                        ((unsigned short*)p.a[2])[base + k * (OH_ * OW_)] = (unsigned short)(__float_as_uint(acc[e]) >> 16);      // (truncation)
#else
                        ((float*)p.a[2])[base + k * (OH_ * OW_)] = acc[e];
#endif
                    }
                });
#endif
            }
        }
    }
}
