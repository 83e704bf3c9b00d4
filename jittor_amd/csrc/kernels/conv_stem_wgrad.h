// Weight gradient of a float32 convolution of images with few channels, the first layer of a network, from windows that lie in LDS:
//   dw[k][c][r][s] = sum_{n,oh,ow} dy[n][k][oh][ow] * x[n][c][oh*SH-PH+r*DH][ow*2-PW+s]
// (python/jittor/nn.py:1251-1262 differentiated by ops/reduce_op.cc:339-362; opt/tuner/conv_tuner.cc:375-397 relays it) with horizontal stride 2.  Every
// value becomes three bfloat16 parts, six of whose nine products are summed (split.h has the reasoning), in float32.
//
// What it replaces, the product that gathers both operands (gemm_mfma.h, CONV 2), loads x once for each tap that sees it and multiplies with
// float32 MFMAs.  Here the rows of x under TR output rows lie in LDS, split, even and odd columns apart: a column (c, r, s) of the product
// reads the 8 pixels of a step as 8 consecutive values of one of the two, 5 dwords that a shift by its lane's own parity aligns.  dy is
// read once, from memory into registers: lane (k, half) of v_mfma_f32_32x32x16 holds 8 pixels of channel k and splits them for all columns.
// Four waves: KH halves of the channels times groups that take every (4 / KH)-th step of 16 pixels of a row; the groups' sums meet in LDS.
// A workgroup walks `per` tiles and leaves a slice of the sum, which a reduce launch adds up.
//
// us with the fold, product that gathers / this: 32 x 3 x 224 x 224 7x7 -> 64 107 / 59.6, -> 16 103.5 / 36, 32 x 3 x 190 x 190 -> 51 99.6 / 65.5; relative error against 64 bits
// 2.4e-7 / 1.8e-7 at 1 x 3 x 224 x 224.  What bounds it: 49 GFLOP of parts and padding on the MFMAs (39 at the rate of a large bfloat16 product) beside 5 dwords of LDS
// and 4 shifts for every operand of 8 pixels; the fold takes 10.
//
// Sums that are not finite are thrown away, and the workgroup's slice comes from float32 MFMAs over memory.
//
// Supplied by the host: C_, H_, W_, K_, R_, S_, OH_, OW_, SH, PH, PW, DH, TR (output rows of a tile).

typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mjt_h8, a), __builtin_bit_cast(mjt_h8, b), c, 0, 0, 0)
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros

template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

struct Params { void* a[7]; };       // x, dy, partial, images, tiles a workgroup, bytes of x, bytes of dy

constexpr int CRS = C_ * R_ * S_, NT = (CRS + 31) / 32;
constexpr int KH = K_ > 32 ? 2 : 1, KBLOCKS = (K_ + 32 * KH - 1) / (32 * KH), GROUPS = 4 / KH;
constexpr int LP = (PW + 3) / 4 * 4, XR = (TR - 1) * SH + (R_ - 1) * DH + 1, TPI = (OH_ + TR - 1) / TR;
constexpr int NS = (OW_ + 15) / 16, UNITS = TR * NS;                    // steps of a row, of a tile
constexpr int REACH = NS * 16 + (S_ - 1 - PW + LP) / 2 + 2, HALFW = (LP + W_ + 1) / 2 > REACH ? (LP + W_ + 1) / 2 : REACH;
constexpr int PL = (HALFW + 1) / 2 % 2 == 1 ? (HALFW + 1) / 2 * 2 : (HALFW + 1) / 2 * 2 + 2;       // values of a row's even or odd columns: an odd number of dwords
constexpr int PARTB = C_ * XR * 2 * PL * 2;
constexpr int OUTB = 32 * KH * NT * 32 * 4, LDSB = (3 * PARTB > OUTB ? 3 * PARTB : OUTB) + 16;
constexpr int G = W_ % 4 == 0 ? 4 : W_ % 2 == 0 ? 2 : 1, XU = C_ * XR * (W_ / G), NI = (XU + 255) / 256;
constexpr int GY = OW_ % 4 == 0 ? 4 : OW_ % 2 == 0 ? 2 : 1;            // values of a load of x, of dy
static_assert(LDSB <= 160 * 1024, "LDS");

// G values from byte `off` on
template <int N> __device__ __forceinline__ void mjt_load(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned* to) {
    if constexpr (N == 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
        to[0] = v[0]; to[1] = v[1]; to[2] = v[2]; to[3] = v[3];
    } else if constexpr (N == 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
        to[0] = v[0]; to[1] = v[1];
    } else {
        to[0] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
    }
}

extern "C" __global__ __launch_bounds__(256, 2) void ENTRY(Params p) {
    const int N = (int)(long long)p.a[3], per = (int)(long long)p.a[4], tiles = N * TPI;
    const int kb = blockIdx.x % KBLOCKS, slice = blockIdx.x / KBLOCKS, first = slice * per, last = first + per < tiles ? first + per : tiles;
    if (first >= tiles) return;
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDSB];
    __shared__ unsigned unsound;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5, wk = wave % KH, group = wave / KH;
    const int k = (kb * KH + wk) * 32 + l32;
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[0], 0, (int)(long long)p.a[5], 0x00020000);
    const __amdgpu_buffer_rsrc_t d_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[1], 0, (int)(long long)p.a[6], 0x00020000);

    unsigned xv[NI][G];
    auto fetch = [&](int tile) {
        const int n = tile / TPI, ih0 = (tile - n * TPI) * TR * SH - PH;
        unsigned t = tid;
        asm volatile("" : "+v"(t));                    // (worked out anew for every tile: kept, the offsets would push the accumulators out)
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int u = (int)t + i * 256, row = u / (W_ / G), q = u - row * (W_ / G), c = row / XR, ih = ih0 + row - c * XR;
            const bool in = (i * 256 + 255 < XU || u < XU) && ih >= 0 && ih < H_;
            mjt_load<G>(x_rsrc, in ? (unsigned)(((n * C_ + c) * H_ + ih) * W_ + q * G) * 4u : MJT_NONE, xv[i]);
        });
    };
    auto commit = [&]() {                              // to LDS, as parts: [part][c][row][even, odd columns][column / 2]
        unsigned t = tid;
        asm volatile("" : "+v"(t));
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int u = (int)t + i * 256, row = u / (W_ / G), col = LP + (u - row * (W_ / G)) * G;
            if (i * 256 + 255 < XU || u < XU) {
                unsigned e[3], o[3];                   // even columns and odd ones, two each (or one)
                unsigned char* const to = lds + (row * 2 * PL + (col >> 1)) * 2;
                if constexpr (G == 4) {
                    mjt_split(xv[i][0], xv[i][G / 2], e[0], e[1], e[2]);
                    mjt_split(xv[i][G / 4], xv[i][G - 1], o[0], o[1], o[2]);
                    mjt_static_for<0, 3>([&](auto pc) {
                        constexpr int part = decltype(pc)::v;
                        *(unsigned*)(to + part * PARTB) = e[part];
                        *(unsigned*)(to + part * PARTB + PL * 2) = o[part];
                    });
                } else {
                    mjt_split(xv[i][0], xv[i][G - 1], e[0], e[1], e[2]);
                    mjt_static_for<0, 3>([&](auto pc) {
                        constexpr int part = decltype(pc)::v;
                        if constexpr (G == 2) {
                            *(unsigned short*)(to + part * PARTB) = (unsigned short)e[part];
                            *(unsigned short*)(to + part * PARTB + PL * 2) = (unsigned short)(e[part] >> 16);
                        } else {
                            *(unsigned short*)(to + part * PARTB + (col & 1) * (PL * 2)) = (unsigned short)e[part];
                        }
                    });
                }
            }
        });
    };
    // 8 pixels of the lane's channel in step u of a tile
    auto fetch_dy = [&](int n, int oh0, int u, unsigned (&to)[8]) {
        const int row = u / NS, px = (u - row * NS) * 16 + half * 8, oh = oh0 + row;
        const bool in = u < UNITS && k < K_ && oh < OH_;
        const unsigned off = (unsigned)(((n * K_ + k) * OH_ + oh) * OW_ + px) * 4u;
        mjt_static_for<0, 8 / GY>([&](auto ic) {
            constexpr int e = decltype(ic)::v * GY;
            mjt_load<GY>(d_rsrc, in && px + e < OW_ ? off + e * 4u : MJT_NONE, to + e);
        });
    };

    // where the lane's columns read: 5 dwords from there on, 0 or 16 bits to the right (columns past the last repeat the first)
    int at[NT];
    unsigned odd = 0;                                  // bit t: the window of column tile t begins in the upper half of its dword
    mjt_static_for<0, NT>([&](auto tc) {
        constexpr int t = decltype(tc)::v;
        const int col = t * 32 + l32 < CRS ? t * 32 + l32 : 0, c = col / (R_ * S_), r = col / S_ % R_, v = col % S_ - PW + LP, j = v >> 1;
        at[t] = (((c * XR + r * DH) * 2 + (v & 1)) * PL + (j & ~1) + half * 8) * 2;
        odd |= (unsigned)(j & 1) << t;
    });
    mjt_f32x16 acc[NT];
    mjt_static_for<0, NT>([&](auto tc) { acc[decltype(tc)::v] = (mjt_f32x16)(0.0f); });

    fetch(first);
    if (tid == 0) unsound = 0;
    for (int i = tid * 16; i < LDSB / 16 * 16; i += 256 * 16) *(mjt_u32x4v*)(lds + i) = (mjt_u32x4v)(0u);      // (margins stay zero)
#pragma unroll 1
    for (int tile = first; tile < last; tile++) {
        const int n = tile / TPI, oh0 = (tile - n * TPI) * TR;
        unsigned dv[8];
        fetch_dy(n, oh0, group, dv);
        __syncthreads();
        commit();
        __syncthreads();
        if (tile + 1 < last) fetch(tile + 1);
#pragma unroll 1
        for (int u = group; u < UNITS; u += GROUPS) {
            unsigned a[3][4];
            mjt_static_for<0, 4>([&](auto ec) {
                constexpr int e = decltype(ec)::v;
                mjt_split(dv[2 * e], dv[2 * e + 1], a[0][e], a[1][e], a[2][e]);
            });
            fetch_dy(n, oh0, u + GROUPS, dv);
            const mjt_u32x4v ah = {a[0][0], a[0][1], a[0][2], a[0][3]}, am = {a[1][0], a[1][1], a[1][2], a[1][3]}, al = {a[2][0], a[2][1], a[2][2], a[2][3]};
            const int row = u / NS, step = (row * SH * 2 * PL + (u - row * NS) * 16) * 2;
            // operand f: part 2, 1 or 0 of column tile f / 3, asked for two operands ahead of its MFMAs
            unsigned ring[3][5];
            auto request = [&](auto fc) {
                constexpr int f = decltype(fc)::v, t = f / 3, part = 2 - f % 3;
                const unsigned char* const from = lds + at[t] + step + part * PARTB;
                mjt_static_for<0, 5>([&](auto ec) { ring[f % 3][decltype(ec)::v] = *(const unsigned*)(from + decltype(ec)::v * 4); });
            };
            request(mjt_ic<0>());
            request(mjt_ic<1>());
            mjt_static_for<0, NT * 3>([&](auto fc) {
                constexpr int f = decltype(fc)::v, t = f / 3, part = 2 - f % 3;
                __builtin_amdgcn_sched_barrier(0);         // (left to itself the compiler asks for an operand where it is needed)
                if constexpr (f + 2 < NT * 3) request(mjt_ic<f + 2>());
                const unsigned shift = (odd >> t & 1) * 16;
                const unsigned (&d)[5] = ring[f % 3];
                mjt_u32x4v b;
                mjt_static_for<0, 4>([&](auto ec) { b[decltype(ec)::v] = __builtin_amdgcn_alignbit(d[decltype(ec)::v + 1], d[decltype(ec)::v], shift); });
                if constexpr (part == 0) acc[t] = MJT_MFMA(al, b, acc[t]);
                if constexpr (part != 2) acc[t] = MJT_MFMA(am, b, acc[t]);
                acc[t] = MJT_MFMA(ah, b, acc[t]);
            });
        }
    }
    {
        float z = 0.0f;                                // not zero if any sum is not finite
        mjt_static_for<0, NT * 16>([&](auto ec) { z += acc[decltype(ec)::v / 16][decltype(ec)::v % 16] * 0.0f; });
        if (!(z == 0.0f)) unsound = 1;
        mjt_static_for<0, NT>([&](auto tc) { acc[decltype(tc)::v] *= MJT_SPLIT_DOWN; });
    }
    __syncthreads();
    if (unsound) {
        mjt_static_for<0, NT>([&](auto tc) { acc[decltype(tc)::v] = (mjt_f32x16)(0.0f); });
#pragma unroll 1
        for (int tile = first; tile < last; tile++) {
            const int n = tile / TPI, oh0 = (tile - n * TPI) * TR;
#pragma unroll 1
            for (int u = group; u < TR * OW_ / 2 + TR; u += GROUPS) {      // two pixels of a row: the lanes' halves
                constexpr int PAIRS = (OW_ + 1) / 2;
                const int row = u / PAIRS, ow = (u - row * PAIRS) * 2 + half, oh = oh0 + row;
                const bool px = row < TR && oh < OH_ && ow < OW_;
                const float a = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(d_rsrc, px && k < K_ ? (int)((unsigned)(((n * K_ + k) * OH_ + oh) * OW_ + ow) * 4u) : (int)MJT_NONE, 0, 0));
                mjt_static_for<0, NT>([&](auto tc) {
                    const int col = decltype(tc)::v * 32 + l32, c = col / (R_ * S_), ih = oh * SH - PH + col / S_ % R_ * DH, iw = ow * 2 - PW + col % S_;
                    const bool in = px && col < CRS && ih >= 0 && ih < H_ && iw >= 0 && iw < W_;
                    const float b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(x_rsrc, in ? (int)((unsigned)(((n * C_ + c) * H_ + ih) * W_ + iw) * 4u) : (int)MJT_NONE, 0, 0));
                    acc[decltype(tc)::v] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[decltype(tc)::v], 0, 0, 0);
                });
            }
        }
    }
    // D of a 32 x 32 tile: lane holds column (c, r, s) lane % 32, rows (k) 8 * (e / 4) + 4 * (lane / 32) + e % 4; the groups' sums meet in LDS
    float* const out = (float*)lds;
    auto place = [&](int t, int e) { return (wk * 32 + 8 * (e / 4) + 4 * half + e % 4) * (NT * 32) + t * 32 + l32; };
    mjt_static_for<1, GROUPS>([&](auto gc) {
        if (group == decltype(gc)::v)
            mjt_static_for<0, NT * 16>([&](auto ec) { out[place(decltype(ec)::v / 16, decltype(ec)::v % 16)] = acc[decltype(ec)::v / 16][decltype(ec)::v % 16]; });
        __syncthreads();
        if (group == 0)
            mjt_static_for<0, NT * 16>([&](auto ec) { acc[decltype(ec)::v / 16][decltype(ec)::v % 16] += out[place(decltype(ec)::v / 16, decltype(ec)::v % 16)]; });
        __syncthreads();
    });
    if (group != 0) return;
    float* const part = (float*)p.a[2] + (long long)slice * (K_ * CRS);
    mjt_static_for<0, NT * 16>([&](auto ec) {
        constexpr int t = decltype(ec)::v / 16, e = decltype(ec)::v % 16;
        const int ko = (kb * KH + wk) * 32 + 8 * (e / 4) + 4 * half + e % 4, col = t * 32 + l32;
        if ((K_ % 32 == 0 || ko < K_) && (CRS % 32 == 0 || col < CRS)) part[ko * CRS + col] = acc[t][e];
    });
}
