// Input gradient of a strided convolution, all stride phases in one pass:
//   dx[n][c][oh*SH-PH+r*DH][ow*SW-PW+s*DW] += dy[n][k][oh][ow] * w[k][c][r][s]
// (python/jittor/nn.py:1251-1262 differentiated by ops/reindex_op.cc:170-190) for bfloat16 (IN_F16: float16) operands, exact products, float32
// sums, one rounding of a 16-bit result.
//
// A phase (a, b) of dx, the positions (SH*i + a, SW*j + b), is a convolution of dy with its own taps: tap r belongs to the phase
// a = (r*DH - PH) mod SH and reads dy at row i + (a + PH - r*DH) / SH, columns alike.  No product has a zero factor between dy's rows.
//
// What it replaces, a convolution per phase into its own buffer and a pass that interleaves them, read dy once a phase, wrote and read dx one
// time more and was ten launches.  Here a workgroup takes 64 channels and 64 * PT base positions (n, i, j) with the accumulators of all
// phases, so dy comes in once and phases that share a row leave as pairs.
//
// Layout.  A stage is KU * 16 channels of dy.  dy lies in LDS as [8 channels of 2 KU][position][channel], positions being those of dy with
// the margins that the taps' shifts reach (zeros), SPAN of them from the tile's first on: a shift is a constant distance.  A thread makes 8
// channels' pieces of one position from single values, or of two from dwords where rows are even.  Weights come packed as
// [64 channels][stage][16 channels of KU][tap][8 channels of dy][channel of dx][channel of dy].  Both are runs of 16 bytes that neighbouring lanes read side by
// side (rows of 32 bytes, the halves side by side, met in the banks: 64 x 512 x 14 x 14 3x3 -> 512 43.1 us so, 40.4 now).
// v_mfma_f32_32x32x16, weights the first operand: a lane ends up with one position and 16 channels.  Four waves, 2 halves of the channels x
// 2 of the positions; two LDS buffers, the next stage is loaded into registers ahead of a stage's MFMAs and written behind them; two
// workgroups on a compute unit hide one another's barriers.
// us a call, packing included, phase by phase / this: 64 x 256 x 28 x 28 3x3 -> 256 96 / 32.0; 64 x 128 x 56 x 56 -> 128 82 / 33.4; 64 x 512 x 14 x 14 -> 512 134 /
// 40.4; 1 x 256 x 28 x 28 -> 256 76 / 15.1; 32 x 64 x 32 x 32 5x5 -> 128 66 / 16.9; 64 x 256 x 28 x 28 1x1 -> 512 49 / 18.8; odd maps, with dy spread out / this: 64 x 64 x
// 31 x 31 3x3 -> 64 47 / 11.1; closest 1 x 512 x 7 x 7 -> 512 26.9 / 25.2.  What bounds the first of these: the 16 stages of a workgroup, 0.9 us each of which the
// MFMAs are half, on 392 of 512 places; the packing takes 5.
//
// Supplied by the host: C_, H_, W_, K_, R_, S_, OH_, OW_, SH, SW, PH, PW, DH, DW, IN_F16, Y_16 (result in the operands' type, else float32), KU, PT, SPAN.

#if IN_F16
typedef _Float16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_f16
#else
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_bf16
#endif
typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
typedef float mjt_f32x2v __attribute__((ext_vector_type(2)));
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros

template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

struct Params { void* a[6]; };       // packed weights, dy, dx, images, bytes of dy, bytes of the packed weights

constexpr int mod_of(int a, int b) { return a % b < 0 ? a % b + b : a % b; }
constexpr int row_phase(int r) { return mod_of(r * DH - PH, SH); }
constexpr int col_phase(int s) { return mod_of(s * DW - PW, SW); }
constexpr int row_shift(int r) { return (row_phase(r) + PH - r * DH) / SH; }
constexpr int col_shift(int s) { return (col_phase(s) + PW - s * DW) / SW; }
constexpr int least(bool cols) {
    int v = 0;
    for (int t = 0; t < (cols ? S_ : R_); t++) { const int d = cols ? col_shift(t) : row_shift(t); if (d < v) v = d; }
    return v;
}
constexpr int most(bool cols) {
    int v = 0;
    for (int t = 0; t < (cols ? S_ : R_); t++) { const int d = cols ? col_shift(t) : row_shift(t); if (d > v) v = d; }
    return v;
}
constexpr int TAPS = R_ * S_, PHASES = SH * SW, OHW = OH_ * OW_;
constexpr int RLO = least(false), RHI = most(false), CLO = least(true), CHI = most(true), NRS = RHI - RLO + 1, NCS = CHI - CLO + 1;
constexpr int UNIT = OW_ % 2 == 0 ? 2 : 1;                                      // positions of one load
constexpr int HB = (H_ + SH - 1) / SH, WB = (W_ + SW - 1) / SW;                 // base positions of an image
constexpr int LPC = (-CLO + UNIT - 1) / UNIT * UNIT;                            // margin left of a row
constexpr int PR = HB + RHI - RLO, PC = (LPC + WB + CHI + UNIT - 1) / UNIT * UNIT;   // rows and columns of an image with its margins
constexpr bool shift_used(int dr, int dc) {
    bool r_ = false, c_ = false;
    for (int r = 0; r < R_; r++) r_ = r_ || row_shift(r) == dr;
    for (int s = 0; s < S_; s++) c_ = c_ || col_shift(s) == dc;
    return r_ && c_;
}
constexpr int TILE = 64 * PT, KC = 16 * KU, STAGES = (K_ + KC - 1) / KC, CT = (C_ + 63) / 64;
constexpr int AB = KU * TAPS * 2048, DB = KU * SPAN * 32, BUFB = AB + DB;
constexpr int NA = (AB / 16 + 255) / 256;                                       // 16-byte pieces of the weights a thread copies
constexpr int UNITS = SPAN / UNIT, ITEMS = UNITS * 2 * KU, NI = (ITEMS + 255) / 256;
static_assert(SPAN % UNIT == 0 && 2 * BUFB <= 160 * 1024, "LDS");

__device__ __forceinline__ unsigned mjt_narrow2(float x, float y) {
#if IN_F16
    return (unsigned)__builtin_bit_cast(unsigned short, (_Float16)x) | (unsigned)__builtin_bit_cast(unsigned short, (_Float16)y) << 16;
#else
    return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);       // (truncation)
#endif
}

extern "C" __global__ __launch_bounds__(256, 2) void ENTRY(Params p) {
    const int N = (int)(long long)p.a[3], total = N * (HB * WB);
    // every XCD takes a run of neighbouring (positions, channels) pairs: the blocks of channels of a tile read the same dy
    const int pairs = (total + TILE - 1) / TILE * CT, run = (pairs + 7) / 8, pair = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= run || pair >= pairs) return;
    const int tile = pair / CT, ct = pair - tile * CT, f0 = tile * TILE;

    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * BUFB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5, wc = wave & 1, wp = wave >> 1;
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[0], 0, (int)(long long)p.a[5], 0x00020000);
    const __amdgpu_buffer_rsrc_t d_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[1], 0, (int)(long long)p.a[4], 0x00020000);
    auto pos_of = [](int f) {
        const int n = f / (HB * WB), q = f - n * (HB * WB), i = q / WB;
        return (n * PR + i - RLO) * PC + (q - i * WB) + LPC;
    };
    const int q0 = (pos_of(f0) + RLO * PC + CLO) / UNIT * UNIT;

    // staging of dy: item it = (8 channels, unit of positions); where it comes from but for the stage, and where it goes
    unsigned from[NI];
    mjt_static_for<0, NI>([&](auto ic) {
        const int it = tid + decltype(ic)::v * 256, h = it / UNITS, q = q0 + (it - h * UNITS) * UNIT;
        const int n = q / (PR * PC), e = q - n * (PR * PC), row = e / PC + RLO, col = e % PC - LPC;
        const bool in = it < ITEMS && n < N && row >= 0 && row < OH_ && col >= 0 && col < OW_;
        from[decltype(ic)::v] = in ? (unsigned)((n * K_ + h * 8) * OHW + row * OW_ + col) * 2u : MJT_NONE;
    });
    unsigned dv[NI][8];
    mjt_u32x4v av[NA];
    auto fetch = [&](int st) {
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const unsigned off = from[i] + (unsigned)st * (unsigned)(KC * OHW * 2);
            mjt_static_for<0, 8>([&](auto kc) {
                constexpr int k = decltype(kc)::v;
                unsigned o = off + k * OHW * 2;
                if constexpr (K_ % KC != 0) {
                    const int h = (tid + i * 256) / UNITS;
                    if (st * KC + h * 8 + k >= K_) o = MJT_NONE;
                }
                if constexpr (UNIT == 2) dv[i][k] = __builtin_amdgcn_raw_buffer_load_b32(d_rsrc, (int)o, 0, 0);
                else dv[i][k] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(d_rsrc, (int)o, 0, 0);
            });
        });
        const unsigned w0 = (unsigned)((ct * STAGES + st) * AB) + (unsigned)tid * 16u;
        mjt_static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)(w0 + i * 4096), 0, 0);
            av[i] = (mjt_u32x4v){v[0], v[1], v[2], v[3]};
        });
    };
    auto commit = [&](int st) {
        unsigned char* const buf = lds + (st & 1) * BUFB;
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int it = tid + i * 256, h = it / UNITS, u = it - h * UNITS;
            if (i * 256 + 255 < ITEMS || it < ITEMS) {
                unsigned char* const to = buf + AB + (h * SPAN + u * UNIT) * 16;
                mjt_u32x4v lo, hi;
                mjt_static_for<0, 4>([&](auto ec) {
                    constexpr int e = decltype(ec)::v;
                    lo[e] = __builtin_amdgcn_perm(dv[i][2 * e + 1], dv[i][2 * e], 0x05040100u);
                    hi[e] = __builtin_amdgcn_perm(dv[i][2 * e + 1], dv[i][2 * e], 0x07060302u);
                });
                *(mjt_u32x4v*)to = lo;
                if constexpr (UNIT == 2) *(mjt_u32x4v*)(to + 16) = hi;
            }
        });
        mjt_static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            if (i * 256 + 255 < AB / 16 || tid + i * 256 < AB / 16) *(mjt_u32x4v*)(buf + (tid + i * 256) * 16) = av[i];
        });
    };

    const unsigned char* const al = lds + half * 1024 + (wc * 32 + l32) * 16;
    const unsigned char* bl[PT];
    mjt_static_for<0, PT>([&](auto tc) {
        constexpr int t = decltype(tc)::v;
        bl[t] = lds + AB + (half * SPAN + pos_of(f0 + (wp * PT + t) * 32 + l32) - q0) * 16;
    });
    mjt_f32x16 acc[PHASES][PT];
    mjt_static_for<0, PHASES * PT>([&](auto ic) { acc[decltype(ic)::v / PT][decltype(ic)::v % PT] = (mjt_f32x16)(0.0f); });

    fetch(0);
    commit(0);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < STAGES; st++) {
        if (st + 1 < STAGES) fetch(st + 1);
        const int buf = (st & 1) * BUFB;
        mjt_static_for<0, KU * NRS * NCS>([&](auto sc) {
            constexpr int s = decltype(sc)::v, ku = s / (NRS * NCS), dr = s / NCS % NRS + RLO, dc = s % NCS + CLO;
            if constexpr (shift_used(dr, dc)) {
                mjt_u32x4v b[PT];
                mjt_static_for<0, PT>([&](auto tc) { b[decltype(tc)::v] = *(const mjt_u32x4v*)(bl[decltype(tc)::v] + buf + (2 * ku * SPAN + dr * PC + dc) * 16); });
                mjt_static_for<0, TAPS>([&](auto tapc) {
                    constexpr int tap = decltype(tapc)::v, r = tap / S_, c = tap % S_;
                    if constexpr (row_shift(r) == dr && col_shift(c) == dc) {
                        const mjt_u32x4v a = *(const mjt_u32x4v*)(al + buf + (ku * TAPS + tap) * 2048);
                        mjt_static_for<0, PT>([&](auto tc) {
                            mjt_f32x16& to = acc[row_phase(r) * SW + col_phase(c)][decltype(tc)::v];
                            to = MJT_MFMA(__builtin_bit_cast(mjt_h8, a), __builtin_bit_cast(mjt_h8, b[decltype(tc)::v]), to, 0, 0, 0);
                        });
                    }
                });
            }
        });
        if (st + 1 < STAGES) commit(st + 1);            // (into the buffer that nobody has read since the last barrier)
        __syncthreads();
    }

    // D of a 32 x 32 tile: lane holds column (position) lane % 32, rows (c) 8 * (e / 4) + 4 * (lane / 32) + e % 4
#if Y_16
    typedef unsigned short mjt_y;
#else
    typedef float mjt_y;
#endif
    mjt_static_for<0, PT>([&](auto tc) {
        constexpr int t = decltype(tc)::v;
        const int f = f0 + (wp * PT + t) * 32 + l32;
        if (f >= total) return;
        const int n = f / (HB * WB), q = f - n * (HB * WB), i = q / WB, j = q - i * WB;
        const int c0 = ct * 64 + wc * 32 + 4 * half;
        mjt_y* const to = (mjt_y*)p.a[2] + ((long long)(n * C_ + c0) * H_ + i * SH) * W_ + j * SW;
        mjt_static_for<0, 16 * SH>([&](auto ec) {
            constexpr int e = decltype(ec)::v / SH, a = decltype(ec)::v % SH, c = 8 * (e / 4) + e % 4;
            if ((C_ % 64 == 0 || c0 + c < C_) && (H_ % SH == 0 || i * SH + a < H_)) {
                mjt_y* const at = to + (c * H_ + a) * W_;
                if constexpr (SW == 2 && W_ % 2 == 0) {
                    const float x = acc[a * SW][t][e], y = acc[a * SW + SW - 1][t][e];
#if Y_16
                    *(unsigned*)at = mjt_narrow2(x, y);
#else
                    *(mjt_f32x2v*)at = (mjt_f32x2v){x, y};
#endif
                } else {
                    mjt_static_for<0, SW>([&](auto bc) {
                        constexpr int b = decltype(bc)::v;
                        if (W_ % SW == 0 || j * SW + b < W_) {
#if Y_16
                            at[b] = (unsigned short)mjt_narrow2(acc[a * SW + b][t][e], 0.0f);
#else
                            at[b] = acc[a * SW + b][t][e];
#endif
                        }
                    });
                }
            }
        });
    });
}
