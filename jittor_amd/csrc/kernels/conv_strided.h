// Forward convolution with horizontal stride 2 (vertical 1 or 2) from windows in LDS:
//   y[n][k][oh][ow] = sum_{c,r,s} w[k][c][r][s] * x[n][c][oh*SH-PH+r*DH][ow*2-PW+s*DW]
// (python/jittor/nn.py:1251-1262, recognised by opt/tuner/conv_tuner.cc:218-411) for bfloat16 (IN_F16: float16) operands, exact products, float32 sums,
// one rounding of a 16-bit result.  The counterpart of conv_dgrad_phases.h: there the result has phases, here x has.
//
// x falls into planes by (row mod SH, column mod 2); tap (r, s) reads plane ((r*DH - PH) mod SH, (s*DW - PW) mod 2) a constant shift away from the
// output's own position.  A stage is KU * 16 channels: the planes lie in LDS as [16 channels of KU][row phase][column phase][8 channels][position][channel], positions
// being those of y with the margins the shifts reach (zeros), SPAN of them from the tile's first on.  A dword of x is a value of either column phase, so a
// thread makes 8 channels' pieces of both from 8 dwords.  Weights come packed as [32 * WK channels of y][stage][16 channels of KU][tap][8 channels][channel of y]
// [channel].  Both are runs of 16 bytes that neighbouring lanes read side by side (rows of 32 bytes, the halves of a wave side by side, met in the banks: 40.5 us
// instead of 36.1 for the first of the layers below).
// v_mfma_f32_32x32x16, weights the first operand.  A workgroup takes 32 * WK channels and 64 * PT positions, a wave 32 channels and 32 * PT positions; two LDS
// buffers, the next stage is loaded into registers ahead of a stage's MFMAs and written behind them.  (Two stages ahead changes nothing.)
// us, row kernel (conv_mfma.h) / this, packing included: 64 x 256 x 28 x 28 3x3 -> 256 46.0 / 36.1; 8 x 256 x 28 x 28 -> 256 37.9 / 22.0; 64 x 128 x 28 x 28 -> 128 26.3 / 17.6;
// 2 x 512 x 28 x 28 -> 128 72.3 / 35.6; 64 x 512 x 28 x 28 1x1 -> 256 58.1 / 18.0.  What bounds it: LDS, 27 KB of operands for 18 MFMAs of a wave, and
// a stage's barrier.
//
// Supplied by the host: C_, H_, W_, K_, R_, S_, OH_, OW_, SH, PH, PW, DH, DW, IN_F16, Y_16 (result in the operands' type, else float32), KU, PT, WK, SPAN.

#if IN_F16
typedef _Float16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_f16
#else
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_bf16
#endif
typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros

template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

struct Params { void* a[6]; };       // packed weights, x, y, images, bytes of x, bytes of the packed weights

constexpr int floor_of(int a, int b) { return a >= 0 ? a / b : -((b - 1 - a) / b); }
constexpr int row_shift(int r) { return floor_of(r * DH - PH, SH); }
constexpr int col_shift(int s) { return floor_of(s * DW - PW, 2); }
constexpr int row_phase(int r) { return r * DH - PH - SH * row_shift(r); }
constexpr int col_phase(int s) { return s * DW - PW - 2 * col_shift(s); }
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
constexpr bool row_phase_used(int a) { for (int r = 0; r < R_; r++) if (row_phase(r) == a) return true; return false; }
constexpr int FIRST_ROW = row_phase_used(0) ? 0 : 1, NRP = SH == 2 && row_phase_used(0) && row_phase_used(1) ? 2 : 1;      // row phases that taps read
constexpr int TAPS = R_ * S_, HW = H_ * W_;
constexpr int RLO = least(false), RHI = most(false), CLO = least(true), CHI = most(true);
constexpr int LPC = -CLO, PR = OH_ + RHI - RLO, PC = LPC + OW_ + CHI;           // rows and columns of an image's positions with their margins
constexpr int TILE = 64 * PT, KT = 32 * WK, THREADS = 128 * WK, KC = 16 * KU, STAGES = C_ / KC, KB = K_ / KT;
constexpr int PLANEB = SPAN * 32, AB = KU * TAPS * KT * 32, DB = KU * NRP * 2 * PLANEB, BUFB = AB + DB;
constexpr int NA = (AB / 16 + THREADS - 1) / THREADS;                           // 16-byte pieces of the weights a thread copies
constexpr int ITEMS = SPAN * NRP * 2 * KU, NI = (ITEMS + THREADS - 1) / THREADS;
static_assert(C_ % KC == 0 && K_ % KT == 0, "packed weights are as many bytes as w");
static_assert(W_ % 2 == 0 && 2 * BUFB <= 160 * 1024, "dwords of two columns; LDS");

__device__ __forceinline__ unsigned short mjt_narrow(float x) {
#if IN_F16
    return __builtin_bit_cast(unsigned short, (_Float16)x);
#else
    return (unsigned short)(__float_as_uint(x) >> 16);       // (truncation)
#endif
}

extern "C" __global__ __launch_bounds__(THREADS, 2) void ENTRY(Params p) {
    const int N = (int)(long long)p.a[3], total = N * (OH_ * OW_);
    // every XCD takes a run of neighbouring (positions, channels) pairs: the blocks of channels of a tile read the same x
    const int pairs = (total + TILE - 1) / TILE * KB, run = (pairs + 7) / 8, pair = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= run || pair >= pairs) return;
    const int tile = pair / KB, kb = pair - tile * KB, f0 = tile * TILE;

    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * BUFB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5, wk = wave % WK, wp = wave / WK;
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[0], 0, (int)(long long)p.a[5], 0x00020000);
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[1], 0, (int)(long long)p.a[4], 0x00020000);
    auto pos_of = [](int f) {
        const int n = f / (OH_ * OW_), q = f - n * (OH_ * OW_), i = q / OW_;
        return (n * PR + i - RLO) * PC + (q - i * OW_) + LPC;
    };
    const int q0 = pos_of(f0) + RLO * PC + CLO;

    // staging of x: item it = ((8 channels, row phase), position); where its columns come from but for the stage
    unsigned from[NI];
    mjt_static_for<0, NI>([&](auto ic) {
        constexpr int i = decltype(ic)::v;
        const int it = tid + i * THREADS, g = it / SPAN, q = q0 + it - g * SPAN, h = g / NRP, a = FIRST_ROW + g - h * NRP;
        const int n = q / (PR * PC), e = q - n * (PR * PC), row = (e / PC + RLO) * SH + a, col = (e % PC - LPC) * 2;
        const bool in = it < ITEMS && n < N && row >= 0 && row < H_ && col >= 0 && col < W_;
        from[i] = in ? (unsigned)((n * C_ + h * 8) * HW + row * W_ + col) * 2u : MJT_NONE;
    });
    unsigned xv[NI][8];
    mjt_u32x4v av[NA];
    auto fetch = [&](int st) {
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const unsigned off = from[i] + (unsigned)st * (unsigned)(KC * HW * 2);
            mjt_static_for<0, 8>([&](auto kc) {
                constexpr int k = decltype(kc)::v;
                xv[i][k] = __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)(off + k * HW * 2), 0, 0);
            });
        });
        const unsigned w0 = (unsigned)((kb * STAGES + st) * AB) + (unsigned)tid * 16u;
        mjt_static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)(w0 + i * (THREADS * 16)), 0, 0);
            av[i] = (mjt_u32x4v){v[0], v[1], v[2], v[3]};
        });
    };
    auto commit = [&](int st) {
        unsigned char* const buf = lds + (st & 1) * BUFB;
        mjt_static_for<0, NI>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            const int it = tid + i * THREADS, g = it / SPAN, q = it - g * SPAN, h = g / NRP, a = g - h * NRP;
            if (i * THREADS + THREADS - 1 < ITEMS || it < ITEMS) {
                unsigned char* const to = buf + AB + ((h >> 1) * NRP + a) * (2 * PLANEB) + ((h & 1) * SPAN + q) * 16;
                mjt_u32x4v even, odd;
                mjt_static_for<0, 4>([&](auto ec) {
                    constexpr int e = decltype(ec)::v;
                    even[e] = __builtin_amdgcn_perm(xv[i][2 * e + 1], xv[i][2 * e], 0x05040100u);
                    odd[e] = __builtin_amdgcn_perm(xv[i][2 * e + 1], xv[i][2 * e], 0x07060302u);
                });
                *(mjt_u32x4v*)to = even;
                *(mjt_u32x4v*)(to + PLANEB) = odd;
            }
        });
        mjt_static_for<0, NA>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            if (i * THREADS + THREADS - 1 < AB / 16 || tid + i * THREADS < AB / 16) *(mjt_u32x4v*)(buf + (tid + i * THREADS) * 16) = av[i];
        });
    };

    const unsigned char* const al = lds + half * (KT * 16) + (wk * 32 + l32) * 16;
    const unsigned char* bl[PT];
    mjt_static_for<0, PT>([&](auto tc) {
        constexpr int t = decltype(tc)::v;
        bl[t] = lds + AB + (half * SPAN + pos_of(f0 + (wp * PT + t) * 32 + l32) - q0) * 16;
    });
    mjt_f32x16 acc[PT];
    mjt_static_for<0, PT>([&](auto tc) { acc[decltype(tc)::v] = (mjt_f32x16)(0.0f); });

    fetch(0);
    commit(0);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < STAGES; st++) {
        if (st + 1 < STAGES) fetch(st + 1);
        const int buf = (st & 1) * BUFB;
        // the operands of a tap are asked for two taps ahead of its MFMAs
        mjt_u32x4v a[3], b[3][PT];
        auto request = [&](auto sc) {
            constexpr int i = decltype(sc)::v, ku = i / TAPS, tap = i % TAPS, r = tap / S_, s = tap % S_;
            constexpr int at = ((ku * NRP + row_phase(r) - FIRST_ROW) * 2 + col_phase(s)) * PLANEB + (row_shift(r) * PC + col_shift(s)) * 16;
            a[i % 3] = *(const mjt_u32x4v*)(al + buf + (ku * TAPS + tap) * (KT * 32));
            mjt_static_for<0, PT>([&](auto tc) { b[i % 3][decltype(tc)::v] = *(const mjt_u32x4v*)(bl[decltype(tc)::v] + buf + at); });
        };
        mjt_static_for<0, (KU * TAPS < 2 ? KU * TAPS : 2)>(request);
        mjt_static_for<0, KU * TAPS>([&](auto sc) {
            constexpr int i = decltype(sc)::v;
            __builtin_amdgcn_sched_barrier(0);         // (left to itself the compiler asks for an operand where it is needed)
            if constexpr (i + 2 < KU * TAPS) request(mjt_ic<i + 2>());
            mjt_static_for<0, PT>([&](auto tc) {
                acc[decltype(tc)::v] = MJT_MFMA(__builtin_bit_cast(mjt_h8, a[i % 3]), __builtin_bit_cast(mjt_h8, b[i % 3][decltype(tc)::v]), acc[decltype(tc)::v], 0, 0, 0);
            });
        });
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < STAGES) commit(st + 1);            // (into the buffer that nobody has read since the last barrier)
        __syncthreads();
    }

    // D of a 32 x 32 tile: lane holds column (position) lane % 32, rows (k) 8 * (e / 4) + 4 * (lane / 32) + e % 4
    mjt_static_for<0, PT>([&](auto tc) {
        constexpr int t = decltype(tc)::v;
        const int f = f0 + (wp * PT + t) * 32 + l32, n = f / (OH_ * OW_), k0 = kb * KT + wk * 32 + 4 * half;
        if (f >= total) return;
        const long long base = (long long)(n * K_ + k0) * (OH_ * OW_) + (f - n * (OH_ * OW_));
        mjt_static_for<0, 16>([&](auto ec) {
            constexpr int e = decltype(ec)::v, k = 8 * (e / 4) + e % 4;
#if Y_16
            ((unsigned short*)p.a[2])[base + k * (OH_ * OW_)] = mjt_narrow(acc[t][e]);
#else
            ((float*)p.a[2])[base + k * (OH_ * OW_)] = acc[t][e];
#endif
        });
    });
}
