// Matrix product on MFMA:  C[b][M][N] = sum_k A'[b][M][K] * B'[b][K][N]
// (reference: the broadcast * broadcast -> reduce.add pattern that
// python/jittor/src/opt/tuner/matmul_tuner.cc:16-104 relays to a library GEMM,
// python/jittor/extern/cuda/cublas/ops/cublas_matmul_op.cc:27-126; batched form
// cublas_batched_matmul_op.cc:63-85).  Row-major operands; A' is a, or a
// transposed when A_KCONT == 0 (memory [K][M]); B' is b, or b transposed when
// B_KCONT == 1 (memory [N][K]).  bfloat16 / float16 operands with exact products
// and float32 accumulation, or float32 throughout.
//
// Supplied by the host: IN (0 bfloat16, 1 float16, 2 float32), OUT (0 bfloat16 by
// truncation, 1 float16 rounded to nearest even, 2 float32), MI, NI (32x32 accumulator
// tiles per wave along m and n), A_KCONT, B_KCONT (the operand's memory has k innermost).
//
// Mapping.  A workgroup of four waves (2 x 2; SPLIT: eight) owns a TM x TN = 64 MI x 64 NI tile of C and
// walks K in stages of KS elements (eight 16-byte chunks per row: 64 for 16-bit operands,
// 32 for float32).  Both operand tiles of a stage sit in LDS with k innermost,
// [row][8 chunks + one chunk of padding] (144 bytes per row: 16-byte fragment reads of
// 16 neighbouring rows then do not meet in a bank), which is the order an MFMA operand
// wants: lane (row = lane % 32, half = lane / 32) of v_mfma_f32_32x32x16 reads the 8
// consecutive k of its row and half with one ds_read_b128.  An operand whose memory has k
// innermost is copied as it is (a lane moves 16 bytes; 8 lanes read one 128-byte line).
// The other kind (m or n innermost) is transposed on the way in registers: 8 lanes load
// 16 bytes of 8 consecutive k rows, exchange among themselves with three butterfly steps
// (4 lanes and two steps for float32) until each owns one column for the 8 (4) k, and
// write 16 bytes.  A stage's tiles are loaded into registers one or two stages ahead and move to the other LDS buffer piece by
// piece between the MFMAs of the current stage; its barrier and the first fragment reads of the next stage stand in front
// of the last MFMAs.  (With these one after the other at the end of each stage the matrix cores stood still for 570 of the
// 1700 cycles of a 64 x 64 float32 stage.  us before / now, in turn: float32 a b^T 2048 x 1024 x 1024 51 / 43,
// 2048^3 163 / 143, a^T b 1024 x 1024 x 2048 72 / 58; bfloat16 2048 x 2048 x 2048 32.5 / 23, 12544 x 256 x 1024 18.8 / 14.)
// SPLIT = 1 (float32): the float32 MFMAs, 140 TFLOP/s measured, bound the large products, and the bfloat16 ones run at 16 times their
// rate.  On its way to LDS every value becomes three bfloat16 parts (split.h, which has the reasoning and the error).  A
// workgroup whose sums are not all finite throws them away and runs the float32 loop.  Eight waves share a tile,
// two to a SIMD: one splits while the other's MFMAs run (a b^T 2048 x 1024 x 1024 on 128 x 64 tiles 36.1 us with four waves, 31.0 with
// eight; 4096 x 4096 x 2048 on 128 x 128 415 / 375).  What bounds it: splitting, 13 vector instructions for two values, takes as
// long as the MFMAs on 128 x 64 tiles, LDS carries 6 bytes for each value (without the writes 28.5 us, without the loads 24.8, with
// one MFMA of six 21); a third buffer changes nothing (33), nor does splitting by truncation (30.4) or by v_dot2 (31.2).
// float32 uses v_mfma_f32_32x32x2: a lane's 16-byte read holds 4 k of its row, which feed
// four MFMAs (lanes 32..63 read the next chunk, so that an MFMA sums k and k + 4 of a
// chunk pair; any pairing is right as long as both operands use the same one).
//
// CONV = 1 makes the kernel an implicit-GEMM convolution, the meta-op group of
// python/jittor/nn.py:1251-1262 that opt/tuner/conv_tuner.cc:233-240,365-373 relays for every float type:
// A = the weights [K_][C_*R_*S_] (rows padded to 16 bytes by the host), B'[k = (c, r, s)][j = (image, oh, ow)] =
// x[image][c][oh*SH-PH+r*DH][ow*SW-PW+s*DW] (0 outside the image) is never written to memory -- the B tile of a
// stage is gathered from x element by element on its way to LDS (a float32 MFMA runs at a sixteenth of the 16-bit
// rate, so the gather's address arithmetic hides behind it; with 16-bit operands the gather is what bounds the
// kernel, which then serves the shapes the MFMA convolution kernel does not take) -- and C[k][j] is stored as
// y[image][k][oh][ow].
// Geometry comes as C_, H_, W_, K_, R_, S_, OH_, OW_, SH, SW, PH, PW, DH, DW; N = images * OH_ * OW_.
//
// CONV = 2 makes it the weight gradient of that convolution (opt/tuner/conv_tuner.cc:375-397):
//   dw[k][(c, r, s)] = sum over q = (image, oh, ow) of dy[image][k][oh][ow] * x[image][c][oh*SH-PH+r*DH][ow*SW-PW+s*DW]
// A = dy with rows k, B' = the shifted planes of x with columns (c, r, s), both with the summed index q innermost, gathered on their
// way to LDS: a lane owns one chunk of EPC pixels per stage and works out their image, row and column once for all rows and
// columns it loads; dy is loaded in the widest pieces that a plane consists of, as is x
// for taps of 1 x 1 without stride and padding; otherwise x is loaded by elements.  The sum over q is cut into slices of a[9] stages; the slices' float32 partial
// results are added up by a reduce launch.  Before, the shifted planes were written to memory, multiplied image by image
// and the images' results added (float32 32 x 3 x 224 x 224, 7x7 stride 2 -> 64: 110 + 337 + 9 us; 116 here).
//
// Rows of A' and columns of B' beyond M and N are read from the last valid row (their
// results are not stored); k beyond K is zeroed in both operands.  Leading dimensions are
// multiples of 16 bytes and the operand pointers 16-byte aligned (the host sends
// everything else to the plain kernel below).

#if IN == 2
typedef float TIN;
#define EPC 4                    // elements per 16-byte chunk
#else
typedef unsigned short TIN;
#define EPC 8
#endif
#define KC 8                     // chunks per row and stage
#define KS (KC * EPC)            // k per stage
#define TM (64 * MI)
#define TN (64 * NI)
#define ROWB 144                 // bytes per LDS row: 8 chunks + 1 of padding
#ifndef SPLIT
#define SPLIT 0                  // 1: float32 products from bfloat16 parts (below)
#endif
// Waves: WM x WN, of FI x FJ accumulator tiles each.
#if SPLIT
#define SPLIT_ROWB 208           // of a float32 row as three rows of bfloat16: 3 x 64 bytes + 16 of padding
#define WM (MI >= NI ? 4 : 2)
#define WN (8 / WM)
#else
#define SPLIT_ROWB ROWB
#define WM 2
#define WN 2
#endif
#define NTHR (64 * WM * WN)
#define FI (TM / 32 / WM)
#define FJ (TN / 32 / WN)
#ifndef CONV
#define CONV 0
#endif
#ifndef SLICED
#define SLICED 0                 // 1: workgroup (tile, slice) sums stages slice * a[9] .. of K into its own float32 C (or y), a[11] apart
#endif
// A convolution's sum is known here, and images have few channels: a single stage takes one buffer, so that eight workgroups share a
// compute unit instead of four, two stages one register set, and the loop of whole stages is left out where it would not be entered.
// (us with the general form / this: bfloat16 32 x 3 x 224 x 224 3x3 stride 2 -> 32 43.3 / 30.5, 32 x 3 x 112 x 112 7x7 stride 2 -> 64
// 28.9 / 23.7; float16 43 x 1 x 56 x 56 5x5 -> 16 16.8 / 13.6, 12 x 31 x 14 x 14 2x2 -> 224 10.7 / 10.2, 16 x 100 x 9 x 9 3x3 stride 2 -> 70
// 25.8 / 21.3; float32 32 x 3 x 64 x 64 3x3 -> 96 27.0 / 23.6, 64 x 64 x 56 x 56 3x3 -> 64 177 / 174.)
#if CONV == 1
#define STAGES ((C_ * R_ * S_ + KS - 1) / KS)
#else
#define STAGES 0
#endif
#ifndef NBUF
#define NBUF (CONV == 1 && STAGES == 1 ? 1 : 2)      // staging buffers: 2, or 1 for a product of a single stage (K <= KS)
#endif

typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
#if IN == 0
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)
#elif IN == 1
typedef _Float16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0)
#endif

template <int V> struct mjt_ic { static constexpr int v = V; };
#ifndef EPI
#define EPI 0
#define EPI_WORDS 0
#endif
struct Params { void* a[12 + EPI_WORDS]; };
// a[0] A  a[1] B  a[2] C  a[3] M (upper half: matrices of the batch)  a[4] N  a[5] K  a[6] lda  a[7] ldb  a[8] ldc (elements)
// a[9] batch stride of A  a[10] of B  a[11] of C (elements)

__device__ __forceinline__ unsigned mjt_dpp_xor1(unsigned v) { return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ unsigned mjt_dpp_xor2(unsigned v) { return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true); }
__device__ __forceinline__ unsigned mjt_dpp_xor4(unsigned v) {   // mirror of each group of 8 lanes, then a reversal inside each quad
    return (unsigned)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
}

// 8 lanes hold 8 rows (k) x 8 columns of 16-bit values, lane r = row r with d[j] = columns 2j, 2j+1.
// Returns column r for the 8 rows: d'[j] = rows 2j, 2j+1.
__device__ __forceinline__ mjt_u32x4v mjt_transpose8x8_b16(mjt_u32x4v d, int lane) {
    const bool b2 = lane & 4, b1 = lane & 2, b0 = lane & 1;
    const unsigned sel_t = b0 ? 0x05040100u : 0x07060302u;
    const unsigned sel_a = b0 ? 0x03020504u : 0x05040100u;
    const unsigned sel_b = b0 ? 0x03020706u : 0x07060100u;
    const unsigned g0 = mjt_dpp_xor4(b2 ? d[0] : d[2]), g1 = mjt_dpp_xor4(b2 ? d[1] : d[3]);
    const unsigned a0 = b2 ? g0 : d[0], a1 = b2 ? g1 : d[1];
    const unsigned a2 = b2 ? d[2] : g0, a3 = b2 ? d[3] : g1;
    const unsigned h0 = mjt_dpp_xor2(b1 ? a0 : a1), h1 = mjt_dpp_xor2(b1 ? a2 : a3);
    const unsigned c0 = b1 ? h0 : a0, c1 = b1 ? a1 : h0;
    const unsigned c2 = b1 ? h1 : a2, c3 = b1 ? a3 : h1;
    const unsigned s0 = mjt_dpp_xor1(__builtin_amdgcn_perm(c1, c0, sel_t)), s1 = mjt_dpp_xor1(__builtin_amdgcn_perm(c3, c2, sel_t));
    mjt_u32x4v f;
    f[0] = __builtin_amdgcn_perm(s0, c0, sel_a);
    f[1] = __builtin_amdgcn_perm(s0, c1, sel_b);
    f[2] = __builtin_amdgcn_perm(s1, c2, sel_a);
    f[3] = __builtin_amdgcn_perm(s1, c3, sel_b);
    return f;
}
// 4 lanes hold 4 rows x 4 columns of 32-bit values, lane r = row r.  Returns column r for the 4 rows.
__device__ __forceinline__ mjt_u32x4v mjt_transpose4x4_b32(mjt_u32x4v v, int lane) {
    const bool b1 = lane & 2, b0 = lane & 1;
    const unsigned g0 = mjt_dpp_xor1(b0 ? v[0] : v[1]), g1 = mjt_dpp_xor1(b0 ? v[2] : v[3]);
    const unsigned a0 = b0 ? g0 : v[0], a1 = b0 ? v[1] : g0;
    const unsigned a2 = b0 ? g1 : v[2], a3 = b0 ? v[3] : g1;
    const unsigned h0 = mjt_dpp_xor2(b1 ? a0 : a2), h1 = mjt_dpp_xor2(b1 ? a1 : a3);
    mjt_u32x4v y;
    y[0] = b1 ? h0 : a0;
    y[1] = b1 ? h1 : a1;
    y[2] = b1 ? a2 : h0;
    y[3] = b1 ? a3 : h1;
    return y;
}

#if SPLIT
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
typedef unsigned mjt_u32x2v __attribute__((ext_vector_type(2)));
#define MJT_MFMA16(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)
#endif
// One 16-byte chunk on its way to LDS.  SP: as its three bfloat16 parts.
template <bool SP> __device__ __forceinline__ void mjt_put(unsigned char* lds, int row, int kc, mjt_u32x4v v) {
#if SPLIT
    if constexpr (SP) {
        unsigned char* const at = lds + row * SPLIT_ROWB + kc * 8;
        unsigned h[2], m[2], l[2];
        mjt_split(v[0], v[1], h[0], m[0], l[0]);
        mjt_split(v[2], v[3], h[1], m[1], l[1]);
        *(mjt_u32x2v*)at = (mjt_u32x2v){h[0], h[1]};
        *(mjt_u32x2v*)(at + 64) = (mjt_u32x2v){m[0], m[1]};
        *(mjt_u32x2v*)(at + 128) = (mjt_u32x2v){l[0], l[1]};
        return;
    }
#endif
    *(mjt_u32x4v*)(lds + row * ROWB + kc * 16) = v;
}

template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

// One operand tile of a stage on its way from memory to LDS.  ROWS = tile rows (m or n), KCONT = memory has k
// innermost.  p = first element of the operand (of this batch), ld = leading dimension in elements, r0 = first
// tile row, rmax = rows of the operand, k0 = first k of the stage, K = total k.
// A tile moves in PER pieces, one 16-byte move per thread each.  fetch() only issues piece I's load (unconditional: nothing in it
// looks at a loaded value, so no wait is needed before the MFMAs that follow); commit() zeroes what lies beyond K, transposes
// and writes to LDS.  FULL: the stage does not reach beyond K.
template <int ROWS, bool KCONT> struct mjt_stager {
    static constexpr int PER = ROWS * KC / NTHR;          // 16-byte moves per thread
    mjt_u32x4v reg[PER];

    template <int I, bool FULL> __device__ __forceinline__ void fetch(const TIN* __restrict__ p, long long ld, int r0, int rmax, int k0, int K, int tid) {
        if constexpr (KCONT) {
            // chunk c = tid + I * NTHR: row c / KC, k-chunk c % KC (8 consecutive lanes read one 128-byte line)
            const int c = tid + I * NTHR;
            int row = r0 + c / KC;
            row = row < rmax ? row : rmax - 1;
            const int k = k0 + (c % KC) * EPC;
            const int kk = FULL || k < K ? k : 0;         // a chunk past the end reads chunk 0 and is zeroed in commit
            reg[I] = *(const mjt_u32x4v*)(p + (long long)row * ld + kk);
        } else {
            // blocks of EPC k-rows x EPC columns: EPC lanes each load 16 bytes (EPC columns) of one k-row.
            // Block b = tid / EPC + I * (NTHR / EPC): column group b % (ROWS / EPC), k-chunk b / (ROWS / EPC);
            // the blocks of a wave are neighbouring column groups, so a k-row's loads of a wave are contiguous.
            const int b = tid / EPC + I * (NTHR / EPC);
            const int cg = b % (ROWS / EPC), kc = b / (ROWS / EPC);
            int col = r0 + cg * EPC;
            col = col < rmax ? col : ((rmax - 1) / EPC) * EPC;      // a group outside the operand reads the last one (ld is a multiple of EPC: a group never leaves its row)
            const int k = k0 + kc * EPC + tid % EPC;
            const int kk = FULL || k < K ? k : 0;
            reg[I] = *(const mjt_u32x4v*)(p + (long long)kk * ld + col);
        }
    }
    template <int I, bool FULL, bool SP> __device__ __forceinline__ void commit(unsigned char* lds, int k0, int K, int tid) const {
        mjt_u32x4v v = reg[I];
        int row, kc;
        if constexpr (KCONT) {
            const int c = tid + I * NTHR;
            row = c / KC;
            kc = c % KC;
            if constexpr (!FULL) {
                const int valid = K - (k0 + kc * EPC);    // elements of this chunk that exist
#if IN == 2
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = e < valid ? v[e] : 0u;
#else
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = 2 * e + 1 < valid ? v[e] : 2 * e < valid ? (v[e] & 0xffffu) : 0u;
#endif
            }
        } else {
            const int b = tid / EPC + I * (NTHR / EPC);
            row = (b % (ROWS / EPC)) * EPC + tid % EPC;
            kc = b / (ROWS / EPC);
            if constexpr (!FULL) {
                if (k0 + kc * EPC + tid % EPC >= K) v = (mjt_u32x4v)(0u);
            }
#if IN == 2
            v = mjt_transpose4x4_b32(v, tid);
#else
            v = mjt_transpose8x8_b16(v, tid);
#endif
        }
        mjt_put<SP>(lds, row, kc, v);
    }
};

#if CONV
constexpr int ESZ = (int)sizeof(TIN);
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros
__device__ __forceinline__ unsigned mjt_wg_load(__amdgpu_buffer_rsrc_t d, unsigned off) {
#if IN == 2
    return __builtin_amdgcn_raw_buffer_load_b32(d, (int)off, 0, 0);
#else
    return (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(d, (int)off, 0, 0);
#endif
}
__device__ __forceinline__ mjt_u32x4v mjt_wg_pack(const unsigned (&v)[EPC]) {
    mjt_u32x4v r;
#if IN == 2
    r[0] = v[0]; r[1] = v[1]; r[2] = v[2]; r[3] = v[3];
#else
    r[0] = v[0] | (v[1] << 16); r[1] = v[2] | (v[3] << 16); r[2] = v[4] | (v[5] << 16); r[3] = v[6] | (v[7] << 16);
#endif
    return r;
}
#endif

#if CONV == 1
// The B tile of a stage of the implicit-GEMM convolution.  Same blocks as mjt_stager<TN, false>: EPC lanes hold EPC
// k-rows x EPC columns (4 x 4 float32 values, 8 x 8 16-bit ones), lane tid % EPC the k-row.  What depends on a column
// alone (its image and pixel) is worked out once per workgroup (mjt_conv_cols): base = element offset of
// x[image][0][oh*SH-PH][ow*SW-PW], hw = that row and column, both biased by 0x4000, in one word (0 for a column past
// N: every tap of it then fails the range check).
struct mjt_conv_cols {
    static constexpr int PER = TN * KC / NTHR;
    int base[PER][EPC];
    unsigned hw[PER][EPC];
    // (compile-time loop indices throughout: with run-time ones the compiler keeps these arrays in scratch memory
    // once the loops are too long for it to unroll them itself)
    __device__ __forceinline__ void init(int n0, int N, int img0, int tid) {
        mjt_static_for<0, PER * EPC>([&](auto ic) {
            constexpr int i = decltype(ic)::v / EPC, e = decltype(ic)::v % EPC;
            const int b = tid / EPC + i * (NTHR / EPC);
            const int j = n0 + (b % (TN / EPC)) * EPC + e;
            const int img = j / (OH_ * OW_), px = j - img * (OH_ * OW_);
            const int oh = px / OW_, ow = px - oh * OW_;
            const int ih = oh * SH - PH, iw = ow * SW - PW;
            base[i][e] = j < N ? ((img - img0) * C_ * H_ + ih) * W_ + iw : 0;
            hw[i][e] = j < N ? ((unsigned)(ih + 0x4000) << 16) | (unsigned)(iw + 0x4000) : 0u;
        });
    }
};
// XBUF 1: x is read through a buffer descriptor that begins at the tile's first image (the host promises that a tile's images
// are less than 2 GB), unconditionally: a tap outside the image gets an offset past the buffer's end and reads zero, so nothing
// has to be looked at before the value is written to LDS.  XBUF 0: plain loads, zeroed afterwards, which wait for them.
struct mjt_conv_stager {
    static constexpr int PER = TN * KC / NTHR;
    static constexpr int RS = R_ * S_, CRS = C_ * R_ * S_;
    unsigned v[PER][EPC];

    template <int I> __device__ __forceinline__ void fetch(const TIN* __restrict__ x, __amdgpu_buffer_rsrc_t d, const mjt_conv_cols& cols, int k0, int tid) {
        const int b = tid / EPC + I * (NTHR / EPC);
        const int k = k0 + (b / (TN / EPC)) * EPC + tid % EPC;
        const bool kvalid = k < CRS;
        const int kk = kvalid ? k : 0;
        const int c = kk / RS, rs = kk - c * RS;
        const int r = rs / S_, t = rs - r * S_;
        const int koff = (c * H_ + r * DH) * W_ + t * DW;
        const unsigned dhw = ((unsigned)(r * DH) << 16) | (unsigned)(t * DW);
        mjt_static_for<0, EPC>([&](auto ec) {
            constexpr int e = decltype(ec)::v;
            const unsigned q = cols.hw[I][e] + dhw;
            const bool ok = kvalid && (q >> 16) - 0x4000u < (unsigned)H_ && (q & 0xffffu) - 0x4000u < (unsigned)W_;
#if XBUF
            v[I][e] = mjt_wg_load(d, ok ? (unsigned)(cols.base[I][e] + koff) * ESZ : MJT_NONE);
#else
#if IN == 2
            const unsigned ld = __float_as_uint(x[ok ? cols.base[I][e] + koff : 0]);
#else
            const unsigned ld = x[ok ? cols.base[I][e] + koff : 0];
#endif
            v[I][e] = ok ? ld : 0u;
#endif
        });
    }
    template <int I, bool SP> __device__ __forceinline__ void commit(unsigned char* lds, int tid) const {
        const int b = tid / EPC + I * (NTHR / EPC);
        const int row = (b % (TN / EPC)) * EPC + tid % EPC, kc = b / (TN / EPC);
#if IN == 2
        mjt_put<SP>(lds, row, kc, mjt_transpose4x4_b32(mjt_wg_pack(v[I]), tid));
#else
        mjt_put<SP>(lds, row, kc, mjt_transpose8x8_b16(mjt_wg_pack(v[I]), tid));
#endif
    }
};
#endif

#if CONV == 2
constexpr int P_ = OH_ * OW_;
// The pixels of the lane's chunk of a stage (chunk tid % KC), the same for all rows and columns that it loads.  All loads go
// through buffer descriptors, unconditionally: what lies outside the image or past the sum gets an offset past the buffer's
// end and reads zero, so nothing has to be looked at before it is written to LDS.
constexpr int PU = P_ % EPC == 0 ? EPC : P_ % 4 == 0 ? 4 : P_ % 2 == 0 ? 2 : 1;     // pixels of a plane that one load takes
constexpr int NL = EPC / PU;
#define XPLANE (R_ * S_ == 1 && SH == 1 && SW == 1 && PH == 0 && PW == 0)             /* x is read in planes, as dy is */
struct mjt_wg_chunk {
    unsigned dy[NL];                 // byte offsets of dy[image][0][pixel], or MJT_NONE
    unsigned x[EPC];                 // byte offset of x[image][0][oh*SH-PH][ow*SW-PW] (may wrap below zero); XPLANE: as dy
    unsigned hw[EPC];                // that row and column, both biased by 0x4000; 0 for a pixel past the sum
    __device__ __forceinline__ void at(int k0, int K, int tid) {
        const int q = k0 + (tid % KC) * EPC;
        mjt_static_for<0, EPC>([&](auto ec) {
            constexpr int e = decltype(ec)::v;
            constexpr bool decode = OW_ % EPC != 0 || e == 0;          // a row of outputs is whole chunks: neighbours of the first
            if constexpr (e % PU == 0) {
                const int qe = q + e, img = qe / P_, px = qe - img * P_;
                dy[e / PU] = qe < K ? (unsigned)(img * (K_ * P_) + px) * ESZ : MJT_NONE;
                if constexpr (XPLANE) x[e / PU] = qe < K ? (unsigned)(img * (C_ * P_) + px) * ESZ : MJT_NONE;
            }
            if constexpr (!XPLANE && decode) {
                const int qe = q + e;
                const int img = qe / P_, px = qe - img * P_;
                const int oh = px / OW_, ow = px - oh * OW_;
                const int ih = oh * SH - PH, iw = ow * SW - PW;
                x[e] = (unsigned)((img * C_ * H_ + ih) * W_ + iw) * ESZ;
                hw[e] = qe < K ? ((unsigned)(ih + 0x4000) << 16) | (unsigned)(iw + 0x4000) : 0u;
            } else if constexpr (!XPLANE) {
                x[e] = x[0] + e * SW * ESZ;
                hw[e] = hw[0] + e * SW;                                // (0 + e * SW stays far below the bias)
            }
        });
    }
};
// An operand read in planes: the lane's chunk of PER channels, NL loads of PU pixels each.  A load's pixels lie in one plane (PU
// divides the planes) at an address that is a multiple of its size.
template <int ROWS> struct mjt_wg_plane {
    static constexpr int PER = ROWS * KC / NTHR;
    mjt_u32x4v reg[PER];
    unsigned row[PER];               // byte offset of the lane's channels inside an image
    __device__ __forceinline__ void init(int r0, int rmax, int tid) {
        mjt_static_for<0, PER>([&](auto ic) {
            const int r = r0 + tid / KC + decltype(ic)::v * (NTHR / KC);
            row[decltype(ic)::v] = (unsigned)((r < rmax ? r : rmax - 1) * P_) * ESZ;
        });
    }
    template <int I> __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t d, const unsigned* at) {
        if constexpr (PU * ESZ == 2) {
            unsigned v[EPC];
            mjt_static_for<0, EPC>([&](auto ec) { constexpr int e = decltype(ec)::v; v[e] = mjt_wg_load(d, (at[e] + row[I]) | (at[e] & MJT_NONE)); });
            reg[I] = mjt_wg_pack(v);
        } else {
            mjt_static_for<0, NL>([&](auto gc) {
                constexpr int g = decltype(gc)::v;
                const int off = (int)((at[g] + row[I]) | (at[g] & MJT_NONE));
                if constexpr (PU * ESZ == 16) {
                    reg[I] = __builtin_amdgcn_raw_buffer_load_b128(d, off, 0, 0);
                } else if constexpr (PU * ESZ == 8) {
                    const auto two = __builtin_amdgcn_raw_buffer_load_b64(d, off, 0, 0);
                    reg[I][2 * g] = two[0];
                    reg[I][2 * g + 1] = two[1];
                } else {
                    reg[I][g] = __builtin_amdgcn_raw_buffer_load_b32(d, off, 0, 0);
                }
            });
        }
    }
    template <int I, bool SP> __device__ __forceinline__ void commit(unsigned char* lds, int tid) const {
        mjt_put<SP>(lds, tid / KC + I * (NTHR / KC), tid % KC, reg[I]);
    }
};
typedef mjt_wg_plane<TM> mjt_wg_dy;
#if XPLANE
typedef mjt_wg_plane<TN> mjt_wg_x;
#else
struct mjt_wg_x {
    static constexpr int PER = TN * KC / NTHR;
    unsigned v[PER][EPC];
    unsigned koff[PER], dhw[PER];    // of the lane's columns (c, r, s): byte offset inside an image, row and column shift
    __device__ __forceinline__ void init(int n0, int N, int tid) {
        mjt_static_for<0, PER>([&](auto ic) {
            constexpr int i = decltype(ic)::v;
            int k = n0 + tid / KC + i * (NTHR / KC);
            k = k < N ? k : N - 1;
            const int c = k / (R_ * S_), rs = k - c * (R_ * S_), r = rs / S_, t = rs - r * S_;
            koff[i] = (unsigned)((c * H_ + r * DH) * W_ + t * DW) * ESZ;
            dhw[i] = ((unsigned)(r * DH) << 16) | (unsigned)(t * DW);
        });
    }
    template <int I> __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t d, const mjt_wg_chunk& ch) {
        mjt_static_for<0, EPC>([&](auto ec) {
            constexpr int e = decltype(ec)::v;
            const unsigned h = ch.hw[e] + dhw[I];
            const bool in = (h >> 16) - 0x4000u < (unsigned)H_ && (h & 0xffffu) - 0x4000u < (unsigned)W_;
            v[I][e] = mjt_wg_load(d, in ? ch.x[e] + koff[I] : MJT_NONE);
        });
    }
    template <int I, bool SP> __device__ __forceinline__ void commit(unsigned char* lds, int tid) const {
        mjt_put<SP>(lds, tid / KC + I * (NTHR / KC), tid % KC, mjt_wg_pack(v[I]));
    }
};
#endif
#endif

extern "C" __global__ __launch_bounds__(NTHR) void ENTRY(Params p) {
    const int M = (int)(long long)p.a[3], N = (int)(long long)p.a[4];
#if CONV == 1
    constexpr int K = C_ * R_ * S_;
#else
    const int K = (int)(long long)p.a[5];
#endif
    const long long lda = (long long)p.a[6], ldb = (long long)p.a[7], ldc = (long long)p.a[8];
#if CONV == 2
    const TIN* __restrict__ A = (const TIN*)p.a[0];
    const TIN* __restrict__ B = (const TIN*)p.a[1];
    const __amdgpu_buffer_rsrc_t dy_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)(K * K_) * ESZ, 0x00020000);
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, (int)(long long)p.a[10], 0x00020000);   // a[10]: bytes of x
#endif
    // Workgroups go round-robin over the 8 XCDs: every XCD takes a run of neighbouring (matrix of the batch or slice of the sum, tile)
    // pairs, so that the tiles that read the same operands run next to each other and share an L2 (weight gradient 64 x 64 x 56 x 56,
    // 3x3 -> 64: 269 us with the tiles dealt out one by one, 162 with runs), and all XCDs have work however few tiles a matrix has
    // (us, a b^T, each matrix on the same first XCDs / so: float32 256 x 64 x 64 x 64 20.4 / 10.6, 512 x 32 x 128 x 64 66 / 31;
    // bfloat16 the same 8.7 / 7.2, 18.1 / 10.2).  (Before, each matrix had a row of the
    // grid to itself, rounded up to eight workgroups, and which compute units the empty ones kept from work was chance: float32
    // 64 x 256 x 196 x 1024 on 128 x 128 tiles, four a matrix, 92 / 56; 256 x 64 x 64 x 64 9.2 / 5.2; bfloat16 the same 7.1 / 4.0,
    // 100 x 200 x 200 x 128 22.2 / 12.2.)
    const int tiles_m = (M + TM - 1) / TM, tiles_n = (N + TN - 1) / TN, tiles = tiles_m * tiles_n;
#if CONV == 2 || SLICED
    const int per_slice = (int)(long long)p.a[9], pairs = ((K + KS - 1) / KS + per_slice - 1) / per_slice * tiles;
#else
    const int pairs = (CONV ? 1 : (int)((long long)p.a[3] >> 32)) * tiles;
#endif
    const int run = (pairs + 7) / 8, pair = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= run || pair >= pairs) return;
    const int outer = pair / tiles, L = pair - outer * tiles;        // slice or matrix; tile
#if CONV == 2 || SLICED
    const int first_stage = outer * per_slice;
#endif
#if CONV != 2
#if SLICED
    const TIN* __restrict__ A = (const TIN*)p.a[0];
    const TIN* __restrict__ B = (const TIN*)p.a[1];
#else
    const TIN* __restrict__ A = (const TIN*)p.a[0] + (long long)outer * (long long)p.a[9];
    const TIN* __restrict__ B = (const TIN*)p.a[1] + (long long)outer * (long long)p.a[10];
#endif
#endif
    // NBUF 1: the host promises K <= KS, a single stage -- one staging buffer, so twice as many workgroups fit a compute unit
    __shared__ __attribute__((aligned(16))) unsigned char lds[NBUF][(TM + TN) * SPLIT_ROWB];
#if SPLIT
    __shared__ int in_float32;                                 // some sum is not finite
    if (threadIdx.x == 0) in_float32 = 0;
    __syncthreads();
#endif

    // Tile order inside a matrix: panels of 4 tile rows, inside a panel column by column, so that a run of tiles is compact and
    // finds the operand rows and columns it shares in its XCD's L2.
    int tm, tn;
    {
        const int panel = L / (4 * tiles_n);
        const int rows_here = tiles_m - panel * 4 < 4 ? tiles_m - panel * 4 : 4;
        const int within = L - panel * 4 * tiles_n;
        tn = within / rows_here;
        tm = panel * 4 + within - tn * rows_here;
    }
    const int m0 = tm * TM, n0 = tn * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;

    // The operand tiles of a stage are asked for NSET stages ahead: one stage of MFMAs is shorter than a trip to memory on tiles
    // up to 128 x 128 of 16-bit and on all float32 tiles that are run (us with one set / two / three, float32: 1024 x 1024 x 2048
    // on 64 x 64 57.7 / 55.4 / 57.1, 2048^3 on 128 x 128 133 / 127 / -).  Larger tiles have no registers to spare.
    // The gathering operands hold more registers: two sets on 64 x 64 tiles only (64 x 512 x 7 x 7 3x3 -> 512 247 / 218;
    // 64 x 128 x 28 x 28 3x3 -> 128 on 128 x 128 186 / 194).
    auto multiply = [&](auto spc) -> bool {
    constexpr bool SP = decltype(spc)::v != 0;
    constexpr int RB = SP ? SPLIT_ROWB : ROWB, BUFB = (TM + TN) * RB;
    constexpr int NSET = NBUF > 1 && STAGES != 2 && MI * NI <= (CONV ? 1 : 4) ? 2 : 1;
#if CONV == 2
    const int all_stages = (K + KS - 1) / KS;
    const int nstages = all_stages - first_stage < per_slice ? all_stages - first_stage : per_slice;
    mjt_wg_dy sa[NSET];
    mjt_wg_x sb[NSET];
    mjt_static_for<0, NSET>([&](auto tc) { sa[decltype(tc)::v].init(m0, M, tid); sb[decltype(tc)::v].init(n0, N, tid); });
    mjt_wg_chunk ch;
    constexpr int PA = mjt_wg_dy::PER, PIECES = PA + mjt_wg_x::PER;
    auto fetch = [&](auto ic, auto setc, auto, int stage) {
        constexpr int I = decltype(ic)::v, SET = decltype(setc)::v;
        if constexpr (I == 0) ch.at((first_stage + stage) * KS, K, tid);
        if constexpr (I < PA) sa[SET].template fetch<I>(dy_rsrc, ch.dy);
#if XPLANE
        else sb[SET].template fetch<I - PA>(x_rsrc, ch.x);
#else
        else sb[SET].template fetch<I - PA>(x_rsrc, ch);
#endif
    };
    auto commit = [&](auto ic, auto setc, auto, int stage) {
        constexpr int I = decltype(ic)::v, SET = decltype(setc)::v;
        unsigned char* buf = &lds[0][0] + (stage & (NBUF - 1)) * BUFB;
        if constexpr (I < PA) sa[SET].template commit<I, SP>(buf, tid);
        else sb[SET].template commit<I - PA, SP>(buf + TM * RB, tid);
    };
#else
#if SLICED
    const int all_stages = (K + KS - 1) / KS;
    const int nstages = all_stages - first_stage < per_slice ? all_stages - first_stage : per_slice;
#else
    constexpr int first_stage = 0;
    const int nstages = NBUF == 1 ? 1 : (K + KS - 1) / KS;
#endif
    mjt_stager<TM, A_KCONT> sa[NSET];
    const int arows = M, brows = N;
#if CONV
    const int img0 = n0 / (OH_ * OW_);
    mjt_conv_cols cols;
    cols.init(n0, N, XBUF ? img0 : 0, tid);
    mjt_conv_stager sb[NSET];
    const long long x_bytes = ((long long)(N / (OH_ * OW_)) - img0) * (C_ * H_) * W_ * ESZ;
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(B + (long long)img0 * (C_ * H_) * W_), 0,
                                                                            (int)(x_bytes < 0x7fffffffll ? x_bytes : 0x7fffffffll), 0x00020000);
#else
    mjt_stager<TN, B_KCONT> sb[NSET];
#endif
    constexpr int PA = TM * KC / NTHR, PIECES = PA + TN * KC / NTHR;
    auto fetch = [&](auto ic, auto setc, auto fullc, int stage) {
        constexpr int I = decltype(ic)::v, SET = decltype(setc)::v;
        constexpr bool FULL = decltype(fullc)::v != 0;
        if constexpr (I < PA) sa[SET].template fetch<I, FULL>(A, lda, m0, arows, (first_stage + stage) * KS, K, tid);
#if CONV
        else sb[SET].template fetch<I - PA>(B, x_rsrc, cols, (first_stage + stage) * KS, tid);
#else
        else sb[SET].template fetch<I - PA, FULL>(B, ldb, n0, brows, (first_stage + stage) * KS, K, tid);
#endif
    };
    auto commit = [&](auto ic, auto setc, auto fullc, int stage) {
        constexpr int I = decltype(ic)::v, SET = decltype(setc)::v;
        constexpr bool FULL = decltype(fullc)::v != 0;
        unsigned char* buf = &lds[0][0] + (stage & (NBUF - 1)) * BUFB;
        if constexpr (I < PA) sa[SET].template commit<I, FULL, SP>(buf, (first_stage + stage) * KS, K, tid);
#if CONV
        else sb[SET].template commit<I - PA, SP>(buf + TM * RB, tid);
#else
        else sb[SET].template commit<I - PA, FULL, SP>(buf + TM * RB, (first_stage + stage) * KS, K, tid);
#endif
    };
#endif
    mjt_static_for<0, NSET>([&](auto tc) {
        if (decltype(tc)::v < nstages) mjt_static_for<0, PIECES>([&](auto ic) { fetch(ic, tc, mjt_ic<0>(), decltype(tc)::v); });
    });

    mjt_f32x16 acc[FI][FJ], low[SP ? FI : 1][SP ? FJ : 1];
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                acc[i][j][e] = 0.0f;
                if constexpr (SP) low[i][j][e] = 0.0f;
            }

    mjt_static_for<0, PIECES>([&](auto ic) { commit(ic, mjt_ic<0>(), mjt_ic<0>(), 0); });
    if (NSET < nstages) mjt_static_for<0, PIECES>([&](auto ic) { fetch(ic, mjt_ic<0>(), mjt_ic<0>(), NSET); });
    __syncthreads();

    // fragment addresses of this lane: row lane % 32 of its wave's tile rows, chunk lane / 32
    const int frow = lane & 31, fhalf = lane >> 5;
    const unsigned char* const la = &lds[0][0] + (wm * 32 * FI + frow) * RB + fhalf * 16;
    const unsigned char* const lb = &lds[0][0] + (TM + wn * 32 * FJ + frow) * RB + fhalf * 16;
    // a pair of chunks per step; the fragments of the next step, across the end of a stage too, are requested before the MFMAs of
    // this one (the scheduling barriers keep them there: the compiler would move every read next to its first use)
    constexpr int PARTS = SP ? 3 : 1, STEPS = SP ? KS / 16 : KC / 2;
    mjt_u32x4v fa[2][FI][PARTS], fb[2][FJ][PARTS];
    auto request = [&](auto ksc, auto setc, const int s) {
        constexpr int KSX = decltype(ksc)::v, SET = decltype(setc)::v;
        const int off = (s & (NBUF - 1)) * BUFB + KSX * 32;
        mjt_static_for<0, PARTS>([&](auto pc) {
            constexpr int part = decltype(pc)::v;
            mjt_static_for<0, FI>([&](auto ic) { fa[SET][decltype(ic)::v][part] = *(const mjt_u32x4v*)(la + off + part * 64 + decltype(ic)::v * 32 * RB); });
            mjt_static_for<0, FJ>([&](auto jc) { fb[SET][decltype(jc)::v][part] = *(const mjt_u32x4v*)(lb + off + part * 64 + decltype(jc)::v * 32 * RB); });
        });
    };
    request(mjt_ic<0>(), mjt_ic<0>(), 0);
    // Stage s: its tiles sit in LDS buffer s % NBUF, its first fragments are on their way, and the register sets hold the stages
    // s + 1 .. s + NSET.  Piece by piece between the MFMAs of all steps but the last, stage s + 1 goes to the other buffer, which
    // nobody has read since the barrier of stage s - 1, and its registers take stage s + 1 + NSET.  The barrier stands in front
    // of the last step's MFMAs (SP, two long steps: of the last half of them): every wave has then read the last fragments of this
    // stage and written the next one, whose first fragments arrive during these MFMAs.
    // FULL: stages s + 1 and s + 1 + NSET exist and do not reach beyond K -- no branches, so that the pieces' instructions can
    // stand between MFMAs.
    auto run_stage = [&](auto parc, auto fullc, const int s) {
        constexpr int PAR = decltype(parc)::v, SET = (PAR + 1) % NSET;
        constexpr bool FULL = decltype(fullc)::v != 0;
        mjt_static_for<0, STEPS>([&](auto ksc) {
            constexpr int ks = decltype(ksc)::v, cur = ks & 1, nxt = cur ^ 1;
            constexpr int EK = SP ? 6 : IN == 2 ? 4 : 1, PER_STEP = EK * FI * FJ;
            constexpr int BARRIER = SP ? PER_STEP * STEPS - PER_STEP / 2 : PER_STEP * (STEPS - 1), SLOTS = SP ? BARRIER * 3 / 4 : BARRIER - PER_STEP / 2;
            if constexpr (ks + 1 < STEPS) request(mjt_ic<ks + 1>(), mjt_ic<nxt>(), s);
            mjt_static_for<0, PER_STEP>([&](auto mc) {
                constexpr int m = decltype(mc)::v, e = m / (FI * FJ), i = m / FJ % FI, j = m % FJ, slot = ks * PER_STEP + m;
                if constexpr (slot == BARRIER) {
                    if (FULL || s + 1 < nstages) {
                        __syncthreads();
                        request(mjt_ic<0>(), mjt_ic<nxt>(), s + 1);
                    }
                }
                if constexpr (m == 0 || slot == BARRIER) __builtin_amdgcn_sched_barrier(0);
#if IN == 2
#if SPLIT
                if constexpr (SP) {
                    constexpr int pa = e == 0 ? 2 : e == 2 || e == 3 ? 1 : 0, pb = e == 1 ? 2 : e == 2 || e == 4 ? 1 : 0;
                    mjt_f32x16& sum = e == 5 ? acc[i][j] : low[i][j];
                    sum = MJT_MFMA16(__builtin_bit_cast(mjt_h8, fa[cur][i][pa]), __builtin_bit_cast(mjt_h8, fb[cur][j][pb]), sum);
                } else
#endif
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(fa[cur][i][0][e & 3]), __uint_as_float(fb[cur][j][0][e & 3]), acc[i][j], 0, 0, 0);
#else
                acc[i][j] = MJT_MFMA16(__builtin_bit_cast(mjt_h8, fa[cur][i][0]), __builtin_bit_cast(mjt_h8, fb[cur][j][0]), acc[i][j]);
#endif
                if constexpr (NBUF > 1 && slot < SLOTS) {
                    constexpr int first = PIECES * slot / SLOTS, last = PIECES * (slot + 1) / SLOTS;
                    if constexpr (FULL && last > first) {
                        __builtin_amdgcn_sched_barrier(0);
                        mjt_static_for<first, last>([&](auto ic) {
                            commit(ic, mjt_ic<SET>(), mjt_ic<1>(), s + 1);
                            fetch(ic, mjt_ic<SET>(), mjt_ic<1>(), s + 1 + NSET);
                        });
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            });
            if constexpr (!FULL && NBUF > 1 && ks == STEPS - 2) {
                if (s + 1 < nstages) {
                    mjt_static_for<0, PIECES>([&](auto ic) { commit(ic, mjt_ic<SET>(), mjt_ic<0>(), s + 1); });
                    if (s + 1 + NSET < nstages) mjt_static_for<0, PIECES>([&](auto ic) { fetch(ic, mjt_ic<SET>(), mjt_ic<0>(), s + 1 + NSET); });
                }
            }
        });
    };
    const int nstages_full = CONV == 2 ? nstages : K / KS - first_stage < nstages ? K / KS - first_stage : nstages;     // (the weight gradient's operands read zeros beyond K by themselves)
    int s0 = 0;
#if CONV == 1
    constexpr bool LONG = K / KS > 2 * NSET;
#else
    constexpr bool LONG = NBUF > 1;
#endif
    if constexpr (LONG)
#pragma unroll 1
        for (; s0 + 2 * NSET < nstages_full; s0 += NSET)
            mjt_static_for<0, NSET>([&](auto parc) { run_stage(parc, mjt_ic<1>(), s0 + decltype(parc)::v); });
#pragma unroll 1
    for (; s0 < nstages; s0 += NSET)
        mjt_static_for<0, NSET>([&](auto parc) {
            if (s0 + decltype(parc)::v < nstages) run_stage(parc, mjt_ic<0>(), s0 + decltype(parc)::v);
        });

#if SPLIT
    if constexpr (SP) {
        float z = 0.0f;                                        // not zero if any sum is not finite
#pragma unroll
        for (int i = 0; i < FI; i++)
#pragma unroll
            for (int j = 0; j < FJ; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    acc[i][j][e] += low[i][j][e];
                    z = __builtin_fmaf(acc[i][j][e], 0.0f, z);
                    acc[i][j][e] *= MJT_SPLIT_DOWN;
                }
        if (z != 0.0f) in_float32 = 1;
        __syncthreads();
        if (in_float32) return false;
    }
#endif

    // D of a 32x32 tile: lane holds column lane % 32, rows 8 * (e / 4) + 4 * (lane / 32) + e % 4
    const long long c0 = (long long)outer * (long long)p.a[11];
#pragma unroll
    for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++) {
            const int col = n0 + wn * 32 * FJ + j * 32 + (lane & 31);
#if CONV == 1
            const int img = col / (OH_ * OW_), px = col - img * (OH_ * OW_);      // y[img][row][px]
#endif
            auto row_of = [&](int e) { return m0 + wm * 32 * FI + i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e & 3); };
            auto place_of = [&](int row) {
#if CONV == 1
                return (SLICED ? c0 : 0) + ((long long)img * K_ + row) * (OH_ * OW_) + px;
#else
                return c0 + (long long)row * ldc + col;
#endif
            };
#if EPI
            // what the group reads of all sixteen places is asked for before the first is finished
            mjt_epi_in<1> read[16];
#pragma unroll
            for (int e = 0; e < 16; e++) mjt_epi_load(p, read[e], (MJT_EPI_INDEX)(row_of(e) < M && col < N ? place_of(row_of(e)) : 0));
#endif
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int row = row_of(e);
                if (row < M && col < N) {
                    const float v = acc[i][j][e];
                    const long long at = place_of(row);
#if EPI
                    mjt_epi_finish(p, read[e], (MJT_EPI_INDEX)at, {v});
#elif OUT == 2
                    ((float*)p.a[2])[at] = v;
#elif OUT == 0
                    ((unsigned short*)p.a[2])[at] = (unsigned short)(__float_as_uint(v) >> 16);     // truncation (type/fp16_compute.h:238-241)
#else
                    const _Float16 h = (_Float16)v;                        // nearest even (type/fp16_compute.h:147-198)
                    ((unsigned short*)p.a[2])[at] = __builtin_bit_cast(unsigned short, h);
#endif
                }
            }
        }
    return true;
    };
#if SPLIT
    if (multiply(mjt_ic<1>())) return;
    __syncthreads();
#endif
    multiply(mjt_ic<0>());
}
