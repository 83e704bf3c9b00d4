// Weight gradient of the meta-op convolution from windows that lie in LDS:
//   dW[k][c][r][s] = sum_{n,oh,ow} dy[n][k][oh][ow] * x[n][c][oh*SH-PH+r*DH][ow*SW-PW+s*DW]
// (python/jittor/nn.py:1251-1262 differentiated by ops/reduce_op.cc:339-362; opt/tuner/conv_tuner.cc:375-397 relays it) for bfloat16
// (IN_F16: float16) operands with exact products and float32 accumulation; taps outside the image contribute 0.
//
// What it replaces, the product over gathered operands (gemm_mfma.h, CONV 2), loads every element of x by itself, once for each
// tap: the loads bound it.  Here a workgroup copies RB output rows' worth of x (or IB whole images) of 64 input channels, and the same
// pixels of dy of 64 output channels, into LDS once and makes the operands of all R_ * S_ taps from there.
//
// Layout.  An output row is cut into pieces of 8 pixels, OW_ rounded up (what is beyond OW_ is zero in dy and cleared in x, so that
// infinities of x stay where they belong).  dy: [channel][row][piece].  x: [channel][row][column % SW][LP zeros, column / SW], so that the 8 pixels of a piece, shifted by tap s,
// are 8 consecutive values from a 16-byte aligned place, shifted by floor((s*DW-PW) / SW) values: a lane reads the 16 bytes
// there and the dwords beside them once for all taps of a row, and makes odd shifts with v_alignbit.  v_mfma_f32_32x32x16 takes
// two pieces; lane (l32, half) holds channel l32 and piece 2*step + half.
// Eight waves: 2 x 2 tiles of 32 x 32 channels, each with R_ * S_ accumulators, times two groups that take every other step; the
// groups' sums meet in LDS at the end, where a row of 64 * R_ * S_ results is contiguous as it is in memory.  Two LDS buffers: the next
// stage is asked for ahead of a stage's MFMAs and written between them.
// The sum over stages is cut into slices, whose float32 results a reduce launch adds up.
// What bounds it, 64 x 256 x 14 x 14 3x3 -> 256 (us; product over gathered operands / this, folds included: 59.9 / 39.4; 64 x 512 x 7 x 7 -> 512 91.8 / 42.9;
// 64 x 256 x 28 x 28 stride 2 -> 256 63.9 / 50.9): of the kernel's 32, the results of the slices (147 KB a workgroup, all at the same time)
// take 10, whatever the stores' cache policy and layout, the meeting of the groups 3, the first loads and the launch 5; the four stages 14, of which
// 8 are MFMAs.  Over many stages (256 images) a stage takes 3.5 us: without its LDS writes 2.5, without fragment reads 2.6, MFMAs alone 2.2.
//
// Supplied by the host: C_, H_, W_, K_, R_, S_, OH_, OW_, SH, SW (1 or 2), PH, PW, DH, DW, IN_F16, RB (output rows of a stage), IB (images of a
// stage; more than one only with RB == OH_).

#if IN_F16
typedef _Float16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_f16
#else
typedef __bf16 mjt_h8 __attribute__((ext_vector_type(8)));
#define MJT_MFMA __builtin_amdgcn_mfma_f32_32x32x16_bf16
#endif
typedef float mjt_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned mjt_u32x4v __attribute__((ext_vector_type(4)));
typedef unsigned mjt_u32x2v __attribute__((ext_vector_type(2)));
#define MJT_NONE 0x80000000u         // an offset beyond every buffer (they are smaller than 2 GB): the load delivers zeros

template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}

struct Params { void* a[8]; };       // x, dy, partial, images, stages, stages per slice, bytes of x, bytes of dy

constexpr int TAPS = R_ * S_;
constexpr bool WHOLE = RB == OH_;    // a stage is whole images: the rows around them stay zero in LDS
constexpr int SPI = (OH_ + RB - 1) / RB;                     // stages of an image (WHOLE: 1)
constexpr int NPW = (OW_ + 7) / 8, NP = RB * NPW, SPG = (NP + 3) / 4;     // pieces of a row, of a stage's image; steps of a group
constexpr int VD = OW_ - (NPW - 1) * 8;                      // pixels of a row's last piece
constexpr int floor_div(int a, int b) { return a >= 0 ? a / b : -((b - 1 - a) / b); }
constexpr int tap_shift(int s) { return floor_div(s * DW - PW, SW); }
constexpr int tap_phase(int s) { return s * DW - PW - tap_shift(s) * SW; }
constexpr int lo_of(int ph) {        // first and last dword, relative to the piece, that the taps of a column phase read
    int lo = 0;
    for (int s = 0; s < S_; s++) if (tap_phase(s) == ph && floor_div(tap_shift(s), 2) < lo) lo = floor_div(tap_shift(s), 2);
    return lo;
}
constexpr int hi_of(int ph) {
    int hi = 3;
    for (int s = 0; s < S_; s++) {
        const int h = floor_div(tap_shift(s), 2) + 3 + (tap_shift(s) & 1);
        if (tap_phase(s) == ph && h > hi) hi = h;
    }
    return hi;
}
constexpr bool phase_used(int ph) {
    for (int s = 0; s < S_; s++) if (tap_phase(s) == ph) return true;
    return false;
}
constexpr int LO = lo_of(0) < lo_of(SW - 1) ? lo_of(0) : lo_of(SW - 1), HI = hi_of(0) > hi_of(SW - 1) ? hi_of(0) : hi_of(SW - 1);
constexpr int LP = (-2 * LO + 7) / 8 * 8 < 8 ? 8 : (-2 * LO + 7) / 8 * 8;
constexpr int PWID = (W_ + SW - 1) / SW, NEED = NPW * 8 - 8 + 2 * HI + 2 - LP;       // (the next row's zeros serve as this one's)
constexpr int RW = (LP + (PWID > NEED ? PWID : NEED) + 7) / 8 * 8;
constexpr int XROWB = SW * RW * 2, XR = (RB - 1) * SH + (R_ - 1) * DH + 1;
constexpr int XCB = ((XR * XROWB + LP * 2) / 16 | 1) * 16;   // bytes of a channel: an odd number of 16-byte pieces, against bank conflicts
constexpr int DCB = (SPG * 4 | 1) * 16;
constexpr int XB = 64 * XCB, DB = 64 * DCB, BUFB = IB * (XB + DB);
constexpr int ZB = LP * 2 + SW * RW * 2 + HI * 4 + 16;       // zeros that pieces past the rows read
constexpr bool CHECKED = OH_ % RB != 0 || NP % 4 != 0 || IB > 1;
constexpr int OUTS = 64 * TAPS + 8, OUTB = 64 * OUTS * 4;    // floats of a row of results in LDS: rows 4 apart, which a wave writes together, lie 32 banks apart
constexpr int LDSB = 2 * BUFB + (CHECKED ? ZB : 0) > OUTB ? 2 * BUFB + (CHECKED ? ZB : 0) : OUTB;
static_assert(LDSB <= 160 * 1024, "LDS");
static_assert(LP * 2 + ((RB - 1) * SH + (R_ - 1) * DH) * XROWB + (SW - 1) * RW * 2 + (NPW - 1) * 16 + HI * 4 + 4 <= XCB, "reads stay inside a channel");
static_assert(NPW == 1 || NPW == 2 || NPW % 4 == 0, "the pieces of a step lie at the same distances in every step");

// where the pieces of a group's step lie from those of its first: 4 / NPW rows on, or 4 pieces of a row
constexpr int step_row(int t) { return NPW <= 2 ? t % SPG * (4 / NPW) : t % SPG * 4 / NPW; }
constexpr int step_col(int t) { return NPW <= 2 ? 0 : t % SPG * 4 % NPW; }

constexpr int unit_of(int n) { return n % 8 == 0 ? 8 : n % 4 == 0 ? 4 : n % 2 == 0 ? 2 : 1; }
// values of one load, of one piece of it that stays inside a row, loads of a channel and of each of its 8 threads
constexpr int GX = unit_of(WHOLE ? H_ * W_ : W_), LX = unit_of(W_) < GX ? unit_of(W_) : GX, UX = (WHOLE ? H_ : XR) * W_ / GX, NX = (UX + 7) / 8;
constexpr int GD = unit_of(WHOLE ? OH_ * OW_ : OW_), LD = unit_of(OW_) < GD ? unit_of(OW_) : GD, UD = RB * OW_ / GD, ND = (UD + 7) / 8;

template <int G> struct mjt_unit {   // G 16-bit values on their way to LDS
    unsigned d[G < 2 ? 1 : G / 2];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned off) {
        if constexpr (G == 1) {
            d[0] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
        } else if constexpr (G == 2) {
            d[0] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
        } else if constexpr (G == 4) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
            d[0] = v[0]; d[1] = v[1];
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
            d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
        }
    }
    // values FIRST .. FIRST + N of it, side by side
    template <int FIRST, int N> __device__ __forceinline__ void put(unsigned char* at) const {
        if constexpr (N == 1) *(unsigned short*)at = (unsigned short)(d[FIRST / 2] >> (FIRST % 2 * 16));
        else if constexpr (N == 2) *(unsigned*)at = d[FIRST / 2];
        else if constexpr (N == 4) *(mjt_u32x2v*)at = (mjt_u32x2v){d[FIRST / 2], d[FIRST / 2 + 1]};
        else *(mjt_u32x4v*)at = (mjt_u32x4v){d[0], d[1], d[2], d[3]};
    }
    // the even ones of values FIRST .. FIRST + N to `even`, the odd ones to `odd`
    template <int FIRST, int N> __device__ __forceinline__ void put_phases(unsigned char* even, unsigned char* odd) const {
        if constexpr (N == 2) {
            *(unsigned short*)even = (unsigned short)d[FIRST / 2];
            *(unsigned short*)odd = (unsigned short)(d[FIRST / 2] >> 16);
        } else if constexpr (N == 4) {
            *(unsigned*)even = __builtin_amdgcn_perm(d[FIRST / 2 + 1], d[FIRST / 2], 0x05040100u);
            *(unsigned*)odd = __builtin_amdgcn_perm(d[FIRST / 2 + 1], d[FIRST / 2], 0x07060302u);
        } else {
            *(mjt_u32x2v*)even = (mjt_u32x2v){__builtin_amdgcn_perm(d[1], d[0], 0x05040100u), __builtin_amdgcn_perm(d[3], d[2], 0x05040100u)};
            *(mjt_u32x2v*)odd = (mjt_u32x2v){__builtin_amdgcn_perm(d[1], d[0], 0x07060302u), __builtin_amdgcn_perm(d[3], d[2], 0x07060302u)};
        }
    }
};

extern "C" __global__ __launch_bounds__(512) void ENTRY(Params p) {
    const int N = (int)(long long)p.a[3], stages = (int)(long long)p.a[4], per_slice = (int)(long long)p.a[5];
    // every XCD takes a run of neighbouring (slice, block) pairs: the blocks of a slice read the same pixels and share an L2
    constexpr int KB = (K_ + 63) / 64, CB = (C_ + 63) / 64, BLOCKS = KB * CB;
    const int pairs = (stages + per_slice - 1) / per_slice * BLOCKS;
    const int run = (pairs + 7) / 8, pair = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= run || pair >= pairs) return;
    const int slice = pair / BLOCKS, block = pair - slice * BLOCKS;
    const int k0 = block % KB * 64, c0 = block / KB * 64;
    const int first = slice * per_slice, last = first + per_slice < stages ? first + per_slice : stages;

    __shared__ __attribute__((aligned(16))) unsigned char lds[LDSB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[0], 0, (int)(long long)p.a[6], 0x00020000);
    const __amdgpu_buffer_rsrc_t d_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.a[1], 0, (int)(long long)p.a[7], 0x00020000);

    // staging: 8 threads per channel
    const int ch = tid >> 3;
    const unsigned x_ch = (unsigned)((c0 + ch) * (H_ * W_)) * 2u, x_none = c0 + ch < C_ ? 0u : MJT_NONE;
    const unsigned d_ch = (unsigned)((k0 + ch) * (OH_ * OW_)) * 2u, d_none = k0 + ch < K_ ? 0u : MJT_NONE;
    mjt_unit<GX> ux[IB][NX];
    mjt_unit<GD> ud[IB][ND];
    auto fetch = [&](int st, unsigned never) {       // never: MJT_NONE for a stage that does not exist
        const int n = WHOLE ? st * IB : st / SPI, oh0 = WHOLE ? 0 : (st - n * SPI) * RB, xr0 = oh0 * SH - PH;
        unsigned j = tid & 7;
        asm volatile("" : "+v"(j));              // (worked out anew in every stage: kept, the offsets would push the accumulators out)
        mjt_static_for<0, IB>([&](auto bc) {
            constexpr int b = decltype(bc)::v;
            const unsigned gone = never | (n + b < N ? 0u : MJT_NONE);
            const unsigned xb = (unsigned)((n + b) * (C_ * H_ * W_) + (WHOLE ? 0 : xr0 * W_)) * 2u + x_ch, db = (unsigned)((n + b) * (K_ * OH_ * OW_) + oh0 * OW_) * 2u + d_ch;
            // (the thread's first load; a constant further lies each other one, beyond the buffer if there is nothing to load)
            const unsigned xno = (unsigned)((int)(gone | x_none) >> 31), dno = (unsigned)((int)(gone | d_none) >> 31);
            const unsigned x0 = ((xb + j * (GX * 2u)) & ~xno) | (xno & MJT_NONE), d0 = ((db + j * (GD * 2u)) & ~dno) | (dno & MJT_NONE);
            mjt_static_for<0, NX>([&](auto ic) {
                constexpr int i = decltype(ic)::v;
                const int u = 8 * i + 7 < UX || (int)j + 8 * i < UX ? 8 * i : UX - 1 - (int)j;      // (a thread past the end copies the last one again)
                unsigned out = 0;
                if constexpr (!WHOLE) out = (unsigned)(xr0 + (int)((unsigned)(j + u) / (unsigned)(W_ / GX))) >= (unsigned)H_ ? MJT_NONE : 0u;
                ux[b][i].load(x_rsrc, (x0 + u * (GX * 2)) | out);
            });
            mjt_static_for<0, ND>([&](auto ic) {
                constexpr int i = decltype(ic)::v;
                const int u = 8 * i + 7 < UD || (int)j + 8 * i < UD ? 8 * i : UD - 1 - (int)j;
                unsigned out = 0;
                if constexpr (!WHOLE && OH_ % RB != 0) out = oh0 + (int)((unsigned)(j + u) / (unsigned)(OW_ / GD)) >= OH_ ? MJT_NONE : 0u;
                ud[b][i].load(d_rsrc, (d0 + u * (GD * 2)) | out);
            });
        });
    };
    // Where the values from FIRST of unit j + 8 Q of a channel go (rows of WIDTH values, PITCH bytes apart): a constant from where the
    // thread's first unit goes, or a row further.  (In bytes of the phase the columns lie in; `row` is needed only where it is looked at.)
    auto place = [](auto gc, auto widthc, auto pitchc, auto stridec, auto countc, auto qc, auto firstc, unsigned j, unsigned& row) -> unsigned {
        constexpr unsigned G = decltype(gc)::v, WIDTH = decltype(widthc)::v, PITCH = decltype(pitchc)::v, STRIDE = decltype(stridec)::v, COUNT = decltype(countc)::v;
        constexpr unsigned Q = decltype(qc)::v, FIRST = decltype(firstc)::v;
        if constexpr (8 * Q + 7 < COUNT && STRIDE == 1) {
            const unsigned row0 = j * G / WIDTH, col0 = j * G - row0 * WIDTH;
            constexpr unsigned e = 8 * Q * G + FIRST, er = e / WIDTH, ec = e - er * WIDTH;
            const bool wraps = col0 >= WIDTH - ec;
            row = row0 + er + (wraps ? 1 : 0);
            return row0 * PITCH + col0 * 2 + (wraps ? (er + 1) * PITCH + ec * 2 - WIDTH * 2 : er * PITCH + ec * 2);
        } else {
            const unsigned u = j + 8 * Q < COUNT ? j + 8 * Q : COUNT - 1, e = u * G + FIRST, col = e % WIDTH;
            row = e / WIDTH;
            return row * PITCH + (STRIDE == 1 ? col * 2 : col / STRIDE * 2 + col % STRIDE * (RW * 2));
        }
    };
    constexpr int PIECES = IB * (NX + ND);
    auto commit = [&](auto pc, int st, unsigned j) {
        constexpr int P = decltype(pc)::v, b = P / (NX + ND), q = P % (NX + ND);
        unsigned char* const buf = lds + (st & 1) * BUFB + b * (XB + DB);
        if constexpr (q < NX) {
            mjt_static_for<0, GX / LX>([&](auto kc) {
                constexpr int k = decltype(kc)::v;
                unsigned row;
                unsigned char* const to = buf + ch * XCB + LP * 2 + (WHOLE ? PH * XROWB : 0) +
                                          place(mjt_ic<GX>(), mjt_ic<W_>(), mjt_ic<XROWB>(), mjt_ic<SW>(), mjt_ic<UX>(), mjt_ic<q>(), mjt_ic<k * LX>(), j, row);
                if (!WHOLE || H_ + PH <= XR || (int)row + PH < XR) {
                    if constexpr (SW == 1 || LX == 1) ux[b][q].template put<k * LX, LX>(to);
                    else ux[b][q].template put_phases<k * LX, LX>(to, to + RW * 2);
                }
            });
        } else {
            constexpr int i = q - NX;
            mjt_static_for<0, GD / LD>([&](auto kc) {
                constexpr int k = decltype(kc)::v;
                unsigned row;
                ud[b][i].template put<k * LD, LD>(buf + XB + ch * DCB + place(mjt_ic<GD>(), mjt_ic<OW_>(), mjt_ic<NPW * 16>(), mjt_ic<1>(), mjt_ic<UD>(), mjt_ic<i>(), mjt_ic<k * LD>(), j, row));
            });
        }
    };

    const int group = wave >> 2, wk = wave >> 1 & 1, wc = wave & 1, l32 = lane & 31, half = lane >> 5;
    const int ql = 2 * group + half;                                   // the lane's piece in step 0; 4 further in the next
    const int ql_row = ql / NPW, ql_col = ql % NPW;
    const unsigned char* const xl = lds + (wc * 32 + l32) * XCB + LP * 2 + ql_row * SH * XROWB + ql_col * 16;
    const unsigned char* const dl = lds + XB + (wk * 32 + l32) * DCB + ql * 16;
    mjt_f32x16 acc[TAPS];
    mjt_static_for<0, TAPS>([&](auto tc) { acc[decltype(tc)::v] = (mjt_f32x16)(0.0f); });

    fetch(first, 0u);
    for (int i = tid * 16; i < LDSB; i += 512 * 16) *(mjt_u32x4v*)(lds + i) = (mjt_u32x4v)(0u);
    __syncthreads();
    mjt_static_for<0, PIECES>([&](auto pc) { commit(pc, first, tid & 7); });
    __syncthreads();

    constexpr int NS = IB * SPG, SUBS = NS * R_;                       // a sub-step: one row of taps of a step
    unsigned raw[2][SW][HI - LO + 1];
    mjt_u32x4v fd[2];
#pragma unroll 1
    for (int st = first; st < last; st++) {
        const int n = WHOLE ? st * IB : st / SPI, rows = WHOLE ? OH_ : OH_ - (st - n * SPI) * RB;
        const int buf = (st & 1) * BUFB;
        fetch(st + 1, st + 1 < last ? 0u : MJT_NONE);
        unsigned j = tid & 7;
        asm volatile("" : "+v"(j));
        auto request = [&](auto sc) {
            constexpr int sub = decltype(sc)::v, t = sub / R_, r = sub % R_, b = t / SPG;
            constexpr int at = b * (XB + DB) + (step_row(t) * SH + r * DH) * XROWB + step_col(t) * 16;
            const unsigned char* from = xl + buf + at;
            if constexpr (CHECKED) {
                const int row = ql_row + step_row(t);
                const bool in = row < (rows < RB ? rows : RB) && (IB == 1 || n + b < N);
                from = in ? from : lds + 2 * BUFB + LP * 2;
            }
            mjt_static_for<0, SW>([&](auto phc) {
                constexpr int ph = decltype(phc)::v;
                if constexpr (phase_used(ph)) {
                    unsigned (&d)[HI - LO + 1] = raw[sub & 1][ph];
                    const mjt_u32x4v v = *(const mjt_u32x4v*)(from + ph * RW * 2);
                    d[-LO] = v[0]; d[1 - LO] = v[1]; d[2 - LO] = v[2]; d[3 - LO] = v[3];
                    mjt_static_for<0, HI - LO + 1>([&](auto wc_) {
                        constexpr int w = decltype(wc_)::v + LO;
                        if constexpr ((w < 0 && w >= lo_of(ph)) || (w > 3 && w <= hi_of(ph))) d[w - LO] = *(const unsigned*)(from + ph * RW * 2 + w * 4);
                    });
                }
            });
            if constexpr (r == 0) fd[t & 1] = *(const mjt_u32x4v*)(dl + buf + b * (XB + DB) + (t % SPG) * 64);
        };
        request(mjt_ic<0>());
        mjt_static_for<0, SUBS>([&](auto sc) {
            constexpr int sub = decltype(sc)::v, t = sub / R_, r = sub % R_;
            __builtin_amdgcn_sched_barrier(0);         // (reads of later sub-steps, moved up, would push the accumulators out)
            if constexpr (sub + 1 < SUBS) request(mjt_ic<sub + 1>());
            const bool edge = NPW == 1 || ql_col + step_col(t) == NPW - 1;      // the lane holds a row's last piece
            mjt_static_for<0, S_>([&](auto tc) {
                constexpr int s = decltype(tc)::v, ph = tap_phase(s), w = floor_div(tap_shift(s), 2) - LO;
                const unsigned (&d)[HI - LO + 1] = raw[sub & 1][ph];
                mjt_u32x4v f;
                mjt_static_for<0, 4>([&](auto ec) {
                    constexpr int e = decltype(ec)::v;
                    if constexpr (tap_shift(s) & 1) f[e] = __builtin_amdgcn_alignbit(d[w + e + 1], d[w + e], 16);
                    else f[e] = d[w + e];
                    if constexpr (2 * e >= VD) f[e] = edge ? 0u : f[e];
                    else if constexpr (2 * e + 1 >= VD) f[e] = edge ? f[e] & 0xffffu : f[e];
                });
                acc[r * S_ + s] = MJT_MFMA(__builtin_bit_cast(mjt_h8, fd[t & 1]), __builtin_bit_cast(mjt_h8, f), acc[r * S_ + s], 0, 0, 0);
                // the next stage moves to the other buffer, which nobody has read since the last barrier, between all but the first MFMAs
                constexpr int slot = sub * S_ + s, SLOTS = SUBS * S_, BEGIN = SLOTS / 4;
                if constexpr (slot >= BEGIN) {
                    constexpr int from = PIECES * (slot - BEGIN) / (SLOTS - BEGIN), to = PIECES * (slot + 1 - BEGIN) / (SLOTS - BEGIN);
                    if constexpr (to > from) mjt_static_for<from, to>([&](auto pc) { commit(pc, st + 1, j); });     // (zeros behind the last stage)
                }
            });
        });
        __syncthreads();
    }

    // D of a 32 x 32 tile: lane holds column (c) lane % 32, rows (k) 8 * (e / 4) + 4 * (lane / 32) + e % 4
    // the groups' sums meet there: each adds what the other has written of one half of the taps
    float* const out = (float*)lds;
    auto at = [&](int tap, int e) -> float& { return out[(wk * 32 + 8 * (e / 4) + 4 * half + (e & 3)) * OUTS + (wc * 32 + l32) * TAPS + tap]; };
    auto put = [&](auto tc) {
#pragma unroll
        for (int e = 0; e < 16; e++) at(decltype(tc)::v, e) = acc[decltype(tc)::v][e];
    };
    auto add = [&](auto tc) {
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; e++) v[e] = at(decltype(tc)::v, e);
#pragma unroll
        for (int e = 0; e < 16; e++) at(decltype(tc)::v, e) = acc[decltype(tc)::v][e] + v[e];
    };
    if (group == 1) mjt_static_for<0, TAPS / 2>(put);
    else mjt_static_for<TAPS / 2, TAPS>(put);
    __syncthreads();
    if (group == 0) mjt_static_for<0, TAPS / 2>(add);
    else mjt_static_for<TAPS / 2, TAPS>(add);
    __syncthreads();
    float* const part = (float*)p.a[2] + (long long)slice * ((long long)K_ * C_ * TAPS);
    const int krows = K_ - k0 < 64 ? K_ - k0 : 64, width = (C_ - c0 < 64 ? C_ - c0 : 64) * TAPS;
    constexpr int V = C_ * TAPS % 4 == 0 ? 4 : 1;                      // floats of a store: rows and blocks begin at multiples of 16 bytes, or not
    auto store = [&](int row, int col) {
        float* const to = part + (long long)(k0 + row) * (C_ * TAPS) + c0 * TAPS + col;
        if constexpr (V == 4) *(mjt_u32x4v*)to = *(const mjt_u32x4v*)(out + row * OUTS + col);
        else *to = out[row * OUTS + col];
    };
    // (whole tiles without a condition, so that the reads of several stores are on their way together)
    constexpr int MOVES = 64 * 64 * TAPS / V / 512;
    if (krows == 64 && width == 64 * TAPS) {
#pragma unroll 6
        for (int m = 0; m < MOVES; m++) {
            const int i = tid + m * 512, row = i / (64 * TAPS / V), col = (i - row * (64 * TAPS / V)) * V;
            store(row, col);
        }
    } else {
#pragma unroll 1
        for (int i = tid; i < 64 * (64 * TAPS / V); i += 512) {
            const int row = i / (64 * TAPS / V), col = (i - row * (64 * TAPS / V)) * V;
            if (row < krows && col < width) store(row, col);
        }
    }
}
