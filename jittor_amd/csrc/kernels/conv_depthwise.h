// Depthwise convolution (one input channel per group) and its two gradients
// (python/jittor/nn.py:1272-1294 with C / G == 1; the gradients are the ones
// python/jittor/src/opt/tuner/conv_tuner.cc:375-397 relays).  Nothing is contracted over channels, so the work is
// bound by memory: one read of x (or dy) and one write of the result.  With one lane per output every tap was a load
// of its own through the caches; here a workgroup stages planes in LDS once, vector loads in, and a lane computes a
// strip of RS rows x CW columns from it, reading every row of the strip's window as 16-byte pieces and using it for
// all taps and output rows that touch it.  us before / after, 32 x 128 x 56 x 56, 3x3, float32 (51 MB read, 51 written:
// 16 us at the rate of a copy): forward 35.8 / 17.8, input gradient 40.4 (with the rearranged weights) / 16.5, weight
// gradient with its fold 55.4 / 26.5; on 64 x 256 x 14 x 14 the three take 8.0 / 8.0 / 12.4.
//
// MODE 0: y[n, ko] = conv(x[n, ko / MULT], w[ko]).  The input gradient is the same with dy in x's place, the taps flipped (FLIP)
//         and, for a strided convolution, the rows and columns of dy UH and UW apart in LDS with zeros between them.
// MODE 1: partial[slice][ko][tap] = sum over the slice's images and all positions of dy * x; the slices are added up by
//         a reduce launch.
// MODE 2: both gradients of a convolution of stride 1 without dilation at once.  dy is staged as for the input gradient; the lane that makes a
//         strip of dx has the same strip of x in registers and multiplies the window's rows with it as well, which gives the weight
//         gradient's terms: dy is read once, x once, dx written once.  Cells around dy are zeros that are no terms of the weight
//         gradient, harmless unless x is infinite there; and a zero around x times an infinite dy is a term that this way does not
//         see.  Either leaves some sum of the workgroup not finite, and then its sums are taken again, term by term.
//         us with the fold, input and weight gradient / both: float32 3x3 32 x 128 x 56 x 56 49.8 / 37.0 (154 MB: 24.5 at the rate of a copy),
//         64 x 256 x 14 x 14 21.6 / 19.2, 8 x 32 x 112 x 112 25.3 / 18.4, 4 x 512 x 7 x 7 7.9 / 5.2, 5x5 64 x 24 x 56 x 56 34.0 / 26.1; bfloat16 3x3
//         32 x 128 x 56 x 56 35.1 / 26.3.  (x asked for ahead of the window, like dy: 148 registers instead of 126, three workgroups a
//         unit instead of four, 39.9; held to 128 registers it spills, 46.6.)
// Supplied by the host: TIN, TOUT, the geometry (H_, W_ of the staged planes, OH_, OW_ of the planes a lane's strips lie
// in, R_, S_, SH, SW, PH, PW, DH, DW), UH, UW, MULT, K_ (planes per image of y / dy), TH (rows of a plane per
// workgroup, NTILE such tiles per plane), PPW (planes, or images of one channel in MODE 1, staged together), VEC (elements
// per staging load), CW, RS, STVEC (elements per access of y / dy).

struct Params { void* a[7]; };   // MODE 0: x, w, y, planes of y;  MODE 1: x, dy, partial, images, images per slice;  MODE 2: dy, x, partial, images, images per slice, w, dx

constexpr int NV = ((CW - 1) * SW + (S_ - 1) * DW + 1 + 3) / 4;        // 16-byte pieces of a strip's row
constexpr int NCG = (OW_ + CW - 1) / CW;                               // column groups of a row
constexpr int NST = (TH + RS - 1) / RS;                                // strips of a tile
constexpr int LR = (NST * RS - 1) * SH + (R_ - 1) * DH + 1;            // rows of a staged tile
constexpr int LC = ((NCG - 1) * CW * SW + NV * 4 + 3) / 4 * 4;         // its columns
constexpr int NIR = NTILE == 1 ? H_ : ((LR - 1) / UH + 2 < H_ ? (LR - 1) / UH + 2 : H_);   // rows of the plane a tile may need
constexpr int WV = W_ / VEC;
constexpr int NLD = PPW * NIR * WV;                                    // staging loads of a tile
constexpr int NIT = (NLD + 255) / 256;
constexpr int BATCH = NIT < 8 ? NIT : 8;                               // of them under way per lane
constexpr int TASKS = PPW * NST * NCG;

__shared__ __attribute__((aligned(16))) float tile[PPW * LR * LC];

__device__ __forceinline__ void mjt_dw_clear() {
    typedef float f4 __attribute__((ext_vector_type(4)));
    for (int i = threadIdx.x; i < PPW * LR * LC / 4; i += 256) ((f4*)tile)[i] = (f4)(0.0f);
}

// Loads `b` .. `b` + BATCH - 1 of a lane's share of `count` planes (plane i at xp + i * pstride), rows from ih0 on.
// Unconditional: a lane without a share loads the first element.
__device__ __forceinline__ void mjt_dw_load(mjt_pack<TIN, VEC> (&v)[BATCH], const TIN* __restrict__ xp, long long pstride, int count, int ih0, int b) {
#pragma unroll
    for (int u = 0; u < BATCH; u++) {
        const int i = (b + u) * 256 + (int)threadIdx.x;
        const int pl = i / (NIR * WV), rest = i - pl * (NIR * WV), row = rest / WV, cv = rest - row * WV;
        const bool on = i < NLD && pl < count;
        mjt_load(v[u], xp + (on ? pl * pstride + (long long)((ih0 + row) * W_ + cv * VEC) : 0));
    }
}
// ... and into LDS, whose row 0 is row `first` of the planes (counted with the zeros of UH and UW in between)
__device__ __forceinline__ void mjt_dw_fill(const mjt_pack<TIN, VEC> (&v)[BATCH], int count, int ih0, int first, int b) {
#pragma unroll
    for (int u = 0; u < BATCH; u++) {
        const int i = (b + u) * 256 + (int)threadIdx.x;
        const int pl = i / (NIR * WV), rest = i - pl * (NIR * WV), row = rest / WV, cv = rest - row * WV;
        const int lr = (ih0 + row) * UH - first, lc = cv * VEC * UW + PW;
        if (i < NLD && pl < count && lr >= 0 && lr < LR) {
            float* const dst = tile + (pl * LR + lr) * LC + lc;
#pragma unroll
            for (int k = 0; k < VEC; k++)
                if (lc + k * UW < LC) dst[k * UW] = (float)v[u].v[k];
        }
    }
}
__device__ __forceinline__ int mjt_dw_first_row(int oh0) {
    if (NTILE == 1) return 0;
    const int first = oh0 * SH - PH, ih0 = first > 0 ? first / UH : 0;
    return ih0 > H_ - NIR ? H_ - NIR : ih0;
}
// the rows that the tile at output row oh0 needs into LDS; cells outside the planes stay zero
__device__ __forceinline__ void mjt_dw_stage(const TIN* __restrict__ xp, long long pstride, int count, int oh0) {
    const int ih0 = mjt_dw_first_row(oh0);
    for (int b = 0; b < NIT; b += BATCH) {
        mjt_pack<TIN, VEC> v[BATCH];
        mjt_dw_load(v, xp, pstride, count, ih0, b);
        mjt_dw_fill(v, count, ih0, oh0 * SH - PH, b);
    }
}

// f(row of LDS inside the strip, its values) for the strip's rows from the top
template <class F> __device__ __forceinline__ void mjt_dw_rows(int pl, int strip, int cg, F&& f) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4* const src = (const f4*)(tile + (pl * LR + strip * RS * SH) * LC + cg * CW * SW);
#pragma unroll
    for (int lr = 0; lr < (RS - 1) * SH + (R_ - 1) * DH + 1; lr++) {
        float x[NV * 4];
#pragma unroll
        for (int q = 0; q < NV; q++) {
            const f4 t = src[lr * (LC / 4) + q];
            x[q * 4] = t[0]; x[q * 4 + 1] = t[1]; x[q * 4 + 2] = t[2]; x[q * 4 + 3] = t[3];
        }
        f(lr, x);
    }
}

extern "C" __global__ __launch_bounds__(256) void ENTRY(Params p) {
    const TIN* __restrict__ xp = (const TIN*)p.a[0];
#if MODE == 0
    const TIN* __restrict__ wp = (const TIN*)p.a[1];
    TOUT* __restrict__ yp = (TOUT*)p.a[2];
    const long long planes = (long long)(unsigned long long)p.a[3];
    const int oh0 = (int)(blockIdx.x % NTILE) * TH;
    const long long p0 = (long long)(blockIdx.x / NTILE) * PPW;         // first plane of y (the host makes PPW 1 when MULT > 1)
    const int count = planes - p0 < PPW ? (int)(planes - p0) : PPW;
    mjt_dw_clear();
    __syncthreads();
    mjt_dw_stage(xp + p0 / MULT * (H_ * W_), H_ * W_, count, oh0);
    __syncthreads();
    for (int t = threadIdx.x; t < TASKS; t += 256) {
        const int pl = t / (NST * NCG), rest = t - pl * (NST * NCG), strip = rest / NCG, cg = rest - strip * NCG;
        if (pl >= count) break;
        const int ko = (int)((p0 + pl) % K_);
        float w[R_ * S_];
#pragma unroll
        for (int k = 0; k < R_ * S_; k++) w[k] = (float)wp[ko * (R_ * S_) + (FLIP ? R_ * S_ - 1 - k : k)];
        float acc[RS][CW];
#pragma unroll
        for (int r = 0; r < RS; r++)
#pragma unroll
            for (int j = 0; j < CW; j++) acc[r][j] = 0.0f;
        mjt_dw_rows(pl, strip, cg, [&](int lr, const float* x) {
#pragma unroll
            for (int ro = 0; ro < RS; ro++)
#pragma unroll
                for (int r = 0; r < R_; r++)
                    if (ro * SH + r * DH == lr) {
#pragma unroll
                        for (int s = 0; s < S_; s++)
#pragma unroll
                            for (int j = 0; j < CW; j++) acc[ro][j] = acc[ro][j] + x[j * SW + s * DW] * w[r * S_ + s];
                    }
        });
        TOUT* const dst = yp + (p0 + pl) * (OH_ * OW_);
#pragma unroll
        for (int ro = 0; ro < RS; ro++) {
            const int oh = oh0 + strip * RS + ro;
            if (strip * RS + ro < TH && oh < OH_) {
#pragma unroll
                for (int j = 0; j < CW; j += STVEC) {
                    if (cg * CW + j < OW_) {
                        mjt_pack<TOUT, STVEC> o;
#pragma unroll
                        for (int k = 0; k < STVEC; k++) o.v[k] = (TOUT)acc[ro][j + k];
                        mjt_store(dst + oh * OW_ + cg * CW + j, o);
                    }
                }
            }
        }
    }
#else
    const TIN* __restrict__ dyp = (const TIN*)p.a[1];
    float* __restrict__ part = (float*)p.a[2];
    const long long n_img = (long long)(unsigned long long)p.a[3], ips = (long long)(unsigned long long)p.a[4];
    const int ko = (int)(blockIdx.x % K_);
    const long long slice = blockIdx.x / K_;
    const long long n1 = (slice + 1) * ips < n_img ? (slice + 1) * ips : n_img;
    constexpr int C = K_ / MULT;
    float acc[R_ * S_];
#pragma unroll
    for (int k = 0; k < R_ * S_; k++) acc[k] = 0.0f;
#if MODE == 2
    const TIN* __restrict__ wp = (const TIN*)p.a[5];
    TOUT* __restrict__ dxp = (TOUT*)p.a[6];
    float w[R_ * S_];
#pragma unroll
    for (int k = 0; k < R_ * S_; k++) w[k] = (float)wp[ko * (R_ * S_) + R_ * S_ - 1 - k];
    auto both = [&](long long n, int count, int oh0) {
        for (int t = threadIdx.x; t < TASKS; t += 256) {
            const int pl = t / (NST * NCG), rest = t - pl * (NST * NCG), row = rest / NCG, cg = rest - row * NCG;
            if (pl >= count) break;
            const long long at = ((n + pl) * K_ + ko) * (OH_ * OW_);
            float xv[RS][CW], dx[RS][CW];
#pragma unroll
            for (int ro = 0; ro < RS; ro++) {
                const int oh = oh0 + row * RS + ro;
                const bool row_in = row * RS + ro < TH && oh < OH_;
#pragma unroll
                for (int j = 0; j < CW; j += STVEC) {                   // out of range: the first element, replaced by zero
                    const bool in = row_in && cg * CW + j < OW_;
                    mjt_pack<TIN, STVEC> v;
                    mjt_load(v, dyp + at + (in ? oh * OW_ + cg * CW + j : 0));
#pragma unroll
                    for (int k = 0; k < STVEC; k++) {
                        xv[ro][j + k] = in ? (float)v.v[k] : 0.0f;
                        dx[ro][j + k] = 0.0f;
                    }
                }
            }
            mjt_dw_rows(pl, row, cg, [&](int lr, const float* d) {
#pragma unroll
                for (int ro = 0; ro < RS; ro++)
#pragma unroll
                    for (int r = 0; r < R_; r++)
                        if (ro + r == lr) {
#pragma unroll
                            for (int s = 0; s < S_; s++)
#pragma unroll
                                for (int j = 0; j < CW; j++) {
                                    dx[ro][j] = dx[ro][j] + d[j + s] * w[r * S_ + s];
                                    acc[(R_ - 1 - r) * S_ + S_ - 1 - s] = acc[(R_ - 1 - r) * S_ + S_ - 1 - s] + d[j + s] * xv[ro][j];
                                }
                        }
            });
            TOUT* const dst = dxp + at;
#pragma unroll
            for (int ro = 0; ro < RS; ro++) {
                const int oh = oh0 + row * RS + ro;
                if (row * RS + ro < TH && oh < OH_) {
#pragma unroll
                    for (int j = 0; j < CW; j += STVEC) {
                        if (cg * CW + j < OW_) {
                            mjt_pack<TOUT, STVEC> o;
#pragma unroll
                            for (int k = 0; k < STVEC; k++) o.v[k] = (TOUT)dx[ro][j + k];
                            mjt_store(dst + oh * OW_ + cg * CW + j, o);
                        }
                    }
                }
            }
        }
    };
#else
    auto sums = [&](long long n, int count, int oh0) {
        for (int t = threadIdx.x; t < TASKS; t += 256) {
            const int pl = t / (NST * NCG), rest = t - pl * (NST * NCG), strip = rest / NCG, cg = rest - strip * NCG;
            if (pl >= count) break;
            const TIN* const src = dyp + ((n + pl) * K_ + ko) * (OH_ * OW_);
            float dy[RS][CW];
#pragma unroll
            for (int ro = 0; ro < RS; ro++) {
                const int oh = oh0 + strip * RS + ro;
                const bool row_in = strip * RS + ro < TH && oh < OH_;
#pragma unroll
                for (int j = 0; j < CW; j += STVEC) {                   // out of range: the first element, replaced by zero
                    const bool in = row_in && cg * CW + j < OW_;
                    mjt_pack<TIN, STVEC> v;
                    mjt_load(v, src + (in ? oh * OW_ + cg * CW + j : 0));
#pragma unroll
                    for (int k = 0; k < STVEC; k++) dy[ro][j + k] = in ? (float)v.v[k] : 0.0f;
                }
            }
            // A strip may reach past the map's last row and column, over pixels that exist: those positions are no term of the sum, and
            // a product with their zero would be one (0 times an infinity).  Columns are taken out of x once per row, rows are skipped.
            constexpr bool PART_ROWS = OH_ % RS != 0 || OH_ % TH != 0, PART_COLS = OW_ % CW != 0;
            const int rows = OH_ - oh0 < TH ? OH_ - oh0 - strip * RS : TH - strip * RS;
            mjt_dw_rows(pl, strip, cg, [&](int lr, const float* x) {
                float xv[S_][CW];
#pragma unroll
                for (int s = 0; s < S_; s++)
#pragma unroll
                    for (int j = 0; j < CW; j++) xv[s][j] = !PART_COLS || cg * CW + j < OW_ ? x[j * SW + s * DW] : 0.0f;
#pragma unroll
                for (int ro = 0; ro < RS; ro++)
#pragma unroll
                    for (int r = 0; r < R_; r++)
                        if (ro * SH + r * DH == lr && (!PART_ROWS || ro < rows)) {
#pragma unroll
                            for (int s = 0; s < S_; s++)
#pragma unroll
                                for (int j = 0; j < CW; j++) acc[r * S_ + s] = acc[r * S_ + s] + dy[ro][j] * xv[s][j];
                        }
            });
        }
    };
#endif
    auto images = [&](long long n) { return n1 - n < PPW ? (n1 > n ? (int)(n1 - n) : 0) : PPW; };
    const TIN* __restrict__ xc = xp + (ko / MULT) * (H_ * W_);
    const long long istride = (long long)C * (H_ * W_);
    mjt_dw_clear();
    if constexpr (NTILE == 1 && NIT == BATCH) {                         // the next planes are on their way while these are summed
        long long n = slice * ips;
        mjt_pack<TIN, VEC> v[BATCH];
        mjt_dw_load(v, xc + n * istride, istride, images(n), 0, 0);
        for (; n < n1; n += PPW) {
            __syncthreads();                                            // everybody is done with the planes before
            mjt_dw_fill(v, images(n), 0, -PH, 0);
            __syncthreads();
            const long long next = n + PPW < n1 ? n + PPW : n;
            mjt_dw_load(v, xc + next * istride, istride, images(next), 0, 0);
#if MODE == 2
            both(n, images(n), 0);
#else
            sums(n, images(n), 0);
#endif
        }
    } else {
        for (long long n = slice * ips; n < n1; n += PPW)
            for (int tl = 0; tl < NTILE; tl++) {
                __syncthreads();
                if (NTILE > 1 && tl + n > slice * ips) {                // another tile leaves other rows empty
                    mjt_dw_clear();
                    __syncthreads();
                }
#if MODE == 2
                mjt_dw_stage(xc + n * istride, istride, images(n), tl * TH);
                __syncthreads();
                both(n, images(n), tl * TH);
#else
                mjt_dw_stage(xc + n * istride, istride, images(n), tl * TH);
                __syncthreads();
                sums(n, images(n), tl * TH);
#endif
            }
    }
#if MODE == 2
    {
        float z = 0.0f;                                                 // not zero if any sum is not finite
#pragma unroll
        for (int k = 0; k < R_ * S_; k++) z = z + acc[k] * 0.0f;
        if (__syncthreads_or(!(z == 0.0f))) {
            constexpr int PADH = R_ - 1 - PH, PADW = S_ - 1 - PW;       // the convolution's own padding
#pragma unroll
            for (int k = 0; k < R_ * S_; k++) acc[k] = 0.0f;
            for (long long n = slice * ips; n < n1; n++) {
                const TIN* const d = xp + (n * K_ + ko) * (H_ * W_);
                const TIN* const x = dyp + (n * K_ + ko) * (OH_ * OW_);
                for (int i = threadIdx.x; i < H_ * W_; i += 256) {
                    const int oh = i / W_, ow = i - oh * W_;
                    const float dv = (float)d[i];
#pragma unroll
                    for (int k = 0; k < R_ * S_; k++) {
                        const int h = oh - PADH + k / S_, c = ow - PADW + k % S_;
                        const bool in = h >= 0 && h < OH_ && c >= 0 && c < OW_;
                        const float xv = (float)x[in ? h * OW_ + c : 0];
                        acc[k] = acc[k] + dv * (in ? xv : 0.0f);
                    }
                }
            }
        }
    }
#endif
    __shared__ float fold[4][R_ * S_];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < R_ * S_; k++) {
        float v = acc[k];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off, 64);
        if (lane == 0) fold[wave][k] = v;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < R_ * S_; k += 256)
        part[(slice * K_ + ko) * (R_ * S_) + k] = (fold[0][k] + fold[1][k]) + (fold[2][k] + fold[3][k]);
#endif
}
