// Windows folded where they lie: z[b.., oh, ow] = fold over (kh, kw) of x[b.., oh*SH + kh*DH + CH, ow*SW + kw*DW + CW], the overflow value
// outside x (reference: python/jittor/src/ops/reindex_op.cc:111-139 with the reduce that consumes it; pooling, python/jittor/pool.py:200-208).
//
// Supplied by the host: TX, TZ, TACC, LV (elements of x in 16 bytes), OR x OV (outputs a lane owns; OV*SW is a multiple of LV), ZV (outputs
// stored together), KH, KW, SH, SW, DH, DW, CH, CW, H_, W_ (a multiple of LV), OH_, OW_, INIT, COMBINE(a, x).
//
// Bound by memory: x once, z once.  A lane that folds one output loads its window element by element, 9 loads for a 3x3 window that its
// neighbours load again; here a lane owns OV neighbouring outputs of OR rows and loads the rows beneath as 16-byte pieces, which begin at
// multiples of 16 bytes and lie wholly inside or outside a row: 15 loads for eight outputs of 3x3 stride 2 against 72 (32 x 64 x 112 x 112
// float32 35.9 -> 28.4 us, 4.5 TB/s; bfloat16 38.2 -> 13.0, 5.9 TB/s).  Every output meets its
// window in the order of the taps, as in the kernel of one output a lane, so the results are the same bits.

struct Params { void* a[5]; };

constexpr int mjt_floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }
#define FIRST mjt_floor_div(CW, LV)                                              // first and last piece that a lane's windows touch, from its first column on
#define LAST mjt_floor_div((OV - 1) * SW + (CW) + (KW - 1) * DW, LV)
#define NP (LAST - FIRST + 1)
#define NR ((OR - 1) * SH + (KH - 1) * DH + 1)                                   // rows of x beneath a lane's outputs

extern "C" __global__ __launch_bounds__(256) void ENTRY(Params p) {
    const TX* __restrict__ xp = (const TX*)p.a[0];
    TZ* __restrict__ zp = (TZ*)p.a[1];
    const unsigned lanes = (unsigned)(unsigned long long)p.a[2];
    const TX ovalue = (TX)__longlong_as_double((long long)(unsigned long long)p.a[3]);
    const TACC rcount = (TACC)__longlong_as_double((long long)(unsigned long long)p.a[4]);
    (void)rcount;
    const unsigned lane = blockIdx.x * 256 + threadIdx.x;
    if (lane >= lanes) return;
    constexpr unsigned ACROSS = (OW_ + OV - 1) / OV, DOWN = (OH_ + OR - 1) / OR;
    const int ow0 = (int)(lane % ACROSS) * OV;
    const unsigned t = lane / ACROSS;
    const int oh0 = (int)(t % DOWN) * OR;
    const int plane = (int)(t / DOWN);

    TX got[NR][NP * LV];
#pragma unroll
    for (int j = 0; j < NR; j++) {
        const int h = oh0 * SH + (CH) + j;
        const bool in_h = h >= 0 && h < H_;
#pragma unroll
        for (int q = 0; q < NP; q++) {
            const int c = ow0 * SW + (FIRST + q) * LV;
            const bool in = in_h && c >= 0 && c < W_;
            mjt_pack<TX, LV> piece;
            mjt_load(piece, xp + (in ? (plane * H_ + h) * W_ + c : 0));              // (unconditional: the loads of a lane are under way together)
#pragma unroll
            for (int e = 0; e < LV; e++) got[j][q * LV + e] = in ? piece.v[e] : ovalue;
        }
    }
#pragma unroll
    for (int r = 0; r < OR; r++) {
        if (oh0 + r >= OH_) break;
        mjt_pack<TZ, OV> out;
#pragma unroll
        for (int k = 0; k < OV; k++) {
            TACC acc = INIT;
#pragma unroll
            for (int kh = 0; kh < KH; kh++)
#pragma unroll
                for (int kw = 0; kw < KW; kw++) acc = (TACC)(COMBINE(acc, (got[r * SH + kh * DH][k * SW + (CW) + kw * DW - FIRST * LV])));
            out.v[k] = (TZ)acc;
        }
        TZ* const to = zp + (plane * OH_ + oh0 + r) * OW_ + ow0;
#pragma unroll
        for (int k = 0; k < OV; k += ZV) {
            mjt_pack<TZ, ZV> some;
#pragma unroll
            for (int e = 0; e < ZV; e++) some.v[e] = out.v[k + e];
            if (ow0 + k < OW_) mjt_store(to + k, some);
        }
    }
}
