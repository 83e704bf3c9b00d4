// Scatter through a window pattern, turned into a gather
// (reference: python/jittor/src/ops/reindex_reduce_op.cc:93-131; the gradient of pooling, python/jittor/pool.py:200-208).
//
// x[b.., oh*SH + kh*DH + CH, ow*SW + kw*DW + CW] op= y[b.., oh, ow, kh, kw]: with windows that overlap, neighbouring
// elements of y meet in the same element of x and atomic updates queue up behind each other.  Every element of x knows
// which windows reach it, so one lane per element of x folds them itself: no atomics, no identity fill, one coalesced
// store.  Row h is reached from output row oh through tap kh when oh*SH + kh*DH + CH == h; the candidates are the NCH
// output rows at and below (h - CH) / SH (NCH = (KH-1)*DH / SH + 1), likewise for columns, where a lane looks at the NCU that
// reach any of its elements (NCU = (VEC-1 + (KW-1)*DW) / SW + 1).
//
// Constants and fragments supplied by the host:
//   TX, TACC, index_t, VEC, NPARAM, NB (batch axes), KH, KW, SH, SW, DH, DW, CH, CW, NCH, NCU, BLOCKS
//   MJT_RX_SETUP    xshapeK, yshapeK and strides (the names the index language uses)
//   MJT_WS_BATCH    coordinates i0 .. i{NB-1} of plane number plane_
//   I_OH, I_OW, I_KH, I_KW   the names of the four window coordinates (i{NB} .. i{NB+3})
//   INIT, COMBINE(a, v)
//   SC_PROLOGUE, MJT_SC_SCALARS, MJT_SC_VALUE   as in the generic scatter kernel: the scattered value `val_` of element e_
//                   of y, computed from the group's inputs (a gathered input is read at xid, which is this lane's element)
//
// BLOCKS 1 (VEC is a multiple of SW): a lane owns SH rows x VEC columns, from a row and a column that are multiples of the stride on, so
// that which windows reach which element through which tap is known when the kernel is built: the candidates that reach none are
// not looked at (3x3 stride 2: 18 of the 48 that two rows of four have), a window that reaches several rows is loaded once for all of
// them, and of the address arithmetic the bounds remain (with the group below 59.5 -> 49.0 us, 5.3 TB/s).
//
// An element group behind the scatter (epilogue.h: the mask of the relu in front of a pooling) runs on the lane's elements before they are
// stored: 3x3 stride-2 maximum of 32 x 64 x 112 x 112 float32, gradient and mask 62.6 + 35.7 us / together 60.2 (a row a lane), and the mask is not stored in the
// forward pass (convolution with relu 72.5 -> 68.1).
//
// A candidate that does not exist is computed at clamped coordinates and dropped afterwards, so that no branch separates
// the loads of a lane.

#ifndef EPI
#define EPI 0
#endif
struct Params { void* a[NPARAM]; };
#if BLOCKS
template <int V> struct mjt_ic { static constexpr int v = V; };
template <int I, int N, class F> __device__ __forceinline__ void mjt_static_for(F&& f) {
    if constexpr (I < N) {
        f(mjt_ic<I>());
        mjt_static_for<I + 1, N>(f);
    }
}
constexpr int mjt_floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }
#else
static_assert(NCH * NCU * VEC <= 40, "bodies that a lane unrolls");
#endif

extern "C" __global__ __launch_bounds__(256) void ENTRY(Params p) {
    TX* __restrict__ xp = (TX*)p.a[0];
    const TX* __restrict__ yp = (const TX*)p.a[1];
    (void)yp;
    const index_t nx = (index_t)(unsigned long long)p.a[2];
    MJT_RX_SETUP
#if SC_PROLOGUE
    MJT_SC_SCALARS
#endif
#if BLOCKS
    // lane: block of SH rows x VEC columns (W is a multiple of VEC) of a plane; a[2] is the number of blocks
    const index_t lane_ = (index_t)blockIdx.x * 256 + threadIdx.x;
    if (lane_ >= nx) return;
    const index_t H_ = xshape_h, W_ = xshape_w, OH_ = yshape_oh, OW_ = yshape_ow;
    const index_t w0_ = lane_ % (W_ / VEC) * VEC;
    const index_t t_ = lane_ / (W_ / VEC);
    const index_t hb_ = t_ % ((H_ + SH - 1) / SH);
    const index_t plane_ = t_ / ((H_ + SH - 1) / SH);
    MJT_WS_BATCH
    const index_t wb_ = w0_ / SW;
    // rows past the last one are computed at the last one's place and not stored
    auto row_of_ = [&](int r) { const index_t h = hb_ * SH + r; return (plane_ * H_ + (h < H_ ? h : H_ - 1)) * W_ + w0_; };
    TACC acc_[SH][VEC];
#pragma unroll
    for (int r = 0; r < SH; r++)
#pragma unroll
        for (int k = 0; k < VEC; k++) acc_[r][k] = INIT;
#if EPI
    mjt_epi_in<VEC> behind_[SH];                               // what the group behind the scatter reads of the lane's elements
#pragma unroll
    for (int r = 0; r < SH; r++) mjt_epi_load(p, behind_[r], (MJT_EPI_INDEX)row_of_(r));
#endif
    // Rows and columns of windows, both falling, as every element meets them (below): row hb_ + TOP - a, column wb_ + RIGHT - b.
    constexpr int TOP = mjt_floor_div(SH - 1 - (CH), SH), RIGHT = mjt_floor_div(VEC - 1 - (CW), SW);
    constexpr int ROWS = TOP - mjt_floor_div(-(CH) - (KH - 1) * DH, SH) + 1, COLS = RIGHT - mjt_floor_div(-(CW) - (KW - 1) * DW, SW) + 1;
    mjt_static_for<0, ROWS>([&](auto ac) {
        constexpr int a = decltype(ac)::v;
        const index_t oh_c = hb_ + (TOP - a);
        const bool ok_h = oh_c >= 0 && oh_c < OH_;
        const index_t I_OH = ok_h ? oh_c : (index_t)0;
        mjt_static_for<0, COLS>([&](auto bc) {
            constexpr int b = decltype(bc)::v;
            const index_t ow_c = wb_ + (RIGHT - b);
            const bool ok_o = ok_h && ow_c >= 0 && ow_c < OW_;
            const index_t I_OW = ok_o ? ow_c : (index_t)0;
            mjt_static_for<0, SH * VEC>([&](auto ec) {
                constexpr int r = decltype(ec)::v / VEC, k = decltype(ec)::v % VEC;
                constexpr int rh = r - (CH) - (TOP - a) * SH, rw = k - (CW) - (RIGHT - b) * SW;       // kh * DH and kw * DW, if such taps exist
                if constexpr (rh >= 0 && rh % DH == 0 && rh / DH < KH && rw >= 0 && rw % DW == 0 && rw / DW < KW) {
                    const index_t I_KH = rh / DH, I_KW = rw / DW;
                    const index_t xid = row_of_(r) + k;
                    const index_t e_ = (((plane_ * OH_ + I_OH) * OW_ + I_OW) * KH + I_KH) * KW + I_KW;
                    (void)xid;
                    (void)e_;
                    MJT_SC_VALUE
                    const TACC next_ = (TACC)(COMBINE(acc_[r][k], val_));
                    acc_[r][k] = ok_o ? next_ : acc_[r][k];
                }
            });
        });
    });
#pragma unroll
    for (int r = 0; r < SH; r++) {
        if (hb_ * SH + r >= H_) break;
#if EPI
        float sum_[VEC];
#pragma unroll
        for (int k = 0; k < VEC; k++) sum_[k] = (float)(TX)acc_[r][k];
        mjt_epi_finish(p, behind_[r], (MJT_EPI_INDEX)row_of_(r), sum_);
#else
        mjt_pack<TX, VEC> out_;
#pragma unroll
        for (int k = 0; k < VEC; k++) out_.v[k] = (TX)acc_[r][k];
        mjt_store(xp + row_of_(r), out_);
#endif
    }
#else
    // a lane owns VEC adjacent elements of a row of x (W is a multiple of VEC) and stores them as one vector
    const index_t xbase_ = ((index_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (xbase_ >= nx) return;
    const index_t H_ = xshape_h, W_ = xshape_w, OH_ = yshape_oh, OW_ = yshape_ow;
    const index_t w0_ = xbase_ % W_;
    const index_t t_ = xbase_ / W_;
    const index_t h_ = t_ % H_;
    const index_t plane_ = t_ / H_;
    MJT_WS_BATCH
    const index_t th_ = h_ - (CH);
    const index_t oh_hi = th_ >= 0 ? th_ / SH : (index_t)-1;
    // Windows outside, the lane's elements inside: what a window holds (the result and its gradient of a pooling) is loaded once
    // for all elements that it reaches.  A lane's elements are reached from NCU columns of windows.  Every element meets its
    // windows in the same order, rows and columns falling.  (Elements outside, every element loaded its windows' values for
    // itself, 32 scattered loads a lane against 12: gradient of a 3x3 stride-2 maximum pooling of 32 x 64 x 112 x 112 float32
    // 111 -> 63 us, 4.1 TB/s of what it cannot do without.)
    const index_t tw0_ = w0_ - (CW), tw1_ = tw0_ + (VEC - 1);
    const index_t ow_hi = tw1_ >= 0 ? tw1_ / SW : (index_t)-1;
    TACC acc_[VEC];
#pragma unroll
    for (int k = 0; k < VEC; k++) acc_[k] = INIT;
#if EPI
    mjt_epi_in<VEC> behind_;                                   // what the group behind the scatter reads of the lane's elements
    mjt_epi_load(p, behind_, (MJT_EPI_INDEX)xbase_);
#endif
#pragma unroll
    for (int a = 0; a < NCH; a++) {
        const index_t oh_c = oh_hi - a;
        const index_t rh_ = th_ - oh_c * SH;                   // kh * DH, if this row of windows reaches the lane's row
        const bool ok_h = oh_c >= 0 && oh_c < OH_ && rh_ % DH == 0 && rh_ / DH < KH;
        const index_t I_OH = ok_h ? oh_c : (index_t)0;
        const index_t I_KH = ok_h ? rh_ / DH : (index_t)0;
#pragma unroll
        for (int b = 0; b < NCU; b++) {
            const index_t ow_c = ow_hi - b;
            const bool ok_o = ok_h && ow_c >= 0 && ow_c < OW_;
            const index_t I_OW = ok_o ? ow_c : (index_t)0;
#pragma unroll
            for (int k = 0; k < VEC; k++) {
                const index_t xid = xbase_ + k;
                const index_t rw_ = tw0_ + k - ow_c * SW;
                const bool ok_w = ok_o && rw_ >= 0 && rw_ % DW == 0 && rw_ / DW < KW;
                const index_t I_KW = ok_w ? rw_ / DW : (index_t)0;
                const index_t e_ = (((plane_ * OH_ + I_OH) * OW_ + I_OW) * KH + I_KH) * KW + I_KW;
                (void)xid;
                (void)e_;
#if SC_PROLOGUE
                MJT_SC_VALUE
#else
                const TX val_ = yp[e_];
#endif
                const TACC next_ = (TACC)(COMBINE(acc_[k], val_));
                acc_[k] = ok_w ? next_ : acc_[k];
            }
        }
    }
#if EPI
    float sum_[VEC];
#pragma unroll
    for (int k = 0; k < VEC; k++) sum_[k] = (float)(TX)acc_[k];
    mjt_epi_finish(p, behind_, (MJT_EPI_INDEX)xbase_, sum_);
#else
    mjt_pack<TX, VEC> out_;
#pragma unroll
    for (int k = 0; k < VEC; k++) out_.v[k] = (TX)acc_[k];
    mjt_store(xp + xbase_, out_);
#endif
#endif
}
