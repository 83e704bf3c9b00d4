// Input gradient of a small strided convolution, whole in one launch (python/jittor/nn.py:1251-1262 differentiated; the relay is
// opt/tuner/conv_tuner.cc:375-397):
//   dx[n][c][h][x] = sum over (k, r, s) of dy[n][k][oh][ow] * w[k][c][r][s],  h = oh*SH - PH + r*DH,  x = ow*SW - PW + s*DW
// Supplied by the host: TIN (dy and w), TOUT, LPO (lanes that share a result: a power of two), C_, H_, W_, K_, R_, S_, OH_, OW_ and the geometry.
//
// Bound by latency: a few thousand results.  LPO lanes share one, each takes every LPO-th channel of dy, and which taps reach the result is
// worked out once for all channels; weights and dy are read as they lie.  Phase by phase the same took six launches: the weights rearranged, a
// convolution a phase, the phases woven together.
#ifndef EPI
#define EPI 0
#define EPI_WORDS 0
#endif
struct Params { void* a[4 + EPI_WORDS]; };       // dy, w, dx, number of results

extern "C" __global__ __launch_bounds__(256) void ENTRY(Params p) {
    const TIN* __restrict__ dy = (const TIN*)p.a[0];
    const TIN* __restrict__ w = (const TIN*)p.a[1];
    const int total = (int)(long long)p.a[3];
    const int lane = (int)(blockIdx.x * 256 + threadIdx.x), mine = lane / LPO, part = lane % LPO;
    const int o = mine < total ? mine : total - 1;               // (every lane of a wave takes part in the sum across lanes)
    const int x = o % W_, h = o / W_ % H_, c = o / (W_ * H_) % C_, n = o / (W_ * H_ * C_);
    int at[R_ * S_];                                             // place of the tap's dy inside a plane, or -1
#pragma unroll
    for (int r = 0; r < R_; r++)
#pragma unroll
        for (int s = 0; s < S_; s++) {
            const int th = h + PH - r * DH, tx = x + PW - s * DW;
            at[r * S_ + s] = th >= 0 && tx >= 0 && th % SH == 0 && tx % SW == 0 && th / SH < OH_ && tx / SW < OW_ ? th / SH * OW_ + tx / SW : -1;
        }
    float sum = 0.0f;
    for (int k = part; k < K_; k += LPO) {
        const TIN* const d = dy + (n * K_ + k) * (OH_ * OW_);
        const TIN* const v = w + (k * C_ + c) * (R_ * S_);
#pragma unroll
        for (int t = 0; t < R_ * S_; t++) {
            const float term = (float)d[at[t] < 0 ? 0 : at[t]] * (float)v[t];        // (unconditional loads; a tap that does not reach adds nothing)
            sum += at[t] < 0 ? 0.0f : term;
        }
    }
#pragma unroll
    for (int off = 1; off < LPO; off *= 2) sum += __shfl_xor(sum, off);
    if (part || mine >= total) return;
#if EPI
    mjt_epi_in<1> read;
    mjt_epi_load(p, read, (MJT_EPI_INDEX)o);
    mjt_epi_finish(p, read, (MJT_EPI_INDEX)o, {sum});
#else
    ((TOUT*)p.a[2])[o] = (TOUT)sum;
#endif
}
