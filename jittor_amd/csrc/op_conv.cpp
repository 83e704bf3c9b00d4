// mjt_conv2d_meta: host side of the meta-op convolution (the group
// python/jittor/nn.py:1251-1262 builds; parameters as solved by
// python/jittor/src/opt/tuner/conv_tuner.cc:312-356).
#include "common.h"
#include <array>
#include <cmath>
#include <map>
#include <functional>
#include <mutex>
#include <unordered_map>

namespace mjt {

namespace {
std::mutex g_mu;
std::unordered_map<std::string, JitKernel*> g_kernels;
JitKernel* cached(const std::string& key) {
    std::lock_guard<std::mutex> lock(g_mu);
    auto it = g_kernels.find(key);
    return it == g_kernels.end() ? nullptr : it->second;
}
void remember(const std::string& key, JitKernel* k) {
    std::lock_guard<std::mutex> lock(g_mu);
    g_kernels.emplace(key, k);
}
void* g_wpack = nullptr;
size_t g_wpack_bytes = 0;
void* g_wgrad_part = nullptr;      // per-slice partial weight gradients (its own buffer: the reduce that folds them uses the arena)
size_t g_wgrad_bytes = 0;
// column matrices of a chunk of images; float32 copy of a bfloat16 result; for the input gradient: rearranged weights,
// and dy spread out with zeros or the results of the stride phases
// [4]: weights with rows padded to 16 bytes for the product; [5]: the product of a whole batch, channels outermost
void* g_conv_scratch[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
size_t g_conv_scratch_bytes[6] = {0, 0, 0, 0, 0, 0};

void forget() {
    std::lock_guard<std::mutex> lock(g_mu);
    for (auto& kv : g_kernels)
        if (kv.first.size() > 5 && kv.first.compare(kv.first.size() - 5, 5, "|pack") == 0) delete kv.second;   // shares its module with the main kernel
    g_kernels.clear();                                  // the kernels themselves belong to the run-time compiler's cache
    if (!ctx().dry_run) {
        if (g_wpack) (void)hipFree(g_wpack);
        if (g_wgrad_part) (void)hipFree(g_wgrad_part);
        for (void* b : g_conv_scratch)
            if (b) (void)hipFree(b);
    }
    g_wpack = g_wgrad_part = nullptr;
    g_wpack_bytes = g_wgrad_bytes = 0;
    for (int i = 0; i < 6; i++) {
        g_conv_scratch[i] = nullptr;
        g_conv_scratch_bytes[i] = 0;
    }
}
const bool g_registered = (at_shutdown(&forget), true);

// One of the two growing buffers of the GEMM path.
void* conv_scratch(int which, size_t bytes) {
    Context& c = ctx();
    if (c.dry_run) return (void*)(uintptr_t)0x1000;
    if (bytes > g_conv_scratch_bytes[which]) {
        kept_buffer_moved();
        if (g_conv_scratch[which]) {
            HIP_CHECK(hipStreamSynchronize(c.stream));
            HIP_CHECK(hipFree(g_conv_scratch[which]));
            g_conv_scratch[which] = nullptr;
            g_conv_scratch_bytes[which] = 0;
        }
        HIP_CHECK(hipMalloc(&g_conv_scratch[which], bytes));
        g_conv_scratch_bytes[which] = bytes;
    }
    return g_conv_scratch[which];
}
}  // namespace

void matmul_impl(const mjt_tensor* a, const mjt_tensor* b, const mjt_tensor* c, int trans_a, int trans_b, bool share_a);
bool matmul_available();
void gemm_launch(int in_dtype, int out_dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                 int64_t lda, int64_t ldb, int64_t ldc, int64_t sa, int64_t sb, int64_t sc, int64_t batch, bool a_kcont,
                 bool b_kcont, int tile_m = 0, int tile_n = 0, bool allow_direct = true);
bool gemm_pixels(int in_dtype, int out_dtype, const void* A, const void* x, void* y, int64_t M, int64_t K, int64_t P, int64_t images, bool a_kcont);

// ---- depthwise convolution (kernels/conv_depthwise.h) ----------------------------------
namespace {
struct DepthwiseShape {                       // see the kernel's header: staged planes H x W, strips in planes of OH x OW
    int64_t H, W, OH, OW, R, S, SH, SW, PH, PW, DH, DW, UH, UW, K, mult;
    bool flip;
};
struct DepthwisePlan {
    int64_t TH, NTILE, PPW, VEC, STVEC, RS;
};
constexpr int kDwCW = 4, kDwRS = 4;           // a lane's strip: 4 columns (16 bytes of float32) x at most 4 rows

// Tile and vector widths, or false when the shape does not fit: at most 49 taps (they live in registers) and a window of
// strip rows that fits LDS.  A workgroup stages whole planes while one is at most 40 KB (four workgroups or more then share a
// compute unit and one loads while another computes), else rows of one plane; small planes together, as many as give every
// lane a strip, as long as 512 workgroups are left.
bool depthwise_plan(const DepthwiseShape& g, int in_size, int strip_size, const void* x, const void* strips, int64_t planes, int64_t most_ppw, DepthwisePlan* out) {
    if (g.R * g.S > 49 || g.PH < 0 || g.PW < 0 || g.H * g.W >= (int64_t(1) << 31) || g.OH * g.OW >= (int64_t(1) << 31)) return false;
    const int64_t ncg = (g.OW + kDwCW - 1) / kDwCW;
    const int64_t nv = ((kDwCW - 1) * g.SW + (g.S - 1) * g.DW + 1 + 3) / 4;
    const int64_t lc = ((ncg - 1) * kDwCW * g.SW + nv * 4 + 3) / 4 * 4;
    if (nv > 8) return false;
    auto bytes = [&](int64_t th) { return (((th + kDwRS - 1) / kDwRS * kDwRS - 1) * g.SH + (g.R - 1) * g.DH + 1) * lc * 4; };
    int64_t th = g.OH;
    while (th > kDwRS && bytes(th) > 40 * 1024) th = ((th + 1) / 2 + kDwRS - 1) / kDwRS * kDwRS;
    if (bytes(th) > 60 * 1024) return false;
    // a plane or so a call: rows of it for as many workgroups (forward float32, 1 x 32 x 56 x 56 3x3: 3.4 / 2.9 us)
    while (th > 8 && planes * ((g.OH + th - 1) / th) < 128) th = ((th + 1) / 2 + kDwRS - 1) / kDwRS * kDwRS;
    out->TH = th;
    out->NTILE = (g.OH + th - 1) / th;
    int64_t ppw = 1;
    if (out->NTILE == 1) {
        ppw = 256 / (((th + kDwRS - 1) / kDwRS) * ncg);
        if (ppw > 40 * 1024 / bytes(th)) ppw = 40 * 1024 / bytes(th);
        if (ppw > planes / 512) ppw = planes / 512;
        if (ppw > most_ppw) ppw = most_ppw;
        if (ppw < 1) ppw = 1;
    }
    out->PPW = ppw;
    // Few small planes leave most lanes without a strip of 4 rows, and each of those with all the work: shorter strips then (forward
    // float32, us with 4 rows / as chosen: 16 x 128 x 7 x 7 5x5 4.1 / 2.9; 4 x 512 x 14 x 14 3x3 stride 2 3.4 / 3.2)
    out->RS = kDwRS;
    while (out->RS > 1 && ppw * ((th + out->RS - 1) / out->RS) * ncg < 48) out->RS /= 2;
    int64_t vec = 16 / in_size;
    while (vec > 1 && (g.W % vec || (uintptr_t)x % (size_t)(vec * in_size))) vec /= 2;
    out->VEC = vec;
    int64_t sv = kDwCW;
    while (sv > 1 && (g.OW % sv || (uintptr_t)strips % (size_t)(sv * strip_size))) sv /= 2;
    out->STVEC = sv;
    return true;
}

JitKernel* depthwise_kernel(int mode, const DepthwiseShape& g, const DepthwisePlan& q, int tin, int tout) {
    std::ostringstream key;
    key << "dw|" << mode << "|" << tin << "|" << tout << "|" << g.H << "|" << g.W << "|" << g.OH << "|" << g.OW << "|" << g.R << "|" << g.S << "|" << g.SH << "|" << g.SW
        << "|" << g.PH << "|" << g.PW << "|" << g.DH << "|" << g.DW << "|" << g.UH << "|" << g.UW << "|" << g.K << "|" << g.mult << "|" << g.flip << "|" << q.TH << "|" << q.RS << "|"
        << q.PPW << "|" << q.VEC << "|" << q.STVEC;
    JitKernel* k = cached(key.str());
    if (k) return k;
    std::ostringstream name;
    name << (mode == 2 ? "mjt_conv_backward_direct_" : mode ? "mjt_conv_wgrad_direct_" : "mjt_conv_direct_") << mjt_dtype_name(tin);
    if (mode != 1) name << "_" << mjt_dtype_name(tout);
    name << "_depthwise_" << g.H << "x" << g.W << "_r" << g.R << "x" << g.S << "_s" << g.SH << "x" << g.SW << "_p" << g.PH << "x" << g.PW << "_d" << g.DH
         << "x" << g.DW << "_u" << g.UH << "x" << g.UW << (g.flip ? "_flip" : "") << (g.mult > 1 ? "_m" + std::to_string(g.mult) : std::string()) << "_g" << g.K / g.mult;
    std::ostringstream src;
    src << "#define ENTRY " << name.str() << "\n#define MODE " << mode << "\n#define TIN " << dtype_cname(tin) << "\n#define TOUT " << dtype_cname(tout) << "\n#define H_ " << g.H
        << "\n#define W_ " << g.W << "\n#define OH_ " << g.OH << "\n#define OW_ " << g.OW << "\n#define R_ " << g.R << "\n#define S_ " << g.S << "\n#define SH " << g.SH
        << "\n#define SW " << g.SW << "\n#define PH " << g.PH << "\n#define PW " << g.PW << "\n#define DH " << g.DH << "\n#define DW " << g.DW << "\n#define UH " << g.UH
        << "\n#define UW " << g.UW << "\n#define MULT " << g.mult << "\n#define K_ " << g.K << "\n#define FLIP " << (g.flip ? 1 : 0) << "\n#define TH " << q.TH
        << "\n#define NTILE " << q.NTILE << "\n#define PPW " << q.PPW << "\n#define VEC " << q.VEC << "\n#define CW " << kDwCW << "\n#define RS " << q.RS
        << "\n#define STVEC " << q.STVEC << "\n";
    src << embedded_source("prelude.h") << "\n" << embedded_source("conv_depthwise.h") << "\n";
    k = jit_get(src.str(), name.str());
    remember(key.str(), k);
    return k;
}

// y[planes of OH x OW] = convolution of x[planes of H x W] (or, with flip, the input gradient); false: not covered
bool depthwise_run(const DepthwiseShape& g, const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y) {
    const int64_t planes = y->shape[0] * y->shape[1];
    DepthwisePlan q;
    if (getenv("MJT_NO_FASTPATH") ||
        !depthwise_plan(g, dtype_size(x->dtype), dtype_size(y->dtype), x->ptr, y->ptr, planes, g.mult == 1 ? planes : 1, &q))
        return false;
    const int64_t blocks = (planes + q.PPW - 1) / q.PPW * q.NTILE;
    if (blocks >= (int64_t(1) << 31)) return false;
    JitKernel* k = depthwise_kernel(0, g, q, x->dtype, y->dtype);
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(w->ptr), bits_of_ptr(y->ptr), (uint64_t)planes, 0, 0, 0};
    jit_launch(k, (unsigned)blocks, 1, 256, 0, a);
    return true;
}
}  // namespace

// The first layer of a network, few channels and long rows of taps at horizontal stride 2, from windows in LDS (kernels/conv_stem.h).  False: not covered.
static bool conv_stem(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = w->shape[0], R = w->shape[2], S = w->shape[3], OH = y->shape[2], OW = y->shape[3], SH = p->stride_h, PH = p->pad_h, PW = p->pad_w, DH = p->dil_h;
    const int in = x->dtype == MJT_BFLOAT16 ? 0 : x->dtype == MJT_FLOAT16 ? 1 : 2;
    const int64_t esz = dtype_size(x->dtype), shift = PW & 1, steps = (C * R + 1) / 2, parts = in == 2 ? 3 : 1;
    const bool narrow = y->dtype != MJT_FLOAT32;
    if (p->stride_w != 2 || (p->dil_w != 1 && S > 1) || S + shift > 8 || steps * parts > 36 || getenv("MJT_CONV_NO_IGEMM")) return false;
    // (a row of taps is 8 places of the sum whatever S is: half of them at least are to be taps)
    if (2 * C * R * S < 16 * steps || numel(x) * esz >= (int64_t(1) << 31) || H > 8192 || W > 4096 || PH > 64 || PW > 64 || SH > 8 || (R - 1) * DH > 64 || (uintptr_t)x->ptr % 16) return false;
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    // float32 and more than 32 channels: a workgroup's way to its weights costs a few tiles more than it gives (us, gather / this: 1 x 224 x 224 -> 64 10.4 /
    // 14.6, 4 x 96 x 96 -> 48 10.7 / 12.7, 2 x 224 x 224 -> 64 15.4 / 15.7, 3 x 224 x 224 19.9 / 19.2, 4 x 224 x 224 24.3 / 19.7; up to 32 channels 4 x 160 x 160 -> 16
    // 14.4 / 11.5, 3 x 48 x 48 -> 17 10.2 / 9.0; bfloat16 1 x 224 x 224 -> 64 9.6 / 8.8, 4 x 128 x 128 -> 32 9.1 / 5.8).
    if (in == 2 && K > 32 && (N * OH * OW + 63) / 64 * ((K + 63) / 64) < 2 * cus) return false;
    const int64_t KH = K > 32 ? 2 : 1, kblocks = (K + 32 * KH - 1) / (32 * KH), waves = 4 / KH, unit = W % 4 == 0 ? 4 : W % 2 == 0 ? 2 : 1;
    const int64_t lp = (PW + shift + 3) / 4 * 4, pitch = (std::max(lp + W, lp - PW - shift + 2 * OW + 6) + 3) / 4 * 4;
    // Rows of a tile and tiles of a workgroup by what they are estimated to take, in cycles: a wave's 32 pixels their MFMAs and 300, a tile
    // its values' way to LDS and 1000, a workgroup 6000 for the weights; two workgroups share a compute unit in 1.6 times the time of one.
    int64_t TR = 0, per = 1;
    double best = 1e300;
    for (int64_t tr = 1; tr <= 8 && tr <= OH; tr++) {
        const int64_t xr = (tr - 1) * SH + (R - 1) * DH + 1, units = C * xr * (W / unit), ni = (units + 255) / 256;
        const int64_t lds = std::max(parts * C * xr * pitch * 2, 32 * KH * (C * R * S | 1) * 4);
        if (lds > 78 * 1024 || ni * std::max<int64_t>(1, unit * esz / 4) > 40) continue;
        const int64_t pts = (tr * OW + 31) / 32, tiles = N * ((OH + tr - 1) / tr);
        const double tile = (double)((pts + waves - 1) / waves) * (double)(steps * (in == 2 ? 6 : 1) * 32 + 300) + 1000.0 + (double)(ni * unit) * (in == 2 ? 40.0 : 15.0);
        for (int64_t n = 1; n <= 16 && n <= tiles; n++) {
            const int64_t wgs = (tiles + n - 1) / n * kblocks;
            const double t = wgs <= cus ? 6000.0 + (double)n * tile : std::ceil((double)wgs / (2 * cus)) * 1.6 * (6000.0 + (double)n * tile);
            if (t < best) { best = t; TR = tr; per = n; }
        }
    }
    if (TR == 0) return false;
    const int64_t tiles = N * ((OH + TR - 1) / TR), grid = (tiles + per - 1) / per * kblocks;
    if (tiles >= (1 << 28) || grid >= (1 << 28)) return false;
    const EpilogueCode ep = epilogue_code(1, 6, y->dtype, numel(y));
    std::ostringstream key;
    key << "stem|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << SH << "|" << PH << "|" << PW << "|" << DH << "|" << in << narrow << "|" << TR << ep.key;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_igemm_" << mjt_dtype_name(x->dtype) << (y->dtype != x->dtype ? "_of32" : "") << "_stem_c" << C << "_k" << K << "_r" << R << "x" << S << "_s" << SH << "x2_p" << PH << "x" << PW << "_d"
             << DH << "x1_rows" << TR << "_" << H << "x" << W << ep.suffix();
        std::ostringstream src;
        src << ep.defs << "#define ENTRY " << name.str() << "\n#define IN " << in << "\n#define Y_16 " << narrow << "\n#define TR " << TR << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W
            << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH << "\n#define OW_ " << OW << "\n#define SH " << SH << "\n#define PH " << PH
            << "\n#define PW " << PW << "\n#define DH " << DH << "\n";
        src << embedded_source("split.h") << "\n" << embedded_source("conv_stem.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0) {
        if (ep.on) check_no_epilogue();                     // (the convolution without the group is the better one)
        return false;
    }
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(w->ptr), bits_of_ptr(y->ptr), (uint64_t)N, (uint64_t)per, (uint64_t)(numel(x) * esz)};
    a.insert(a.end(), ep.words.begin(), ep.words.end());
    epilogue_taken(ep);
    jit_launch(k, (unsigned)grid, 1, 256, 0, a);
    set_last_kernel(k->name.c_str());
    return true;
}

// The layout that kernels/conv_strided.h and conv_dgrad_phases.h keep in LDS: outputs or base positions of images of P in rows of W, in planes of PR x PC with
// the margins that the taps' shifts reach (rlo .. rhi, clo .. chi; `left` columns ahead of a row), loaded `unit` positions at a time.
struct MarginPlanes {
    int64_t total, P, W, PR, PC, rlo, rhi, clo, chi, left, unit;
    // The most positions between the first and the last that a tile of `tile` outputs reads.  Tiles begin at the same places of an image again after P of
    // them, which a call would have to walk over (us of host time a call: 64 x 32 x 224 x 224 stride 2 256 forward, 98 input gradient), so what was
    // found is kept.
    int64_t span(int64_t tile) const {
        static std::mutex mu;
        static std::map<std::array<int64_t, 12>, int64_t> kept;
        const int64_t tiles = std::min((total + tile - 1) / tile, P);
        const std::array<int64_t, 12> key{tile, tiles, P, W, PR, PC, rlo, rhi, clo, chi, left, unit};
        {
            std::lock_guard<std::mutex> lock(mu);
            auto it = kept.find(key);
            if (it != kept.end()) return it->second;
        }
        auto pos = [&](int64_t f) { return (f / P * PR + f % P / W - rlo) * PC + f % W + left; };
        int64_t most = 0;
        for (int64_t t = 0; t < tiles; t++) most = std::max(most, pos(t * tile + tile - 1) + rhi * PC + chi + 1 - (pos(t * tile) + rlo * PC + clo) / unit * unit);
        most = (most + unit - 1) / unit * unit;
        std::lock_guard<std::mutex> lock(mu);
        if (kept.size() >= 1024) kept.clear();
        kept.emplace(key, most);
        return most;
    }
};

// Convolutions of 16-bit operands with horizontal stride 2 from windows in LDS (kernels/conv_strided.h), for shapes that the row kernel takes too.  False: not
// covered, or the row kernel is the faster one: more than one tap on maps of less than 100 pixels, whose tiles hold mostly margins, or on more tiles than
// compute units.  us, row kernel / this: 32 x 256 x 14 x 14 3x3 -> 256 20.7 / 22.3, 32 x 128 x 14 x 14 5x5 -> 128 17.9 / 21.4, 64 x 512 x 14 x 14 3x3 -> 512 45.0 / 56.4, 64 x 128 x
// 56 x 56 3x3 -> 128 34.5 / 36.8; on this side 1 x 64 x 32 x 32 3x3 -> 128 18.0 / 9.5, 2 x 512 x 28 x 28 3x3 -> 128 72.3 / 35.6, 64 x 32 x 28 x 28 5x5 -> 128 16.6 / 12.8; single
// taps 64 x 256 x 28 x 28 -> 512 32.1 / 18.9, 64 x 512 x 14 x 14 -> 512 24.7 / 17.6, 64 x 64 x 32 x 32 -> 128 16.2 / 14.1.
// `packed`, `pack_mode`: as below; the packed weights are as many bytes as w.
static bool conv_strided(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p, void* packed, int pack_mode) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = w->shape[0], R = w->shape[2], S = w->shape[3], OH = y->shape[2], OW = y->shape[3], taps = R * S;
    const int64_t SH = p->stride_h, PH = p->pad_h, PW = p->pad_w, DH = p->dil_h, DW = p->dil_w;
    const bool half = x->dtype == MJT_FLOAT16, narrow = y->dtype == x->dtype;
    if (!(half || x->dtype == MJT_BFLOAT16) || p->stride_w != 2 || SH > 2 || taps < 1 || taps > 25) return false;
    if (numel(x) < 1 || numel(x) * 2 >= (int64_t(1) << 31) || numel(y) >= (int64_t(1) << 31) || H > 4096 || W > 4096 || PH > 64 || PW > 64 || (R - 1) * DH > 64 || (S - 1) * DW > 64 || (uintptr_t)x->ptr % 4 || W % 2 || C % 32 || (taps > 1 && OH * OW < 100))
        return false;
    // the kernel's layout: margins that the taps' shifts reach, row phases of x that are read, and the positions between the first and the last that a tile reads
    auto floor_of = [](int64_t a, int64_t b) { return a >= 0 ? a / b : -((b - 1 - a) / b); };
    int64_t rlo = 0, rhi = 0, clo = 0, chi = 0;
    bool phase[2] = {false, false};
    for (int64_t r = 0; r < R; r++) {
        const int64_t d = floor_of(r * DH - PH, SH);
        phase[r * DH - PH - SH * d] = true;
        rlo = std::min(rlo, d);
        rhi = std::max(rhi, d);
    }
    for (int64_t s = 0; s < S; s++) {
        const int64_t d = floor_of(s * DW - PW, 2);
        clo = std::min(clo, d);
        chi = std::max(chi, d);
    }
    const int64_t PR = OH + rhi - rlo, PC = OW + chi - clo, P = OH * OW, total = N * P, nrp = phase[0] && phase[1] ? 2 : 1;
    if (N * PR * PC >= (int64_t(1) << 30)) return false;
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    if (taps > 1 && (total + 127) / 128 * (K / (K % 128 == 0 ? 128 : K % 64 == 0 ? 64 : 32)) > cus) return false;      // (the fewest tiles there are)
    const MarginPlanes planes{total, P, OW, PR, PC, rlo, rhi, clo, chi, -clo, 1};
    const int64_t spans[2] = {planes.span(64), planes.span(128)};
    const int64_t KU = taps >= 6 ? 1 : taps >= 3 || C % 64 ? 2 : 4, stages = C / (16 * KU);      // (C is a multiple of 32)
    // Channels and positions of a workgroup by what a stage is estimated to take: its operands' way out of LDS and the next stage's way in, at 128
    // bytes a cycle, and 400 cycles for its barrier and what nothing hides.
    int64_t WK = 0, PT = 0, span = 0;
    double best = 1e300;
    for (int64_t wk = K % 64 ? 1 : 2; wk <= 4 && K % (32 * wk) == 0; wk *= 2)
        for (int64_t pt = 1; pt <= 2; pt++) {
            const int64_t sp = spans[pt - 1], stage_bytes = KU * (taps * wk * 1024 + nrp * 2 * sp * 32);
            if (2 * stage_bytes > 160 * 1024 || (sp * nrp * 2 * KU + 128 * wk - 1) / (128 * wk) > 6) continue;
            const int64_t wgs = (total + 64 * pt - 1) / (64 * pt) * (K / (32 * wk));
            const double t = std::ceil((double)wgs / cus) * ((double)(2 * wk * KU * taps * (1 + pt) * 1024 + stage_bytes) / 128 + 400.0);
            if (t < best) { best = t; WK = wk; PT = pt; span = sp; }
        }
    if (WK == 0) return false;
    const int64_t KB = K / (32 * WK), bytes = numel(w) * 2, tiles = (total + 64 * PT - 1) / (64 * PT) * KB;
    if (bytes >= (int64_t(1) << 31) || tiles >= (1 << 28) || (taps > 1 && tiles > cus)) return false;
    std::ostringstream key;
    key << "strided|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << SH << "|" << PH << "|" << PW << "|" << DH << "|" << DW << "|" << half << narrow << "|"
        << PT << "|" << WK << "|" << span;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_mfma_" << (half ? "f16" : "bf16") << "_strided_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << SH << "x2_p" << PH << "x" << PW << "_d" << DH << "x" << DW
             << "_o" << (narrow ? (half ? "f16" : "bf16") : "f32") << "_t" << 32 * WK << "x" << 64 * PT;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define IN_F16 " << half << "\n#define Y_16 " << narrow << "\n#define KU " << KU << "\n#define PT " << PT << "\n#define WK " << WK << "\n#define SPAN " << span
            << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH
            << "\n#define OW_ " << OW << "\n#define SH " << SH << "\n#define PH " << PH << "\n#define PW " << PW << "\n#define DH " << DH << "\n#define DW " << DW << "\n";
        src << embedded_source("conv_strided.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0) return false;
    if (pack_mode) MJT_CHECK(packed && (uintptr_t)packed % 16 == 0, "conv: packed weights must be a 16-byte aligned device buffer");
    void* wbuf = pack_mode ? packed : conv_scratch(2, (size_t)bytes);
    if (pack_mode != 2) {
        mjt_tensor tw;
        memset(&tw, 0, sizeof(tw));
        tw.ptr = wbuf;
        tw.dtype = w->dtype;
        for (int64_t e : {KB, stages, KU, taps, int64_t(2), 32 * WK, int64_t(8)}) tw.shape[tw.ndim++] = e;
        const std::string ks = "i0*" + std::to_string(32 * WK) + "+i5", cs = "i1*" + std::to_string(16 * KU) + "+i2*16+i4*8+i6", rs = "i3/" + std::to_string(S), ss = "i3%" + std::to_string(S);
        const char* idx[4] = {ks.c_str(), cs.c_str(), rs.c_str(), ss.c_str()};
        if (mjt_reindex(w, &tw, 4, idx, 0.0, 0, nullptr, 0, nullptr) != MJT_OK) MJT_FAIL(MJT_ERR_DEVICE, "conv: packing the weights failed: " << mjt_last_error());
    }
    if (pack_mode == 1) {
        set_last_kernel((k->name + "_pack").c_str());
        return true;
    }
    std::vector<uint64_t> a{bits_of_ptr(wbuf), bits_of_ptr(x->ptr), bits_of_ptr(y->ptr), (uint64_t)N, (uint64_t)(numel(x) * 2), (uint64_t)bytes};
    jit_launch(k, (unsigned)((tiles + 7) / 8 * 8), 1, (unsigned)(128 * WK), 0, a);
    set_last_kernel(k->name.c_str());
    return true;
}

// free_extent: y's rows and columns are taken as they are instead of checked against the extents that stride, padding and
// taps give (output (oh, ow) reads x around (oh*sh - ph, ow*sw - pw) whatever oh and ow; outside the image x is 0): what the
// stride phases of an input gradient need, whose zero margins differ between the two ends of an axis.
// packed / pack_mode: 0 the call packs the weights itself (into the library's buffer) and runs; 1 it only packs them
// into `packed`; 2 it runs on weights packed by an earlier call of mode 1 for the same shapes and parameters.  Modes 1
// and 2 exist for the MFMA kernel only and fail with MJT_ERR_UNSUPPORTED for a convolution that takes another route.
// flipped: w [K,C,R,S] is still to be written, by fill(): it is the transpose of forward [C,K,R,S] with the taps from the last to the first
// (an input gradient).  The MFMA kernel packs it from there in one pass (256 x 256 x 3 x 3 bfloat16, us: transposed 5.0 and packed 4.8, 4.8 so);
// the other routes have it filled in first.
struct FlippedWeights {
    const mjt_tensor* forward;
    std::function<void()> fill;
};
static void conv_run(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p, int64_t G, bool free_extent,
                     int pack_mode, void* packed, const FlippedWeights* flipped) {
    auto need_weights = [&] {
        if (flipped) flipped->fill();
        flipped = nullptr;
    };
    require_init();
    check_tensor(x, "conv x");
    check_tensor(w, "conv w");
    check_tensor(y, "conv y");
    MJT_CHECK(p, "conv: null parameters");
    MJT_CHECK(x->ndim == 4 && w->ndim == 4 && y->ndim == 4, "conv: x, w and y must have rank 4");
    MJT_CHECK(x->dtype == w->dtype && (x->dtype == MJT_BFLOAT16 || x->dtype == MJT_FLOAT16 || x->dtype == MJT_FLOAT32),
              "conv: x and w must both be bfloat16, float16 or float32");
    MJT_CHECK(y->dtype == MJT_FLOAT32 || y->dtype == x->dtype, "conv: y must be float32 or the input dtype");
    MJT_CHECK(G >= 1, "conv: groups must be >= 1, got " << G);
    // C is the number of channels one output channel sees: all of x's, or those of its group
    const int64_t N = x->shape[0], C = w->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = w->shape[0], R = w->shape[2], S = w->shape[3];
    MJT_CHECK(x->shape[1] == C * G, "conv: weight channels " << C << " x " << G << " group(s) != input channels " << x->shape[1]);
    MJT_CHECK(K % G == 0, "conv: " << K << " output channels do not divide into " << G << " groups");
    MJT_CHECK(p->stride_h >= 1 && p->stride_w >= 1 && p->dil_h >= 1 && p->dil_w >= 1 && p->pad_h >= 0 && p->pad_w >= 0,
              "conv: bad stride / padding / dilation");
    const int64_t OH = free_extent ? y->shape[2] : (H + 2 * p->pad_h - p->dil_h * (R - 1) - 1) / p->stride_h + 1;
    const int64_t OW = free_extent ? y->shape[3] : (W + 2 * p->pad_w - p->dil_w * (S - 1) - 1) / p->stride_w + 1;
    MJT_CHECK(OH >= 1 && OW >= 1, "conv: empty output");
    MJT_CHECK(y->shape[0] == N && y->shape[1] == K && y->shape[2] == OH && y->shape[3] == OW,
              "conv: y shape " << shape_str(y) << " != [" << N << "," << K << "," << OH << "," << OW << "]");
    if (N == 0 || K == 0) return;
    MJT_CHECK(numel(x) < (int64_t(1) << 40) && numel(y) < (int64_t(1) << 40), "conv: too large");
    Context& c = ctx();

    if (R * S == 1 || G > 1 || p->stride_h > 1 || p->stride_w > 1) need_weights();
    // a 1x1 convolution on large enough planes of an even number of pixels: one product for the batch, x read as it lies
    if (G == 1 && R == 1 && S == 1 && p->stride_h == 1 && p->stride_w == 1 && p->pad_h == 0 && p->pad_w == 0 && OH == H && OW == W && pack_mode == 0 &&
        !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_NO_GEMM") && !getenv("MJT_CONV_FLAT") && (double)N * K * C * H * W >= (double)(1 << 22) &&
        gemm_pixels(x->dtype, y->dtype, w->ptr, x->ptr, y->ptr, K, C, H * W, N, true)) {
        set_last_kernel("conv_as_gemm");
        return;
    }

    std::ostringstream geo;
    geo << "#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R
        << "\n#define S_ " << S << "\n#define OH_ " << OH << "\n#define OW_ " << OW << "\n#define SH " << p->stride_h
        << "\n#define SW " << p->stride_w << "\n#define PH " << p->pad_h << "\n#define PW " << p->pad_w << "\n#define DH "
        << p->dil_h << "\n#define DW " << p->dil_w << "\n";

    // ---- MFMA path ----------------------------------------------------------------
    const int64_t WPX = 2;                                  // pixel halves per workgroup (1: one wave per SIMD with 224-pixel wave tiles, 224-227 us on the 3x3 256-channel 56x56 layer against 215)
    const int64_t max_px = WPX == 1 ? 224 : 112;            // pixels per wave: 16 per accumulator tile
    const int64_t WPS = max_px == 224 ? 1 : 2;              // waves per SIMD the register budget is set for
    // output channels per wave: 16 per accumulator-tile row; per workgroup: up to 256
    const int64_t Kg = K / G;                                // output channels of one group: the K of the MFMA kernel
    // accumulator-tile rows (of 16 output channels) per wave: 4; 2 for groups of 64 or 128 output channels, which then have four
    // waves share an input tile instead of two (64 x 64 x 56 x 56 3x3 -> 64: 42.9 -> 31.7 us; 64 x 256 x 56 x 56 -> 64:
    // 124 -> 86; 64 x 64 x 28 x 28 -> 64: 20.8 -> 14.3)
    // (groups of 128: eight waves of 32 channels instead of four of 64: 64 x 128 x 28 x 28 3x3 -> 128: 25.4 -> 24.6 us,
    // with 8 images 23.0 -> 18.4)
    int64_t MT = Kg == 32 || Kg == 64 || Kg == 128 ? 2 : 4;
    auto widest = [&]() {                                   // groups of output channels per workgroup: up to 256 channels, eight waves
        const int64_t v = Kg % 256 == 0 ? 256 / (16 * MT) : Kg % 128 == 0 ? 128 / (16 * MT) : Kg % 64 == 0 ? 64 / (16 * MT) : 32 / (16 * MT);
        return v > 4 ? int64_t(4) : v;
    };
    int64_t WKO = widest();
    // LDS: two buffers of input rows (one block of CB channels each), a ring of NS weight slabs (64 bytes per output
    // channel of the workgroup each) and a spare KB that takes the writes of idle lanes.  Blocks of 32 channels
    // leave room for a deeper ring, which is what hides the latency of the slabs; the ring needs three slabs at least.
    const int64_t lds_total = 160 * 1024;
    const int64_t CBLK = 32;
    const int64_t slab0 = 64 * 16 * MT * WKO, spare0 = 1024;
    const int64_t tile_limit = (lds_total - 4 * slab0 - spare0) / 2;         // leaves room for four slabs of the widest workgroup
    int64_t TRW = OW <= max_px ? max_px / OW : 0;
    if (TRW > OH) TRW = OH;
    while (TRW > 1 && WPX * TRW > OH && (OH % (WPX * TRW)) != 0 && (WPX * (TRW - 1)) >= OH) TRW--;
    auto lds_rows = [&](int64_t trw) { return (WPX * trw - 1) * p->stride_h + (R - 1) * p->dil_h + 1; };
    const int64_t LCOLS = (OW - 1) * p->stride_w + (S - 1) * p->dil_w + 1 > W + 2 * p->pad_w
                              ? (OW - 1) * p->stride_w + (S - 1) * p->dil_w + 1
                              : W + 2 * p->pad_w;
    while (TRW > 1 && lds_rows(TRW) * LCOLS * CBLK * 2 > tile_limit) TRW--;
    const int64_t NT = TRW ? (TRW * OW + 15) / 16 : 0;
    const int64_t LROWS = lds_rows(TRW);
    {
        // fewer output channels per workgroup while the grid would leave compute units idle (small maps, small batches):
        // the same input tile is then staged by more workgroups, which the L2 absorbs
        const int64_t cus0 = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
        const int64_t tile_rows = WPX * (TRW > 0 ? TRW : 1);
        const int64_t min_ranges = N * ((OH + tile_rows - 1) / tile_rows);
        // (down to 128 channels per workgroup, four waves, never to workgroups of two waves: 64 x 256 x 14 x 14 3x3 -> 256 on 128
        // workgroups of four waves 48 us, on 256 of two waves 61, on 64 of eight 65; with 8 images 48 against 58)
        const int64_t before = WKO;
        while (WKO > 2 && 2 * min_ranges * (Kg / (16 * MT * WKO)) <= cus0) WKO /= 2;
        // such a small grid with more channels: wave tiles of 32 channels as well, so that twice as many workgroups of four
        // waves share the work (64 x 256 x 14 x 14 3x3 -> 256: 48 -> 39 us; 64 x 256 x 14 x 14 3x3 stride 2 -> 512: 42 -> 37)
        if (WKO < before && MT == 4) {
            MT = 2;
            WKO = widest();
            while (WKO > 2 && 2 * min_ranges * (Kg / (16 * MT * WKO)) <= cus0) WKO /= 2;
        }
    }
    const bool half = x->dtype == MJT_FLOAT16;
    // Small maps with long sums that the MFMA kernel below does not take (7 x 7 and 13 x 13 maps: odd widths): one
    // product for the whole batch, y'[K][N * P] = w [K][C*R*S] x cols [C*R*S][N * P], on column matrices with the images
    // side by side, then y' -> y [N][K][P] by one permutation.  The gather of the implicit GEMM is paid once per 64 or
    // 128 output channels, the column matrices once (us, bf16, gather / per-image column matrices / this:
    // 64 x 512 x 7 x 7 3x3 -> 512: 126 / 85 / 60; 64 x 256 x 13 x 13 3x3 -> 384: 76 / 103 / 69; 1x1 on 7 x 7 maps,
    // gather / this: 2048 -> 512: 60 / 35; 1024 -> 1024: 38 / 29; 512 -> 2048: 38 / 31; on 14 x 14: 1024 -> 512: 63 / 51;
    // 512 -> 512: 36 / 36; 1024 -> 256: 36 / 41; short sums, few output channels and larger maps stay with the gather:
    // 64 x 48 x 28 x 28 3x3 -> 96: 35 / 69 / 62; with fewer than 64 tiles of 128 x 128 the per-image matrices win:
    // 32 x 512 x 7 x 7 3x3 -> 512: 70 against 79; where the MFMA kernel applies it wins: 64 x 256 x 14 x 14 3x3 -> 256:
    // 61 against 71).  MJT_CONV_FLAT=1 sends every eligible shape this way, =0 none.
    const int64_t esz0 = dtype_size(x->dtype), NP0 = N * OH * OW, CRS0 = C * R * S;
    const bool flat_ok = G == 1 && pack_mode == 0 && esz0 == 2 && !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_NO_GEMM") && matmul_available() &&
                         (NP0 * esz0) % 16 == 0 && (uintptr_t)x->ptr % 16 == 0 && (uintptr_t)y->ptr % 16 == 0 && NP0 < (int64_t(1) << 31) &&
                         CRS0 * NP0 * esz0 <= (int64_t(1) << 30) && CRS0 * esz0 >= 128 && (double)N * K * OH * OW * CRS0 >= (double)(1 << 22);
    const char* flat_env = getenv("MJT_CONV_FLAT");
    const bool flat_forced = flat_ok && flat_env && atoi(flat_env) != 0;
    const bool flat = flat_forced || (flat_ok && !flat_env && OH * OW <= 256 && ((K + 127) / 128) * ((NP0 + 127) / 128) >= 64 &&
                                      ((K >= 512 && CRS0 >= 512) || (K >= 256 && CRS0 >= 2048)));
    // (a grouped convolution is one launch per group on the group's channels: worth it from 32 x 64 channels per group)
    const bool mfma_ok = !flat_forced && (x->dtype == MJT_BFLOAT16 || half) && !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_NO_MFMA") && C % CBLK == 0 && (Kg % 64 == 0 || Kg == 32) && G <= 64 &&
                         W % 2 == 0 && TRW >= 1 && NT <= max_px / 16 && LROWS * LCOLS * CBLK * 2 <= tile_limit &&
                         // tap shift + k-step plane offset of a fragment read must fit the 16-bit offset field
                         ((R - 1) * p->dil_h * LCOLS + (S - 1) * p->dil_w) * 16 + (CBLK == 64 ? 4 * LROWS * LCOLS * 16 : 0) < 65536 &&
                         (uintptr_t)x->ptr % 16 == 0 && (uintptr_t)y->ptr % 16 == 0 && R * S <= 49 &&
                         // byte offsets inside one image and inside the weights are 32-bit in the kernel
                         C * G * H * W * 2 < (int64_t(1) << 31) && K * OH * OW * 4 < (int64_t(1) << 31) && numel(w) * 2 < (int64_t(1) << 31) &&
                         // a 1x1 convolution of stride 1 is a matrix product per image: when the rows of a plane are 16-byte
                         // multiples the product kernel below reads x as it lies and is as fast or faster for every shape
                         // measured (64 x 512 x 28 x 28 -> 128 channels: 22 us against 42; 64 x 256 x 56 x 56 -> 64: 31 against
                         // 73; 64 x 1024 x 16 x 16 -> 2048: 82 against 387; closest 64 x 512 x 28 x 28 -> 512: 74 against 74),
                         // this kernel walking one-step channel blocks.  With other plane sizes the product kernel gathers x
                         // (its CONV mode; long sums have gone to the product over pieces above), which wins with more than 64 output channels and enough 128 x 64 tiles for the chip
                         // (64 x 512 x 14 x 14 -> 512: 36 against 61; 64 x 1024 x 14 x 14 -> 512: 63 against 100; -> 256: 37
                         // against 142) and with many more input than output channels and few output channels or a small map
                         !(R * S == 1 && G == 1 && p->stride_h == 1 && p->stride_w == 1 && matmul_available() && !getenv("MJT_CONV_NO_GEMM") &&
                           ((p->pad_h == 0 && p->pad_w == 0 && OH == H && OW == W && (OH * OW * 2) % 16 == 0 && (uintptr_t)w->ptr % 16 == 0) ||
                            (C >= 4 * K && (K <= 64 || OH * OW <= 256)) ||
                            (K > 64 && !getenv("MJT_CONV_NO_IGEMM") && ((K + 127) / 128) * ((N * OH * OW + 63) / 64) >= 256)));
    if (mfma_ok && G == 1 && !free_extent && !getenv("MJT_ABLATE_CONV") && !getenv("MJT_CONV_RPW") && conv_strided(x, w, y, p, packed, pack_mode)) return;
    if (mfma_ok) {
        // Rows per workgroup: a workgroup walks RPW output rows as NFULL tiles of TR rows plus one
        // shorter tile.  Pick the RPW that minimises (rounds of workgroups over the compute units) x
        // (accumulator tiles a workgroup computes, plus a per-tile overhead worth half a tile column).
        const int64_t TR = WPX * TRW, KPARTS = Kg / (16 * MT * WKO);
        const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
        auto tail_of = [&](int64_t rpw, int64_t* trw_t, int64_t* nt_t) {
            const int64_t t = rpw % TR;
            *trw_t = (t + WPX - 1) / WPX;
            *nt_t = (*trw_t * OW + 15) / 16;
        };
        int64_t RPW = TR;
        {
            // Workgroups of at most four waves whose LDS is at most half a compute unit's run two to a compute unit, each
            // SIMD then holding two waves that fill each other's gaps: a pair gets through its work in 1.4 times the time
            // of one workgroup alone (64 x 64 x 56 x 56 3x3 -> 64: 256 workgroups of 14 rows 29.7 us, 448 of 8 rows 25.1,
            // 896 of 4 rows 28.4; 64 x 256 x 56 x 56 -> 64: 91.9 -> 75.9 us per call).  Such a grid pays for more, shorter
            // workgroups; a workgroup's set-up counts as one accumulator tile there, a short last tile as half a one more.
            const int64_t lds_need = 2 * LROWS * LCOLS * CBLK * 2 + 8 * (64 * 16 * MT * WKO) + 1024;
            const bool pairs = WPX * WKO <= 4 && lds_need <= lds_total / 2;
            double best = 1e300;
            for (int64_t r = TR; r <= OH || r == TR; r++) {
                int64_t trw_t, nt_t;
                tail_of(r, &trw_t, &nt_t);
                const int64_t wgs = N * ((OH + r - 1) / r) * KPARTS;
                const int64_t ntiles = r / TR + (trw_t ? 1 : 0);
                const double work = (double)(r / TR) * NT + nt_t + 0.5 * ntiles;
                double cost;
                if (pairs && wgs > cus)
                    cost = (double)((wgs + 2 * cus - 1) / (2 * cus)) * 1.4 * (work + 1.0 + (trw_t ? 0.5 : 0.0));
                else
                    cost = (double)((wgs + cus - 1) / cus) * work;
                if (cost < best - 1e-9) { best = cost; RPW = r; }
            }
            const char* e = getenv("MJT_CONV_RPW");
            if (e && *e && atoi(e) >= TR) RPW = atoi(e);
        }
        int64_t TAIL_TRW, TAIL_NT;
        tail_of(RPW, &TAIL_TRW, &TAIL_NT);
        const int64_t NFULL = RPW / TR;
        const int64_t TAIL_LROWS = TAIL_TRW ? lds_rows(TAIL_TRW) : 0;
        std::ostringstream key;
        const int64_t slab = 64 * 16 * MT * WKO;
        const int64_t spare = 1024;
        int64_t NSLAB = (lds_total - 2 * LROWS * LCOLS * CBLK * 2 - spare) / slab;
        if (NSLAB > 8) NSLAB = 8;
        MJT_CHECK(NSLAB >= 3, "conv: internal: no room for the weight ring");
        const int stage_depth = 4;                          // steps between asking for an input row and writing it to LDS (2-7: +-2 us)
        const int abl = getenv("MJT_ABLATE_CONV") ? atoi(getenv("MJT_ABLATE_CONV")) : 0;   // timing-only ablations (bench.py --ablate): results are wrong
        MJT_CHECK(abl == 0 || abl == 1 || abl == 2 || abl == 3 || abl == 7 || abl == 16 || abl == 17,
                  "conv: MJT_ABLATE_CONV must be one of 0, 1, 2, 3, 7, 16, 17");
        std::ostringstream geo_g;                        // the kernel's K_ is a group's; XC_ / YK_ are the strides of x and y between images
        geo_g << geo.str() << "#undef K_\n#define K_ " << Kg << "\n#define XC_ " << C * G << "\n#define YK_ " << K << "\n";
        key << "mfma|" << half << "|" << geo_g.str() << TRW << "|" << (y->dtype != MJT_FLOAT32) << "|" << WKO << "|" << WPX << "|" << RPW << "|" << MT << "|" << WPS
            << "|" << stage_depth << "|" << CBLK << "|" << NSLAB << "|" << abl;
        const EpilogueCode ep = epilogue_code(OW % 4 == 0 ? 4 : OW % 2 == 0 ? 2 : 1, 4, y->dtype, numel(y));
        key << ep.key;
        JitKernel* k = cached(key.str());
        JitKernel* kp = cached(key.str() + "|pack");
        if (!k || !kp) {
            std::ostringstream name;
            name << "mjt_conv_mfma_" << (half ? "f16" : "bf16") << "_c" << C << "_k" << Kg << (G > 1 ? "_g" + std::to_string(G) : std::string()) << "_" << H << "x" << W << "_r" << R << "x" << S << "_s"
                 << p->stride_h << "x" << p->stride_w << "_p" << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x"
                 << p->dil_w << "_rows" << RPW << (y->dtype == MJT_FLOAT32 ? "_of32" : half ? "_of16" : "_obf16") << ep.suffix();
            std::ostringstream src;
            src << ep.defs << "#define ENTRY " << name.str() << "\n#define ENTRY_PACK " << name.str() << "_pack\n" << geo_g.str()
                << "#define MT " << MT << "\n#define WKO " << WKO << "\n#define WPX " << WPX << "\n#define TRW " << TRW << "\n#define NT " << NT << "\n#define LROWS " << LROWS << "\n#define LCOLS " << LCOLS
                << "\n#define RPW " << RPW << "\n#define NFULL " << NFULL << "\n#define TAIL_TRW " << TAIL_TRW << "\n#define TAIL_NT "
                << TAIL_NT << "\n#define TAIL_LROWS " << TAIL_LROWS << "\n#define Y_BF16 " << (y->dtype != MJT_FLOAT32 ? 1 : 0) << "\n#define IN_F16 " << (half ? 1 : 0)
                << "\n#define ABL " << abl << "\n#define WPS " << WPS << "\n#define CB " << CBLK << "\n#define NS " << NSLAB << "\n#define STAGE_DEPTH " << stage_depth << "\n";
            src << embedded_source("conv_mfma.h") << "\n";
            k = jit_get(src.str(), name.str());
            kp = new JitKernel();
            kp->name = name.str() + "_pack";
            kp->module = k->module;
            if (!c.dry_run) HIP_CHECK(hipModuleGetFunction(&kp->fn, k->module, kp->name.c_str()));
            remember(key.str(), k);
            remember(key.str() + "|pack", kp);
        }
        // The kernel keeps loads and LDS reads under way in registers behind the compiler's back (it takes a spelled-out load
        // for finished when issued).  That is sound while the compiler moves no register aside; a build that needed more
        // registers than a wave has (accumulation registers beyond the accumulators, scratch memory) may have moved one
        // whose load had not landed, so such a build is not run: the convolution takes the routes below.
        const bool regs_ok = k->spilled == 0 && k->agprs >= 0 && k->agprs <= MT * NT * 4;
        if (!regs_ok && ep.on) check_no_epilogue();           // (the convolution without the group is the better one)
        if (regs_ok) {
            size_t wbytes = (size_t)numel(w) * 2;
            if (pack_mode) MJT_CHECK(packed && (uintptr_t)packed % 16 == 0, "conv: packed weights must be a 16-byte aligned device buffer");
            if (!pack_mode && !c.dry_run && wbytes > g_wpack_bytes) {
                kept_buffer_moved();
                if (g_wpack) {
                    HIP_CHECK(hipStreamSynchronize(c.stream));
                    HIP_CHECK(hipFree(g_wpack));
                }
                HIP_CHECK(hipMalloc(&g_wpack, wbytes));
                g_wpack_bytes = wbytes;
            }
            const int64_t ranges = N * ((OH + RPW - 1) / RPW);
            const int64_t ranges8 = (ranges + 7) / 8 * 8;
            const int64_t blocks = ranges8 * KPARTS;
            MJT_CHECK(blocks < (int64_t(1) << 31), "conv: launch too large");
            const int64_t wg = Kg * C * R * S;               // weights of one group
            int64_t pblocks = (wg + 255) / 256;
            if (pblocks > 2048) pblocks = 2048;
            // one launch for all groups (the group is the grid's second axis)
            char* wdst = (char*)(pack_mode ? packed : g_wpack);
            if (pack_mode != 2) {
                std::vector<uint64_t> pa{bits_of_ptr(flipped ? flipped->forward->ptr : w->ptr), bits_of_ptr(wdst), (uint64_t)(flipped ? 1 : 0), 0};
                pa.resize(4 + ep.words.size());
                Preparing preparing;
                jit_launch(kp, (unsigned)pblocks, (unsigned)G, 256, 0, pa);
            }
            if (pack_mode != 1) {
                std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(wdst), bits_of_ptr(y->ptr), (uint64_t)N};
                a.insert(a.end(), ep.words.begin(), ep.words.end());
                epilogue_taken(ep);
                jit_launch(k, (unsigned)blocks, (unsigned)G, (unsigned)(64 * WPX * WKO), 0, a);
            }
            return;
        }
    }

    if (pack_mode) MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv: this convolution does not run on packed weights (mjt_conv2d_meta takes it)");

    // ---- column matrices x weights on the GEMM kernel -----------------------------------
    // What the MFMA convolution kernel does not take (float32, odd widths, channel counts that are no multiple of 64,
    // tiles that do not fit) and is large enough to matter: y[n] [K, P] = w [K, C*R*S] x cols[n] [C*R*S, P], cols = the
    // shifted input planes written by one reindex per chunk of images (a 1x1 convolution of stride 1 without padding
    // reads x itself), the product on kernels/gemm_mfma.h with the weights shared across the batch.  Rows of cols are
    // padded to a multiple of 16 bytes when the pixel count is not one (the GEMM kernel's fast path wants aligned rows).
    // Small ones with long sums as well: the kernel of one lane a result below walks them in 0.05 (1x1) to 0.1 us a term, the product's
    // kernel in 0.03 behind 3 us, and 3 more where the weights' rows are copied (us, one lane a result / this: float32 4 x 16 x 6 x 6 3x3
    // stride 2 -> 16 10.4 / 7.0, 8 x 39 x 6 x 6 3x3 stride 2 -> 39 26.0 / 12.4, 2 x 256 x 7 x 7 1x1 -> 64 15.6 / 8.7, 1 x 16 x 8 x 8 3x3 -> 16
    // 6.6 / 6.8; float16 2 x 18 x 10 x 10 3x3 -> 16 15.6 / 8.1; bfloat16 1 x 215 x 7 x 7 3x3 -> 17 167 / 15.8; on the other side float32
    // 2 x 8 x 10 x 10 3x3 -> 8 4.6 / 5.7, 3 x 100 x 9 x 9 1x1 -> 100 6.7 / 7.4).
    const int64_t P = OH * OW, CRS = C * R * S;
    const bool long_sum = (x->dtype == MJT_FLOAT32 || x->dtype == MJT_BFLOAT16 || x->dtype == MJT_FLOAT16) &&
                          CRS >= ((CRS * dtype_size(x->dtype)) % 16 || (uintptr_t)w->ptr % 16 ? 160 : 128);
    if (G == 1 && !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_NO_GEMM") && ((double)N * K * P * CRS >= (double)(1 << 22) || long_sum) &&
        P < (int64_t(1) << 31) && CRS < (int64_t(1) << 31) && matmul_available()) {
        if (!flat_forced && !flipped && conv_stem(x, w, y, p)) return;       // (of stride 2)
        const int64_t esz = dtype_size(x->dtype);
        const int64_t Ppad = (P * esz + 15) / 16 * 16 / esz;
        const bool plain = R == 1 && S == 1 && p->stride_h == 1 && p->stride_w == 1 && p->pad_h == 0 && p->pad_w == 0 && Ppad == P && OH == H && OW == W;
        auto view = [](void* ptr, int dtype, std::initializer_list<int64_t> shape) {
            mjt_tensor t;
            memset(&t, 0, sizeof(t));
            t.ptr = ptr;
            t.dtype = dtype;
            for (int64_t e : shape) t.shape[t.ndim++] = e;
            return t;
        };
        // The product's MFMA kernel wants operand rows that are 16-byte multiples at 16-byte aligned addresses.  Weight
        // rows that are not (3 x 7 x 7 float32 taps: 588 bytes) are copied into rows padded with zeros once per call.
        const void* wmat = w->ptr;
        int64_t lda = CRS;
        auto weight_rows = [&] {                                // (each route below, once it is sure to run)
            need_weights();
            if ((CRS * esz) % 16 == 0 && (uintptr_t)w->ptr % 16 == 0) return;
            lda = (CRS * esz + 15) / 16 * 16 / esz;
            void* wpad = conv_scratch(4, (size_t)(K * lda * esz));
            mjt_tensor tw = view(w->ptr, w->dtype, {K, CRS}), tp = view(wpad, w->dtype, {K, lda});
            Preparing preparing;
            const char* widx[2] = {"i0", "i1"};                 // columns past CRS lie outside w: overflow value 0
            if (mjt_reindex(&tw, &tp, 2, widx, 0.0, 0, nullptr, 0, nullptr) != MJT_OK)
                MJT_FAIL(MJT_ERR_DEVICE, "conv: padding the weight rows failed: " << mjt_last_error());
            wmat = wpad;
        };
        if (flat && !plain) {
            check_no_epilogue();                                // (column matrices take no group: refused before the weights are touched)
            weight_rows();
            const int64_t osz = dtype_size(y->dtype);
            void* cols = conv_scratch(0, (size_t)(CRS * NP0 * esz));
            void* yt = conv_scratch(5, (size_t)(K * NP0 * osz));
            const std::string ih = "i4*" + std::to_string(p->stride_h) + "-" + std::to_string(p->pad_h) + "+i1*" + std::to_string(p->dil_h);
            const std::string iw = "i5*" + std::to_string(p->stride_w) + "-" + std::to_string(p->pad_w) + "+i2*" + std::to_string(p->dil_w);
            const char* cidx[4] = {"i3", "i0", ih.c_str(), iw.c_str()};
            mjt_tensor tx = view(x->ptr, x->dtype, {N, C, H, W}), tc = view(cols, x->dtype, {C, R, S, N, OH, OW});
            if (mjt_reindex(&tx, &tc, 4, cidx, 0.0, 0, nullptr, 0, nullptr) != MJT_OK)
                MJT_FAIL(MJT_ERR_DEVICE, "conv: writing the column matrices failed: " << mjt_last_error());
            gemm_launch(x->dtype, y->dtype, wmat, cols, yt, K, NP0, CRS, lda, NP0, NP0, 0, 0, 0, 1, true, false);
            const char* pidx[3] = {"i1", "i0", "i2"};
            mjt_tensor tt = view(yt, y->dtype, {K, N, P}), ty = view(y->ptr, y->dtype, {N, K, P});
            if (mjt_reindex(&tt, &ty, 3, pidx, 0.0, 0, nullptr, 0, nullptr) != MJT_OK)
                MJT_FAIL(MJT_ERR_DEVICE, "conv: rearranging the product failed: " << mjt_last_error());
            set_last_kernel("conv_as_batch_gemm");
            return;
        }
        // The product kernel gathers its second operand from x on the fly (kernels/gemm_mfma.h with CONV): no column
        // matrices.  float32 convolutions, and the 16-bit ones the MFMA convolution kernel above does not take (odd widths,
        // channel counts that are no multiple of 32 / 64, long rows).  Offsets inside x and y and the column number are
        // 32-bit there, rows and columns of the image and the reach of the taps 14-bit.
        const bool ig16 = x->dtype == MJT_BFLOAT16 || x->dtype == MJT_FLOAT16;
        const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
        const int64_t NP = N * P, tiles64 = ((K + 63) / 64) * ((NP + 63) / 64);
        // (16-bit operands with a long sum and fewer 64 x 64 tiles than compute units stay on the column matrices, whose
        // product picks its tiles for a part-filled chip: 32 x 512 x 7 x 7 3x3 -> 512, 200 tiles: 102 us here, 71 there)
        // (above 18 stages, tiles for at most a quarter of the chip, or half of it where one row of tiles has all output channels and the gather
        // is not repeated, take slices of the sum here; us, column matrices / so: 6 x 160 x 9 x 9 3x3 -> 100 16.8 / 11.4, 51 x 133 x 11 x 11 3x3 -> 16
        // 33.7 / 19.5, 64 x 200 x 11 x 11 5x5 -> 64 76.0 / 41.8; on the other side 20 x 256 x 9 x 9 3x3 -> 256 28.6 / 30.8, 12 x 130 x 13 x 13 3x3 -> 250 22.1 /
        // 25.5; 18 stages, 2 x 128 x 7 x 7 3x3 -> 128 13.5 / 9.4, are left there)
        const bool ig_fits = !ig16 || tiles64 >= cus || CRS <= 1024 || (CRS > 18 * 64 && tiles64 * (K <= 64 ? 2 : 4) <= cus);
        // (a 1x1 convolution whose product would leave most of the chip idle comes here for the slices: the product below takes the images
        // as a batch, whose sums stay whole; float32 3 x 1024 x 14 x 14 -> 256 25.0 us there, 15.8 here; 10 x 512 x 16 x 16 -> 128 15.3, 13.8)
        const bool few_long = CRS >= (ig16 ? 512 : 256) && tiles64 * 2 <= cus;
        if ((!plain || few_long) && ((x->dtype == MJT_FLOAT32 && y->dtype == MJT_FLOAT32) || ig16) && ig_fits && !getenv("MJT_CONV_NO_IGEMM") &&
            numel(x) < (int64_t(1) << 31) && numel(y) < (int64_t(1) << 31) && H < 16384 && W < 16384 &&
            (R - 1) * p->dil_h < 16384 && (S - 1) * p->dil_w < 16384 && p->pad_h < 16384 && p->pad_w < 16384 &&
            OH * p->stride_h < 16384 && OW * p->stride_w < 16384) {
            // Tile, float32, sums of less than four stages (32 elements): 64 output channels x 64 pixels, or 128 x 128 when there
            // are more than 64 output channels and enough tiles of that size for every compute unit.  Longer sums: float32
            // MFMAs on 64 x 64 tiles, of which four workgroups share a compute unit, so that the gather's address arithmetic of one
            // overlaps the MFMAs of another, or products of bfloat16 parts on 128 x 64 or 128 x 128 tiles, by what they are
            // estimated to take: 0.92, 1.05 or 1.85 us a stage and 3, 4 or 5 for each round's first loads and results, four 64 x 64
            // workgroups running at once on a unit (us, 64x64 / 64x128 / 128x64 / 128x128:
            // 64x64x56x56 3x3 -> 64: 178 / 190 / 286 / 261; 64x3x224x224 7x7 stride 2 -> 64: 229 / 278 / 434 / 361; 64x128x28x28 3x3 ->
            // 128: 213 / 199 / 172 / 137; 64x256x14x14 3x3 -> 256: 214 / 192 / 166 / 151; 64x512x7x7 3x3 -> 512: 220 / 186 / 163 / 255;
            // 32x64x56x56 3x3 stride 2 -> 128: 62 / 57 / 50 / 43; 16x256x14x14 3x3 -> 256: 66 / 83 / 71 / 124).
            // 16-bit: the gather bounds the kernel and every 64 rows of output channels repeat it, so 128 x 64 when
            // such tiles fill the chip (us, 64x64 / 128x64 / 256x64 / column matrices: 64x1024x14x14 1x1 -> 256: 51 / 37 /
            // 36 / 68; 64x256x13x13 3x3 -> 384: 116 / 76 / 139 / 103; 64x64x27x27 3x3 stride 2 -> 128: 20 / 18 / 23 / 29;
            // 64x48x28x28 3x3 -> 96: 40 / 35 / 67 / 69; 64x3x224x224 7x7 stride 2 -> 64: 114 / - / - / 285).
            const bool big = !ig16 && K > 64 && ((K + 127) / 128) * ((NP + 127) / 128) >= cus;
            const bool tall = ig16 && K > 64 && ((K + 127) / 128) * ((NP + 63) / 64) >= cus;
            int MI = big || tall ? 2 : 1, NI = big ? 2 : 1;
            bool split = false;
            // Few tiles and a long sum: the sum is cut into up to 16 slices, whose float32 results are added up by a launch behind them,
            // which also takes a group behind the convolution along.  A stage (32 float32 or 64 16-bit elements of the sum) of a 64 x 64 tile
            // takes as long as above, 1.1 us in 16 bits; that launch 5 us and its traffic.  (us, whole / in slices: float32 3 x 272 x 7 x 7 3x3 -> 470 65 / 16.0, 1 x 512 x 7 x 7 3x3
            // -> 512 122 / 17.9, 16 x 256 x 14 x 14 3x3 -> 256 69.5 / 45.9, 4 x 64 x 14 x 14 3x3 -> 64 19.4 / 10.0, 32 x 128 x 9 x 9 3x3 -> 128 35.3 /
            // 19.0, 6 x 256 x 14 x 14 3x3 stride 2 -> 512 64.5 / 18.6; 16 bits, column matrices / so: 6 x 400 x 14 x 14 5x5 -> 51 77.9 / 24.4,
            // 12 x 300 x 15 x 15 5x5 -> 20 76.2 / 29.9, 20 x 500 x 7 x 7 3x3 -> 256 45.9 / 36.1.)
            const int64_t ks = ig16 ? 64 : 32, stages = (CRS + ks - 1) / ks;
            int64_t slices = 1, per = stages;
            auto estimate = [&](int t, int64_t n) {
                const int mi = t ? 2 : 1, ni = t == 2 ? 2 : 1;
                const double tiles = (double)(((K + 64 * mi - 1) / (64 * mi)) * ((NP + 64 * ni - 1) / (64 * ni)));
                const double rounds = std::ceil(tiles * (double)n / cus), st = (double)((stages + n - 1) / n);
                const double us = t == 0 ? ((ig16 ? 1.1 : 0.92) * st + 3.0) * (0.25 + 0.75 * rounds) : t == 1 ? (1.05 * st + 4.0) * rounds : (1.85 * st + 5.0) * rounds;
                return us + (n == 1 ? 0.0 : 5.0 + (double)n * K * NP * 8 / 3e6);
            };
            double least = 1e30;
            if (!ig16 && CRS >= 128)
                for (int t = big ? 1 : 0; t < 3; t++) {
                    const double us = estimate(t, 1);
                    if (us < least) { least = us; MI = t ? 2 : 1; NI = t == 2 ? 2 : 1; split = t > 0; }
                }
            else if (!big && !tall)
                least = estimate(0, 1);
            for (int64_t n = 2; n <= 16 && n <= stages / 2 && least < 1e30; n++) {
                const int64_t pn = (stages + n - 1) / n, nn = (stages + pn - 1) / pn;
                for (int t = 0; t < (ig16 || CRS < 128 ? 1 : 3); t++) {
                    const double us = estimate(t, nn);
                    if (us < least && nn * K * NP * 4 <= (int64_t(256) << 20)) {
                        least = us; slices = nn; per = pn; MI = t ? 2 : 1; NI = t == 2 ? 2 : 1; split = t > 0;
                    }
                }
            }
            if (const char* e = getenv("MJT_CONV_SLICES")) {         // for tests: at most so many slices (1: none) of the tile chosen
                const int64_t n = std::max(1, std::min(atoi(e), 16));
                per = (stages + n - 1) / n;
                slices = (stages + per - 1) / per;
            }
            void* part_mem = slices > 1 ? scratch_if_any((size_t)(slices * K * NP * 4)) : nullptr;
            if (!part_mem) slices = 1;
            const int in = x->dtype == MJT_BFLOAT16 ? 0 : x->dtype == MJT_FLOAT16 ? 1 : 2;
            const int out = slices > 1 ? 2 : y->dtype == MJT_BFLOAT16 ? 0 : y->dtype == MJT_FLOAT16 ? 1 : 2;
            std::ostringstream key;
            const bool xbuf = (64 * NI / P + 2) * C * H * W * esz < (int64_t(1) << 31);      // a tile's images through one buffer descriptor
            const EpilogueCode ep = epilogue_code(1, 12, y->dtype, slices > 1 ? -1 : numel(y));      // (a group behind slices runs where they are added up)
            key << "igemm|" << geo.str() << MI << NI << in << out << xbuf << split << (slices > 1) << ep.key;
            JitKernel* k = cached(key.str());
            if (!k) {
                std::ostringstream name;
                name << "mjt_conv_igemm_" << mjt_dtype_name(x->dtype) << (y->dtype != x->dtype ? "_of32" : "") << "_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << p->stride_h << "x"
                     << p->stride_w << "_p" << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w << (slices > 1 ? "_slices" : "") << (split ? "_parts_" : "_") << 64 * MI << "x" << 64 * NI << ep.suffix();
                std::ostringstream src;
                src << ep.defs << "#define ENTRY " << name.str() << "\n#define SPLIT " << (split ? 1 : 0) << "\n#define SLICED " << (slices > 1 ? 1 : 0) << "\n#define CONV 1\n#define IN " << in << "\n#define OUT " << out << "\n#define MI " << MI << "\n#define NI " << NI
                    << "\n#define A_KCONT 1\n#define B_KCONT 0\n#define XBUF " << (xbuf ? 1 : 0) << "\n" << geo.str();
                if (split) src << embedded_source("split.h") << "\n";
                src << embedded_source("gemm_mfma.h") << "\n";
                k = jit_get(src.str(), name.str());
                remember(key.str(), k);
            }
            const int64_t tiles = ((K + 64 * MI - 1) / (64 * MI)) * ((NP + 64 * NI - 1) / (64 * NI));
            const int64_t grid = (tiles * slices + 7) / 8 * 8;
            MJT_CHECK(grid < (int64_t(1) << 31), "conv: launch too large");
            auto args = [&] {
                weight_rows();
                std::vector<uint64_t> a{bits_of_ptr(wmat), bits_of_ptr(x->ptr), bits_of_ptr(slices > 1 ? part_mem : y->ptr), (uint64_t)K, (uint64_t)NP, (uint64_t)CRS,
                                        (uint64_t)lda, 0, 0, (uint64_t)(slices > 1 ? per : 0), 0, (uint64_t)(slices > 1 ? K * NP : 0)};
                a.insert(a.end(), ep.words.begin(), ep.words.end());
                return a;
            };
            if (slices == 1) {
                if (!ep.on) check_no_epilogue();
                const std::vector<uint64_t> a = args();
                epilogue_taken(ep);
                jit_launch(k, (unsigned)grid, 1, product_threads(split), 0, a);
                return;
            }
            SliceFold fold(part_mem, y->ptr, y->dtype, K * NP, slices);
            const std::vector<uint64_t> a = args();
            {
                Preparing preparing;
                jit_launch(k, (unsigned)grid, 1, product_threads(split), 0, a);
            }
            fold.launch();
            set_last_kernel(k->name.c_str());
            return;
        }
        if (!plain) check_no_epilogue();
        weight_rows();
        int64_t chunk = (int64_t(1) << 30) / (CRS * Ppad * esz);
        if (const char* e = getenv("MJT_CONV_GEMM_CHUNK"))      // images per chunk, for tests of the chunk loop
            if (atoi(e) >= 1) chunk = atoi(e);
        if (chunk < 1) chunk = 1;
        if (chunk > N) chunk = N;
        if (chunk > 65535) chunk = 65535;                       // the images of a chunk are the batch of one product launch
        void* cols = plain ? nullptr : conv_scratch(0, (size_t)(chunk * CRS * Ppad * esz));
        // index strings of the column matrices: [n, c, kh, kw, oh, ow] when a row needs no padding (the window
        // pattern of the reindex fast path), else [n, c, kh, kw, pixel] with the pixel split by division and
        // remainder and the padding marked as overflow
        std::string sh, sw, over;
        if (Ppad == P) {
            sh = "i4*" + std::to_string(p->stride_h) + "-" + std::to_string(p->pad_h) + "+i2*" + std::to_string(p->dil_h);
            sw = "i5*" + std::to_string(p->stride_w) + "-" + std::to_string(p->pad_w) + "+i3*" + std::to_string(p->dil_w);
        } else {
            sh = "i4/" + std::to_string(OW) + "*" + std::to_string(p->stride_h) + "-" + std::to_string(p->pad_h) + "+i2*" + std::to_string(p->dil_h);
            sw = "i4%" + std::to_string(OW) + "*" + std::to_string(p->stride_w) + "-" + std::to_string(p->pad_w) + "+i3*" + std::to_string(p->dil_w);
            over = "i4>=" + std::to_string(P);
        }
        const char* idx[4] = {"i0", "i1", sh.c_str(), sw.c_str()};
        const char* ovc[1] = {over.c_str()};

        for (int64_t n0 = 0; n0 < N; n0 += chunk) {
            const int64_t nb = N - n0 < chunk ? N - n0 : chunk;
            char* xn = (char*)x->ptr + n0 * C * H * W * esz;
            if (!plain) {
                mjt_tensor tx = view(xn, x->dtype, {nb, C, H, W});
                mjt_tensor tc = Ppad == P ? view(cols, x->dtype, {nb, C, R, S, OH, OW}) : view(cols, x->dtype, {nb, C, R, S, Ppad});
                if (mjt_reindex(&tx, &tc, 4, idx, 0.0, Ppad == P ? 0 : 1, ovc, 0, nullptr) != MJT_OK)
                    MJT_FAIL(MJT_ERR_DEVICE, "conv: writing the column matrices failed: " << mjt_last_error());
            }
            char* yn = (char*)y->ptr + n0 * K * P * dtype_size(y->dtype);
            // a short sum (a 1x1 convolution, few channels) is bound by how many workgroups a compute unit holds, not by
            // operand reuse: tiles of 128 x 128 (64 for at most 64 output channels or pixels, or when there would be fewer
            // tiles than compute units; at most 64 output channels with four or more 64 x 128 tiles per compute unit:
            // 64 x 64), and the direct-copy kernel from two stages of the sum on, its 256 x 256 tiles from four
            // (16-bit operands, us with / without the tile named here: 64 x 64 x 56 x 56 -> 256: 43 / 55;
            // 64 x 512 x 28 x 28 -> 64: 19 / 37; 64 x 256 x 56 x 56 -> 64: 37 / 44 with 64 x 128;
            // general kernel / direct-copy kernel on 128 x 128 tiles: 64 x 512 x 28 x 28 -> 128: 21.8 / 19.8; -> 512: 77 / 64;
            // 64 x 256 x 56 x 56 -> 128: 56 / 47; 64 x 128 x 28 x 28 -> 512: 32 / 26)
            const bool short_sum = CRS <= 1024 && esz == 2 && !getenv("MJT_CONV_GEMM_NO_HINT");
            const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
            const bool few = ((K + 127) / 128) * ((P + 127) / 128) * nb < cus;       // tiles of 128 x 128 would leave compute units idle
            const bool many = ((P + 127) / 128) * nb >= 4 * cus;                     // plenty of 64 x 128 tiles
            const int tile_m = !short_sum ? 0 : K <= 64 || few ? 64 : 128;
            const int tile_n = !short_sum ? 0 : P <= 64 || few || (K <= 64 && many) ? 64 : 128;
            gemm_launch(x->dtype, y->dtype, wmat, plain ? (void*)xn : cols, yn, K, P, CRS, lda, Ppad, P, 0, CRS * Ppad, K * P, nb, true, false,
                        tile_m, tile_n, !short_sum || CRS >= 128);
        }
        set_last_kernel(plain ? "conv_as_gemm" : "conv_as_reindex_gemm");
        return;
    }

    need_weights();
    // ---- depthwise: one input channel per group -----------------------------------------
    if (G > 1 && C == 1 && !free_extent) {
        const DepthwiseShape g{H, W, OH, OW, R, S, p->stride_h, p->stride_w, p->pad_h, p->pad_w, p->dil_h, p->dil_w, 1, 1, K, K / G, false};
        if (depthwise_run(g, x, w, y)) return;
    }

    // ---- direct path ----------------------------------------------------------------
    const bool idx32 = numel(x) < (int64_t(1) << 31) && numel(y) < (int64_t(1) << 31) - 256 && numel(w) < (int64_t(1) << 31);
    std::ostringstream key;
    const EpilogueCode ep = epilogue_code(1, 4, y->dtype, numel(y));
    key << "direct|" << geo.str() << x->dtype << "|" << y->dtype << "|" << G << "|" << idx32 << ep.key;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_direct_" << mjt_dtype_name(x->dtype) << "_" << mjt_dtype_name(y->dtype) << "_c" << C << "_k" << K
             << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << p->stride_h << "x" << p->stride_w << "_p" << p->pad_h
             << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w;
        if (G > 1) name << "_g" << G;
        if (!idx32) name << "_i64";
        name << ep.suffix();
        std::ostringstream src;
        src << ep.defs << "#define ENTRY " << name.str() << "\n#define TIN " << dtype_cname(x->dtype) << "\n#define TOUT "
            << dtype_cname(y->dtype) << "\n#define G_ " << G << "\n#define IDX " << (idx32 ? "int" : "long long")
            << "\n" << geo.str();
        if (!ep.on) src << embedded_source("prelude.h") << "\n";
        src << embedded_source("conv_direct.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    const int64_t total = numel(y);
    const int64_t blocks = (total + 255) / 256;
    MJT_CHECK(blocks < (int64_t(1) << 31), "conv: launch too large");
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(w->ptr), bits_of_ptr(y->ptr), (uint64_t)total};
    a.insert(a.end(), ep.words.begin(), ep.words.end());
    epilogue_taken(ep);
    jit_launch(k, (unsigned)blocks, 1, 256, 0, a);
}

void conv_impl(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p, int64_t G, bool free_extent = false,
               int pack_mode = 0, void* packed = nullptr) {
    conv_run(x, w, y, p, G, free_extent, pack_mode, packed, nullptr);
}

// The buffer of per-slice partial weight gradients, grown to `bytes`.
static void* wgrad_partials(size_t bytes) {
    if (ctx().dry_run) return (void*)(uintptr_t)0x1000;
    if (!grow_kept(&g_wgrad_part, &g_wgrad_bytes, bytes)) MJT_FAIL(MJT_ERR_DEVICE, "conv wgrad: no device memory for " << bytes << " bytes of partial sums");
    return g_wgrad_part;
}

// [slices, numel(dw)] float partial sums summed over axis 0 into dw, rounded once if dw is a 16-bit type.
static void fold_wgrad_slices(void* part, int64_t slices, const mjt_tensor* dw) {
    mjt_tensor tp, td;
    memset(&tp, 0, sizeof(tp));
    memset(&td, 0, sizeof(td));
    tp.ptr = part;
    tp.dtype = MJT_FLOAT32;
    tp.ndim = 2;
    tp.shape[0] = slices;
    tp.shape[1] = numel(dw);
    td.ptr = dw->ptr;
    td.dtype = dw->dtype;
    td.ndim = 1;
    td.shape[0] = numel(dw);
    if (mjt_reduce(&tp, &td, MJT_OP_ADD, 0b01) != MJT_OK) MJT_FAIL(MJT_ERR_DEVICE, "conv wgrad: folding the partial sums failed: " << mjt_last_error());
}

// The direct weight-gradient kernel (kernels/conv_wgrad_direct.h): any groups, any geometry, float32 / bfloat16 / float16.
static void conv_wgrad_direct(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p, int64_t G) {
    const int64_t N = x->shape[0], C = x->shape[1] / G, H = x->shape[2], W = x->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = dw->shape[2], S = dw->shape[3];
    const bool flt = x->dtype == MJT_FLOAT32 || x->dtype == MJT_BFLOAT16 || x->dtype == MJT_FLOAT16;
    if (!flt || dy->dtype != x->dtype || !(dw->dtype == MJT_FLOAT32 || dw->dtype == x->dtype))
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv wgrad: x and dy must share one of float32 / bfloat16 / float16 and dw be of that type or float32");
    MJT_CHECK(H * W < (int64_t(1) << 31) && OH * OW < (int64_t(1) << 31), "conv wgrad: image too large");
    if (N == 0 || OH * OW == 0) {                                // a sum over nothing: zeros, written by the reduce kernel
        fold_wgrad_slices(wgrad_partials(4), 0, dw);
        return;
    }
    if (C == 1 && G > 1 && !getenv("MJT_NO_FASTPATH")) {           // depthwise: planes through LDS
        const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
        // slices of images: about four workgroups per compute unit, each of which has the planes of its next images on their way
        // while it sums; every slice ends in a fold of its lanes' sums and a row of partial results (us with the fold, float32, 3x3,
        // 2 / 4 / 8 / 16 workgroups a unit: 32 x 128 x 56 x 56 34.6 / 26.5 / 30.6 / 32.7; 64 x 256 x 14 x 14 - / 12.4 / 15.8 / 18.5).
        // Below 2048 positions a channel one slice, whose sums are the result of a float32 gradient (in slices / in one, 3x3:
        // 4 x 512 x 7 x 7 8.4 / 4.9, 16 x 128 x 7 x 7 8.3 / 5.0, 64 x 256 x 7 x 7 stride 2 8.8 / 5.6).
        int64_t slices = (4 * cus + K - 1) / K;
        if (slices > N) slices = N;
        if (N * OH * OW < 2048) slices = 1;
        const int64_t ips = (N + slices - 1) / slices;
        slices = (N + ips - 1) / ips;
        const DepthwiseShape g{H, W, OH, OW, R, S, p->stride_h, p->stride_w, p->pad_h, p->pad_w, p->dil_h, p->dil_w, 1, 1, K, K / G, false};
        DepthwisePlan q;
        if (slices * K < (int64_t(1) << 31) &&
            depthwise_plan(g, dtype_size(x->dtype), dtype_size(dy->dtype), x->ptr, dy->ptr, int64_t(1) << 40, ips, &q)) {
            JitKernel* k = depthwise_kernel(1, g, q, x->dtype, x->dtype);
            const bool in_place = slices == 1 && dw->dtype == MJT_FLOAT32;
            void* part = in_place ? dw->ptr : wgrad_partials((size_t)slices * (size_t)numel(dw) * 4);
            std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(dy->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)ips, 0, 0};
            jit_launch(k, (unsigned)(slices * K), 1, 256, 0, a);
            if (!in_place) fold_wgrad_slices(part, slices, dw);
            set_last_kernel(k->name.c_str());
            return;
        }
    }
    const int64_t taps = R * S;
    const int64_t TCH = taps <= 49 ? taps : 32;
    int64_t CT = taps <= 49 ? 40 / taps : 1;
    if (CT > 4) CT = 4;
    if (CT > C) CT = C;
    if (CT < 1) CT = 1;
    const int64_t per_slice = K * ((C + CT - 1) / CT) * ((taps + TCH - 1) / TCH);
    Context& c = ctx();
    const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
    // slices of whole images: about four workgroups per compute unit, at least a thousand positions per slice
    int64_t slices = (4 * cus + per_slice - 1) / per_slice;
    if (slices > N * OH * OW / 1024) slices = N * OH * OW / 1024;
    if (slices > N) slices = N;
    if (slices < 1) slices = 1;
    const int64_t ips = (N + slices - 1) / slices;
    slices = (N + ips - 1) / ips;
    MJT_CHECK(slices * per_slice < (int64_t(1) << 31), "conv wgrad: launch too large");

    std::ostringstream key;
    key << "wgrad_direct|" << x->dtype << "|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|"
        << p->stride_h << "|" << p->stride_w << "|" << p->pad_h << "|" << p->pad_w << "|" << p->dil_h << "|" << p->dil_w << "|" << G << "|" << CT;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_wgrad_direct_" << mjt_dtype_name(x->dtype) << "_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s"
             << p->stride_h << "x" << p->stride_w << "_p" << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w << "_g" << G;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define TIN " << dtype_cname(x->dtype) << "\n#define C_ " << C << "\n#define H_ " << H
            << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH
            << "\n#define OW_ " << OW << "\n#define SH " << p->stride_h << "\n#define SW " << p->stride_w << "\n#define PH " << p->pad_h
            << "\n#define PW " << p->pad_w << "\n#define DH " << p->dil_h << "\n#define DW " << p->dil_w << "\n#define G_ " << G
            << "\n#define CT " << CT << "\n#define TCH " << TCH << "\n";
        src << embedded_source("prelude.h") << "\n" << embedded_source("conv_wgrad_direct.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    const bool in_place = slices == 1 && dw->dtype == MJT_FLOAT32;       // one slice of float sums is the result
    void* part = in_place ? dw->ptr : wgrad_partials((size_t)slices * (size_t)numel(dw) * 4);
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(dy->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)ips, 0};
    jit_launch(k, (unsigned)(slices * per_slice), 1, 256, 0, a);
    if (!in_place) fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
}

// Weight gradient from windows in LDS (kernels/conv_wgrad_window.h): 16-bit operands, 2 to 9 taps, horizontal strides 1 and 2.
// False: not covered, or estimated to take longer than `other` us.
static bool conv_wgrad_window(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p, double other) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = dw->shape[2], S = dw->shape[3];
    const int64_t SH = p->stride_h, SW = p->stride_w, PW = p->pad_w, DH = p->dil_h, DW = p->dil_w, taps = R * S, npw = (OW + 7) / 8;
    const bool half = x->dtype == MJT_FLOAT16;
    if (!(half || x->dtype == MJT_BFLOAT16) || dy->dtype != x->dtype || !(dw->dtype == MJT_FLOAT32 || dw->dtype == x->dtype) || getenv("MJT_NO_FASTPATH") || getenv("MJT_CONV_NO_IGEMM")) return false;
    if (taps < 2 || taps > 9 || SW > 2 || PW > 8 || (S - 1) * DW > 8 || !(npw == 1 || npw == 2 || npw % 4 == 0) || H > 1024 || W > 256 || numel(x) * 2 >= (int64_t(1) << 31) ||
        numel(dy) * 2 >= (int64_t(1) << 31) || (uintptr_t)x->ptr % 16 || (uintptr_t)dy->ptr % 16)
        return false;
    // The kernel's layout for `rb` output rows and `ib` images a stage: its bytes of LDS, and the dwords a thread holds on their way there.
    auto floor_div = [](int64_t a, int64_t b) { return a >= 0 ? a / b : -((b - 1 - a) / b); };
    int64_t lo = 0, hi = 3;
    for (int64_t s = 0; s < S; s++) {
        const int64_t shift = floor_div(s * DW - PW, SW);
        lo = std::min(lo, floor_div(shift, 2));
        hi = std::max(hi, floor_div(shift, 2) + 3 + (shift & 1));
    }
    const int64_t lp = std::max<int64_t>(8, (-2 * lo + 7) / 8 * 8), rw = (lp + std::max((W + SW - 1) / SW, npw * 8 - 8 + 2 * hi + 2 - lp) + 7) / 8 * 8, xrow = SW * rw * 2;
    auto unit = [](int64_t n) { return n % 8 == 0 ? 8 : n % 4 == 0 ? 4 : n % 2 == 0 ? 2 : 1; };
    auto lds_bytes = [&](int64_t rb, int64_t ib) {
        const int64_t xr = (rb - 1) * SH + (R - 1) * DH + 1, steps = (rb * npw + 3) / 4;
        const int64_t xcb = ((xr * xrow + lp * 2) / 16 | 1) * 16, dcb = (steps * 4 | 1) * 16;
        const bool checked = OH % rb != 0 || rb * npw % 4 != 0 || ib > 1;
        return std::max(2 * ib * 64 * (xcb + dcb) + (checked ? lp * 2 + xrow + hi * 4 + 16 : 0), 64 * (64 * taps + 8) * 4);
    };
    auto dwords = [&](int64_t rb, int64_t ib) {
        const bool whole = rb == OH;
        const int64_t xr = (rb - 1) * SH + (R - 1) * DH + 1, gx = unit(whole ? H * W : W), gd = unit(whole ? OH * OW : OW);
        const int64_t nx = ((whole ? H : xr) * W / gx + 7) / 8, nd = (rb * OW / gd + 7) / 8;
        return ib * (nx * std::max<int64_t>(1, gx / 2) + nd * std::max<int64_t>(1, gd / 2));
    };
    const int64_t blocks = ((K + 63) / 64) * ((C + 63) / 64), cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    // Rows, images and slices by what they are estimated to take: 0.8 us and 0.04 for each row of 32 x 32 products of a wave a stage, 11.5 for
    // the launches, the first loads and the meeting of the groups, the slices' results written (3 TB/s: all compute units at once) and read by
    // the fold, 4 more for a fold in two launches.  us, estimated / measured: 64 x 256 x 14 x 14 -> 256 41.8 / 39.4, 64 x 512 x 7 x 7 -> 512 46.4 / 42.9,
    // 64 x 256 x 28 x 28 stride 2 -> 256 52.8 / 50.9, 4 x 256 x 16 x 16 -> 256 20.2 / 18.5.  (Twenty-eight dwords on their way are what a thread
    // has registers for beside nine accumulators.)
    int64_t RB = 0, IB = 1, slices = 1;
    double least = 1e30;
    for (int64_t rb = 1; rb <= OH; rb++)
        for (int64_t ib = 1; ib <= (rb == OH ? 4 : 1); ib++) {
            if (lds_bytes(rb, ib) > 160 * 1024 || dwords(rb, ib) > 28) continue;
            const int64_t stages = rb == OH ? (N + ib - 1) / ib : N * ((OH + rb - 1) / rb);
            const double stage = 0.8 + 0.04 * (double)(ib * ((rb * npw + 3) / 4) * taps);
            const int64_t most = std::min(stages, std::max<int64_t>(1, cus / blocks));
            for (int64_t n = 1; n <= most; n++) {
                const int64_t per = (stages + n - 1) / n, nn = (stages + per - 1) / per;
                const double t = 11.5 + std::ceil((double)(nn * blocks) / cus) * (double)per * stage + (double)nn * numel(dw) * 4 * (C * taps % 4 ? 0.7e-6 : 0.45e-6) + (nn > 16 ? 4.0 : 0.0);
                if (t < least) { least = t; RB = rb; IB = ib; slices = nn; }
            }
        }
    if (RB == 0 || least >= other) return false;
    const int64_t stages = RB == OH ? (N + IB - 1) / IB : N * ((OH + RB - 1) / RB), per = (stages + slices - 1) / slices;
    slices = (stages + per - 1) / per;
    if (slices * numel(dw) * 4 > (int64_t(1) << 30) || slices * blocks > (1 << 28)) return false;
    const bool in_place = slices == 1 && dw->dtype == MJT_FLOAT32 && (uintptr_t)dw->ptr % 16 == 0;
    const size_t part_bytes = (size_t)slices * (size_t)numel(dw) * 4;
    if (!in_place && !(workspace_allowed(part_bytes) && (ctx().dry_run || grow_kept(&g_wgrad_part, &g_wgrad_bytes, part_bytes)))) return false;
    std::ostringstream key;
    key << "wgwin|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << SH << "|" << SW << "|" << p->pad_h << "|" << PW
        << "|" << DH << "|" << DW << "|" << half << "|" << RB << "|" << IB;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_wgrad_mfma_" << (half ? "f16" : "bf16") << "_window_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << SH << "x" << SW << "_p"
             << p->pad_h << "x" << PW << "_d" << DH << "x" << DW << "_rows" << RB << "_images" << IB;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define IN_F16 " << half << "\n#define RB " << RB << "\n#define IB " << IB
            << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH
            << "\n#define OW_ " << OW << "\n#define SH " << SH << "\n#define SW " << SW << "\n#define PH " << p->pad_h << "\n#define PW " << PW << "\n#define DH " << DH << "\n#define DW " << DW << "\n";
        src << embedded_source("conv_wgrad_window.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0) return false;
    void* part = in_place ? dw->ptr : wgrad_partials(part_bytes);
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(dy->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)stages, (uint64_t)per, (uint64_t)(numel(x) * 2), (uint64_t)(numel(dy) * 2)};
    jit_launch(k, (unsigned)((slices * blocks + 7) / 8 * 8), 1, 512, 0, a);
    if (!in_place) fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
    return true;
}

// Weight gradient of the first layer of a network, float32, few channels at horizontal stride 2, from windows in LDS (kernels/conv_stem_wgrad.h).
// False: not covered, or estimated to take longer than `other` us.
static bool conv_wgrad_stem(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p, double other) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = dw->shape[2], S = dw->shape[3], CRS = C * R * S, NT = (CRS + 31) / 32;
    const int64_t SH = p->stride_h, PH = p->pad_h, PW = p->pad_w, DH = p->dil_h;
    if (x->dtype != MJT_FLOAT32 || dw->dtype != MJT_FLOAT32 || p->stride_w != 2 || (p->dil_w != 1 && S > 1) || NT < 3 || NT > 5 || H > 8192 || W > 4096 || PH > 64 || PW > 64 || SH > 8 || (R - 1) * DH > 64 ||
        (uintptr_t)x->ptr % 16 || (uintptr_t)dy->ptr % 16 || numel(x) * 4 >= (int64_t(1) << 31) || numel(dy) * 4 >= (int64_t(1) << 31))
        return false;
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    const int64_t KH = K > 32 ? 2 : 1, kblocks = (K + 32 * KH - 1) / (32 * KH), groups = 4 / KH, unit = W % 4 == 0 ? 4 : W % 2 == 0 ? 2 : 1, steps = (OW + 15) / 16;
    const int64_t lp = (PW + 3) / 4 * 4, halfw = std::max((lp + W + 1) / 2, steps * 16 + (S - 1 - PW + lp) / 2 + 2), dwords = (halfw + 1) / 2 | 1;
    // Rows of a tile and tiles of a workgroup by what they are estimated to take, in us: terms as for the forward kernel, the slices' fold as for the
    // gathering product, whose estimate `other` is.  us, gather / this: 32 x 3 x 224 x 224 7x7 -> 64 107 / 59.6, -> 16 103.5 / 36; 8 x 3 x 224 x 224 -> 64 35.8 / 25.3;
    // 32 x 3 x 125 x 125 -> 64 53.7 / 43.1; on the other side 1 x 3 x 224 x 224 -> 64 14.8 / 19.9, 4 x 3 x 96 x 96 -> 48 13.8 / 18.3.  (Up to 64 columns, such as 3 x 3 taps
    // of 3 channels, the waves have few MFMAs to a step: 16 x 3 x 128 x 128 3x3 -> 64 16.6 / 16.6, 64 x 3 x 32 x 32 -> 16 11.1 / 13.6.)
    int64_t TR = 0, per = 1;
    double best = other;
    for (int64_t tr = 1; tr <= 8 && tr <= OH; tr++) {
        const int64_t xr = (tr - 1) * SH + (R - 1) * DH + 1, ni = (C * xr * (W / unit) + 255) / 256;
        if (std::max(3 * C * xr * dwords * 8, 32 * KH * NT * 128) > 78 * 1024 || ni * unit > 36) continue;
        const int64_t tiles = N * ((OH + tr - 1) / tr);
        const double tile = (double)((tr * steps + groups - 1) / groups) * (double)(NT * 6 * 32 + 200) + 1000.0 + (double)(ni * unit) * 40.0;
        for (int64_t n = 1; n <= 64 && n <= tiles; n++) {
            const int64_t nn = (tiles + n - 1) / n, wgs = nn * kblocks;
            const double cycles = wgs <= cus ? 3000.0 + (double)n * tile : std::ceil((double)wgs / (2 * cus)) * 1.6 * (3000.0 + (double)n * tile);
            const double t = cycles / 2200.0 + 3.0 + (nn > 1 ? (nn > 16 ? 8.0 : 5.0) + (double)nn * numel(dw) * 8 / 5e6 : 0.0);
            if (t < best) { best = t; TR = tr; per = n; }
        }
    }
    if (TR == 0) return false;
    const int64_t tiles = N * ((OH + TR - 1) / TR), slices = (tiles + per - 1) / per;
    if (tiles >= (1 << 28) || slices * kblocks >= (1 << 28) || slices * numel(dw) * 4 > (int64_t(1) << 30)) return false;
    const size_t part_bytes = (size_t)slices * (size_t)numel(dw) * 4;
    if (slices > 1 && !(workspace_allowed(part_bytes) && (ctx().dry_run || grow_kept(&g_wgrad_part, &g_wgrad_bytes, part_bytes)))) return false;
    std::ostringstream key;
    key << "wgstem|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << SH << "|" << PH << "|" << PW << "|" << DH << "|" << TR;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_wgrad_igemm_float32_stem_c" << C << "_k" << K << "_r" << R << "x" << S << "_s" << SH << "x2_p" << PH << "x" << PW << "_d" << DH << "x1_rows" << TR << "_" << H << "x" << W;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define TR " << TR << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R
            << "\n#define S_ " << S << "\n#define OH_ " << OH << "\n#define OW_ " << OW << "\n#define SH " << SH << "\n#define PH " << PH << "\n#define PW " << PW << "\n#define DH " << DH << "\n";
        src << embedded_source("split.h") << "\n" << embedded_source("conv_stem_wgrad.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0) return false;
    void* part = slices == 1 ? dw->ptr : wgrad_partials(part_bytes);
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(dy->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)per, (uint64_t)(numel(x) * 4), (uint64_t)(numel(dy) * 4)};
    jit_launch(k, (unsigned)(slices * kblocks), 1, 256, 0, a);
    if (slices > 1) fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
    return true;
}

// Weight gradient as an implicit product (kernels/gemm_mfma.h with CONV 2): both operands are gathered on their way to LDS and
// the sum over images and pixels is cut into slices.  False: not covered.
static bool conv_wgrad_product(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p) {
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = dw->shape[2], S = dw->shape[3];
    const int64_t P = OH * OW, CRS = C * R * S, Q = N * P;
    const bool half = x->dtype == MJT_FLOAT16 || x->dtype == MJT_BFLOAT16;
    if (!(x->dtype == MJT_FLOAT32 || half) || dy->dtype != x->dtype || !(dw->dtype == MJT_FLOAT32 || dw->dtype == x->dtype) || getenv("MJT_NO_FASTPATH") || getenv("MJT_CONV_NO_IGEMM")) return false;
    const int64_t esz = dtype_size(x->dtype);
    // (offsets inside x and dy are 31-bit bytes, rows and columns 14-bit; a few million multiply-adds are worth the set-up)
    if ((double)Q * K * CRS < (double)(1 << 22) || Q >= (int64_t(1) << 31) - 64 ||
        numel(x) * esz >= (int64_t(1) << 31) || numel(dy) * esz >= (int64_t(1) << 31) || H >= 16384 || W >= 16384 || (R - 1) * p->dil_h >= 16384 || (S - 1) * p->dil_w >= 16384 || p->pad_h >= 16384 || p->pad_w >= 16384 ||
        OH * p->stride_h >= 16384 || OW * p->stride_w >= 16384 || (uintptr_t)dy->ptr % 16 || (uintptr_t)x->ptr % 16)
        return false;
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    const int in = x->dtype == MJT_BFLOAT16 ? 0 : half ? 1 : 2;
    const int64_t KS = half ? 64 : 32;
    // Tile and slices of the sum by what they are estimated to take.  Slices end in a fold: 5 us, 8 with more than 16 of them (the
    // reduce is then two launches), and its traffic.
    auto tiles_of = [&](int64_t t) { return ((K + t - 1) / t) * ((CRS + t - 1) / t); };
    const int64_t stages = (Q + KS - 1) / KS;
    int64_t slices = 1;
    int MI = 1;
    double least = 1e30;
    if (!half) {
        // float32: a stage of a 64 x 64 tile takes 0.78 us with a compute unit to itself and 0.9 of that more for each further
        // workgroup there (four fit), one of a 128 x 128 tile, which multiplies bfloat16 parts, 1.75 us, one workgroup at a time; its
        // first operands and its results 5 us more.  Slices that give every compute unit one, two, four or eight workgroups (128: one,
        // two or four), down to a single stage each; more 64 x 64 tiles than compute units share less and take 1.25 times that.
        // us, 64 x 64 / 128 x 128 tiles at their best slices: 16 x 100 x 9 x 9 3x3 stride 2 -> 70 9.1 / 12.0; 8 x 64 x 28 x 28 3x3 -> 64 15.8 /
        // 19.5; 64 x 64 x 56 x 56 3x3 -> 64 152 / 221; 32 x 64 x 56 x 56 3x3 stride 2 -> 128 59 / 40; 64 x 128 x 28 x 28 3x3 -> 128 168 / 101;
        // 64 x 256 x 14 x 14 3x3 -> 256 189 / 108; 64 x 512 x 7 x 7 3x3 -> 512 216 / 131 (128 x 128 with float32 MFMAs 140, 141, 156).
        for (int mi = 1; mi <= 2; mi++)
            for (int64_t r = 1; r <= (mi == 1 ? 8 : 4); r *= 2) {
                int64_t n = r * cus / tiles_of(64 * mi);
                n = n < 1 ? 1 : n > stages ? stages : n;
                const int64_t pn = (stages + n - 1) / n, nn = (stages + pn - 1) / pn;
                const double wgs = std::ceil((double)(nn * tiles_of(64 * mi)) / cus);
                const double st = mi == 1 ? 0.78 * (1.0 + 0.9 * (wgs - 1.0)) : 1.75 * wgs;
                const double t = (double)pn * st * (mi == 1 && tiles_of(64) > cus ? 1.25 : 1.0) + (mi == 2 ? 5.0 * wgs : 0.0) +
                                 (nn > 1 ? (nn > 16 ? 8.0 : 5.0) + (double)nn * numel(dw) * 8 / 5e6 : 0.0);
                if (t < least) { least = t; MI = mi; slices = nn; }
            }
    } else {
        // 16 bits: the loads bound a stage, 0.045 us for each that a thread issues on 128 x 128 tiles (four chunks of each operand)
        // and 0.05 on 64 x 64 (two), 0.7 and 0.37 at least; a further workgroup on a compute unit adds 0.7 of that time.
        // us at 64 images, tile / slices as found here, and others: 1024 x 14 x 14 1x1 -> 256 128 / 16 21.7 (64 / 4 24.8, 128 / 8 26.7, 128 / 48 32.1); 256 x 14 x 14 3x3 -> 256 128 / 14 60.7 (128 / 4 90.5, 64 / 12
        // 96.5); 256 x 28 x 28 1x1 -> 128 64 / 32 16.5 (128 / 64 20.3).
        const bool planes = R * S == 1 && p->stride_h == 1 && p->stride_w == 1 && p->pad_h == 0 && p->pad_w == 0;
        const int nl = P % 8 == 0 ? 1 : P % 4 == 0 ? 2 : P % 2 == 0 ? 4 : 8, loads = nl + (planes ? nl : 8);
        for (int mi = 1; mi <= 2; mi++)
            for (int64_t n = 1; n <= 64 && (n == 1 || n <= stages / 4); n++) {
                const int64_t pn = (stages + n - 1) / n, nn = (stages + pn - 1) / pn;
                const double st = mi == 2 ? std::max(0.7, 0.045 * 4 * loads) : std::max(0.37, 0.05 * 2 * loads);
                const double t = (double)pn * st * (1.0 + 0.7 * (std::ceil((double)(nn * tiles_of(64 * mi)) / cus) - 1.0)) + 5.0 + (double)nn * numel(dw) * 8 / 5e6;
                if (t < least) { least = t; MI = mi; slices = nn; }
            }
    }
    // us at 16 bits, this / the windows: 64 x 256 x 14 x 14 3x3 -> 256 59.9 / 39.4; 64 x 512 x 7 x 7 -> 512 91.8 / 42.9; 64 x 256 x 28 x 28 stride 2 ->
    // 256 63.9 / 50.9; 16 x 512 x 14 x 14 -> 512 64.2 / 38.9; 4 x 128 x 12 x 12 -> 256 11.9 / 15.6, 64 x 64 x 14 x 14 -> 64 18.2 / 25.0 stay.
    if (half && R * S > 1 && conv_wgrad_window(x, dy, dw, p, least)) return true;
    if (!half && conv_wgrad_stem(x, dy, dw, p, least)) return true;
    const int NI = MI;
    const bool split = !half && MI == 2;
    const int64_t tiles = tiles_of(64 * MI);
    if (slices * numel(dw) * 4 > (int64_t(1) << 30)) return false;
    const int64_t per = (stages + slices - 1) / slices;
    slices = (stages + per - 1) / per;
    const bool in_place = slices == 1 && dw->dtype == MJT_FLOAT32;
    const size_t part_bytes = (size_t)slices * (size_t)numel(dw) * 4;
    if (!in_place && !(workspace_allowed(part_bytes) && (ctx().dry_run || grow_kept(&g_wgrad_part, &g_wgrad_bytes, part_bytes)))) return false;
    std::ostringstream key;
    key << "wgprod|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << p->stride_h << "|" << p->stride_w << "|" << p->pad_h << "|" << p->pad_w
        << "|" << p->dil_h << "|" << p->dil_w << "|" << MI << NI << in;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_wgrad_igemm_" << mjt_dtype_name(x->dtype) << "_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << p->stride_h << "x" << p->stride_w << "_p"
             << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w << (split ? "_parts_" : "_") << 64 * MI << "x" << 64 * NI;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define SPLIT " << (split ? 1 : 0) << "\n#define CONV 2\n#define IN " << in << "\n#define OUT 2\n#define MI " << MI << "\n#define NI " << NI << "\n#define A_KCONT 1\n#define B_KCONT 1"
            << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH
            << "\n#define OW_ " << OW << "\n#define SH " << p->stride_h << "\n#define SW " << p->stride_w << "\n#define PH " << p->pad_h << "\n#define PW " << p->pad_w << "\n#define DH " << p->dil_h
            << "\n#define DW " << p->dil_w << "\n";
        if (split) src << embedded_source("split.h") << "\n";
        src << embedded_source("gemm_mfma.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    void* part = in_place ? dw->ptr : wgrad_partials(part_bytes);
    std::vector<uint64_t> a{bits_of_ptr(dy->ptr), bits_of_ptr(x->ptr), bits_of_ptr(part), (uint64_t)K, (uint64_t)CRS, (uint64_t)Q, 0, 0, (uint64_t)CRS, (uint64_t)per,
                            (uint64_t)(numel(x) * esz), (uint64_t)(K * CRS)};
    const int64_t grid = (slices * tiles + 7) / 8 * 8;
    MJT_CHECK(grid < (int64_t(1) << 31), "conv wgrad: launch too large");
    jit_launch(k, (unsigned)grid, 1, product_threads(split), 0, a);
    if (!in_place) fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
    return true;
}

// Weight gradient: dw[k,c,r,s] = sum_{n,oh,ow} dy[n,k,oh,ow] * x[n,c,oh*sh-ph+r*dh,ow*sw-pw+s*dw].
// With `any_shape` (the grouped entry point) what the MFMA kernel does not cover runs on the direct kernel instead of
// being handed back; G > 1: x has G groups of dw->shape[1] channels, dy G groups of K / G (python/jittor/nn.py:1272-1294).
void conv_wgrad_impl(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p, int64_t G, bool any_shape) {
    require_init();
    check_tensor(x, "conv wgrad x");
    check_tensor(dy, "conv wgrad dy");
    check_tensor(dw, "conv wgrad dw");
    MJT_CHECK(p, "conv wgrad: null parameters");
    MJT_CHECK(x->ndim == 4 && dy->ndim == 4 && dw->ndim == 4, "conv wgrad: x, dy and dw must have rank 4");
    MJT_CHECK(p->stride_h >= 1 && p->stride_w >= 1 && p->dil_h >= 1 && p->dil_w >= 1 && p->pad_h >= 0 && p->pad_w >= 0,
              "conv wgrad: bad stride / padding / dilation");
    MJT_CHECK(G >= 1, "conv wgrad: groups must be positive");
    const int64_t N = x->shape[0], H = x->shape[2], W = x->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3];
    const int64_t R = dw->shape[2], S = dw->shape[3];
    MJT_CHECK(x->shape[1] % G == 0 && K % G == 0, "conv wgrad: " << x->shape[1] << " input and " << K << " output channels do not split into " << G << " groups");
    const int64_t C = x->shape[1] / G;                           // input channels per group
    MJT_CHECK(dy->shape[0] == N, "conv wgrad: dy has " << dy->shape[0] << " images, x " << N);
    MJT_CHECK(dw->shape[0] == K && dw->shape[1] == C, "conv wgrad: dw shape " << shape_str(dw) << " != [" << K << "," << C << ",R,S]");
    MJT_CHECK(OH == (H + 2 * p->pad_h - p->dil_h * (R - 1) - 1) / p->stride_h + 1 &&
                  OW == (W + 2 * p->pad_w - p->dil_w * (S - 1) - 1) / p->stride_w + 1,
              "conv wgrad: dy shape " << shape_str(dy) << " does not follow from x " << shape_str(x) << " and the " << R << "x" << S
                                      << " kernel");
    if (numel(dw) == 0) return;
    // what the MFMA kernel covers; anything else is for the caller's general path
    const int64_t KG = K % 256 == 0 ? 4 : K % 128 == 0 ? 2 : 1;
    const int64_t CTW = 8 / KG;
    const bool half = x->dtype == MJT_FLOAT16;
    const bool ok = G == 1 && (x->dtype == MJT_BFLOAT16 || half) && dy->dtype == x->dtype && (dw->dtype == MJT_FLOAT32 || dw->dtype == x->dtype) &&
                    p->stride_w == 1 && p->pad_w <= 2 && (S - 1) * p->dil_w - p->pad_w <= 4 && K % 64 == 0 && C % 16 == 0 && (C % (16 * CTW) == 0 || C % (16 * CTW) >= 8 * CTW) && R * S <= 9 && OW % 2 == 0 &&
                    W % 2 == 0 && N >= 1 && numel(x) * 2 < (int64_t(1) << 31) && numel(dy) * 2 < (int64_t(1) << 31) &&
                    (uintptr_t)x->ptr % 4 == 0 && (uintptr_t)dy->ptr % 16 == 0 &&
                    !getenv("MJT_NO_FASTPATH");
    // 16-bit operands: the product instead of the MFMA kernel for 1x1 taps without stride and padding, whose operands it reads as they
    // lie, and for maps that fill less than 0.6 of the kernel's chunks of 32 columns (us at 64 images, kernel / product:
    // 1024 x 14 x 14 1x1 -> 256 65.9 / 21.7; 256 x 28 x 28 1x1 -> 128 25.5 / 16.5; 256 x 14 x 14 3x3 -> 256 70.6 / 60.7;
    // 128 x 28 x 28 3x3 -> 128 54.8 / 62.0 stays), from 2^27 multiply-adds on.  Smaller layers stay on the kernel they had (16 x 64 x
    // 14 x 14 3x3 -> 64 20.5 / 12.0, 8 x 256 x 14 x 14 1x1 -> 256 14.1 / 8.3, 4 x 64 x 6 x 6 3x3 -> 64 12.8 / 8.7); the front end sends the
    // narrow ones of them to the product over chunks of images instead of here.
    const bool narrow = OW % 8 != 0 && (double)OW < 0.6 * 32 * (double)((OW + 31) / 32);
    const bool planes = R * S == 1 && p->stride_h == 1 && p->stride_w == 1 && p->pad_h == 0 && p->pad_w == 0;
    const bool large = (double)N * OH * OW * K * C * R * S >= (double)(1 << 27);
    if ((!ok || (OH * OW % 2 == 0 && (planes || narrow) && large)) && G == 1 && N >= 1 && conv_wgrad_product(x, dy, dw, p)) return;
    // What is left for the MFMA kernel, on maps whose rows the windows take (us, kernel / windows: 64 x 128 x 28 x 28 3x3 -> 128 55.0 / 41.7;
    // 64 x 512 x 8 x 8 -> 512 93.9 / 37.0; 64 x 64 x 28 x 28 -> 64 39.1 / 30.3; 1 x 128 x 8 x 8 -> 64 15.0 / 13.2; a few images of few
    // channels stay: 1 x 64 x 14 x 14 -> 64 12.0 / 13.3, 1 x 64 x 28 x 28 -> 64 13.0 / 13.7).
    // (MJT_WGRAD_IPS, MJT_WGRAD_RPS: that kernel's slices, for experiments)
    if (ok && R * S > 1 && !getenv("MJT_WGRAD_IPS") && !getenv("MJT_WGRAD_RPS") && (K * C >= 8192 || (double)N * OH * OW * K * C * R * S >= (double)(1 << 25)) && conv_wgrad_window(x, dy, dw, p, 1e30)) return;
    if (!ok && any_shape) {
        conv_wgrad_direct(x, dy, dw, p, G);
        return;
    }
    if (!ok)
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv wgrad: only bfloat16 or float16 operands with horizontal stride 1, column shifts of the taps within -2 .. 4, at most 9 taps, "
                                      "K % 64 == 0, C % 16 == 0 (the last block of " << 16 * CTW << " channels at least half full), even OW and tensors below 2 GB run on the MFMA kernel");
    Context& c = ctx();
    const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
    const int64_t blocks_per_slice = (K / (64 * KG)) * ((C + 16 * CTW - 1) / (16 * CTW));   // the last block of channels may be partly idle
    // slices of consecutive output rows of the batch (a part of an image, or several images): enough workgroups for every
    // compute unit, at least 4 rows per slice (with whole images per slice, 64 x 64 x 56 x 56 with 3x3 taps ran 64
    // workgroups: 158 us)
    const int64_t rows = N * OH;
    int64_t slices = (cus + blocks_per_slice - 1) / blocks_per_slice;
    if (slices > (rows + 3) / 4) slices = (rows + 3) / 4;
    if (slices < 1) slices = 1;
    int64_t rps = (rows + slices - 1) / slices;
    if (const char* e = getenv("MJT_WGRAD_IPS"))             // images per slice, for experiments
        if (atoi(e) >= 1) rps = (atoi(e) < N ? atoi(e) : N) * OH;
    if (const char* e = getenv("MJT_WGRAD_RPS"))             // rows per slice, likewise
        if (atoi(e) >= 1) rps = atoi(e) < rows ? atoi(e) : rows;
    slices = (rows + rps - 1) / rps;

    const int abl = getenv("MJT_ABLATE_WGRAD") ? atoi(getenv("MJT_ABLATE_WGRAD")) : 0;    // timing-only ablations (bench.py --ablate): results are wrong
    MJT_CHECK(abl >= 0 && abl <= 63, "conv wgrad: MJT_ABLATE_WGRAD must be 0 .. 63");
    std::ostringstream key;
    key << "wgrad|" << abl << "|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << p->stride_h << "|"
        << p->pad_h << "|" << p->pad_w << "|" << p->dil_h << "|" << p->dil_w << "|" << KG << "|" << half;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_wgrad_mfma_" << (half ? "f16" : "bf16") << "_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << p->stride_h
             << "x1_p" << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K
            << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH << "\n#define OW_ " << OW << "\n#define SH "
            << p->stride_h << "\n#define PH " << p->pad_h << "\n#define PW " << p->pad_w << "\n#define DH " << p->dil_h << "\n#define DW "
            << p->dil_w << "\n#define KG " << KG << "\n#define IN_F16 " << (half ? 1 : 0) << "\n#define ABL " << abl << "\n";
        src << embedded_source("conv_wgrad_mfma.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    // (as in the forward kernel: a build that had to move registers aside is not run; its accumulators are vector registers)
    if (k->spilled != 0 || k->agprs != 0) {
        if (any_shape) {
            conv_wgrad_direct(x, dy, dw, p, G);
            return;
        }
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv wgrad: the MFMA kernel for this shape needs more registers than a wave has");
    }
    void* part = wgrad_partials((size_t)slices * (size_t)numel(dw) * 4);
    std::vector<uint64_t> a{bits_of_ptr(x->ptr), bits_of_ptr(dy->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)rps, 0};
    jit_launch(k, (unsigned)((slices + 7) / 8 * 8 * blocks_per_slice), 1, 512, 0, a);
    fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
}

}  // namespace mjt

extern "C" int mjt_conv2d_meta_wgrad(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p) {
    return mjt::guarded([&] { mjt::conv_wgrad_impl(x, dy, dw, p, 1, false); });
}

extern "C" int mjt_conv2d_meta_wgrad_grouped(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* dw, const mjt_conv_params* p,
                                             int groups) {
    return mjt::guarded([&] { mjt::conv_wgrad_impl(x, dy, dw, p, groups, true); });
}

namespace mjt {
// All stride phases of an input gradient in one launch behind the weights' packing (kernels/conv_dgrad_phases.h): 16-bit operands, strides 1 and 2, any
// padding and dilation; no shape of these that was timed is slower than before.  False: not covered.
static bool conv_dgrad_all_phases(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p) {
    const int64_t N = dx->shape[0], C = dx->shape[1], H = dx->shape[2], W = dx->shape[3];
    const int64_t K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = w->shape[2], S = w->shape[3], taps = R * S;
    const int64_t SH = p->stride_h, SW = p->stride_w, PH = p->pad_h, PW = p->pad_w, DH = p->dil_h, DW = p->dil_w;
    const bool half = dy->dtype == MJT_FLOAT16, narrow = dx->dtype == dy->dtype;
    if (!(half || dy->dtype == MJT_BFLOAT16) || SH > 2 || SW > 2 || SH * SW == 1 || taps < 1 || taps > 25 || getenv("MJT_NO_FASTPATH") || getenv("MJT_CONV_DGRAD_NO_PHASES")) return false;
    if (numel(dy) < 1 || numel(dy) * 2 >= (int64_t(1) << 31) || numel(dx) >= (int64_t(1) << 31) || H > 4096 || W > 4096 || (R - 1) * DH > 64 || (S - 1) * DW > 64 ||
        (uintptr_t)dy->ptr % 4 || (uintptr_t)dx->ptr % 8)
        return false;
    // the kernel's layout: margins that the taps' shifts reach, and the positions between the first and the last that a tile reads
    auto phase = [](int64_t t, int64_t stride) { return (t % stride + stride) % stride; };
    int64_t rlo = 0, rhi = 0, clo = 0, chi = 0;
    for (int64_t r = 0; r < R; r++) {
        const int64_t d = (phase(r * DH - PH, SH) + PH - r * DH) / SH;
        rlo = std::min(rlo, d);
        rhi = std::max(rhi, d);
    }
    for (int64_t s = 0; s < S; s++) {
        const int64_t d = (phase(s * DW - PW, SW) + PW - s * DW) / SW;
        clo = std::min(clo, d);
        chi = std::max(chi, d);
    }
    const int64_t unit = OW % 2 == 0 ? 2 : 1, HB = (H + SH - 1) / SH, WB = (W + SW - 1) / SW, lpc = (-clo + unit - 1) / unit * unit;
    const int64_t PR = HB + rhi - rlo, PC = (lpc + WB + chi + unit - 1) / unit * unit, total = N * HB * WB, CT = (C + 63) / 64;
    if (N * PR * PC >= (int64_t(1) << 30)) return false;
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    const int64_t PT = (total + 127) / 128 * CT >= cus ? 2 : 1, span = MarginPlanes{total, HB * WB, WB, PR, PC, rlo, rhi, clo, chi, lpc, unit}.span(64 * PT), tiles = (total + 64 * PT - 1) / (64 * PT) * CT;
    // A stage of 6 to 9 taps is 16 channels of dy, of fewer taps more, so that its MFMAs take longer than its barrier.  Where every workgroup has
    // a compute unit to itself nothing hides a stage's latency: twice as many (us, 16 / 32 channels: 1 x 512 x 7 x 7 -> 512 29.0 / 26.4, 8 x 256 x 28 x 28 -> 256 17.8 / 16.7).
    auto fits = [&](int64_t ku) { return 2 * ku * (taps * 2048 + span * 32) <= 160 * 1024 && span / unit * 2 * ku <= 4 * 256; };
    int64_t KU = taps >= 6 ? 1 : taps >= 3 ? 2 : 4;
    if (tiles <= cus && KU * 16 < K && fits(2 * KU)) KU *= 2;
    const int64_t stages = (K + 16 * KU - 1) / (16 * KU), packed = CT * stages * KU * taps * 2048;
    if (!fits(KU) || packed >= (int64_t(1) << 31) || tiles >= (1 << 28)) return false;
    std::ostringstream key;
    key << "dgphases|" << C << "|" << H << "|" << W << "|" << K << "|" << R << "|" << S << "|" << OH << "|" << OW << "|" << SH << "|" << SW << "|" << PH << "|" << PW << "|" << DH << "|" << DW
        << "|" << half << narrow << "|" << PT << "|" << KU << "|" << span;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_conv_mfma_" << (half ? "f16" : "bf16") << "_dgrad_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << SH << "x" << SW << "_p" << PH << "x" << PW
             << "_d" << DH << "x" << DW << "_o" << (narrow ? (half ? "f16" : "bf16") : "f32") << "_t" << 64 * PT << "_ku" << KU;
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define IN_F16 " << half << "\n#define Y_16 " << narrow << "\n#define KU " << KU << "\n#define PT " << PT << "\n#define SPAN " << span
            << "\n#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH
            << "\n#define OW_ " << OW << "\n#define SH " << SH << "\n#define SW " << SW << "\n#define PH " << PH << "\n#define PW " << PW << "\n#define DH " << DH << "\n#define DW " << DW << "\n";
        src << embedded_source("conv_dgrad_phases.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0) return false;
    void* wbuf = conv_scratch(2, (size_t)packed);
    mjt_tensor tw;
    memset(&tw, 0, sizeof(tw));
    tw.ptr = wbuf;
    tw.dtype = w->dtype;
    for (int64_t e : {CT, stages, KU, taps, int64_t(2), int64_t(64), int64_t(8)}) tw.shape[tw.ndim++] = e;
    const std::string ks = "i1*" + std::to_string(16 * KU) + "+i2*16+i4*8+i6", cs = "i0*64+i5", rs = "i3/" + std::to_string(S), ss = "i3%" + std::to_string(S);
    const std::string over_k = ks + ">=" + std::to_string(K), over_c = cs + ">=" + std::to_string(C);
    const char* idx[4] = {ks.c_str(), cs.c_str(), rs.c_str(), ss.c_str()};
    const char* over[2] = {over_k.c_str(), over_c.c_str()};
    if (mjt_reindex(w, &tw, 4, idx, 0.0, 2, over, 0, nullptr) != MJT_OK) MJT_FAIL(MJT_ERR_DEVICE, "conv dgrad: a rearrangement failed: " << mjt_last_error());
    std::vector<uint64_t> a{bits_of_ptr(wbuf), bits_of_ptr(dy->ptr), bits_of_ptr(dx->ptr), (uint64_t)N, (uint64_t)(numel(dy) * 2), (uint64_t)packed};
    jit_launch(k, (unsigned)((tiles + 7) / 8 * 8), 1, 256, 0, a);
    set_last_kernel(k->name.c_str());
    return true;
}

// The same for a few thousand results of any of the types, from dy and w as they lie (kernels/conv_dgrad_direct.h).
static void conv_dgrad_direct(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p) {
    const int64_t C = dx->shape[1], H = dx->shape[2], W = dx->shape[3], K = dy->shape[1], OH = dy->shape[2], OW = dy->shape[3], R = w->shape[2], S = w->shape[3];
    const int64_t total = numel(dx), lpo = K >= 32 ? 16 : K >= 8 ? 8 : K >= 4 ? 4 : 1;
    std::ostringstream geo, name;
    geo << "#define C_ " << C << "\n#define H_ " << H << "\n#define W_ " << W << "\n#define K_ " << K << "\n#define R_ " << R << "\n#define S_ " << S << "\n#define OH_ " << OH << "\n#define OW_ " << OW
        << "\n#define SH " << p->stride_h << "\n#define SW " << p->stride_w << "\n#define PH " << p->pad_h << "\n#define PW " << p->pad_w << "\n#define DH " << p->dil_h << "\n#define DW " << p->dil_w
        << "\n#define LPO " << lpo << "\n#define TIN " << dtype_cname(dy->dtype) << "\n#define TOUT " << dtype_cname(dx->dtype) << "\n";
    const EpilogueCode ep = epilogue_code(1, 4, dx->dtype, total);
    const std::string key = "dgdirect|" + geo.str() + ep.key;
    JitKernel* k = cached(key);
    if (!k) {
        name << "mjt_conv_direct_dgrad_" << mjt_dtype_name(dy->dtype) << "_" << mjt_dtype_name(dx->dtype) << "_c" << C << "_k" << K << "_" << H << "x" << W << "_r" << R << "x" << S << "_s" << p->stride_h << "x"
             << p->stride_w << "_p" << p->pad_h << "x" << p->pad_w << "_d" << p->dil_h << "x" << p->dil_w << ep.suffix();
        k = jit_get(ep.defs + "#define ENTRY " + name.str() + "\n" + geo.str() + (ep.on ? "" : embedded_source("prelude.h")) + "\n" + embedded_source("conv_dgrad_direct.h") + "\n", name.str());
        remember(key, k);
    }
    std::vector<uint64_t> a{bits_of_ptr(dy->ptr), bits_of_ptr(w->ptr), bits_of_ptr(dx->ptr), (uint64_t)total};
    a.insert(a.end(), ep.words.begin(), ep.words.end());
    epilogue_taken(ep);
    jit_launch(k, (unsigned)((total * lpo + 255) / 256), 1, 256, 0, a);
    set_last_kernel(k->name.c_str());
}

// Input gradient of the convolution y = conv(x, w): dx[n,c,h,w] = sum over (k, r, s) of dy[n,k,oh,ow] * w[k,c,r,s] with
// h = oh*sh - ph + r*dh, w = ow*sw - pw + s*dw.  It is itself a convolution of dy, run on the forward kernels:
//   * 16-bit operands at strides 1 and 2 other than 1 x 1: one launch for all phases (above);
//   * any other stride above 1 with few multiply-adds: one launch, a result at a time (conv_dgrad_direct);
//   * stride 1: with the weights transposed and their taps flipped, padding d*(R-1) - p;
//   * a stride without dilation, H and W multiples of it: one stride-1 convolution per stride phase.  The rows
//     h = sh*i + a of dx see only the taps r = r_a + sh*u (r_a = (a + ph) % sh, u = 0 .. U_a - 1) and
//     dx[sh*i + a] = sum_u dy[i + d_a - u] * w[r_a + sh*u] with d_a = (a + ph) / sh: a convolution of dy with U_a taps
//     (flipped) and left padding U_a - 1 - d_a, likewise for columns.  No product has a zero factor; the phases
//     are written one after the other and interleaved by one reindex;
//   * otherwise: dy with sh-1 (sw-1) zeros between its rows (columns), then as for stride 1.
void conv_dgrad_impl(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p) {
    require_init();
    check_tensor(dy, "conv dgrad dy");
    check_tensor(w, "conv dgrad w");
    check_tensor(dx, "conv dgrad dx");
    MJT_CHECK(p, "conv dgrad: null parameters");
    MJT_CHECK(dy->ndim == 4 && w->ndim == 4 && dx->ndim == 4, "conv dgrad: dy, w and dx must have rank 4");
    MJT_CHECK(dy->dtype == w->dtype && (dy->dtype == MJT_BFLOAT16 || dy->dtype == MJT_FLOAT16 || dy->dtype == MJT_FLOAT32),
              "conv dgrad: dy and w must both be bfloat16, float16 or float32");
    MJT_CHECK(dx->dtype == MJT_FLOAT32 || dx->dtype == dy->dtype, "conv dgrad: dx must be float32 or the operands' dtype");
    const int64_t N = dx->shape[0], C = dx->shape[1], H = dx->shape[2], W = dx->shape[3];
    const int64_t K = w->shape[0], R = w->shape[2], S = w->shape[3];
    const int64_t sh = p->stride_h, sw = p->stride_w, ph = p->pad_h, pw = p->pad_w, dh = p->dil_h, dw = p->dil_w;
    MJT_CHECK(sh >= 1 && sw >= 1 && dh >= 1 && dw >= 1 && ph >= 0 && pw >= 0, "conv dgrad: bad stride / padding / dilation");
    MJT_CHECK(w->shape[1] == C, "conv dgrad: weight channels " << w->shape[1] << " != dx channels " << C);
    const int64_t OH = (H + 2 * ph - dh * (R - 1) - 1) / sh + 1, OW = (W + 2 * pw - dw * (S - 1) - 1) / sw + 1;
    MJT_CHECK(dy->shape[0] == N && dy->shape[1] == K && dy->shape[2] == OH && dy->shape[3] == OW,
              "conv dgrad: dy shape " << shape_str(dy) << " != [" << N << "," << K << "," << OH << "," << OW << "]");
    MJT_CHECK(dh * (R - 1) >= ph && dw * (S - 1) >= pw, "conv dgrad: padding beyond the taps' reach is not supported");
    if (N == 0 || C == 0) return;
    if (conv_dgrad_all_phases(dy, w, dx, p)) return;
    const int64_t esz = dtype_size(w->dtype);
    auto view = [](void* ptr, int dtype, std::initializer_list<int64_t> shape) {
        mjt_tensor t;
        memset(&t, 0, sizeof(t));
        t.ptr = ptr;
        t.dtype = dtype;
        for (int64_t e : shape) t.shape[t.ndim++] = e;
        return t;
    };
    auto reindex = [&](const mjt_tensor& src, const mjt_tensor& dst, std::initializer_list<std::string> idx, std::initializer_list<std::string> over) {
        std::vector<const char*> ip, op;
        for (const std::string& e : idx) ip.push_back(e.c_str());
        for (const std::string& e : over) op.push_back(e.c_str());
        if (mjt_reindex(&src, &dst, (int)ip.size(), ip.data(), 0.0, (int)op.size(), op.data(), 0, nullptr) != MJT_OK)
            MJT_FAIL(MJT_ERR_DEVICE, "conv dgrad: a rearrangement failed: " << mjt_last_error());
    };
    auto str = [](int64_t v) { return std::to_string(v); };
    void* wbuf = conv_scratch(2, (size_t)(numel(w) * esz));

    // the taps of each stride phase along one axis: first tap, number of taps, left padding (-1: not expressible)
    struct Phase { int64_t first, taps, pad; };
    auto phases = [](int64_t stride, int64_t pad, int64_t taps) {
        std::vector<Phase> v;
        for (int64_t a = 0; a < stride; a++) {
            Phase q;
            q.first = (a + pad) % stride;
            q.taps = q.first < taps ? (taps - q.first + stride - 1) / stride : 0;
            q.pad = q.taps ? q.taps - 1 - (a + pad) / stride : 0;
            v.push_back(q);
        }
        return v;
    };
    bool by_phase = (sh > 1 || sw > 1) && dh == 1 && dw == 1 && H % sh == 0 && W % sw == 0 && !getenv("MJT_CONV_DGRAD_NO_PHASES");
    std::vector<Phase> rows, cols;
    if (by_phase) {
        rows = phases(sh, ph, R);
        cols = phases(sw, pw, S);
        for (const Phase& q : rows) by_phase = by_phase && q.pad >= 0;
        for (const Phase& q : cols) by_phase = by_phase && q.pad >= 0;
    }
    // Few multiply-adds: all phases in one launch, a result at a time.  It looks at every tap of every channel, 1.2 us a million (float32, us,
    // phase by phase in five or six launches / so: 4 x 16 x 6 x 6 3x3 -> 16 22.8 / 3.6, 4 x 16 x 16 x 16 -> 16 17.8 / 5.3, 2 x 8 x 8 x 8 -> 8 10.6 / 2.9; on the
    // other side, 47 and 58 million, 13 x 48 x 18 x 18 3x3 -> 26 28.8 / 53.9, 8 x 64 x 14 x 14 3x3 -> 64 34.0 / 77.2).
    if ((sh > 1 || sw > 1) && K > 0 && !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_DGRAD_NO_DIRECT") && !getenv("MJT_CONV_DGRAD_NO_PHASES") && R * S <= 49 && numel(dx) >= 1 && numel(dy) >= 1 &&
        numel(dy) < (int64_t(1) << 30) && (double)numel(dx) * K * R * S < (double)(1 << 23)) {
        conv_dgrad_direct(dy, w, dx, p);
        return;
    }
    if (by_phase) {
        const int64_t Hs = H / sh, Ws = W / sw, dsz = dtype_size(dx->dtype);
        const int64_t plane = N * C * Hs * Ws;
        char* part = (char*)conv_scratch(3, (size_t)(sh * sw * plane * dsz));
        const mjt_conv_params unit = {1, 1, 0, 0, 1, 1};
        std::string kernels;
        // The weights of all phases in one pass (the phases partition the taps): w [K,C,R,S] -> one block [C,K,U,V] per
        // phase, the phase's taps flipped, the blocks one after the other.  Seen from the flat offset i0 of that buffer,
        // block p covers [off_p, off_p + C*K*U*V) and its element (c, k, u, v) reads w[k, c, first_r + sh*(U-1-u),
        // first_c + sw*(V-1-v)]: four index expressions, each a chain of conditions on i0.
        std::vector<int64_t> woff((size_t)(sh * sw), -1);
        {
            std::string ek = "0", ec = "0", er = "0", es = "0";
            int64_t off = 0;
            std::vector<std::array<std::string, 4>> pieces;
            std::vector<int64_t> ends;
            for (int64_t a = 0; a < sh; a++)
                for (int64_t b = 0; b < sw; b++) {
                    const Phase &qr = rows[a], &qc = cols[b];
                    if (qr.taps == 0 || qc.taps == 0) continue;
                    woff[(size_t)(a * sw + b)] = off;
                    const int64_t U = qr.taps, V = qc.taps;
                    const std::string l = "(i0-" + str(off) + ")";
                    pieces.push_back({l + "/" + str(U * V) + "%" + str(K), l + "/" + str(K * U * V),
                                      str(qr.first) + "+" + str(sh) + "*(" + str(U - 1) + "-" + l + "/" + str(V) + "%" + str(U) + ")",
                                      str(qc.first) + "+" + str(sw) + "*(" + str(V - 1) + "-" + l + "%" + str(V) + ")"});
                    off += C * K * U * V;
                    ends.push_back(off);
                }
            if (!pieces.empty()) {
                std::array<std::string, 4> e = pieces.back();
                for (int i = (int)pieces.size() - 2; i >= 0; i--)
                    for (int j = 0; j < 4; j++) e[j] = "(i0<" + str(ends[i]) + " ? " + pieces[i][j] + " : " + e[j] + ")";
                mjt_tensor tall = view(wbuf, w->dtype, {off});
                reindex(*w, tall, {e[0], e[1], e[2], e[3]}, {});
            }
        }
        for (int64_t a = 0; a < sh; a++)
            for (int64_t b = 0; b < sw; b++) {
                const Phase &qr = rows[a], &qc = cols[b];
                mjt_tensor ty = view(part + (a * sw + b) * plane * dsz, dx->dtype, {N, C, Hs, Ws});
                if (qr.taps == 0 || qc.taps == 0) {                 // no tap reaches these positions: zeros (the source, of the same type, is not read)
                    reindex(ty, ty, {"0", "0", "0", "0"}, {"1"});
                    continue;
                }
                mjt_tensor tw = view((char*)wbuf + woff[(size_t)(a * sw + b)] * esz, w->dtype, {C, K, qr.taps, qc.taps});
                mjt_conv_params q = unit;
                q.pad_h = (int32_t)qr.pad;
                q.pad_w = (int32_t)qc.pad;
                conv_impl(dy, &tw, &ty, &q, 1, true);
                if (kernels.empty()) kernels = mjt_last_kernel();
            }
        mjt_tensor tp = view(part, dx->dtype, {sh * sw, N, C, Hs, Ws});
        reindex(tp, *dx, {"i2%" + str(sh) + "*" + str(sw) + "+i3%" + str(sw), "i0", "i1", "i2/" + str(sh), "i3/" + str(sw)}, {});
        set_last_kernel(("conv_dgrad_phases:" + kernels).c_str());
        return;
    }
    // a 1x1 convolution: the product takes the weights as they lie
    if (R == 1 && S == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0 && !getenv("MJT_NO_FASTPATH") && !getenv("MJT_CONV_NO_GEMM") &&
        (double)N * K * C * H * W >= (double)(1 << 22) && gemm_pixels(dy->dtype, dx->dtype, w->ptr, dy->ptr, dx->ptr, C, K, H * W, N, false)) {
        set_last_kernel("conv_as_gemm");
        return;
    }
    mjt_tensor tw = view(wbuf, w->dtype, {C, K, R, S});
    const FlippedWeights flipped{w, [&] {
        Preparing preparing;
        reindex(*w, tw, {"i1", "i0", str(R - 1) + "-i2", str(S - 1) + "-i3"}, {});
    }};
    const mjt_conv_params q = {1, 1, (int32_t)(dh * (R - 1) - ph), (int32_t)(dw * (S - 1) - pw), (int32_t)dh, (int32_t)dw};
    if (sh == 1 && sw == 1) {
        conv_run(dy, &tw, dx, &q, 1, false, 0, nullptr, &flipped);
        return;
    }
    flipped.fill();
    const int64_t ZH = H + 2 * ph - dh * (R - 1), ZW = W + 2 * pw - dw * (S - 1);
    mjt_tensor tz = view(conv_scratch(3, (size_t)(N * K * ZH * ZW * esz)), dy->dtype, {N, K, ZH, ZW});
    {
        Preparing preparing;
        reindex(*dy, tz, {"i0", "i1", "i2/" + str(sh), "i3/" + str(sw)}, {"i2%" + str(sh) + "!=0", "i3%" + str(sw) + "!=0"});
    }
    conv_impl(&tz, &tw, dx, &q, 1);
}
}  // namespace mjt

namespace mjt {
// Input gradient of a depthwise convolution with as many output as input channels: one launch on the forward kernel, which
// reads the taps from the last to the first and keeps the rows and columns of a strided dy apart.
void conv_dgrad_depthwise(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p, int64_t G) {
    require_init();
    check_tensor(dy, "conv dgrad dy");
    check_tensor(w, "conv dgrad w");
    check_tensor(dx, "conv dgrad dx");
    MJT_CHECK(p, "conv dgrad: null parameters");
    MJT_CHECK(dy->ndim == 4 && w->ndim == 4 && dx->ndim == 4, "conv dgrad: dy, w and dx must have rank 4");
    MJT_CHECK(dy->dtype == w->dtype && (dy->dtype == MJT_BFLOAT16 || dy->dtype == MJT_FLOAT16 || dy->dtype == MJT_FLOAT32),
              "conv dgrad: dy and w must both be bfloat16, float16 or float32");
    MJT_CHECK(dx->dtype == MJT_FLOAT32 || dx->dtype == dy->dtype, "conv dgrad: dx must be float32 or the operands' dtype");
    MJT_CHECK(p->stride_h >= 1 && p->stride_w >= 1 && p->dil_h >= 1 && p->dil_w >= 1 && p->pad_h >= 0 && p->pad_w >= 0,
              "conv dgrad: bad stride / padding / dilation");
    const int64_t C = dx->shape[1], H = dx->shape[2], W = dx->shape[3], R = w->shape[2], S = w->shape[3];
    const int64_t OH = (H + 2 * p->pad_h - p->dil_h * (R - 1) - 1) / p->stride_h + 1, OW = (W + 2 * p->pad_w - p->dil_w * (S - 1) - 1) / p->stride_w + 1;
    MJT_CHECK(G >= 1 && C % G == 0 && w->shape[0] % G == 0, "conv dgrad: channels do not split into " << G << " groups");
    MJT_CHECK(dy->shape[0] == dx->shape[0] && dy->shape[1] == w->shape[0] && dy->shape[2] == OH && dy->shape[3] == OW,
              "conv dgrad: dy shape " << shape_str(dy) << " does not follow from dx " << shape_str(dx) << " and w " << shape_str(w));
    if (G < 2 || C != G || w->shape[0] != G || w->shape[1] != 1) MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv dgrad: only depthwise convolutions with as many output as input channels");
    if (numel(dx) == 0) return;
    const DepthwiseShape g{OH, OW, H, W, R, S, 1, 1, p->dil_h * (R - 1) - p->pad_h, p->dil_w * (S - 1) - p->pad_w, p->dil_h, p->dil_w, p->stride_h, p->stride_w, C, 1, true};
    if (numel(dy) == 0 || !depthwise_run(g, dy, w, dx)) MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv dgrad: this shape takes another route");
}

// Both gradients of a depthwise convolution of stride 1 with as many output as input channels, in one kernel over dy and x.
void conv_backward_depthwise(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_tensor* dw, const mjt_conv_params* p,
                             int64_t G) {
    require_init();
    check_tensor(x, "conv backward x");
    check_tensor(dy, "conv backward dy");
    check_tensor(w, "conv backward w");
    check_tensor(dx, "conv backward dx");
    check_tensor(dw, "conv backward dw");
    MJT_CHECK(p, "conv backward: null parameters");
    MJT_CHECK(x->ndim == 4 && dy->ndim == 4 && w->ndim == 4 && dx->ndim == 4 && dw->ndim == 4, "conv backward: every tensor must have rank 4");
    MJT_CHECK(x->dtype == dy->dtype && x->dtype == w->dtype && (x->dtype == MJT_BFLOAT16 || x->dtype == MJT_FLOAT16 || x->dtype == MJT_FLOAT32),
              "conv backward: x, dy and w must share one of float32 / bfloat16 / float16");
    MJT_CHECK((dx->dtype == MJT_FLOAT32 || dx->dtype == x->dtype) && (dw->dtype == MJT_FLOAT32 || dw->dtype == x->dtype), "conv backward: dx and dw must be float32 or the operands' dtype");
    const int64_t N = x->shape[0], C = x->shape[1], H = x->shape[2], W = x->shape[3], R = w->shape[2], S = w->shape[3], OH = dy->shape[2], OW = dy->shape[3];
    for (int i = 0; i < 4; i++) MJT_CHECK(dx->shape[i] == x->shape[i] && dw->shape[i] == w->shape[i], "conv backward: dx and dw must have the shapes of x and w");
    MJT_CHECK(dy->shape[0] == N && dy->shape[1] == w->shape[0], "conv backward: dy " << shape_str(dy) << " does not follow from x " << shape_str(x) << " and w " << shape_str(w));
    if (G < 2 || C != G || w->shape[0] != G || w->shape[1] != 1 || p->stride_h != 1 || p->stride_w != 1 || p->dil_h != 1 || p->dil_w != 1)
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv backward: only depthwise convolutions of stride 1 without dilation, with as many output as input channels");
    MJT_CHECK(OH == H + 2 * p->pad_h - R + 1 && OW == W + 2 * p->pad_w - S + 1, "conv backward: dy " << shape_str(dy) << " does not follow from x " << shape_str(x));
    if (numel(x) == 0 || numel(dy) == 0 || p->pad_h < 0 || p->pad_w < 0 || p->pad_h > R - 1 || p->pad_w > S - 1 || getenv("MJT_NO_FASTPATH"))
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv backward: this shape takes another route");
    const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
    // slices of images: as many workgroups as the compute units hold at once, four each, or two where more taps take more registers (us
    // with 2 / 3 / 4 / 6 a unit: 32 x 128 x 56 x 56 3x3 float32 38.0 / 39.3 / 37.0 / 38.6, 32 x 96 x 31 x 29 19.1 / 17.6 / 18.5 / 21.2; 5x5 64 x 24 x 56 x 56
    // 26.1 / 33.7 / 34.3 / 39.2, 64 x 512 x 14 x 14 30.7 / 30.2 / 39.8 / 49.0)
    int64_t slices = (R * S <= 9 ? 4 : 2) * cus / C;
    if (slices < 1) slices = 1;
    if (slices > N) slices = N;
    if (N * OH * OW < 2048) slices = 1;
    const int64_t ips = (N + slices - 1) / slices;
    slices = (N + ips - 1) / ips;
    const DepthwiseShape g{OH, OW, H, W, R, S, 1, 1, R - 1 - p->pad_h, S - 1 - p->pad_w, 1, 1, 1, 1, C, 1, true};
    DepthwisePlan q;
    // (strips are read from x and written to dx: vectors that suit both)
    const int wide = std::max(dtype_size(x->dtype), dtype_size(dx->dtype));
    const void* strips = (const void*)((uintptr_t)x->ptr | (uintptr_t)dx->ptr);
    if (slices * C >= (int64_t(1) << 31) || !depthwise_plan(g, dtype_size(dy->dtype), wide, dy->ptr, strips, int64_t(1) << 40, ips, &q))
        MJT_FAIL(MJT_ERR_UNSUPPORTED, "conv backward: this shape takes another route");
    JitKernel* k = depthwise_kernel(2, g, q, x->dtype, dx->dtype);
    const bool in_place = slices == 1 && dw->dtype == MJT_FLOAT32;
    void* part = in_place ? dw->ptr : wgrad_partials((size_t)slices * (size_t)numel(dw) * 4);
    std::vector<uint64_t> a{bits_of_ptr(dy->ptr), bits_of_ptr(x->ptr), bits_of_ptr(part), (uint64_t)N, (uint64_t)ips, bits_of_ptr(w->ptr), bits_of_ptr(dx->ptr)};
    jit_launch(k, (unsigned)(slices * C), 1, 256, 0, a);
    if (!in_place) fold_wgrad_slices(part, slices, dw);
    set_last_kernel(k->name.c_str());
}
}  // namespace mjt

extern "C" int mjt_conv2d_meta_backward_depthwise(const mjt_tensor* x, const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_tensor* dw,
                                                  const mjt_conv_params* p, int groups) {
    return mjt::guarded([&] { mjt::conv_backward_depthwise(x, dy, w, dx, dw, p, groups); });
}

extern "C" int mjt_conv2d_meta_dgrad_depthwise(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p, int groups) {
    return mjt::guarded([&] { mjt::conv_dgrad_depthwise(dy, w, dx, p, groups); });
}

extern "C" int mjt_conv2d_meta_dgrad(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p) {
    return mjt::guarded([&] { mjt::conv_dgrad_impl(dy, w, dx, p); });
}

extern "C" int mjt_conv2d_meta(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p) {
    return mjt::guarded([&] { mjt::conv_impl(x, w, y, p, 1); });
}

extern "C" int mjt_conv2d_meta_pack(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p,
                                    void* packed, size_t packed_bytes) {
    return mjt::guarded([&] {
        mjt::check_tensor(w, "conv w");
        MJT_CHECK(packed_bytes >= (size_t)mjt::numel(w) * mjt::dtype_size(w->dtype), "conv: the packed weights need as many bytes as w");
        mjt::conv_impl(x, w, y, p, 1, false, 1, packed);
    });
}

extern "C" int mjt_conv2d_meta_packed(const mjt_tensor* x, const mjt_tensor* w, const void* packed, const mjt_tensor* y,
                                      const mjt_conv_params* p) {
    return mjt::guarded([&] { mjt::conv_impl(x, w, y, p, 1, false, 2, const_cast<void*>(packed)); });
}

extern "C" int mjt_conv2d_meta_grouped(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p,
                                       int groups) {
    return mjt::guarded([&] { mjt::conv_impl(x, w, y, p, groups); });
}
