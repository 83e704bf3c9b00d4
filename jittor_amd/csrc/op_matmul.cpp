// Matrix product behind the reference's matmul relay.
//
// The reference recognises broadcast * broadcast -> reduce.add over 2-d
// operands (opt/tuner/matmul_tuner.cc:16-104) and relays it to a library GEMM:
// cublas_matmul(a, b, trans_a, trans_b) on the GPU
// (extern/cuda/cublas/ops/cublas_matmul_op.cc:27-56, batched form
// cublas_batched_matmul_op.cc:63-85).  Here the product runs on the library's
// own kernels: kernels/gemm_mfma.h (MFMA, LDS-tiled; bfloat16, float16 and
// float32 operands whose rows are 16-byte aligned) and kernels/gemm_plain.h
// (everything else, float64 included).  Float accumulation for every input
// type (double for float64).
#include "common.h"
#include <algorithm>
#include <cmath>
#include <mutex>
#include <unordered_map>

namespace mjt {

void launch_fill_pattern(void* dst, uint64_t pattern, int elem_size, size_t n);

namespace {
std::mutex g_mu;
std::unordered_map<std::string, JitKernel*> g_kernels;
void* g_rows[2] = {nullptr, nullptr};      // operands with rows padded to 16 bytes (guarded by the library's lock, as the scratch memory)
size_t g_rows_bytes[2] = {0, 0};
void forget() {   // the kernels belong to the run-time compiler's cache, which mjt_shutdown empties
    std::lock_guard<std::mutex> lock(g_mu);
    g_kernels.clear();
    for (int i = 0; i < 2; i++) {
        if (g_rows[i] && !ctx().dry_run) (void)hipFree(g_rows[i]);
        g_rows[i] = nullptr;
        g_rows_bytes[i] = 0;
    }
}
const bool g_registered = (at_shutdown(&forget), true);

JitKernel* cached(const std::string& key) {
    std::lock_guard<std::mutex> lock(g_mu);
    auto it = g_kernels.find(key);
    return it == g_kernels.end() ? nullptr : it->second;
}
void remember(const std::string& key, JitKernel* k) {
    std::lock_guard<std::mutex> lock(g_mu);
    g_kernels.emplace(key, k);
}
int env_int(const char* name, int dflt) {
    const char* v = getenv(name);
    return v && *v ? atoi(v) : dflt;
}

// [rows, ld] copied into rows of `ldp` elements (zeros behind each), into the buffer of operand `which`; null where there is no
// memory for it.
const void* padded_rows(int which, const void* src, int dtype, int64_t rows, int64_t ld, int64_t ldp) {
    Context& c = ctx();
    const size_t bytes = (size_t)(rows * ldp * dtype_size(dtype));
    if (!workspace_allowed(bytes) || !(c.dry_run || grow_kept(&g_rows[which], &g_rows_bytes[which], bytes))) return nullptr;
    mjt_tensor t{}, d{};
    t.ptr = (void*)src;
    d.ptr = c.dry_run ? (void*)(uintptr_t)0x1000 : g_rows[which];
    t.dtype = d.dtype = dtype;
    t.ndim = d.ndim = 2;
    t.shape[0] = d.shape[0] = rows;
    t.shape[1] = ld;
    d.shape[1] = ldp;
    Preparing preparing;
    const char* idx[2] = {"i0", "i1"};                          // columns past ld lie outside the source: overflow value 0
    if (mjt_reindex(&t, &d, 2, idx, 0.0, 0, nullptr, 0, nullptr) != MJT_OK) MJT_FAIL(MJT_ERR_DEVICE, "matmul: padding the rows failed: " << mjt_last_error());
    return d.ptr;
}
}  // namespace

// One strided-batched product C[b] = A'[b] * B'[b] over plain pointers: M x K times K x N, leading dimensions and
// batch strides in elements (a batch stride of 0 shares the operand).  a_kcont / b_kcont: the operand's memory has
// k innermost (a as given, b transposed).
void gemm_launch(int in_dtype, int out_dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                 int64_t lda, int64_t ldb, int64_t ldc, int64_t sa, int64_t sb, int64_t sc, int64_t batch, bool a_kcont,
                 bool b_kcont, int tile_m = 0, int tile_n = 0, bool allow_direct = true) {
    Context& c = ctx();
    const int esz = dtype_size(in_dtype);
    const bool mfma_type = in_dtype == MJT_BFLOAT16 || in_dtype == MJT_FLOAT16 || in_dtype == MJT_FLOAT32;
    const bool out_ok = out_dtype == MJT_FLOAT32 || (out_dtype == in_dtype && esz == 2);
    auto al16 = [&](const void* p, int64_t ld, int64_t stride) {
        return (uintptr_t)p % 16 == 0 && (ld * esz) % 16 == 0 && (stride * esz) % 16 == 0;
    };
    const bool fast = mfma_type && out_ok && !getenv("MJT_GEMM_PLAIN") && al16(A, lda, sa) && al16(B, ldb, sb) &&
                      M < (int64_t(1) << 31) && N < (int64_t(1) << 31) && K < (int64_t(1) << 31) && batch < 65536;
    std::vector<uint64_t> args{bits_of_ptr(A), bits_of_ptr(B), bits_of_ptr(C), (uint64_t)M, (uint64_t)N, (uint64_t)K,
                               (uint64_t)lda, (uint64_t)ldb, (uint64_t)ldc, (uint64_t)sa, (uint64_t)sb, (uint64_t)sc};
    // 16-bit operands, K a multiple of 64 and enough tiles of 256 x 256 to go round: the kernel whose operands reach LDS
    // without passing through registers (any of the four layouts).  Offsets inside an operand's tile are 32-bit there:
    // 256 rows of an operand with k innermost, all K rows of one with m or n innermost.
    auto fits32 = [&](bool kcont, int64_t ld) { return (kcont ? ld * 2 * 256 : ld * 2 * K) < (int64_t(1) << 31); };
    if (fast && allow_direct && esz == 2 && K % 64 == 0 && !getenv("MJT_GEMM_NO_DMA") && fits32(a_kcont, lda) && fits32(b_kcont, ldb)) {
        const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
        // 256 x 256 tiles on two stage buffers, or 128 x 128 tiles on a ring of four (a 128-tile's stage is a quarter of
        // the MFMA time, so more stages have to be on their way): the smaller tile where the larger one leaves compute
        // units without work
        int tile = 0;
        // a caller that names its tile has measured the general kernel against the 256 x 256 tiles; 128 x 128 tiles of this
        // kernel are still better than the general kernel's from two stages on (measured on 1x1 convolutions below)
        const bool hinted = tile_m || tile_n;
        const int smallest = hinted && !(tile_m == 128 && tile_n == 128 && K >= 128) ? 256 : 128;
        for (int t = 256; t >= smallest && !tile; t /= 2) {
            const int64_t tm = (M + t - 1) / t, tn = (N + t - 1) / t;
            const double edge = ((double)M * N) / ((double)tm * t * tn * t);
            const double tiles = (double)tm * tn * batch;
            const double util = tiles / (std::ceil(tiles / cus) * cus);
            // (a sum of fewer than four stages does not fill the time a 256 x 256 tile's operands take to arrive, and only
            // one such workgroup fits a compute unit)
            if (edge >= 0.85 && util >= (t == 256 ? 0.7 : 0.25) && (t == 128 || K >= 256)) tile = t;
        }
        if (const char* e = getenv("MJT_GEMM_DMA")) tile = atoi(e) == 128 ? 128 : 256;
        if (tile) {
            const int64_t tm = (M + tile - 1) / tile, tn = (N + tile - 1) / tile;
            const int in = in_dtype == MJT_BFLOAT16 ? 0 : 1;
            const int out = out_dtype == MJT_BFLOAT16 ? 0 : out_dtype == MJT_FLOAT16 ? 1 : 2;
            // a short sum on 128 x 128 tiles: two stage buffers, so that a compute unit holds two workgroups and one
            // computes or stores while the other waits for its operands
            // 128 x 128 tiles: with more tiles than compute units two stage buffers, so that a compute unit holds two
            // workgroups and one computes or stores while the other waits for its operands (us, ring of four / two
            // workgroups: 3072 x 3072 x 1024 35.4 / 31.7; 8192 x 1024 x 1024 26.8 / 22.1; 64 x 512 x 28 x 28 -> 512 as a
            // product 82.3 / 63.7); with at most one tile each a ring of four (2048^3 21.7 / 24.8; 1536^3 15.3 / 20.5)
            const int nbuf = tile == 256 ? 2 : (double)tm * tn * batch > (double)cus ? 2 : 4, wpe = tile == 128 && nbuf == 2 ? 2 : 1;
            // adjacent results that a lane stores: rows of C have to be such vectors, wherever a tile ends
            const int osz = dtype_size(out_dtype);
            auto whole = [&](int v) { return N % v == 0 && ldc % v == 0 && sc % v == 0 && (uintptr_t)C % (size_t)(v * osz) == 0; };
            const int vs = whole(4) ? 4 : whole(2) ? 2 : 1;
            const EpilogueCode ep = epilogue_code(vs, 12, out_dtype, ldc == N && (batch == 1 || sc == M * N) ? M * N * batch : -1);
            std::ostringstream key;
            key << "gemmd|" << in << out << a_kcont << b_kcont << tile << nbuf << vs << ep.key;
            JitKernel* k = cached(key.str());
            if (!k) {
                std::ostringstream name;
                name << "mjt_gemm_mfma_" << mjt_dtype_name(in_dtype) << "_" << mjt_dtype_name(out_dtype) << "_" << tile << "x" << tile << (a_kcont ? "_n" : "_t")
                     << (b_kcont ? "t" : "n") << "_direct" << (wpe == 2 ? "2" : "") << ep.suffix();
                std::ostringstream src;
                src << ep.defs << "#define VS " << vs << "\n#define ENTRY " << name.str() << "\n#define IN " << in << "\n#define OUT " << out << "\n#define A_KCONT " << (a_kcont ? 1 : 0)
                    << "\n#define B_KCONT " << (b_kcont ? 1 : 0) << "\n#define TILE " << tile << "\n#define NBUF " << nbuf << "\n#define WPE " << wpe << "\n";
                src << embedded_source("gemm_dma.h") << "\n";
                k = jit_get(src.str(), name.str());
                remember(key.str(), k);
            }
            // (the kernel keeps LDS reads under way in registers behind the compiler's back: a build that had to move
            // registers aside, into accumulation registers beyond the tile / 256 accumulators or into scratch memory,
            // is not run; the general kernel below takes the product)
            if (k->spilled == 0 && k->agprs >= 0 && k->agprs <= tile * tile / 256) {
                const int64_t grid = (tm * tn + 7) / 8 * 8;
                MJT_CHECK(grid < (int64_t(1) << 31), "matmul: launch too large");
                args.insert(args.end(), ep.words.begin(), ep.words.end());
                epilogue_taken(ep);
                jit_launch(k, (unsigned)grid, (unsigned)batch, 256, 0, args);
                return;
            }
            if (ep.on) check_no_epilogue();                      // (the product without the group is the better one)
        }
    }
    if (fast) {
        // Tile: the largest of 64 MI x 64 NI (MI, NI in 1, 2, 4) that still gives every compute unit work and wastes
        // little on the edges; larger tiles read each operand element less often.
        const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
        int best_mi = 1, best_ni = 1;
        double best = -1.0;
        for (int mi = 4; mi >= 1; mi /= 2)
            for (int ni = 4; ni >= 1; ni /= 2) {
                const int64_t tm = (M + 64 * mi - 1) / (64 * mi), tn = (N + 64 * ni - 1) / (64 * ni);
                const double tiles = (double)tm * tn * batch;
                const double edge = ((double)M * N) / ((double)tm * 64 * mi * tn * 64 * ni);
                const double waves = std::ceil(tiles / cus);
                const double util = tiles / (waves * cus);
                const double reuse = 1.0 / (1.0 / (64.0 * mi) + 1.0 / (64.0 * ni)) / 128.0;   // 1 for 256 x 256
                const double score = edge * util * (0.55 + 0.45 * reuse);
                if (score > best) { best = score; best_mi = mi; best_ni = ni; }
            }
        // the caller's tile, if it names one (tile_m x tile_n of 64, 128 or 256)
        if (tile_m == 64 || tile_m == 128 || tile_m == 256) best_mi = tile_m / 64;
        if (tile_n == 64 || tile_n == 128 || tile_n == 256) best_ni = tile_n / 64;
        // Few tiles and a long sum: the sum is cut into slices, whose float32 results a reduce launch adds up.  A stage (32 float32 or 64
        // 16-bit elements of the sum) of a 64 x 64 tile takes about 0.75 us in float32 and 0.5 in 16 bits with a compute unit to itself, 1.75 / 2.6 / 3.4 times that
        // with two / three / four workgroups a unit; the reduce launch 5 us and its traffic.  At most 16 slices: their reduce is
        // a single launch, which leaves the scratch memory alone.  (us whole / in slices; a^T b: 512 x 512 x 8192 float32
        // 183 / 50, bfloat16 64.5 / 22.7; 64 x 64 x 4096 float32 94 / 13.5; 1024 x 512 x 4096 float32 96 / 50; a b^T:
        // 256 x 1024 x 1024 float32 20.1 / 12.4; 1024 x 1024 x 2048 a^T b, 256 tiles, 50.4 / 50.6, stays whole.)
        const int64_t ks = esz == 2 ? 64 : 32, stages = (K + ks - 1) / ks;
        int64_t slices = 1, per = stages;
        bool split = false;
        const bool sliceable = batch == 1 && !tile_m && !tile_n && ldc == N;
        const double tiles64 = (double)((M + 63) / 64) * ((N + 63) / 64) * batch;
        auto crowd = [&](double wgs) { const double r = std::ceil(wgs / cus); return 1.0 + 0.8 * (r - 1.0); };
        const double st = esz == 2 ? 0.5 : 0.75;
        double least = (double)stages * st * crowd(tiles64) * (best_mi * best_ni > 1 ? 0.95 : 1.0);
        // float32 sums of four stages and more go as products of bfloat16 parts (kernels/gemm_mfma.h) on 128 x 64, 64 x 128 or
        // 128 x 128 tiles, whole or in slices, where that is estimated to take less.  A stage takes 0.92 us on 128 x 64 tiles and 1.45
        // on 128 x 128, a little more where an operand is transposed on the way; a round of workgroups adds a first load and a
        // store that nothing overlaps.  64 x 64 tiles stay with the float32 MFMAs: their stage is bound by the splitting (46 to
        // 56 us / 52 to 57 for a^T b 1024 x 1024 x 2048, 17.1 / 15.7 for a b^T 8192 x 64 x 1024).
        // us, float32 MFMAs on the tiles chosen before / so: a b^T 2048 x 1024 x 1024 38.4 / 31.5 (128 x 64), a b 40.0 / 31.7, a^T b 1024 x
        // 1024 x 2048 50.3 / 36.7 (128 x 128, 4 slices), a b^T 2048^3 126 / 92.5 (128 x 128), 4096^3 966 / 703, 512 x 512 x 8192 a^T b
        // 51 / 35.4, 64 x 512 x 512 x 256 143 / 65.5, 12 x 384 x 384 x 384 35.5 / 17.2.
        const bool parts = in_dtype == MJT_FLOAT32 && stages >= 4;
        for (int t = 0; t < (parts ? 4 : 1); t++) {
            const int mi = t == 1 || t == 3 ? 2 : 1, ni = t >= 2 ? 2 : 1;
            const double tiles = (double)((M + 64 * mi - 1) / (64 * mi)) * ((N + 64 * ni - 1) / (64 * ni)) * batch;
            for (int64_t n = t ? 1 : 2; n == 1 || (sliceable && n <= 16 && n <= stages / 4); n++) {
                const int64_t pn = (stages + n - 1) / n, nn = (stages + pn - 1) / pn;
                const double rounds = std::ceil(tiles * nn / cus);
                double us = t ? (nn > 1 ? 4.0 + (double)nn * M * N * 8 / 4.5e6 : -2.0) : nn > 1 ? 5.0 + (double)nn * M * N * 8 / 3e6 : 0.0;
                if (t == 0) us = (us + (double)pn * st * crowd(tiles * nn)) / 0.9;
                else if (t == 3) us += rounds * ((double)pn * (a_kcont && b_kcont ? 1.45 : 1.55) + 6.5);
                else us += rounds * ((double)pn * (a_kcont && b_kcont ? 0.92 : 1.05) * (rounds > 1 ? 0.9 : 1.0) * (t == 2 ? 1.06 : 1.0) + 3.5);
                if (us < least && (nn == 1 || nn * M * N * 4 <= (int64_t(256) << 20))) {
                    least = us; slices = nn; per = pn; split = t > 0; best_mi = mi; best_ni = ni;
                }
            }
        }
        void* part_mem = slices > 1 ? scratch_if_any((size_t)(slices * M * N * 4)) : nullptr;
        if (!part_mem) slices = 1;
        const int MI = best_mi, NI = best_ni;
        const int in = in_dtype == MJT_BFLOAT16 ? 0 : in_dtype == MJT_FLOAT16 ? 1 : 2;
        const int out = slices > 1 || out_dtype == MJT_FLOAT32 ? 2 : out_dtype == MJT_BFLOAT16 ? 0 : 1;
        const bool one_stage = stages == 1 && !getenv("MJT_GEMM_TWO_BUFFERS");       // a single stage of the kernel's k loop
        const EpilogueCode ep = epilogue_code(1, 12, out_dtype, slices == 1 && ldc == N && (batch == 1 || sc == M * N) ? M * N * batch : -1);
        std::ostringstream key;
        key << "gemm|" << in << out << MI << NI << a_kcont << b_kcont << one_stage << (slices > 1) << split << ep.key;
        JitKernel* k = cached(key.str());
        if (!k) {
            std::ostringstream name;
            name << "mjt_gemm_mfma_" << mjt_dtype_name(in_dtype) << "_" << (out == 2 ? "float32" : mjt_dtype_name(out_dtype)) << "_" << 64 * MI << "x" << 64 * NI
                 << (a_kcont ? "_n" : "_t") << (b_kcont ? "t" : "n") << (one_stage ? "_k1" : "") << (split ? "_parts" : "") << (slices > 1 ? "_slices" : "") << ep.suffix();
            std::ostringstream src;
            src << ep.defs << "#define NBUF " << (one_stage ? 1 : 2) << "\n#define SLICED " << (slices > 1 ? 1 : 0) << "\n#define SPLIT " << (split ? 1 : 0) << "\n";
            src << "#define ENTRY " << name.str() << "\n#define IN " << in << "\n#define OUT " << out << "\n#define MI " << MI
                << "\n#define NI " << NI << "\n#define A_KCONT " << (a_kcont ? 1 : 0) << "\n#define B_KCONT " << (b_kcont ? 1 : 0) << "\n";
            if (split) src << embedded_source("split.h") << "\n";
            src << embedded_source("gemm_mfma.h") << "\n";
            k = jit_get(src.str(), name.str());
            remember(key.str(), k);
        }
        const int64_t tiles = ((M + 64 * MI - 1) / (64 * MI)) * ((N + 64 * NI - 1) / (64 * NI));
        const int64_t grid = (tiles * (slices > 1 ? slices : batch) + 7) / 8 * 8;
        MJT_CHECK(grid < (int64_t(1) << 31), "matmul: launch too large");
        if (slices == 1) {
            args[3] |= (uint64_t)batch << 32;
            args.insert(args.end(), ep.words.begin(), ep.words.end());
            epilogue_taken(ep);
            jit_launch(k, (unsigned)grid, 1, product_threads(split), 0, args);
            return;
        }
        args[2] = bits_of_ptr(part_mem);
        args[9] = (uint64_t)per;
        args[11] = (uint64_t)(M * N);
        SliceFold fold(part_mem, C, out_dtype, M * N, slices);
        {
            Preparing preparing;
            jit_launch(k, (unsigned)grid, 1, product_threads(split), 0, args);
        }
        fold.launch();
        set_last_kernel(k->name.c_str());
        return;
    }
    std::ostringstream key;
    key << "gemmp|" << in_dtype << "|" << out_dtype << a_kcont << b_kcont;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_gemm_plain_" << mjt_dtype_name(in_dtype) << "_" << mjt_dtype_name(out_dtype) << (a_kcont ? "_n" : "_t") << (b_kcont ? "t" : "n");
        std::ostringstream src;
        src << "#define ENTRY " << name.str() << "\n#define TIN " << dtype_cname(in_dtype) << "\n#define TOUT " << dtype_cname(out_dtype)
            << "\n#define TACC " << (in_dtype == MJT_FLOAT64 ? "double" : "float") << "\n#define A_KCONT " << (a_kcont ? 1 : 0)
            << "\n#define B_KCONT " << (b_kcont ? 1 : 0) << "\n";
        src << embedded_source("prelude.h") << "\n" << embedded_source("gemm_plain.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    MJT_CHECK(batch < 65536 && (M + 63) / 64 < 65536, "matmul: launch too large");
    jit_launch(k, (unsigned)((N + 63) / 64), (unsigned)((M + 63) / 64), 256, 0, args, (unsigned)batch);
}

// 1x1 convolution of stride 1 over a batch of planes that need not be 16-byte multiples (kernels/gemm_dma.h with IMG):
// y[image][m][p] = sum over k of A'[m][k] * x[image][k][p], 16-bit operands, an even number of pixels.  a_kcont: A' = A [M][K], else
// A [K][M] (the input gradient takes the weights as they lie).  False: not covered.
bool gemm_pixels(int in_dtype, int out_dtype, const void* A, const void* x, void* y, int64_t M, int64_t K, int64_t P, int64_t images, bool a_kcont) {
    Context& c = ctx();
    const int64_t lda = a_kcont ? K : M, pieces = (P + 7) / 8, N = images * pieces * 8;
    if ((in_dtype != MJT_BFLOAT16 && in_dtype != MJT_FLOAT16) || !(out_dtype == MJT_FLOAT32 || out_dtype == in_dtype) || K % 64 || P % 2 || K < 64 ||
        lda % 8 || (uintptr_t)A % 16 || (uintptr_t)x % 4 || images * K * P * 2 >= (int64_t(1) << 31) || N >= (int64_t(1) << 31) || M * P >= (int64_t(1) << 31) ||
        (a_kcont ? lda * 2 * 256 : lda * 2 * K) >= (int64_t(1) << 31) || getenv("MJT_GEMM_NO_DMA"))
        return false;
    const int64_t cus = c.dry_run || c.prop.multiProcessorCount <= 0 ? 256 : c.prop.multiProcessorCount;
    // 128 x 128 tiles, also where they are few: the alternatives gather x by elements or run image by image (us at 64 images,
    // forward, before / tiles of 128 / of 256: 1024 x 14 x 14 -> 256: 37.9 / 14.1 / 31.2; 256 x 14 x 14 -> 1024: 40.2 / 18.7 / 20.8;
    // 512 x 28 x 28 -> 128: 20.0 / 15.4 / 24.8; 256 x 28 x 28 -> 512: 36.7 / 31.5 / 35.2; 8 images of 1024 x 14 x 14 -> 256: 24.7 / 11.5 /
    // 29.3).  Not for a half-empty tile of output channels where the plain product per image takes the planes (256 x 56 x 56 -> 64:
    // 37.8 / 40.6), nor, in the forward direction, for short sums and a handful of tiles of odd-sized planes, where little is to be
    // had (64 x 14 x 14 -> 64: 9.0 / 6.1; 128 x 28 x 28 -> 128: 10.9 / 9.5) and the convolution kernels stay; an input gradient also
    // saves the transposed copy of the weights (the same two: 11.9 / 5.9, 15.1 / 9.7).
    const int tile = 128;
    const int64_t tm = (M + tile - 1) / tile, tn = (N + tile - 1) / tile;
    if (P % 8 == 0 ? (double)M < 0.7 * (double)(tm * tile) && tm * tn > cus : a_kcont && (K < 256 || tm * tn < 16)) return false;
    // nor, forward on planes that the plain product takes too, for a sum of one stage, or one of less than eight on few tiles (us
    // plain / this: 8 x 64 x 28 x 28 -> 64 3.7 / 6.3, 32 x 64 x 28 x 28 -> 384 10.0 / 12.5; 4 x 128 x 16 x 16 -> 512 4.8 / 6.4, 8 x 256 x 28 x 28
    // -> 256 7.3 / 7.7, but 32 x 256 x 28 x 28 -> 256 12.3 / 11.2 and 8 x 512 x 16 x 16 -> 128 8.7 / 8.3).
    if (P % 8 == 0 && a_kcont && (K < 128 || (K < 512 && tm * tn <= cus / 2))) return false;
    const int in = in_dtype == MJT_BFLOAT16 ? 0 : 1, out = out_dtype == MJT_BFLOAT16 ? 0 : out_dtype == MJT_FLOAT16 ? 1 : 2;
    const int nbuf = tm * tn > cus ? 2 : 4, wpe = nbuf == 2 ? 2 : 1;      // as for the plain product: two workgroups a unit, or a deeper ring
    const int osz = dtype_size(out_dtype), vs = P % 4 == 0 && (uintptr_t)y % (size_t)(4 * osz) == 0 ? 4 : (uintptr_t)y % (size_t)(2 * osz) == 0 ? 2 : 1;
    const EpilogueCode ep = epilogue_code(vs, 12, out_dtype, M * P * images);
    std::ostringstream key;
    key << "gemmpx|" << in << out << a_kcont << tile << nbuf << vs << "|" << P << ep.key;
    JitKernel* k = cached(key.str());
    if (!k) {
        std::ostringstream name;
        name << "mjt_gemm_mfma_" << mjt_dtype_name(in_dtype) << "_" << mjt_dtype_name(out_dtype) << "_" << tile << "x" << tile << (a_kcont ? "_n" : "_t") << "_pixels" << P << (wpe == 2 ? "_direct2" : "_direct") << ep.suffix();
        std::ostringstream src;
        src << ep.defs << "#define VS " << vs << "\n#define ENTRY " << name.str() << "\n#define IN " << in << "\n#define OUT " << out << "\n#define A_KCONT " << (a_kcont ? 1 : 0) << "\n#define B_KCONT 0\n#define IMG " << P
            << "\n#define TILE " << tile << "\n#define NBUF " << nbuf << "\n#define WPE " << wpe << "\n";
        src << embedded_source("gemm_dma.h") << "\n";
        k = jit_get(src.str(), name.str());
        remember(key.str(), k);
    }
    if (k->spilled != 0 || k->agprs < 0 || k->agprs > tile * tile / 256) {                 // (see gemm_launch)
        if (ep.on) check_no_epilogue();
        return false;
    }
    std::vector<uint64_t> args{bits_of_ptr(A), bits_of_ptr(x), bits_of_ptr(y), (uint64_t)M, (uint64_t)N, (uint64_t)K, (uint64_t)lda, (uint64_t)(K * P), (uint64_t)(M * P), 0,
                               (uint64_t)(images * K * P * 2), 0};
    args.insert(args.end(), ep.words.begin(), ep.words.end());
    epilogue_taken(ep);
    jit_launch(k, (unsigned)((tm * tn + 7) / 8 * 8), 1, 256, 0, args);
    return true;
}

// With `share_a` every matrix of the batch is multiplied by the first matrix of a (batch stride 0: the weights of a
// convolution against the column matrices of a chunk of images).
void matmul_impl(const mjt_tensor* a, const mjt_tensor* b, const mjt_tensor* c, int trans_a, int trans_b, bool share_a) {
    require_init();
    MJT_CHECK(a && b && c, "matmul: null tensor");
    // the relay's own checks (cublas_matmul_op.cc:34-52)
    // 2-d operands, or the same leading (batch) extents on all three (cublas_batched_matmul_op.cc:63-85)
    MJT_CHECK(a->ndim >= 2 && a->ndim == b->ndim && a->ndim == c->ndim, "matmul: operands must have the same rank >= 2");
    const int nd = a->ndim;
    int64_t batch = 1;
    for (int i = 0; i < nd - 2; i++) {
        MJT_CHECK(a->shape[i] == b->shape[i] && a->shape[i] == c->shape[i], "matmul: batch extents differ at axis " << i);
        batch *= a->shape[i];
    }
    auto is_float = [](int d) { return d == MJT_FLOAT32 || d == MJT_FLOAT64 || d == MJT_FLOAT16 || d == MJT_BFLOAT16; };
    MJT_CHECK(is_float(a->dtype) && a->dtype == b->dtype, "matmul: type of two inputs should be the same (float)");
    // the result has the inputs' type; float32 is also accepted for 16-bit inputs (the sum before it is narrowed)
    MJT_CHECK(c->dtype == a->dtype || (c->dtype == MJT_FLOAT32 && dtype_size(a->dtype) == 2), "matmul: result dtype");
    int64_t n = a->shape[nd - 2], m = a->shape[nd - 1], m2 = b->shape[nd - 2], k = b->shape[nd - 1];
    if (trans_a) std::swap(n, m);
    if (trans_b) std::swap(m2, k);
    MJT_CHECK(m == m2, "matmul: inner extents " << m << " and " << m2 << " differ");
    MJT_CHECK(c->shape[nd - 2] == n && c->shape[nd - 1] == k,
              "matmul: result shape " << shape_str(c) << " does not end in [" << n << "," << k << "]");
    MJT_CHECK(n < (int64_t(1) << 31) && m < (int64_t(1) << 31) && k < (int64_t(1) << 31) && batch < (int64_t(1) << 31),
              "matmul: extent too large");
    if (batch == 0) return;
    if (n == 0 || k == 0) return;
    Context& ctxt = ctx();
    if (!ctxt.dry_run) MJT_CHECK(a->ptr && b->ptr && c->ptr, "matmul: null data");
    if (m == 0) {                                             // an empty sum
        if (!ctxt.dry_run) launch_fill_pattern(c->ptr, 0, dtype_size(c->dtype), (size_t)batch * n * k);
        return;
    }
    // c[n,k] = a'[n,m] * b'[m,k]: rows n, columns k, sum over m
    const int64_t lda = a->shape[nd - 1], ldb = b->shape[nd - 1];
    // Rows that are no 16-byte multiples, or operands that do not begin at one, are what only the kernel without MFMAs takes as
    // they lie, 0.14 us for every element of the sum however few tiles there are.  They are copied into padded rows first, 6 to 9 us
    // with the launches, where that is less: from a million multiply-adds on with a sum of 96 and more; from four million with one
    // of 40 (one operand copied) or 48 (both); with a shorter one, down to 16, from 33 million or 67 million (us as they lie /
    // copied: bfloat16 a b^T 1000 x 500 x 900 111 / 15.8, a b 300 x 300 x 700 86.5 / 14.2, a b^T 100 x 1000 x 300 38.3 / 11.7;
    // float32 a b^T 130 x 100 x 333 45.3 / 14.7, 4097 x 49 x 513 17.2 / 14.7; on the other side bfloat16 a^T b 1025 x 5 x 1025 5.6 / 10.3,
    // a b^T 4097 x 17 x 65 6.4 / 9.5, a b 1025 x 33 x 1025 9.7 / 10.6; again worth it: a b 4097 x 33 x 513 12.0 / 11.1, with one copy
    // 1001 x 33 x 2000 10.7 / 8.1).
    {
        const int esz = dtype_size(a->dtype);
        const int64_t ra = batch * a->shape[nd - 2], rb = batch * b->shape[nd - 2], epc = 16 / esz;
        const int64_t lap = (lda + epc - 1) / epc * epc, lbp = (ldb + epc - 1) / epc * epc;
        const bool pad_a = lda != lap || (uintptr_t)a->ptr % 16, pad_b = ldb != lbp || (uintptr_t)b->ptr % 16;
        const int64_t most = int64_t(1) << 30, copies = (pad_a ? 1 : 0) + (pad_b ? 1 : 0);
        auto worth = [&](double macs) { return macs >= (double)(1 << (m >= 96 ? 20 : m >= 32 + 8 * copies ? 22 : 24 + copies)) && m >= 16; };
        // Nor in a batch of small matrices, whose many rows share little work: a copied element takes 4e-6 us (16 bits 2.2e-6),
        // every element of the sum gives back 0.09 us for each round of 64 x 64 tiles, of which the launches take 3.5 to 5 us (us as
        // they lie / copied, a b^T: float32 256 x 50 x 50 x 63 11.1 / 18.0, x 111 18.5 / 26.1; 17 x 816 x 48 x 63 10.9 / 13.9, x 131
        // 22.2 / 21.5; 8 x 512 x 512 x 41 12.4 / 14.6; bfloat16 256 x 50 x 50 x 63 9.6 / 13.7, x 131 18.9 / 16.9; 17 x 816 x 48 x 71
        // 11.1 / 12.8, x 97 14.9 / 13.6).
        const int64_t units = ctxt.dry_run || ctxt.prop.multiProcessorCount <= 0 ? 256 : ctxt.prop.multiProcessorCount;
        const double rounds = std::max(1.0, 0.5 + (double)(batch * ((n + 63) / 64) * ((k + 63) / 64)) / (double)(2 * units));
        const double copied = (double)((pad_a ? ra * lap : 0) + (pad_b ? rb * lbp : 0)) * (esz == 2 ? 2.2e-6 : 4e-6);
        const bool pays = batch == 1 || ((m >= 48 || copies == 1) && copied <= 0.09 * (double)m * rounds - (esz == 2 ? 5.0 : 3.5) + (copies == 1 ? 2.5 : 0.0));
        if ((pad_a || pad_b) && a->dtype != MJT_FLOAT64 && !share_a && batch < 65536 && !getenv("MJT_GEMM_PLAIN") && !getenv("MJT_NO_FASTPATH") &&
            worth((double)batch * n * k * m) && pays && (!pad_a || ra * lap * esz <= most) && (!pad_b || rb * lbp * esz <= most)) {
            const void* pa = pad_a ? padded_rows(0, a->ptr, a->dtype, ra, lda, lap) : a->ptr;
            const void* pb = !pad_b ? b->ptr : pa ? padded_rows(1, b->ptr, b->dtype, rb, ldb, lbp) : nullptr;
            const int64_t la = pad_a ? lap : lda, lb = pad_b ? lbp : ldb;
            if (pa && pb) {
                gemm_launch(a->dtype, c->dtype, pa, pb, c->ptr, n, k, m, la, lb, k, a->shape[nd - 2] * la, b->shape[nd - 2] * lb, n * k, batch, !trans_a, trans_b != 0, 0, 0, k % 8 == 0);
                return;
            }
        }
    }
    const int64_t per_launch = 65535;                         // the batch rides on a grid axis
    for (int64_t b0 = 0; b0 < batch; b0 += per_launch) {
        const int64_t nb = batch - b0 < per_launch ? batch - b0 : per_launch;
        const char* pa = (const char*)a->ptr + (share_a ? 0 : b0 * n * m * dtype_size(a->dtype));
        const char* pb = (const char*)b->ptr + b0 * m * k * dtype_size(b->dtype);
        char* pc = (char*)c->ptr + b0 * n * k * dtype_size(c->dtype);
        gemm_launch(a->dtype, c->dtype, pa, pb, pc, n, k, m, lda, ldb, k, share_a ? 0 : n * m, m * k, n * k, nb, !trans_a, trans_b != 0);
    }
}

}  // namespace mjt

extern "C" int mjt_matmul(const mjt_tensor* a, const mjt_tensor* b, const mjt_tensor* c, int trans_a, int trans_b) {
    return mjt::guarded([&] { mjt::matmul_impl(a, b, c, trans_a, trans_b, false); });
}

namespace mjt {
bool matmul_available() { return true; }
}  // namespace mjt

extern "C" int mjt_matmul_available(void) { return 1; }
