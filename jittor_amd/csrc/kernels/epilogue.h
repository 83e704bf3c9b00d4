// The element-wise group behind a product, pasted into the kernel that computes it: where the kernel would store adjacent values
// of the result it runs the group on them (the reference's fuser keeps such ops in the product's own loop nest,
// python/jittor/src/executor.cc:555), so that bias, relu or a residual sum cost no pass over memory of their own.
//
// Supplied by the host (as for kernels/fused.h): MJT_EPI_VEC, MJT_EPI_INDEX, the fragments MJT_EPI_SCALARS .. MJT_EPI_STORES, EPI_WORDS
// parameter words behind the kernel's own, MJT_EPI_PRODUCT (the product's name in the fragments), MJT_EPI_TYPE (its dtype: the value is
// rounded to it first, as the plain kernel stores it).
//
// What it saves is the group's read of the product and a launch; what else the group reads and writes stays, which the product kernel's
// waves overlap with their MFMAs.  us, product + group / together, 64 images bfloat16: 1024 x 14 x 14 -> 256 1x1 with relu 15.7 + 5.6 / 17.1,
// 256 x 14 x 14 3x3 with relu 24.5 + 5.6 / 27.9, 256 x 14 x 14 -> 1024 1x1 with a sum, relu and that relu's gradient 18.4 + 21.5 / 30.7, its
// input gradient with a mask 14.3 + 5.3 / 15.6, the other 1x1's with a sum 18.6 + 11.7 / 20.7; float32 32 x 3 x 224 x 224 7x7 -> 64 with relu
// 66.4 + 32.6 / 72.5, 2048 x 1024 x 1024 with a bias 31.4 + 4.8 / 32.6.
//
// Two steps, so that a kernel can ask for what the group reads of many places before it finishes the first.
#define EPI 1

template <int V> struct mjt_epi_in {
    static_assert(V % MJT_EPI_VEC == 0, "whole vectors");
    struct part { MJT_EPI_DECL } part[V / MJT_EPI_VEC];
};

// What the group reads for V adjacent elements from number `at` of the result on.
template <int V, class P> __device__ __forceinline__ void mjt_epi_load(const P& p, mjt_epi_in<V>& in, MJT_EPI_INDEX at) {
#pragma unroll
    for (int q_ = 0; q_ < V / MJT_EPI_VEC; q_++) {
        const MJT_EPI_INDEX e = at + q_ * MJT_EPI_VEC;
        auto& t = in.part[q_];
        (void)e;
        (void)t;
        MJT_EPI_DECODE
        MJT_EPI_LOADS
    }
}

// The group on the product's values there, and its stores.
template <int V, class P> __device__ __forceinline__ void mjt_epi_finish(const P& p, const mjt_epi_in<V>& in, MJT_EPI_INDEX at, const float (&product)[V]) {
    MJT_EPI_SCALARS
#pragma unroll
    for (int q_ = 0; q_ < V / MJT_EPI_VEC; q_++) {
        const MJT_EPI_INDEX e = at + q_ * MJT_EPI_VEC;
        const auto& t = in.part[q_];
        (void)t;
        MJT_EPI_OUTS
#pragma unroll
        for (int k = 0; k < MJT_EPI_VEC; k++) {
            const MJT_EPI_TYPE MJT_EPI_PRODUCT = (MJT_EPI_TYPE)product[q_ * MJT_EPI_VEC + k];
            MJT_EPI_BODY
        }
        MJT_EPI_STORES
    }
}
