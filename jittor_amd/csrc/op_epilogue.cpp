// Products and scatters with an element-wise group behind them: mjt_conv2d_meta_then, mjt_conv2d_meta_dgrad_then, mjt_matmul_then,
// mjt_fused_reindex_reduce_then.
#include "common.h"

namespace mjt {

void conv_impl(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p, int64_t G, bool free_extent, int pack_mode,
               void* packed);
void conv_dgrad_impl(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p);
void matmul_impl(const mjt_tensor* a, const mjt_tensor* b, const mjt_tensor* c, int trans_a, int trans_b, bool share_a);
void fused_reindex_reduce_impl(const mjt_fused_desc* d, const mjt_tensor* x, int op, int n_idx, const char* const* idx, int n_ofc,
                               const char* const* ofc, int n_ex, const mjt_tensor* ex);

namespace {

struct Waiting {
    const mjt_fused_desc* d;
    std::vector<int> inputs;
    std::vector<FusedCode::Dim> dims;
    int64_t total;
    int dtype;
    bool taken = false, refused = false;
};
thread_local Waiting* t_waiting = nullptr;
thread_local int t_preparing = 0;

// Runs `product` on a result tensor of y's shape with the group waiting for it.
template <class F> void then(const mjt_tensor* y, const mjt_fused_desc* d, F&& product) {
    require_init();
    MJT_CHECK(y && d, "product and group: null descriptor");
    Waiting w;
    w.d = d;
    w.total = fused_validate(d, &w.inputs, true, MJT_VAR_PRODUCT);
    int var = -1, out = -1;
    for (int i = 0; i < d->n_vars; i++) {
        if (d->vars[i].role == MJT_VAR_PRODUCT) {
            MJT_CHECK(var < 0, "product and group: more than one product var");
            var = i;
        }
        if (d->vars[i].role == MJT_VAR_OUTPUT && out < 0) out = i;
    }
    MJT_CHECK(var >= 0 && out >= 0, "product and group: the group needs a product var and an output var");
    MJT_CHECK(d->vars[var].dtype == y->dtype, "product and group: the product var must have the result's dtype");
    MJT_CHECK(d->vars[var].bcast_mask == 0, "product and group: the product var has the group's shape");
    MJT_CHECK(y->ndim >= 0 && y->ndim <= MJT_MAX_DIM && numel(y) == w.total, "product and group: the group's shape must be the result's");
    if (w.total == 0) return;
    w.dims = fused_dims(d, w.inputs);
    w.dtype = y->dtype;
    mjt_tensor result = *y;
    result.ptr = d->vars[out].ptr;         // (looked at for its alignment only: nothing but the group's stores is launched)
    struct Scope {
        Scope(Waiting* w) { t_waiting = w; }
        ~Scope() { t_waiting = nullptr; }
    } scope(&w);
    try {
        product(&result);
    } catch (const Error&) {
        if (!w.refused) throw;             // (a refused launch may come back as another failure, from an entry point inside)
    }
    if (!w.taken) MJT_FAIL(MJT_ERR_UNSUPPORTED, "product and group: this product's route takes no group");
}

}  // namespace

EpilogueCode epilogue_code(int vec, int first, int dtype, int64_t covered) {
    EpilogueCode e;
    Waiting* w = t_waiting;
    if (!w || w->taken || t_preparing || dtype != w->dtype || covered != w->total) return e;
    if (dtype != MJT_FLOAT32 && dtype != MJT_BFLOAT16 && dtype != MJT_FLOAT16) return e;          // (handed over as float32)
    while (vec > 1 && !fused_aligned(w->d, w->inputs, w->dims, vec)) vec /= 2;
    if (!fused_aligned(w->d, w->inputs, w->dims, vec)) return e;
    const FusedCode code(w->d, w->inputs, w->dims, vec, w->total >= (int64_t(1) << 31), first);
    std::ostringstream defs;
    defs << embedded_source("prelude.h") << "\n" << code.text("MJT_EPI", "mjt_load", "mjt_store") << "#define EPI_WORDS " << code.words.size() << "\n";
    for (int i = 0; i < w->d->n_vars; i++)
        if (w->d->vars[i].role == MJT_VAR_PRODUCT) defs << "#define MJT_EPI_PRODUCT v" << i << "\n#define MJT_EPI_TYPE " << dtype_cname(dtype) << "\n";
    defs << embedded_source("epilogue.h") << "\n";
    e.on = true;
    e.ops = w->d->n_ops;
    e.key = "|then|" + code.key();
    e.defs = defs.str();
    e.words = code.words;
    return e;
}

void epilogue_taken(const EpilogueCode& code) {
    if (code.on && t_waiting) t_waiting->taken = true;
}

bool epilogue_waits() { return t_waiting && !t_waiting->taken && !t_preparing; }

void check_no_epilogue() {
    if (!epilogue_waits()) return;
    t_waiting->refused = true;
    MJT_FAIL(MJT_ERR_UNSUPPORTED, "product and group: this product's route takes no group");
}

Preparing::Preparing() { t_preparing++; }
Preparing::~Preparing() { t_preparing--; }

}  // namespace mjt

extern "C" int mjt_conv2d_meta_then(const mjt_tensor* x, const mjt_tensor* w, const mjt_tensor* y, const mjt_conv_params* p, int groups,
                                    const mjt_fused_desc* desc) {
    return mjt::guarded([&] { mjt::then(y, desc, [&](const mjt_tensor* r) { mjt::conv_impl(x, w, r, p, groups, false, 0, nullptr); }); });
}
extern "C" int mjt_conv2d_meta_dgrad_then(const mjt_tensor* dy, const mjt_tensor* w, const mjt_tensor* dx, const mjt_conv_params* p,
                                          const mjt_fused_desc* desc) {
    return mjt::guarded([&] { mjt::then(dx, desc, [&](const mjt_tensor* r) { mjt::conv_dgrad_impl(dy, w, r, p); }); });
}
extern "C" int mjt_fused_reindex_reduce_then(const mjt_fused_desc* desc, const mjt_tensor* x, int op, int n_indexes, const char* const* indexes,
                                             int n_overflow_conditions, const char* const* overflow_conditions, int n_extras, const mjt_tensor* extras,
                                             const mjt_fused_desc* behind) {
    return mjt::guarded([&] {
        mjt::then(x, behind, [&](const mjt_tensor* r) {
            mjt::fused_reindex_reduce_impl(desc, r, op, n_indexes, indexes, n_overflow_conditions, overflow_conditions, n_extras, extras);
        });
    });
}
extern "C" int mjt_matmul_then(const mjt_tensor* a, const mjt_tensor* b, const mjt_tensor* c, int trans_a, int trans_b, const mjt_fused_desc* desc) {
    return mjt::guarded([&] { mjt::then(c, desc, [&](const mjt_tensor* r) { mjt::matmul_impl(a, b, r, trans_a, trans_b, false); }); });
}
