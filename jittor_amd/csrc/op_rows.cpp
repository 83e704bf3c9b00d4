// mjt_fused_rows: fused groups and the row reductions between them as one kernel over the rows (kernels/rows.h).
// The reference's executor lets element, broadcast and reduce ops share a group (python/jittor/src/executor.cc:555,
// fused_op.cc:41-118); the ops' formulas are those of mjt_fused_elementwise and mjt_reduce.
#include "common.h"
#include <algorithm>
#include <mutex>
#include <unordered_map>

namespace mjt {

namespace {

struct Built {
    JitKernel* rows = nullptr;
    JitKernel* fold = nullptr;
};
std::mutex g_mu;
std::unordered_map<std::string, Built> g_kernels;
void* g_part = nullptr;               // the workgroups' column sums (guarded by the library's lock, as the scratch memory)
size_t g_part_bytes = 0;
void forget() {   // the kernels belong to the run-time compiler's cache, which mjt_shutdown empties
    std::lock_guard<std::mutex> lock(g_mu);
    g_kernels.clear();
    if (g_part && !ctx().dry_run) (void)hipFree(g_part);
    g_part = nullptr;
    g_part_bytes = 0;
}
const bool g_registered = (at_shutdown(&forget), true);

std::string vname(int i) { return "v" + std::to_string(i); }

enum Space { FULL = MJT_SPACE_FULL, ROW = MJT_SPACE_ROW, COLUMN = MJT_SPACE_COLUMN, SINGLE = 3 };

bool summed_in_float(int dtype) { return dtype == MJT_FLOAT32 || dtype == MJT_FLOAT16 || dtype == MJT_BFLOAT16; }

}  // namespace

static void rows_impl(const mjt_fused_desc* d, int n_row_axes) {
    require_init();
    MJT_CHECK(d && d->vars && d->ops, "rows: null descriptor");
    MJT_CHECK(d->ndim >= 2 && d->ndim <= MJT_MAX_DIM && n_row_axes >= 1 && n_row_axes < d->ndim, "rows: rank " << d->ndim << ", " << n_row_axes << " row axes");
    const int nv = d->n_vars, nops = d->n_ops, first = d->ndim - n_row_axes;
    MJT_CHECK(nv > 0 && nops > 0, "rows: empty group");
    if (nv > 256 || nops > 256) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: group too large");
    int64_t rows = 1, cols = 1;
    for (int a = 0; a < d->ndim; a++) {
        MJT_CHECK(d->shape[a] >= 0, "rows: negative extent");
        (a < first ? rows : cols) *= d->shape[a];
    }
    if (rows == 0 || cols == 0 || cols > 16384 || rows >= (int64_t(1) << 31)) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: " << rows << " x " << cols << " is not covered");

    // ---- where every var lives; how many reductions lie in front of it -----------------------
    std::vector<int> space(nv, -1), level(nv, 0), maker(nv, -1);
    auto mask_space = [&](uint32_t mask) {
        bool lead = true, no_lead = true, tail = true, no_tail = true;
        for (int a = 0; a < d->ndim; a++) {
            if (d->shape[a] == 1) continue;
            const bool b = mask >> a & 1;
            (a < first ? (b ? no_lead : lead) : (b ? no_tail : tail)) = false;
        }
        // (lead: every leading axis of extent > 1 is in the mask; no_lead: none is)
        if (no_lead && no_tail) return (int)FULL;
        if (no_lead && tail) return (int)ROW;
        if (lead && no_tail) return (int)COLUMN;
        return lead && tail ? (int)SINGLE : -1;
    };
    int maxsize = 1;
    for (int i = 0; i < nv; i++) {
        const mjt_fused_var& v = d->vars[i];
        dtype_size(v.dtype);
        MJT_CHECK(v.role >= MJT_VAR_INPUT && v.role <= MJT_VAR_SCALAR, "rows: var " << i << " has role " << v.role);
        if (v.role == MJT_VAR_INPUT) {
            MJT_CHECK(v.ptr, "rows: input var " << i << " has no data");
            MJT_CHECK((v.bcast_mask >> d->ndim) == 0, "rows: bcast_mask of var " << i << " exceeds the rank");
            space[i] = mask_space(v.bcast_mask);
            if (space[i] < 0) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: var " << i << " is broadcast along part of the rows or columns");
        } else if (v.role == MJT_VAR_SCALAR)
            space[i] = SINGLE;
        if (v.role == MJT_VAR_OUTPUT) MJT_CHECK(v.ptr, "rows: output var " << i << " has no data");
    }
    int levels = 0, n_sums = 0;
    std::vector<int> sums;
    for (int k = 0; k < nops; k++) {
        const mjt_fused_op& o = d->ops[k];
        const bool reduces = o.kind == MJT_FOP_ROW_REDUCE || o.kind == MJT_FOP_COLUMN_SUM;
        MJT_CHECK(o.kind >= MJT_FOP_UNARY && o.kind <= MJT_FOP_COLUMN_SUM, "rows: op " << k << " has kind " << o.kind);
        const int nin = o.kind == MJT_FOP_BINARY ? 2 : o.kind == MJT_FOP_TERNARY ? 3 : 1;
        int from = SINGLE, lv = 0;
        for (int j = 0; j < nin; j++) {
            MJT_CHECK(o.in[j] >= 0 && o.in[j] < nv && space[o.in[j]] >= 0, "rows: op " << k << " reads var " << o.in[j] << " before it is produced");
            const int s = space[o.in[j]];
            MJT_CHECK(maker[o.in[j]] < 0 || d->ops[maker[o.in[j]]].kind != MJT_FOP_COLUMN_SUM, "rows: op " << k << " reads a column sum");
            from = from == SINGLE ? s : s == SINGLE || s == from ? from : (int)FULL;
            lv = std::max(lv, level[o.in[j]]);
        }
        MJT_CHECK(o.out >= 0 && o.out < nv && space[o.out] < 0, "rows: op " << k << " output");
        const mjt_fused_var& ov = d->vars[o.out];
        MJT_CHECK(ov.role == MJT_VAR_INTERMEDIATE || ov.role == MJT_VAR_OUTPUT, "rows: op " << k << " writes var " << o.out);
        if (o.kind == MJT_FOP_UNARY) MJT_CHECK(o.op >= MJT_OP_ABS && o.op <= MJT_OP_SIGMOID, "rows: op " << k << ": not a unary op");
        if (o.kind == MJT_FOP_BINARY) MJT_CHECK(o.op >= MJT_OP_POW && o.op <= MJT_OP_MEAN, "rows: op " << k << ": not a binary op");
        const int declared = (int)(ov.reserved & 3);
        if (reduces) {
            const bool row = o.kind == MJT_FOP_ROW_REDUCE;
            if (!summed_in_float(ov.dtype) || !summed_in_float(d->vars[o.in[0]].dtype) || space[o.in[0]] != FULL ||
                !(o.op == MJT_OP_ADD || (row && (o.op == MJT_OP_MEAN || o.op == MJT_OP_MAXIMUM || o.op == MJT_OP_MINIMUM))))
                MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: reduction " << k << " is not covered");
            MJT_CHECK(declared == (row ? ROW : COLUMN) && (row || ov.role == MJT_VAR_OUTPUT), "rows: reduction " << k << " writes var " << o.out);
            space[o.out] = declared;
            level[o.out] = lv + 1;
            if (row) levels = std::max(levels, lv + 1);
            else { sums.push_back(k); n_sums++; }
        } else {
            // an op works where it is declared: on every element, or once per row
            MJT_CHECK(declared == FULL || (declared == ROW && (from == ROW || from == SINGLE)), "rows: op " << k << " has inputs that do not fit its result");
            space[o.out] = declared;
            level[o.out] = lv;
        }
        maker[o.out] = k;
    }
    for (int i = 0; i < nv; i++) MJT_CHECK(space[i] >= 0, "rows: var " << i << " is never produced");
    if (levels == 0 || n_sums > 8) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: " << levels << " rounds of row reductions, " << n_sums << " column sums");
    int n_full = 0, n_cols = 0;
    for (int i = 0; i < nv; i++) {
        const mjt_fused_var& v = d->vars[i];
        if (v.role == MJT_VAR_INPUT) (space[i] == FULL ? n_full : n_cols) += space[i] == FULL || space[i] == COLUMN;
        if ((v.role == MJT_VAR_INPUT || v.role == MJT_VAR_OUTPUT) && (space[i] == FULL || (v.role == MJT_VAR_INPUT && space[i] == COLUMN))) maxsize = std::max(maxsize, dtype_size(v.dtype));
    }

    // ---- vectors, lanes of a row, rows of a workgroup ------------------------------------------
    int vec = std::min(8, 16 / maxsize);
    auto aligned = [&](int w) {
        if (cols % w) return false;
        for (int i = 0; i < nv; i++) {
            const mjt_fused_var& v = d->vars[i];
            if (v.role == MJT_VAR_INTERMEDIATE || v.role == MJT_VAR_SCALAR || !(space[i] == FULL || (space[i] == COLUMN && v.role == MJT_VAR_INPUT))) continue;
            if ((uintptr_t)v.ptr % (size_t)(w * dtype_size(v.dtype))) return false;
        }
        return true;
    };
    while (vec > 1 && !aligned(vec)) vec /= 2;
    const int64_t packs = (cols + vec - 1) / vec;
    // about eight elements a lane: few enough for the registers of several inputs, enough that a row's reductions cost
    // little beside its elements (see kernels/rows.h)
    const int want = std::max(1, 8 / vec);
    int64_t g = 1;
    while (g < 1024 && g * want < packs) g *= 2;
    const int nvp = (int)((packs + g - 1) / g);
    if (nvp * vec > 16) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: rows of " << cols << " elements in vectors of " << vec);
    if ((n_full + n_cols + n_sums) * nvp * vec > 160) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: " << n_full + n_cols << " inputs of " << nvp * vec << " elements a lane");
    const int block = g > 256 ? (int)g : 256;
    const int64_t rpb = block / g, passes = (rows + rpb - 1) / rpb;
    int64_t blocks = std::min(passes, int64_t(1) << 20);       // (they walk over the rest: a launch is less than 2^32 lanes)
    if (n_sums) {
        // the partial sums are written and read once more, so a workgroup takes four rows at least; and one for every compute unit at
        // least, four of 256 lanes at most (4096 x 2048 float32, rows a workgroup 16 / 8 / 4: 48 / 34 / 30.5)
        const int64_t cus = ctx().dry_run || ctx().prop.multiProcessorCount <= 0 ? 256 : ctx().prop.multiProcessorCount;
        blocks = std::min(passes, std::max(cus, std::min((1024 / block) * cus, rows / 4)));
    }
    // a workgroup counts rows in 32 bits, up to one step past the last
    if (rows + blocks * rpb >= int64_t(1) << 31) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: " << rows << " rows are not covered");
    const bool streams = rows * cols * maxsize >= (int64_t(32) << 20);

    // ---- parameters -----------------------------------------------------------------------------
    const size_t part_bytes = (size_t)blocks * n_sums * cols * 4;
    if (n_sums && !(workspace_allowed(part_bytes) && (ctx().dry_run || grow_kept(&g_part, &g_part_bytes, part_bytes)))) MJT_FAIL(MJT_ERR_UNSUPPORTED, "rows: no memory for partial sums");
    void* const part = ctx().dry_run ? (void*)(uintptr_t)0x1000 : g_part;
    std::vector<uint64_t> args{(uint64_t)rows, (uint64_t)cols, bits_of(1.0 / (double)cols), n_sums ? bits_of_ptr(part) : 0};
    std::vector<int> at(nv, -1);
    for (int i = 0; i < nv; i++) {
        const mjt_fused_var& v = d->vars[i];
        if (v.role == MJT_VAR_INTERMEDIATE || (v.role == MJT_VAR_OUTPUT && space[i] == COLUMN)) continue;
        at[i] = (int)args.size();
        if (v.role == MJT_VAR_SCALAR) args.push_back(dtype_is_float(v.dtype) ? bits_of(v.fvalue) : (uint64_t)v.ivalue);
        else args.push_back(bits_of_ptr(v.ptr));
    }
    std::ostringstream key;
    key << vec << "|" << g << "|" << nvp << "|" << (packs < g * nvp) << streams << "|";
    for (int i = 0; i < nv; i++) key << d->vars[i].role << ":" << d->vars[i].dtype << ":" << space[i] << ":" << (d->vars[i].reserved & MJT_ROUNDED) << ";";
    for (int k = 0; k < nops; k++) {
        const mjt_fused_op& o = d->ops[k];
        key << o.kind << ":" << o.op << ":" << o.in[0] << ":" << (o.kind == MJT_FOP_BINARY || o.kind == MJT_FOP_TERNARY ? o.in[1] : -1) << ":" << (o.kind == MJT_FOP_TERNARY ? o.in[2] : -1) << ">" << o.out << ";";
    }
    Built built;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = g_kernels.find(key.str());
        if (it != g_kernels.end()) built = it->second;
    }
    if (!built.rows) {
        // ---- the kernel's text ------------------------------------------------------------------
        std::ostringstream scal, colp, loads, body, sumdef;
        auto type = [&](int i) { return std::string(dtype_cname(d->vars[i].dtype)); };
        // (only a lane's last pack can lie past the row's end; it is then the row's last one again, read but neither summed nor stored:
        // no branch in front of a load or of arithmetic)
        const bool tail = packs < g * nvp;
        const std::string valid = tail ? "if (t < NV - 1 || inside) " : "", keep = tail ? "t < NV - 1 || inside ? " : "";
        const std::string col = tail ? "(t < NV - 1 ? (t * G + lane) * VEC : last)" : "(t * G + lane) * VEC";
        const bool late = nvp * vec > 8 && vec > 1;                       // a value per column is loaded where it is used, not held from row to row
        for (int i = 0; i < nv; i++) {
            const mjt_fused_var& v = d->vars[i];
            const std::string T = type(i), P = "p.a[" + std::to_string(at[i]) + "]", I = std::to_string(i);
            if (v.role == MJT_VAR_SCALAR) {
                scal << "const " << T << " " << vname(i) << " = (" << T << ")" << (dtype_is_float(v.dtype) ? "__longlong_as_double((long long)(unsigned long long)" + P + ")" : "(long long)(unsigned long long)" + P) << "; ";
            } else if (v.role == MJT_VAR_INPUT && space[i] == SINGLE) {
                scal << "const " << T << " " << vname(i) << " = *(const " << T << "*)" << P << "; ";
            } else if (v.role == MJT_VAR_INPUT && space[i] == COLUMN) {
                if (!late) colp << "mjt_pack<" << T << ", VEC> in" << I << "[NV]; _Pragma(\"unroll\") for (int t = 0; t < NV; t++) mjt_load(in" << I << "[t], (const " << T << "*)" << P << " + " << col << "); ";
            } else if (v.role == MJT_VAR_INPUT && space[i] == FULL) {
                loads << "mjt_pack<" << T << ", VEC> in" << I << "[NV]; _Pragma(\"unroll\") for (int t = 0; t < NV; t++) mjt_load(in" << I << "[t], (const " << T << "*)" << P << " + base + " << col << "); ";
            } else if (v.role == MJT_VAR_INPUT) {
                loads << "const " << T << " " << vname(i) << " = ((const " << T << "*)" << P << ")[row]; ";
            }
        }
        // the value of one op: `const auto vI`, or its declared type where the value is stored or would have been
        auto statement = [&](int k) {
            const mjt_fused_op& o = d->ops[k];
            const mjt_fused_var& ov = d->vars[o.out];
            const std::string e = fused_op_expr(d, o);
            if (ov.role == MJT_VAR_OUTPUT || (ov.reserved & MJT_ROUNDED)) return "const " + type(o.out) + " " + vname(o.out) + " = (" + type(o.out) + ")(" + e + "); ";
            return "const auto " + vname(o.out) + " = " + e + "; ";
        };
        // the element ops behind `wanted`, in order, with the elements of the inputs that they read
        std::string pack_loads;                                // what the last element_code wants loaded per pack
        auto element_code = [&](const std::vector<int>& wanted) {
            pack_loads.clear();
            std::vector<char> need(nv, 0);
            for (int v : wanted) need[v] = 1;
            std::vector<int> run;
            for (int k = nops - 1; k >= 0; k--) {
                const mjt_fused_op& o = d->ops[k];
                if (!need[o.out] || space[o.out] != FULL || o.kind > MJT_FOP_BROADCAST) continue;
                run.push_back(k);
                for (int j = 0; j < (o.kind == MJT_FOP_BINARY ? 2 : o.kind == MJT_FOP_TERNARY ? 3 : 1); j++) need[o.in[j]] = 1;
            }
            std::string s;
            for (int i = 0; i < nv; i++)
                if (need[i] && d->vars[i].role == MJT_VAR_INPUT && space[i] == COLUMN && late)
                    pack_loads += "mjt_pack<" + type(i) + ", VEC> in" + std::to_string(i) + "[NV]; mjt_load(in" + std::to_string(i) + "[t], (const " + type(i) + "*)p.a[" + std::to_string(at[i]) + "] + " + col + "); ";
            for (int i = 0; i < nv; i++)
                if (need[i] && d->vars[i].role == MJT_VAR_INPUT && (space[i] == FULL || space[i] == COLUMN)) s += "const " + type(i) + " " + vname(i) + " = in" + std::to_string(i) + "[t].v[k]; ";
            for (size_t q = run.size(); q-- > 0;) s += statement(run[q]);
            return s;
        };
        auto row_ops = [&](int lv) {
            for (int k = 0; k < nops; k++) {
                const mjt_fused_op& o = d->ops[k];
                if (o.kind > MJT_FOP_BROADCAST || space[o.out] != ROW || level[o.out] != lv) continue;
                body << statement(k);
                if (d->vars[o.out].role == MJT_VAR_OUTPUT) body << "if (mine && lane == 0) ((" << type(o.out) << "*)p.a[" << at[o.out] << "])[row] = " << vname(o.out) << "; ";
            }
        };
        row_ops(0);
        int most = 1;
        for (int lv = 0; lv < levels; lv++) {
            std::vector<int> reds, ins;
            for (int k = 0; k < nops; k++)
                if (d->ops[k].kind == MJT_FOP_ROW_REDUCE && level[d->ops[k].out] == lv + 1) { reds.push_back(k); ins.push_back(d->ops[k].in[0]); }
            most = std::max(most, (int)reds.size());
            // (up to eight accumulators a lane, then a tree: chains of two roundings)
            for (int k : reds) {
                const std::string I = std::to_string(d->ops[k].out);
                body << "float q" << I << "[ACCS]; _Pragma(\"unroll\") for (int k = 0; k < ACCS; k++) q" << I << "[k] = mjt_init_" << (d->ops[k].op == MJT_OP_MEAN ? "add" : mjt_op_name(d->ops[k].op)) << "<float>(); ";
            }
            const std::string code = element_code(ins);
            body << "_Pragma(\"unroll\") for (int t = 0; t < NV; t++) { " << pack_loads << "_Pragma(\"unroll\") for (int k = 0; k < VEC; k++) { " << code;
            for (int k : reds) {
                const mjt_fused_op& o = d->ops[k];
                const std::string q = "q" + std::to_string(o.out) + "[(t * VEC + k) % ACCS]", no = tail ? " : " + q : "";
                if (o.op == MJT_OP_MEAN) body << q << " = " << keep << q << " + float(" << vname(o.in[0]) << ") * rcount" << no << "; ";
                else body << q << " = " << keep << "mjt_" << mjt_op_name(o.op) << "<float>(" << q << ", " << vname(o.in[0]) << ")" << no << "; ";
            }
            body << "} } ";
            for (int k : reds) {
                const mjt_fused_op& o = d->ops[k];
                const std::string q = "q" + std::to_string(o.out);
                body << "_Pragma(\"unroll\") for (int off = ACCS / 2; off > 0; off /= 2) _Pragma(\"unroll\") for (int k = 0; k < off; k++) " << q << "[k] = mjt_"
                     << (o.op == MJT_OP_MEAN ? "add" : mjt_op_name(o.op)) << "<float>(" << q << "[k], " << q << "[k + off]); float r" << o.out << " = " << q << "[0]; ";
            }
            auto merge = [&](const mjt_fused_op& o, const std::string& b) {
                const std::string r = "r" + std::to_string(o.out);
                return r + " = mjt_" + (o.op == MJT_OP_MEAN ? "add" : mjt_op_name(o.op)) + "<float>(" + r + ", " + b + "); ";
            };
            body << "_Pragma(\"unroll\") for (int off = (G < 64 ? G : 64) / 2; off > 0; off /= 2) { ";
            for (int k : reds) body << merge(d->ops[k], "mjt_rows_xor(r" + std::to_string(d->ops[k].out) + ", off)");
            body << "} ";
            if (g > 64) {
                body << "if ((tid & 63) == 0) { ";
                for (size_t q = 0; q < reds.size(); q++) body << "slots[turn][" << lv << "][" << q << "][tid >> 6] = r" << d->ops[reds[q]].out << "; ";
                body << "} __syncthreads(); ";
                for (size_t q = 0; q < reds.size(); q++) {
                    const mjt_fused_op& o = d->ops[reds[q]];
                    const std::string w = "w" + std::to_string(o.out);
                    body << "float " << w << "[GW]; _Pragma(\"unroll\") for (int i = 0; i < GW; i++) " << w << "[i] = slots[turn][" << lv << "][" << q << "][sub * GW + i]; "
                         << "_Pragma(\"unroll\") for (int off = GW / 2; off > 0; off /= 2) _Pragma(\"unroll\") for (int i = 0; i < off; i++) " << w << "[i] = mjt_"
                         << (o.op == MJT_OP_MEAN ? "add" : mjt_op_name(o.op)) << "<float>(" << w << "[i], " << w << "[i + off]); r" << o.out << " = " << w << "[0]; ";
                }
            }
            for (int k : reds) {
                const int o = d->ops[k].out;
                body << "const " << type(o) << " " << vname(o) << " = (" << type(o) << ")r" << o << "; ";
                if (d->vars[o].role == MJT_VAR_OUTPUT) body << "if (mine && lane == 0) ((" << type(o) << "*)p.a[" << at[o] << "])[row] = " << vname(o) << "; ";
            }
            row_ops(lv + 1);
        }
        std::vector<int> wanted, outs;
        for (int i = 0; i < nv; i++)
            if (d->vars[i].role == MJT_VAR_OUTPUT && space[i] == FULL) { wanted.push_back(i); outs.push_back(i); }
        for (int k : sums) wanted.push_back(d->ops[k].in[0]);
        const std::string code = element_code(wanted);
        body << "_Pragma(\"unroll\") for (int t = 0; t < NV; t++) { " << pack_loads;
        for (int i : outs) body << "mjt_pack<" << type(i) << ", VEC> out" << i << "; ";
        body << "_Pragma(\"unroll\") for (int k = 0; k < VEC; k++) { " << code;
        for (int i : outs) body << "out" << i << ".v[k] = " << vname(i) << "; ";
        for (size_t j = 0; j < sums.size(); j++) body << "sums[" << j << "][t][k] += mine" << (tail ? " && (t < NV - 1 || inside)" : "") << " ? float(" << vname(d->ops[sums[j]].in[0]) << ") : 0.0f; ";
        body << "} if (mine) " << valid << "{ ";
        for (int i : outs) body << "MJT_ST((" << type(i) << "*)p.a[" << at[i] << "] + base + (t * G + lane) * VEC, out" << i << "); ";
        body << "} } ";
        if (n_sums) sumdef << "float sums[NSUMS][NV][VEC] = {}; ";

        int accs = 1;
        while (accs < 8 && accs * 2 <= nvp * vec) accs *= 2;
        std::ostringstream frag;
        frag << "#define NPARAM " << args.size() << "\n#define BLOCK " << block << "\n#define G " << g << "\n#define VEC " << vec << "\n#define NV " << nvp << "\n#define ACCS " << accs << "\n#define LEVELS " << levels
             << "\n#define MOST " << most << "\n#define TAIL " << (packs < g * nvp ? 1 : 0) << "\n#define NSUMS " << n_sums << "\n#define MJT_ST " << (streams ? "mjt_store_nt" : "mjt_store") << "\n";
        frag << "#define MJT_ROWS_SCALARS " << scal.str() << "\n#define MJT_ROWS_COLS " << colp.str() << "\n#define MJT_ROWS_SUMS " << sumdef.str() << "\n#define MJT_ROWS_LOADS " << loads.str()
             << "\n#define MJT_ROWS_BODY " << body.str() << "\n";
        auto named = [](const char* what, int n, const std::string& text) {
            uint64_t h = 1469598103934665603ull;
            for (unsigned char c : text) h = (h ^ c) * 1099511628211ull;
            char name[64];
            snprintf(name, sizeof(name), "mjt_%s_%d_%016llx", what, n, (unsigned long long)h);
            return std::string(name);
        };
        std::string name = named("rows", nops, frag.str());
        built.rows = jit_get("#define ENTRY " + name + "\n" + frag.str() + embedded_source("prelude.h") + "\n" + embedded_source("rows.h") + "\n", name);
        if (n_sums) {
            std::ostringstream f;
            f << "#define FOLD 1\n#define NPARAM " << 3 + n_sums << "\n#define BLOCK 1024\n#define G 64\n#define NSUMS " << n_sums << "\n#define MJT_FOLD_STORE ";
            for (int j = 0; j < n_sums; j++) {
                const std::string T = type(d->ops[sums[j]].out);
                f << "if (j == " << j << ") ((" << T << "*)p.a[" << 3 + j << "])[c] = (" << T << ")all; ";
            }
            f << "\n";
            name = named("rows_fold", n_sums, f.str());
            built.fold = jit_get("#define ENTRY " + name + "\n" + f.str() + embedded_source("prelude.h") + "\n" + embedded_source("rows.h") + "\n", name);
        }
        std::lock_guard<std::mutex> lock(g_mu);
        g_kernels.emplace(key.str(), built);
    }
    MJT_CHECK(blocks < (int64_t(1) << 31), "rows: launch too large");
    jit_launch(built.rows, (unsigned)blocks, 1, (unsigned)block, 0, args);
    if (n_sums) {
        std::vector<uint64_t> fa{(uint64_t)blocks, (uint64_t)cols, bits_of_ptr(part)};
        for (int k : sums) fa.push_back(bits_of_ptr(d->vars[d->ops[k].out].ptr));
        jit_launch(built.fold, (unsigned)((cols + 31) / 32), (unsigned)n_sums, 1024, 0, fa);
        set_last_kernel(built.rows->name.c_str());
    }
}

}  // namespace mjt

extern "C" int mjt_fused_rows(const mjt_fused_desc* desc, int n_row_axes) {
    return mjt::guarded([&] { mjt::rows_impl(desc, n_row_axes); });
}
