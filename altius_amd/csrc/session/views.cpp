// The session's copy avoidance: strided views (Split / Transpose results that only MatMuls read), operand
// descriptions for the GEMM, activations deferred into the next product's operand split, and
// MatMul -> Softmax -> MatMul deferred into the one-kernel attention.  Counterparts in the reference always
// copy: compute_transpose (crates/session_interpreter/src/session.rs:1179-1278), compute_split (1488-1548),
// compute_mat_mul (621-684), compute_softmax (990-1026).
#include <algorithm>
#include <functional>

#include "views.h"

namespace altius {

using namespace detail;

bool HipSession::materialize(DeviceTensor *t, SessionError *err) {
    if (t->strides.empty()) return true;
    DeviceTensor dense;
    if (!allocate(TypedFixedShape{t->dims, t->elem_ty}, &dense, err)) return false;
    std::vector<int64_t> d;
    for (auto x : t->dims.as_vec()) d.push_back((int64_t)x);
    const std::vector<int64_t> os = dense_strides(t->dims);
    const int rc = launch_copy_strided(ctx_, dense.ptr, t->ptr, (int)elem_size(t->elem_ty), (int)d.size(), d.data(), os.data(),
                                       t->strides.data());
    if (rc) return fail_code(err, rc, ctx_.last_error);
    dense.host = t->host;
    *t = std::move(dense);
    return true;
}

bool HipSession::flush_add(DeviceTensor *t, SessionError *err) {
    if (!t->owes_add()) return true;
    PendingAdd &p = *t->pending_add;
    const int64_t n = (int64_t)p.elems, one = 1;
    const int rc = launch_binary(ctx_, AHIP_ADD, static_cast<float *>(t->ptr), p.a, p.b, 1, &n, &one, &one);
    if (rc) return fail_code(err, rc, ctx_.last_error);
    p.done = true;
    p.a_block.reset();
    p.b_block.reset();
    return true;
}

bool HipSession::apply_pending(DeviceTensor *t, SessionError *err) {
    if (!flush_add(t, err)) return false;
    if (t->pending_op < 0) return true;
    if (t->pending_op == PENDING_ATTENTION)  // callers that know the value's id flush it instead (flush_attention)
        return fail(err, SessionError::Message, "internal: a deferred attention product was read by an operator that cannot finish it");
    if (!materialize(t, err)) return false;
    DeviceTensor done;
    if (!allocate(TypedFixedShape{t->dims, t->elem_ty}, &done, err)) return false;
    const int rc = launch_unary(ctx_, t->pending_op, static_cast<float *>(done.ptr), static_cast<const float *>(t->ptr),
                                t->dims.total_elems(), 0.0f, 0.0f);
    if (rc) return fail_code(err, rc, ctx_.last_error);
    *t = std::move(done);
    return true;
}

bool HipSession::describe_operand(DeviceTensor *t, MatOperand *o, SessionError *err) {
    for (int attempt = 0; attempt < 2; attempt++) {
        const size_t r = t->dims.len();
        const std::vector<int64_t> st = strides_of(*t);
        o->rows = t->dims[r - 2], o->cols = t->dims[r - 1];
        const int64_t sr = st[r - 2], sc = st[r - 1];
        bool ok = true;
        if (sc == 1 || o->cols == 1) {
            o->stored_transposed = false;
            o->ld = o->rows == 1 ? o->cols : (size_t)sr;
            ok = o->ld >= o->cols;
        } else if (sr == 1 || o->rows == 1) {
            o->stored_transposed = true;
            o->ld = o->cols == 1 ? o->rows : (size_t)sc;
            ok = o->ld >= o->rows;
        } else {
            ok = false;
        }
        o->batch = 1;
        o->bdims.clear(), o->bstr.clear();
        for (size_t i = 0; i + 2 < r; i++) {
            o->batch *= t->dims[i];
            o->bdims.push_back(t->dims[i]);
            o->bstr.push_back(st[i]);
            ok = ok && st[i] >= 0;
        }
        if (ok) return true;
        if (t->strides.empty()) break;
        if (!materialize(t, err)) return false;
    }
    return fail(err, SessionError::Message, "MatMul: an operand's layout could not be read");
}

namespace {
// Batch strides of an operand over the batch axes bd (extent-1 axes already dropped from both): a dense
// operand counts its matrices in bd's order whatever its own leading shape.
bool operand_batch_strides(const std::vector<size_t> &bd, const std::vector<size_t> &own_dims, const std::vector<int64_t> &own_strides,
                           bool dense, size_t matrix_elems, size_t batch, std::vector<int64_t> *out) {
    out->assign(bd.size(), 0);
    if (batch == 1) return true;
    if (dense) {
        int64_t acc = (int64_t)matrix_elems;
        for (size_t i = bd.size(); i-- > 0;) (*out)[i] = acc, acc *= (int64_t)bd[i];
        return true;
    }
    std::vector<size_t> d;
    std::vector<int64_t> s;
    for (size_t i = 0; i < own_dims.size(); i++)
        if (own_dims[i] != 1) d.push_back(own_dims[i]), s.push_back(own_strides[i]);
    if (d != bd) return false;
    *out = s;
    return true;
}
bool aligned_operand(const void *p, size_t ld, const std::vector<int64_t> &bs) {
    bool ok = (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && ld % 4 == 0;
    for (int64_t s : bs) ok = ok && s % 4 == 0;
    return ok;
}
}  // namespace

bool HipSession::flush_attention(ValueId scores, DeviceTensor *placeholder, SessionError *err) {
    auto it = pending_attn_.find(scores);
    if (it == pending_attn_.end()) return fail(err, SessionError::Message, "internal: no operands kept for a deferred attention product");
    PendingAttention pa = std::move(it->second);
    pending_attn_.erase(it);
    DeviceTensor out;
    if (!allocate(TypedFixedShape{pa.score_dims, TensorElemType::F32}, &out, err)) return false;
    const size_t tq = pa.Q.stored_transposed ? pa.Q.cols : pa.Q.rows, tk = pa.K.stored_transposed ? pa.K.cols : pa.K.rows;
    auto two = [](const std::vector<int64_t> &s, size_t out2[2]) {
        out2[0] = s.size() > 0 ? (size_t)s[0] : 0;
        out2[1] = s.size() > 1 ? (size_t)s[1] : 0;
    };
    const size_t outer = pa.bd.size() > 0 ? pa.bd[0] : 1, inner = pa.bd.size() > 1 ? pa.bd[1] : 1;
    size_t q2[2], k2[2], c2[2] = {inner * tq * tk, pa.bd.size() > 1 ? tq * tk : 0};
    two(pa.Q.bstr, q2), two(pa.K.bstr, k2);
    // Q rows [tq, 64] times the transpose of K rows [tk, 64].
    const int rc = launch_gemm_batch2(ctx_, static_cast<float *>(out.ptr), static_cast<const float *>(pa.q.ptr),
                                      static_cast<const float *>(pa.k.ptr), nullptr, outer, inner, tq, tk, 64, 0, 1, pa.Q.ld, pa.K.ld, tk, q2,
                                      k2, c2, 0, 1, 1.0f, 0.0f);
    if (rc) return fail_code(err, rc, ctx_.last_error);
    *placeholder = std::move(out);
    return true;
}

// The first product of MatMul -> Softmax -> MatMul: if the one-kernel attention can take it (64-wide heads,
// at most two batch axes, aligned operands), leave a placeholder and remember Q and K.
bool HipSession::try_defer_attention(const Node &node, const Op &op, const std::vector<DeviceTensor *> &in,
                                     const std::vector<TypedFixedShape> &shapes, std::vector<DeviceTensor> *outs, SessionError *err) {
    if (in.size() != 2 || !in[0] || !in[1] || in[0]->elem_ty != TensorElemType::F32 || in[1]->elem_ty != TensorElemType::F32) return true;
    if (in[0]->dims.len() < 2 || in[1]->dims.len() < 2 || in[0]->pending_op >= 0 || in[1]->pending_op >= 0) return true;
    PendingAttention pa;
    if (!describe_operand(in[0], &pa.Q, err) || !describe_operand(in[1], &pa.K, err)) return false;
    // Q as stored rows [tq, d]; the logical second operand is K^T, so K must be stored as rows [tk, d].
    const bool q_rows = !((op.trans_a ? 1 : 0) ^ (pa.Q.stored_transposed ? 1 : 0));
    const bool k_rows = ((op.trans_b ? 1 : 0) ^ (pa.K.stored_transposed ? 1 : 0)) != 0;
    if (!q_rows || !k_rows) return true;
    const size_t tq = pa.Q.stored_transposed ? pa.Q.cols : pa.Q.rows, d = pa.Q.stored_transposed ? pa.Q.rows : pa.Q.cols;
    const size_t tk = pa.K.stored_transposed ? pa.K.cols : pa.K.rows, dk = pa.K.stored_transposed ? pa.K.rows : pa.K.cols;
    if (d != 64 || dk != 64 || tk == 0 || tq == 0) return true;
    const FixedDimensions &od = shapes[0].dims;
    size_t batch = 1;
    for (size_t i = 0; i + 2 < od.len(); i++) {
        batch *= od[i];
        if (od[i] != 1) pa.bd.push_back(od[i]);
    }
    if (pa.bd.size() > 2 || pa.Q.batch != batch || pa.K.batch != batch) return true;
    std::vector<int64_t> qs, ks;
    if (!operand_batch_strides(pa.bd, pa.Q.bdims, pa.Q.bstr, in[0]->strides.empty(), tq * d, pa.Q.batch, &qs) ||
        !operand_batch_strides(pa.bd, pa.K.bdims, pa.K.bstr, in[1]->strides.empty(), tk * d, pa.K.batch, &ks))
        return true;
    if (!aligned_operand(in[0]->ptr, pa.Q.ld, qs) || !aligned_operand(in[1]->ptr, pa.K.ld, ks)) return true;
    pa.Q.bstr = qs, pa.K.bstr = ks;  // now per axis of bd
    pa.q = *in[0], pa.k = *in[1];
    pa.score_dims = od;
    pending_attn_[node.outputs[0]] = std::move(pa);
    DeviceTensor o;
    o.dims = od;
    o.elem_ty = TensorElemType::F32;
    o.pending_op = PENDING_ATTENTION;
    copies_avoided_++;
    outs->push_back(std::move(o));
    return true;
}

// The second product: O = Softmax(scale(Q K^T)) V in one kernel, into `out` (dense, or in the layout of the
// Transpose behind this node).
bool HipSession::run_attention_tail(const Op &op, const std::vector<DeviceTensor *> &in, DeviceTensor *out, SessionError *err) {
    const Node &node = model_.graph.nodes[current_node_];
    auto it = pending_attn_.find(node.inputs[0]);
    if (it == pending_attn_.end()) return fail(err, SessionError::Message, "MatMul: deferred attention operands are missing");
    PendingAttention pa = std::move(it->second);
    pending_attn_.erase(it);
    // Which attention this is (for the scale): the head that names this node as its tail.
    const AttentionPlan *plan = nullptr;
    for (const auto &kv : attn_head_)
        if (kv.second.tail == current_node_) plan = &kv.second;
    if (!plan) return fail(err, SessionError::Message, "MatMul: no attention plan for this node");
    if (op.trans_a || in.size() != 2 || !in[1] || in[1]->elem_ty != TensorElemType::F32 || in[1]->dims.len() < 2)
        return fail(err, SessionError::Message, "MatMul: the second product of an attention has an unexpected form");
    const size_t tq = pa.Q.stored_transposed ? pa.Q.cols : pa.Q.rows, tk = pa.K.stored_transposed ? pa.K.cols : pa.K.rows;
    MatOperand V;
    std::vector<int64_t> vs;
    for (int attempt = 0;; attempt++) {
        if (!describe_operand(in[1], &V, err)) return false;
        const bool v_rows = !((op.trans_b ? 1 : 0) ^ (V.stored_transposed ? 1 : 0));
        size_t batch = 1;
        for (size_t x : pa.bd) batch *= x;
        bool ok = v_rows && V.rows == tk && V.cols == 64 && (V.batch == batch || V.batch == 1) &&
                  operand_batch_strides(pa.bd, V.bdims, V.bstr, in[1]->strides.empty(), tk * 64, V.batch, &vs) &&
                  aligned_operand(in[1]->ptr, V.ld, vs);
        if (ok) break;
        if (attempt > 0 || in[1]->strides.empty())
            return fail(err, SessionError::Message, "MatMul: the values of an attention do not fit its keys");
        if (!materialize(in[1], err)) return false;
    }
    // Output strides: dense, or the Transpose's layout behind this node.
    std::vector<int64_t> c_str = dense_strides(out->dims);
    auto pv = matmul_out_perm_.find(current_node_);
    if (pv != matmul_out_perm_.end() && pv->second.size() == out->dims.len()) {
        FixedDimensions td = out->dims;
        for (size_t i = 0; i < td.len(); i++) td[i] = out->dims[(size_t)pv->second[i]];
        const std::vector<int64_t> ts = dense_strides(td);
        std::vector<int64_t> cand = c_str;
        for (size_t i = 0; i < td.len(); i++) cand[(size_t)pv->second[i]] = ts[i];
        bool aligned = true;
        for (size_t i = 0; i + 1 < cand.size(); i++) aligned = aligned && (out->dims[i] == 1 || cand[i] % 4 == 0);
        if (aligned && !is_dense(out->dims, cand)) out->strides = c_str = cand;
    }
    const size_t rank = out->dims.len();
    std::vector<int64_t> os;
    for (size_t i = 0; i + 2 < rank; i++)
        if (out->dims[i] != 1) os.push_back(c_str[i]);
    const size_t ldo = out->dims[rank - 2] > 1 ? (size_t)c_str[rank - 2] : 64;
    auto two = [](const std::vector<int64_t> &s, size_t out2[2]) {
        out2[0] = s.size() > 0 ? (size_t)s[0] : 0;
        out2[1] = s.size() > 1 ? (size_t)s[1] : 0;
    };
    size_t q2[2], k2[2], v2[2], o2[2];
    two(pa.Q.bstr, q2), two(pa.K.bstr, k2), two(vs, v2), two(os, o2);
    const size_t outer = pa.bd.size() > 0 ? pa.bd[0] : 1, inner = pa.bd.size() > 1 ? pa.bd[1] : 1;
    // O as the operand planes of the product behind it: O is [outer, inner, tq, 64] written as [outer, tq, inner * 64]
    // (the Transpose's layout), which that product reads as [outer * tq, inner * 64].
    void *planes_ptr = nullptr;
    auto ap = attn_planes_.find(current_node_);
    if (ap != attn_planes_.end() && pa.bd.size() == 2 && rank == 4 && !out->strides.empty() && ldo == inner * 64 && o2[0] == tq * ldo && o2[1] == 64 &&
        attention_writes_planes(ctx_, outer, inner, tq) && gemm_takes_split(ctx_, outer * tq, ap->second.next_n, inner * 64)) {
        DeviceTensor planes;
        if (!allocate_bytes(gemm_planes_bytes(outer * tq, inner * 64), &planes, err)) return false;
        out->block = planes.block;  // the fp32 block goes back to the pool unused
        out->ptr = planes.ptr;
        out->planes = true;
        out->planes_rows = outer * tq, out->planes_k = inner * 64;
        planes_ptr = planes.ptr;
        copies_avoided_++;  // the operand split of the product behind
    }
    const int rc = launch_attention(ctx_, planes_ptr ? nullptr : static_cast<float *>(out->ptr), static_cast<const float *>(pa.q.ptr),
                                    static_cast<const float *>(pa.k.ptr), static_cast<const float *>(in[1]->ptr), outer, inner, tq, tk, 64,
                                    pa.Q.ld, pa.K.ld, V.ld, ldo, q2, k2, v2, o2, plan->scale_op, plan->scale,
                                    pa.mask.ptr ? static_cast<const float *>(pa.mask.ptr) : nullptr, pa.mask_outer_stride, planes_ptr);
    if (rc) return fail_code(err, rc, ctx_.last_error);
    return true;
}

// A Split or Transpose hands out views when everything downstream of it can read them in place:
// MatMul operands, possibly through reshapes and further transposes.  A MatMul whose only reader is
// a Transpose that keeps the last axis writes its result directly in that Transpose's layout.
HipSession::ViewPlan HipSession::find_views() const {
    const auto users = model_.get_value_users();
    const Graph &g = model_.graph;
    auto is_output = [&](ValueId v) { return std::find(g.outputs.begin(), g.outputs.end(), v) != g.outputs.end(); };
    std::function<bool(ValueId, int)> view_ok = [&](ValueId v, int depth) -> bool {
        if (depth > 8 || is_output(v)) return false;
        auto it = users.find(v);
        if (it == users.end() || it->second.empty()) return false;
        for (NodeId u : it->second) {
            const Node &n = g.nodes[u];
            if (n.op.kind == OpKind::MatMul) {
                if (n.inputs.size() > 2 && n.inputs[2] == v) return false;
            } else if (is_alias_op(n.op.kind) || n.op.kind == OpKind::Transpose) {
                if (n.inputs.empty() || n.inputs[0] != v || n.outputs.empty()) return false;
                for (size_t i = 1; i < n.inputs.size(); i++)
                    if (n.inputs[i] == v) return false;
                if (!view_ok(n.outputs[0], depth + 1)) return false;
            } else {
                return false;
            }
        }
        return true;
    };
    ViewPlan plan;
    for (const NodeExecutionPlan &step : plan_) {
        const NodeId id = step.node_id;
        const Node &n = g.nodes[id];
        if (n.op.kind == OpKind::Split || n.op.kind == OpKind::Transpose) {
            bool all = !n.outputs.empty();
            for (ValueId v : n.outputs) all = all && view_ok(v, 0);
            if (all) plan.lazy.insert(id);
        } else if (n.op.kind == OpKind::MatMul && n.outputs.size() == 1 && !is_output(n.outputs[0])) {
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1) continue;
            const Node &t = g.nodes[*it->second.begin()];
            if (t.op.kind != OpKind::Transpose || t.inputs.size() != 1) continue;
            const auto &perm = t.op.perm;
            if (perm.size() < 3 || perm.back() != (int64_t)perm.size() - 1) continue;
            plan.out_perm[id] = perm;
        }
    }
    return plan;
}

// The strides in which a result of these dims is dense once it is transposed by perm.
static std::vector<int64_t> strides_ahead_of(const FixedDimensions &dims, const std::vector<int64_t> &perm) {
    FixedDimensions td = dims;
    for (size_t i = 0; i < td.len(); i++) td[i] = dims[(size_t)perm[i]];
    const std::vector<int64_t> ts = dense_strides(td);
    std::vector<int64_t> s(td.len());
    for (size_t i = 0; i < td.len(); i++) s[(size_t)perm[i]] = ts[i];
    return s;
}

// Which products read their weights' planes, from the graph and its inferred shapes alone: with the views that a session may hand out
// (`views`) and without, a product runs the same sums.  By planes the first operand is one tall matrix and the result dense; gemm_takes_planes
// counts the copies that this takes of a view and ahead of a Transpose.
void HipSession::plan_planes(const ViewPlan &views) {
    struct View {
        FixedDimensions dims;
        std::vector<int64_t> strides;
    };
    std::map<ValueId, View> view_of;  // values that are views where views are handed out
    const Graph &g = model_.graph;
    for (const NodeExecutionPlan &step : plan_) {
        const NodeId id = step.node_id;
        const Node &n = g.nodes[id];
        auto it = inferred_.find(id);
        if (it == inferred_.end() || n.inputs.empty() || n.outputs.empty() || it->second.second.size() < n.outputs.size()) continue;
        const Op &op = it->second.first;
        const std::vector<TypedFixedShape> &shapes = it->second.second;
        const FixedDimensions &od = shapes[0].dims;
        auto in = view_of.find(n.inputs[0]);
        auto hand_out = [&](size_t i, const std::vector<int64_t> &strides) {
            if (!is_dense(shapes[i].dims, strides)) view_of[n.outputs[i]] = View{shapes[i].dims, strides};
        };
        if (is_alias_op(op.kind)) {
            std::vector<int64_t> s;
            if (in != view_of.end() && reshape_strides(in->second.dims, in->second.strides, od, &s)) hand_out(0, s);
        } else if (op.kind == OpKind::Transpose && views.lazy.count(id) && op.perm.size() == od.len()) {
            FixedDimensions d = od;
            for (size_t i = 0; i < od.len(); i++) d[(size_t)op.perm[i]] = od[i];
            const std::vector<int64_t> s = in != view_of.end() ? in->second.strides : dense_strides(d);
            std::vector<int64_t> ps(od.len());
            for (size_t i = 0; i < od.len(); i++) ps[i] = s[(size_t)op.perm[i]];
            hand_out(0, ps);
        } else if (op.kind == OpKind::Split && views.lazy.count(id)) {
            const size_t axis = (size_t)(op.axis < 0 ? op.axis + (int64_t)od.len() : op.axis);
            if (axis >= od.len()) continue;
            FixedDimensions d = od;
            d[axis] = 0;
            for (size_t p = 0; p < n.outputs.size(); p++) d[axis] += shapes[p].dims[axis];
            const std::vector<int64_t> s = in != view_of.end() ? in->second.strides : dense_strides(d);
            for (size_t p = 0; p < n.outputs.size(); p++) hand_out(p, s);
        } else if (op.kind == OpKind::MatMul || op.kind == OpKind::Gemm) {
            auto pv = views.out_perm.find(id);
            std::vector<int64_t> ahead;  // of a Transpose behind the product
            if (pv != views.out_perm.end() && pv->second.size() == od.len()) ahead = strides_ahead_of(od, pv->second);
            if (!ahead.empty() && is_dense(od, ahead)) ahead.clear();
            auto w = n.inputs.size() > 1 ? g.inits.find(n.inputs[1]) : g.inits.end();
            if (!op.trans_a && w != g.inits.end() && w->second.elem_ty() == TensorElemType::F32 && w->second.dims().len() == 2 && od.len() >= 2 &&
                std::find(g.inputs.begin(), g.inputs.end(), n.inputs[1]) == g.inputs.end()) {
                const FixedDimensions &wd = w->second.dims();
                size_t matrices = 1;
                for (size_t i = 0; i + 2 < od.len(); i++) matrices *= od[i];
                const bool turned = op.kind == OpKind::MatMul && in != view_of.end() && !rows_at_one_pitch(in->second.dims, in->second.strides);
                if (gemm_takes_planes(ctx_, matrices * od[od.len() - 2], op.trans_b ? wd[0] : wd[1], op.trans_b ? wd[1] : wd[0], matrices, turned, !ahead.empty()))
                    by_planes_.insert(id);
            }
            if (!ahead.empty() && !by_planes_.count(id)) hand_out(0, ahead);
        }
    }
}

void HipSession::plan_views(bool fused_attention) {
    const auto users = model_.get_value_users();
    const auto parents = model_.get_value_parents();
    const Graph &g = model_.graph;
    auto is_output = [&](ValueId v) { return std::find(g.outputs.begin(), g.outputs.end(), v) != g.outputs.end(); };
    // The [k, n] f32 weights of a product, which no input of the graph can stand in for.
    auto weight_matrix = [&](const Node &product) -> const Tensor * {
        auto w = product.inputs.size() > 1 ? g.inits.find(product.inputs[1]) : g.inits.end();
        if (w == g.inits.end() || std::find(g.inputs.begin(), g.inputs.end(), product.inputs[1]) != g.inputs.end()) return nullptr;
        return w->second.dims().len() == 2 && w->second.elem_ty() == TensorElemType::F32 ? &w->second : nullptr;
    };
    // Product or convolution -> activation, or -> Add(residual): done by its own kernel when that is an fp32 one.
    // v: the result as that node reads it.
    auto plan_post = [&](NodeId id, ValueId v, MatMulPost mp) {
        auto it = users.find(v);
        if (it == users.end() || it->second.size() != 1 || is_output(v)) return;
        const NodeId uid = *it->second.begin();
        const Node &u = g.nodes[uid];
        if (const int act = u.inputs.size() == 1 && u.outputs.size() == 1 ? activation_of(u.op, &mp.alpha, &mp.beta) : 0) {
            mp.act = act;
            matmul_post_[id] = mp;
        } else if (u.op.kind == OpKind::Add && u.inputs.size() == 2 && u.outputs.size() == 1 && u.inputs[0] != u.inputs[1]) {
            mp.has_add = true;
            mp.add_node = uid;
            mp.add_input = u.inputs[0] == v ? 0 : 1;
            mp.residual = u.inputs[1 - mp.add_input];
            matmul_post_[id] = mp;
        }
    };
    for (const NodeExecutionPlan &step : plan_) {
        const NodeId id = step.node_id;
        const Node &n = g.nodes[id];
        if ((n.op.kind == OpKind::Gelu || n.op.kind == OpKind::ReLU) && n.outputs.size() == 1 && n.inputs.size() == 1 &&
                   !is_output(n.outputs[0])) {
            // The activation between two products: its only reader is a MatMul's first operand.
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1) continue;
            const Node &mm = g.nodes[*it->second.begin()];
            if (mm.op.kind != OpKind::MatMul || mm.inputs.size() < 2 || mm.inputs[0] != n.outputs[0]) continue;
            bool elsewhere = false;
            for (size_t i = 1; i < mm.inputs.size(); i++) elsewhere = elsewhere || mm.inputs[i] == n.outputs[0];
            if (elsewhere) continue;
            deferred_unary_.insert(id);
            auto par = parents.find(n.inputs[0]);
            if (par == parents.end() || is_output(n.inputs[0])) continue;
            const Node &first = g.nodes[par->second];
            auto fu = users.find(n.inputs[0]);
            const Tensor *w = weight_matrix(mm);
            if (first.op.kind != OpKind::MatMul || first.outputs.size() != 1 || first.op.trans_a || mm.op.trans_a || fu == users.end() || fu->second.size() != 1 ||
                !weight_matrix(first) || !w)
                continue;
            ActPlanesPlan ap;
            ap.next.consumer = *it->second.begin();
            ap.next.next_n = mm.op.trans_b ? w->dims()[0] : w->dims()[1];
            ap.act = n.op.kind == OpKind::Gelu ? AHIP_GELU : AHIP_RELU;
            act_planes_[par->second] = ap;
            planes_consumer_.insert(ap.next.consumer);
            planes_pass_.insert(id);
        } else if (n.op.kind == OpKind::LayerNormalization && n.outputs.size() == 1 && n.inputs.size() == 3 && !is_output(n.outputs[0])) {
            // LayerNormalization read only by a product with a weight matrix: it can write that product's operand planes.
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1) continue;
            const Node &mm = g.nodes[*it->second.begin()];
            if (mm.op.kind != OpKind::MatMul || mm.inputs.size() < 2 || mm.inputs[0] != n.outputs[0] || mm.op.trans_a) continue;
            bool elsewhere = false;
            for (size_t i = 1; i < mm.inputs.size(); i++) elsewhere = elsewhere || mm.inputs[i] == n.outputs[0];
            const Tensor *w = weight_matrix(mm);
            if (elsewhere || !w) continue;
            PlanesPlan pp;
            pp.consumer = *it->second.begin();
            pp.next_n = mm.op.trans_b ? w->dims()[0] : w->dims()[1];
            planes_out_[id] = pp;
            planes_consumer_.insert(pp.consumer);
            // The residual Add in front of it (two tensors of one shape) can leave its sum to this kernel.
            auto par = parents.find(n.inputs[0]);
            if (par != parents.end()) {
                const Node &add = g.nodes[par->second];
                if (add.op.kind == OpKind::Add && add.inputs.size() == 2 && add.outputs.size() == 1 && add.inputs[0] != add.inputs[1])
                    add_into_ln_[par->second] = id;
            }
        } else if (n.op.kind == OpKind::Conv2d && n.outputs.size() == 1 && !is_output(n.outputs[0])) {
            MatMulPost mp;
            ValueId v = n.outputs[0];
            auto it = users.find(v);
            if (it == users.end() || it->second.size() != 1) continue;
            const Node &bn = g.nodes[*it->second.begin()];
            if (bn.op.kind == OpKind::BatchNormalization && !bn.op.training_mode && bn.inputs.size() == 5 && bn.inputs[0] == v && bn.outputs.size() == 1) {
                bool constant = true;  // its four parameters are weights that no input of the graph can stand in for
                for (size_t k = 1; k < 5; k++)
                    constant = constant && bn.inputs[k] != v && g.inits.count(bn.inputs[k]) &&
                               std::find(g.inputs.begin(), g.inputs.end(), bn.inputs[k]) == g.inputs.end();
                if (constant) {
                    mp.has_norm = true;
                    mp.norm = *it->second.begin();
                    matmul_post_[id] = mp;
                    v = bn.outputs[0];
                }
            }
            plan_post(id, v, mp);
        } else if (n.op.kind == OpKind::FusedElemwise && n.outputs.size() == 1 && !is_output(n.outputs[0])) {
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1) continue;
            MatMulPost mp;
            if (is_hard_swish(g.nodes[*it->second.begin()].op, &mp.alpha, &mp.beta)) {
                mp.act = ACT_HARD_SWISH;
                chain_post_[id] = mp;
            }
        } else if (n.op.kind == OpKind::Gemm && n.outputs.size() == 1) {
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1 || is_output(n.outputs[0])) continue;
            const Node &r = g.nodes[*it->second.begin()];
            MatMulPost mp;
            if (r.op.kind == OpKind::Reshape && !r.inputs.empty() && r.inputs[0] == n.outputs[0] && r.outputs.size() == 1) {
                mp.reshaped = true;
                mp.reshape = *it->second.begin();
            }
            plan_post(id, mp.reshaped ? r.outputs[0] : n.outputs[0], mp);
        } else if (n.op.kind == OpKind::MatMul && n.outputs.size() == 1 && !is_output(n.outputs[0])) {
            auto it = users.find(n.outputs[0]);
            if (it == users.end() || it->second.size() != 1) continue;
            plan_post(id, n.outputs[0], MatMulPost());
            // MatMul -> Softmax(last axis, optional scalar scale, no mask) -> MatMul(first operand): one attention kernel.
            if (fused_attention) {
                const NodeId sid = *it->second.begin();
                const Node &sm = g.nodes[sid];
                if (sm.op.kind == OpKind::Softmax && n.inputs.size() == 2 && !sm.inputs.empty() && sm.inputs[0] == n.outputs[0] &&
                    sm.outputs.size() == 1 && !is_output(sm.outputs[0])) {
                    bool last_axis = sm.op.axis == -1;
                    auto sh = inferred_.find(sid);
                    if (!last_axis && sh != inferred_.end() && !sh->second.second.empty())
                        last_axis = sm.op.axis == (int64_t)sh->second.second[0].dims.len() - 1;
                    AttentionPlan ap;
                    ap.has_mask = sm.op.prologue_mask != 0;
                    bool scale_ok = true;
                    if (sm.op.prologue_scale) {
                        auto init = sm.inputs.size() > 1 ? g.inits.find(sm.inputs[1]) : g.inits.end();
                        scale_ok = init != g.inits.end() && init->second.elem_ty() == TensorElemType::F32 &&
                                   init->second.dims().total_elems() == 1 && init->second.has_data();
                        if (scale_ok) ap.scale_op = sm.op.prologue_scale, ap.scale = init->second.data_f32()[0];
                    }
                    auto su = users.find(sm.outputs[0]);
                    if (last_axis && scale_ok && su != users.end() && su->second.size() == 1) {
                        const NodeId tid = *su->second.begin();
                        const Node &mm = g.nodes[tid];
                        if (mm.op.kind == OpKind::MatMul && mm.inputs.size() == 2 && mm.inputs[0] == sm.outputs[0] &&
                            mm.inputs[1] != sm.outputs[0] && !mm.op.trans_a) {
                            ap.softmax = sid, ap.tail = tid;
                            attn_head_[id] = ap;
                            attn_softmax_.insert(sid);
                            attn_tail_.insert(tid);
                            continue;
                        }
                    }
                }
            }
        }
    }
    // An attention whose result goes, through the Transpose it is written ahead of and one Reshape, into a product with a
    // weight matrix and nowhere else: the attention kernel can write that product's operand planes.
    for (NodeId tid : attn_tail_) {
        auto pv = matmul_out_perm_.find(tid);
        if (pv == matmul_out_perm_.end() || pv->second != std::vector<int64_t>{0, 2, 1, 3}) continue;
        auto single_user = [&](ValueId v, NodeId *u) {
            auto it = users.find(v);
            if (it == users.end() || it->second.size() != 1 || is_output(v)) return false;
            *u = *it->second.begin();
            return true;
        };
        NodeId tr, rs, mm;
        if (!single_user(g.nodes[tid].outputs[0], &tr) || g.nodes[tr].op.kind != OpKind::Transpose || g.nodes[tr].outputs.size() != 1) continue;
        if (!single_user(g.nodes[tr].outputs[0], &rs) || g.nodes[rs].op.kind != OpKind::Reshape || g.nodes[rs].outputs.size() != 1 ||
            g.nodes[rs].inputs.empty() || g.nodes[rs].inputs[0] != g.nodes[tr].outputs[0])
            continue;
        if (!single_user(g.nodes[rs].outputs[0], &mm)) continue;
        const Node &m = g.nodes[mm];
        if (m.op.kind != OpKind::MatMul || m.inputs.size() < 2 || m.inputs[0] != g.nodes[rs].outputs[0] || m.op.trans_a ||
            planes_consumer_.count(mm) || matmul_out_perm_.count(mm))
            continue;
        bool elsewhere = false;
        for (size_t i = 1; i < m.inputs.size(); i++) elsewhere = elsewhere || m.inputs[i] == m.inputs[0];
        const Tensor *w = weight_matrix(m);
        if (elsewhere || !w) continue;
        // The planes are laid out for [b * t, h * 64] x weights [h * 64, n]: the attention's result must be [b, h, t, 64],
        // the Reshape must merge exactly the heads into the last axis (any other valid reshape, [b, t * h, 64] say, would
        // read the planes with another geometry), and the weights must have h * 64 rows.  Shapes that are not known
        // before the run leave the plan out.
        auto at = inferred_.find(tid), rt = inferred_.find(rs);
        if (at == inferred_.end() || rt == inferred_.end() || at->second.second.empty() || rt->second.second.empty()) continue;
        const FixedDimensions &ad = at->second.second[0].dims, &rd = rt->second.second[0].dims;
        if (ad.len() != 4 || ad[3] != 64 || rd.len() < 2) continue;
        const size_t merged = ad[1] * 64, rows = ad[0] * ad[2];
        size_t lead = 1;
        for (size_t i = 0; i + 1 < rd.len(); i++) lead *= rd[i];
        if (rd[rd.len() - 1] != merged || lead != rows || (m.op.trans_b ? w->dims()[1] : w->dims()[0]) != merged) continue;
        PlanesPlan pp;
        pp.consumer = mm;
        pp.next_n = m.op.trans_b ? w->dims()[0] : w->dims()[1];
        attn_planes_[tid] = pp;
        planes_consumer_.insert(mm);
        planes_pass_.insert(tr);
        planes_pass_.insert(rs);
    }
}

bool HipSession::act_planes_due(const Op &op, const std::vector<DeviceTensor *> &in) const {
    auto ap = act_planes_.find(current_node_);
    if (ap == act_planes_.end() || in.size() < 2 || !in[0] || !in[1] || !in[0]->strides.empty() || !in[1]->strides.empty() || in[0]->pending_op == PENDING_ATTENTION ||
        in[0]->elem_ty != TensorElemType::F32 || in[1]->elem_ty != TensorElemType::F32 || in[0]->dims.len() < 2 || in[1]->dims.len() != 2 || op.trans_a ||
        matmul_out_perm_.count(current_node_) || matmul_out_perm_.count(ap->second.next.consumer))
        return false;
    const FixedDimensions &ad = in[0]->dims, &wd = in[1]->dims;
    const size_t k = ad[ad.len() - 1], m = k ? ad.total_elems() / k : 0, n = op.trans_b ? wd[0] : wd[1];
    // The second product reads [m, n]; it is given planes only if it would have split its operand itself.
    return m && n && (op.trans_b ? wd[1] : wd[0]) == k && gemm_takes_split(ctx_, m, n, k) && gemm_takes_split(ctx_, m, ap->second.next.next_n, n);
}

bool HipSession::take_act_planes(size_t m, size_t n, DeviceTensor *out, void **planes, int *act, SessionError *err) {
    if (!allocate_bytes(gemm_planes_bytes(m, n), out, err)) return false;
    *planes = out->ptr;
    out->planes = true;
    out->planes_rows = m, out->planes_k = n;
    out->applied_op = *act = act_planes_.at(current_node_).act;
    activation_planes_++;
    return true;
}

void HipSession::plan_norm_chains() {
    const auto users = model_.get_value_users();
    const Graph &g = model_.graph;
    auto listed = [](const std::vector<ValueId> &l, ValueId v) { return std::find(l.begin(), l.end(), v) != l.end(); };
    // An initializer no input of the graph can stand in for.
    auto constant = [&](ValueId v) -> const Tensor * {
        auto it = g.inits.find(v);
        return it == g.inits.end() || listed(g.inputs, v) || it->second.elem_ty() != TensorElemType::F32 || !it->second.has_data() ? nullptr : &it->second;
    };
    auto scalar = [&](ValueId v) -> const Tensor * {
        const Tensor *t = constant(v);
        return t && t->dims().total_elems() == 1 && t->dims().len() <= 1 ? t : nullptr;
    };
    auto row = [&](ValueId v, size_t len) {
        const Tensor *t = constant(v);
        return t && t->dims().len() == 1 && t->dims()[0] == len;
    };
    // The node of kind `k` that reads v, where v has exactly `readers` readers and is no output of the graph.
    auto reader = [&](ValueId v, OpKind k, size_t readers, NodeId *id) -> const Node * {
        auto it = users.find(v);
        if (it == users.end() || it->second.size() != readers || listed(g.outputs, v)) return nullptr;
        const Node *found = nullptr;
        for (NodeId u : it->second)
            if (g.nodes[u].op.kind == k && g.nodes[u].inputs.size() == (k == OpKind::Sqrt || k == OpKind::ReduceMean ? 1u : 2u) && g.nodes[u].outputs.size() == 1) {
                if (found) return nullptr;
                found = &g.nodes[u], *id = u;
            }
        return found;
    };
    for (const NodeExecutionPlan &step : plan_) {
        const Node &mean = g.nodes[step.node_id];
        if (mean.op.kind != OpKind::ReduceMean || mean.inputs.size() != 1 || mean.outputs.size() != 1) continue;
        const ValueId x = mean.inputs[0];
        auto inferred = inferred_.find(step.node_id);
        if (inferred == inferred_.end() || inferred->second.second.empty()) continue;
        const int64_t rank = (int64_t)inferred->second.second[0].dims.len();  // of x as well: the axis is kept
        auto last_axis = [&](const Node &n) {
            return n.op.keep_dims && n.op.axes.size() == 1 && (n.op.axes[0] == -1 || n.op.axes[0] == rank - 1);
        };
        if (rank < 1 || !last_axis(mean)) continue;
        NormChainPlan c;
        c.rest.resize(8);
        const Node *sub = reader(mean.outputs[0], OpKind::Sub, 1, &c.rest[0]);
        if (!sub || sub->inputs[0] != x || sub->inputs[1] != mean.outputs[0] || x == mean.outputs[0]) continue;
        const ValueId d = sub->outputs[0];
        const Node *pow = reader(d, OpKind::Pow, 2, &c.rest[1]), *div = reader(d, OpKind::Div, 2, &c.rest[6]);
        if (!pow || !div || pow->inputs[0] != d || div->inputs[0] != d || div->inputs[1] == d) continue;
        const Tensor *two = scalar(pow->inputs[1]);
        if (!two || two->data_f32()[0] != 2.0f) continue;
        const Node *var = reader(pow->outputs[0], OpKind::ReduceMean, 1, &c.rest[2]);
        if (!var || !last_axis(*var)) continue;
        const Node *add = reader(var->outputs[0], OpKind::Add, 1, &c.rest[3]);
        if (!add) continue;
        const Tensor *eps = scalar(add->inputs[add->inputs[0] == var->outputs[0] ? 1 : 0]);
        const Node *sqrt = eps ? reader(add->outputs[0], OpKind::Sqrt, 1, &c.rest[4]) : nullptr;
        NodeId div_id = 0;
        if (!sqrt || reader(sqrt->outputs[0], OpKind::Div, 1, &div_id) != div || div->inputs[1] != sqrt->outputs[0]) continue;
        const Node *mul = reader(div->outputs[0], OpKind::Mul, 1, &c.rest[5]);
        if (!mul) continue;
        const Node *shift = reader(mul->outputs[0], OpKind::Add, 1, &c.rest[7]);
        if (!shift) continue;
        // The row length: gamma's, checked against x when the chain runs.
        c.gamma = mul->inputs[mul->inputs[0] == div->outputs[0] ? 1 : 0];
        c.beta = shift->inputs[shift->inputs[0] == mul->outputs[0] ? 1 : 0];
        const Tensor *gamma = constant(c.gamma);
        if (!gamma || gamma->dims().len() != 1 || !row(c.beta, gamma->dims()[0])) continue;
        c.result = shift->outputs[0];
        c.eps = eps->data_f32()[0];
        norm_chains_[step.node_id] = std::move(c);
    }
}

bool HipSession::run_norm_chain(NodeId id, const DeviceTensor &x, std::map<ValueId, DeviceTensor> &values, bool *done, SessionError *err) {
    const NormChainPlan &c = norm_chains_[id];
    const DeviceTensor &gamma = inits_.at(c.gamma), &beta = inits_.at(c.beta);
    const size_t rank = x.dims.len(), len = rank ? x.dims[rank - 1] : 0;
    if (x.elem_ty != TensorElemType::F32 || len == 0 || gamma.dims[0] != len || !x.strides.empty()) return true;
    const size_t rows = x.dims.total_elems() / len;
    DeviceTensor out;
    const float *in = static_cast<const float *>(x.ptr), *gp = static_cast<const float *>(gamma.ptr), *bp = static_cast<const float *>(beta.ptr);
    if (!norm_chain_fits(in, in, gp, bp, rows, len)) return true;  // the result's block is aligned like every other
    if (!allocate({x.dims, x.elem_ty}, &out, err)) return false;
    const int rc = launch_norm_chain(ctx_, static_cast<float *>(out.ptr), in, gp, bp, rows, len, c.eps);
    if (rc) return fail_code(err, rc, ctx_.last_error);
    values[c.result] = std::move(out);
    passed_over_.insert(c.rest.begin(), c.rest.end());
    copies_avoided_ += c.rest.size();
    *done = true;
    return true;
}

void HipSession::plan_attention_rows() {
    const auto users = model_.get_value_users();
    const Graph &g = model_.graph;
    auto listed = [](const std::vector<ValueId> &l, ValueId v) { return std::find(l.begin(), l.end(), v) != l.end(); };
    // One f32 value that nothing can stand in for.
    auto scalar = [&](ValueId v, float *value) {
        auto it = g.inits.find(v);
        if (it == g.inits.end() || listed(g.inputs, v) || it->second.elem_ty() != TensorElemType::F32 || it->second.dims().total_elems() != 1 ||
            !it->second.has_data())
            return false;
        *value = it->second.data_f32()[0];
        return true;
    };
    // The only reader of v, which is no output of the graph and read once.
    auto reader = [&](ValueId v, NodeId *id) -> const Node * {
        auto it = users.find(v);
        if (it == users.end() || it->second.size() != 1 || listed(g.outputs, v)) return nullptr;
        const Node &n = g.nodes[*id = *it->second.begin()];
        return n.outputs.size() == 1 && std::count(n.inputs.begin(), n.inputs.end(), v) == 1 ? &n : nullptr;
    };
    for (const NodeExecutionPlan &step : plan_) {
        const Node &head = g.nodes[step.node_id];
        if (head.op.kind != OpKind::MatMul || head.inputs.size() != 2 || head.outputs.size() != 1 || attn_head_.count(step.node_id)) continue;
        auto scores = inferred_.find(step.node_id);
        if (scores == inferred_.end() || scores->second.second.empty()) continue;
        const FixedDimensions &dims = scores->second.second[0].dims;
        if (dims.len() < 2) continue;
        auto same_shape = [&](NodeId id) {
            auto it = inferred_.find(id);
            return it != inferred_.end() && !it->second.second.empty() && it->second.second[0].dims == dims;
        };
        AttentionRowsPlan p;
        ValueId v = head.outputs[0];
        NodeId id = 0;
        const Node *n = reader(v, &id);
        if (n && (n->op.kind == OpKind::Div || n->op.kind == OpKind::Mul) && n->inputs.size() == 2 && same_shape(id)) {
            const bool first = n->inputs[0] == v;
            if (!(first || n->op.kind == OpKind::Mul) || !scalar(n->inputs[first ? 1 : 0], &p.scale)) continue;
            p.scale_op = n->op.kind == OpKind::Mul ? 1 : 2;
            p.rest.push_back(id);
            v = n->outputs[0];
            n = reader(v, &id);
        }
        if (n && n->op.kind == OpKind::Where && n->inputs.size() == 3 && n->inputs[1] == v && same_shape(id)) {
            if (!scalar(n->inputs[2], &p.fill)) continue;
            p.has_where = true;
            p.cond = n->inputs[0];
            p.rest.push_back(id);
            v = n->outputs[0];
            n = reader(v, &id);
        }
        bool added = false;  // a mask that the Softmax has not absorbed
        if (n && n->op.kind == OpKind::Add && n->inputs.size() == 2 && same_shape(id)) {
            added = true;
            p.mask = n->inputs[n->inputs[0] == v ? 1 : 0];
            p.rest.push_back(id);
            v = n->outputs[0];
            n = reader(v, &id);
        }
        if (!n || n->op.kind != OpKind::Softmax || n->inputs.empty() || n->inputs[0] != v || !same_shape(id)) continue;
        if (added && (n->op.prologue_scale || n->op.prologue_mask)) continue;
        if (n->op.axis != -1 && n->op.axis != (int64_t)dims.len() - 1) continue;
        p.softmax_op = n->op.prologue_scale, p.has_mask = n->op.prologue_mask;
        if (n->inputs.size() != 1u + (p.softmax_op ? 1 : 0) + (p.has_mask ? 1 : 0)) continue;
        if (p.softmax_op && !scalar(n->inputs[1], &p.softmax_scale)) continue;
        if (p.has_mask) p.mask = n->inputs.back();
        p.has_mask = p.has_mask || added;
        p.rest.push_back(id);
        v = n->outputs[0];
        n = reader(v, &id);
        if (!n || n->op.kind != OpKind::MatMul || n->inputs.size() != 2 || n->inputs[0] != v || n->op.trans_a) continue;
        auto result = inferred_.find(id);
        if (result == inferred_.end() || result->second.second.empty()) continue;
        p.rest.push_back(id);
        attention_rows_[step.node_id] = std::move(p);
    }
}

namespace {
// An operand whose values are there, as fp32 (or as conditions).
bool readable(const DeviceTensor *t, TensorElemType ty) {
    return t && t->ptr && t->elem_ty == ty && t->pending_op < 0 && t->applied_op < 0 && !t->planes && !t->owes_add() && t->dims.len() >= 2;
}
}  // namespace

bool HipSession::attention_rows_takes(NodeId id, const std::vector<DeviceTensor *> &in) const {
    const FixedDimensions &sd = inferred_.at(id).second[0].dims, &od = inferred_.at(attention_rows_.at(id).rest.back()).second[0].dims;
    if (in.size() != 2 || !readable(in[0], TensorElemType::F32) || !readable(in[1], TensorElemType::F32) || od.len() != sd.len()) return false;
    const size_t rank = sd.len();
    size_t batch = 1, axes = 0;
    for (size_t i = 0; i + 2 < rank; i++) {
        if (od[i] != sd[i]) return false;
        batch *= sd[i];
        axes += sd[i] != 1;
    }
    const bool wide = (inferred_.at(id).first.trans_a ? in[0]->dims[in[0]->dims.len() - 2] : in[0]->dims[in[0]->dims.len() - 1]) == 64;
    if (!wide || axes > 2 || od[rank - 2] != sd[rank - 2] || od[rank - 1] != 64) return false;
    return attention_rows_fits(ctx_, batch, sd[rank - 2], sd[rank - 1]);
}

bool HipSession::finish_attention_rows(NodeId id, NodeId tail, std::map<ValueId, DeviceTensor> &values, SessionError *err) {
    const AttentionRowsPlan &p = attention_rows_.at(id);
    for (NodeId n : p.rest) attention_held_.erase(n);
    bool done = false;
    if (!run_attention_rows(id, values, &done, err)) return false;
    if (!done) {
        // What they read may have been let go in the meantime.
        std::vector<ValueId> again;
        for (auto &kv : attention_operands_[id])
            if (values.emplace(kv.first, kv.second).second) again.push_back(kv.first);
        attention_apart_ = true;
        bool ok = run_node(id, values, err);
        for (NodeId n : p.rest) ok = ok && run_node(n, values, err);
        attention_apart_ = false;
        if (!ok) return false;
        for (ValueId v : again) values.erase(v);
        values.erase(model_.graph.nodes[id].outputs[0]);
        for (NodeId n : p.rest)
            if (n != tail) values.erase(model_.graph.nodes[n].outputs[0]);
    }
    attention_operands_.erase(id);
    return true;
}

bool HipSession::run_attention_rows(NodeId id, std::map<ValueId, DeviceTensor> &values, bool *done, SessionError *err) {
    const AttentionRowsPlan &p = attention_rows_.at(id);
    const Node &head = model_.graph.nodes[id], &tail = model_.graph.nodes[p.rest.back()];
    const Op &head_op = inferred_.at(id).first, &tail_op = inferred_.at(p.rest.back()).first;
    const FixedDimensions &sd = inferred_.at(id).second[0].dims, &od = inferred_.at(p.rest.back()).second[0].dims;
    const size_t rank = sd.len(), tq = sd[rank - 2], tk = sd[rank - 1];
    std::vector<size_t> bd;
    size_t batch = 1;
    for (size_t i = 0; i + 2 < rank; i++) {
        batch *= sd[i];
        if (sd[i] != 1) bd.push_back(sd[i]);
    }
    std::map<ValueId, DeviceTensor> &operands = attention_operands_[id];
    auto value = [&](ValueId v) -> DeviceTensor * {
        auto it = operands.find(v);
        if (it != operands.end()) return &it->second;
        auto ii = inits_.find(v);
        return ii != inits_.end() ? &ii->second : nullptr;
    };
    DeviceTensor *in[2] = {value(head.inputs[0]), value(head.inputs[1])};
    DeviceTensor *vt = value(tail.inputs[1]), *ct = p.has_where ? value(p.cond) : nullptr, *mt = p.has_mask ? value(p.mask) : nullptr;
    if (!in[0] || !in[1] || !readable(vt, TensorElemType::F32)) return true;
    auto over = [&](const DeviceTensor *t, TensorElemType ty) { return t && t->ptr && t->elem_ty == ty && t->pending_op < 0 && t->applied_op < 0 && !t->planes && !t->owes_add() && t->strides.empty(); };
    if ((p.has_where && !over(ct, TensorElemType::Bool)) || (p.has_mask && !over(mt, TensorElemType::F32))) return true;
    MatOperand Q, K, V;
    if (!describe_operand(in[0], &Q, err) || !describe_operand(in[1], &K, err) || !describe_operand(vt, &V, err)) return false;
    // Q [tq, 64], K [tk, 64] and V [tk, 64] as stored rows.
    const bool q_rows = head_op.trans_a == Q.stored_transposed, k_rows = head_op.trans_b != K.stored_transposed, v_rows = tail_op.trans_b == V.stored_transposed;
    auto extent = [](const MatOperand &o, size_t r) { return (o.stored_transposed ? o.cols : o.rows) == r && (o.stored_transposed ? o.rows : o.cols) == 64; };
    if (!q_rows || !k_rows || !v_rows || !extent(Q, tq) || !extent(K, tk) || !extent(V, tk)) return true;
    // (Keys or values that all heads share make one tall product of the heads' rows, which may add up in another order.)
    if (Q.batch != batch || K.batch != batch || V.batch != batch) return true;
    std::vector<int64_t> qs, ks, vs;
    if (!operand_batch_strides(bd, Q.bdims, Q.bstr, in[0]->strides.empty(), tq * 64, Q.batch, &qs) ||
        !operand_batch_strides(bd, K.bdims, K.bstr, in[1]->strides.empty(), tk * 64, K.batch, &ks) ||
        !operand_batch_strides(bd, V.bdims, V.bstr, vt->strides.empty(), tk * 64, V.batch, &vs))
        return true;
    AttentionRows a;
    auto two = [&](const std::vector<int64_t> &s, size_t out2[2]) {
        out2[0] = s.size() > 0 ? (size_t)s[0] : 0;
        out2[1] = s.size() > 1 ? (size_t)s[1] : 0;
    };
    two(qs, a.q_bs), two(ks, a.k_bs), two(vs, a.v_bs);
    // A condition or mask over the scores: strides of the batch axes, the query and the key.
    auto over_scores = [&](const DeviceTensor *t, size_t out4[4]) {
        auto st = t->dims.strides_for_broadcasting_to(sd);
        if (!st || st->len() != rank) return false;
        std::vector<int64_t> b;
        for (size_t i = 0; i + 2 < rank; i++)
            if (sd[i] != 1) b.push_back((int64_t)(*st)[i]);
        two(b, out4);
        out4[2] = (*st)[rank - 2], out4[3] = (*st)[rank - 1];
        return true;
    };
    if ((ct && !over_scores(ct, a.cond_strides)) || (mt && !over_scores(mt, a.mask_strides))) return true;

    DeviceTensor out;
    if (!allocate({od, TensorElemType::F32}, &out, err)) return false;
    // Dense, or the layout of the Transpose behind the last product.
    std::vector<int64_t> c_str = dense_strides(od);
    auto pv = matmul_out_perm_.find(p.rest.back());
    if (pv != matmul_out_perm_.end() && pv->second.size() == rank) {
        FixedDimensions td = od;
        for (size_t i = 0; i < rank; i++) td[i] = od[(size_t)pv->second[i]];
        const std::vector<int64_t> ts = dense_strides(td);
        for (size_t i = 0; i < rank; i++) c_str[(size_t)pv->second[i]] = ts[i];
        if (!is_dense(od, c_str)) out.strides = c_str;
    }
    std::vector<int64_t> os;
    for (size_t i = 0; i + 2 < rank; i++)
        if (od[i] != 1) os.push_back(c_str[i]);
    two(os, a.o_bs);
    auto f = [](const DeviceTensor *t) { return static_cast<const float *>(t->ptr); };
    a.q = f(in[0]), a.k = f(in[1]), a.v = f(vt), a.o = static_cast<float *>(out.ptr);
    a.mask = mt ? f(mt) : nullptr, a.cond = ct ? static_cast<const uint8_t *>(ct->ptr) : nullptr;
    a.batch_outer = bd.size() > 0 ? bd[0] : 1, a.batch_inner = bd.size() > 1 ? bd[1] : 1;
    a.tq = tq, a.tk = tk, a.ldq = Q.ld, a.ldk = K.ld, a.ldv = V.ld, a.ldo = tq > 1 ? (size_t)c_str[rank - 2] : 64;
    a.scale_op = p.scale_op, a.scale = p.scale, a.softmax_op = p.softmax_op, a.softmax_scale = p.softmax_scale, a.fill = p.fill;
    const int rc = launch_attention_rows(ctx_, a);
    if (rc == AHIP_ERR_UNSUPPORTED) return true;
    if (rc) return fail_code(err, rc, ctx_.last_error);
    values[tail.outputs[0]] = std::move(out);
    attentions_++;
    *done = true;
    return true;
}

}  // namespace altius
