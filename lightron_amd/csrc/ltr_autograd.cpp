// C++ autograd node of the attention library: the host side of lightron_amd.attention.BlockAttentionFunction (a Q chunk against a table
// of K/V chunks: a ring's share, or the one chunk of an SDPA call site of the reference, model/model.py:193-198 and
// parallel/parallel_cp.py:224-229) moved out of Python.  The same C-ABI calls (ltr_attn_fwd, ltr_attn_bwd_delta, ltr_attn_bwd_ws,
// ltr_cast_f32_to_bf16), but arguments are filled here and the backward runs on the autograd thread as a C++ node - no
// interpreter lock to take, no Python frames - which is where the time of short calls goes: four ranks of 256 fp32 tokens
// forward and backward: 846 us through the Python node, 389 us through this one.  A bf16 call of 4 x 12 heads x 128 tokens takes
// 70 us (41 - 87 by process), its three kernels 29 us; this node with the same allocations and no launches 55 - 56 us, a
// training pass of one torch.addcmul in the same process 69 us: what is left there is torch's engine.
// No device code here: torch is used for tensors and autograd only, the kernels are those of libltr_attn.so.
#include <torch/extension.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "ltr_attn.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void strides3(const Tensor &t, int64_t *out) {
    out[0] = t.stride(0);
    out[1] = t.stride(1);
    out[2] = t.stride(2);
}

void require_bshd(const Tensor &t, const char *name) {
    TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor (the HIP library has no CPU path)");
    TORCH_CHECK(t.dim() == 4 && (t.numel() == 0 || t.stride(3) == 1), name, " must be [B,S,H,D] with a contiguous last dim");
}

void check_rc(int rc, const char *what) { TORCH_CHECK(rc == 0, what, " failed: ", ltr_strerror(rc), " (", rc, ")"); }

bool same_strides(const Tensor &a, const Tensor &b) { return a.stride(0) == b.stride(0) && a.stride(1) == b.stride(1) && a.stride(2) == b.stride(2); }

// One entry of the chunk table: `rows` keys of tensor `t` from row `row0` on, the first of them at global position pos0.
struct Entry {
    int64_t t, row0, rows, pos0;
};

// Everything of a call but the differentiable tensors; kept by the node for its backward.
struct Call : torch::CustomClassHolder {
    std::vector<Entry> entries;
    int64_t q_pos0[2] = {0, 0}, q_split = 0;
    bool causal = false;
    double scale = 0;
    int64_t stream = 0;
    int64_t step = 0;               // 0: one launch over the table; g: one launch per g entries, merged into an fp32 (O, LSE)
    bool out_f32 = false;           // O is returned in fp32
    std::vector<Tensor> dk, dv;     // fp32 accumulators shaped like the K / V tensors: dK / dV are added there, none are returned
    Tensor rope;                    // fp32 [n_pos, D/2, 2] (cos, sin) table indexed by global position, or undefined (no fused RoPE)
};

char *row_ptr(const Tensor &t, int64_t row) { return (char *)t.data_ptr() + row * t.stride(1) * t.element_size(); }

// Saved-tensor hooks may hand a tensor back in another layout than it was saved in; the kernels want whole rows, and one stride
// triple for all K and one for all V tensors of a table.
Tensor rows_contiguous(const Tensor &t) {
    const bool cols = t.size(3) != 64 && t.size(3) != 128 && ((t.stride(0) | t.stride(1) | t.stride(2)) % 8 || (uintptr_t)t.data_ptr() % 16);
    return (t.numel() == 0 || t.stride(3) == 1) && !cols ? t : t.clone(at::MemoryFormat::Contiguous);
}

std::vector<Tensor> one_layout(const Tensor *t, int64_t n) {
    std::vector<Tensor> out;
    bool alike = true;
    for (int64_t i = 0; i < n; i++) {
        out.push_back(rows_contiguous(t[i]));
        alike = alike && same_strides(out[i], out[0]);
    }
    if (alike) return out;
    const Tensor all = at::cat(out, 1);
    for (int64_t i = 0, row = 0; i < n; row += out[i++].size(1)) out[i] = all.narrow(1, row, out[i].size(1));
    return out;
}

// The arithmetic of both nodes below.  kv: the K tensors, then as many V tensors
struct ChunksFunction {
    static variable_list forward(AutogradContext *ctx, const Tensor &q, at::TensorList kv, const c10::intrusive_ptr<Call> &call) {
        const c10::DeviceGuard on_q_device(q.device());   // the library launches on the CURRENT device
        const Call &c = *call;
        const int64_t n_t = (int64_t)kv.size() / 2, B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3), n = (int64_t)c.entries.size();
        const Tensor &k0 = kv[0], &v0 = kv[n_t];
        const bool f32 = q.scalar_type() == at::kFloat, stepwise = c.step > 0, o_f32 = stepwise || c.out_f32;
        Tensor o = torch::empty({B, Sq, Hq, D}, q.options().dtype(o_f32 ? at::kFloat : at::kBFloat16));
        Tensor lse = torch::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
        Tensor q_rot;
        const bool with_rope = c.rope.defined();
        if (with_rope) q_rot = torch::empty({B, Sq, Hq, D}, q.options());
        if (q.numel() > 0) {
            ltr_attn_fwd_args a{};
            a.q = q.data_ptr();
            a.o = o.data_ptr();
            a.lse = lse.data_ptr<float>();
            a.B = (int32_t)B;
            a.Hq = (int32_t)Hq;
            a.Hkv = (int32_t)k0.size(2);
            a.D = (int32_t)D;
            a.Sq = Sq;
            strides3(q, a.q_stride);
            strides3(o, a.o_stride);
            strides3(k0, a.k_stride);
            strides3(v0, a.v_stride);
            a.q_pos0[0] = c.q_pos0[0];
            a.q_pos0[1] = c.q_pos0[1];
            a.q_split = c.q_split;
            a.scale = (float)c.scale;
            a.io_dtype = f32 ? LTR_F32 : LTR_BF16;
            a.o_dtype = o_f32 ? LTR_F32 : LTR_BF16;
            const uint32_t cols = D == 64 || D == 128 ? 0u : LTR_HEAD_COLS;
            if (with_rope) {
                a.rope_freqs = c.rope.data_ptr<float>();
                a.rope_len = c.rope.size(0);
                a.q_rot = q_rot.data_ptr();
                strides3(q_rot, a.q_rot_stride);
            }
            const int64_t group = std::min<int64_t>(stepwise ? c.step : n, LTR_MAX_CHUNKS);
            for (int64_t first = 0; first < n; first += group) {
                a.n_chunks = (int32_t)std::min(group, n - first);
                for (int64_t i = 0; i < a.n_chunks; i++) {
                    const Entry &e = c.entries[first + i];
                    a.chunk[i].k = row_ptr(kv[e.t], e.row0);
                    a.chunk[i].v = row_ptr(kv[n_t + e.t], e.row0);
                    a.chunk[i].sk = e.rows;
                    a.chunk[i].pos0 = e.pos0;
                }
                a.flags = cols | (c.causal ? LTR_CAUSAL : 0u) | (with_rope ? LTR_ROPE_Q : 0u) | (first > 0 ? LTR_MERGE : 0u);
                check_rc(ltr_attn_fwd(&a, (void *)c.stream), "ltr_attn_fwd");
                a.q_rot = nullptr;   // stored by the first launch
            }
        }
        if (o_f32 && !c.out_f32) o = o.to(at::kBFloat16);
        variable_list saved{with_rope ? q_rot : q, o, lse, c.rope};
        saved.insert(saved.end(), kv.begin(), kv.end());
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["call"] = c10::IValue::make_capsule(call);   // with its stream: the engine runs the backward on the forward's
        ctx->mark_non_differentiable({lse});
        ctx->set_materialize_grads(false);                           // no zero tensor for the gradient of lse
        return {o, lse};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
        const Call &c = *call;
        const Tensor q = rows_contiguous(saved[0]), o = rows_contiguous(saved[1]), lse = saved[2].contiguous();
        const Tensor &rope = saved[3];
        const int64_t n_t = ((int64_t)saved.size() - 4) / 2, n = (int64_t)c.entries.size();
        const std::vector<Tensor> ks = one_layout(&saved[4], n_t), vs = one_layout(&saved[4] + n_t, n_t);
        variable_list out(1 + 2 * n_t + 1);
        if (!grads[0].defined()) return out;
        const c10::DeviceGuard on_q_device(q.device());
        const bool f32 = q.scalar_type() == at::kFloat, own_acc = !c.dk.empty();
        Tensor d_o = grads[0];
        if (d_o.scalar_type() != q.scalar_type()) d_o = d_o.to(q.scalar_type());
        if (d_o.stride(3) != 1) d_o = d_o.contiguous();
        const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = ks[0].size(2);
        const uint32_t cols = D == 64 || D == 128 ? 0u : LTR_HEAD_COLS;
        if (cols && ((d_o.stride(0) | d_o.stride(1) | d_o.stride(2)) % 8 || (uintptr_t)d_o.data_ptr() % 16)) d_o = d_o.clone(at::MemoryFormat::Contiguous);
        // gradients of the K / V tensors: one tensor each when their strides then agree, else slices of one buffer
        std::vector<Tensor> dk(n_t), dv(n_t);
        if (own_acc) {
            dk = c.dk;
            dv = c.dv;
        } else {
            bool alike = true;
            int64_t total = 0;
            for (int64_t t = 0; t < n_t; t++) {
                alike = alike && (B == 1 || ks[t].size(1) == ks[0].size(1));
                total += ks[t].size(1);
            }
            const auto fresh = [&](int64_t rows) {
                return f32 ? torch::zeros({B, rows, Hkv, D}, q.options()) : torch::empty({B, rows, Hkv, D}, q.options());
            };
            if (alike) {
                for (int64_t t = 0; t < n_t; t++) dk[t] = fresh(ks[t].size(1)), dv[t] = fresh(ks[t].size(1));
            } else {
                const Tensor kb = fresh(total), vb = fresh(total);
                for (int64_t t = 0, at = 0; t < n_t; at += ks[t++].size(1))
                    dk[t] = kb.narrow(1, at, ks[t].size(1)), dv[t] = vb.narrow(1, at, ks[t].size(1));
            }
            for (int64_t t = 0; t < n_t; t++) out[1 + t] = dk[t], out[1 + n_t + t] = dv[t];
        }
        if (q.numel() == 0) {
            out[0] = torch::empty(q.sizes(), q.options());
            if (!own_acc && !f32)
                for (int64_t t = 0; t < n_t; t++) dk[t].zero_(), dv[t].zero_();
            return out;
        }
        // one launch sees every chunk: dQ is written by the kernel; otherwise it accumulates in fp32
        const bool direct = !f32 && n <= LTR_MAX_CHUNKS;
        const bool direct32 = f32 && n <= LTR_MAX_CHUNKS && o.scalar_type() == at::kFloat && (o.stride(0) | o.stride(1) | o.stride(2)) % 4 == 0 &&
                              (uintptr_t)o.data_ptr() % 16 == 0;
        const bool delta_from_o = direct32 || (!f32 && o.scalar_type() == at::kBFloat16);
        Tensor dq = direct || direct32 ? torch::empty({B, Sq, Hq, D}, q.options()) : torch::zeros({B, Sq, Hq, D}, q.options().dtype(at::kFloat));
        Tensor delta = torch::empty({B, Hq, Sq}, lse.options());   // with delta_from_o a workspace: filled by the dQ kernel, or before a joint launch
        if (!delta_from_o) {
            ltr_attn_delta_args d{};
            d.o = o.data_ptr();
            d.d_o = d_o.data_ptr();
            d.delta = delta.data_ptr<float>();
            d.B = (int32_t)B;
            d.Hq = (int32_t)Hq;
            d.D = (int32_t)D;
            d.Sq = Sq;
            strides3(o, d.o_stride);
            strides3(d_o, d.do_stride);
            d.o_dtype = o.scalar_type() == at::kFloat ? LTR_F32 : LTR_BF16;
            d.do_dtype = f32 ? LTR_F32 : LTR_BF16;
            check_rc(ltr_attn_bwd_delta(&d, (void *)c.stream), "ltr_attn_bwd_delta");
        }
        ltr_attn_bwd_args a{};
        a.q = q.data_ptr();
        a.d_o = d_o.data_ptr();
        a.lse = lse.data_ptr<float>();
        a.delta = delta.data_ptr<float>();
        a.dq = dq.data_ptr();
        a.B = (int32_t)B;
        a.Hq = (int32_t)Hq;
        a.Hkv = (int32_t)Hkv;
        a.D = (int32_t)D;
        a.Sq = Sq;
        strides3(q, a.q_stride);
        strides3(d_o, a.do_stride);
        strides3(dq, a.dq_stride);
        strides3(ks[0], a.k_stride);
        strides3(vs[0], a.v_stride);
        strides3(dk[0], a.dk_stride);
        strides3(dv[0], a.dv_stride);
        if (delta_from_o) {
            a.o = o.data_ptr();
            strides3(o, a.o_stride);
        }
        a.q_pos0[0] = c.q_pos0[0];
        a.q_pos0[1] = c.q_pos0[1];
        a.q_split = c.q_split;
        a.scale = (float)c.scale;
        a.io_dtype = f32 ? LTR_F32 : LTR_BF16;
        if (rope.defined()) {
            a.rope_freqs = rope.data_ptr<float>();
            a.rope_len = rope.size(0);
        }
        for (int64_t first = 0; first < n; first += LTR_MAX_CHUNKS) {
            a.n_chunks = (int32_t)std::min<int64_t>(LTR_MAX_CHUNKS, n - first);
            for (int64_t i = 0; i < a.n_chunks; i++) {
                const Entry &e = c.entries[first + i];
                a.chunk[i].k = row_ptr(ks[e.t], e.row0);
                a.chunk[i].v = row_ptr(vs[e.t], e.row0);
                a.chunk[i].dk = row_ptr(dk[e.t], e.row0);
                a.chunk[i].dv = row_ptr(dv[e.t], e.row0);
                a.chunk[i].sk = e.rows;
                a.chunk[i].pos0 = e.pos0;
            }
            // this node holds every key these rows see and every row of it that sees these keys: the kernels write bf16 results
            a.flags = cols | (c.causal ? LTR_CAUSAL : 0u) | (direct ? LTR_DQ_BF16 : 0u) | (!f32 && !own_acc ? LTR_DKDV_BF16 : 0u) |
                      (direct32 ? LTR_DQ_F32_RESULT : delta_from_o && first == 0 ? LTR_DELTA_FROM_O : 0u) | (rope.defined() ? LTR_ROPE_DQ : 0u) | LTR_BWD_JOINT;   // the results are fresh tensors or the ring's accumulators
            // few key tiles: blocks share them and leave partial sums in a workspace (from torch's caching allocator)
            int64_t part_bytes = 0;
            check_rc(ltr_attn_bwd_workspace(&a, &part_bytes), "ltr_attn_bwd_workspace");
            Tensor part;
            if (part_bytes > 0) part = torch::empty({part_bytes}, q.options().dtype(at::kByte));
            check_rc(ltr_attn_bwd_ws(&a, part_bytes > 0 ? part.data_ptr() : nullptr, part_bytes, (void *)c.stream), "ltr_attn_bwd");
        }
        if (!direct && !f32) {
            Tensor dq16 = torch::empty({B, Sq, Hq, D}, q.options());
            check_rc(ltr_cast_f32_to_bf16(dq.data_ptr<float>(), dq16.data_ptr(), dq.numel(), (void *)c.stream), "ltr_cast_f32_to_bf16");
            dq = dq16;
        }
        out[0] = dq;
        return out;
    }
};

struct ChunksNode : torch::autograd::Function<ChunksNode> {
    static variable_list forward(AutogradContext *ctx, const Tensor &q, at::TensorList kv, const c10::intrusive_ptr<Call> &call) {
        return ChunksFunction::forward(ctx, q, kv, call);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) { return ChunksFunction::backward(ctx, std::move(grads)); }
};

// the same under the name that profiles of a one-chunk call show
struct SingleChunkNode : torch::autograd::Function<SingleChunkNode> {
    static variable_list forward(AutogradContext *ctx, const Tensor &q, at::TensorList kv, const c10::intrusive_ptr<Call> &call) {
        return ChunksFunction::forward(ctx, q, kv, call);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) { return ChunksFunction::backward(ctx, std::move(grads)); }
};

void require_rope(const Tensor &rope, const Tensor &q) {
    TORCH_CHECK(q.scalar_type() == at::kBFloat16, "the fused RoPE prologue is implemented for bf16 q");
    TORCH_CHECK(rope.scalar_type() == at::kFloat && rope.dim() == 3 && rope.size(1) == q.size(3) / 2 && rope.size(2) == 2 && rope.is_contiguous() &&
                    rope.device() == q.device(),
                "the RoPE table must be a contiguous fp32 [n_pos, D/2, 2] (cos, sin) tensor on q's device");
}

// (O [B,Sq,Hq,D] bf16, LSE [B,Hq,Sq] fp32) of one bf16 chunk; stream = hipStream_t of torch's current stream on q's device, as an integer
std::vector<Tensor> single_chunk(const Tensor &q, const Tensor &k, const Tensor &v, int64_t k_pos0, int64_t q_pos0a, int64_t q_pos0b,
                                 int64_t q_split, bool causal, double scale, int64_t stream, const c10::optional<Tensor> &rope) {
    require_bshd(q, "q");
    require_bshd(k, "k");
    require_bshd(v, "v");
    TORCH_CHECK(q.scalar_type() == at::kBFloat16 && k.scalar_type() == at::kBFloat16 && v.scalar_type() == at::kBFloat16, "q, k, v must be bf16");
    TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3) && k.device() == q.device() && v.device() == q.device(),
                "k/v chunk shape or device mismatch");
    auto c = c10::make_intrusive<Call>();
    c->entries = {{0, 0, k.size(1), k_pos0}};
    c->q_pos0[0] = q_pos0a;
    c->q_pos0[1] = q_pos0b;
    c->q_split = q_split;
    c->causal = causal;
    c->scale = scale;
    c->stream = stream;
    if (rope.has_value()) {
        require_rope(*rope, q);
        c->rope = *rope;
    }
    const Tensor kv[2] = {k, v};
    return SingleChunkNode::apply(q, at::TensorList(kv, 2), c);
}

// A table of chunks: kv = the K tensors, then the V tensors; entries = flat (tensor, first row, rows, position of the first) per
// table entry; dk / dv = fp32 accumulators per tensor, or empty.  Empty result: tensors whose strides do not agree (one stride
// triple describes all K, one all V chunks of a launch); the caller packs them.
std::vector<Tensor> chunks(const Tensor &q, std::vector<Tensor> kv, const std::vector<int64_t> &entries, int64_t q_pos0a, int64_t q_pos0b,
                           int64_t q_split, bool causal, double scale, int64_t stream, int64_t step, bool out_f32, std::vector<Tensor> dk,
                           std::vector<Tensor> dv, const c10::optional<Tensor> &rope) {
    require_bshd(q, "q");
    TORCH_CHECK(q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kFloat, "q must be bf16 or fp32");
    const size_t n_t = kv.size() / 2;
    TORCH_CHECK(n_t > 0 && kv.size() == 2 * n_t && entries.size() % 4 == 0 && !entries.empty(), "a chunk table needs K and V tensors and entries");
    for (size_t t = 0; t < 2 * n_t; t++) {
        const Tensor &x = kv[t];
        require_bshd(x, t < n_t ? "k" : "v");
        TORCH_CHECK(x.scalar_type() == q.scalar_type() && x.sizes() == kv[t % n_t].sizes() && x.size(0) == q.size(0) && x.size(3) == q.size(3) &&
                        x.size(2) == kv[0].size(2) && x.device() == q.device(),
                    "k/v chunk shape, dtype or device mismatch");
        if (!same_strides(x, kv[t < n_t ? 0 : n_t])) return {};
    }
    TORCH_CHECK(dk.size() == dv.size() && (dk.empty() || dk.size() == n_t), "one dK and one dV accumulator per K / V tensor");
    for (size_t t = 0; t < dk.size(); t++) {
        for (const Tensor *x : {&dk[t], &dv[t]})
            TORCH_CHECK(x->scalar_type() == at::kFloat && x->sizes() == kv[t].sizes() && x->stride(3) == 1 && x->device() == q.device(),
                        "accumulators must be fp32 tensors shaped like their chunks");
        if (!same_strides(dk[t], dk[0]) || !same_strides(dv[t], dv[0])) return {};
    }
    auto c = c10::make_intrusive<Call>();
    for (size_t i = 0; i < entries.size(); i += 4) {
        const Entry e{entries[i], entries[i + 1], entries[i + 2], entries[i + 3]};
        TORCH_CHECK(e.t >= 0 && e.t < (int64_t)n_t && e.row0 >= 0 && e.rows > 0 && e.row0 + e.rows <= kv[e.t].size(1), "chunk table entry outside its tensor");
        c->entries.push_back(e);
    }
    c->q_pos0[0] = q_pos0a;
    c->q_pos0[1] = q_pos0b;
    c->q_split = q_split;
    c->causal = causal;
    c->scale = scale;
    c->stream = stream;
    c->step = step;
    c->out_f32 = out_f32;
    c->dk = std::move(dk);
    c->dv = std::move(dv);
    if (rope.has_value()) {
        require_rope(*rope, q);
        c->rope = *rope;
    }
    return ChunksNode::apply(q, at::TensorList(kv), c);
}

// The exchange of a rank-stacked tensor x [W, *shard]: out[i] = cat_j(split(x[j], scatter)[i], gather) for every rank i at once, as one
// pass over the data.
Tensor exchange(const Tensor &x0, int64_t scatter, int64_t gather, int64_t W, int64_t stream) {
    const Tensor x = x0.resolve_conj().resolve_neg();   // the bytes that are copied have to be the values (a gradient may come as a conjugated view)
    const int64_t nd = x.dim() - 1, chunk = x.size(scatter + 1) / W;
    std::vector<int64_t> size{W}, stride{chunk * x.stride(scatter + 1)}, out_size{W};
    for (int64_t i = 0; i < nd; i++) {
        if (i == gather) size.push_back(W), stride.push_back(x.stride(0));
        size.push_back(i == scatter ? chunk : x.size(i + 1));
        stride.push_back(x.stride(i + 1));
        out_size.push_back((i == scatter ? chunk : x.size(i + 1)) * (i == gather ? W : 1));
    }
    // neighbouring dimensions that are one run in memory are one dimension
    std::vector<int64_t> cs, ct;
    for (size_t i = 0; i < size.size(); i++) {
        if (size[i] == 1) continue;
        if (!cs.empty() && ct.back() == size[i] * stride[i]) cs.back() *= size[i], ct.back() = stride[i];
        else cs.push_back(size[i]), ct.push_back(stride[i]);
    }
    const int64_t e = x.element_size();
    Tensor out = torch::empty(out_size, x.options());
    if (x.numel() == 0) return out;
    ltr_copy_args a{};
    bool fits = !cs.empty() && ct.back() == 1 && cs.back() * e % 16 == 0 && (int64_t)cs.size() - 1 <= LTR_COPY_DIMS && x.numel() * e / 16 < 0x7fff0000LL &&
                ((uintptr_t)x.data_ptr() | (uintptr_t)out.data_ptr()) % 16 == 0;
    for (size_t i = 0; fits && i + 1 < cs.size(); i++) {
        a.size[i] = cs[i];
        a.stride_bytes[i] = ct[i] * e;
        fits = a.stride_bytes[i] % 16 == 0;
    }
    if (!fits) return x.as_strided(size, stride).reshape(out_size).contiguous();
    const c10::DeviceGuard on_x_device(x.device());
    a.src = x.data_ptr();
    a.dst = out.data_ptr();
    a.n_outer = (int32_t)cs.size() - 1;
    a.run_bytes = cs.back() * e;
    check_rc(ltr_copy_strided(&a, (void *)stream), "ltr_copy_strided");
    return out;
}

struct ExchangeNode : torch::autograd::Function<ExchangeNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, int64_t scatter, int64_t gather, int64_t W, int64_t stream) {
        ctx->saved_data["dims"] = std::vector<int64_t>{scatter, gather, W, stream};
        return exchange(x, scatter, gather, W, stream);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {   // the exchange with the two dims swapped
        const auto d = ctx->saved_data["dims"].toIntVector();
        return {ExchangeNode::apply(grads[0], d[1], d[0], d[2], d[3]), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

Tensor seq_all_to_all(const Tensor &x, int64_t scatter, int64_t gather, int64_t W, int64_t stream) {
    const int64_t nd = x.dim() - 1;
    TORCH_CHECK(x.is_cuda() && nd > 0 && W > 0 && scatter >= 0 && scatter < nd && gather >= 0 && gather < nd && x.size(0) == W && x.size(scatter + 1) % W == 0,
                "a rank-stacked GPU tensor whose scattered dim divides by the number of ranks");
    return ExchangeNode::apply(x, scatter, gather, W, stream);
}

// RoPE of one [B, S, H, D] tensor (ltr_rope_apply); its gradient is the rotation by the conjugate angles.
Tensor rope_pass(const Tensor &x0, const Tensor &table, bool conj, int64_t stream) {
    const Tensor x = x0.stride(3) == 1 ? x0 : x0.contiguous();
    const c10::DeviceGuard on_x_device(x.device());
    Tensor out = torch::empty(x.sizes(), x.options());
    ltr_rope_args a{};
    a.x = x.data_ptr();
    a.out = out.data_ptr();
    a.freqs = table.data_ptr<float>();
    a.B = (int32_t)x.size(0);
    a.S = x.size(1);
    a.H = (int32_t)x.size(2);
    a.D = (int32_t)x.size(3);
    strides3(x, a.x_stride);
    strides3(out, a.out_stride);
    a.flags = conj ? LTR_ROPE_CONJ : 0u;
    a.io_dtype = x.scalar_type() == at::kBFloat16 ? LTR_BF16 : LTR_F32;
    check_rc(ltr_rope_apply(&a, (void *)stream), "ltr_rope_apply");
    return out;
}

struct RopeNode : torch::autograd::Function<RopeNode> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &table, int64_t stream) {
        ctx->save_for_backward({table});
        ctx->saved_data["stream"] = stream;
        return rope_pass(x, table, false, stream);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        return {rope_pass(grads[0], ctx->get_saved_variables()[0], true, ctx->saved_data["stream"].toInt()), Tensor(), Tensor()};
    }
};

// table: fp32 [S, D/2, 2] (cos, sin) rows of x's sequence indices
Tensor rope(const Tensor &x, const Tensor &table, int64_t stream) {
    TORCH_CHECK(x.is_cuda() && x.dim() == 4 && (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat), "x must be a bf16 or fp32 [B,S,H,D] GPU tensor");
    TORCH_CHECK(table.scalar_type() == at::kFloat && table.is_contiguous() && table.dim() == 3 && table.size(0) == x.size(1) && table.size(1) == x.size(3) / 2 &&
                    table.size(2) == 2 && table.device() == x.device(),
                "the RoPE table must be a contiguous fp32 [S, D/2, 2] (cos, sin) tensor on x's device");
    return RopeNode::apply(x, table, stream);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("single_chunk", &single_chunk, "one bf16 KV chunk, forward with a C++ autograd node behind it");
    m.def("chunks", &chunks, "a table of KV chunks, forward with a C++ autograd node behind it");
    m.def("rope", &rope, "rotary position embedding of one tensor, differentiable");
    m.def("seq_all_to_all", &seq_all_to_all, "the exchange of a rank-stacked tensor, differentiable");
    m.def("exchange", [](const Tensor &x, int64_t s, int64_t g, int64_t W, int64_t stream) { return exchange(x, s, g, W, stream); }, "its data movement");
    m.def("abi_version", []() { return ltr_abi_version(); });
}
