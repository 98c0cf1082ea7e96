// PyTorch-ROCm extension over the C ABI of libmhc_hip.so: allocates outputs, passes raw device
// pointers and torch's current HIP stream, and implements the autograd functions in C++.
//
// Counterpart of the reference's pybind module `mhc_cuda` (src/python/bindings.cu:544-554) and of
// the autograd classes of src/python/mhc/ops.py:13-417.  No torch type crosses into the library:
// every mhc_* call below is the C ABI of include/mhc_hip.h.
#include <torch/extension.h>

#include <ATen/FuncTorchTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <array>
#include <mutex>
#include <unordered_map>

#include "../../include/mhc_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using OptTensor = c10::optional<Tensor>;

struct MhcError : std::runtime_error {
    std::string fn;
    int status;
    MhcError(const char *f, int s)
        : std::runtime_error(std::string(f) + " failed: " + mhc_status_string(s) + " (status " + std::to_string(s) + ")"),
          fn(f), status(s) {}
};

inline void check(const char *fn, int status) {
    if (status != MHC_OK) throw MhcError(fn, status);
}

inline int dt(const Tensor &t) {
    if (t.scalar_type() == at::kFloat) return MHC_F32;
    if (t.scalar_type() == at::kBFloat16) return MHC_BF16;
    TORCH_CHECK(false, "mhc: unsupported dtype ", t.scalar_type(), ": the HIP library takes float32 or bfloat16");
}
inline bool is_act(at::ScalarType st) { return st == at::kFloat || st == at::kBFloat16; }
inline bool is_act_dtype(const Tensor &t) { return is_act(t.scalar_type()); }

inline void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

inline void require_gpu(const Tensor &t) {
    if (!t.defined()) return;
    TORCH_CHECK(t.is_cuda(), "mhc: tensors must live on a HIP (cuda) device; there is no CPU path");
}

// contiguous, on the device, and with a 16-byte aligned base (a contiguous view at an odd offset is copied)
inline Tensor act(const Tensor &t) {
    require_gpu(t);
    Tensor c = t.contiguous();
    if ((reinterpret_cast<uintptr_t>(c.data_ptr()) & 15u) != 0) c = c.clone();
    return c;
}
inline Tensor f32c(const Tensor &t) {
    require_gpu(t);
    return (t.scalar_type() == at::kFloat ? t : t.to(at::kFloat)).contiguous();
}

inline void *stream_of(const Tensor &t) {
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Scratch memory per (device, stream), grown on demand and held while a call enqueues its launches: on the stream
// the calls are then ordered one after the other, each with the memory to itself.  Two host threads that use one
// stream (a forward beside the backward of another thread, which the engine runs on the forward's stream) would
// otherwise enqueue their launches in between each other's.
struct Scratch {
    Tensor retired;  // a smaller buffer that this call replaced; released after the lock
    std::unique_lock<std::mutex> held;
    char *ptr;
    size_t bytes;
};

Scratch scratch(const Tensor &like, size_t nbytes) {
    struct Slot {
        std::mutex mu;
        Tensor buf;
    };
    static std::mutex mu;
    static std::unordered_map<uint64_t, Slot> slots;  // (references to its elements stay valid)
    const uint64_t key = (static_cast<uint64_t>(like.device().index()) << 56) ^
                         reinterpret_cast<uint64_t>(stream_of(like));
    Slot *slot;
    {
        std::lock_guard<std::mutex> lock(mu);
        slot = &slots[key];
    }
    // While a slot is held nothing but library calls may run (no tensor is made, converted or freed): torch may ask
    // for the interpreter's lock there, which a thread that waits for the slot holds.
    Tensor buf;
    std::unique_lock<std::mutex> held(slot->mu);
    while (!slot->buf.defined() || static_cast<size_t>(slot->buf.numel()) < nbytes) {
        held.unlock();
        buf = at::empty({static_cast<int64_t>(std::max<size_t>(nbytes, 1 << 20))}, like.options().dtype(at::kByte));
        held.lock();
        if (!slot->buf.defined() || slot->buf.numel() < buf.numel()) std::swap(slot->buf, buf);
    }
    char *p = static_cast<char *>(slot->buf.data_ptr());
    const size_t n = static_cast<size_t>(slot->buf.numel());
    return Scratch{std::move(buf), std::move(held), p, n};
}

// ---------------------------------------------------------------------------------------------
// what the two autograd nodes share
//
// A forward + backward of a small layer is bound by the host, so the two layers are autograd nodes of
// their own (torch::autograd::Node) instead of torch::autograd::Function: no string-keyed dictionary of
// saved values, no generic argument extraction and output wrapping; everything a call keeps sits in ONE
// byte buffer, dphi in another and the small parameter gradients in a third, and the gradients handed back are
// tensors built directly over those buffers' storage (nine narrow / select / reshape calls through the dispatcher cost
// more than the backward's kernel launches).  B=320 C=1280 n=4, same box: forward + backward 126 -> 105 us;
// B=7 forward without gradients 19.8 -> 14.3 us.  Where the host's time of a step goes (B=8 n=4 C=256, 67 us with
// nothing to wait for on the device): the forward call 11, the backward call about 8, the engine's hand-over to
// its device thread and back about 16, and 3.2 for each of the ten parameter leaves.
// ---------------------------------------------------------------------------------------------
inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

inline Tensor byte_buffer(const Tensor &like, size_t bytes) {
    return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
}

// A contiguous tensor over part of `base`'s storage (base at offset 0, byte_off a multiple of the element size).
Tensor over(const Tensor &base, at::ScalarType st, size_t byte_off, at::IntArrayRef sizes) {
    Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(base.storage()), base.key_set(),
                                                        c10::scalarTypeToTypeMeta(st));
    c10::TensorImpl *impl = t.unsafeGetTensorImpl();
    impl->set_storage_offset((int64_t)(byte_off / c10::elementSize(st)));
    impl->set_sizes_contiguous(sizes);
    return t;
}

inline Tensor cast_to(Tensor t, at::ScalarType st) { return t.scalar_type() == st ? t : t.to(st); }

// What torch::autograd::Function refuses by itself and a node of one's own does not: the function transforms
// (vmap, grad, jvp ... of torch.func), whose wrapped tensors no kernel can read, and forward mode.
inline void refuse_transforms(std::initializer_list<const Tensor *> inputs) {
    if (const auto &tls = at::functorch::functorchTLSAccessor()) tls->checkSupportsCppAutogradFunction();
    // outside a dual level no tensor has a tangent (asking all of them costs a lock each, 1.5 us a call)
    if (!torch::autograd::ForwardADLevel::try_get_by_idx(0)) return;
    for (const Tensor *t : inputs)
        TORCH_CHECK(!t->defined() || !t->_fw_grad(0).defined(), "mhc: forward-mode differentiation is not implemented");
}

inline const Tensor &optional_tensor(const OptTensor &t) {
    static const Tensor none;
    return t.has_value() ? *t : none;
}

// The incoming gradient as the kernels take it.  bfloat16 activations with a float32 result hand back a
// float32 gradient: it is rounded to the activations' format here, so that the backward runs the kernels
// that take both in 2 bytes (the mixed pair goes through slower general kernels: 111 against 20 us for dx
// at B=128 n=32 C=1280).  One pass also when the gradient arrives as a broadcast view (the backward of a sum).
Tensor incoming_gradient(const Tensor &g, const Tensor &x, at::ScalarType y_type) {
    if (!g.defined()) return at::zeros(x.sizes(), x.options().dtype(x.scalar_type() == at::kBFloat16 ? at::kBFloat16 : y_type));
    const bool round_dy = x.scalar_type() == at::kBFloat16 && g.scalar_type() == at::kFloat;
    return act(round_dy ? g.to(g.options().dtype(at::kBFloat16), false, false, at::MemoryFormat::Contiguous) : g);
}

// A saved tensor as the backward takes it; what a hook of torch.autograd.graph.saved_tensors_hooks handed back has to be
// of the type and size that was saved.
inline Tensor unpacked(const SavedVariable &v, at::ScalarType st, int64_t numel) {
    const Tensor t = act(v.unpack());
    TORCH_CHECK(t.scalar_type() == st && t.numel() >= numel,
                "mhc: a saved-tensor hook changed the type or the size of a tensor saved for the backward");
    return t;
}

template <typename N> std::shared_ptr<N> make_node(torch::autograd::edge_list &&edges) {
    std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
    node->set_next_edges(std::move(edges));
    return node;
}

// ---------------------------------------------------------------------------------------------
// parameter packing (dynamic H): phi [D, nC] in the compute dtype, [bias (D) | alpha (3)] in fp32
// ---------------------------------------------------------------------------------------------
struct DynParams {
    const Tensor *src[9];  // phi_pre, phi_post, phi_res, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res
};

// the parameters as the library takes them: device, dtype and shape checked; m keeps converted copies alive
struct mhc_dynamic_params library_params(const DynParams &p, int n, int C, Tensor (&m)[9]) {
    // the three phi matrices in one source dtype the kernels read (float32 or bfloat16)
    const bool same_dt = p.src[0]->scalar_type() == p.src[1]->scalar_type() && p.src[0]->scalar_type() == p.src[2]->scalar_type() &&
                         is_act_dtype(*p.src[0]);
    for (int i = 0; i < 9; i++) {
        require_gpu(*p.src[i]);
        m[i] = i < 3 && same_dt ? p.src[i]->contiguous() : f32c(*p.src[i]);
    }
    TORCH_CHECK(m[0].numel() == (int64_t)n * n * C && m[1].numel() == m[0].numel() && m[2].numel() == (int64_t)n * n * n * C,
                "mhc: phi shapes do not match expansion rate ", n, " and hidden size ", C);
    TORCH_CHECK(m[6].numel() == n && m[7].numel() == n && m[8].numel() == n * n, "mhc: bias shapes do not match n = ", n);
    return {ptr(m[0]), ptr(m[1]), ptr(m[2]), dt(m[0]), m[6].data_ptr<float>(), m[7].data_ptr<float>(), m[8].data_ptr<float>(),
            m[3].data_ptr<float>(), m[4].data_ptr<float>(), m[5].data_ptr<float>()};
}

bool g_param_cache = false;

struct Packed {
    Tensor phi, ba;
};

// The opt-in cache of packed parameters.  An entry is valid while the very same tensor objects are alive
// (weak references: a new tensor that happens to reuse the address of a freed one never matches) and their
// storage addresses and in-place version counters are unchanged.
struct CacheEntry {
    std::vector<c10::weak_intrusive_ptr<c10::TensorImpl>> impl;
    void *ptrs[9];
    uint32_t versions[9];
    int cd;
    Packed packed;
};

Packed cached_params(const DynParams &p, const Tensor &x, int n, int C, int cd) {
    static std::mutex mu;
    static std::unordered_map<void *, CacheEntry> cache;
    {
        std::lock_guard<std::mutex> lock(mu);
        auto it = cache.find(p.src[0]->data_ptr());
        if (it != cache.end() && it->second.cd == cd) {
            bool same = true;
            for (int i = 0; i < 9; i++)
                same = same && !it->second.impl[i].expired() &&
                       it->second.impl[i]._unsafe_get_target() == p.src[i]->unsafeGetTensorImpl() &&
                       it->second.ptrs[i] == p.src[i]->data_ptr() && it->second.versions[i] == p.src[i]->_version();
            if (same) return it->second.packed;
        }
    }
    const int D = n * n + 2 * n;
    Packed out;
    out.phi = at::empty({D, (int64_t)n * C}, x.options().dtype(cd == MHC_BF16 ? at::kBFloat16 : at::kFloat));
    out.ba = at::empty({D + 3}, x.options().dtype(at::kFloat));
    Tensor m[9];
    const struct mhc_dynamic_params lp = library_params(p, n, C, m);
    float *ba = out.ba.data_ptr<float>();
    check("mhc_pack_dynamic_params",
          mhc_pack_dynamic_params(lp.phi_pre, lp.phi_post, lp.phi_res, lp.phi_dtype, lp.b_pre, lp.b_post, lp.b_res, lp.alpha_pre,
                                  lp.alpha_post, lp.alpha_res, out.phi.data_ptr(), cd, ba, ba + D, n, C, stream_of(x)));
    std::lock_guard<std::mutex> lock(mu);
    if (cache.size() >= 4096) cache.clear();
    CacheEntry e;
    for (int i = 0; i < 9; i++) {
        e.impl.emplace_back(p.src[i]->getIntrusivePtr());
        e.ptrs[i] = p.src[i]->data_ptr();
        e.versions[i] = p.src[i]->_version();
    }
    e.cd = cd;
    e.packed = out;
    cache.erase(p.src[0]->data_ptr());
    cache.emplace(p.src[0]->data_ptr(), std::move(e));
    return out;
}

// ---------------------------------------------------------------------------------------------
// dynamic-H layer (reference ops.py:154-417, bindings.cu:405-542)
// ---------------------------------------------------------------------------------------------
// What a call keeps, in one byte buffer: fp32 Hpre | Hpost | M | P | r | q | Sinkhorn state, then the packed
// [bias | alpha] and phi (each at a multiple of 256 bytes) unless those come from the parameter cache.
struct DynLayout {
    int B, n, C, D;
    size_t state, ba, phi, bytes;  // floats of state; byte offsets
    DynLayout(int B_, int n_, int C_, int iters, bool for_backward, int cd, bool packed_here)
        : B(B_), n(n_), C(C_), D(n_ * n_ + 2 * n_) {
        // the Sinkhorn denominators are only worth writing when a backward call will read them
        state = for_backward ? mhc_layer_sinkhorn_state_floats(B, n, iters) : 0;
        ba = align256(((size_t)B * (2 * n + n * n + D + 2) + state) * 4);
        phi = ba + (packed_here ? align256((size_t)(D + 3) * 4) : 0);
        bytes = phi + (packed_here ? (size_t)D * n * C * (cd == MHC_BF16 ? 2 : 4) : 0);
    }
};

struct DynViews {
    float *Hp, *Ho, *M, *P, *r, *q, *sk, *ba;
    void *phi;
    DynViews(char *b, const DynLayout &l) {
        const size_t B = l.B, n = l.n;
        Hp = reinterpret_cast<float *>(b);
        Ho = Hp + B * n; M = Ho + B * n; P = M + B * n * n; r = P + B * l.D; q = r + B;
        sk = l.state ? q + B : nullptr;
        ba = reinterpret_cast<float *>(b + l.ba);
        phi = b + l.phi;
    }
};

struct MHCDynamicBackward final : public torch::autograd::Node {
    SavedVariable x_, w_, f_, kept_, phi_, ba_;  // phi_, ba_: only with the parameter cache
    bool has_w = false, has_f = false, cached = false, released = false;
    std::array<int64_t, 3> shape;  // of x
    int iters = 0, x_code = 0, cd = 0;
    double eps = 0.0;
    at::ScalarType x_type, w_type, f_type, y_type, p_type[9];
    std::vector<int64_t> b_res_sizes;

    std::string name() const override { return "MHCLayerDynamicBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data(); w_.reset_data(); f_.reset_data(); kept_.reset_data(); phi_.reset_data(); ba_.reset_data();
        released = true;
    }

    // edges: x, w, f_inject, then the nine parameters in the order of DynParams
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
        const at::ScalarType act_type = x_code == MHC_BF16 ? at::kBFloat16 : at::kFloat;
        const int B = (int)shape[0], n = (int)shape[1], C = (int)shape[2], D = n * n + 2 * n;
        const int64_t nC = (int64_t)n * C;
        const DynLayout l(B, n, C, iters, true, cd, !cached);
        const Tensor x = unpacked(x_, act_type, B * nC), kept = unpacked(kept_, at::kByte, (int64_t)l.bytes);
        const Tensor w = has_w ? unpacked(w_, is_act(w_type) ? w_type : at::kFloat, C) : Tensor();
        const Tensor f = has_f ? unpacked(f_, act_type, (int64_t)B * C) : Tensor();
        const Tensor phi_c = cached ? unpacked(phi_, cd == MHC_BF16 ? at::kBFloat16 : at::kFloat, D * nC) : Tensor();
        const Tensor ba_c = cached ? unpacked(ba_, at::kFloat, D + 3) : Tensor();
        at::AutoDispatchBelowADInplaceOrView below;
        c10::DeviceGuard guard(x.device());
        DynViews v(static_cast<char *>(kept.data_ptr()), l);
        if (cached) { v.phi = phi_c.data_ptr(); v.ba = ba_c.data_ptr<float>(); }
        const Tensor dy = incoming_gradient(grads[0], x, y_type);
        Tensor dx = at::empty(shape, x.options());
        Tensor df = has_f ? at::empty(f.sizes(), f.options()) : Tensor();
        // dphi [D, nC], fp32; in a buffer of their own, so that keeping one of them does not keep dphi, the small ones:
        // dbias [D] dalpha [3], fp32 | dw [C] in the weight's type where the library writes it
        const at::ScalarType dw_type = w_type == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
        Tensor g = at::empty({D, nC}, x.options().dtype(at::kFloat));
        const size_t off_w = align256((size_t)(D + 3) * 4);
        Tensor gs = byte_buffer(x, off_w + (size_t)C * 4);
        char *gp = static_cast<char *>(gs.data_ptr());
        float *dphi = g.data_ptr<float>(), *dba = reinterpret_cast<float *>(gp);
        Scratch ws = scratch(x, mhc_layer_dynamic_workspace_bytes(B, n, C));
        check("mhc_layer_bwd_dynamic",
              mhc_layer_bwd_dynamic_dw(ptr(dy), dt(dy), ptr(x), x_code, ptr(w), has_w ? dt(w) : 0, v.phi, cd, v.ba, v.ba + D, ptr(f),
                                    v.Hp, v.Ho, v.M, v.P, v.r, v.q, v.sk, ptr(dx), ptr(df),
                                    has_f ? nullptr : gp + off_w, dw_type == at::kBFloat16 ? MHC_BF16 : MHC_F32, dphi, dba, dba + D, B, n, C, iters,
                                    (float)eps, ws.ptr, ws.bytes, stream_of(x)));
        ws.held.unlock();
        variable_list out(12);
        if (task_should_compute_output(0)) out[0] = cast_to(dx, x_type);
        if (has_w && !has_f && task_should_compute_output(1)) out[1] = cast_to(over(gs, dw_type, off_w, {C}), w_type);
        if (has_f && task_should_compute_output(2)) out[2] = cast_to(df, f_type);
        const int64_t rows[3] = {n, n, (int64_t)n * n}, row0[3] = {0, n, 2 * n};
        for (int i = 0; i < 3; i++) {
            if (task_should_compute_output(3 + i))
                out[3 + i] = cast_to(over(g, at::kFloat, (size_t)row0[i] * nC * 4, {rows[i], nC}), p_type[i]);
            if (task_should_compute_output(6 + i)) out[6 + i] = cast_to(over(gs, at::kFloat, (size_t)(D + i) * 4, {}), p_type[3 + i]);
            if (task_should_compute_output(9 + i)) {
                const at::IntArrayRef sizes = i < 2 ? at::IntArrayRef(rows[i]) : at::IntArrayRef(b_res_sizes);
                out[9 + i] = cast_to(over(gs, at::kFloat, (size_t)row0[i] * 4, sizes), p_type[6 + i]);
            }
        }
        return out;
    }
};

Tensor mhc_layer_dynamic(const Tensor &x_in, const OptTensor &w_opt, const Tensor &phi_pre, const Tensor &phi_post,
                         const Tensor &phi_res, const Tensor &alpha_pre, const Tensor &alpha_post, const Tensor &alpha_res,
                         const Tensor &b_pre, const Tensor &b_post, const Tensor &b_res, int64_t iters, double eps,
                         c10::optional<at::ScalarType> out_dtype, const OptTensor &f_opt, bool compute_bf16) {
    TORCH_CHECK(x_in.dim() == 3, "mhc: x must be [B, n, C]");
    const Tensor &w_in = optional_tensor(w_opt), &f_in = optional_tensor(f_opt);
    refuse_transforms({&x_in, &w_in, &f_in, &phi_pre, &phi_post, &phi_res, &alpha_pre, &alpha_post, &alpha_res, &b_pre, &b_post, &b_res});
    const bool record = torch::autograd::compute_requires_grad(x_in, w_in, f_in, phi_pre, phi_post, phi_res, alpha_pre,
                                                               alpha_post, alpha_res, b_pre, b_post, b_res);
    std::shared_ptr<MHCDynamicBackward> node;
    if (record)
        node = make_node<MHCDynamicBackward>(torch::autograd::collect_next_edges(
            x_in, w_in, f_in, phi_pre, phi_post, phi_res, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res));
    const at::ScalarType y_type = out_dtype.value_or(at::kFloat);
    const bool cached = g_param_cache;
    Tensor y, x, w, f, kept;
    Packed pk;
    int x_code = 0, cd = 0;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        // compute_bf16 with float32 activations (the reference's default contract: float32 in and out
        // around a bf16 kernel path): where the library's kernels load fp32 storage themselves, x is
        // handed over as it is and rounded in registers; elsewhere it is cast here, as the reference
        // casts it (bindings.cu:421-423)
        x = act(is_act_dtype(x_in) ? x_in : x_in.to(at::kFloat));
        const int B = x.size(0), n = x.size(1), C = x.size(2), D = n * n + 2 * n;
        c10::DeviceGuard guard(x.device());
        x_code = dt(x);
        if (compute_bf16 && x_code == MHC_F32) {
            if (y_type == at::kFloat && mhc_layer_dynamic_accepts_f32_as_bf16(B, n, C, (int)iters))
                x_code = MHC_F32_AS_BF16;
            else {
                x = x.to(at::kBFloat16);
                x_code = MHC_BF16;
            }
        }
        if (w_in.defined()) w = act(is_act_dtype(w_in) ? w_in : w_in.to(at::kFloat));
        if (f_in.defined()) f = act(f_in.to(x.scalar_type()));
        cd = x_code == MHC_F32 ? MHC_F32 : MHC_BF16;
        const DynParams params{{&phi_pre, &phi_post, &phi_res, &alpha_pre, &alpha_post, &alpha_res, &b_pre, &b_post, &b_res}};
        if (cached) pk = cached_params(params, x, n, C, cd);
        y = at::empty({B, n, C}, x.options().dtype(y_type));
        const DynLayout l(B, n, C, (int)iters, record, cd, !cached);
        // Without a backward nothing of it outlives the call: a small one lies behind the workspace then, one allocation
        // less.  It pays where the host bounds the call (n=4 C=1280, phi 0.25 MB: B=7 10.72 us against 11.17 with a buffer
        // of its own, B=200 10.76 against 11.15); from 0.8 MB of phi on the device does (n=4 C=4096 12.68 against 12.56,
        // n=8 C=1280 14.94 against 14.91), and the workspace, which is held on to, need not grow for it.
        const bool own = record || l.bytes > ((size_t)512 << 10);
        const size_t ws_bytes = align256(mhc_layer_dynamic_workspace_bytes(B, n, C));
        if (own) kept = byte_buffer(x, l.bytes);
        Tensor m[9];
        struct mhc_dynamic_params lp;
        if (!cached) lp = library_params(params, n, C, m);
        const int w_dt = w.defined() ? dt(w) : 0, y_dt = dt(y);
        const Scratch ws = scratch(x, ws_bytes + (own ? 0 : l.bytes));
        DynViews v(own ? static_cast<char *>(kept.data_ptr()) : ws.ptr + ws_bytes, l);
        if (cached) {
            v.phi = pk.phi.data_ptr();
            v.ba = pk.ba.data_ptr<float>();
            check("mhc_layer_fwd_dynamic",
                  mhc_layer_fwd_dynamic(ptr(x), x_code, ptr(w), w_dt, v.phi, cd, v.ba, v.ba + D, ptr(f), ptr(y), y_dt, v.Hp, v.Ho,
                                        v.M, v.P, v.r, v.q, v.sk, B, n, C, (int)iters, (float)eps, ws.ptr, ws_bytes,
                                        stream_of(x)));
        } else {
            check("mhc_layer_fwd_dynamic",
                  mhc_layer_fwd_dynamic_params(ptr(x), x_code, ptr(w), w_dt, &lp, v.phi, cd, v.ba, v.ba + D, ptr(f), ptr(y), y_dt,
                                               v.Hp, v.Ho, v.M, v.P, v.r, v.q, v.sk, B, n, C, (int)iters, (float)eps,
                                               ws.ptr, ws_bytes, stream_of(x)));
        }
    }
    if (record) {
        // outside the guard: the hooks of torch.autograd.graph.saved_tensors_hooks run here and are user code
        node->x_ = SavedVariable(x, false);
        node->kept_ = SavedVariable(kept, false);
        if ((node->has_w = w.defined())) node->w_ = SavedVariable(w, false);
        if ((node->has_f = f.defined())) node->f_ = SavedVariable(f, false);
        if ((node->cached = cached)) {
            node->phi_ = SavedVariable(pk.phi, false);
            node->ba_ = SavedVariable(pk.ba, false);
        }
        node->iters = (int)iters;
        node->eps = eps;
        node->x_code = x_code;
        node->cd = cd;
        node->shape = {x.size(0), x.size(1), x.size(2)};
        node->x_type = x_in.scalar_type();
        node->y_type = y_type;
        node->w_type = w_in.defined() ? w_in.scalar_type() : at::kFloat;
        node->f_type = f_in.defined() ? f_in.scalar_type() : at::kFloat;
        const Tensor *src[9] = {&phi_pre, &phi_post, &phi_res, &alpha_pre, &alpha_post, &alpha_res, &b_pre, &b_post, &b_res};
        for (int i = 0; i < 9; i++) node->p_type[i] = src[i]->scalar_type();
        node->b_res_sizes = b_res.sizes().vec();
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------
// static-H layer (reference ops.py:55-151, bindings.cu:221-401)
// ---------------------------------------------------------------------------------------------
struct MHCStaticBackward final : public torch::autograd::Node {
    SavedVariable x_, w_, f_, hp_, ho_, hr_, kept_;  // kept: fp32 Hpre | Hpost | M | q
    bool has_w = false, has_f = false, released = false;
    int iters = 0;
    double eps = 0.0;
    at::ScalarType x_type, act_type, w_type, f_type, y_type, h_type[3];  // act_type: of the saved x
    std::array<int64_t, 3> shape;                                         // of x
    std::vector<int64_t> h_res_sizes;

    std::string name() const override { return "MHCLayerStaticBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data(); w_.reset_data(); f_.reset_data(); hp_.reset_data(); ho_.reset_data(); hr_.reset_data(); kept_.reset_data();
        released = true;
    }

    // edges: x, w, f_inject, H_pre, H_post, H_res
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
        const int B = (int)shape[0], n = (int)shape[1], C = (int)shape[2];
        const Tensor x = unpacked(x_, act_type, (int64_t)B * n * C), kept = unpacked(kept_, at::kFloat, 2 * n + n * n + B);
        const Tensor hp = unpacked(hp_, at::kFloat, n), ho = unpacked(ho_, at::kFloat, n), hr = unpacked(hr_, at::kFloat, n * n);
        const Tensor w = has_w ? unpacked(w_, is_act(w_type) ? w_type : at::kFloat, C) : Tensor();
        const Tensor f = has_f ? unpacked(f_, act_type, (int64_t)B * C) : Tensor();
        at::AutoDispatchBelowADInplaceOrView below;
        c10::DeviceGuard guard(x.device());
        const Tensor dy = incoming_gradient(grads[0], x, y_type);
        Tensor dx = at::empty(shape, x.options());
        Tensor df = has_f ? at::empty(f.sizes(), f.options()) : Tensor();
        // dH_pre | dH_post | dH_res, fp32 | dw [C] in the weight's type where the library writes it
        const at::ScalarType dw_type = w_type == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
        const size_t off_w = align256((size_t)(2 * n + n * n) * 4);
        Tensor g = byte_buffer(x, off_w + (size_t)C * 4);
        float *d = static_cast<float *>(g.data_ptr()), *s = kept.data_ptr<float>();
        Scratch ws = scratch(x, mhc_layer_static_workspace_bytes(B, n, C));
        check("mhc_layer_bwd",
              mhc_layer_bwd_dw(ptr(dy), dt(dy), ptr(x), dt(x), ptr(w), has_w ? dt(w) : 0, hp.data_ptr<float>(), ho.data_ptr<float>(),
                            hr.data_ptr<float>(), ptr(f), s, s + n, s + 2 * n, s + 2 * n + n * n, ptr(dx), ptr(df),
                            has_f ? nullptr : d + off_w / 4, dw_type == at::kBFloat16 ? MHC_BF16 : MHC_F32, d, d + n, d + 2 * n, B, n, C, iters, (float)eps, ws.ptr,
                            ws.bytes, stream_of(x)));
        ws.held.unlock();
        variable_list out(6);
        if (task_should_compute_output(0)) out[0] = cast_to(dx, x_type);
        if (has_w && !has_f && task_should_compute_output(1)) out[1] = cast_to(over(g, dw_type, off_w, {C}), w_type);
        if (has_f && task_should_compute_output(2)) out[2] = cast_to(df, f_type);
        if (task_should_compute_output(3)) out[3] = cast_to(over(g, at::kFloat, 0, {n}), h_type[0]);
        if (task_should_compute_output(4)) out[4] = cast_to(over(g, at::kFloat, (size_t)n * 4, {n}), h_type[1]);
        if (task_should_compute_output(5)) out[5] = cast_to(over(g, at::kFloat, (size_t)n * 8, h_res_sizes), h_type[2]);
        return out;
    }
};

Tensor mhc_layer_static(const Tensor &x_in, const OptTensor &w_opt, const Tensor &H_pre, const Tensor &H_post,
                        const Tensor &H_res, int64_t iters, double eps, c10::optional<at::ScalarType> out_dtype,
                        const OptTensor &f_opt) {
    TORCH_CHECK(x_in.dim() == 3, "mhc: x must be [B, n, C]");
    const Tensor &w_in = optional_tensor(w_opt), &f_in = optional_tensor(f_opt);
    refuse_transforms({&x_in, &w_in, &f_in, &H_pre, &H_post, &H_res});
    const bool record = torch::autograd::compute_requires_grad(x_in, w_in, f_in, H_pre, H_post, H_res);
    std::shared_ptr<MHCStaticBackward> node;
    if (record)
        node = make_node<MHCStaticBackward>(torch::autograd::collect_next_edges(x_in, w_in, f_in, H_pre, H_post, H_res));
    const at::ScalarType y_type = out_dtype.value_or(at::kFloat);
    Tensor y, x, w, f, hp, ho, hr, kept;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        x = act(is_act_dtype(x_in) ? x_in : x_in.to(at::kFloat));
        const int B = x.size(0), n = x.size(1), C = x.size(2);
        c10::DeviceGuard guard(x.device());
        if (w_in.defined()) w = act(is_act_dtype(w_in) ? w_in : w_in.to(at::kFloat));
        if (f_in.defined()) f = act(f_in.to(x.scalar_type()));
        hp = f32c(H_pre); ho = f32c(H_post); hr = f32c(H_res);
        TORCH_CHECK(hp.numel() == n && ho.numel() == n && hr.numel() == n * n, "mhc: H shapes do not match n = ", n);
        y = at::empty({B, n, C}, x.options().dtype(y_type));
        kept = at::empty({2 * n + n * n + B}, x.options().dtype(at::kFloat));
        float *s = kept.data_ptr<float>();
        const Scratch ws = scratch(x, mhc_layer_static_workspace_bytes(B, n, C));
        check("mhc_layer_fwd",
              mhc_layer_fwd(ptr(x), dt(x), ptr(w), w.defined() ? dt(w) : 0, hp.data_ptr<float>(), ho.data_ptr<float>(),
                            hr.data_ptr<float>(), ptr(f), ptr(y), dt(y), s, s + n, s + 2 * n, s + 2 * n + n * n, B, n, C,
                            (int)iters, (float)eps, ws.ptr, ws.bytes, stream_of(x)));
    }
    if (record) {
        node->x_ = SavedVariable(x, false);
        node->kept_ = SavedVariable(kept, false);
        node->hp_ = SavedVariable(hp, false);
        node->ho_ = SavedVariable(ho, false);
        node->hr_ = SavedVariable(hr, false);
        if ((node->has_w = w.defined())) node->w_ = SavedVariable(w, false);
        if ((node->has_f = f.defined())) node->f_ = SavedVariable(f, false);
        node->iters = (int)iters;
        node->eps = eps;
        node->shape = {x.size(0), x.size(1), x.size(2)};
        node->x_type = x_in.scalar_type();
        node->act_type = x.scalar_type();
        node->y_type = y_type;
        node->w_type = w_in.defined() ? w_in.scalar_type() : at::kFloat;
        node->f_type = f_in.defined() ? f_in.scalar_type() : at::kFloat;
        node->h_type[0] = H_pre.scalar_type();
        node->h_type[1] = H_post.scalar_type();
        node->h_type[2] = H_res.scalar_type();
        node->h_res_sizes = H_res.sizes().vec();
        torch::autograd::set_history(y, node);
    }
    return y;
}

// forward only: nothing is kept for a backward pass (coefficients stay in the workspace)
Tensor mhc_layer_inference(const Tensor &x_in, const Tensor &w_in, const Tensor &H_pre, const Tensor &H_post,
                           const Tensor &H_res, int64_t iters, double eps, c10::optional<at::ScalarType> out_dtype) {
    const Tensor x = act(is_act_dtype(x_in) ? x_in : x_in.to(at::kFloat));
    const Tensor w = act(is_act_dtype(w_in) ? w_in : w_in.to(at::kFloat));
    const int B = x.size(0), n = x.size(1), C = x.size(2);
    c10::DeviceGuard guard(x.device());
    const Tensor hp = f32c(H_pre), ho = f32c(H_post), hr = f32c(H_res);
    Tensor y = at::empty({B, n, C}, x.options().dtype(out_dtype.value_or(at::kFloat)));
    const Scratch ws = scratch(x, mhc_layer_static_workspace_bytes(B, n, C));
    check("mhc_layer_fwd",
          mhc_layer_fwd(ptr(x), dt(x), ptr(w), dt(w), hp.data_ptr<float>(), ho.data_ptr<float>(), hr.data_ptr<float>(),
                        nullptr, ptr(y), dt(y), nullptr, nullptr, nullptr, nullptr, B, n, C, (int)iters, (float)eps,
                        ws.ptr, ws.bytes, stream_of(x)));
    return y;
}

// ---------------------------------------------------------------------------------------------
// stand-alone operators (reference ops.py:13-52, bindings.cu:115-164)
// ---------------------------------------------------------------------------------------------
struct SinkhornFn : public torch::autograd::Function<SinkhornFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &inp_in, int64_t iters, double eps) {
        const Tensor inp = f32c(inp_in);
        TORCH_CHECK(inp.dim() >= 2, "mhc: sinkhorn_knopp takes [..., rows, cols]");
        c10::DeviceGuard guard(inp.device());
        const int rows = inp.size(-2), cols = inp.size(-1);
        const int batch = (int)(inp.numel() / ((int64_t)rows * cols));
        Tensor out = at::empty_like(inp);
        check("mhc_sinkhorn_knopp_fwd", mhc_sinkhorn_knopp_fwd(inp.data_ptr<float>(), out.data_ptr<float>(), batch, rows,
                                                                cols, (int)iters, (float)eps, stream_of(inp)));
        ctx->save_for_backward({inp});
        ctx->saved_data["iters"] = iters;
        ctx->saved_data["eps"] = eps;
        ctx->saved_data["dtype"] = (int64_t)inp_in.scalar_type();
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const Tensor inp = ctx->get_saved_variables()[0];
        c10::DeviceGuard guard(inp.device());
        const Tensor go = f32c(grads[0]);
        const int rows = inp.size(-2), cols = inp.size(-1);
        const int batch = (int)(inp.numel() / ((int64_t)rows * cols));
        const int iters = (int)ctx->saved_data["iters"].toInt();
        const double eps = ctx->saved_data["eps"].toDouble();
        const auto sd = (at::ScalarType)ctx->saved_data["dtype"].toInt();
        Tensor d_inp = at::empty_like(inp);
        Scratch ws = scratch(inp, mhc_sinkhorn_knopp_bwd_workspace_bytes(batch, rows, cols, iters));
        check("mhc_sinkhorn_knopp_bwd",
              mhc_sinkhorn_knopp_bwd(go.data_ptr<float>(), inp.data_ptr<float>(), d_inp.data_ptr<float>(), batch, rows, cols,
                                     iters, (float)eps, ws.ptr, ws.bytes, stream_of(inp)));
        ws.held.unlock();
        return {d_inp.scalar_type() == sd ? d_inp : d_inp.to(sd), Tensor(), Tensor()};
    }
};

struct RMSNormFn : public torch::autograd::Function<RMSNormFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &inp_in, const Tensor &w_in, double eps) {
        TORCH_CHECK(is_act_dtype(inp_in) && is_act_dtype(w_in), "mhc: rmsnorm takes float32 or bfloat16 tensors");
        const Tensor inp = act(inp_in), w = act(w_in);
        c10::DeviceGuard guard(inp.device());
        const int C = inp.size(-1);
        const int rows = (int)(inp.numel() / C);
        Tensor out = at::empty_like(inp);
        Tensor rms = at::empty({rows}, inp.options().dtype(at::kFloat));
        check("mhc_rmsnorm_fwd", mhc_rmsnorm_fwd(ptr(inp), dt(inp), ptr(w), dt(w), ptr(out), rms.data_ptr<float>(), rows, C,
                                                  (float)eps, stream_of(inp)));
        ctx->save_for_backward({inp, w, rms});
        return out;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &inp = saved[0], &w = saved[1], &rms = saved[2];
        c10::DeviceGuard guard(inp.device());
        const Tensor go = act(grads[0].scalar_type() == inp.scalar_type() ? grads[0] : grads[0].to(inp.scalar_type()));
        const int C = inp.size(-1);
        const int rows = (int)(inp.numel() / C);
        Tensor d_inp = at::empty_like(inp);
        Tensor d_w = at::empty({C}, inp.options().dtype(at::kFloat));
        Scratch ws = scratch(inp, mhc_rmsnorm_bwd_workspace_bytes(rows, C));
        check("mhc_rmsnorm_bwd",
              mhc_rmsnorm_bwd(ptr(go), ptr(inp), dt(inp), ptr(w), dt(w), rms.data_ptr<float>(), ptr(d_inp),
                              d_w.data_ptr<float>(), rows, C, ws.ptr, ws.bytes, stream_of(inp)));
        ws.held.unlock();
        return {d_inp, d_w.scalar_type() == w.scalar_type() ? d_w : d_w.to(w.scalar_type()), Tensor()};
    }
};

py::object g_error_class;  // mhc._lib.MHCError, handed over at import

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "PyTorch-ROCm binding of libmhc_hip.so (C ABI: include/mhc_hip.h)";
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const MhcError &e) {
            if (g_error_class) {
                py::object exc = g_error_class(e.fn, e.status);
                PyErr_SetObject(g_error_class.ptr(), exc.ptr());
            } else {
                PyErr_SetString(PyExc_RuntimeError, e.what());
            }
        }
    });
    m.def("set_error_class", [](py::object cls) { g_error_class = std::move(cls); });
    m.def("set_param_cache", [](bool on) { g_param_cache = on; },
          "Opt in to reusing the packed phi / bias / alpha of a layer while the parameters' storage addresses and "
          "in-place version counters are unchanged.  Writes through `.data` do not bump the counters: leave it off "
          "(the default) if parameters are ever updated that way.");
    m.def("abi_version", []() { return mhc_abi_version(); });
    m.def("mhc_layer_dynamic", &mhc_layer_dynamic, py::arg("x"), py::arg("w"), py::arg("phi_pre"), py::arg("phi_post"),
          py::arg("phi_res"), py::arg("alpha_pre"), py::arg("alpha_post"), py::arg("alpha_res"), py::arg("b_pre"),
          py::arg("b_post"), py::arg("b_res"), py::arg("iters"), py::arg("eps"), py::arg("out_dtype"), py::arg("f_inject"),
          py::arg("compute_bf16") = false,
          "mhc_layer_fwd_dynamic / mhc_layer_bwd_dynamic with autograd (reference bindings.cu:405-542)");
    m.def("mhc_layer_static", &mhc_layer_static, "mhc_layer_fwd / mhc_layer_bwd with autograd (reference bindings.cu:264-401)");
    m.def("mhc_layer_inference", &mhc_layer_inference, "mhc_layer_fwd_inference (reference bindings.cu:221-262)");
    m.def("sinkhorn_knopp", [](const Tensor &inp, int64_t iters, double eps) { return SinkhornFn::apply(inp, iters, eps); });
    m.def("rmsnorm", [](const Tensor &inp, const Tensor &w, double eps) { return RMSNormFn::apply(inp, w, eps); });
}
