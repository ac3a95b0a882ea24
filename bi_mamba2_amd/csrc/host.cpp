// The host path of the operator and of the BiMamba2 layer in native code: argument checks, parameter block, memory and the
// autograd functions around bimamba2_fwd / bimamba2_bwd and the layer's other kernels.
//
// Why it exists: a forward + backward pass through Python (ctypes parameter block, autograd functions whose backward needs
// the interpreter lock, one torch op per small map) took the host 0.18 - 0.37 ms, the layer's 1.0 ms, which is more than the
// kernels take at every small or ordinary size.  The functions here do the same checks, make the same launches and leave the
// same tensors for the backward pass; the interpreter lock is released while they run.
//
// Built as a Python module (bi_mamba2_amd/_host.so); load(path) opens libbimamba2_hip.so and resolves the C ABI, so the
// module follows the library the Python side was told to use.
#include <dlfcn.h>
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <c10/hip/HIPGuard.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <array>
#include <optional>
#include <string>
#include <vector>

#include "../../include/bimamba2.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

struct AssertionFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
#define BM2_ASSERT(cond, what) \
    do {                       \
        if (!(cond)) throw AssertionFailure(what); \
    } while (0)

struct Api {
    decltype(&bimamba2_fwd) fwd = nullptr;
    decltype(&bimamba2_bwd) bwd = nullptr;
    decltype(&bimamba2_workspace_bytes) workspace_bytes = nullptr;
    decltype(&bimamba2_state_copies) state_copies = nullptr;
    decltype(&bimamba2_chunk_scan_reads_cb) reads_cb = nullptr;
    decltype(&bimamba2_chunk_for) chunk_for = nullptr;
    decltype(&bimamba2_seq_boundaries) seq_boundaries = nullptr;
    decltype(&bimamba2_strerror) strerror = nullptr;
    decltype(&bimamba2_rmsnorm_gated_fwd) norm_fwd = nullptr;
    decltype(&bimamba2_rmsnorm_gated_workspace_bytes) norm_workspace = nullptr;
    decltype(&bimamba2_conv1d_silu_fwd) conv_fwd = nullptr;
    decltype(&bimamba2_conv1d_silu_workspace_bytes) conv_workspace = nullptr;
    decltype(&bimamba2_cast_many) cast_many = nullptr;
    decltype(&bimamba2_norm_scan_conv_bwd) norm_scan_conv_bwd = nullptr;
    decltype(&bimamba2_gemm) gemm = nullptr;
    decltype(&bimamba2_gemm_workspace_bytes) gemm_workspace = nullptr;
    decltype(&bimamba2_gemm_plan) gemm_plan = nullptr;
} api;

void load(const std::string &path) {
    void *lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(lib, "cannot open ", path, ": ", dlerror());
    auto get = [&](auto &fn, const char *name) {
        fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(dlsym(lib, name));
        TORCH_CHECK(fn, path, " does not export ", name);
    };
    size_t (*params_size)() = nullptr, (*norm_size)() = nullptr, (*conv_size)() = nullptr, (*cast_size)() = nullptr, (*gemm_size)() = nullptr;
    get(params_size, "bimamba2_params_size");
    get(norm_size, "bimamba2_norm_params_size");
    get(conv_size, "bimamba2_conv_params_size");
    get(cast_size, "bimamba2_cast_params_size");
    get(gemm_size, "bimamba2_gemm_params_size");
    TORCH_CHECK(params_size() == sizeof(bimamba2_params) && norm_size() == sizeof(bimamba2_norm_params) &&
                    conv_size() == sizeof(bimamba2_conv_params) && cast_size() == sizeof(bimamba2_cast_params) &&
                    gemm_size() == sizeof(bimamba2_gemm_params),
                path, " was built from another version of include/bimamba2.h");
    get(api.fwd, "bimamba2_fwd");
    get(api.bwd, "bimamba2_bwd");
    get(api.workspace_bytes, "bimamba2_workspace_bytes");
    get(api.state_copies, "bimamba2_state_copies");
    get(api.reads_cb, "bimamba2_chunk_scan_reads_cb");
    get(api.chunk_for, "bimamba2_chunk_for");
    get(api.seq_boundaries, "bimamba2_seq_boundaries");
    get(api.strerror, "bimamba2_strerror");
    get(api.norm_fwd, "bimamba2_rmsnorm_gated_fwd");
    get(api.norm_workspace, "bimamba2_rmsnorm_gated_workspace_bytes");
    get(api.conv_fwd, "bimamba2_conv1d_silu_fwd");
    get(api.conv_workspace, "bimamba2_conv1d_silu_workspace_bytes");
    get(api.cast_many, "bimamba2_cast_many");
    get(api.norm_scan_conv_bwd, "bimamba2_norm_scan_conv_bwd");
    get(api.gemm, "bimamba2_gemm");
    get(api.gemm_workspace, "bimamba2_gemm_workspace_bytes");
    get(api.gemm_plan, "bimamba2_gemm_plan");
}

void check(int rc, const char *entry) {
    if (rc == BIMAMBA2_OK) return;
    const std::string msg = std::string(entry) + ": " + api.strerror(rc) + " (code " + std::to_string(rc) + ")";
    if (rc == BIMAMBA2_EINVAL || rc == BIMAMBA2_EUNSUPPORTED || rc == BIMAMBA2_ESCRATCH) TORCH_CHECK_VALUE(false, msg);
    TORCH_CHECK(false, msg);
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int dtype_code(at::ScalarType t, const char *what) {
    switch (t) {
        case at::kFloat: return BIMAMBA2_F32;
        case at::kBFloat16: return BIMAMBA2_BF16;
        case at::kHalf: return BIMAMBA2_F16;
        default: TORCH_CHECK_VALUE(false, "unsupported ", what, " ", t, " (need float32, bfloat16 or float16)"); return -1;
    }
}

void require_gpu(const Tensor &t, const char *name) {
    TORCH_CHECK(t.is_cuda(), name, " is on ", t.device(),
                ": the bidirectional SSD kernels run on an AMD GPU only (there is no CPU fallback)");
}

// device memory from torch's allocator without the dispatcher in front of it (1.6 -> 0.8 us; a training step makes about twenty)
inline Tensor device_empty(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor &beside) {
    return at::detail::empty_cuda(sizes, dtype, beside.device(), std::nullopt);
}

inline bool aligned16(const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }
inline size_t round_up(size_t n, size_t to) { return (n + to - 1) / to * to; }
inline Tensor as_type(const Tensor &t, at::ScalarType dtype) { return t.scalar_type() == dtype ? t : t.to(dtype); }
inline Tensor undef(const OptTensor &t) { return t ? *t : Tensor(); }

// float32 contiguous form of a parameter (A, D, dt_bias) or state
inline Tensor f32c(const Tensor &t) { return as_type(t, at::kFloat).contiguous(); }

// The gradients that the kernels write have no history.  Where a backward pass is itself recorded (create_graph), they are given
// one that leads back to what they were computed from and refuses to be differentiated: as one term of a loss they would
// otherwise count as constants without a word.
struct NoSecondDerivative : torch::autograd::Node {
    const char *of;
    explicit NoSecondDerivative(const char *of_) : of(of_) {}
    std::string name() const override { return "NoSecondDerivative"; }
    variable_list apply(variable_list &&) override { TORCH_CHECK(false, of, " has no second derivative: its gradients cannot be differentiated again"); }
};

variable_list once_differentiable(variable_list grads, const variable_list &from, const variable_list &upstream, const char *of) {
    if (!at::GradMode::is_enabled()) return grads;
    variable_list all = from;
    all.insert(all.end(), upstream.begin(), upstream.end());
    const std::shared_ptr<torch::autograd::Node> node(new NoSecondDerivative(of), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(all));
    for (Tensor &g : grads)
        if (g.defined()) torch::autograd::set_history(g, node);
    return grads;
}

// ---------------------------------------------------------------------------------------------------------------------
// the operator
// ---------------------------------------------------------------------------------------------------------------------
struct ScanOpts : torch::CustomClassHolder {
    int64_t chunk = 0;
    bool dt_softplus = false, want_final = false;
    bool copies = false;          // the forward kept the states in 16 bits
    bool cb = false;              // the forward kept C.B^T
    double dt_min = 0, dt_max = 0;
};

// The operands in the form the kernels take (16-bit or float32 rows with the last dimension contiguous, float32
// parameters) and the parameter block that points at them.
struct Problem {
    bimamba2_params p{};
    Tensor x, dt, A, B, C, D, z, bias, init_f, init_b, seq;

    Tensor strided(const Tensor &t, const char *name, const void *&ptr, int64_t &s0, int64_t &s1, int64_t &s2) {
        require_gpu(t, name);
        Tensor r = as_type(t, x.scalar_type());
        if (r.stride(-1) != 1) r = r.contiguous();
        ptr = r.const_data_ptr();
        s0 = r.stride(0);
        s1 = r.stride(1);
        s2 = r.stride(2);
        return r;
    }
    Tensor param(const Tensor &t, const char *name, const float *&ptr) {
        require_gpu(t, name);
        Tensor r = f32c(t);
        ptr = r.const_data_ptr<float>();
        return r;
    }

    Problem(const Tensor &x_, const Tensor &dt_, const Tensor &A_, const Tensor &B_, const Tensor &C_, const Tensor &D_,
            const Tensor &z_, const Tensor &bias_, const Tensor &init_f_, const Tensor &init_b_, const Tensor &seq_,
            const ScanOpts &o) {
        BM2_ASSERT(x_.dim() == 4 && B_.dim() == 4, "x: expected (batch, seqlen, nheads, headdim), B: (batch, seqlen, ngroups, dstate)");
        const int64_t batch = x_.size(0), seqlen = x_.size(1), nheads = x_.size(2), headdim = x_.size(3);
        const int64_t ngroups = B_.size(2), dstate = B_.size(3);
        BM2_ASSERT(ngroups > 0 && nheads % ngroups == 0, "nheads must be a multiple of ngroups");
        BM2_ASSERT(B_.size(0) == batch && B_.size(1) == seqlen, "B: expected (batch, seqlen, ngroups, dstate)");
        BM2_ASSERT(dt_.sizes() == at::IntArrayRef({batch, seqlen, nheads}), "dt: expected (batch, seqlen, nheads)");
        BM2_ASSERT(A_.sizes() == at::IntArrayRef({nheads}), "A: expected (nheads,)");
        BM2_ASSERT(C_.sizes() == B_.sizes(), "C: expected the shape of B");
        BM2_ASSERT(o.chunk >= 32, "chunk_size must be at least 32 (as in the reference) and at most 256");
        BM2_ASSERT(!z_.defined() || z_.sizes() == x_.sizes(), "z: expected the shape of x");
        BM2_ASSERT(!D_.defined() || D_.sizes() == at::IntArrayRef({nheads}) || D_.sizes() == at::IntArrayRef({nheads, headdim}),
                   "D: expected (nheads,) or (nheads, headdim)");
        BM2_ASSERT(!bias_.defined() || bias_.sizes() == at::IntArrayRef({nheads}), "dt_bias: expected (nheads,)");
        require_gpu(x_, "x");
        p.batch = batch; p.seqlen = seqlen; p.nheads = nheads; p.headdim = headdim;
        p.ngroups = ngroups; p.dstate = dstate; p.chunk_size = o.chunk;
        p.dtype = dtype_code(x_.scalar_type(), "dtype");
        p.dt_dtype = dtype_code(dt_.scalar_type(), "dt dtype");
        p.dt_softplus = o.dt_softplus;
        p.dt_min = (float)o.dt_min;
        p.dt_max = (float)o.dt_max;
        x = x_;
        x = strided(x_, "x", p.x, p.x_sb, p.x_sl, p.x_sh);
        require_gpu(dt_, "dt");
        dt = dt_;
        p.dt = dt.const_data_ptr();
        p.dt_sb = dt.stride(0); p.dt_sl = dt.stride(1); p.dt_sh = dt.stride(2);
        A = param(A_, "A", p.A);
        B = strided(B_, "Bm", p.Bm, p.B_sb, p.B_sl, p.B_sg);
        C = strided(C_, "Cm", p.Cm, p.C_sb, p.C_sl, p.C_sg);
        if (D_.defined()) {
            p.has_D = 1;
            p.D_has_hdim = D_.dim() == 2;
            D = param(D_, "D", p.D);
        }
        if (z_.defined()) {
            p.has_z = 1;
            z = strided(z_, "z", p.z, p.z_sb, p.z_sl, p.z_sh);
        }
        if (bias_.defined()) {
            p.has_dt_bias = 1;
            bias = param(bias_, "dt_bias", p.dt_bias);
        }
        if (init_f_.defined()) {
            BM2_ASSERT(init_f_.sizes() == at::IntArrayRef({batch, nheads, headdim, dstate}), "initial_f: expected (batch, nheads, headdim, dstate)");
            init_f = param(init_f_, "initial_f", p.initial_f);
        }
        if (init_b_.defined()) {
            BM2_ASSERT(init_b_.sizes() == at::IntArrayRef({batch, nheads, headdim, dstate}), "initial_b: expected (batch, nheads, headdim, dstate)");
            init_b = param(init_b_, "initial_b", p.initial_b);
        }
        if (seq_.defined()) {
            BM2_ASSERT(seq_.sizes() == at::IntArrayRef({batch, seqlen}), "seq_idx: expected (batch, seqlen)");
            require_gpu(seq_, "seq_idx");
            seq = as_type(seq_, at::kInt).contiguous();
            p.seq_idx = seq.const_data_ptr<int32_t>();
        }
        p.stream = stream_of(x);
    }
};

// What the forward pass leaves for the backward pass besides its operands, in one float32 allocation: dt_out, cs_f, cs_b, the
// states entering the chunks (copies: in the operands' 16-bit type, where the kernels can keep them that way) and, with cb,
// C.B^T and its transpose.  One chunk without states of its own (final: the caller takes the final states) has no states to keep.
struct Kept {
    size_t n1 = 0, ns = 0, ncb = 0;
    bool copies = false;
    Kept(const bimamba2_params &p, bool copies_, bool cb, bool final) : copies(copies_) {
        const size_t nc = (p.seqlen + p.chunk_size - 1) / p.chunk_size;
        n1 = round_up((size_t)p.batch * p.nheads * nc * p.chunk_size, 64);
        ns = round_up((size_t)p.batch * nc * p.nheads * p.headdim * p.dstate, 64);
        if (copies) ns /= 2;
        if (p.seqlen <= p.chunk_size && !p.initial_f && !p.initial_b && !final) ns = 0;
        if (cb) ncb = round_up((size_t)p.batch * nc * p.ngroups * p.chunk_size * p.chunk_size, 64);
    }
    int64_t floats() const { return (int64_t)(3 * n1 + 2 * ns + 2 * ncb); }
    void point(bimamba2_params &p, float *base) const {
        p.dt_out = base;
        p.cs_f = base + n1;
        p.cs_b = base + 2 * n1;
        float *st = base + 3 * n1;
        if (ns && copies) {
            p.states16_f = st;
            p.states16_b = st + ns;
        } else if (ns) {
            p.states_f = st;
            p.states_b = st + ns;
        }
        if (ncb) {
            p.CB = st + 2 * ns;
            p.CBT = p.CB + ncb;
        }
    }
    // what bimamba2_fwd and bimamba2_bwd are told about these
    int kept() const { return ns ? 0 : 4; }
    int saved() const { return kept() | (ncb ? 3 : 1); }
};

// Whether the forward pass keeps C.B^T and its transpose for the backward pass: where the backward's kernels read them and they
// are no larger than what the call holds between the passes anyway (x, the decays and the states), so that a model's layers
// hold at most twice as much.  The forward pass forms the product for itself there; the backward's launch for both took 9 to 13 us
// (float32 with 16 heads in 2 groups over 2 x 1111 positions, 10 MB beside 15; bfloat16 at state dimension 128 over 2 x 3001, 13
// MB beside 57).  With few narrow heads per group it would be many times that: 17 MB beside 1.5 at 4 heads of 16 in 4 groups.
bool keeps_cb(const bimamba2_params &p) {
    if (!api.reads_cb(&p, 0) || !api.reads_cb(&p, 1)) return false;
    const size_t e = p.dtype == BIMAMBA2_F32 ? 4 : 2, x = e * p.batch * p.seqlen * p.nheads * p.headdim;
    // (beside the states of the chunks, also where there are none to keep)
    const Kept without(p, false, false, true), with(p, false, true, true);
    return 8 * with.ncb <= x + 4 * (size_t)without.floats();
}

Tensor attach_workspace(bimamba2_params &p, bool bwd, const Tensor &like) {
    Tensor ws = device_empty({(int64_t)std::max<size_t>(api.workspace_bytes(&p, bwd), 1)}, at::kByte, like);
    p.workspace = ws.mutable_data_ptr();
    p.workspace_bytes = ws.numel();
    return ws;
}

struct ScanResult {
    Tensor out, out_x, final_f, final_b, kept;
};

ScanResult scan_forward(Problem &q, ScanOpts &o, bool keep) {
    bimamba2_params &p = q.p;
    ScanResult r;
    if (keep) {
        o.copies = api.state_copies(&p) != 0;
        o.cb = !o.copies && keeps_cb(p);
        const Kept k(p, o.copies, o.cb, o.want_final);
        r.kept = device_empty({k.floats()}, at::kFloat, q.x);
        k.point(p, r.kept.mutable_data_ptr<float>());
        p.fwd_saved = k.kept();
    }
    r.out = device_empty(q.x.sizes(), q.x.scalar_type(), q.x);
    p.out = r.out.mutable_data_ptr();
    if (keep && p.has_z) {        // the pre-gate output is what a backward pass needs; without one the store is skipped
        r.out_x = device_empty(q.x.sizes(), q.x.scalar_type(), q.x);
        p.out_x = r.out_x.mutable_data_ptr();
    }
    if (o.want_final) {
        const std::array<int64_t, 4> st = {p.batch, p.nheads, p.headdim, p.dstate};
        r.final_f = device_empty(st, at::kFloat, q.x);
        r.final_b = device_empty(st, at::kFloat, q.x);
        p.final_f = r.final_f.mutable_data_ptr<float>();
        p.final_b = r.final_b.mutable_data_ptr<float>();
    }
    const Tensor ws = attach_workspace(p, false, q.x);
    check(api.fwd(&p), "bimamba2_fwd");
    return r;
}

// Packed sequences: the largest number of boundaries that falls into one chunk.  The count is taken on the device and written
// to pinned host memory; the host waits for that kernel only, after it has enqueued the forward pass at the usual chunk
// size, so that the GPU has work while the host reads the answer (which nearly always is that the chunk size may stay).
constexpr int64_t max_boundaries = BIMAMBA2_MAX_SEQ_BOUNDARIES;

struct EventCache {
    std::vector<hipEvent_t> of_device;
    hipEvent_t get(int device) {
        if ((int)of_device.size() <= device) of_device.resize(device + 1, nullptr);
        if (!of_device[device]) TORCH_CHECK(hipEventCreateWithFlags(&of_device[device], hipEventDisableTiming) == hipSuccess, "hipEventCreate failed");
        return of_device[device];
    }
    ~EventCache() {
        for (hipEvent_t e : of_device)
            if (e) (void)hipEventDestroy(e);
    }
};

struct BoundaryCount {
    Tensor counts;
    hipEvent_t event = nullptr;
    explicit BoundaryCount(const bimamba2_params &p, int device) {
        static thread_local EventCache events;
        const int64_t nc = (p.seqlen + p.chunk_size - 1) / p.chunk_size;
        counts = at::empty({p.batch * nc}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        check(api.seq_boundaries(&p, counts.mutable_data_ptr<int32_t>()), "bimamba2_seq_boundaries");
        const hipEvent_t e = events.get(device);
        TORCH_CHECK(hipEventRecord(e, static_cast<hipStream_t>(p.stream)) == hipSuccess, "hipEventRecord failed");
        event = e;
    }
    BoundaryCount(const BoundaryCount &) = delete;
    // (an exception between the launch and wait(): the pinned memory goes back only when the kernel has written it)
    ~BoundaryCount() {
        if (event) (void)hipEventSynchronize(event);
    }
    int64_t wait() {
        const hipEvent_t recorded = event;
        event = nullptr;
        TORCH_CHECK(hipEventSynchronize(recorded) == hipSuccess, "waiting for the count of sequence boundaries failed");
        const int32_t *c = counts.const_data_ptr<int32_t>();
        return counts.numel() ? *std::max_element(c, c + counts.numel()) : 0;
    }
};

template <typename MakeProblem> ScanResult scan_checked(MakeProblem make, ScanOpts &o, bool keep) {
    {
        Problem q = make(o);
        q.p.chunk_size = o.chunk = api.chunk_for(&q.p, keep);
        if (!q.p.seq_idx || o.chunk <= max_boundaries) return scan_forward(q, o, keep);
        BoundaryCount first(q.p, q.x.device().index());
        ScanResult r = scan_forward(q, o, keep);
        if (first.wait() <= max_boundaries) return r;
    }        // (the pass that does not count gives its memory back before the one that does takes its own)
    for (int64_t c : {128, 64, 32}) {
        if (c >= o.chunk) continue;
        o.chunk = c;
        Problem smaller = make(o);
        if (c <= max_boundaries || BoundaryCount(smaller.p, smaller.x.device().index()).wait() <= max_boundaries) return scan_forward(smaller, o, keep);
    }
    TORCH_CHECK_VALUE(false, "seq_idx puts more than ", max_boundaries, " sequence boundaries into every chunk size down to 32 positions");
}

class ScanFn : public torch::autograd::Function<ScanFn> {
public:
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &dt, const Tensor &A, const Tensor &B,
                                 const Tensor &C, const OptTensor &D, const OptTensor &z, const OptTensor &bias,
                                 const OptTensor &init_f, const OptTensor &init_b, const OptTensor &seq,
                                 c10::intrusive_ptr<ScanOpts> o) {
        ScanResult r = scan_checked([&](const ScanOpts &opts) {
            return Problem(x, dt, A, B, C, undef(D), undef(z), undef(bias), undef(init_f), undef(init_b), undef(seq), opts);
        }, *o, true);
        ctx->save_for_backward({x, dt, A, B, C, undef(D), undef(z), undef(bias), undef(init_f), undef(init_b), undef(seq), r.out_x, r.kept});
        ctx->saved_data["opts"] = c10::IValue::make_capsule(o);
        ctx->set_materialize_grads(false);
        if (!o->want_final) return {r.out};
        return {r.out, r.final_f, r.final_b};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const auto capsule = ctx->saved_data["opts"].toCapsule();
        const ScanOpts &o = *static_cast<const ScanOpts *>(capsule.get());
        const Tensor &x = s[0], &dt = s[1], &A = s[2], &B = s[3], &C = s[4], &D = s[5], &bias = s[7];
        const c10::DeviceGuard guard(x.device());
        Problem q(x, dt, A, B, C, D, s[6], bias, s[8], s[9], s[10], o);
        bimamba2_params &p = q.p;
        Tensor dout = grads[0].defined() ? grads[0] : at::zeros(x.sizes(), q.x.options());
        BM2_ASSERT(dout.sizes() == x.sizes(), "gradient of the output: expected the shape of x");
        dout = as_type(dout, x.scalar_type());
        // the kernels that read the kept 16-bit states take aligned rows: a gradient view that is not (a slice of a wider
        // tensor at an odd offset) is copied (clone: contiguous() leaves a contiguous tensor at an odd address where it is)
        bool even = dout.stride(-1) == 1;
        if (even && p.dtype != BIMAMBA2_F32)
            even = aligned16(dout.const_data_ptr()) && dout.stride(0) % 8 == 0 && dout.stride(1) % 8 == 0 && dout.stride(2) % 8 == 0;
        if (!even) dout = dout.clone(at::MemoryFormat::Contiguous);
        p.dout = dout.const_data_ptr();
        p.dout_sb = dout.stride(0); p.dout_sl = dout.stride(1); p.dout_sh = dout.stride(2);
        Tensor dfin_f, dfin_b, dinit_f, dinit_b;
        if (grads.size() > 1 && grads[1].defined()) dfin_f = q.param(grads[1], "dfinal_f", p.dfinal_f);
        if (grads.size() > 2 && grads[2].defined()) dfin_b = q.param(grads[2], "dfinal_b", p.dfinal_b);
        const std::array<int64_t, 4> st = {p.batch, p.nheads, p.headdim, p.dstate};
        if (q.init_f.defined()) {
            dinit_f = device_empty(st, at::kFloat, q.x);
            p.dinitial_f = dinit_f.mutable_data_ptr<float>();
        }
        if (q.init_b.defined()) {
            dinit_b = device_empty(st, at::kFloat, q.x);
            p.dinitial_b = dinit_b.mutable_data_ptr<float>();
        }
        Tensor kept = s[12].contiguous();
        const Kept k(p, o.copies, o.cb, o.want_final);
        k.point(p, kept.mutable_data_ptr<float>());
        p.fwd_saved = k.saved();
        Tensor dz, dD, dbias, out_x = s[11];
        if (p.has_z) {
            out_x = out_x.contiguous();
            p.out_x = out_x.mutable_data_ptr();
            dz = device_empty(x.sizes(), q.x.scalar_type(), q.x);
            p.dz = dz.mutable_data_ptr();
        }
        Tensor dx = device_empty(x.sizes(), q.x.scalar_type(), q.x), ddt = device_empty(dt.sizes(), dt.scalar_type(), dt), dB = device_empty(B.sizes(), q.x.scalar_type(), q.x),
               dC = device_empty(C.sizes(), q.x.scalar_type(), q.x), dA = device_empty(A.sizes(), at::kFloat, q.x);
        p.dx = dx.mutable_data_ptr();
        p.ddt = ddt.mutable_data_ptr();
        p.dB = dB.mutable_data_ptr();
        p.dC = dC.mutable_data_ptr();
        p.dA = dA.mutable_data_ptr<float>();
        if (D.defined()) {
            dD = device_empty(D.sizes(), at::kFloat, q.x);
            p.dD = dD.mutable_data_ptr<float>();
        }
        if (bias.defined()) {
            dbias = device_empty(bias.sizes(), at::kFloat, q.x);
            p.ddt_bias = dbias.mutable_data_ptr<float>();
        }
        const Tensor ws = attach_workspace(p, true, q.x);
        check(api.bwd(&p), "bimamba2_bwd");
        auto like = [](const Tensor &g, const Tensor &t) { return g.defined() ? as_type(g, t.scalar_type()) : g; };
        return once_differentiable({dx, ddt, like(dA, A), like(dB, B), like(dC, C), like(dD, D), dz.defined() ? like(dz, s[6]) : dz,
                                    like(dbias, bias), dinit_f, dinit_b, Tensor(), Tensor()}, s, grads, "bimamba_chunk_scan_combined");
    }
};

// forward-mode tangents: the call goes through the autograd function whether or not gradients are enabled, which says that
// there is no such derivative
inline bool has_tangent(const Tensor &t) { return t.defined() && t._fw_grad(0).defined(); }

inline bool wants_autograd(std::initializer_list<const Tensor *> ts) {
    const bool grads = at::GradMode::is_enabled();
    for (const Tensor *t : ts)
        if ((grads && t->defined() && t->requires_grad()) || has_tangent(*t)) return true;
    return false;
}

variable_list scan(const Tensor &x, const Tensor &dt, const Tensor &A, const Tensor &B, const Tensor &C, int64_t chunk,
                   const OptTensor &D, const OptTensor &z, const OptTensor &bias, bool dt_softplus, double dt_min, double dt_max,
                   bool want_final, const OptTensor &init_f, const OptTensor &init_b, const OptTensor &seq) {
    const Tensor D_ = undef(D), z_ = undef(z), b_ = undef(bias), f_ = undef(init_f), r_ = undef(init_b);
    auto o = c10::make_intrusive<ScanOpts>();
    o->chunk = chunk;
    o->dt_softplus = dt_softplus;
    o->want_final = want_final;
    o->dt_min = dt_min;
    o->dt_max = dt_max;
    c10::OptionalDeviceGuard guard;
    if (x.is_cuda()) guard.reset_device(x.device());
    if (wants_autograd({&x, &dt, &A, &B, &C, &D_, &z_, &b_, &f_, &r_})) return ScanFn::apply(x, dt, A, B, C, D, z, bias, init_f, init_b, seq, o);
    at::AutoDispatchBelowADInplaceOrView below;
    ScanResult r = scan_checked([&](const ScanOpts &opts) { return Problem(x, dt, A, B, C, D_, z_, b_, f_, r_, undef(seq), opts); }, *o, false);
    if (!want_final) return {r.out};
    return {r.out, r.final_f, r.final_b};
}

// ---------------------------------------------------------------------------------------------------------------------
// the BiMamba2 layer: in_proj -> [z | xBC | dt] -> conv + SiLU -> operator -> gated RMS norm -> out_proj
// ---------------------------------------------------------------------------------------------------------------------
struct LayerOpts : torch::CustomClassHolder {
    int64_t inner = 0, nheads = 0, headdim = 0, ngroups = 0, dstate = 0, chunk = 0, norm_group = 0;
    bool norm_before_gate = true;
    uint32_t needs = 0;           // bit i: input i of LayerFn takes a gradient
    uint32_t converted = 0;       // bit i: the forward took small parameter i from its float32 copy
    bool copies = false;          // the forward kept the states in 16 bits
    bool cb = false;              // the forward kept C.B^T
    double dt_min = 0, dt_max = 0, eps = 0;
};

// The layer's small parameters as the kernels take them: float32, A = -exp(A_log).  One launch for all of them.
struct Params32 {
    // A_log, D, dt_bias, conv weight, conv bias, norm weight
    static constexpr int N = 6;
    std::array<const float *, N> ptr{};
    Tensor buf;       // holds what had to be converted; null where the parameters are used as they are
};

void add_cast(bimamba2_cast_params &c, const Tensor &src, void *dst, int dst_dtype, int op, const float *aux = nullptr) {
    bimamba2_cast_item &it = c.item[c.count++];
    it.src = src.const_data_ptr();
    it.dst = dst;
    it.aux = aux;
    it.n = src.numel();
    it.src_dtype = dtype_code(src.scalar_type(), "parameter dtype");
    it.dst_dtype = dst_dtype;
    it.op = op;
}

// The parameters that need a float32 copy (bit i: parameter i; A = -exp(A_log) always is one).
uint32_t params_to_convert(const std::array<Tensor, Params32::N> &prm) {
    uint32_t mask = 0;
    for (int i = 0; i < Params32::N; ++i)
        if (prm[i].defined() && (i == 0 || prm[i].scalar_type() != at::kFloat || !prm[i].is_contiguous())) mask |= 1u << i;
    return mask;
}

// offsets (in floats, 256-byte steps so that every piece is aligned for vector loads) of the pieces in Params32::buf; the
// backward pass finds them again from the forward's mask
std::array<int64_t, Params32::N + 1> param_offsets(const std::array<Tensor, Params32::N> &prm, uint32_t converted) {
    std::array<int64_t, Params32::N + 1> off{};
    for (int i = 0; i < Params32::N; ++i) off[i + 1] = off[i] + (converted >> i & 1 ? (int64_t)round_up(prm[i].numel(), 64) : 0);
    return off;
}

// (a parameter that is used as it is has to be contiguous; the caller holds it)
Params32 point_params(const std::array<Tensor, Params32::N> &prm, uint32_t converted, const Tensor &buf) {
    const auto off = param_offsets(prm, converted);
    Params32 r;
    r.buf = buf;
    float *base = buf.mutable_data_ptr<float>();
    for (int i = 0; i < Params32::N; ++i)
        if (prm[i].defined()) r.ptr[i] = converted >> i & 1 ? base + off[i] : prm[i].const_data_ptr<float>();
    return r;
}

Params32 params_as_float32(std::array<Tensor, Params32::N> &prm, uint32_t converted, void *stream) {
    const auto off = param_offsets(prm, converted);
    const Tensor buf = device_empty({off.back()}, at::kFloat, prm[0]);
    Params32 r = point_params(prm, converted, buf);
    bimamba2_cast_params c{};
    c.stream = stream;
    std::array<Tensor, Params32::N> rows;
    for (int i = 0; i < Params32::N; ++i)
        if (converted >> i & 1) {
            rows[i] = prm[i].contiguous();
            add_cast(c, rows[i], const_cast<float *>(r.ptr[i]), BIMAMBA2_F32, i == 0 ? BIMAMBA2_CAST_NEG_EXP : BIMAMBA2_CAST_COPY);
        }
    check(api.cast_many(&c), "bimamba2_cast_many");
    return r;
}

struct LayerShape {
    int64_t batch, seqlen, rows, inner, conv, proj, width;
    int64_t pitch;      // of the rows of the projection's output: whole cache lines, and aligned for vector loads whatever nheads is
    size_t e;
    LayerShape(const Tensor &u, const Tensor &cw, const LayerOpts &o)
        : batch(u.size(0)), seqlen(u.size(1)), rows(batch * seqlen), inner(o.inner), conv(o.inner + 2 * o.ngroups * o.dstate),
          proj(o.inner + conv + o.nheads), width(cw.size(-1)), pitch((proj + 63) / 64 * 64), e(u.element_size()) {}
};

inline char *at_byte(const Tensor &t, size_t elements) { return static_cast<char *>(t.mutable_data_ptr()) + elements * t.element_size(); }

bimamba2_conv_params conv_params(const LayerShape &s, const Tensor &zx, const Params32 &w, void *stream) {
    bimamba2_conv_params c{};
    c.batch = s.batch; c.seqlen = s.seqlen; c.channels = s.conv; c.width = s.width;
    c.dtype = dtype_code(zx.scalar_type(), "dtype");
    c.has_bias = w.ptr[4] != nullptr;
    c.x = at_byte(zx, s.inner);
    c.x_sb = s.seqlen * s.pitch;
    c.x_sl = s.pitch;
    c.weight = w.ptr[3];
    c.bias = w.ptr[4];
    c.stream = stream;
    return c;
}

bimamba2_params layer_scan_params(const LayerShape &s, const LayerOpts &o, const Tensor &zx, const Tensor &xbc, const Params32 &w, void *stream) {
    bimamba2_params p{};
    p.batch = s.batch; p.seqlen = s.seqlen; p.nheads = o.nheads; p.headdim = o.headdim;
    p.ngroups = o.ngroups; p.dstate = o.dstate; p.chunk_size = o.chunk;
    p.dtype = p.dt_dtype = dtype_code(zx.scalar_type(), "dtype");
    p.dt_softplus = 1;
    p.dt_min = (float)o.dt_min; p.dt_max = (float)o.dt_max;
    p.has_D = 1; p.has_dt_bias = 1;
    p.x = at_byte(xbc, 0);
    p.x_sb = s.seqlen * s.conv; p.x_sl = s.conv; p.x_sh = o.headdim;
    p.Bm = at_byte(xbc, s.inner);
    p.Cm = at_byte(xbc, s.inner + o.ngroups * o.dstate);
    p.B_sb = p.C_sb = s.seqlen * s.conv; p.B_sl = p.C_sl = s.conv; p.B_sg = p.C_sg = o.dstate;
    p.dt = at_byte(zx, s.inner + s.conv);
    p.dt_sb = s.seqlen * s.pitch; p.dt_sl = s.pitch; p.dt_sh = 1;
    p.A = w.ptr[0]; p.D = w.ptr[1]; p.dt_bias = w.ptr[2];
    p.stream = stream;
    return p;
}

bimamba2_norm_params layer_norm_params(const LayerShape &s, const LayerOpts &o, const Tensor &zx, const Tensor &y, const Params32 &w, void *stream) {
    bimamba2_norm_params n{};
    n.rows = s.rows; n.cols = s.inner; n.group_size = o.norm_group;
    n.dtype = dtype_code(zx.scalar_type(), "dtype");
    n.has_z = 1;
    n.norm_before_gate = o.norm_before_gate;
    n.eps = (float)o.eps;
    n.x = y.const_data_ptr(); n.x_rs = s.inner;
    n.z = at_byte(zx, 0); n.z_rs = s.pitch;
    n.weight = w.ptr[5];
    n.stream = stream;
    return n;
}

// ---- the projections' matrix products -------------------------------------------------------------------------------
// c (m x n, row pitch ldc) = sum_k A(m, k) B(n, k) (+ bias), by this library's kernel; false where it does not take the problem.
// a, b: 2-d with unit stride along columns; a_kc: k along a's columns (else along its rows), b_kc likewise.
bool own_product(const Tensor &a, bool a_kc, const Tensor &b, bool b_kc, const Tensor &bias, const Tensor &c) {
    if (c.scalar_type() == at::kFloat || a.stride(1) != 1 || b.stride(1) != 1 || c.stride(1) != 1) return false;
    bimamba2_gemm_params g{};
    g.m = c.size(0);
    g.n = c.size(1);
    g.k = a.size(a_kc ? 1 : 0);
    g.dtype = dtype_code(c.scalar_type(), "dtype");
    g.a_kcontig = a_kc;
    g.b_kcontig = b_kc;
    g.lda = a.stride(0);
    g.ldb = b.stride(0);
    g.ldc = c.stride(0);
    g.a = a.const_data_ptr();
    g.b = b.const_data_ptr();
    g.bias = bias.defined() ? bias.const_data_ptr() : nullptr;
    g.c = c.mutable_data_ptr();
    g.stream = stream_of(c);
    const size_t need = api.gemm_workspace(&g);
    Tensor ws;
    if (need) {
        ws = device_empty({(int64_t)need}, at::kByte, c);
        g.partial = static_cast<float *>(ws.mutable_data_ptr());
        g.partial_bytes = need;
    }
    const int rc = api.gemm(&g);
    if (rc == BIMAMBA2_EUNSUPPORTED) return false;
    check(rc, "bimamba2_gemm");
    return true;
}

// Which products the own kernel takes, in operations.  A library call costs the host 18 us, which shows where a layer's kernels do not
// hide it: a forward pass without gradients up to some 65 us, a training step up to some 230.  Where the host is hidden, or a
// replayed graph does without it, the library's kernel is the faster one of the large products.  One layer of dstate 64 in bfloat16
// over rows x d_model, us a pass with the library -> with the own kernel (eager, as a replayed graph):
//   without gradients: 197 x 384 (0.25 and 0.12 GFLOP) 67 -> 51, 47 -> 48; 197 x 768 (0.98 and 0.46) 67 -> 55, 50 -> 52; 1024 x 384 (1.3
//     and 0.6) 67 -> 58, 56 -> 56; above the line 1024 x 768 (5.1, 2.4) 66 -> 70, 65 -> 70 for the second, 512 x 1024 (4.5, 2.2) 65 -> 72, 64 -> 73
//   forward products of a training step: 2048 x 384 (2.6, 1.2) 255 -> 228, 223 -> 223; 1024 x 576 (2.9, 1.4) 247 -> 232, 227 -> 229; 512 x 1024
//     (4.5, 2.2) 257 -> 262, 251 -> 259 for the second; above the line 2048 x 768 (10, 4.8) 308 -> 315, 307 -> 314
//   gradients of the inputs: 197 x 384 241 -> 214, 170 -> 163; 512 x 768 240 -> 230, 231 -> 228; 512 x 1024 273 -> 264, 270 -> 262; 2048 x 768 (4.8 for
//     the second) 314 -> 316, 313 -> 314
constexpr double OWN_INFERENCE_FLOPS = 1.5e9, OWN_TRAINING_FLOPS = 3e9, OWN_GRADIENT_FLOPS = 5e9;
// Gradients of inputs go further: own_input_gradient().  So do forward products whose columns are no multiple of 64 (the library has fast kernels for some of these
// numbers only), of 1024 to 4095 rows, 256 to 576 inputs and up to 2600 columns: 0.82 of the library's time over 30 with 3 GFLOP and more, 0.73 to 1.04, 0.77 over 16 with
// 1.5 to 3 (replayed graphs, operands from memory).  The others of 227 such products of 3 to 20 GFLOP below 16384 rows: fewer rows 1.15, 0.93 to 1.53 (116 x 2176 by 8900 19 ->
// 29 us), other inputs 0.99, 0.76 to 1.37, more rows 1.00 of what SPLIT_ROWS gives, 0.59 to 1.57 (15617 x 192 by 1030 16 -> 25).
constexpr int64_t RAGGED_ROWS = 1024, RAGGED_ROWS_END = 4096, RAGGED_INPUTS = 256, RAGGED_INPUTS_END = 577, RAGGED_COLUMNS_END = 2601;

// From so many rows or operations on, the columns of a forward product behind the last multiple of 256 go to the own kernel where the
// number of columns is no multiple of 64: the library has fast kernels for some of these numbers only.  us, library alone -> in
// two: 16384 x 768 by 3224 columns 128 -> 84; 24063 x 384 by 2060 109 -> 73; 4715 x 832 by 3482 53 -> 36; 19687 x 128 by 772 47 -> 20; but 5044 x 448
// by 1934 27 -> 33, 8931 x 704 by 2966 58 -> 71.  315 such products of layers of 128 to 1024 columns, operands from memory, above 1
// GFLOP: 0.92 of the library's time (0.89 with the better of both each time).  Fewer rows: 3233 x 896 by 3740 35 -> 48, 1658 x 768 by 3352
// 20 -> 27.  A multiple of 64 columns stays whole at any size: 188 products would take 1.2 times as long (15642 x 768 by 384 18 -> 35).
constexpr int64_t SPLIT_ROWS = 4096;
constexpr double SPLIT_FLOPS = 25e9;

// whether a forward product (rows x columns, a sum of `inputs`) goes to the own kernel
bool own_forward_product(int64_t rows, int64_t columns, int64_t inputs, bool training) {
    if (2.0 * rows * columns * inputs <= (training ? OWN_TRAINING_FLOPS : OWN_INFERENCE_FLOPS)) return true;
    return columns % 64 && rows >= RAGGED_ROWS && rows < RAGGED_ROWS_END && inputs >= RAGGED_INPUTS && inputs < RAGGED_INPUTS_END && columns < RAGGED_COLUMNS_END;
}

// c = x w^T (+ bias): the forward product.  c may be a view with a row pitch.
void product_nt(const Tensor &x, const Tensor &w, const Tensor &bias, Tensor c, bool training) {
    const int64_t m = c.size(0), n = c.size(1), whole = n / 256 * 256;
    const double per_column = 2.0 * m * x.size(1);
    if (own_forward_product(m, n, x.size(1), training) && own_product(x, true, w, true, bias, c)) return;
    if ((m >= SPLIT_ROWS || per_column * whole >= SPLIT_FLOPS) && n % 64 && whole && c.scalar_type() != at::kFloat && !bias.defined() &&
        own_product(x, true, w.narrow(0, whole, n - whole), true, Tensor(), c.narrow(1, whole, n - whole))) {
        Tensor front = c.narrow(1, 0, whole);
        at::mm_out(front, x, w.narrow(0, 0, whole).t());
        return;
    }
    if (bias.defined()) at::addmm_out(c, bias, x, w.t());
    else at::mm_out(c, x, w.t());
}

// Whether the gradient of a projection's input (rows x columns, a sum of `terms`) goes to the own kernel.  Beyond the line above, with twice as many terms as columns (in
// front of the first projection), own over library, replayed graphs, operands from memory, 403 products of layers of 128 to 4096 columns over 64 to 65536 rows:
//   below 2560 rows, where the library does not cut the sum: 0.70 over 130, 0.37 (128 x 3328 from 13672) to 0.99
//   large tiles, the sum in one piece, up to 1024 columns, 256 x 256 tiles from 384 columns on: 0.91 over 62, 0.74 (16960 x 1024 from 4384) to 1.09 (35085 x 512 from
//     2320), six of them above 1.02; 16384 x 768 from 3224 82 -> 71 us
//   the other 211, which the library keeps: 0.98, up to 1.31 (10736 x 576 from 2834; 14629 x 1280 from 5288 207 -> 258 us, 9152 x 1984 from 8126 285 -> 366)
bool own_input_gradient(int64_t rows, int64_t columns, int64_t terms) {
    if (2.0 * rows * columns * terms <= OWN_GRADIENT_FLOPS) return true;
    if (terms < 2 * columns || columns > 4096) return false;
    if (rows < 2560) return true;
    if (columns > 1024) return false;
    bimamba2_gemm_params g{};
    g.m = rows;
    g.n = columns;
    g.k = terms;
    g.a_kcontig = 1;
    int slices = 0;
    const int tile = api.gemm_plan(&g, &slices);
    return slices == 1 && (tile == 1 || (tile == 0 && columns >= 384));
}

// c = dy w: the gradient of a projection's input
void product_nn(const Tensor &dy, const Tensor &w, Tensor c) {
    if (own_input_gradient(c.size(0), c.size(1), dy.size(1)) && own_product(dy, true, w, false, Tensor(), c)) return;
    at::mm_out(c, dy, w);
}

// c = dy^T x: the gradient of a projection's weight.  Always the own kernel where it exists: the library does not cut the long
// sum over the rows.  us, library -> own: 3224 x 768 over 16384 rows 185 -> 88; 768 x 1536 145 -> 54; 4256 x 1024 over 65536 706 -> 493;
// 2320 x 512 over 4096 35 -> 27; 1676 x 384 over 992 15 -> 11; 1676 x 384 over 197 7.6 -> 5.9.
void product_tn(const Tensor &dy, const Tensor &x, Tensor c) {
    if (own_product(dy, false, x, false, Tensor(), c)) return;
    at::mm_out(c, dy.t(), x);
}

struct LayerKept {
    Tensor zx_rows, xbc, y, yn, rstd, kept, prm32;
};

Tensor layer_forward(const Tensor &u, const Tensor &w_in, const Tensor &b_in, std::array<Tensor, Params32::N> prm, const Tensor &w_out,
                     const Tensor &b_out, LayerOpts &o, bool keep, LayerKept *left) {
    const LayerShape s(u, prm[3], o);
    void *stream = stream_of(u);
    const Tensor u2 = u.reshape({s.rows, u.size(2)});
    const Tensor zx_rows = device_empty({s.rows, s.pitch}, u.scalar_type(), u), zx = zx_rows.narrow(1, 0, s.proj);
    product_nt(u2, w_in, b_in, zx, keep);
    o.converted = params_to_convert(prm);
    const Params32 w = params_as_float32(prm, o.converted, stream);

    const Tensor xbc = device_empty({s.rows, s.conv}, u.scalar_type(), u);
    bimamba2_conv_params c = conv_params(s, zx, w, stream);
    c.out = xbc.mutable_data_ptr();
    check(api.conv_fwd(&c), "bimamba2_conv1d_silu_fwd");

    const Tensor y = device_empty({s.rows, s.inner}, u.scalar_type(), u);
    bimamba2_params p = layer_scan_params(s, o, zx, xbc, w, stream);
    p.chunk_size = o.chunk = api.chunk_for(&p, keep);
    p.out = y.mutable_data_ptr();
    Tensor kept;
    if (keep) {
        o.copies = api.state_copies(&p) != 0;
        o.cb = !o.copies && keeps_cb(p);
        const Kept k(p, o.copies, o.cb, false);
        kept = device_empty({k.floats()}, at::kFloat, u);
        k.point(p, kept.mutable_data_ptr<float>());
        p.fwd_saved = k.kept();
    }
    const Tensor ws = attach_workspace(p, false, u);
    check(api.fwd(&p), "bimamba2_fwd");

    const Tensor yn = device_empty({s.rows, s.inner}, u.scalar_type(), u);
    Tensor rstd;
    bimamba2_norm_params n = layer_norm_params(s, o, zx, y, w, stream);
    n.out = yn.mutable_data_ptr();
    n.out_rs = s.inner;
    if (keep) {
        rstd = device_empty({s.rows, s.inner / o.norm_group}, at::kFloat, u);
        n.rstd = rstd.mutable_data_ptr<float>();
    }
    check(api.norm_fwd(&n), "bimamba2_rmsnorm_gated_fwd");
    const Tensor out = device_empty({s.batch, s.seqlen, w_out.size(0)}, u.scalar_type(), u);
    product_nt(yn, w_out, b_out, out.view({s.rows, w_out.size(0)}), keep);
    if (left) *left = {zx_rows, xbc, y, yn, rstd, kept, w.buf};
    return out;
}

class LayerFn : public torch::autograd::Function<LayerFn> {
public:
    static Tensor forward(AutogradContext *ctx, const Tensor &u, const Tensor &w_in, const OptTensor &b_in, const Tensor &A_log,
                          const Tensor &D, const Tensor &dt_bias, const Tensor &cw, const OptTensor &cb, const Tensor &nw,
                          const Tensor &w_out, const OptTensor &b_out, c10::intrusive_ptr<LayerOpts> o) {
        LayerKept k;
        const Tensor out = layer_forward(u, w_in, undef(b_in), {A_log, D, dt_bias, cw, undef(cb), nw}, w_out, undef(b_out), *o, true, &k);
        ctx->save_for_backward({u, w_in, A_log, D, dt_bias, cw, undef(cb), nw, w_out, k.zx_rows, k.xbc, k.y, k.yn, k.rstd, k.kept, k.prm32});
        ctx->saved_data["opts"] = c10::IValue::make_capsule(o);
        return out;
    }

    // The gradient of the projection's output is one buffer: the norm writes dz, the operator ddt and the convolution dxBC
    // into its columns (and the operator dx, dB and dC into the columns of the gradient of the convolution's output), so
    // nothing is concatenated.
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list v = ctx->get_saved_variables();
        const auto capsule = ctx->saved_data["opts"].toCapsule();
        const LayerOpts &o = *static_cast<const LayerOpts *>(capsule.get());
        auto needs = [&](int i) { return (o.needs >> i & 1) != 0; };
        const Tensor &u = v[0], &w_in = v[1], &w_out = v[8];
        // (a saved-tensor hook may hand back another layout than it was given: zx is kept with its padding columns, so that
        // contiguous is the layout the kernels were told)
        const Tensor zx = v[9].contiguous(), xbc = v[10].contiguous(), y = v[11].contiguous(), yn = v[12].contiguous(),
                     rstd = v[13].contiguous(), kept = v[14].contiguous(), prm32 = v[15].contiguous();
        std::array<Tensor, Params32::N> prm = {v[2], v[3], v[4], v[5], v[6], v[7]};
        for (int i = 0; i < Params32::N; ++i)
            if (prm[i].defined() && !(o.converted >> i & 1)) prm[i] = prm[i].contiguous();
        const c10::DeviceGuard guard(u.device());
        void *stream = stream_of(u);
        at::AutoDispatchBelowADInplaceOrView below;
        const LayerShape s(u, prm[3], o);
        const Params32 w = point_params(prm, o.converted, prm32);
        const Tensor dout = as_type(grads[0], u.scalar_type()).reshape({s.rows, w_out.size(0)});
        Tensor dw_in, db_in, dw_out, db_out, du;
        if (needs(9)) product_tn(dout, yn, dw_out = device_empty(w_out.sizes(), u.scalar_type(), u));
        if (needs(10)) db_out = dout.sum(0);

        // float32 gradients of the small parameters, one buffer: A, D, dt_bias, conv weight, conv bias, norm weight
        std::array<int64_t, Params32::N + 1> off{};
        for (int i = 0; i < Params32::N; ++i) off[i + 1] = off[i] + (prm[i].defined() ? (int64_t)round_up(prm[i].numel(), 64) : 0);
        const Tensor g32 = device_empty({off.back()}, at::kFloat, u);
        float *g = g32.mutable_data_ptr<float>();

        const Tensor dyn = device_empty({s.rows, s.inner}, u.scalar_type(), u), dy = device_empty({s.rows, s.inner}, u.scalar_type(), u);
        const Tensor dzx = device_empty({s.rows, s.pitch}, u.scalar_type(), u).narrow(1, 0, s.proj);
        product_nn(dout, w_out, dyn);
        bimamba2_norm_params n = layer_norm_params(s, o, zx, y, w, stream);
        n.rstd = rstd.mutable_data_ptr<float>();
        n.dout = dyn.const_data_ptr(); n.dout_rs = s.inner;
        n.dx = dy.mutable_data_ptr(); n.dx_rs = s.inner;
        n.dz = at_byte(dzx, 0); n.dz_rs = s.pitch;
        n.dweight = g + off[5];
        Tensor norm_ws = device_empty({(int64_t)std::max<size_t>(api.norm_workspace(&n), 1)}, at::kByte, u);
        n.workspace = norm_ws.mutable_data_ptr();
        n.workspace_bytes = norm_ws.numel();

        const Tensor dxbc = device_empty({s.rows, s.conv}, u.scalar_type(), u);
        bimamba2_params p = layer_scan_params(s, o, zx, xbc, w, stream);
        const Kept k(p, o.copies, o.cb, false);
        k.point(p, kept.mutable_data_ptr<float>());
        p.fwd_saved = k.saved();
        p.dout = dy.const_data_ptr();
        p.dout_sb = s.seqlen * s.inner; p.dout_sl = s.inner; p.dout_sh = o.headdim;
        p.dx = at_byte(dxbc, 0);
        p.dB = at_byte(dxbc, s.inner);
        p.dC = at_byte(dxbc, s.inner + o.ngroups * o.dstate);
        p.dx_sb = p.dB_sb = p.dC_sb = s.seqlen * s.conv;
        p.dx_sl = p.dB_sl = p.dC_sl = s.conv;
        p.ddt = at_byte(dzx, s.inner + s.conv);
        p.ddt_sb = s.seqlen * s.pitch; p.ddt_sl = s.pitch;
        p.dA = g + off[0]; p.dD = g + off[1]; p.ddt_bias = g + off[2];
        Tensor scan_ws = attach_workspace(p, true, u);

        bimamba2_conv_params cv = conv_params(s, zx, w, stream);
        cv.dout = dxbc.const_data_ptr();
        cv.dout_sb = s.seqlen * s.conv; cv.dout_sl = s.conv;
        cv.dx = at_byte(dzx, s.inner);
        cv.dx_sb = s.seqlen * s.pitch; cv.dx_sl = s.pitch;
        cv.dweight = g + off[3];
        if (prm[4].defined()) cv.dbias = g + off[4];
        Tensor conv_ws = device_empty({(int64_t)std::max<size_t>(api.conv_workspace(&cv), 1)}, at::kByte, u);
        cv.workspace = conv_ws.mutable_data_ptr();
        cv.workspace_bytes = conv_ws.numel();
        // the small gradients in their parameters' types; dA_log = dA * A
        std::array<Tensor, Params32::N> dprm;
        bimamba2_cast_params c{};
        c.stream = stream;
        static constexpr int input_of[Params32::N] = {3, 4, 5, 6, 7, 8};
        for (int i = 0; i < Params32::N; ++i) {
            if (!prm[i].defined() || !needs(input_of[i])) continue;
            const Tensor part = g32.narrow(0, off[i], prm[i].numel());
            if (i && prm[i].scalar_type() == at::kFloat) {
                dprm[i] = part.view(prm[i].sizes());
                continue;
            }
            dprm[i] = device_empty(prm[i].sizes(), prm[i].scalar_type(), prm[i]);
            add_cast(c, part, dprm[i].mutable_data_ptr(), dtype_code(prm[i].scalar_type(), "parameter dtype"),
                     i == 0 ? BIMAMBA2_CAST_MUL : BIMAMBA2_CAST_COPY, i == 0 ? w.ptr[0] : nullptr);
        }
        check(api.norm_scan_conv_bwd(&n, &p, &cv, &c), "bimamba2_norm_scan_conv_bwd");
        norm_ws = scan_ws = conv_ws = Tensor();           // (what follows may have their memory)
        if (needs(0)) {
            du = device_empty(u.sizes(), u.scalar_type(), u);
            product_nn(dzx, w_in, du.view({s.rows, u.size(2)}));
        }
        if (needs(1)) product_tn(dzx, u.reshape({s.rows, u.size(2)}), dw_in = device_empty(w_in.sizes(), u.scalar_type(), u));
        if (needs(2)) db_in = dzx.sum(0);
        return once_differentiable({du, dw_in, db_in, dprm[0], dprm[1], dprm[2], dprm[3], dprm[4], dprm[5], dw_out, db_out, Tensor()},
                                   v, grads, "BiMamba2");
    }
};

// Whether the layer's tensors have the shapes, the device and the types that its kernels are told; what does not (a parameter
// that was replaced, an input of another width, no rows at all) is left to the composition of the operators, whose own checks
// say what is wrong with it.
bool layer_fits(const Tensor &u, const Tensor &w_in, const Tensor &b_in, const std::array<Tensor, Params32::N> &prm, const Tensor &w_out,
                const Tensor &b_out, const LayerOpts &o) {
    if (u.dim() != 3 || u.numel() == 0 || w_in.dim() != 2 || w_out.dim() != 2 || w_out.numel() == 0) return false;
    if (o.headdim <= 0 || o.ngroups <= 0 || o.nheads * o.headdim != o.inner || o.nheads % o.ngroups || o.norm_group <= 0 || o.inner % o.norm_group)
        return false;
    const int64_t conv = o.inner + 2 * o.ngroups * o.dstate;
    auto is = [](const Tensor &t, at::IntArrayRef sizes) { return !t.defined() || t.sizes() == sizes; };
    if (!is(w_in, {o.inner + conv + o.nheads, u.size(2)}) || !is(b_in, {w_in.size(0)}) || !is(b_out, {w_out.size(0)})) return false;
    for (int i = 0; i < 3; ++i)
        if (!is(prm[i], {o.nheads})) return false;
    const Tensor &cw = prm[3];
    if (cw.dim() != 3 || cw.size(0) != conv || cw.size(1) != 1 || !is(prm[4], {conv}) || !is(prm[5], {o.inner})) return false;
    for (const Tensor *t : {&w_in, &b_in, &w_out, &b_out})
        if (t->defined() && t->scalar_type() != u.scalar_type()) return false;
    auto here = [&](const Tensor &t) { return !t.defined() || (t.device() == u.device() && t.layout() == at::kStrided); };
    for (const Tensor *t : {&u, &w_in, &b_in, &w_out, &b_out})
        if (!here(*t)) return false;
    return std::all_of(prm.begin(), prm.end(), here);
}

// nullopt: see layer_fits
OptTensor layer(const Tensor &u, const Tensor &w_in, const OptTensor &b_in, const Tensor &A_log, const Tensor &D, const Tensor &dt_bias,
             const Tensor &cw, const OptTensor &cb, const Tensor &nw, const Tensor &w_out, const OptTensor &b_out, int64_t headdim,
             int64_t ngroups, int64_t dstate, int64_t chunk, double dt_min, double dt_max, double eps, int64_t norm_group, bool norm_before_gate) {
    auto o = c10::make_intrusive<LayerOpts>();
    o->inner = w_out.size(1);
    o->headdim = headdim;
    o->nheads = o->inner / headdim;
    o->ngroups = ngroups;
    o->dstate = dstate;
    o->chunk = chunk;
    o->dt_min = dt_min;
    o->dt_max = dt_max;
    o->eps = eps;
    o->norm_group = norm_group;
    o->norm_before_gate = norm_before_gate;
    const Tensor bi = undef(b_in), bc = undef(cb), bo = undef(b_out);
    if (!layer_fits(u, w_in, bi, {A_log, D, dt_bias, cw, bc, nw}, w_out, bo, *o)) return std::nullopt;
    const c10::DeviceGuard guard(u.device());
    bool tangents = false;
    int i = 0;
    for (const Tensor *t : {&u, &w_in, &bi, &A_log, &D, &dt_bias, &cw, &bc, &nw, &w_out, &bo}) {
        if (at::GradMode::is_enabled() && t->defined() && t->requires_grad()) o->needs |= 1u << i;
        tangents |= has_tangent(*t);
        ++i;
    }
    if (o->needs || tangents)
        return LayerFn::apply(u, w_in, b_in, A_log, D, dt_bias, cw, cb, nw, w_out, b_out, o);
    at::AutoDispatchBelowADInplaceOrView below;
    return layer_forward(u, w_in, bi, {A_log, D, dt_bias, cw, bc, nw}, w_out, bo, *o, false, nullptr);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::register_exception_translator([](std::exception_ptr e) {
        try {
            if (e) std::rethrow_exception(e);
        } catch (const AssertionFailure &f) {
            PyErr_SetString(PyExc_AssertionError, f.what());
        } catch (python_error &f) {              // raised by a saved-tensor hook: the hook's own exception goes on
            f.restore();
        }
    });
    m.def("load", &load);
    m.def("scan", &scan, py::call_guard<py::gil_scoped_release>());
    m.def("own_forward_product", &own_forward_product);
    m.def("own_input_gradient", &own_input_gradient);
    m.def("layer", &layer, py::call_guard<py::gil_scoped_release>());
}
