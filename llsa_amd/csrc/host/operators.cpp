// The host side of the fused operators (llsa_l1 / l2 / l3 / lk) and of the token permutation: argument checks, one arena
// per call, the sequence of C-ABI calls of include/llsa_hip.h, and the autograd nodes.
//
//     forward   pool_pyramid_fwd (q, k, v: pooled rows, RoPE, operand tiles) [+ deeper levels]
//               topk_dense / topk_cascade [+ topk_sparse ...]
//               attn_fwd_lists  (the attention kernel, the transposed selections in the same launch), or at the long sequences
//               attn_fwd and, on a second stream beside it, transpose_indices_multi
//     backward  attn_bwd with fold_pooled = 1  (dq, dk, dv complete, rotated back and back through the qk-norm)
//
// Native because at the short sequences a step is bound by its host side: at B=1, H=6, N=1024 the kernels of a forward
// take about 13 us and those of a forward + backward 47, while the same sequence issued from Python took 33 and 100 to
// 180 (a backward written in Python also has to win the interpreter lock on the autograd thread).
//
// The library's entry points are called through the table of addresses its ctypes binding (llsa_amd/_lib.py) passes in, so
// that this file works on whatever build of the library the binding has loaded.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <array>
#include <mutex>
#include <optional>
#include <string>
#include <utility>
#include <vector>

#include "../../../include/llsa_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---------------------------------------------------------------------------------------
// errors: which Python exception, and its text
// ---------------------------------------------------------------------------------------
struct Failure {
    enum Kind { kValue, kNotImplemented, kRuntime, kLibrary } kind;
    std::string text;
};
PyObject* g_library_error = nullptr;      // llsa_amd._lib.LlsaError

[[noreturn]] void fail(Failure::Kind kind, std::string text) { throw Failure{kind, std::move(text)}; }

void set_python_error(const Failure& f) {                 // with the interpreter lock held
    PyObject* type = f.kind == Failure::kValue            ? PyExc_ValueError
                     : f.kind == Failure::kNotImplemented ? PyExc_NotImplementedError
                     : f.kind == Failure::kLibrary && g_library_error != nullptr ? g_library_error
                                                          : PyExc_RuntimeError;
    PyErr_SetString(type, f.text.c_str());
}

template <typename Fn>
auto without_interpreter(Fn fn) {
    std::optional<Failure> failure;
    {
        py::gil_scoped_release release;
        try {
            return fn();
        } catch (const Failure& f) {
            failure = f;
        }
    }
    set_python_error(*failure);
    throw py::error_already_set();
}
// the same on a thread of the autograd engine, which does not hold the lock
template <typename Fn>
auto in_engine(Fn fn) {
    try {
        return fn();
    } catch (const Failure& f) {
        py::gil_scoped_acquire acquire;
        set_python_error(f);
        python_error e;
        e.persist();
        throw e;
    }
}

// ---------------------------------------------------------------------------------------
// the library
// ---------------------------------------------------------------------------------------
struct Library {
    decltype(&llsa_last_error_string) last_error_string;
    decltype(&llsa_pool_pyramid_fwd) pool_pyramid_fwd;
    decltype(&llsa_topk_dense_tiles) topk_dense_tiles;
    decltype(&llsa_topk_sparse_tiles) topk_sparse_tiles;
    decltype(&llsa_topk_cascade_tiles) topk_cascade_tiles;
    decltype(&llsa_topk_cascade_max_parents) topk_cascade_max_parents;
    decltype(&llsa_attn_fwd) attn_fwd;
    decltype(&llsa_attn_fwd_lists) attn_fwd_lists;
    decltype(&llsa_attn_fwd_selects) attn_fwd_selects;
    decltype(&llsa_transpose_indices_multi) transpose_indices_multi;
    decltype(&llsa_transpose_one_launch) transpose_one_launch;
    decltype(&llsa_transpose_nested_bytes) transpose_nested_bytes;
    decltype(&llsa_work_list_len) work_list_len;
    decltype(&llsa_fine_chunk_for) fine_chunk_for;
    decltype(&llsa_attn_bwd_workspace_bytes) attn_bwd_workspace_bytes;
    decltype(&llsa_attn_bwd) attn_bwd;
    decltype(&llsa_gather_rows) gather_rows;
    bool device;                          // false: the CPU emulation build the tests install

    Library(const std::map<std::string, uintptr_t>& at_, bool device_) : device(device_) {
        auto get = [&](const char* name, auto& fn) { fn = reinterpret_cast<std::decay_t<decltype(fn)>>(at_.at(name)); };
        get("llsa_last_error_string", last_error_string);
        get("llsa_pool_pyramid_fwd", pool_pyramid_fwd);
        get("llsa_topk_dense_tiles", topk_dense_tiles);
        get("llsa_topk_sparse_tiles", topk_sparse_tiles);
        get("llsa_topk_cascade_tiles", topk_cascade_tiles);
        get("llsa_topk_cascade_max_parents", topk_cascade_max_parents);
        get("llsa_attn_fwd", attn_fwd);
        get("llsa_attn_fwd_lists", attn_fwd_lists);
        get("llsa_attn_fwd_selects", attn_fwd_selects);
        get("llsa_transpose_indices_multi", transpose_indices_multi);
        get("llsa_transpose_one_launch", transpose_one_launch);
        get("llsa_transpose_nested_bytes", transpose_nested_bytes);
        get("llsa_work_list_len", work_list_len);
        get("llsa_fine_chunk_for", fine_chunk_for);
        get("llsa_attn_bwd_workspace_bytes", attn_bwd_workspace_bytes);
        get("llsa_attn_bwd", attn_bwd);
        get("llsa_gather_rows", gather_rows);
    }
    void check(int rc, const char* what) const {
        if (rc != 0) fail(Failure::kLibrary, std::string(what) + " failed (" + std::to_string(rc) + "): " + last_error_string());
    }
    void on_device(const Tensor& t) const {
        if (device && !t.is_cuda())
            fail(Failure::kRuntime, "llsa_amd runs on an AMD GPU only (got a CPU tensor); there is no CPU implementation");
    }
    void* stream(const Tensor& t) const {
        return device ? static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream()) : nullptr;
    }
};

std::string text_of(at::IntArrayRef v) {
    std::string s = "(";
    for (size_t i = 0; i < v.size(); i++) s += (i ? ", " : "") + std::to_string(v[i]);
    return s + ")";
}

bool strides_multiple(at::IntArrayRef st, int64_t m) {
    for (size_t i = 0; i + 1 < st.size(); i++)
        if (st[i] % m != 0) return false;
    return true;
}
// Whether no two elements of such a tensor share memory (an expanded one's do): every dimension steps over all that the smaller steps span.
bool own_places(const std::array<int64_t, 4>& sizes, const std::array<int64_t, 4>& st) {
    std::array<std::pair<int64_t, int64_t>, 4> dims;          // step, entries
    for (int i = 0; i < 4; i++) dims[i] = {sizes[i] > 1 ? st[i] : 0, sizes[i]};
    std::sort(dims.begin(), dims.end());
    int64_t span = 1;
    for (const auto& [step, n] : dims) {
        if (n > 1 && step < span) return false;
        span += step * (n - 1);
    }
    return true;
}
// last stride 1 and every row 16-byte aligned: what the kernels' 16-byte loads need
bool rows_ok(const Tensor& t) {
    return t.stride(-1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && strides_multiple(t.strides(), 8);
}
Tensor as_rows(const Tensor& t) { return rows_ok(t) ? t : t.contiguous(); }
// a tensor as the kernels need it, wherever and with whatever strides a caller or a saved-tensor hook has put it
Tensor restored(const Tensor& t, bool contiguous = false) {
    const bool usable = !t.defined() || (rows_ok(t) && (!contiguous || t.is_contiguous()));
    return usable ? t : t.clone(at::MemoryFormat::Contiguous);
}

int64_t align_up(int64_t n, int64_t a) { return (n + a - 1) / a * a; }

// What torch.autograd.Function refuses for the operators written in Python, an operator whose node is native has to refuse itself:
// inputs that carry a tangent (the kernels have no forward-mode rule; without this the result would carry none, which reads
// as a derivative of zero) and torch.func's transforms, whose tensors have no data.
void refuse_transforms(std::initializer_list<const Tensor*> inputs) {
    const c10::DispatchKeySet active = c10::impl::tls_local_dispatch_key_set().included_;
    if (active.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || active.has(c10::DispatchKey::FuncTorchDynamicLayerBackMode))
        fail(Failure::kRuntime, "llsa_amd operators do not work under functorch transforms (vmap, grad, jvp, jacrev, ...)");
    for (const Tensor* t : inputs)
        if (t != nullptr && t->_fw_grad(/*level=*/0).defined())
            fail(Failure::kNotImplemented, "llsa_amd operators have no jvp function: forward mode AD is not supported");
}
const Tensor* address(const std::optional<Tensor>& t) { return t.has_value() ? &*t : nullptr; }

// ---------------------------------------------------------------------------------------
// The second stream of a device, and the two events that tie it to the caller's.  The events are a thread's own: a wait
// refers to the last record before it in issue order, so a thread may record them again in its next call.
// ---------------------------------------------------------------------------------------
struct SideStream {
    hipEvent_t ready = nullptr, done = nullptr;
    explicit SideStream() {
        if (hipEventCreateWithFlags(&ready, hipEventDisableTiming) != hipSuccess || hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess)
            fail(Failure::kRuntime, "llsa_amd: cannot create an event");
    }
};
constexpr int kMaxDevices = 64;
hipStream_t side_stream(int device) {
    static std::mutex mutex;
    static std::array<hipStream_t, kMaxDevices> streams{};
    std::lock_guard<std::mutex> lock(mutex);
    if (streams.at(device) == nullptr) streams.at(device) = c10::hip::getStreamFromPool(false, static_cast<c10::DeviceIndex>(device)).stream();
    return streams[device];
}
SideStream& side_events(int device) {
    static thread_local std::array<std::unique_ptr<SideStream>, kMaxDevices> events;
    if (!events.at(device)) events.at(device) = std::make_unique<SideStream>();
    return *events[device];
}
void hip_check(hipError_t e) {
    if (e != hipSuccess) fail(Failure::kRuntime, std::string("llsa_amd: ") + hipGetErrorString(e));
}

// ---------------------------------------------------------------------------------------
// Where everything the forward produces lives: one arena (bytes), every section contiguous (B*H, ...) and 256-byte aligned.
// Level 0 is the tokens themselves, level l = 1..L the pooled levels (n[l] = N / 16^l tokens each).
// ---------------------------------------------------------------------------------------
constexpr int kL = LLSA_MAX_LEVELS;
struct Layout {
    int64_t n[kL + 2];
    int L, chunk;
    bool rows;                                              // the forward reads q and v as rows (no gradients wanted)
    int32_t topk[kL];
    int64_t pq[kL + 1], pk[kL + 1], pv[kL + 1];             // pooled rows, index = level
    int64_t qr, kr, vr;                                     // operand tiles of the tokens
    int64_t pkr[kL + 1], pvr[kL + 1], pvt[kL + 1];          // and of the pooled levels
    int64_t sel[kL], off[kL], flat[kL], inv[kL], work = -1; // sel[0]: fine blocks per query block, sel[l]: blocks of level l per group of 16^(l+1) queries
    int64_t lse, bytes;
    int64_t nested_bytes = 0;                               // scratch of the lists made from those of the level above: of the forward only, not in the arena
    int64_t dpk[kL + 1], dpv[kL + 1], ws, ws_bytes = 0, bwd_bytes;       // the backward's arena

    Layout(const Library& lib, int64_t B, int64_t H, int64_t N, const std::vector<int64_t>& topks, bool grad) {
        const int64_t BH = B * H;
        L = static_cast<int>(topks.size());
        n[0] = N;
        for (int l = 1; l < L + 2; l++) n[l] = n[l - 1] / 16;
        for (int l = 0; l < L; l++) topk[l] = static_cast<int32_t>(topks[l]);
        int64_t o = 0;
        auto take = [&](int64_t per_bh, bool on = true) -> int64_t {
            if (!on) return -1;
            const int64_t at = o;
            o = align_up(o + BH * std::max<int64_t>(per_bh, 0), 256);      // (a topk below 1 is the library's to reject)
            return at;
        };
        for (int l = 1; l <= L; l++) pq[l] = take(n[l] * 128);
        // (the selection reads the keys as tiles: rows of k and v are wanted only where the next pooling pass starts from them)
        for (int l = 1; l <= L; l++) pk[l] = take(n[l] * 128, l % 2 == 0 && l < L);
        for (int l = 1; l <= L; l++) pv[l] = take(n[l] * 128, l % 2 == 0 && l < L);
        // Without gradients the forward reads q and v as rows, and the pooling pass writes no tiles of them: 8 x 65536 tokens of one level 683 -> 660 us, 96 x
        // 4096 143 -> 132, 6 x 65536 of two levels 214 -> 199, 3 x 49152 193.0 -> 191.2.  But a wave then starts with rows that are further away and have to be
        // rotated, which a short pass waits for: 8 x 16384 53.4 / 54.9, 15 x 7168 57.4 / 58.9, 24 x 4096 50.8 / 51.0, 6 x 1024 16.6 / 16.8; 2 x 65536 196.2 / 193.3.
        // With the norm and the rotation both, even up to 200000 tokens (tiles / rows, 24 x 7168 89.3 / 90.7, 12 x 16384 96.6 / 96.3, 192 x 1024 61.8 / 63.7;  without
        // either 84.8 / 79.1, 90.3 / 83.4, 55.9 / 49.5), less beyond (96 x 4096 137.3 / 126.8);  8 heads of (B,N,H,64) views, whose rows lie 1 KB
        // apart, with the rotation 433 / 445 at 49152 tokens, topk 64/32, 156 / 158 at 32768, 32/16.
        rows = !grad && BH * N > (int64_t(1) << 17);
        qr = take(n[1] * 2048, !rows);
        kr = take(n[1] * 2048);
        vr = take(n[1] * 2048, !rows);
        for (int l = 1; l <= L; l++) {
            pkr[l] = take(n[l + 1] * 2048);
            pvr[l] = take(n[l + 1] * 2048, grad);
            pvt[l] = take(n[l + 1] * 2048);
        }
        for (int l = 0; l < L; l++) sel[l] = take(4 * n[l + 1] * topk[l]);
        lse = take(4 * N, !rows);
        chunk = lib.fine_chunk_for(static_cast<int>(B), static_cast<int>(H), static_cast<int>(N), topk[0]);
        if (grad) {
            for (int l = 0; l < L; l++) {
                off[l] = take(4 * (n[l + 1] + 1));
                flat[l] = take(4 * n[l + 1] * topk[l]);
                inv[l] = take(4 * n[l + 1] * topk[l], l > 0);
            }
            work = take(4 * lib.work_list_len(static_cast<int>(n[1]), static_cast<int>(n[1]), topk[0], chunk));
            // (lists too long for one launch are made from those of the level above, which the selection is nested in)
            const int m = static_cast<int>(n[1]), b = static_cast<int>(B), h = static_cast<int>(H);
            if (L > 1 && !lib.transpose_one_launch(m, m, topk[0], b, h)) nested_bytes = std::max<int64_t>(lib.transpose_nested_bytes(m, m, topk[1], b, h), 0);
        }
        bytes = o;
        o = 0;
        if (grad) {
            ws_bytes = lib.attn_bwd_workspace_bytes(static_cast<int>(B), static_cast<int>(H), static_cast<int>(N), topk, L);
            for (int l = 1; l <= L; l++) {
                dpk[l] = take(n[l] * 128);
                dpv[l] = take(n[l] * 128);
            }
        }
        ws = o;
        bwd_bytes = o + ws_bytes;
    }
};

// ---------------------------------------------------------------------------------------
// backward node
// ---------------------------------------------------------------------------------------
struct LlsaBackward : public Node {
    std::shared_ptr<Library> lib;
    std::optional<Layout> lay;
    int64_t B, H, N;
    std::array<int64_t, 4> sq, sk, sv;
    double eps;
    bool has_gq = false, has_gk = false;
    at::ScalarType type_gq = at::kFloat, type_gk = at::kFloat;
    // (everything kept is a SavedVariable: saved-tensor hooks -- offloading, the non-reentrant checkpoint -- see all of it)
    SavedVariable arena, o, freq, gq, gk, q, k;
    bool released = false;

    std::string name() const override { return "LlsaBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        released = true;
        for (SavedVariable* s : {&arena, &o, &freq, &gq, &gk, &q, &k}) s->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        return in_engine([&] { return run(grads[0]); });
    }
    Tensor unpack_arena() const {
        const Tensor t = restored(arena.unpack(), true);
        if (t.scalar_type() != at::kByte || t.numel() != lay->bytes)
            fail(Failure::kRuntime, "llsa_amd: a saved-tensor hook returned another tensor than it was given");
        return t;
    }
    variable_list run(const Tensor& grad_out) {
        if (released) fail(Failure::kRuntime, torch::autograd::ERR_BACKWARD_TWICE);
        // (before the autograd keys are left out: a hook may run the forward again)
        const Tensor saved = unpack_arena(), out = restored(o.unpack(shared_from_this()));
        const Tensor fr = restored(freq.unpack(), true), wq = gq.unpack(), wk = gk.unpack();
        const Tensor qs = restored(q.unpack()), ks = restored(k.unpack());
        at::AutoDispatchBelowADInplaceOrView below;
        c10::OptionalDeviceGuard guard(lib->device ? std::optional<at::Device>(out.device()) : std::nullopt);
        const Tensor d = as_rows(grad_out.defined() ? grad_out : at::zeros_like(out));
        const auto opts = out.options();
        const std::array<int64_t, 4> shape{B, H, N, 64};
        auto like = [&](const std::array<int64_t, 4>& st) {  // gradients have the layout of their primals when the 8-byte stores allow it and no rows meet
            return strides_multiple(st, 4) && st[3] == 1 && own_places(shape, st) ? at::empty_strided(shape, st, opts) : at::empty(shape, opts);
        };
        Tensor dq = like(sq), dk = like(sk), dv = like(sv);
        const Tensor W = at::empty({lay->bwd_bytes}, opts.dtype(at::kByte));
        char* const a0 = static_cast<char*>(saved.data_ptr());
        char* const w0 = static_cast<char*>(W.data_ptr());
        const Layout& y = *lay;
        llsa_attn_bwd_args a{};
        a.dout = d.data_ptr(); a.sdob = d.stride(0); a.sdoh = d.stride(1); a.sdon = d.stride(2);
        a.o = out.data_ptr(); a.sob = out.stride(0); a.soh = out.stride(1); a.son = out.stride(2);
        a.lse = reinterpret_cast<const float*>(a0 + y.lse);
        a.qr = a0 + y.qr; a.kr = a0 + y.kr; a.vr = a0 + y.vr;
        auto ints = [&](int64_t at) { return reinterpret_cast<const int32_t*>(a0 + at); };
        a.idx = ints(y.sel[0]); a.off = ints(y.off[0]); a.flat = ints(y.flat[0]); a.work = ints(y.work);
        a.dq = dq.data_ptr(); a.sdqb = dq.stride(0); a.sdqh = dq.stride(1); a.sdqn = dq.stride(2);
        a.dk = dk.data_ptr(); a.sdkb = dk.stride(0); a.sdkh = dk.stride(1); a.sdkn = dk.stride(2);
        a.dv = dv.data_ptr(); a.sdvb = dv.stride(0); a.sdvh = dv.stride(1); a.sdvn = dv.stride(2);
        float w = 1.f;
        for (int l = 1; l <= y.L; l++) {
            llsa_bwd_level& lv = a.lvl[l - 1];
            w *= 16.f;
            lv.kr = a0 + y.pkr[l]; lv.vr = a0 + y.pvr[l];
            lv.dk = w0 + y.dpk[l]; lv.dv = w0 + y.dpv[l];
            // llsa_l1 keeps the reference's quirk: its pooled path is differentiated with weight 1
            // (sparse_attention_res_1.py:388-389) although the forward uses token_weight
            lv.w = w; lv.gw = y.L == 1 ? 1.f : w;
            if (l < y.L) {
                lv.sel = ints(y.sel[l]); lv.off = ints(y.off[l]); lv.inv = ints(y.inv[l]); lv.T = y.topk[l];
            }
        }
        a.workspace = w0 + y.ws; a.workspace_bytes = y.ws_bytes;
        if (fr.defined()) a.freq_dq = a.freq_dk = fr.data_ptr();
        a.B = static_cast<int32_t>(B); a.H = static_cast<int32_t>(H); a.N = static_cast<int32_t>(N); a.T = y.topk[0]; a.levels = y.L;
        a.fold_pooled = 1; a.chunk = y.chunk;
        Tensor dgq, dgk, P;
        if (wq.defined() || wk.defined()) {                  // back through the qk-norm, inside the kernels that write dq and dk
            const auto f32 = opts.dtype(at::kFloat);
            const int64_t rows = B * H * (N / 16);
            P = at::empty({2 * rows * 64}, f32);
            auto norm = [&](llsa_norm_back& nb, const Tensor& gamma, const Tensor& x, int64_t at) {
                const Tensor dg = at::empty({64}, f32);
                nb.x = x.data_ptr(); nb.sxb = x.stride(0); nb.sxh = x.stride(1); nb.sxn = x.stride(2);
                nb.gamma = gamma.data_ptr<float>();
                nb.dgamma = dg.data_ptr<float>();
                nb.partials = P.data_ptr<float>() + at;
                nb.eps = static_cast<float>(eps);
                return dg;
            };
            if (wq.defined()) dgq = norm(a.norm_q, wq, qs, 0);
            if (wk.defined()) dgk = norm(a.norm_k, wk, ks, rows * 64);
        }
        lib->check(lib->attn_bwd(&a, lib->stream(out)), "attn_bwd");
        if (dgq.defined()) dgq = dgq.to(type_gq);
        if (dgk.defined()) dgk = dgk.to(type_gk);
        variable_list r{dq, dk, dv};
        if (has_gq) r.push_back(dgq);
        if (has_gk) r.push_back(dgk);
        return r;
    }
};

bool wants_grad(const std::optional<Tensor>& t) { return t.has_value() && t->requires_grad(); }

// forward(q, k, v, topks, freq, gamma_q, gamma_k, eps) -> o
//
// topks: one entry per pooled level, (topk1, topk2, ...): the fine blocks a query block keeps, then the blocks of
// pooled level 1, 2, ... its ancestor groups keep; one entry is llsa_l1, two are llsa_l2.
// gamma_q / gamma_k ((64,) or none): RMS-normalise q / k over the head dimension first (the qk-norm of the reference's
// attention processor), inside the pooling pass; they receive gradients.
Tensor attend(const std::shared_ptr<Library>& lib, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, std::vector<int64_t> topks,
              const std::optional<Tensor>& freq_in, const std::optional<Tensor>& gq_in, const std::optional<Tensor>& gk_in, double eps) {
    // (a recorded graph would hold the allocations and none of the launches)
    if (torch::jit::tracer::isTracing()) fail(Failure::kRuntime, "llsa_amd attention operators cannot be recorded by torch.jit.trace");
    refuse_transforms({&q_in, &k_in, &v_in, address(freq_in), address(gq_in), address(gk_in)});
    for (const Tensor* t : {&q_in, &k_in, &v_in}) {
        lib->on_device(*t);
        if (t->scalar_type() != at::kBFloat16)
            fail(Failure::kNotImplemented, "llsa_amd attention kernels are bf16 only (got torch." + std::string(torch::getTHPDtype(t->scalar_type())->name) + ")");
    }
    if (q_in.dim() != 4 || q_in.size(3) != 64) fail(Failure::kNotImplemented, "llsa_amd attention kernels need (B,H,N,64) tensors (got " + text_of(q_in.sizes()) + ")");
    if (k_in.sizes() != q_in.sizes() || v_in.sizes() != q_in.sizes()) fail(Failure::kValue, "self-attention only: q, k, v must have the same shape");
    for (const Tensor* t : {&k_in, &v_in, address(freq_in)})  // (a kernel that follows a pointer into other memory faults the GPU)
        if (t != nullptr && t->device() != q_in.device()) fail(Failure::kValue, "q, k, v and the rope table must be on one device");
    const int64_t B = q_in.size(0), H = q_in.size(1), N = q_in.size(2);
    const int L = static_cast<int>(topks.size());
    if (L < 1 || L > kL) fail(Failure::kValue, "1 to " + std::to_string(kL) + " pooled levels (got " + std::to_string(L) + ")");
    int64_t mult = 64, per = 16;
    for (int l = 0; l < L; l++) mult *= 16;
    if (N % mult != 0)
        fail(Failure::kValue, "llsa_l" + std::to_string(L) + " needs a token count that is a multiple of " + std::to_string(mult) + " (got " + std::to_string(N) + ")");
    for (int l = 0; l < L; l++, per *= 16) topks[l] = std::min(topks[l], N / per);

    const bool grad = at::GradMode::is_enabled() && (q_in.requires_grad() || k_in.requires_grad() || v_in.requires_grad() || wants_grad(gq_in) || wants_grad(gk_in));
    Tensor o, arena, freq, q, k, gq, gk;
    std::shared_ptr<LlsaBackward> node;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        c10::OptionalDeviceGuard guard(lib->device ? std::optional<at::Device>(q_in.device()) : std::nullopt);
        if (freq_in.has_value()) {
            if (freq_in->scalar_type() != at::kBFloat16 || freq_in->dim() != 2 || freq_in->size(0) != N || freq_in->size(1) != 64)
                fail(Failure::kValue, "rope table must be bf16 (N, 64)");
            freq = restored(*freq_in, true);                 // (read in 16-byte pieces; a table may start anywhere in its storage)
        }
        const Tensor v = as_rows(v_in);
        q = as_rows(q_in);
        k = as_rows(k_in);
        if (gq_in.has_value()) gq = gq_in->to(q.device(), at::kFloat).contiguous();
        if (gk_in.has_value()) gk = gk_in->to(q.device(), at::kFloat).contiguous();
        for (const Tensor* g : {&gq, &gk})
            if (g->defined() && g->numel() != 64) fail(Failure::kValue, "qk-norm weights must have 64 entries");
        const Layout y(*lib, B, H, N, topks, grad);
        const int64_t* n = y.n;
        arena = at::empty({y.bytes}, q.options().dtype(at::kByte));
        Tensor scratch;                                      // (goes at the end of this block, when the caller's stream waits for all that uses it)
        if (y.nested_bytes > 0) scratch = at::empty({y.nested_bytes}, arena.options());
        o = strides_multiple(q.strides(), 4) ? at::empty_like(q) : at::empty(q.sizes(), q.options());
        char* const a0 = static_cast<char*>(arena.data_ptr());
        auto pa = [&](int64_t at) -> void* { return at < 0 ? nullptr : a0 + at; };
        auto ints = [&](int64_t at) { return static_cast<int32_t*>(pa(at)); };
        auto lev = [&](const int64_t* list, int l) -> void* { return l <= L ? pa(list[l]) : nullptr; };      // section of pooled level l (none beyond the last)
        void* const stream = lib->stream(q);
        const int b = static_cast<int>(B), h = static_cast<int>(H);

        // The pyramid.  One pass over q, k, v gives the rows of levels 1 and 2 and the tiles of levels 0, 1, 2; every
        // further pass starts from the rows of level 2p and gives rows and tiles of levels 2p + 1 and 2p + 2.
        llsa_pool_item it[3];
        for (int l0 = 0; l0 < L; l0 += 2) {
            for (int i = 0; i < 3; i++) {                    // q, k, v
                llsa_pool_item& p = it[i];
                p = llsa_pool_item{};
                const int64_t* rows = i == 0 ? y.pq : i == 1 ? y.pk : y.pv;
                p.n = static_cast<int32_t>(n[l0]);
                p.y1 = lev(rows, l0 + 1);
                p.y2 = lev(rows, l0 + 2);
                if (l0 == 0) {
                    const Tensor& x = i == 0 ? q : i == 1 ? k : v;
                    p.x = x.data_ptr(); p.sxb = x.stride(0); p.sxh = x.stride(1); p.sxn = x.stride(2);
                    p.rope = i < 2 && freq.defined();
                    p.xr = pa(i == 0 ? y.qr : i == 1 ? y.kr : y.vr);
                    p.stream = grad;
                    const Tensor& g = i == 0 ? gq : gk;
                    if (i < 2 && g.defined()) {
                        p.gamma = g.data_ptr<float>();
                        p.eps = static_cast<float>(eps);
                    }
                } else {
                    p.x = pa(rows[l0]); p.sxb = H * n[l0] * 64; p.sxh = n[l0] * 64; p.sxn = 64;
                }
                if (i == 1) {
                    p.y1r = lev(y.pkr, l0 + 1);
                    p.y2r = lev(y.pkr, l0 + 2);
                }
                if (i == 2) {
                    p.y1r = lev(y.pvr, l0 + 1); p.y1t = lev(y.pvt, l0 + 1);
                    p.y2r = lev(y.pvr, l0 + 2); p.y2t = lev(y.pvt, l0 + 2);
                }
            }
            lib->check(lib->pool_pyramid_fwd(it, 3, l0 == 0 && freq.defined() ? freq.data_ptr() : nullptr, b, h, stream), "pool_pyramid");
        }

        // Selection, coarse to fine: a dense top-k over the coarsest level's tokens (each of them is a block of the level
        // below), then level by level among the blocks under the parent's selection.
        int first = L - 1;               // the first parent-guided selection still to do
        // (without gradients nobody else reads the selection of a short sequence: every wave of the forward makes its own)
        const bool selects = !grad && !y.rows && lib->attn_fwd_selects(b, h, static_cast<int>(N), y.topk[0], L) != 0;
        if (selects) {
            first = 0;
        } else if (L >= 2 && n[L] <= lib->topk_cascade_max_parents() && (n[L] <= 64 || (B * H * n[L] < 800 && y.topk[L - 1] > 4))) {
            // The dense selection rides in the workgroups of the first parent-guided one: one launch less.  More than 64 parent tokens cost every
            // workgroup more than sixteen rows of them cost a wave of their own launch: two launches / one, us, by groups over all heads
            //   (topk 8/8) 256 (65536 tokens) 13.1 / 10.8;  384 (32768) 12.3 / 11.2;  576 (49152) 14.0 / 13.2;  1024 (65536) 15.5 / 16.2;  1536 17.6 / 20.4;
            //   1920 (49152) 19.8 / 23.9;  (16/16) 576 17.5 / 16.6;  1024 19.4 / 20.1;  1536 22.8 / 25.6;  (64/32) 576 32.8 / 31.3;  1152 41.4 / 43.6
            //   (8/4), one wave a group: 128 (32768) 11.1 / 13.4;  576 12.9 / 14.6;  1536 13.2 / 16.9
            lib->check(lib->topk_cascade_tiles(pa(y.pq[L]), pa(y.pkr[L]), ints(y.sel[L - 1]), pa(y.pq[L - 1]), pa(y.pkr[L - 1]), ints(y.sel[L - 2]), b, h,
                                               static_cast<int>(n[L - 1]), y.topk[L - 2], y.topk[L - 1], stream),
                       "topk_cascade");
            first = L - 2;
        } else {
            lib->check(lib->topk_dense_tiles(pa(y.pq[L]), pa(y.pkr[L]), ints(y.sel[L - 1]), b, h, static_cast<int>(n[L]), y.topk[L - 1], 1, stream),
                       "gen_sparse_indices");
        }
        for (int l = first; l > 0; l--)
            lib->check(lib->topk_sparse_tiles(pa(y.pq[l]), pa(y.pkr[l]), ints(y.sel[l]), ints(y.sel[l - 1]), b, h, static_cast<int>(n[l]), y.topk[l - 1],
                                              y.topk[l], stream),
                       "compute_topk_indices_sparse");

        // The lists of the backward (the transposed selections of all levels).  Where one launch can make them all they ride in
        // the attention kernel's (llsa_lists_ride) or, if they are too many for that or have more than 8160 key blocks, follow it on the same
        // stream; the several kernels per level of the longest sequences run on a second
        // stream beside the attention kernel: the attention kernel is issued first (the GPU is waiting for it), and an
        // event recorded before it lets the second stream start as soon as the selection is done.  With few tokens over all
        // heads the event calls cost more than the overlap saves: everything then goes to the one stream.  Training steps, us, behind / beside: two levels
        // 16/16, 2 x 131072 552 / 534;  6 x 131072 1481 / 1462;  3 x 196608 1289 / 1268;  6 x 262144 even (3829 / 3827);  32/16, 3 x 65536 488 / 476;  64/32, 3 x
        // 49152 649 / 626;  three levels, 6 x 262144, 2883 / 2876;  one level, topk 32, 6 x 65536 2247 / 2205.  (One launch on the second stream
        // gains nothing either: two levels of 131072 tokens, topk 8, behind / beside, us: 1 head 279 / 293, 2 heads 458 / 468, 6 heads
        // 1293 / 1297, 12 heads 2457 / 2449.)
        const bool beside = grad && lib->device && B * H * N >= (int64_t(1) << 17) &&
                            !lib->transpose_one_launch(static_cast<int>(n[1]), static_cast<int>(n[1]), y.topk[0], b, h);
        const int dev = beside ? q.device().index() : 0;
        if (beside) hip_check(hipEventRecord(side_events(dev).ready, static_cast<hipStream_t>(stream)));

        llsa_attn_fwd_args f{};
        f.qr = pa(y.qr); f.kr = pa(y.kr); f.vt = pa(y.vr); f.idx = ints(y.sel[0]);
        if (selects) f.pq = pa(y.pq[1]);
        if (y.rows) {
            f.q = q.data_ptr(); f.sqb = q.stride(0); f.sqh = q.stride(1); f.sqn = q.stride(2);
            f.v = v.data_ptr(); f.svb = v.stride(0); f.svh = v.stride(1); f.svn = v.stride(2);
            if (freq.defined()) f.freq_q = freq.data_ptr();
            if (gq.defined()) {
                f.gamma_q = gq.data_ptr<float>();
                f.eps_q = static_cast<float>(eps);
            }
        }
        f.o = o.data_ptr(); f.sob = o.stride(0); f.soh = o.stride(1); f.son = o.stride(2);
        f.lse = static_cast<float*>(pa(y.lse));
        f.B = b; f.H = h; f.N = static_cast<int32_t>(N); f.T = y.topk[0]; f.levels = L;
        float w = 1.f;
        for (int l = 1; l <= L; l++) {
            llsa_fwd_level& lv = f.lvl[l - 1];
            w *= 16.f;
            lv.kr = pa(y.pkr[l]); lv.vt = pa(y.pvt[l]); lv.w = w;
            if (l < L) {
                lv.sel = ints(y.sel[l]);
                lv.T = y.topk[l];
            }
        }
        llsa_transpose_job jobs[kL];
        for (int l = 0; l < L && grad; l++) {
            const int32_t m = static_cast<int32_t>(n[l + 1]);
            jobs[l] = llsa_transpose_job{ints(y.sel[l]), ints(y.off[l]), ints(y.flat[l]), l == 0 ? ints(y.work) : nullptr, l == 0 ? nullptr : ints(y.inv[l]),
                                         m, m, y.topk[l], l == 0 ? y.chunk : 1, l == 0 && scratch.defined() ? scratch.data_ptr() : nullptr};
        }
        if (grad && !beside) lib->check(lib->attn_fwd_lists(&f, jobs, L, stream), "attn_fwd");
        else lib->check(lib->attn_fwd(&f, stream), "attn_fwd");

        if (grad) {
            if (beside) {
                void* lists = side_stream(dev);
                hip_check(hipStreamWaitEvent(static_cast<hipStream_t>(lists), side_events(dev).ready, 0));       // (the arena is older than the selection, so this covers it too)
                lib->check(lib->transpose_indices_multi(jobs, L, b, h, lists), "transpose_indices");
                // (and neither the arena nor the scratch is handed out again before the second stream is done)
                hip_check(hipEventRecord(side_events(dev).done, static_cast<hipStream_t>(lists)));
                hip_check(hipStreamWaitEvent(static_cast<hipStream_t>(stream), side_events(dev).done, 0));
            }
            node = std::shared_ptr<LlsaBackward>(new LlsaBackward, torch::autograd::deleteNode);
            node->lib = lib;
            node->lay = y;
            node->B = B; node->H = H; node->N = N;
            for (int i = 0; i < 4; i++) {
                node->sq[i] = q.stride(i);
                node->sk[i] = k.stride(i);
                node->sv[i] = v.stride(i);
            }
            node->eps = eps;
            if (gq.defined()) {
                node->has_gq = true;
                node->type_gq = gq_in->scalar_type();
            }
            if (gk.defined()) {
                node->has_gk = true;
                node->type_gk = gk_in->scalar_type();
            }
        }
    }
    if (node) {
        variable_list inputs{q_in, k_in, v_in};
        if (node->has_gq) inputs.push_back(*gq_in);
        if (node->has_gk) inputs.push_back(*gk_in);
        node->set_next_edges(torch::autograd::collect_next_edges(inputs));
        torch::autograd::set_history(o, node);
        // (in the state the caller is in: a hook that packs a tensor may compute with it)
        node->arena = SavedVariable(arena, false);
        node->o = SavedVariable(o, true);
        if (freq.defined()) node->freq = SavedVariable(freq, false);
        if (gq.defined()) {                                  // (q and k themselves are needed again only by the backward of the qk-norm)
            node->gq = SavedVariable(gq.is_same(*gq_in) ? *gq_in : gq, false);
            node->q = SavedVariable(q.is_same(q_in) ? q_in : q, false);
        }
        if (gk.defined()) {
            node->gk = SavedVariable(gk.is_same(*gk_in) ? *gk_in : gk, false);
            node->k = SavedVariable(k.is_same(k_in) ? k_in : k, false);
        }
    }
    return o;
}

// The blocks the forward that produced `out` chose, finest first: int32 views of the arena its autograd node holds.
std::vector<Tensor> selection(const Tensor& out) {
    auto* node = dynamic_cast<LlsaBackward*>(out.grad_fn().get());
    if (node == nullptr) fail(Failure::kValue, "not an output of a fused operator that records its backward");
    if (node->released) fail(Failure::kRuntime, torch::autograd::ERR_BACKWARD_TWICE);
    const Layout& y = *node->lay;
    const Tensor arena = node->unpack_arena();
    std::vector<Tensor> r;
    for (int l = 0; l < y.L; l++) {
        const int64_t count = node->B * node->H * y.n[l + 1] * y.topk[l];
        r.push_back(arena.narrow(0, y.sel[l], 4 * count).view(at::kInt).view({node->B, node->H, y.n[l + 1], y.topk[l]}));
    }
    return r;
}

// ---------------------------------------------------------------------------------------
// token permutation
// ---------------------------------------------------------------------------------------
Tensor gather(const Library& lib, const Tensor& x_in, const Tensor& index_in) {
    if (x_in.dim() != 3) fail(Failure::kValue, "gather_tokens expects (B, N, C)");
    lib.on_device(x_in);
    lib.on_device(index_in);
    at::AutoDispatchBelowADInplaceOrView below;
    c10::OptionalDeviceGuard guard(lib.device ? std::optional<at::Device>(x_in.device()) : std::nullopt);
    const int64_t B = x_in.size(0), N = x_in.size(1), C = x_in.size(2), es = x_in.element_size();
    if (C * es % 16 != 0) fail(Failure::kNotImplemented, "rows of " + std::to_string(C * es) + " bytes: a multiple of 16 is needed");
    const bool in_place = x_in.stride(2) == 1 && x_in.stride(1) == C && x_in.stride(0) * es % 16 == 0 && reinterpret_cast<uintptr_t>(x_in.data_ptr()) % 16 == 0;
    const Tensor x = in_place ? x_in : x_in.contiguous();
    const Tensor index = index_in.scalar_type() == at::kInt && index_in.is_contiguous() ? index_in : index_in.to(at::kInt).contiguous();
    const int64_t n_out = index.numel();
    Tensor y = at::empty({B, n_out, C}, x.options());
    if (B == 0 || n_out == 0) return y;
    lib.check(lib.gather_rows(x.data_ptr(), y.data_ptr(), static_cast<const int32_t*>(index.data_ptr()), static_cast<int>(B), static_cast<int>(n_out),
                              static_cast<int>(N), static_cast<int>(C * es), x.stride(0) * es, y.stride(0) * es, lib.stream(x)),
              "gather_tokens");
    return y;
}

struct PermuteBackward : public Node {
    std::shared_ptr<Library> lib;
    SavedVariable inv;
    std::string name() const override { return "PermuteTokensBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        inv.reset_data();
        released = true;
    }
    bool released = false;
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        return in_engine([&]() -> variable_list {
            if (released) fail(Failure::kRuntime, torch::autograd::ERR_BACKWARD_TWICE);
            if (!grads[0].defined()) return {Tensor()};
            const Tensor index = inv.unpack();
            if (!index.defined()) fail(Failure::kValue, "permute_tokens: the gradient needs the inverse permutation");
            return {gather(*lib, grads[0], index)};
        });
    }
};

Tensor permute(const std::shared_ptr<Library>& lib, const Tensor& x, const Tensor& perm, const std::optional<Tensor>& inv) {
    refuse_transforms({&x});
    Tensor y = gather(*lib, x, perm);
    if (at::GradMode::is_enabled() && x.requires_grad()) {
        auto node = std::shared_ptr<PermuteBackward>(new PermuteBackward, torch::autograd::deleteNode);
        node->lib = lib;
        if (inv.has_value()) node->inv = SavedVariable(*inv, false);
        node->set_next_edges(torch::autograd::collect_next_edges(x));
        torch::autograd::set_history(y, node);
    }
    return y;
}

}  // namespace

PYBIND11_MODULE(_llsa_host, m) {
    m.doc() = "host side of llsa_amd's fused operators";
    py::class_<Library, std::shared_ptr<Library>>(m, "Library").def(py::init<const std::map<std::string, uintptr_t>&, bool>());
    m.def("set_library_error", [](py::object type) { g_library_error = type.release().ptr(); });
    m.attr("abi_version") = LLSA_ABI_VERSION;
    m.def("attend", torch::wrap_pybind_function([](const std::shared_ptr<Library>& lib, const Tensor& q, const Tensor& k, const Tensor& v,
                                                   const std::vector<int64_t>& topks, const std::optional<Tensor>& freq,
                                                   const std::optional<Tensor>& gq, const std::optional<Tensor>& gk, double eps) {
        return without_interpreter([&] { return attend(lib, q, k, v, topks, freq, gq, gk, eps); });
    }));
    m.def("selection", torch::wrap_pybind_function([](const Tensor& out) { return without_interpreter([&] { return selection(out); }); }));
    m.def("gather", torch::wrap_pybind_function([](const std::shared_ptr<Library>& lib, const Tensor& x, const Tensor& index) {
        return without_interpreter([&] { return gather(*lib, x, index); });
    }));
    m.def("permute", torch::wrap_pybind_function([](const std::shared_ptr<Library>& lib, const Tensor& x, const Tensor& perm, const std::optional<Tensor>& inv) {
        return without_interpreter([&] { return permute(lib, x, perm, inv); });
    }));
}
