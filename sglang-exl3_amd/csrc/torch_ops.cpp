// Native entry of the operators that programs call eagerly, one per layer:
// exl3_gemv, exl3_linear_cat, exl3_linear_part and exl3_gate_up_swiglu.
//
// A one-token call is bound by its host path: from Python (operator wrapper,
// checks, two ctypes calls, stream and device queries) exl3_gemv took 20.5 us
// on the host for a kernel of 12 (4096 x 14336) or 4 us (512 x 512), three shards
// through exl3_linear_cat 29.2.  Here the usual call - dense tensors of the
// current device, a workspace that is large enough, no graph capture - goes
// from the dispatcher to the C ABI: 5.4 and 6.6 us.  Every other call
// (autograd inputs, strided or misaligned tensors, the first call of a shape,
// capture, and whatever is refused) goes to the operator's *_general twin, the
// Python implementation, so its checks, messages and bookkeeping stay the only ones.
//
// The operators are defined in Python; this file adds the kernels of two
// dispatch keys.  The library that holds the C ABI is bound by address, so that it
// is loaded once.
#include <ATen/ATen.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/library.h>

#include <map>
#include <mutex>
#include <utility>

#include "../../include/sglang_exl3_amd.h"

namespace {

struct Abi {
    decltype(&exl3_gemv) gemv;
    decltype(&exl3_gemv_workspace_size) gemv_ws;
    decltype(&exl3_linear_cat_part) cat;
    decltype(&exl3_linear_cat_workspace_size) cat_ws;
    decltype(&exl3_gate_up_swiglu) gate_up;
    decltype(&exl3_gate_up_workspace_size) gate_up_ws;
} abi;

// The buffers of ops.workspace(), by (device, stream); never destroyed (the
// allocator may be gone before this library at exit).
std::mutex& ws_lock() {
    static std::mutex* m = new std::mutex;
    return *m;
}
std::map<std::pair<int64_t, int64_t>, at::Tensor>& ws_map() {
    static auto* m = new std::map<std::pair<int64_t, int64_t>, at::Tensor>;
    return *m;
}

void keep_workspace(const at::Tensor& ws, int64_t stream) {
    std::lock_guard<std::mutex> g(ws_lock());
    ws_map()[{ws.get_device(), stream}] = ws;
}

// Stream and workspace of a call on `dev`; false: the general path.
struct Launch {
    hipStream_t stream;
    at::Tensor ws;
    bool get(int64_t dev, size_t need) {
        const auto s = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev);
        stream = s.stream();
        hipStreamCaptureStatus cap;
        if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return false;
        std::lock_guard<std::mutex> g(ws_lock());
        const auto it = ws_map().find({dev, (int64_t)reinterpret_cast<intptr_t>(stream)});
        if (it == ws_map().end() || (size_t)it->second.numel() < need) return false;
        ws = it->second;
        return true;
    }
};

bool on_current(const at::Tensor& x) {
    int dev = -1;
    return x.is_cuda() && hipGetDevice(&dev) == hipSuccess && dev == x.get_device();
}
const uint16_t* u16(const at::Tensor& t) { return static_cast<const uint16_t*>(t.const_data_ptr()); }
bool at_bytes(const at::Tensor& t, uintptr_t a) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % a == 0; }

// A half vector of at least `len` elements, packed and dword-aligned.
bool half_vec(const at::Tensor& t, int64_t dev, int64_t len) {
    return t.is_cuda() && t.get_device() == dev && t.scalar_type() == at::kHalf && t.is_contiguous() &&
           t.numel() >= len && at_bytes(t, 4);
}
// Trellis words [k/16, n/16, 16 K], packed and 16-byte aligned.
bool trellis_ok(const at::Tensor& t, int64_t dev, int64_t k, int64_t K) {
    return t.is_cuda() && t.get_device() == dev && t.scalar_type() == at::kShort && t.dim() == 3 &&
           t.is_contiguous() && t.size(0) * 16 == k && t.size(1) > 0 && t.size(1) < (1 << 24) && t.size(2) == 16 * K && at_bytes(t, 16);
}
// Rows of x (m x k); 0: the general path.
int64_t rows_of(const at::Tensor& x, bool bf16_too) {
    if (x.dim() < 2 || !on_current(x) || !x.is_contiguous() || !at_bytes(x, 4)) return 0;
    if (x.scalar_type() != at::kHalf && !(bf16_too && x.scalar_type() == at::kBFloat16)) return 0;
    const int64_t k = x.size(-1);
    const int64_t m = k > 0 ? x.numel() / k : 0;
    return k <= (1 << 24) && m <= (1 << 24) ? m : 0;
}
// A failed call may have left counters behind: clean the buffer, then let the
// general path raise (or run).
bool done(int rc, Launch& l) {
    if (rc == EXL3_OK) return true;
    l.ws.zero_();
    return false;
}

// ------------------------------------------------------------------ exl3_gemv

using GemvFn = at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&, c10::SymInt,
                          bool, c10::SymInt);
struct Gemv {
    static constexpr const char *name = "sglang_exl3::exl3_gemv", *general = "sglang_exl3::exl3_gemv_general";
};

at::Tensor gemv(const at::Tensor& x, const at::Tensor& trellis, const at::Tensor& suh, const at::Tensor& svh,
                int64_t K, bool mcg, int64_t mmode) {
    const int64_t m = rows_of(x, false), k = m ? x.size(-1) : 0, dev = m ? x.get_device() : -1;
    if (m >= 1 && m <= 64 && (mmode == 0 || mmode == 1) && K >= 1 && K <= 8 && trellis_ok(trellis, dev, k, K) &&
        half_vec(suh, dev, k) && half_vec(svh, dev, trellis.size(1) * 16)) {
        const int64_t n = trellis.size(1) * 16;
        Launch l;
        if (l.get(dev, abi.gemv_ws((int)m, (int)k, (int)n, (int)K, 1))) {
            at::Tensor y = at::empty({m, n}, x.options());
            if (done(abi.gemv(u16(x), trellis.const_data_ptr<int16_t>(), u16(suh), u16(svh),
                              static_cast<uint16_t*>(y.mutable_data_ptr()), (int)m, (int)k, (int)n, (int)K,
                              mcg ? 1 : 2, l.ws.mutable_data_ptr(), l.ws.numel(), l.stream),
                     l))
                return y;
        }
    }
    static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(Gemv::general, "").typed<GemvFn>();
    return h.call(x, trellis, suh, svh, K, mcg, mmode);
}

// ------------------------------------------------------------ exl3_linear_cat

using CatFn = at::Tensor(const at::Tensor&, at::TensorList, at::TensorList, at::TensorList, c10::SymInt, c10::SymInt,
                         bool);
struct Cat {
    static constexpr const char *name = "sglang_exl3::exl3_linear_cat",
                                *general = "sglang_exl3::exl3_linear_cat_general";
};
using PartFn = at::Tensor(const at::Tensor&, at::TensorList, at::TensorList, at::TensorList, c10::SymInt, c10::SymInt,
                          bool, c10::SymInt);
struct Part {
    static constexpr const char *name = "sglang_exl3::exl3_linear_part",
                                *general = "sglang_exl3::exl3_linear_part_general";
};

// Weights from `first` on, side by side [m, n] or (apart) packed one after the
// other [m * n]; an undefined tensor: the general path.
at::Tensor linear_weights(const at::Tensor& x, at::TensorList trellis, at::TensorList suh, at::TensorList svh,
                          int64_t K, int64_t codebook, bool out_bf16, int64_t first, bool apart) {
    const int64_t m = rows_of(x, true), k = m ? x.size(-1) : 0, dev = m ? x.get_device() : -1;
    const size_t count = trellis.size();
    bool ok = m >= 1 && count >= 1 && count <= 4 && suh.size() == count && svh.size() == count && K >= 1 && K <= 8 &&
              codebook >= 0 && codebook <= 2 && first >= 0 && first < (int64_t)count;
    const int16_t* tr[4];
    const uint16_t *su[4], *sv[4];
    int ns[4];
    int64_t n = 0;
    for (size_t j = 0; ok && j < count; ++j) {
        ok = trellis_ok(trellis[j], dev, k, K) && half_vec(suh[j], dev, k) &&
             half_vec(svh[j], dev, trellis[j].size(1) * 16);
        if (!ok) break;
        tr[j] = trellis[j].const_data_ptr<int16_t>();
        su[j] = u16(suh[j]);
        sv[j] = u16(svh[j]);
        ns[j] = (int)(trellis[j].size(1) * 16);
        if ((int64_t)j >= first) n += ns[j];
    }
    Launch l;
    if (ok && l.get(dev, abi.cat_ws((int)m, (int)k, ns, (int)count, (int)K))) {
        const auto options = x.options().dtype(out_bf16 ? at::kBFloat16 : at::kHalf);
        at::Tensor y = apart ? at::empty({m * n}, options) : at::empty({m, n}, options);
        if (done(abi.cat(x.const_data_ptr(), x.scalar_type() == at::kBFloat16 ? 1 : 0, tr, su, sv, ns, (int)count,
                         (int)first, apart ? 1 : 0, y.mutable_data_ptr(), out_bf16 ? 1 : 0, (int)m, (int)k, (int)K,
                         (int)codebook, l.ws.mutable_data_ptr(), l.ws.numel(), l.stream),
                 l))
            return y;
    }
    return {};
}

at::Tensor linear_cat(const at::Tensor& x, at::TensorList trellis, at::TensorList suh, at::TensorList svh, int64_t K,
                      int64_t codebook, bool out_bf16) {
    at::Tensor y = linear_weights(x, trellis, suh, svh, K, codebook, out_bf16, 0, false);
    if (y.defined()) return y;
    static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(Cat::general, "").typed<CatFn>();
    return h.call(x, trellis, suh, svh, K, codebook, out_bf16);
}

at::Tensor linear_part(const at::Tensor& x, at::TensorList trellis, at::TensorList suh, at::TensorList svh, int64_t K,
                       int64_t codebook, bool out_bf16, int64_t first) {
    at::Tensor y = linear_weights(x, trellis, suh, svh, K, codebook, out_bf16, first, true);
    if (y.defined()) return y;
    static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(Part::general, "").typed<PartFn>();
    return h.call(x, trellis, suh, svh, K, codebook, out_bf16, first);
}

// -------------------------------------------------------- exl3_gate_up_swiglu

using GateUpFn = at::Tensor(const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&,
                            const at::Tensor&, const at::Tensor&, c10::SymInt, c10::SymInt, double);
struct GateUp {
    static constexpr const char *name = "sglang_exl3::exl3_gate_up_swiglu",
                                *general = "sglang_exl3::exl3_gate_up_swiglu_general";
};

at::Tensor gate_up(const at::Tensor& x, const at::Tensor& suh, const at::Tensor& gt, const at::Tensor& gsv,
                   const at::Tensor& ut, const at::Tensor& usv, int64_t K, int64_t codebook, double limit) {
    const int64_t m = rows_of(x, false), k = m ? x.size(-1) : 0, dev = m ? x.get_device() : -1;

    if (m >= 1 && K >= 1 && K <= 8 && codebook >= 0 && codebook <= 2 && limit >= 0.0 && trellis_ok(gt, dev, k, K) &&
        trellis_ok(ut, dev, k, K) && gt.size(1) == ut.size(1) && half_vec(suh, dev, k) &&
        half_vec(gsv, dev, gt.size(1) * 16) && half_vec(usv, dev, gt.size(1) * 16)) {
        const int64_t n = gt.size(1) * 16;
        Launch l;
        if (l.get(dev, abi.gate_up_ws((int)m, (int)k, (int)n, (int)K))) {
            at::Tensor y = at::empty({m, n}, x.options());
            if (done(abi.gate_up(u16(x), u16(suh), gt.const_data_ptr<int16_t>(), u16(gsv),
                                 ut.const_data_ptr<int16_t>(), u16(usv), static_cast<uint16_t*>(y.mutable_data_ptr()),
                                 (int)m, (int)k, (int)n, (int)K, (int)codebook, (float)limit, l.ws.mutable_data_ptr(),
                                 l.ws.numel(), l.stream),
                     l))
                return y;
        }
    }
    static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(GateUp::general, "").typed<GateUpFn>();
    return h.call(x, suh, gt, gsv, ut, usv, K, codebook, limit);
}

// -------------------------------------------------------------------- autograd

bool wants_grad(const at::Tensor& t) { return t.requires_grad(); }
bool wants_grad(at::TensorList ts) {
    for (const auto& t : ts)
        if (t.requires_grad()) return true;
    return false;
}
bool wants_grad(const c10::SymInt&) { return false; }
bool wants_grad(bool) { return false; }
bool wants_grad(double) { return false; }

// Inputs that require grad take the general operator (its autograd kernel);
// others go below autograd, to the modes and keys that follow.
template <class Op, class F>
struct Autograd;
template <class Op, class R, class... A>
struct Autograd<Op, R(A...)> {
    static R call(c10::DispatchKeySet ks, A... a) {
        if (c10::GradMode::is_enabled() && (wants_grad(a) || ...)) {
            static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(Op::general, "").template typed<R(A...)>();
            return h.call(a...);
        }
        static const auto h = c10::Dispatcher::singleton().findSchemaOrThrow(Op::name, "").template typed<R(A...)>();
        at::AutoDispatchBelowAutograd below;
        return h.redispatch(ks & c10::after_autograd_keyset, a...);
    }
};

}  // namespace

TORCH_LIBRARY_IMPL(sglang_exl3, CUDA, m) {
    m.impl("exl3_gemv", gemv);
    m.impl("exl3_linear_cat", linear_cat);
    m.impl("exl3_linear_part", linear_part);
    m.impl("exl3_gate_up_swiglu", gate_up);
    m.impl("keep_workspace", keep_workspace);
}

TORCH_LIBRARY_IMPL(sglang_exl3, AutogradCUDA, m) {
    m.impl("exl3_gemv", Autograd<Gemv, GemvFn>::call);
    m.impl("exl3_linear_cat", Autograd<Cat, CatFn>::call);
    m.impl("exl3_linear_part", Autograd<Part, PartFn>::call);
    m.impl("exl3_gate_up_swiglu", Autograd<GateUp, GateUpFn>::call);
}

// The PyTorch that this was built for (EXL3_TORCH_VERSION), looked up in the file
// before it is loaded: another one's ABI need not fit.
extern "C" __attribute__((used)) const char exl3_ops_torch[] = "exl3-ops-torch:" EXL3_TORCH_VERSION;

// Addresses of the C ABI: gemv, its workspace size, linear_cat_part, .., gate_up, ..
extern "C" void exl3_ops_bind(void* const* fn) {
    abi.gemv = reinterpret_cast<decltype(abi.gemv)>(fn[0]);
    abi.gemv_ws = reinterpret_cast<decltype(abi.gemv_ws)>(fn[1]);
    abi.cat = reinterpret_cast<decltype(abi.cat)>(fn[2]);
    abi.cat_ws = reinterpret_cast<decltype(abi.cat_ws)>(fn[3]);
    abi.gate_up = reinterpret_cast<decltype(abi.gate_up)>(fn[4]);
    abi.gate_up_ws = reinterpret_cast<decltype(abi.gate_up_ws)>(fn[5]);
}
