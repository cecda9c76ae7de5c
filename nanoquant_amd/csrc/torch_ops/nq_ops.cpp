// The torch.ops.binary_kernels operators' device implementations in C++: argument checks, output and
// scratch from torch's caching allocator, one call of the C ABI on torch's current stream.
//
// At decode sizes a launch takes a few microseconds and an operator implemented in Python spent 24 us on the
// host per call (dispatch into Python, its checks, ctypes), so eager calls were bound by it: 4096 x 4096,
// r = 1120, one row 23.5 -> 11.7 us a call, a module call of 21 rows on 4096 x 11008 34.7 -> 21.5. These
// implementations take the well-formed calls; a call that fails any check, or a library that has not been
// loaded yet, goes to the general operator of the same schema (namespace nanoquant_amd, implemented in Python),
// which loads the library, handles the empty sizes and raises the documented errors.
//
// The C ABI's functions come in as addresses (nq_ops_bind), so that this file needs no link to the HIP library.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/library.h>

#include <atomic>

#include "../../../include/nq_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// In the order of nq_ops_bind's array.
struct Library {
    decltype(&nq_gemv_workspace_bytes) gemv_bytes;
    decltype(&nq_gemv) gemv;
    decltype(&nq_gemm_onebit_workspace_bytes) onebit_bytes;
    decltype(&nq_gemm_onebit) onebit;
    decltype(&nq_gemm_nanoquant_workspace_bytes) nanoquant_bytes;
    decltype(&nq_gemm_nanoquant) nanoquant;
};
constexpr int kFunctions = 6;
std::atomic<const Library*> g_library{nullptr};

int dtype_code(at::ScalarType t) { return t == at::kHalf ? NQ_F16 : NQ_BF16; }

// A tensor the kernels read where it lies: on `x`'s device, contiguous, of the given type.
bool plain(const Tensor& t, const Tensor& x, at::ScalarType type) {
    return t.device() == x.device() && t.scalar_type() == type && t.is_contiguous();
}

// A 1-D scale of `size` elements, or none.
bool scale_ok(const OptTensor& s, const Tensor& x, int64_t size) {
    return !s.has_value() || (s->dim() == 1 && s->size(0) == size && plain(*s, x, x.scalar_type()));
}

const void* data_of(const OptTensor& t) { return t.has_value() ? t->const_data_ptr() : nullptr; }

Tensor scratch(size_t bytes, const Tensor& x) {
    return at::empty({static_cast<int64_t>(bytes)}, x.options().dtype(at::kByte));
}

nq_stream_t stream_of(const Tensor& x) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device()).stream();
}

template <typename F>
c10::TypedOperatorHandle<F> general(const char* name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<F>();
}

bool one_of(int64_t v, std::initializer_list<int64_t> choices) {
    for (int64_t c : choices)
        if (v == c) return true;
    return false;
}

Tensor gemv(const Tensor& x, const Tensor& s_in, const Tensor& v_words, const OptTensor& s_mid, const Tensor& u_words,
            const Tensor& s_out, int64_t th1, int64_t th2, int64_t rpw1, int64_t rpw2, int64_t acc1, int64_t acc2,
            int64_t pipe1, int64_t pipe2) {
    const Library* lib = g_library.load(std::memory_order_acquire);
    const auto type = x.scalar_type();
    if (lib && (type == at::kHalf || type == at::kBFloat16) && x.is_cuda() && x.is_contiguous() && x.dim() >= 1 &&
        x.numel() > 0 && v_words.dim() == 2 && u_words.dim() == 2 && s_out.dim() == 1) {
        const int64_t n = x.size(-1), r = v_words.size(0), m = s_out.size(0), batch = x.numel() / n;
        if (m > 0 && plain(s_in, x, type) && s_in.numel() == n && plain(s_out, x, type) && plain(v_words, x, at::kInt) &&
            v_words.size(1) == (n + 31) / 32 && plain(u_words, x, at::kInt) && u_words.size(0) == m &&
            u_words.size(1) == (r + 31) / 32 && scale_ok(s_mid, x, r) && one_of(th1, {64, 128, 256}) &&
            one_of(th2, {64, 128, 256}) && one_of(rpw1, {1, 2, 4, 8}) && one_of(rpw2, {1, 2, 4, 8}) &&
            one_of(acc1, {1, 2}) && one_of(acc2, {1, 2}) && one_of(pipe1, {1, 2, 4, 8, 16}) &&
            one_of(pipe2, {1, 2, 4, 8, 16})) {
            const c10::DeviceGuard guard(x.device());
            std::vector<int64_t> shape = x.sizes().vec();
            shape.back() = m;
            Tensor y = at::empty(shape, x.options());
            const size_t bytes = lib->gemv_bytes(batch, n, r, m);
            const Tensor ws = scratch(bytes, x);
            if (lib->gemv(dtype_code(type), x.const_data_ptr(), s_in.const_data_ptr(),
                          static_cast<const uint32_t*>(v_words.const_data_ptr()), data_of(s_mid),
                          static_cast<const uint32_t*>(u_words.const_data_ptr()), s_out.const_data_ptr(),
                          y.mutable_data_ptr(), batch, n, r, m, ws.mutable_data_ptr(), bytes, stream_of(x)) == NQ_OK)
                return y;
        }
    }
    static const auto op = general<decltype(gemv)>("nanoquant_amd::nanoquant_dyn_forward");
    return op.call(x, s_in, v_words, s_mid, u_words, s_out, th1, th2, rpw1, rpw2, acc1, acc2, pipe1, pipe2);
}

// What both GEMM operators ask of one stage: x [M, K] against Marlin words of K inputs and `out` outputs, with the
// reference's workspace size.
bool stage_ok(const Tensor& x, int64_t K, const Tensor& words, const OptTensor& scale_in, const OptTensor& scale_out,
              const Tensor& workspace) {
    if (words.dim() != 2 || !plain(words, x, at::kInt) || words.size(0) * 16 != K || words.size(1) % 32 != 0) return false;
    const int64_t out = words.size(1) * 2;
    return out > 0 && scale_ok(scale_in, x, K) && scale_ok(scale_out, x, out) && workspace.numel() >= out / 128 * 32;
}

bool x_ok(const Library* lib, const Tensor& x) {
    return lib && (x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16) && x.is_cuda() && x.is_contiguous() &&
           x.dim() == 2 && x.size(0) > 0 && x.size(1) > 0;
}

Tensor onebit(const Tensor& x, const Tensor& weight, const OptTensor& s_in, const OptTensor& s_out, const Tensor& workspace) {
    const Library* lib = g_library.load(std::memory_order_acquire);
    if (x_ok(lib, x) && stage_ok(x, x.size(1), weight, s_in, s_out, workspace)) {
        const c10::DeviceGuard guard(x.device());
        const int64_t M = x.size(0), K = x.size(1), N = weight.size(1) * 2;
        Tensor y = at::empty({M, N}, x.options());
        const size_t bytes = lib->onebit_bytes(M, K, N);
        const Tensor part = bytes ? scratch(bytes, x) : Tensor();
        if (lib->onebit(dtype_code(x.scalar_type()), x.const_data_ptr(), static_cast<const uint32_t*>(weight.const_data_ptr()),
                        data_of(s_in), data_of(s_out), y.mutable_data_ptr(), M, K, N,
                        bytes ? part.mutable_data_ptr() : nullptr, bytes, stream_of(x)) == NQ_OK)
            return y;
    }
    static const auto op = general<decltype(onebit)>("nanoquant_amd::marlin_onebit_forward");
    return op.call(x, weight, s_in, s_out, workspace);
}

Tensor nanoquant(const Tensor& x, const Tensor& v_words, const Tensor& u_words, const OptTensor& s_g, const OptTensor& s_l,
                 const OptTensor& s_h, const Tensor& workspace) {
    const Library* lib = g_library.load(std::memory_order_acquire);
    if (x_ok(lib, x) && stage_ok(x, x.size(1), v_words, s_g, s_l, workspace) &&
        stage_ok(x, v_words.size(1) * 2, u_words, std::nullopt, s_h, workspace)) {
        const c10::DeviceGuard guard(x.device());
        const int64_t M = x.size(0), n = x.size(1), r_pad = v_words.size(1) * 2, m = u_words.size(1) * 2;
        const Tensor imm = at::empty({M, r_pad}, x.options());
        Tensor y = at::empty({M, m}, x.options());
        const size_t bytes = lib->nanoquant_bytes(M, n, r_pad, m);
        const Tensor part = bytes ? scratch(bytes, x) : Tensor();
        if (lib->nanoquant(dtype_code(x.scalar_type()), x.const_data_ptr(),
                           static_cast<const uint32_t*>(v_words.const_data_ptr()),
                           static_cast<const uint32_t*>(u_words.const_data_ptr()), data_of(s_g), data_of(s_l), data_of(s_h),
                           imm.mutable_data_ptr(), y.mutable_data_ptr(), M, n, r_pad, m,
                           bytes ? part.mutable_data_ptr() : nullptr, bytes, stream_of(x)) == NQ_OK)
            return y;
    }
    static const auto op = general<decltype(nanoquant)>("nanoquant_amd::marlin_nanoquant_forward");
    return op.call(x, v_words, u_words, s_g, s_l, s_h, workspace);
}

}  // namespace

// The addresses of the C ABI's functions, in Library's order, once the HIP library is loaded (the table lives as long
// as the process). Returns 0, or 1 where the count is not this build's.
extern "C" int nq_ops_bind(void* const* functions, int count) {
    if (count != kFunctions) return 1;
    static Library library;
    library.gemv_bytes = reinterpret_cast<decltype(library.gemv_bytes)>(functions[0]);
    library.gemv = reinterpret_cast<decltype(library.gemv)>(functions[1]);
    library.onebit_bytes = reinterpret_cast<decltype(library.onebit_bytes)>(functions[2]);
    library.onebit = reinterpret_cast<decltype(library.onebit)>(functions[3]);
    library.nanoquant_bytes = reinterpret_cast<decltype(library.nanoquant_bytes)>(functions[4]);
    library.nanoquant = reinterpret_cast<decltype(library.nanoquant)>(functions[5]);
    g_library.store(&library, std::memory_order_release);
    return 0;
}

// Digest of the header that this library was built from, to be compared with nq_header_digest before binding.
extern "C" const char* nq_ops_header_digest(void) { return NQ_HEADER_DIGEST; }

TORCH_LIBRARY_IMPL(binary_kernels, CUDA, m) {
    m.impl("nanoquant_dyn_forward", &gemv);
    m.impl("marlin_onebit_forward", &onebit);
    m.impl("marlin_nanoquant_forward", &nanoquant);
}
