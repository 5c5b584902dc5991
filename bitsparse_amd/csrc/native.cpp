// Native host path of the codec calls and of the MLP block's forward and
// backward: the allocations and the calls into libbitsparse_hip.so and torch
// without the interpreter between the launches.  At the small sizes the host
// work is the whole time (a 128-token block step: 300 us of Python for 60 us
// of kernels).  Every tensor lives on the current stream of its device; a
// backward runs on its forward's stream (autograd sets it).
#include <dlfcn.h>
#include <torch/extension.h>

#include <ATen/core/grad_mode.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <map>
#include <memory>

#include "bitsparse_hip.h"

namespace {

using at::Tensor;

// ---------------------------------------------------------------------------
// libbitsparse_hip.so (the path Python loads, so that both use one library)
// ---------------------------------------------------------------------------
#define BS_FUNCS(F)                                                                                              \
    F(bs_abi_version) F(bs_last_error) F(bs_compress_workspace_bytes) F(bs_compress) F(bs_compress_packed)       \
    F(bs_compress_act) F(bs_amax) F(bs_amax_relu) F(bs_amax_bias_relu) F(bs_quantize_e4m3fn)                     \
    F(bs_quantize_e4m3fn_t) F(bs_widen_e4m3fn) F(bs_decompress) F(bs_decompress_packed)                          \
    F(bs_relu_grad) F(bs_relu2_grad) F(bs_relu2_grad_packed) F(bs_grad_sums_workspace_bytes) F(bs_act_grad_sums) \
    F(bs_col_sum_workspace_bytes) F(bs_col_sum) F(bs_gemm_compressed_b_workspace_bytes) F(bs_gemm_compressed_b)  \
    F(bs_gemm_compressed_b_packed_workspace_bytes) F(bs_gemm_compressed_b_packed)                                \
    F(bs_gemm_compressed_b_fp8_workspace_bytes) F(bs_gemm_compressed_b_fp8) F(bs_gemm_compressed_b_fp8_packed)   \
    F(bs_workspace_amax_slot)
struct Lib {
#define F(name) decltype(&::name) name = nullptr;
    BS_FUNCS(F)
#undef F
} L;

void init(const std::string& path)
{
    void* h = dlopen(path.c_str(), RTLD_NOW);
    if (h == nullptr) throw py::import_error(std::string("bitsparse_amd: ") + dlerror());
    Lib lib;
#define F(name)                                                      \
    lib.name = reinterpret_cast<decltype(&::name)>(dlsym(h, #name)); \
    if (lib.name == nullptr) throw py::import_error("bitsparse_amd: " #name " missing in " + path);
    BS_FUNCS(F)
#undef F
    // the header compiled in here and the library are built apart: one version, or shifted arguments
    if (lib.bs_abi_version() != BS_ABI_VERSION)
        throw py::import_error("bitsparse_amd/_native was built for ABI " + std::to_string(BS_ABI_VERSION) + ", " + path +
                               " has " + std::to_string(lib.bs_abi_version()) + "; rebuild both");
    L = lib;
}

void check(int rc, const char* what)
{
    if (rc == BS_OK) return;
    const char* msg = L.bs_last_error();
    if (rc == BS_ERR_INVALID) TORCH_CHECK_VALUE(false, what, ": ", msg);
    const py::gil_scoped_acquire gil;       // (a C++ node's backward has no interpreter lock)
    py::set_error(py::module_::import("bitsparse_amd._lib").attr("BitsparseHipError"),
                  (std::string(what) + " failed (" + std::to_string(rc) + "): " + msg).c_str());
    throw py::error_already_set();
}

void* stream_of(const Tensor& t)
{
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream();
}

template <typename T>
T* ptr(const Tensor& t)
{
    return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}
void* raw(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
std::optional<Tensor> optional(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kBFloat16: return 0;
    case at::kFloat8_e4m3fn: return 1;
    case at::kFloat8_e5m2: return 2;
    default: TORCH_CHECK_TYPE(false, "BitsparseTensor supports bfloat16 and FP8 (e4m3fn/e5m2) values");
    }
}

Tensor empty(at::IntArrayRef shape, const Tensor& like, at::ScalarType t)
{
    return at::empty(shape, like.options().dtype(t));
}

// ---------------------------------------------------------------------------
// per-(device, stream) workspace of the single-pass compress and the amax
// ---------------------------------------------------------------------------
constexpr int64_t kEpochLimit = (int64_t(1) << 30) - 1;

// Zero-initialised device scratch with an epoch counter.  Each compress / amax
// call takes a fresh epoch; status words written under older epochs are
// ignored by the kernels, so the buffer never needs clearing between calls.
// When the counter wraps the buffer is zeroed again.
//
// Threads: every use of a workspace is in a call from Python and holds the
// interpreter lock throughout (Biased's backward does not, and has no use of
// one), which is what keeps a sequence that passes an amax through the
// workspace whole, as long as nothing in it runs Python.  So a sequence
// allocates its outputs first, then calls `prepare`, and makes no call into
// torch from there to its last launch; the workspace's own torch calls leave
// the thread's dispatch modes out.  (No mutex: a thread in a mode's Python code
// gives the lock away, and one waiting for the mutex would not.)
struct Workspace {
    explicit Workspace(c10::Device d) : device(d)
    {
        const NoPython guard;
        buf = at::zeros({0}, at::device(d).dtype(at::kByte));
    }
    c10::Device device;
    Tensor buf;
    int64_t epoch = 0;

    struct NoPython {
        c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKeySet(
            {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::PythonDispatcher})};
    };

    // A graph would record the zero fills below instead of running them, and
    // what is captured with an epoch is refused anyway.
    void refuse_capture() const
    {
        if (!device.is_cuda()) return;
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        const hipError_t e = hipStreamIsCapturing(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream(), &cs);
        if (e != hipSuccess) (void)hipGetLastError();
        TORCH_CHECK_VALUE(e != hipSuccess || cs == hipStreamCaptureStatusNone,
                          "bitsparse_amd: compress and amax cannot be captured into a HIP graph: their device state is "
                          "tagged with a per-call epoch that a replay would repeat");
    }
    void ensure(int64_t nbytes)
    {
        if (buf.numel() >= nbytes) return;
        refuse_capture();
        const NoPython guard;
        // grow geometrically; the old contents (amax slot, status words of
        // earlier epochs) move along and the new tail is zero, so epochs
        // already handed out stay meaningful
        const int64_t size = std::max<int64_t>({nbytes, 2 * buf.numel(), 1 << 16});
        Tensor n = at::zeros({size}, buf.options());
        if (buf.numel()) n.narrow(0, 0, buf.numel()).copy_(buf);
        buf = n;
    }
    // room for a sequence: `nbytes`, and `epochs` that the wrap -- which zeroes
    // the buffer, amax slot included -- does not fall between
    void prepare(int64_t nbytes, int64_t epochs)
    {
        ensure(nbytes);
        if (epoch + epochs <= kEpochLimit) return;
        refuse_capture();
        const NoPython guard;
        buf.zero_();
        epoch = 0;
    }
    int64_t next_epoch(int64_t reserve)
    {
        prepare(0, reserve);
        return ++epoch;
    }
    int64_t nbytes() const { return buf.numel(); }
    const uint64_t* slot() const { return L.bs_workspace_amax_slot(buf.data_ptr(), nbytes()); }
    int64_t fallback_count() const
    {
        if (buf.numel() < 12) return 0;
        return buf.narrow(0, 8, 4).view(at::kInt).item<int>();
    }
};

std::shared_ptr<Workspace> workspace(int dev)
{
    static auto* all = new std::map<std::pair<int, void*>, std::shared_ptr<Workspace>>();   // (freed by the process)
    if (dev < 0) dev = c10::hip::current_device();
    void* st = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev).stream();
    auto& w = (*all)[{dev, st}];
    if (!w) w = std::make_shared<Workspace>(c10::Device(c10::kCUDA, dev));
    return w;
}
Workspace& ws_of(const Tensor& t) { return *workspace(t.get_device()); }

// amax of a bf16 tensor (of its relu, of relu(x + bias)) under the next epoch
// of a prepared workspace
constexpr int64_t kAmaxBytes = 256;
int64_t amax(const Tensor& x, bool relu, const Tensor& bias, Workspace& w)
{
    const int64_t e = ++w.epoch;
    void* st = stream_of(x);
    if (bias.defined())
        check(L.bs_amax_bias_relu(x.data_ptr(), x.size(0), x.size(1), bias.data_ptr(), w.buf.data_ptr(), w.nbytes(), e,
                                  st), "bs_amax_bias_relu");
    else
        check((relu ? L.bs_amax_relu : L.bs_amax)(x.data_ptr(), x.numel(), w.buf.data_ptr(), w.nbytes(), e, st),
              "bs_amax");
    return e;
}

// ---------------------------------------------------------------------------
// codec
// ---------------------------------------------------------------------------
// The TensorBuffer's cursor for one compress.  No offset: the buffer was just
// reset, the values start at 0 (no tensor was filled for it) and the kernel
// writes the start that the BitsparseTensor keeps.  In place: the start is a
// snapshot and the cursor tensor itself advances.
struct Cursor {
    Tensor in, next, start, start_out;
    Cursor(const std::optional<Tensor>& offset, bool in_place, bool packed, const Tensor& like)
    {
        TORCH_CHECK_VALUE(offset || !in_place, "no cursor to advance in place");
        if (offset) in = in_place ? offset->clone() : *offset;
        next = in_place ? *offset : empty({1}, like, at::kLong);
        start = in;
        // (a packed run starts at the cursor rounded up)
        if (packed || !offset) start = start_out = empty({1}, like, at::kLong);
    }
};

int64_t tiles(int64_t M, int64_t N) { return ((M + 63) / 64) * ((N + 63) / 64); }

// (bitmask, prefix, start of the values, advanced cursor, dense codes, scale):
// bs_compress / bs_compress_packed of a contiguous dense into a TensorBuffer's
// storage; quantize: of a bf16 dense's e4m3fn codes, with its amax first
std::tuple<Tensor, Tensor, Tensor, Tensor, std::optional<Tensor>, std::optional<Tensor>>
compress(const Tensor& dense, const Tensor& vals, const std::optional<Tensor>& offset, bool in_place,
         const Tensor& err, bool packed, bool quantize, bool dense_out)
{
    const c10::DeviceGuard guard(dense.device());
    const int64_t M = dense.size(0), N = dense.size(1), T = tiles(M, N);
    Workspace& w = ws_of(dense);
    Tensor q, scale;
    if (quantize) {
        if (dense_out) q = empty({M, N}, dense, at::kFloat8_e4m3fn);
        scale = empty({}, dense, at::kFloat);
    }
    Tensor bitmask = empty({T * 512}, dense, at::kByte), prefix = empty({T + 1}, dense, at::kUInt32);
    Cursor c(offset, in_place, packed, dense);
    w.prepare(std::max(kAmaxBytes, L.bs_compress_workspace_bytes(M, N)), 2);
    const int64_t amax_epoch = quantize ? amax(dense, false, Tensor(), w) : 0, epoch = ++w.epoch;
    const uint64_t* slot = quantize ? w.slot() : nullptr;
    if (packed) {
        check(L.bs_compress_packed(dense.data_ptr(), dtype_code(dense.scalar_type()), M, N, quantize, slot, amax_epoch,
                                   ptr<float>(scale), raw(q), ptr<uint8_t>(bitmask), ptr<uint32_t>(prefix),
                                   vals.data_ptr(), vals.numel(), ptr<int64_t>(c.in), ptr<int64_t>(c.next),
                                   ptr<int64_t>(c.start_out), ptr<int32_t>(err), w.buf.data_ptr(), w.nbytes(), epoch, 0,
                                   nullptr, stream_of(dense)), "bs_compress_packed");
    } else {
        check(L.bs_compress(dense.data_ptr(), dtype_code(dense.scalar_type()), M, N, quantize, slot, amax_epoch,
                            ptr<float>(scale), raw(q), ptr<uint8_t>(bitmask), ptr<uint32_t>(prefix), vals.data_ptr(),
                            vals.numel(), ptr<int64_t>(c.in), 0, ptr<int64_t>(c.next), ptr<int64_t>(c.start_out), 1,
                            ptr<int32_t>(err), w.buf.data_ptr(), w.nbytes(), epoch, stream_of(dense)), "bs_compress");
    }
    return {bitmask, prefix, c.start, c.next, optional(q), optional(scale)};
}

void decompress(const Tensor& vals, at::ScalarType stored, bool packed, const Tensor& bitmask, const Tensor& prefix,
                const Tensor& offset, const Tensor& out, int64_t first_m_tile, int64_t grid_n, int64_t K,
                int64_t batch_rows, int64_t num_tiles, bool square, double k, const std::optional<Tensor>& scale)
{
    const c10::DeviceGuard guard(out.device());
    check((packed ? L.bs_decompress_packed : L.bs_decompress)(
              vals.data_ptr(), dtype_code(stored), vals.numel(), ptr<uint8_t>(bitmask), ptr<uint32_t>(prefix),
              ptr<int64_t>(offset), out.data_ptr(), first_m_tile, grid_n, K, batch_rows, num_tiles, square, (float)k,
              scale ? ptr<float>(*scale) : nullptr, stream_of(out)), "bs_decompress");
}

// ---------------------------------------------------------------------------
// fp8 operands
// ---------------------------------------------------------------------------
struct Fp8 {
    Tensor codes, scale;
};

Fp8 rows_like(const Tensor& x) { return {empty(x.sizes(), x, at::kFloat8_e4m3fn), empty({}, x, at::kFloat)}; }
Fp8 transposed_like(const Tensor& x)
{
    return {empty({x.size(1), x.size(0)}, x, at::kFloat8_e4m3fn), empty({}, x, at::kFloat)};
}

// codes of x, whose amax the workspace holds under `amax_epoch`
void quantize_rows(const Tensor& x, const Fp8& o, int64_t amax_epoch, Workspace& w)
{
    check(L.bs_quantize_e4m3fn(x.data_ptr(), x.numel(), o.codes.data_ptr(), ptr<float>(o.scale), w.buf.data_ptr(),
                               w.nbytes(), amax_epoch, stream_of(x)), "bs_quantize_e4m3fn");
}

// codes of x.T as a row-major matrix (and, `rows` defined, those of x)
void quantize_t(const Tensor& x, const Tensor& rows, const Fp8& t, int64_t amax_epoch, Workspace& w)
{
    check(L.bs_quantize_e4m3fn_t(x.data_ptr(), x.size(0), x.size(1), raw(rows), t.codes.data_ptr(), ptr<float>(t.scale),
                                 w.buf.data_ptr(), w.nbytes(), amax_epoch, stream_of(x)), "bs_quantize_e4m3fn_t");
}

// x as the kernels read it: a bf16 matrix on the GPU (the backward's operands
// come from autograd, whose saved-tensor hooks may hand back anything)
Tensor operand(const Tensor& x)
{
    TORCH_CHECK(x.is_cuda(), "bitsparse_amd runs on a ROCm GPU; got a tensor on ", x.device());
    TORCH_CHECK_TYPE(x.scalar_type() == at::kBFloat16, "expected a bfloat16 tensor, got ", x.scalar_type());
    TORCH_CHECK_VALUE(x.dim() == 2, "expected a matrix, got ", x.dim(), " dimensions");
    return x.contiguous();
}

// to_fp8 of a row-major matrix
Fp8 to_fp8(const Tensor& x)
{
    const Tensor c = operand(x);
    Workspace& w = ws_of(c);
    const Fp8 o = rows_like(c);
    w.prepare(kAmaxBytes, 1);
    quantize_rows(c, o, amax(c, false, Tensor(), w), w);
    return o;
}

// an operand multiplied from the right: column-major codes
Fp8 right_operand(const Tensor& x)
{
    Tensor c = operand(x);
    if (reinterpret_cast<uintptr_t>(c.data_ptr()) & 15) c = c.clone();      // the kernel loads 16 bytes
    Workspace& w = ws_of(c);
    const Fp8 t = transposed_like(c);
    w.prepare(kAmaxBytes, 1);
    quantize_t(c, Tensor(), t, amax(c, false, Tensor(), w), w);
    return {t.codes.t(), t.scale};
}

Tensor fp8_mm(const Fp8& a, const Fp8& b, at::ScalarType out)
{
    return at::_scaled_mm(a.codes, b.codes, a.scale, b.scale, std::nullopt, std::nullopt, out, false);
}

// a gradient in e4m3fn widened to bf16 (exact)
Tensor widened(const Tensor& g)
{
    if (g.scalar_type() != at::kFloat8_e4m3fn) return g;
    Tensor o = empty(g.sizes(), g, at::kBFloat16);
    check(L.bs_widen_e4m3fn(g.data_ptr(), g.numel(), o.data_ptr(), stream_of(g)), "bs_widen_e4m3fn");
    return o;
}

// ---------------------------------------------------------------------------
// the MLP block
// ---------------------------------------------------------------------------
// the compressed activation r of a block
struct Held {
    Tensor vals, bitmask, prefix, start, scale;
    int64_t M, N;
    bool packed, fp8, square;
    double k;
};

// `held`: (values, bitmask, prefix, start, scale), taken out of the list, so
// that they go once the last kernel that reads them is queued
Held take_held(const py::list& held, int64_t M, int64_t N, bool packed, bool fp8, bool square, double k)
{
    Held h{held[0].cast<Tensor>(), held[1].cast<Tensor>(), held[2].cast<Tensor>(), held[3].cast<Tensor>(),
           held[4].is_none() ? Tensor() : held[4].cast<Tensor>(), M, N, packed, fp8, square, k};
    held.attr("clear")();
    return h;
}

// C = A @ op(B), B compressed [K, N]: A row-major (a_layout 1) or A.T
// row-major (0) in `a` with row stride lda; a_scale: A is e4m3fn
Tensor gemm_compressed(const Tensor& a, int64_t M, int64_t K, int64_t lda, int64_t a_layout,
                       const std::optional<Tensor>& a_scale, const Tensor& vals, at::ScalarType stored, bool packed,
                       const Tensor& bitmask, const Tensor& prefix, const Tensor& start, int64_t N, bool square,
                       double k, const std::optional<Tensor>& scale, const std::optional<Tensor>& b_scale_out)
{
    const c10::DeviceGuard guard(a.device());
    Tensor C = empty({M, N}, a, at::kBFloat16);
    const int64_t need =
        a_scale ? L.bs_gemm_compressed_b_fp8_workspace_bytes(M, N, K, a_layout, square || packed)
                : (packed ? L.bs_gemm_compressed_b_packed_workspace_bytes : L.bs_gemm_compressed_b_workspace_bytes)(
                      M, N, K, a_layout);
    const Tensor ws = empty({std::max<int64_t>(need, 0)}, a, at::kByte);
    float* const bs = scale ? ptr<float>(*scale) : nullptr;
    if (a_scale)
        check((packed ? L.bs_gemm_compressed_b_fp8_packed : L.bs_gemm_compressed_b_fp8)(
                  a.data_ptr(), ptr<float>(*a_scale), M, K, lda, a_layout, vals.data_ptr(), dtype_code(stored),
                  vals.numel(), ptr<uint8_t>(bitmask), ptr<uint32_t>(prefix), ptr<int64_t>(start), N, square, (float)k,
                  bs, C.data_ptr(), b_scale_out ? ptr<float>(*b_scale_out) : nullptr, ws.data_ptr(), need,
                  stream_of(a)), "bs_gemm_compressed_b_fp8");
    else
        check((packed ? L.bs_gemm_compressed_b_packed : L.bs_gemm_compressed_b)(
                  a.data_ptr(), M, K, lda, a_layout, vals.data_ptr(), dtype_code(stored), vals.numel(),
                  ptr<uint8_t>(bitmask), ptr<uint32_t>(prefix), ptr<int64_t>(start), N, square, (float)k, bs,
                  C.data_ptr(), ws.data_ptr(), need, stream_of(a)), "bs_gemm_compressed_b");
    return C;
}

// dW2 = g^T act(r)
Tensor down_weight_grad(const Tensor& g, const Tensor& g_scale, const Held& h)
{
    Tensor a = g;
    const int64_t M = g.size(1);
    // rows that overlap (a gradient expanded over the tokens has row stride 0) are copied too
    if (!h.fp8 && (a.stride(1) != 1 || a.stride(0) % 8 != 0 || a.stride(0) < M ||
                   (reinterpret_cast<uintptr_t>(a.data_ptr()) & 15))) {
        a = at::zeros({h.M, (M + 7) / 8 * 8}, g.options());
        a.narrow(1, 0, M).copy_(g);
    }
    return gemm_compressed(a, M, h.M, a.stride(0), 0, h.fp8 ? std::optional<Tensor>(g_scale) : std::nullopt,
                           h.vals, h.fp8 ? at::kFloat8_e4m3fn : at::kBFloat16, h.packed, h.bitmask, h.prefix, h.start,
                           h.N, h.square, h.k, h.fp8 ? std::optional<Tensor>(h.scale) : std::nullopt, std::nullopt);
}

Tensor col_sum(const Tensor& g)
{
    // a graph of this gradient (create_graph), a batch of them (no storage of
    // its own), or a layout the kernel does not take: torch's own sum
    if (at::GradMode::is_enabled() || !g.has_storage() || g.scalar_type() != at::kBFloat16 || !g.is_contiguous() || g.size(1) % 8 != 0 || g.numel() == 0 ||
        (reinterpret_cast<uintptr_t>(g.data_ptr()) & 15) || g.numel() >= (int64_t(1) << 31))
        return g.sum(0);
    const int64_t R = g.size(0), C = g.size(1), need = L.bs_col_sum_workspace_bytes(R, C);
    Tensor out = empty({C}, g, at::kBFloat16), part = empty({need}, g, at::kByte);
    check(L.bs_col_sum(g.data_ptr(), R, C, out.data_ptr(), part.data_ptr(), need, stream_of(g)), "bs_col_sum");
    return out;
}

// The block's y, b2 added, as a node of b2's own: the sum is there already, and
// forward gives y in the shape of the block's input, as a tensor of its own (a
// view refuses detach_()).  b2's gradient needs nothing of the block, so a walk
// for b2 alone leaves the compressed activation to a later one.
struct Biased : torch::autograd::Function<Biased> {
    static Tensor forward(torch::autograd::AutogradContext*, const Tensor& y, const Tensor& /*b2*/,
                          const std::vector<int64_t>& shape)
    {
        return at::_unsafe_view(y, shape);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   const torch::autograd::variable_list& grads)
    {
        const Tensor g = grads[0].reshape({-1, grads[0].size(-1)});
        return {ctx->needs_input_grad(0) ? g : Tensor(), ctx->needs_input_grad(1) ? col_sum(g) : Tensor(), Tensor()};
    }
};

// The activation step inside a block, on its up-projection z, which nothing
// reads afterwards: r = relu(z + bias) compressed, and what the down-projection
// multiplies -- r or (square) k r^2, in bf16 (over z where that leaves a recount
// of z, the look-back's fallback, right: no bias to be added again), or (fp8) as
// e4m3fn codes with their scale, as to_fp8 makes them.
struct Activation {
    Tensor operand, operand_scale, bitmask, prefix, start, next, scale;
};

Activation activate(const Tensor& z, const Tensor& bias, const Tensor& vals, const std::optional<Tensor>& offset,
                    const Tensor& err, bool in_place, bool packed, bool fp8, bool square, double k)
{
    const int64_t M = z.size(0), N = z.size(1), T = tiles(M, N);
    Workspace& w = ws_of(z);
    const Cursor c(offset, in_place, packed, z);
    Activation a;
    a.bitmask = empty({T * 512}, z, at::kByte);
    a.prefix = empty({T + 1}, z, at::kUInt32);
    a.start = c.start;
    a.next = c.next;
    if (fp8) {
        a.scale = empty({}, z, at::kFloat);
        a.operand_scale = square ? empty({}, z, at::kFloat) : a.scale;
        a.operand = empty({M, N}, z, at::kFloat8_e4m3fn);
    } else {
        a.operand = bias.defined() ? at::empty_like(z) : z;
    }
    w.prepare(std::max(kAmaxBytes, L.bs_compress_workspace_bytes(M, N)), 2);
    const int64_t amax_epoch = fp8 ? amax(z, true, bias, w) : 0, epoch = ++w.epoch;
    check(L.bs_compress_act(z.data_ptr(), raw(bias), M, N, square, (float)k, fp8, fp8 ? w.slot() : nullptr, amax_epoch,
                            ptr<float>(a.scale), fp8 ? raw(a.operand) : nullptr,
                            square && fp8 ? ptr<float>(a.operand_scale) : nullptr, fp8 ? nullptr : raw(a.operand),
                            ptr<uint8_t>(a.bitmask), ptr<uint32_t>(a.prefix), vals.data_ptr(), vals.numel(), packed,
                            ptr<int64_t>(c.in), ptr<int64_t>(c.next), ptr<int64_t>(c.start_out), ptr<int32_t>(err),
                            w.buf.data_ptr(), w.nbytes(), epoch, stream_of(z)), "bs_compress_act");
    return a;
}

// The activation's gradient, in place: dz = relu'(.) dh or (square) 2 k r dh,
// and from the pass that writes it the bias gradient (its column sums) and its
// e4m3fn codes, row-major (`rows`) and transposed (`cols`), with their scale,
// each if asked for.  Gives the activation's tensors up once they are read.
struct ActGrad {
    Tensor bias;
    Fp8 rows, cols;
};

ActGrad act_grad(const Tensor& dz, Held& h, bool bias, bool rows, bool cols)
{
    // (the product behind dz may have come in another type, under autocast, or of other operands than the forward's)
    TORCH_CHECK_TYPE(dz.scalar_type() == at::kBFloat16, "the activation's gradient: grad must be bfloat16");
    TORCH_CHECK_VALUE(dz.dim() == 2 && dz.size(0) == h.M && dz.size(1) == h.N && dz.is_contiguous(),
                      "the activation's gradient: grad shape ", dz.sizes(), " != ", at::IntArrayRef({h.M, h.N}));
    const int stored = h.fp8 ? 1 : 0;
    ActGrad o;
    if (bias || rows || cols) {
        Workspace& w = ws_of(dz);
        if (bias) o.bias = empty({h.N}, dz, at::kBFloat16);
        const int64_t bytes = L.bs_grad_sums_workspace_bytes(h.M, h.N);
        const Tensor part = empty({bytes}, dz, at::kByte);
        if (rows) o.rows = cols ? Fp8{empty(dz.sizes(), dz, at::kFloat8_e4m3fn), Tensor()} : rows_like(dz);
        if (cols) o.cols = transposed_like(dz);
        int64_t epoch = 0;
        if (rows || cols) {
            w.prepare(kAmaxBytes, 1);
            epoch = ++w.epoch;
        }
        check(L.bs_act_grad_sums(dz.data_ptr(), h.M, h.N, h.square, h.vals.data_ptr(), stored, h.vals.numel(), h.packed,
                                 ptr<uint8_t>(h.bitmask), ptr<uint32_t>(h.prefix), ptr<int64_t>(h.start), (float)h.k,
                                 ptr<float>(h.scale), raw(o.bias), rows || cols ? w.buf.data_ptr() : nullptr, epoch,
                                 part.data_ptr(), bytes, stream_of(dz)), "bs_act_grad_sums");
        if (cols) {
            quantize_t(dz, o.rows.codes, o.cols, epoch, w);
            o.rows.scale = o.cols.scale;
        } else if (rows) {
            quantize_rows(dz, o.rows, epoch, w);
        }
    } else if (h.square) {
        check((h.packed ? L.bs_relu2_grad_packed : L.bs_relu2_grad)(
                  dz.data_ptr(), h.M, h.N, h.vals.data_ptr(), stored, h.vals.numel(), ptr<uint8_t>(h.bitmask),
                  ptr<uint32_t>(h.prefix), ptr<int64_t>(h.start), (float)h.k, ptr<float>(h.scale), stream_of(dz)),
              "bs_relu2_grad");
    } else {
        check(L.bs_relu_grad(dz.data_ptr(), h.M, h.N, ptr<uint8_t>(h.bitmask), stream_of(dz)), "bs_relu_grad");
    }
    h = Held();
    return o;
}

// y = act(x @ W1.T + b1) @ W2.T + b2 with act(z) = relu(z) or k relu(z)^2 saved
// compressed: the products, quantizations and kernels of the separate nodes
// (matmul, the bias adds, ReluLinear / Relu2Linear), with their roundings.
// What one node adds is what crosses them: the bias, square and codes of the
// down-projection's operand ride on the compress pass, the bias gradient and
// the amax on the activation's gradient, and the fp8 operands of the backward
// products are quantized into the layout those take.  The caller (layers.py)
// has checked the operands.
// -> (y, bitmask, prefix, start of the values, advanced cursor, scale)
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, std::optional<Tensor>>
block_forward(const Tensor& x, const Tensor& W1, const std::optional<Tensor>& b1, const Tensor& W2,
              const std::optional<Tensor>& b2, const Tensor& vals, const std::optional<Tensor>& offset,
              const Tensor& err, bool in_place, bool packed, bool fp8, bool square, double k)
{
    const c10::DeviceGuard guard(x.device());
    Tensor z;
    if (fp8) {
        const Fp8 a = to_fp8(x), b = to_fp8(W1);
        z = fp8_mm(a, {b.codes.t(), b.scale}, at::kBFloat16);
    } else {
        z = at::mm(x, W1.t());
    }
    const Activation a = activate(z, b1.value_or(Tensor()), vals, offset, err, in_place, packed, fp8, square, k);
    z.reset();          // (the down-projection does not need its room)
    Tensor y;
    if (fp8) {
        const Fp8 b = to_fp8(W2);
        y = fp8_mm({a.operand, a.operand_scale}, {b.codes.t(), b.scale}, at::kBFloat16);
    } else {
        y = at::mm(a.operand, W2.t());
    }
    if (b2) y.add_(*b2);
    return {y, a.bitmask, a.prefix, a.start, a.next, optional(a.scale)};
}

// `need` (x, W1, b1, W2 ask for gradients) without those that this walk is not
// after (torch.autograd.grad or backward(inputs=) of some of them): the separate
// nodes' products were left out by the engine itself.
std::vector<bool> asked_for(std::vector<bool> need)
{
    const std::shared_ptr<torch::autograd::Node> node = torch::autograd::get_current_node();
    if (!node || node->name() != "_FFNBlockBackward") return need;
    size_t edge = 0;
    for (size_t i = 0; i < need.size(); i++) {
        if (i == 2 && node->num_outputs() < need.size()) continue;      // no b1, no edge to it
        need[i] = need[i] && node->task_should_compute_output(edge);
        edge++;
    }
    return need;
}

// (dx, dW1, db1, dW2), each where `wanted` and this walk ask for it.  `dh`: the product
// g W2 formed by the caller, where its graph is wanted and the operations here
// would not record one (it is overwritten).
std::vector<std::optional<Tensor>>
block_backward(const Tensor& g, const Tensor& x, const Tensor& W1, const Tensor& W2, const py::list& held, int64_t M,
               int64_t N, bool packed, bool fp8, bool square, double k, const std::optional<at::ScalarType>& grad_dtype,
               const std::vector<bool>& wanted, const std::optional<Tensor>& dh)
{
    const c10::DeviceGuard guard(g.device());
    Held h = take_held(held, M, N, packed, fp8, square, k);
    TORCH_CHECK_VALUE(g.dim() == 2 && g.size(0) == M, "the gradient's rows are not the activation's");
    const std::vector<bool> need = asked_for(wanted);
    const bool need_x = need[0], need_W1 = need[1], need_b1 = need[2], need_W2 = need[3];
    std::vector<std::optional<Tensor>> out(4);
    Fp8 g8;
    if (fp8) g8 = to_fp8(g);
    if (need_W2) out[3] = down_weight_grad(fp8 ? g8.codes : g, g8.scale, h);
    if (!(need_x || need_W1 || need_b1)) return out;
    const Tensor dz = dh ? *dh : fp8 ? fp8_mm(g8, right_operand(W2), at::kBFloat16) : at::mm(g, W2);
    g8 = Fp8();
    const bool sums = need_b1 && !at::GradMode::is_enabled();
    const ActGrad a = act_grad(dz, h, sums, fp8 && need_x, fp8 && need_W1);
    if (need_b1) out[2] = sums ? a.bias : col_sum(dz);
    if (fp8) {
        const at::ScalarType gd = grad_dtype.value_or(at::kFloat8_e4m3fn);
        if (need_x) out[0] = widened(fp8_mm(a.rows, right_operand(W1), gd));
        if (need_W1) out[1] = widened(fp8_mm(a.cols, right_operand(x), gd));
    } else {
        if (need_x) out[0] = at::mm(dz, W1);
        if (need_W1) out[1] = at::mm(dz.t(), x);      // W1's own layout, as autograd forms it
    }
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.attr("EPOCH_LIMIT") = kEpochLimit;
    m.def("init", &init);
    m.def("check", &check);
    m.def("abi_version", [] { return L.bs_abi_version(); });
    py::class_<Workspace, std::shared_ptr<Workspace>>(m, "Workspace")
        .def(py::init<c10::Device>())
        .def_readwrite("buf", &Workspace::buf)
        .def_readwrite("epoch", &Workspace::epoch)
        .def_property_readonly("nbytes", &Workspace::nbytes)
        .def("ensure", &Workspace::ensure)
        .def("next_epoch", &Workspace::next_epoch, py::arg("reserve") = 1)
        .def("amax_slot_ptr", [](const Workspace& w) { return reinterpret_cast<uintptr_t>(w.slot()); })
        .def("fallback_count", &Workspace::fallback_count);
    m.def("workspace", &workspace);
    m.def("compress", &compress);
    m.def("decompress", &decompress);
    m.def("gemm_compressed", &gemm_compressed);
    m.def("block_forward", &block_forward);
    m.def("block_backward", &block_backward);
    m.def("biased", [](const Tensor& y, const Tensor& b2, const std::vector<int64_t>& shape) {
        return Biased::apply(y, b2, shape);
    });
    // the block's steps by themselves
    m.def("activate", [](const Tensor& z, const std::optional<Tensor>& bias, const Tensor& vals,
                         const std::optional<Tensor>& offset, const Tensor& err, bool in_place, bool packed, bool fp8,
                         bool square, double k) {
        const c10::DeviceGuard guard(z.device());
        const Activation a = activate(z, bias.value_or(Tensor()), vals, offset, err, in_place, packed, fp8, square, k);
        return std::make_tuple(a.operand, optional(a.operand_scale), a.bitmask, a.prefix, a.start, a.next,
                               optional(a.scale));
    });
    m.def("act_grad", [](const Tensor& dz, const py::list& held, bool packed, bool fp8, bool square, double k, bool bias,
                         bool rows, bool cols) {
        const c10::DeviceGuard guard(dz.device());
        Held h = take_held(held, dz.size(0), dz.size(1), packed, fp8, square, k);
        const ActGrad a = act_grad(dz, h, bias, rows, cols);
        return std::make_tuple(optional(a.bias), optional(a.rows.codes), optional(a.cols.codes), optional(a.rows.scale),
                               optional(a.cols.scale));
    });
    m.def("col_sum", &col_sum);
    m.def("quantize_t", [](const Tensor& x, bool rows) {
        const c10::DeviceGuard guard(x.device());
        Workspace& w = ws_of(x);
        const Fp8 t = transposed_like(x);
        const Tensor q = rows ? empty(x.sizes(), x, at::kFloat8_e4m3fn) : Tensor();
        w.prepare(kAmaxBytes, 1);
        quantize_t(x, q, t, amax(x, false, Tensor(), w), w);
        return std::make_tuple(optional(q), t.codes, t.scale);
    });
}
