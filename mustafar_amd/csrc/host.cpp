// The Python calls of the decode and prefill paths, from argument check to launch, as one native call each.
//
// What such a call does on the host is a few shape checks, one to ten allocations and a C-ABI call of ten to forty
// arguments.  In Python, with ctypes between, that took as long as the kernels of the smaller calls or longer.  Host time of
// a pass, us, before -> now: fused attention of one short request 9.6 -> 5.6, four decode steps 75.7 -> 38.2, the three padded
// fp16 operators with torch's padding 59 -> 41; whole passes of the calls that wait for sizes: keys and values of 128 heads
// x 256 tokens 44.7 -> 34.4, two 2-bit producers of 64 heads x 4096 tokens 120 -> 100, two compressors from the projection
// of 128 heads x 4096 tokens 178 -> 158.6.  Checks, error types and messages are those of the Python layer above (ops.py,
// mustafar_package.py, mustafar_package_quant.py, compression_quant.py), which keeps workspaces and objects.
//
// Scratch memory comes in as a tensor; a function that finds it too small returns the bytes it wants as an int instead of
// its result, and the Python layer provides them and calls again (`strict`: what is there has to do, the C ABI decides).
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>

#include <string>

#include "../../include/mustafar_hip.h"

namespace {

struct PyFail {};  // a Python error is set
[[noreturn]] void fail(PyObject* type, const char* text)
{
    PyErr_SetString(type, text);
    throw PyFail{};
}
void require(bool ok, const char* what)  // as `assert` does
{
    if (!ok) fail(PyExc_AssertionError, what);
}
void check_rt(bool ok, const char* text)
{
    if (!ok) fail(PyExc_RuntimeError, text);
}
void check_rc(int rc, const char* what)
{
    if (rc == 0) return;
    std::string text = std::string(what) + " failed: " + mstf_strerror(rc);
    if (rc == MSTF_ELAUNCH) text += " (hipError " + std::to_string(mstf_last_hip_error()) + ")";
    fail(PyExc_RuntimeError, text.c_str());
}

PyObject* g_stream_of = nullptr;  // torch._C._cuda_getCurrentRawStream
PyObject* g_device = nullptr;     // torch._C._cuda_getDevice
void* current_stream()
{
    PyObject* dev = PyObject_CallNoArgs(g_device);
    if (!dev) throw PyFail{};
    PyObject* st = PyObject_CallOneArg(g_stream_of, dev);
    Py_DECREF(dev);
    if (!st) throw PyFail{};
    void* p = PyLong_AsVoidPtr(st);
    Py_DECREF(st);
    if (!p && PyErr_Occurred()) throw PyFail{};
    return p;
}

// The arguments of a call, taken in order.
struct Args {
    PyObject* const* at;
    Py_ssize_t left;
    PyObject* next()
    {
        if (left-- <= 0) fail(PyExc_TypeError, "too few arguments");
        return *at++;
    }
    const at::Tensor& tensor()
    {
        PyObject* o = next();
        if (!THPVariable_Check(o)) fail(PyExc_TypeError, "a tensor is expected");
        return THPVariable_Unpack(o);
    }
    const at::Tensor* maybe()
    {
        if (left > 0 && *at == Py_None) {
            next();
            return nullptr;
        }
        return &tensor();
    }
    int64_t integer()
    {
        const int64_t v = PyLong_AsLongLong(next());
        if (v == -1 && PyErr_Occurred()) throw PyFail{};
        return v;
    }
    int small()  // an int of the C ABI
    {
        const int64_t v = integer();
        if (v < INT32_MIN || v > INT32_MAX) fail(PyExc_OverflowError, "argument out of range");
        return (int)v;
    }
    void* pointer()
    {
        void* p = PyLong_AsVoidPtr(next());
        if (!p && PyErr_Occurred()) throw PyFail{};
        return p;
    }
    void done() const
    {
        if (left != 0) fail(PyExc_TypeError, "too many arguments");
    }
};
template <class T>
T* ptr(const at::Tensor& t)
{
    return static_cast<T*>(t.data_ptr());
}
template <class T>
T* ptr(const at::Tensor* t)
{
    return t ? static_cast<T*>(t->data_ptr()) : nullptr;
}
int as_int(int64_t v)
{
    if (v < INT32_MIN || v > INT32_MAX) fail(PyExc_OverflowError, "size out of range");
    return (int)v;
}
bool is_half(const at::Tensor& t) { return t.scalar_type() == at::kHalf; }
at::Tensor make(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& beside)
{
    return at::empty(shape, at::TensorOptions().dtype(type).device(beside.device()));
}

// f without the interpreter lock (a launch may wait for a full queue, a sized call for the GPU): nothing in it sets a Python error
template <class F>
int unlocked(F&& f)
{
    struct Unlock {
        PyThreadState* state = PyEval_SaveThread();
        ~Unlock() { PyEval_RestoreThread(state); }
    } unlock;
    return f();
}
bool enough(const at::Tensor* ws, size_t need, bool strict) { return ws && (strict || (size_t)ws->numel() >= need); }
PyObject* wants(size_t bytes) { return PyLong_FromSize_t(bytes); }
size_t room(const at::Tensor* ws) { return ws ? (size_t)ws->numel() : 0; }
size_t bytes_of(const at::Tensor* t) { return t ? (size_t)t->nbytes() : 0; }
// least scratch memory of an attention call (ops.attention_workspace_least)
size_t attention_least(int64_t tokens, int64_t window, int64_t rows)
{
    return (size_t)((rows * ((tokens + 511) / 512 + (window + 63) / 64) * 520 + 255) / 256 * 256);
}

template <PyObject* (*F)(Args&)>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    try {
        Args a{args, n};
        return F(a);
    } catch (const PyFail&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// (k_bmp, k_nz, k_idx, k_nz_off, v_..., q, groups, tokens, head_dim, out, lse, ws, strict) -> out
PyObject* decode_attention(Args& a)
{
    const at::Tensor *s[8];
    for (auto& t : s) t = &a.tensor();
    const at::Tensor& q = a.tensor();
    const int groups = a.small(), tokens = a.small(), D = a.small();
    const at::Tensor *out = a.maybe(), *lse = a.maybe(), *ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    require(is_half(q) && q.is_contiguous(), "q must be contiguous fp16");
    const int Bq = as_int(q.numel() / D);
    const size_t need = mstf_decode_attention_workspace_bytes(tokens, D, Bq, groups);
    if (!enough(ws, need, strict)) return wants(need);
    at::Tensor o = out ? *out : make({Bq, D}, at::kHalf, q);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_decode_attention_f16(st, ptr<uint64_t>(s[0]), ptr<mstf_half>(s[1]), ptr<uint32_t>(s[2]),
                                                  ptr<uint32_t>(s[3]), ptr<uint64_t>(s[4]), ptr<mstf_half>(s[5]),
                                                  ptr<uint32_t>(s[6]), ptr<uint32_t>(s[7]), ptr<mstf_half>(q), ptr<mstf_half>(o),
                                                  ptr<float>(lse), tokens, D, Bq, groups, ptr<void>(ws), room(ws));
             }),
             "mstf_decode_attention_f16");
    return THPVariable_Wrap(std::move(o));
}

// 64 for [B, T] scales (the reference), 32 for [B, T, 2]
int group_size_of(const at::Tensor& bmp, const at::Tensor& scales, const at::Tensor& zeros)
{
    check_rt(scales.sizes() == zeros.sizes(), "scales and zeros must have the same shape.");
    if (scales.numel() == bmp.numel()) return 64;
    check_rt(scales.numel() == 2 * bmp.numel() && scales.dim() > 0 && scales.size(-1) == 2,
             "scales must hold one or two entries per tile.");
    return 32;
}

// (k bmp, offsets, packed, scales, zeros, v ..., q, groups, bit, mode, out, lse, ws, strict) -> out
PyObject* decode_attention_quant(Args& a)
{
    const at::Tensor *s[10];
    for (auto& t : s) t = &a.tensor();
    const at::Tensor& q = a.tensor();
    const int groups = a.small(), bit = a.small(), mode = a.small();
    const at::Tensor *out = a.maybe(), *lse = a.maybe(), *ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    const int D = as_int(q.size(-1)), Bq = as_int(q.numel() / D);
    const int tokens = as_int(s[0]->size(1) * 64 / D);
    const size_t need = groups > 0 ? mstf_decode_attention_workspace_bytes(tokens, D, Bq, groups) : attention_least(tokens, 0, Bq);
    if (!enough(ws, need, strict)) return wants(need);
    const int gs = group_size_of(*s[0], *s[3], *s[4]);
    check_rt(group_size_of(*s[5], *s[8], *s[9]) == gs, "key side and value side must use the same group size.");
    check_rt(bit > 0, "bit must be positive");
    at::Tensor o = out ? *out : make({Bq, D}, at::kHalf, q);
    const at::Tensor qc = q.contiguous();
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_decode_attention_quant_grouped(
                     st, ptr<uint64_t>(s[0]), ptr<uint32_t>(s[2]), ptr<uint32_t>(s[1]), ptr<mstf_half>(s[3]), ptr<mstf_half>(s[4]),
                     ptr<uint64_t>(s[5]), ptr<uint32_t>(s[7]), ptr<uint32_t>(s[6]), ptr<mstf_half>(s[8]), ptr<mstf_half>(s[9]),
                     ptr<mstf_half>(qc), ptr<mstf_half>(o), ptr<float>(lse), tokens, D, Bq, groups, bit, 32 / bit, mode, gs,
                     ptr<void>(ws), room(ws));
             }),
             "mstf_decode_attention_quant");
    return THPVariable_Wrap(std::move(o));
}

// What both step calls take behind their cache arrays.
struct Step {
    const at::Tensor *q_in, *k_in, *v_in, *k_win, *v_win, *cos, *sin, *win_len_dev, *overflow, *out, *lse, *ws;
    int win_len, max_tokens, bs, n_q, n_kv, D, Bq;
    int64_t tile_capacity, rope_stride = 0;
    const at::Tensor* tokens_dev;
    bool strict;
    // (q_in, k_in, v_in, k_win, v_win, win_len, cos, sin, win_len_dev, overflow, out, lse, max_tokens, tokens_dev,
    //  tile_capacity, ws, strict)
    explicit Step(Args& a)
    {
        q_in = &a.tensor(), k_in = &a.tensor(), v_in = &a.tensor(), k_win = &a.tensor(), v_win = &a.tensor();
        win_len = a.small();
        cos = a.maybe(), sin = a.maybe(), win_len_dev = a.maybe(), overflow = a.maybe(), out = a.maybe(), lse = a.maybe();
        max_tokens = a.small();
        tokens_dev = &a.tensor();
        tile_capacity = a.integer();
        ws = a.maybe();
        strict = a.integer() != 0;
        D = as_int(k_win->size(-1));
        require(D > 0 && k_in->dim() > 0, "window and new rows");
        bs = as_int(k_in->size(0));
        n_kv = as_int(k_in->size(-1) / D), n_q = as_int(q_in->size(-1) / D);
        for (const at::Tensor* t : {q_in, k_in, v_in})
            require(is_half(*t) && t->dim() == 2 && t->stride(1) == 1 && t->size(0) == bs, "new rows: fp16 [bs, heads * D]");
        require(is_half(*k_win) && k_win->is_contiguous() && v_win->is_contiguous() && k_win->sizes() == v_win->sizes(),
                "windows: contiguous fp16 of one shape");
        require(k_win->size(0) == (int64_t)bs * n_kv && v_in->size(-1) == (int64_t)n_kv * D && n_kv > 0 && n_q % n_kv == 0,
                "head counts");
        if (cos) {
            require(sin && is_half(*cos) && is_half(*sin) && cos->sizes() == sin->sizes(), "cos and sin: fp16 of one shape");
            require(cos->size(-1) == D && cos->stride(-1) == 1 && sin->stride(-1) == 1, "cos and sin: [D] or [bs, D]");
            if (cos->dim() == 2 && cos->size(0) > 1) {
                require(cos->size(0) == bs && cos->stride(0) == sin->stride(0), "cos and sin: a row per batch entry");
                rope_stride = cos->stride(0);
            }
        }
        Bq = as_int((int64_t)bs * n_q);
    }
    int win_stride() const { return as_int(k_win->size(1)); }
    at::Tensor output() const { return out ? *out : make({Bq, D}, at::kHalf, *q_in); }
};

// (k bmp, nz, idx, nz_off, v ..., Step) -> out
PyObject* decode_step(Args& a)
{
    const at::Tensor *s[8];
    for (auto& t : s) t = &a.tensor();
    const Step e(a);
    a.done();
    const size_t need = mstf_decode_attention_window_workspace_bytes(e.max_tokens, e.win_len, e.D, e.Bq, e.n_q / e.n_kv);
    if (!enough(e.ws, need, e.strict)) return wants(need);
    at::Tensor o = e.output();
    const int win_stride = e.win_stride();
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_decode_step_pool_f16(
                     st, ptr<uint64_t>(s[0]), ptr<mstf_half>(s[1]), ptr<uint32_t>(s[2]), ptr<uint32_t>(s[3]), ptr<uint64_t>(s[4]),
                     ptr<mstf_half>(s[5]), ptr<uint32_t>(s[6]), ptr<uint32_t>(s[7]), ptr<mstf_half>(e.q_in), e.q_in->stride(0),
                     ptr<mstf_half>(e.k_in), e.k_in->stride(0), ptr<mstf_half>(e.v_in), e.v_in->stride(0), e.bs, e.n_q, e.n_kv,
                     ptr<mstf_half>(e.cos), e.cos ? ptr<mstf_half>(e.sin) : nullptr, e.rope_stride, ptr<mstf_half>(e.k_win),
                     ptr<mstf_half>(e.v_win), win_stride, e.win_len, ptr<int32_t>(e.win_len_dev),
                     ptr<uint32_t>(e.overflow), ptr<mstf_half>(o), ptr<float>(e.lse), e.max_tokens, ptr<int32_t>(e.tokens_dev),
                     e.tile_capacity, e.D, ptr<void>(e.ws), room(e.ws));
             }),
             "mstf_decode_step_pool_f16");
    return THPVariable_Wrap(std::move(o));
}

// (bit, mode, k bmp, packed, offsets, scales, zeros, v ..., Step) -> out
PyObject* decode_step_quant(Args& a)
{
    const int bit = a.small(), mode = a.small();
    const at::Tensor *s[10];
    for (auto& t : s) t = &a.tensor();
    const Step e(a);
    a.done();
    const size_t need = mstf_decode_attention_window_workspace_bytes(e.max_tokens, e.win_len, e.D, e.Bq, e.n_q / e.n_kv);
    if (!enough(e.ws, need, e.strict)) return wants(need);
    check_rt(bit > 0, "bit must be positive");
    at::Tensor o = e.output();
    const int win_stride = e.win_stride();
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_decode_step_quant_pool(
                     st, ptr<uint64_t>(s[0]), ptr<uint32_t>(s[1]), ptr<uint32_t>(s[2]), ptr<mstf_half>(s[3]), ptr<mstf_half>(s[4]),
                     ptr<uint64_t>(s[5]), ptr<uint32_t>(s[6]), ptr<uint32_t>(s[7]), ptr<mstf_half>(s[8]), ptr<mstf_half>(s[9]),
                     ptr<mstf_half>(e.q_in), e.q_in->stride(0), ptr<mstf_half>(e.k_in), e.k_in->stride(0), ptr<mstf_half>(e.v_in),
                     e.v_in->stride(0), e.bs, e.n_q, e.n_kv, ptr<mstf_half>(e.cos), e.cos ? ptr<mstf_half>(e.sin) : nullptr,
                     e.rope_stride, ptr<mstf_half>(e.k_win), ptr<mstf_half>(e.v_win), win_stride, e.win_len,
                     ptr<int32_t>(e.win_len_dev), ptr<uint32_t>(e.overflow), ptr<mstf_half>(o), ptr<float>(e.lse), e.max_tokens,
                     ptr<int32_t>(e.tokens_dev), e.tile_capacity, e.D, bit, 32 / bit, mode, ptr<void>(e.ws), room(e.ws));
             }),
             "mstf_decode_step_quant_pool");
    return THPVariable_Wrap(std::move(o));
}

// The reference's checks in front of its fp16 operators (mustafar_wrapper.cu:19-263).
void formulation_checks(const at::Tensor* const (&s)[4], const at::Tensor& B, bool contiguous_b)
{
    for (const at::Tensor* t : s) check_rt(t->device() == B.device(), "All input tensors must be on the same device.");
    check_rt(is_half(B), "Tensor B must be of type float16.");
    check_rt(is_half(*s[1]), "Tensor NZ must be of type float16.");
    check_rt(s[0]->scalar_type() == at::kLong, "Tensor bmp must be of type int64.");
    check_rt(s[2]->scalar_type() == at::kInt, "Tensor idx must be of type int.");
    check_rt(s[3]->scalar_type() == at::kInt, "Tensor NZ_Offset must be of type int.");
    bool contiguous = !contiguous_b || B.is_contiguous(), cuda = B.is_cuda();
    for (const at::Tensor* t : s) contiguous = contiguous && t->is_contiguous(), cuda = cuda && t->is_cuda();
    check_rt(contiguous, "bmp, NZ, idx, B, C, and Reduction_Workspace tensors must be contiguous.");
    check_rt(cuda, "bmp, NZ, idx, B, C, and (not)Reduction_Workspace tensors must be on CUDA device.");
}

// (bmp, NZ, idx, NZ_Offset, B, M, K, Bq, groups) -> C
PyObject* key_formulation(Args& a)
{
    const at::Tensor* s[4];
    for (auto& t : s) t = &a.tensor();
    const at::Tensor& B = a.tensor();
    const int M = a.small(), K = a.small(), Bq = a.small(), groups = a.small();
    a.done();
    formulation_checks(s, B, true);
    check_rt(B.numel() == (int64_t)Bq * 8 * K, "Tensor B must hold Batch_Size x 8 x K_Global elements.");
    at::Tensor C = make({Bq, 8, M}, at::kHalf, B);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_key_spmv_f16(st, ptr<uint64_t>(s[0]), ptr<mstf_half>(s[1]), ptr<uint32_t>(s[2]), ptr<uint32_t>(s[3]),
                                          ptr<mstf_half>(B), ptr<mstf_half>(C), M, K, Bq, groups, 8);
             }),
             "mustafar_key_formulation");
    return THPVariable_Wrap(std::move(C));
}

// (bmp, NZ, idx, NZ_Offset, B, M, K, Bq, groups, ws, strict) -> C
PyObject* value_formulation(Args& a)
{
    const at::Tensor* s[4];
    for (auto& t : s) t = &a.tensor();
    const at::Tensor& B = a.tensor();
    const int M = a.small(), K = a.small(), Bq = a.small(), groups = a.small();
    const at::Tensor* ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    formulation_checks(s, B, false);
    check_rt(B.numel() == (int64_t)Bq * 8 * K, "Tensor B must hold Batch_Size x 8 x K_Global elements.");
    const size_t need = groups > 0 ? mstf_value_spmv_workspace_bytes(M, K, Bq, groups, 8) : 0;
    if (!enough(ws, need, strict)) return wants(need);
    const at::Tensor P = B.contiguous();
    at::Tensor C = make({Bq, 8, M}, at::kHalf, B);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_value_spmv_f16(st, ptr<uint64_t>(s[0]), ptr<mstf_half>(s[1]), ptr<uint32_t>(s[2]), ptr<uint32_t>(s[3]),
                                            ptr<mstf_half>(P), ptr<mstf_half>(C), M, K, Bq, groups, 8, ptr<void>(ws), room(ws));
             }),
             "mustafar_value_formulation");
    return THPVariable_Wrap(std::move(C));
}

// The checks in front of the quantised operators: bmp, NZ_quant, tile_offsets, tile_counts, tile_units (null: not given),
// scales, zeros.
void quant_checks(const at::Tensor* const (&s)[7], const at::Tensor& B)
{
    static const char* const kInts[] = {nullptr, "Tensor NZ_quant must be of type int32.", "Tensor tile_offsets must be of type int32.",
                                        "Tensor tile_counts must be of type int32.", "Tensor tile_units must be of type int32."};
    for (const at::Tensor* t : s)
        if (t) check_rt(t->device() == B.device(), "All input tensors must be on the same device.");
    check_rt(is_half(B), "Tensor B must be of type float16.");
    check_rt(s[0]->scalar_type() == at::kLong, "Tensor bmp must be of type int64.");
    for (int i = 1; i < 5; i++)
        if (s[i]) check_rt(s[i]->scalar_type() == at::kInt, kInts[i]);
    check_rt(is_half(*s[5]), "Tensor scales must be of type float16.");
    check_rt(is_half(*s[6]), "Tensor zeros must be of type float16.");
    bool contiguous = true, cuda = B.is_cuda();
    for (const at::Tensor* t : s)
        if (t) contiguous = contiguous && t->is_contiguous(), cuda = cuda && t->is_cuda();
    check_rt(contiguous, "All tensors must be contiguous.");
    check_rt(cuda, "All tensors must be on CUDA device.");
    check_rt(s[1]->numel() != 0, "NZ_quant is empty.");
}

// (bmp, NZ_quant, tile_offsets, tile_counts, tile_units, scales, zeros, B, M, K, Bq, groups, bit, capacity, mode) -> C
PyObject* key_formulation_quant(Args& a)
{
    const at::Tensor* s[7];
    for (int i = 0; i < 7; i++) s[i] = i == 3 || i == 4 ? a.maybe() : &a.tensor();
    if (!s[3]) s[4] = nullptr;  // (units come with counts or not at all)
    const at::Tensor& B = a.tensor();
    const int M = a.small(), K = a.small(), Bq = a.small(), groups = a.small(), bit = a.small(), cap = a.small(), mode = a.small();
    a.done();
    quant_checks(s, B);
    check_rt(B.is_contiguous(), "All tensors must be contiguous.");
    check_rt(B.numel() == (int64_t)Bq * 8 * K, "Tensor B must hold Batch_Size x 8 x K_Global elements.");
    at::Tensor C = make({Bq, 8, M}, at::kHalf, B);
    const int gs = group_size_of(*s[0], *s[5], *s[6]);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_key_spmv_quant_grouped(st, ptr<uint64_t>(s[0]), ptr<uint32_t>(s[1]), ptr<uint32_t>(s[2]),
                                                    ptr<mstf_half>(s[5]), ptr<mstf_half>(s[6]), ptr<mstf_half>(B), ptr<mstf_half>(C),
                                                    M, K, Bq, groups, 8, bit, cap, mode, gs);
             }),
             "mustafar_key_formulation_quant");
    return THPVariable_Wrap(std::move(C));
}

// (bmp, NZ_quant, tile_offsets, tile_counts, tile_units, scales, zeros, P, n_rows, M, K, Bq, groups, bit, capacity, mode, ws,
//  strict) -> C
PyObject* value_formulation_quant(Args& a)
{
    const at::Tensor* s[7];
    for (auto& t : s) t = &a.tensor();
    const at::Tensor& P = a.tensor();
    const int rows = a.small(), M = a.small(), K = a.small(), Bq = a.small(), groups = a.small(), bit = a.small(), cap = a.small(),
              mode = a.small();
    const at::Tensor* ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    quant_checks(s, P);
    check_rt(P.numel() == (int64_t)Bq * rows * K, "score tensor has the wrong number of elements.");
    const size_t need = groups > 0 ? mstf_value_spmv_quant_workspace_bytes(M, K, Bq, groups, rows) : 0;
    if (!enough(ws, need, strict)) return wants(need);
    const at::Tensor p = P.contiguous();
    at::Tensor C = rows == 8 ? make({Bq, 8, M}, at::kHalf, P) : make({Bq, M}, at::kHalf, P);
    const int gs = group_size_of(*s[0], *s[5], *s[6]);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_value_spmv_quant_grouped(st, ptr<uint64_t>(s[0]), ptr<uint32_t>(s[1]), ptr<uint32_t>(s[2]),
                                                      ptr<mstf_half>(s[5]), ptr<mstf_half>(s[6]), ptr<mstf_half>(p),
                                                      ptr<mstf_half>(C), M, K, Bq, groups, rows, bit, cap, mode, gs, ptr<void>(ws),
                                                      room(ws));
             }),
             rows == 8 ? "mustafar_value_formulation_quant" : "mustafar_value_formulation_quant_decode_n1");
    return THPVariable_Wrap(std::move(C));
}

// (s, head_dim, out) -> probabilities in the shape of s
PyObject* scale_softmax(Args& a)
{
    const at::Tensor& s = a.tensor();
    const int D = a.small();
    const at::Tensor* out = a.maybe();
    a.done();
    require(is_half(s) && s.dim() > 0 && s.stride(-1) == 1, "scores: fp16 with contiguous rows");
    const int L = as_int(s.size(-1));
    const at::Tensor s2 = s.reshape({-1, L});
    const at::Tensor p = out ? out->reshape({-1, L}) : at::empty_like(s2);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 return mstf_scale_softmax_f16(st, ptr<mstf_half>(s2), ptr<mstf_half>(p), s2.size(0), L, s2.stride(0),
                                               p.stride(0), D);
             }),
             "mstf_scale_softmax_f16");
    return THPVariable_Wrap(p.reshape(s.sizes()));
}

PyObject* tuple_of(std::initializer_list<at::Tensor> tensors, PyObject* last = nullptr)
{
    PyObject* t = PyTuple_New((Py_ssize_t)tensors.size() + (last ? 1 : 0));
    if (!t) throw PyFail{};
    Py_ssize_t i = 0;
    for (const at::Tensor& x : tensors) PyTuple_SET_ITEM(t, i++, THPVariable_Wrap(x));
    if (last) PyTuple_SET_ITEM(t, i, last);
    return t;
}

// The arrays of one compressed side.
struct Side {
    at::Tensor bmp, idx, nz_off, total, nz;
    Side(int64_t B, int64_t T, int64_t cap, const at::Tensor& beside)
        : bmp(make({B, T}, at::kLong, beside)), idx(make({B, T + 1}, at::kInt, beside)), nz_off(make({B}, at::kInt, beside)),
          total(make({1}, at::kLong, beside)), nz(make({cap}, at::kHalf, beside))
    {
    }
};

// (k, v, kth_k, kth_v, capacity or -1, landings or 0, status, ws, strict) -> (bmp, idx, nz_off, total, nz) x 2
PyObject* compress_kv(Args& a)
{
    const at::Tensor &k0 = a.tensor(), &v0 = a.tensor();
    const int kth_k = a.small(), kth_v = a.small();
    const int64_t capacity = a.integer();
    int64_t* landings = static_cast<int64_t*>(a.pointer());
    const at::Tensor *status = a.maybe(), *ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    require(k0.is_cuda() && v0.is_cuda() && is_half(k0) && is_half(v0) && k0.dim() == 3 && k0.sizes() == v0.sizes(),
            "k and v: fp16 [B, M, N] of one shape on the GPU");
    const int B = as_int(k0.size(0)), M = as_int(k0.size(1)), N = as_int(k0.size(2));
    const size_t need = mstf_compress_kv_workspace_bytes(B, M, N);
    if (!enough(ws, need, strict)) return wants(need);
    const at::Tensor k = k0.contiguous(), v = v0.contiguous();
    const int64_t T = (int64_t)M * N / 64, cap = capacity < 0 ? (int64_t)B * M * N : capacity;
    const Side ks(B, T, cap, k), vs(B, T, cap, k);
    void* st = current_stream();
    check_rc(unlocked([&] {
                 auto call = [&](auto fn, auto... more) {
                     return fn(st, ptr<mstf_half>(k), ptr<mstf_half>(v), B, M, N, kth_k, kth_v, ptr<uint64_t>(ks.bmp),
                               ptr<uint32_t>(ks.idx), ptr<uint32_t>(ks.nz_off), ptr<uint64_t>(ks.total), ptr<mstf_half>(ks.nz),
                               (uint64_t)cap, ptr<uint64_t>(vs.bmp), ptr<uint32_t>(vs.idx), ptr<uint32_t>(vs.nz_off),
                               ptr<uint64_t>(vs.total), ptr<mstf_half>(vs.nz), (uint64_t)cap, ptr<void>(ws), room(ws), more...);
                 };
                 return call(mstf_compress_kv_landing_f16, ptr<uint64_t>(status), bytes_of(status), landings);
             }),
             "mstf_compress_kv_landing_f16");
    return tuple_of({ks.bmp, ks.idx, ks.nz_off, ks.total, ks.nz, vs.bmp, vs.idx, vs.nz_off, vs.total, vs.nz});
}

// (x, is_value, kth, M, cos, sin, rot, capacity or -1, landing, waits, status, ws, strict) -> (bmp, idx, nz_off, total, nz, size or -1).
// Capacity -1: room for the dense rows, and the size comes to the landing (M > 0; address of a pinned word).  waits: the call waits
// for it, and returns the values cut to size; negative if a workgroup gave up.
PyObject* compress_proj(Args& a)
{
    const at::Tensor& x = a.tensor();
    const int is_value = a.small(), kth = a.small(), M = a.small();
    const at::Tensor *cos = a.maybe(), *sin = a.maybe(), *rot = a.maybe();
    const int64_t capacity = a.integer();
    int64_t* landing = static_cast<int64_t*>(a.pointer());
    const bool waits = a.integer() != 0;
    const at::Tensor *status = a.maybe(), *ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    require(x.is_cuda() && is_half(x) && x.dim() == 4 && x.stride(3) == 1, "x: fp16 [batch, rows, heads, D] on the GPU");
    mstf_proj_source src = {};
    src.x = ptr<mstf_half>(x);
    src.stride_batch = x.stride(0), src.stride_token = x.stride(1), src.stride_head = x.stride(2);
    src.batch = as_int(x.size(0)), src.rows = as_int(x.size(1)), src.heads = as_int(x.size(2));
    if (cos) {
        require(sin && is_half(*cos) && is_half(*sin) && cos->sizes() == sin->sizes(), "cos and sin: fp16 of one shape");
        require(cos->dim() >= 2 && cos->stride(-1) == 1 && sin->strides() == cos->strides() && cos->size(-2) >= x.size(1),
                "cos and sin: a contiguous row per token");
        const at::Tensor& r = rot ? *rot : x;
        require(r.sizes() == x.sizes() && is_half(r) && r.stride(3) == 1, "rot: shaped like x");
        src.cos = ptr<mstf_half>(cos), src.sin = ptr<mstf_half>(sin);
        src.rope_stride_batch = cos->dim() == 3 && cos->size(0) > 1 ? cos->stride(0) : 0;
        src.rope_stride_token = cos->stride(-2);
        src.rot = ptr<mstf_half>(r);
        src.rot_stride_batch = r.stride(0), src.rot_stride_token = r.stride(1), src.rot_stride_head = r.stride(2);
    }
    const int B = as_int((int64_t)src.batch * src.heads), N = as_int(x.size(3));
    const int64_t T = (int64_t)M * N / 64;
    const size_t need = mstf_compress_workspace_bytes(B, M > 64 ? M : 64, N);
    if (!enough(ws, need, strict)) return wants(need);
    const int64_t cap = capacity < 0 ? (int64_t)B * M * N : capacity;
    const Side s(B, T, cap > 8 ? cap : 8, x);
    void* st = current_stream();
    const bool sized = capacity < 0 && M != 0;
    int64_t size = -1;
    check_rc(unlocked([&] {
                 auto call = [&](auto fn, auto... more) {
                     return fn(st, &src, is_value, M, N, kth, ptr<uint64_t>(s.bmp), ptr<uint32_t>(s.idx),
                               ptr<uint32_t>(s.nz_off), ptr<uint64_t>(s.total), ptr<mstf_half>(s.nz), (uint64_t)cap, ptr<void>(ws),
                               room(ws), more...);
                 };
                 if (!sized) return call(mstf_compress_proj_f16);
                 return waits ? call(mstf_compress_proj_sized_f16, ptr<uint64_t>(status), bytes_of(status), landing, &size)
                              : call(mstf_compress_proj_landing_f16, ptr<uint64_t>(status), bytes_of(status), landing);
             }),
             !sized ? "mstf_compress_proj_f16" : (waits ? "mstf_compress_proj_sized_f16" : "mstf_compress_proj_landing_f16"));
    return tuple_of({s.bmp, s.idx, s.nz_off, s.total, sized && size >= 0 ? s.nz.narrow(0, 0, size) : s.nz},
                    PyLong_FromLongLong(size));
}

// (x, is_value, bit, kth, group_size, room or None, landing or 0, status, ws, strict) ->
// (bmp, tile_off, room, counts, units, scales, zeros, total).  landing: address of a pinned word - the call waits for the word
// count, and returns it in the place of the total.
PyObject* produce_quant(Args& a)
{
    const at::Tensor& x0 = a.tensor();
    const int is_value = a.small(), bit = a.small(), kth = a.small(), gs = a.small();
    const at::Tensor* given = a.maybe();
    int64_t* landing = static_cast<int64_t*>(a.pointer());
    const at::Tensor *status = a.maybe(), *ws = a.maybe();
    const bool strict = a.integer() != 0;
    a.done();
    require(x0.is_cuda() && x0.dim() == 3, "inputs: [B, M, N] on the GPU");
    const int B = as_int(x0.size(0)), M = as_int(x0.size(1)), N = as_int(x0.size(2));
    require(M % 64 == 0, "M must be a multiple of 64");
    check_rt(is_half(x0), "inputs must be float16");
    check_rt(gs == 32 || gs == 64, "group_size must be 32 or 64");
    const size_t need = mstf_compress_quant_workspace_bytes(B, M, N);
    if (!enough(ws, need, strict)) return wants(need);
    const at::Tensor x = x0.contiguous();
    const int64_t T = (int64_t)M * N / 64;
    const at::Tensor bmp = make({B, T}, at::kLong, x), off = make({B, T}, at::kInt, x), counts = make({B, T}, at::kInt, x),
                     units = make({B, T}, at::kInt, x);
    const at::Tensor scales = gs == 64 ? make({B, T}, at::kHalf, x) : make({B, T, 2}, at::kHalf, x),
                     zeros = gs == 64 ? make({B, T}, at::kHalf, x) : make({B, T, 2}, at::kHalf, x);
    const at::Tensor total = make({1}, at::kLong, x);
    // one pass with room for the worst case (every element kept: 64 // capacity words per tile)
    int64_t cap = B * T * (64 * (int64_t)bit / 32);
    const at::Tensor words = given ? *given : make({cap > 1 ? cap : 1}, at::kInt, x);
    if (given) cap = words.numel();
    require(words.scalar_type() == at::kInt && words.is_contiguous(), "room: contiguous int32");
    void* st = current_stream();
    int64_t size = -1;
    check_rc(unlocked([&] {
                 auto call = [&](auto fn, auto... more) {
                     return fn(st, ptr<mstf_half>(x), is_value != 0, B, M, N, kth, bit, gs, ptr<uint64_t>(bmp), ptr<uint32_t>(off),
                               ptr<uint32_t>(counts), ptr<uint32_t>(units), ptr<mstf_half>(scales), ptr<mstf_half>(zeros),
                               ptr<uint64_t>(total), ptr<uint32_t>(words), (uint64_t)cap, ptr<void>(ws), room(ws), more...);
                 };
                 return landing ? call(mstf_compress_quant_sized, ptr<uint64_t>(status), bytes_of(status), landing, &size) : call(mstf_compress_quant_grouped);
             }),
             landing ? "mstf_compress_quant_sized" : "mstf_compress_quant_grouped");
    if (landing) return tuple_of({bmp, off, words, counts, units, scales, zeros}, PyLong_FromLongLong(size));
    return tuple_of({bmp, off, words, counts, units, scales, zeros, total});
}

PyMethodDef kMethods[] = {
#define MSTF_ENTRY(F) {#F, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<F>)), METH_FASTCALL, nullptr}
    MSTF_ENTRY(decode_attention), MSTF_ENTRY(decode_attention_quant), MSTF_ENTRY(decode_step), MSTF_ENTRY(decode_step_quant),
    MSTF_ENTRY(key_formulation), MSTF_ENTRY(value_formulation), MSTF_ENTRY(key_formulation_quant),
    MSTF_ENTRY(value_formulation_quant), MSTF_ENTRY(scale_softmax), MSTF_ENTRY(compress_kv), MSTF_ENTRY(compress_proj),
    MSTF_ENTRY(produce_quant), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host()
{
    PyObject* c = PyImport_ImportModule("torch._C");
    if (!c) return nullptr;
    g_stream_of = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
    g_device = PyObject_GetAttrString(c, "_cuda_getDevice");
    Py_DECREF(c);
    if (!g_stream_of || !g_device) return nullptr;
    return PyModule_Create(&kModule);
}
