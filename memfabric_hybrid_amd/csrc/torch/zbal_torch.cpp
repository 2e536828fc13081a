/*
 * The operator layer's calls in native code: tensors in, descriptors built, outputs allocated, the zbal C ABI called,
 * tensors out. The counterpart of the reference's C++ adaptor (app/zbal/src/csrc/adaptor/deepep/zbal_deepep.cpp);
 * operators.py and buffer.py keep the signatures and return tuples on top of it.
 *
 * Small batches are bound by the host: with ctypes descriptors built field by field in Python a low-latency dispatch
 * and its combine took 55-60 us of host time for 16 us of kernels. Here a call costs its launches, an allocation per
 * output and about a microsecond.
 *
 * The library is the one capi.py has loaded (bind() gets its path): one libzbal.so per process.
 */
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <ATen/ops/empty_cuda_dispatch.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>
#include <vector>

#include "zbal.h"
#include "zbal_py_result.h"

namespace {

/* ---- the library ------------------------------------------------------------------------------------------------- */

struct Library {
    decltype(&zbal_moe_topk_route) topk_route;
    decltype(&zbal_dispatch_normal_layout_in_rank) layout;
    decltype(&zbal_dispatch_normal_notify) notify;
    decltype(&zbal_dispatch_normal_notified) notified;
    decltype(&zbal_dispatch_normal_notify_begin) notify_begin;
    decltype(&zbal_dispatch_normal_notify_end) notify_end;
    decltype(&zbal_dispatch_normal) dispatch;
    decltype(&zbal_combine_normal) combine;
    decltype(&zbal_dispatch_low_latency) ll_dispatch;
    decltype(&zbal_combine_low_latency) ll_combine;
    decltype(&zbal_fused_deep_moe) fused;
    decltype(&zbal_fused_deep_moe_workspace_size) fused_workspace;
};
Library L;
PyObject *g_check = nullptr;        /* capi.check(op, code): raises ZbalError */
PyObject *g_out_of_memory = nullptr;   /* torch.OutOfMemoryError */
PyObject *g_prepacked = nullptr;    /* "zbal_prepacked" */

template <typename F> bool find(void *h, const char *name, F *f)
{
    *f = reinterpret_cast<F>(dlsym(h, name));
    if (*f == nullptr) PyErr_Format(PyExc_RuntimeError, "libzbal.so has no symbol %s", name);
    return *f != nullptr;
}

[[noreturn]] void fail(PyObject *type, const char *text)
{
    PyErr_SetString(type, text);
    throw PyFail{};
}

void check(const char *op, int32_t rc)
{
    if (rc == 0) return;
    PyObject *r = PyObject_CallFunction(g_check, "si", op, (int)rc);
    if (r != nullptr) {
        Py_DECREF(r);
        PyErr_Format(PyExc_RuntimeError, "%s returned %d", op, (int)rc);
    }
    throw PyFail{};
}

/* ---- arguments ------------------------------------------------------------------------------------------------- */

const at::Tensor &tensor(PyObject *o)
{
    if (!THPVariable_Check(o)) fail(PyExc_TypeError, "expected a tensor");
    return THPVariable_Unpack(o);
}

int64_t integer(PyObject *o)
{
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyFail{};
    return v;
}

zbal_datatype_t datatype(at::ScalarType t)
{
    switch (t) {
        case at::kChar: return ZBAL_DATA_TYPE_INT8;
        case at::kShort: return ZBAL_DATA_TYPE_INT16;
        case at::kInt: return ZBAL_DATA_TYPE_INT32;
        case at::kLong: return ZBAL_DATA_TYPE_INT64;
        case at::kDouble: return ZBAL_DATA_TYPE_FP64;
        case at::kHalf: return ZBAL_DATA_TYPE_FP16;
        case at::kFloat: return ZBAL_DATA_TYPE_FP32;
        case at::kBFloat16: return ZBAL_DATA_TYPE_BFP16;
        case at::kByte: return ZBAL_DATA_TYPE_UINT8;
        case at::kBool: return ZBAL_DATA_TYPE_UINT8;
        case at::kFloat8_e4m3fn: return ZBAL_DATA_TYPE_FP8_E4M3;
        default: fail(PyExc_KeyError, "the zbal operators have no such tensor type");
    }
}

/* zbal_tensor_info_t of a contiguous tensor */
struct Info {
    zbal_tensor_info_t ti = {};
    Info() = default;
    explicit Info(const at::Tensor &t)
    {
        if (!t.is_contiguous()) fail(PyExc_ValueError, "zbal tensors are dense row-major; got a non-contiguous tensor");
        if (t.dim() > ZBAL_MAX_TENSOR_DIM) fail(PyExc_ValueError, "too many dimensions");
        ti.data = t.data_ptr();
        ti.dataType = datatype(t.scalar_type());
        ti.dim = (uint16_t)t.dim();
        for (int64_t i = 0; i < t.dim(); ++i) ti.shape[i] = (uint32_t)t.size(i);
    }
    Info &prepacked(int quant_mode)
    {
        if (quant_mode == 2) ti.dataType = ZBAL_DATA_TYPE_FP8_E4M3;
        if (quant_mode == 3) ti.dataType = ZBAL_DATA_TYPE_INT4X2;
        ti.reserved[0] = ZBAL_WEIGHT_FORMAT_PREPACKED;
        return *this;
    }
    Info &shape2(int64_t a, int64_t b)
    {
        ti.dim = 2;
        ti.shape[0] = (uint32_t)a;
        ti.shape[1] = (uint32_t)b;
        return *this;
    }
    const zbal_tensor_info_t *operator*() const { return &ti; }
};

/* an optional tensor: an empty descriptor for None */
Info info_or_null(PyObject *o) { return o == Py_None ? Info() : Info(tensor(o)); }

/* expert ids as the kernels take them: int32 or int64 where they lie, anything else converted */
at::Tensor expert_ids(const at::Tensor &t)
{
    const at::ScalarType s = t.scalar_type();
    if (s == at::kInt) return t;
    if (s == at::kLong && t.is_contiguous() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0) return t;
    return t.to(at::kInt);
}

/* ---- outputs ----------------------------------------------------------------------------------------------------- */

/*
 * An output: an allocation of its own, so that it can be freed, saved and kept by itself. Straight from the allocator where the
 * outputs' device is the current one: a low-latency dispatch and its combine have six, and the device's own at::cuda::empty, which
 * sets and resets the current device around each, takes 0.60 us with its free, this 0.27; the pair 13.8 -> 12.1 us (7 tokens bf16),
 * 13.5 -> 12.1 (128 int8). (at::cuda::empty in place of the dispatcher's had been 15.4 -> 13.6.) Memory that deterministic mode
 * wants filled first is at::cuda::empty's business.
 */
at::Tensor empty(c10::Device dev, bool current, at::IntArrayRef sizes, at::ScalarType t)
{
    if (!current || (at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory()))
        return at::cuda::empty(sizes, t, at::kStrided, dev, false, std::nullopt);
    return at::Tensor(at::detail::empty_generic(sizes, at::detail::getCUDAHooks().getCUDADeviceAllocator(),
                                                c10::DispatchKeySet(c10::DispatchKey::CUDA), t, std::nullopt));
}

Owned wrap(at::Tensor t) { return checked(THPVariable_Wrap(std::move(t))); }

/* ---- the frame of a call --------------------------------------------------------------------------------------- */

/* args[0] = communicator handle, args[1] = index of the device the outputs go to */
struct Frame {
    PyObject *const *args;
    zbal_comm_t comm;
    c10::Device dev;
    aclrtStream stream;
    bool current;               /* whether dev is the current device */

    Frame(PyObject *const *a, Py_ssize_t n, Py_ssize_t want) : args(a), dev(c10::DeviceType::CUDA, 0)
    {
        if (n != want) fail(PyExc_TypeError, "wrong number of arguments");
        comm = (zbal_comm_t)(uintptr_t)integer(a[0]);
        dev = c10::Device(c10::DeviceType::CUDA, (c10::DeviceIndex)integer(a[1]));
        const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream();
        stream = (aclrtStream)s.stream();
        current = s.device_index() == dev.index();
    }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType t) const { return ::empty(dev, current, sizes, t); }
    const at::Tensor &t(int i) const { return tensor(args[i]); }
    int64_t n(int i) const { return integer(args[i]); }
};

/* What a call writes and nobody gets to see: pieces of one allocation, each at a 256-byte boundary. */
class Scratch {
public:
    explicit Scratch(const Frame &f) : f_(f) {}

    size_t plan(int64_t numel, at::ScalarType t)
    {
        const size_t at = bytes_;
        bytes_ = (bytes_ + (size_t)numel * c10::elementSize(t) + 255) & ~size_t(255);
        return at;
    }

    /* after every piece has been planned */
    Info info(size_t offset, int64_t numel, at::ScalarType t)
    {
        if (!whole_.defined()) whole_ = f_.empty({(int64_t)bytes_}, at::kByte);
        Info r;
        r.ti.data = static_cast<uint8_t *>(whole_.data_ptr()) + offset;
        r.ti.dataType = datatype(t);
        r.ti.dim = 1;
        r.ti.shape[0] = (uint32_t)numel;
        return r;
    }

private:
    const Frame &f_;
    size_t bytes_ = 0;
    at::Tensor whole_;
};

/* runs `f` with the interpreter lock released, as a ctypes call would */
template <typename F> int32_t unlocked(F f)
{
    PyThreadState *save = PyEval_SaveThread();
    const int32_t rc = f();
    PyEval_RestoreThread(save);
    return rc;
}

template <PyObject *(*F)(PyObject *const *, Py_ssize_t)> PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    try {
        return F(args, n);
    } catch (const PyFail &) {
        return nullptr;
    } catch (const c10::Error &e) {
        PyErr_SetString(dynamic_cast<const c10::OutOfMemoryError *>(&e) ? g_out_of_memory : PyExc_RuntimeError,
                        e.what_without_backtrace());
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

/* ---- the operators ----------------------------------------------------------------------------------------------- */

/* (comm, dev, logits, topk, ids are int64) -> (idx, weights) */
PyObject *topk_route(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 5);
    const at::Tensor &logits = f.t(2);
    const int64_t T = logits.size(0), K = f.n(3);
    const at::ScalarType it = f.n(4) ? at::kLong : at::kInt;
    const at::Tensor idx = f.empty({T, K}, it), w = f.empty({T, K}, at::kFloat);
    const Info il(logits), ii(idx), iw(w);
    check("zbal_moe_topk_route", unlocked([&] { return L.topk_route(*il, K, *ii, *iw, f.comm, f.stream, 0); }));
    return tuple_of(wrap(idx), wrap(w));
}

/* (comm, dev, topk_idx, experts) -> (per_rank, per_expert, send_idx, token_in_rank) */
PyObject *layout(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 4);
    const at::Tensor &idx = f.t(2);
    const int64_t T = idx.size(0), K = idx.size(1), E = f.n(3);
    const at::Tensor per_rank = f.empty({1}, at::kInt), per_expert = f.empty({E}, at::kInt),
                     send = f.empty({T, K}, at::kInt), in_rank = f.empty({T, 1}, at::kInt);
    const Info i0(idx), i1(per_rank), i2(per_expert), i3(send), i4(in_rank);
    check("zbal_dispatch_normal_layout", unlocked([&] {
              return L.layout(*i0, T, E, K, *i1, *i2, *i3, *i4, f.comm, f.stream, 0);
          }));
    return tuple_of(wrap(per_rank), wrap(per_expert), wrap(send), wrap(in_rank));
}

/* (comm, dev, per_expert, topk) -> (recv_data, recv_per_expert, put_offset, balance_matrix, total_recv) */
PyObject *notify(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 4);
    const at::Tensor &per_expert = f.t(2);
    const int64_t E = per_expert.size(0), topk = f.n(3);
    const at::Tensor recv_data = f.empty({1, E}, at::kInt), recv_per_expert = f.empty({E}, at::kLong),
                     put_offset = f.empty({1, E}, at::kInt), balance = f.empty({1, 2}, at::kInt),
                     total = f.empty({1}, at::kInt);
    const Info i0(per_expert), i1(recv_data), i2(total), i3(recv_per_expert), i4(put_offset), i5(balance);
    check("zbal_dispatch_normal_notify", unlocked([&] { return L.notify(*i0, E, topk, *i1, *i2, *i3, *i4, *i5, f.comm, f.stream, 0); }));
    return tuple_of(wrap(recv_data), wrap(recv_per_expert), wrap(put_offset), wrap(balance), wrap(total));
}

/* the receive tensors of `rows` rows for one quantisation mode: rows, scales (one unused scale without quantisation) */
void receive(const Frame &f, int64_t qm, const at::Tensor &x, int64_t rows, at::Tensor *recv, at::Tensor *scales)
{
    const int64_t H = x.size(1);
    if (qm == NO_QUANT) {
        *recv = f.empty({rows, H}, x.scalar_type());
        *scales = f.empty({1}, at::kFloat);
    } else if (qm == QUANT_BF16_2_INT8) {
        *recv = f.empty({rows, H}, at::kChar);
        *scales = f.empty({rows}, at::kFloat);
    } else {
        *recv = f.empty({rows, H}, at::kFloat8_e4m3fn);
        *scales = f.empty({rows, H / 128}, at::kFloat);
    }
}

/* (comm, dev, x, ids, send_idx, put_offset, balance_matrix, experts, quant_mode, rows) -> (recv, scales) */
PyObject *dispatch(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 10);
    const at::Tensor &x = f.t(2);
    const at::Tensor ids = expert_ids(f.t(3));
    const int64_t E = f.n(7), qm = f.n(8);
    at::Tensor recv, scales;
    receive(f, qm, x, f.n(9), &recv, &scales);
    const Info i0(x), i1(ids), i2(f.t(4)), i3(f.t(5)), i4(f.t(6)), i5(recv), i6(scales);
    check("zbal_dispatch_normal", unlocked([&] {
              return L.dispatch(*i0, *i1, *i2, *i3, *i4, E, (zbal_quant_mode_t)qm, *i5, *i6, f.comm, f.stream, 0);
          }));
    return tuple_of(wrap(recv), wrap(scales));
}

/*
 * Notify and dispatch in one call. (comm, dev, x, ids, send_idx, per_expert, quant_mode, worst_rows, running) ->
 * (recv, scales, list of received counts, put_offset, balance_matrix). worst_rows > 0: that many rows, an empty list
 * and no wait for the GPU; else the counts are read back, recv and scales are allocated for their sum of rows (one at
 * least), and the list holds them, or their running sums. The GPU waits for the host in between: dispatching into
 * tensors with a row for every pick before the counts are known saves 3 % (4096 tokens bf16 217 -> 211 us), but leaves
 * the caller with all of those rows however few there are.
 */
PyObject *dispatch_counts(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 9);
    const at::Tensor &x = f.t(2), &per_expert = f.t(5);
    const at::Tensor ids = expert_ids(f.t(3));
    const int64_t worst = f.n(7), E = per_expert.size(0), qm = f.n(6), K = ids.size(1);
    at::Tensor recv, scales;
    const at::Tensor put_offset = f.empty({1, E}, at::kInt), balance = f.empty({1, 2}, at::kInt);
    Scratch tmp(f);
    const size_t o4 = tmp.plan(E, at::kInt), o5 = tmp.plan(1, at::kInt), o6 = tmp.plan(E, at::kLong);
    std::vector<int64_t> counts(worst > 0 ? 0 : (size_t)E);
    const Info i0(x), i1(ids), i2(f.t(4)), i3(per_expert), i4 = tmp.info(o4, E, at::kInt), i5 = tmp.info(o5, 1, at::kInt),
               i6 = tmp.info(o6, E, at::kLong), i7(put_offset), i8(balance);
    const zbal_quant_mode_t mode = (zbal_quant_mode_t)qm;
    if (worst > 0) {
        receive(f, qm, x, worst, &recv, &scales);
        const Info i9(recv), i10(scales);
        check("zbal_dispatch_normal", unlocked([&] {
                  return L.notified(*i0, *i1, *i2, *i3, E, K, *i4, *i5, *i6, *i7, *i8, mode, *i9, *i10, f.comm, f.stream, 0);
              }));
    } else {
        check("zbal_dispatch_normal_notify", unlocked([&] {
                  zbal_pending_counts_t pending = {};
                  const int32_t rc = L.notify_begin(*i3, E, K, *i4, *i5, *i6, *i7, *i8, &pending, f.comm, f.stream, 0);
                  return rc != 0 ? rc : L.notify_end(&pending, E, counts.data(), f.comm, f.stream, 0);
              }));
        int64_t total = 0;
        for (const int64_t c : counts) total += c;
        receive(f, qm, x, total == 0 ? 1 : total, &recv, &scales);
        const Info i9(recv), i10(scales);
        check("zbal_dispatch_normal", unlocked([&] {
                  return L.dispatch(*i0, *i1, *i2, *i7, *i8, E, mode, *i9, *i10, f.comm, f.stream, 0);
              }));
    }
    return tuple_of(wrap(recv), wrap(scales), list_of(counts, f.n(8) != 0), wrap(put_offset), wrap(balance));
}

/* (comm, dev, x, put_offset, weights, ids, send_idx, balance_matrix, experts) -> out */
PyObject *combine(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 9);
    const at::Tensor &x = f.t(2);
    const at::Tensor ids = expert_ids(f.t(5));
    const at::Tensor out = f.empty({ids.size(0), x.size(1)}, x.scalar_type());
    const Info i0(x), i1(f.t(3)), i2(f.t(4)), i3(ids), i4(f.t(6)), i5(f.t(7)), i6(out);
    const int64_t E = f.n(8);
    check("zbal_combine_normal", unlocked([&] {
              return L.combine(*i0, *i1, *i2, *i3, *i4, *i5, (uint16_t)E, *i6, f.comm, f.stream, 0);
          }));
    return wrap(out).release();
}

/* MOE_EXPERT_TOKEN_NUMS_TYPE (zbal_deepep.cpp:497), 1 where it is not set */
int64_t token_nums_type()
{
    const char *v = getenv("MOE_EXPERT_TOKEN_NUMS_TYPE");
    if (v == nullptr) return 1;
    char *end = nullptr;
    const long n = strtol(v, &end, 10);
    if (end == v || *end != 0) fail(PyExc_ValueError, "MOE_EXPERT_TOKEN_NUMS_TYPE is not a number");
    return n;
}

/* (comm, dev, x, ids, max_tokens, experts, quant_mode) -> (recv, scales, recv_count, expand_idx, ep_recv_count) */
PyObject *ll_dispatch(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 7);
    const at::Tensor &x = f.t(2);
    const at::Tensor ids = expert_ids(f.t(3));
    const int64_t T = x.size(0), K = ids.size(1), H = x.size(1), rows = T * K > 0 ? T * K : 1, E = f.n(5), qm = f.n(6), most = f.n(4),
                  type = token_nums_type();
    const at::ScalarType rt = qm == NO_QUANT ? x.scalar_type() : qm == QUANT_BF16_2_INT8 ? at::kChar : at::kFloat8_e4m3fn;
    const at::Tensor recv = f.empty({rows, H}, rt),
                     scales = qm == QUANT_BF16_2_FP8E4M3_B128 ? f.empty({rows, H / 128}, at::kFloat) : f.empty({rows}, at::kFloat),
                     expand_idx = f.empty({rows}, at::kInt), ep_recv = f.empty({E}, at::kInt), nums = f.empty({E}, at::kLong);
    /* putOffset and its status are a group's business: with one rank, as here, they are checked and left alone */
    const Info i0(x), i1(ids), i2(recv), i3(scales), i4(expand_idx), i5(nums), i6(ep_recv);
    check("zbal_dispatch_low_latency", unlocked([&] {
              return L.ll_dispatch(*i0, *i1, E, 1, 0, qm, T > most ? T : most, 0, type, *i2, *i3, *i4, *i5, *i6, *i6, *i6, f.comm,
                                   f.stream, 0);
          }));
    return tuple_of(wrap(recv), wrap(scales), wrap(nums), wrap(expand_idx), wrap(ep_recv));
}

/* (comm, dev, x, ids, expand_idx, ep_recv_count, weights, experts) -> out */
PyObject *ll_combine(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 8);
    const at::Tensor &x = f.t(2);
    const at::Tensor ids = expert_ids(f.t(3));
    const int64_t T = ids.size(0), K = ids.size(1), E = f.n(7);
    const at::Tensor out = f.empty({T, x.size(1)}, x.scalar_type());
    Info i2(f.t(4));
    i2.shape2(T, K);
    const Info i0(x), i1(ids), i3(f.t(5)), i4(f.t(6)), i5(out);
    check("zbal_combine_low_latency", unlocked([&] {
              return L.ll_combine(*i0, *i1, *i2, *i3, *i4, *i5, E, f.comm, f.stream, 0);
          }));
    return wrap(out).release();
}

/* ---- the fused layer --------------------------------------------------------------------------------------------- */

/*
 * Descriptor of a tensor list: shape and type of the stacked tensor, `data` = a device table of the per-expert
 * addresses. Tables are kept in `tables` (a dict, most recently used last), so repeated calls with the same tensors
 * copy nothing; the caller's `live` keeps this call's tables until the call has been issued, since the cache may drop
 * its own reference at any insertion.
 */
constexpr Py_ssize_t kMostTables = 64;

Info list_info(PyObject *seq, int64_t experts, PyObject *tables, c10::Device dev, std::vector<at::Tensor> &live)
{
    PyObject *fast = PySequence_Fast(seq, "a tensor list needs one tensor per expert");
    if (fast == nullptr) throw PyFail{};
    struct Release {
        PyObject *o;
        ~Release() { Py_XDECREF(o); }
    } release_fast{fast};
    if (PySequence_Fast_GET_SIZE(fast) != experts) fail(PyExc_ValueError, "a tensor list needs one tensor per expert");
    PyObject **items = PySequence_Fast_ITEMS(fast);
    const at::Tensor &first = tensor(items[0]);
    std::vector<int64_t> addresses((size_t)experts);
    for (int64_t e = 0; e < experts; ++e) {
        const at::Tensor &t = tensor(items[e]);
        if (!t.is_contiguous() || t.scalar_type() != first.scalar_type() || t.numel() != first.numel())
            fail(PyExc_ValueError, "tensor-list entries must be contiguous and alike");
        addresses[(size_t)e] = (int64_t)(uintptr_t)t.data_ptr();
    }
    PyObject *key = PyBytes_FromStringAndSize(reinterpret_cast<const char *>(addresses.data()), (Py_ssize_t)(experts * 8));
    if (key == nullptr) throw PyFail{};
    Release release_key{key};
    PyObject *found = PyDict_GetItemWithError(tables, key);
    if (found == nullptr && PyErr_Occurred()) throw PyFail{};
    at::Tensor table;
    if (found != nullptr) {
        table = tensor(found);
        if (PyDict_DelItem(tables, key) != 0) throw PyFail{};
    } else {
        table = at::empty({experts}, at::TensorOptions().dtype(at::kLong));
        memcpy(table.data_ptr(), addresses.data(), (size_t)experts * 8);
        table = table.to(dev);
    }
    if (PyDict_SetItem(tables, key, wrap(table).get()) != 0) throw PyFail{};
    while (PyDict_Size(tables) > kMostTables) {
        Py_ssize_t pos = 0;
        PyObject *oldest = nullptr, *value = nullptr;
        if (!PyDict_Next(tables, &pos, &oldest, &value)) break;
        Py_INCREF(oldest);
        Release release_oldest{oldest};
        if (PyDict_DelItem(tables, oldest) != 0) throw PyFail{};
    }
    live.push_back(table);
    Info r(first);
    /* [experts] + the shape of one entry, which may carry a leading 1 */
    const int skip = first.dim() == 3 && first.size(0) == 1 ? 1 : 0;
    r.ti.dim = (uint16_t)(first.dim() - skip + 1);
    r.ti.shape[0] = (uint32_t)experts;
    for (int64_t i = skip; i < first.dim(); ++i) r.ti.shape[1 + i - skip] = (uint32_t)first.size(i);
    r.ti.data = table.data_ptr();
    return r;
}

/*
 * (comm, dev, x, ids, w1, s1, w2, s2, topk_weights, experts, quant_mode, smooth, share_w1, share_s1, share_w2,
 * share_s2, share_smooth, active_mask, workspace, out, share_out, is_tensor_list, tables) ->
 * (out, share_out, token_nums)
 */
PyObject *fused(PyObject *const *args, Py_ssize_t nargs)
{
    const Frame f(args, nargs, 23);
    const at::Tensor &x = f.t(2);
    const at::Tensor ids = expert_ids(f.t(3));
    const int64_t T = x.size(0), H = x.size(1), K = ids.size(1), E = f.n(9);
    const int qm = (int)f.n(10);
    if (qm < 0 || qm > 3) fail(PyExc_KeyError, "quant_mode");
    const bool lists = PyObject_IsTrue(args[21]) == 1, shared = args[12] != Py_None;
    std::vector<at::Tensor> live;
    auto weight = [&](int i) { return lists ? list_info(args[i], E, args[22], f.dev, live) : Info(f.t(i)); };
    const Info i0(x), i1(ids);
    Info w1 = weight(4);
    const Info s1 = weight(5);
    Info w2 = weight(6);
    const Info s2 = weight(7);
    w1.prepacked(qm);
    w2.prepacked(qm);
    /* [experts, N, K]: a list's entries are [1, N, K] or [N, K], so N is the last dimension but one in either case */
    const int64_t n1 = w1.ti.dim >= 2 ? w1.ti.shape[w1.ti.dim - 2] : 0;
    Info sw1 = info_or_null(args[12]), sw2 = shared ? info_or_null(args[14]) : Info();
    const Info ss1 = shared ? info_or_null(args[13]) : Info(), ss2 = shared ? info_or_null(args[15]) : Info();
    const int64_t sn1 = shared && sw1.ti.dim >= 2 ? sw1.ti.shape[sw1.ti.dim - 2] : 0;
    if (shared) {
        sw1.prepacked(qm);
        sw2.prepacked(qm);
    }
    const Info wt(f.t(8)), smooth = info_or_null(args[11]), ssmooth = info_or_null(args[16]), mask = info_or_null(args[17]);

    at::Tensor workspace, out, share_out;
    if (args[18] == Py_None) {
        const uint64_t bytes = L.fused_workspace(T, H, K, E, n1, sn1, qm);
        if (bytes == 0) fail(PyExc_ValueError, "invalid fused MoE shape");
        workspace = f.empty({(int64_t)bytes}, at::kByte);
    } else {
        workspace = f.t(18);
    }
    out = args[19] == Py_None ? f.empty({T, H}, x.scalar_type()) : f.t(19);
    if (shared) share_out = args[20] == Py_None ? f.empty({T, H}, x.scalar_type()) : f.t(20);
    const at::Tensor nums = f.empty({E}, at::kLong);
    const Info iout(out), inums(nums), iws(workspace);
    Info ishare;
    if (shared) ishare = Info(share_out);
    check("zbal_fused_deep_moe", unlocked([&] {
              return L.fused(*i0, *i1, *w1, *s1, *w2, *s2, *wt, *smooth, *sw1, *ss1, *sw2, *ss2, *ssmooth, *mask, *iout, *ishare,
                             *inums, *iws, E, qm, 0, n1, sn1, lists ? 1 : 0, f.comm, f.stream, 0);
          }));
    if (!shared) Py_INCREF(Py_None);
    return tuple_of(wrap(out), shared ? wrap(share_out) : Owned(Py_None), wrap(nums));
}

/* (tensors,) -> whether every one of them is marked as pre-packed */
PyObject *all_prepacked(PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 1) fail(PyExc_TypeError, "wrong number of arguments");
    PyObject *fast = PySequence_Fast(args[0], "expected a sequence of tensors");
    if (fast == nullptr) throw PyFail{};
    bool all = true;
    for (Py_ssize_t i = 0; all && i < PySequence_Fast_GET_SIZE(fast); ++i) {
        PyObject *v = PyObject_GetAttr(PySequence_Fast_GET_ITEM(fast, i), g_prepacked);
        if (v == nullptr) PyErr_Clear();
        all = v != nullptr && PyObject_IsTrue(v) == 1;
        Py_XDECREF(v);
    }
    Py_DECREF(fast);
    return PyBool_FromLong(all);
}

/* () -> the current stream of the current device, as an integer */
PyObject *current_stream(PyObject *const *, Py_ssize_t)
{
    return PyLong_FromVoidPtr((void *)c10::hip::getCurrentHIPStream().stream());
}

/* (path of libzbal.so, capi.check, torch.OutOfMemoryError) */
PyObject *bind(PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 3) fail(PyExc_TypeError, "wrong number of arguments");
    const char *path = PyUnicode_AsUTF8(args[0]);
    if (path == nullptr) throw PyFail{};
    void *h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (h == nullptr) fail(PyExc_RuntimeError, dlerror());
    if (!find(h, "zbal_moe_topk_route", &L.topk_route) || !find(h, "zbal_dispatch_normal_layout_in_rank", &L.layout) ||
        !find(h, "zbal_dispatch_normal_notify", &L.notify) || !find(h, "zbal_dispatch_normal_notified", &L.notified) ||
        !find(h, "zbal_dispatch_normal_notify_begin", &L.notify_begin) ||
        !find(h, "zbal_dispatch_normal_notify_end", &L.notify_end) ||
        !find(h, "zbal_dispatch_normal", &L.dispatch) || !find(h, "zbal_combine_normal", &L.combine) ||
        !find(h, "zbal_dispatch_low_latency", &L.ll_dispatch) || !find(h, "zbal_combine_low_latency", &L.ll_combine) ||
        !find(h, "zbal_fused_deep_moe", &L.fused) || !find(h, "zbal_fused_deep_moe_workspace_size", &L.fused_workspace))
        throw PyFail{};
    Py_INCREF(args[1]);
    Py_XSETREF(g_check, args[1]);
    Py_INCREF(args[2]);
    Py_XSETREF(g_out_of_memory, args[2]);
    at::globalContext().lazyInitDevice(c10::DeviceType::CUDA);
    Py_RETURN_NONE;
}

#define ZB_METHOD(f) {#f, (PyCFunction)(void (*)(void))entry<f>, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {ZB_METHOD(bind),     ZB_METHOD(topk_route),  ZB_METHOD(layout),     ZB_METHOD(notify),
                           ZB_METHOD(dispatch), ZB_METHOD(dispatch_counts), ZB_METHOD(combine), ZB_METHOD(ll_dispatch),
                           ZB_METHOD(ll_combine), ZB_METHOD(fused),     ZB_METHOD(all_prepacked), ZB_METHOD(current_stream),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_zbal_torch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__zbal_torch()
{
    g_prepacked = PyUnicode_InternFromString("zbal_prepacked");
    return g_prepacked == nullptr ? nullptr : PyModule_Create(&g_module);
}
