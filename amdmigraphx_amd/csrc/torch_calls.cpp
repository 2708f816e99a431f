// The front end's plain calls in native code: operands that are ordinary dense device tensors of the current
// device, with nothing that the Python functions of ops.py would convert, copy or refuse.  Every function here
// returns None for any other call, and the Python function that asked goes on by itself, so what is accepted, what is
// refused and with which message is decided there alone.
//
// What bounds a small call is its host side: shapes, strides and a dozen arguments through Python and ctypes
// were 5 to 12 us of it, beside about 2 of the launch.  Measured a pass (one MI355X): see ops.py.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include "mi355_qgemm.h"

#include <array>

namespace {

PyObject* check_status = nullptr; // capi.check

// A call that the Python function has to look at itself.  A return and no exception: such calls are ordinary ones (an
// output or a workspace of the caller's, more dimensions, strides), and a C++ exception costs them 2.3 us where the
// checks cost 0.1 to 0.2.
PyObject* leave() { Py_RETURN_NONE; }

#define PLAIN_IF(...)       \
    do                      \
    {                       \
        if(!(__VA_ARGS__))  \
            return leave(); \
    } while(0)

// The operands' device and stream.  Every check returns false for what is not plain.
struct site
{
    c10::DeviceIndex device = -1;

    static bool modes()
    {
        return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
               at::tracer::impl::is_dispatch_enabled();
    }
    bool tensor(PyObject* o, const at::Tensor*& to)
    {
        if(!THPVariable_CheckExact(o))
            return false;
        const at::Tensor& t = THPVariable_Unpack(o);
        if(!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || !t.has_storage() || t.is_neg() || t.is_conj() ||
           t.is_quantized() || t.numel() <= 0)
            return false;
        if(device < 0)
            device = t.device().index();
        to = &t;
        return t.device().index() == device;
    }
    bool dense(PyObject* o, const at::Tensor*& to) { return tensor(o, to) && to->is_contiguous(); }
    // a dense tensor, or None
    bool room(PyObject* o, const at::Tensor*& to) { return o == Py_None || dense(o, to); }
    // a dense vector of 32-bit floats or integers, or None
    bool vector(PyObject* o, const at::Tensor*& to)
    {
        return o == Py_None || (dense(o, to) && to->element_size() == 4);
    }
    // modes and a trace see the Python function's own torch calls
    bool here() const { return !modes() && c10::hip::current_device() == device; }
    void* stream() const { return c10::hip::getCurrentHIPStream(device).stream(); }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const
    {
        return at::empty(sizes, at::TensorOptions().dtype(type).device(at::Device(at::kCUDA, device)));
    }
};

template <class T>
T* at_data(const at::Tensor* t)
{
    return t == nullptr ? nullptr : static_cast<T*>(t->data_ptr());
}

bool integer(PyObject* o, int64_t& to)
{
    if(!PyLong_CheckExact(o))
        return false;
    int overflow = 0;
    to           = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

template <class T>
bool integer32(PyObject* o, T& to)
{
    int64_t v     = 0;
    const bool ok = integer(o, v);
    to            = (T)v;
    return ok;
}

bool truth(PyObject* o, bool& to)
{
    to = o == Py_True;
    return o == Py_True || o == Py_False;
}

bool code_of(at::ScalarType t, int& to)
{
    switch(t)
    {
    case at::kChar: to = MI355_I8; return true;
    case at::kByte: to = MI355_U8; return true;
    case at::kInt: to = MI355_I32; return true;
    case at::kFloat: to = MI355_F32; return true;
    case at::kHalf: to = MI355_F16; return true;
    case at::kBFloat16: to = MI355_BF16; return true;
    default: return false;
    }
}

bool type_of(int code, at::ScalarType& to)
{
    switch(code)
    {
    case MI355_I8: to = at::kChar; return true;
    case MI355_U8:
    case MI355_FP8:
    case MI355_BF8: to = at::kByte; return true;
    case MI355_I32: to = at::kInt; return true;
    case MI355_F32: to = at::kFloat; return true;
    case MI355_F16: to = at::kHalf; return true;
    case MI355_BF16: to = at::kBFloat16; return true;
    default: return false;
    }
}

// the type that the caller names, or the result's own: float, or bare whole numbers
bool result_type(PyObject* named, bool dequant, bool fp8, at::ScalarType& type, int& code)
{
    if(named != Py_None && !THPDtype_Check(named))
        return false;
    type = named != Py_None ? reinterpret_cast<THPDtype*>(named)->scalar_type : dequant || fp8 ? at::kFloat : at::kInt;
    return code_of(type, code);
}

bool one_or(const at::Tensor* t, int64_t count) { return t == nullptr || t->numel() == 1 || t->numel() == count; }

// The library's calls run without the interpreter's lock, as they do through ctypes.
template <class F>
PyObject* launch(const char* what, const at::Tensor& result, F&& call)
{
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = call();
    Py_END_ALLOW_THREADS;
    if(status != MI355_OK)
        return PyObject_CallFunction(check_status, "is", status, what);
    return THPVariable_Wrap(result);
}

template <int N, PyObject* (*F)(PyObject* const*)>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    if(count != N)
    {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    try
    {
        return F(args);
    }
    catch(const std::exception&) // torch's errors (out of memory): the Python function meets them again and reports them
    {
        return leave();
    }
}

struct rows_cols
{
    int64_t rows, cols;
    bool of(const at::Tensor& x)
    {
        if(x.dim() < 1)
            return false;
        cols = x.size(-1);
        rows = x.numel() / cols;
        return true;
    }
};

struct parameter
{
    void* data = nullptr;
    int64_t row = 0, col = 0;
    bool of(const at::Tensor& p, const rows_cols& x)
    {
        const int64_t count = p.numel();
        if(count != 1)
        {
            if(p.dim() == 1 && count == x.cols)
                col = 1;
            else if(p.dim() == 1 && count == x.rows)
                row = 1;
            else
            {
                row = x.cols;
                col = 1;
                if(count != x.rows * x.cols)
                    return false;
            }
        }
        data = p.data_ptr();
        return true;
    }
};

// (x, scale, zp, out_type)
PyObject* quantizelinear(PyObject* const* a)
{
    site s;
    rows_cols n;
    parameter scale, zp;
    const at::Tensor *x = nullptr, *st = nullptr, *zt = nullptr;
    int in = 0, to = 0;
    at::ScalarType type;
    PLAIN_IF(s.dense(a[0], x) && n.of(*x) && s.dense(a[1], st) && scale.of(*st, n) && s.room(a[2], zt) &&
             (zt == nullptr || zp.of(*zt, n)) && st->scalar_type() == x->scalar_type() && code_of(x->scalar_type(), in) &&
             integer32(a[3], to) && type_of(to, type) && s.here());
    const at::Tensor out = s.empty(x->sizes(), type);
    return launch("mi355_quantizelinear", out, [&, px = x->data_ptr(), po = out.data_ptr(), stream = s.stream()] {
        return mi355_quantizelinear(px, in, scale.data, scale.row, scale.col, zp.data, zp.row, zp.col, po, to, n.rows, n.cols,
                                    stream);
    });
}

// (x, scale, zp, x_type)
PyObject* dequantizelinear(PyObject* const* a)
{
    site s;
    rows_cols n;
    parameter scale, zp;
    const at::Tensor *x = nullptr, *st = nullptr, *zt = nullptr;
    int from = 0, kind = 0;
    PLAIN_IF(s.dense(a[0], x) && n.of(*x) && s.dense(a[1], st) && scale.of(*st, n) && s.room(a[2], zt) &&
             (zt == nullptr || zp.of(*zt, n)) && (a[3] == Py_None ? code_of(x->scalar_type(), from) : integer32(a[3], from)) &&
             code_of(st->scalar_type(), kind) && s.here());
    const at::Tensor out = s.empty(x->sizes(), st->scalar_type());
    return launch("mi355_dequantizelinear", out, [&, px = x->data_ptr(), po = out.data_ptr(), stream = s.stream()] {
        return mi355_dequantizelinear(px, from, scale.data, kind, scale.row, scale.col, zp.data, zp.row, zp.col, po, n.rows,
                                      n.cols, stream);
    });
}

// (x, axis)
template <bool PACK>
PyObject* int4(PyObject* const* a)
{
    site s;
    rows_cols n;
    const at::Tensor* x = nullptr;
    int64_t axis        = 0;
    PLAIN_IF(s.dense(a[0], x) && n.of(*x) && integer(a[1], axis) && (axis == -1 || axis == x->dim() - 1) &&
             (x->scalar_type() == at::kChar || x->scalar_type() == at::kByte) && (!PACK || n.cols % 2 == 0) && s.here());
    auto sizes   = x->sizes().vec();
    sizes.back() = PACK ? n.cols / 2 : n.cols * 2;
    const at::Tensor out  = s.empty(sizes, x->scalar_type());
    const int is_signed   = x->scalar_type() == at::kChar;
    return launch(PACK ? "mi355_pack_int4" : "mi355_unpack_int4", out,
                  [&, px = x->data_ptr(), po = out.data_ptr(), st = s.stream()] {
                      return PACK ? mi355_pack_int4(px, po, is_signed, n.rows, n.cols, st)
                                  : mi355_unpack_int4(px, po, is_signed, n.rows, n.cols, st);
                  });
}

// (trans, ld) of the last two dimensions: rows side by side, or the transpose of such
bool layout(const at::Tensor& t, int32_t& trans, int64_t& ld)
{
    const int64_t r = t.size(-2), c = t.size(-1), sr = t.stride(-2), sc = t.stride(-1);
    if(sc == 1 || c == 1)
    {
        trans = 0;
        ld    = std::max(r > 1 ? sr : c, c);
        return true;
    }
    trans = 1;
    ld    = std::max(c > 1 ? sc : r, r);
    return sr == 1 || r == 1;
}

bool operand_code(bool fp8, const at::Tensor& t, int32_t& to)
{
    to = fp8 ? MI355_FP8 : t.scalar_type() == at::kByte ? MI355_U8 : MI355_I8;
    return t.scalar_type() == at::kByte || t.scalar_type() == at::kChar;
}

// (a, b, fp8, scale_a, scale_b, zp_a, zp_b, colsum_b, rowsum_a, out_dtype, out, bias, workspace)
PyObject* quant_dot(PyObject* const* v)
{
    site s;
    bool fp8 = false;
    const at::Tensor *ta = nullptr, *tb = nullptr;
    PLAIN_IF(v[10] == Py_None && truth(v[2], fp8) && s.tensor(v[0], ta) && s.tensor(v[1], tb));
    const at::Tensor &a = *ta, &b = *tb;
    PLAIN_IF(a.dim() == b.dim() && (a.dim() == 2 || a.dim() == 3) && a.scalar_type() == b.scalar_type());
    mi355_quant_dot_desc d{};
    d.m     = a.size(-2);
    d.k     = a.size(-1);
    d.n     = b.size(-1);
    d.batch = a.dim() == 3 ? a.size(0) : 1;
    PLAIN_IF(b.size(-2) == d.k && (a.dim() == 2 || b.size(0) == d.batch) && layout(a, d.trans_a, d.lda) &&
             layout(b, d.trans_b, d.ldb) && operand_code(fp8, a, d.in_type));
    d.stride_a = a.dim() == 3 ? a.stride(0) : 0;
    d.stride_b = a.dim() == 3 ? b.stride(0) : 0;
    d.ldc      = d.n;
    d.stride_c = d.m * d.n;
    const at::Tensor *sa = nullptr, *sb = nullptr, *colsum = nullptr, *rowsum = nullptr, *bias = nullptr, *room = nullptr;
    PLAIN_IF(s.vector(v[3], sa) && s.vector(v[4], sb) && s.vector(v[7], colsum) && s.vector(v[8], rowsum) &&
             s.vector(v[11], bias) && s.room(v[12], room));
    const bool dequant = sa != nullptr || sb != nullptr || v[9] != Py_None;
    const bool batched = sb != nullptr && d.batch > 1 && sb->dim() >= 2 && sb->numel() == d.batch * d.n;
    at::ScalarType type;
    PLAIN_IF(result_type(v[9], dequant, fp8, type, d.out_type) && one_or(sa, d.m) && (batched || one_or(sb, d.n)) &&
             (bias == nullptr ||
              (dequant && bias->scalar_type() == at::kFloat && bias->numel() == (batched ? d.batch : 1) * d.n)) &&
             integer32(v[5], d.zp_a) && integer32(v[6], d.zp_b) && s.here());
    d.dequant      = dequant;
    d.scale_a_mode = sa == nullptr ? MI355_QP_NONE : sa->numel() == 1 ? MI355_QP_PER_TENSOR : MI355_QP_PER_ROW;
    d.scale_b_mode = sb == nullptr        ? MI355_QP_NONE
                     : sb->numel() == 1   ? MI355_QP_PER_TENSOR
                     : batched            ? MI355_QP_PER_COL_BATCH
                                          : MI355_QP_PER_COL;
    const std::array<int64_t, 3> sizes{d.batch, d.m, d.n};
    const at::Tensor out = s.empty(a.dim() == 3 ? at::IntArrayRef(sizes) : at::IntArrayRef(sizes.data() + 1, 2), type);
    return launch(room != nullptr   ? "mi355_quant_dot_ws"
                  : bias != nullptr ? "mi355_quant_dot_bias"
                                    : "mi355_quant_dot",
                  out,
                  [&, pa = a.data_ptr(), pb = b.data_ptr(), po = out.data_ptr(), fa = at_data<float>(sa),
                   fb = at_data<float>(sb), cs = at_data<int32_t>(colsum), rs = at_data<int32_t>(rowsum),
                   bi = at_data<float>(bias), ws = at_data<void>(room), bytes = room == nullptr ? 0 : room->nbytes(),
                   st = s.stream()] {
                      return mi355_quant_dot_ws(&d, pa, pb, po, fa, fb, cs, rs, bi, ws, bytes, st);
                  });
}

// (a, b_prepacked, n, fp8, scale_a, scale_b, zp_a, zp_b, colsum_b, rowsum_a, out_dtype, out, bias)
PyObject* quant_dot_prepacked(PyObject* const* v)
{
    site s;
    bool fp8 = false;
    const at::Tensor *ta = nullptr, *b = nullptr;
    PLAIN_IF(v[11] == Py_None && truth(v[3], fp8) && s.tensor(v[0], ta) && s.dense(v[1], b));
    const at::Tensor& a = *ta;
    PLAIN_IF(a.dim() == 2 && a.stride(1) == 1);
    mi355_quant_dot_desc d{};
    d.m     = a.size(0);
    d.k     = a.size(1);
    d.batch = 1;
    d.lda   = d.m > 1 ? a.stride(0) : std::max(d.k, a.stride(0));
    const at::Tensor *sa = nullptr, *sb = nullptr, *colsum = nullptr, *rowsum = nullptr, *bias = nullptr;
    PLAIN_IF(integer(v[2], d.n) && d.n > 0 && operand_code(fp8, a, d.in_type) && s.vector(v[4], sa) && s.vector(v[5], sb) &&
             s.vector(v[8], colsum) && s.vector(v[9], rowsum) && s.vector(v[12], bias));
    d.ldb              = d.n;
    d.ldc              = d.n;
    const bool dequant = sa != nullptr || sb != nullptr || v[10] != Py_None;
    at::ScalarType type;
    PLAIN_IF(result_type(v[10], dequant, fp8, type, d.out_type) && one_or(sa, d.m) && one_or(sb, d.n) &&
             integer32(v[6], d.zp_a) && integer32(v[7], d.zp_b) && s.here());
    d.dequant      = dequant;
    d.scale_a_mode = sa == nullptr ? MI355_QP_NONE : sa->numel() == 1 ? MI355_QP_PER_TENSOR : MI355_QP_PER_ROW;
    d.scale_b_mode = sb == nullptr ? MI355_QP_NONE : sb->numel() == 1 ? MI355_QP_PER_TENSOR : MI355_QP_PER_COL;
    const std::array<int64_t, 2> sizes{d.m, d.n};
    const at::Tensor out = s.empty(sizes, type);
    return launch("mi355_quant_dot_prepacked", out,
                  [&, pa = a.data_ptr(), pb = b->data_ptr(), po = out.data_ptr(), fa = at_data<float>(sa),
                   fb = at_data<float>(sb), cs = at_data<int32_t>(colsum), rs = at_data<int32_t>(rowsum),
                   bi = at_data<float>(bias), st = s.stream()] {
                      return mi355_quant_dot_prepacked(&d, pa, pb, po, fa, fb, cs, rs, bi, st);
                  });
}

// one float for each element of a block-scaled operand, or for each block of 32
bool scale_strides(const at::Tensor& t, int64_t k, int64_t& batch, int64_t& row, int64_t& block, int64_t& elem)
{
    const int64_t cols = t.size(1);
    batch = t.size(0) * cols;
    row   = cols;
    block = cols == k ? 32 : 1;
    elem  = cols == k ? 1 : 0;
    return cols == k || cols * 32 == k;
}

// (a, b_nk, scale_a, scale_b, a_fp4, b_fp4, out, workspace): matrices without batches
PyObject* quant_dot_mx(PyObject* const* v)
{
    site s;
    bool a4 = false, b4 = false;
    const at::Tensor *ta = nullptr, *tb = nullptr, *sat = nullptr, *sbt = nullptr, *given = nullptr;
    PLAIN_IF(v[6] == Py_None && truth(v[4], a4) && truth(v[5], b4) && s.dense(v[0], ta) && s.dense(v[1], tb) &&
             s.dense(v[2], sat) && s.dense(v[3], sbt) && s.room(v[7], given));
    const at::Tensor &a = *ta, &b = *tb, &sa = *sat, &sb = *sbt;
    PLAIN_IF(a.dim() == 2 && b.dim() == 2 && sa.dim() == 2 && sb.dim() == 2 && a.scalar_type() == at::kByte &&
             b.scalar_type() == at::kByte && sa.scalar_type() == at::kFloat && sb.scalar_type() == at::kFloat);
    mi355_mx_dot_desc d{};
    d.m        = a.size(0);
    d.n        = b.size(0);
    d.k        = a.size(1) * (a4 ? 2 : 1);
    d.batch    = 1;
    d.lda      = a.size(1);
    d.ldb      = b.size(1);
    d.ldc      = d.n;
    d.stride_a = d.m * d.lda;
    d.stride_b = d.n * d.ldb;
    d.stride_c = d.m * d.n;
    d.a_type   = a4 ? MI355_FP4X2 : MI355_FP8;
    d.b_type   = b4 ? MI355_FP4X2 : MI355_FP8;
    PLAIN_IF(b.size(1) * (b4 ? 2 : 1) == d.k && sa.size(0) == d.m && sb.size(0) == d.n &&
             scale_strides(sa, d.k, d.sa_batch, d.sa_row, d.sa_block, d.sa_elem) &&
             scale_strides(sb, d.k, d.sb_batch, d.sb_row, d.sb_block, d.sb_elem));
    const size_t need = mi355_quant_dot_mx_workspace_size(&d);
    PLAIN_IF((given == nullptr || given->nbytes() >= need) && s.here());
    const std::array<int64_t, 2> sizes{d.m, d.n};
    const int64_t bytes[1] = {(int64_t)std::max<size_t>(need, 16)};
    const at::Tensor out   = s.empty(sizes, at::kFloat);
    const at::Tensor room  = given == nullptr ? s.empty(bytes, at::kByte) : *given;
    return launch("mi355_quant_dot_mx", out,
                  [&, pa = a.data_ptr(), pb = b.data_ptr(), po = static_cast<float*>(out.data_ptr()), fa = at_data<float>(&sa),
                   fb = at_data<float>(&sb), ws = room.data_ptr(), st = s.stream()] {
                      return mi355_quant_dot_mx(&d, pa, pb, po, fa, fb, ws, need, st);
                  });
}

// (a, w_packed, scales, group, zp, zp_mode, out, workspace)
PyObject* w4a16_gemm(PyObject* const* v)
{
    site s;
    const at::Tensor *ta = nullptr, *wt = nullptr, *scales = nullptr, *room = nullptr, *z = nullptr;
    int64_t group = 0;
    PLAIN_IF(v[6] == Py_None && s.tensor(v[0], ta) && s.dense(v[1], wt) && s.dense(v[2], scales) && s.room(v[7], room) &&
             integer(v[3], group));
    const at::Tensor &a = *ta, &w = *wt;
    PLAIN_IF(a.dim() == 2 && w.dim() == 2 && a.stride(1) == 1 && a.scalar_type() == at::kHalf && w.element_size() == 1 &&
             scales->scalar_type() == at::kHalf && w.size(1) * 2 == a.size(1));
    const int64_t m = a.size(0), k = a.size(1), n = w.size(0);
    int mode = MI355_W4_ZP_SCALAR, scalar = 0;
    if(PyLong_CheckExact(v[4]))
        PLAIN_IF(integer32(v[4], scalar));
    else
    {
        mode = MI355_W4_ZP_GROUP;
        PLAIN_IF(s.dense(v[4], z) && z->element_size() == 1 && (v[5] == Py_None || integer32(v[5], mode)));
    }
    PLAIN_IF(s.here());
    const std::array<int64_t, 2> sizes{m, n};
    const at::Tensor out = s.empty(sizes, at::kHalf);
    return launch(room != nullptr ? "mi355_w4a16_gemm_ws" : "mi355_w4a16_gemm", out,
                  [&, pa = a.data_ptr(), lda = a.stride(0), pw = w.data_ptr(), ps = scales->data_ptr(), po = out.data_ptr(),
                   zp = at_data<void>(z), ws = at_data<void>(room), bytes = room == nullptr ? 0 : room->nbytes(),
                   st = s.stream()] {
                      return mi355_w4a16_gemm_ws(pa, lda, pw, ps, zp, mode, scalar, po, n, m, n, k, group, ws, bytes, st);
                  });
}

// (a, prepacked, n, out)
PyObject* w4a16_gemm_prepacked(PyObject* const* v)
{
    site s;
    const at::Tensor *a = nullptr, *w = nullptr;
    int64_t n = 0;
    PLAIN_IF(v[3] == Py_None && s.tensor(v[0], a) && s.dense(v[1], w) && a->dim() == 2 && a->stride(1) == 1 &&
             a->scalar_type() == at::kHalf && integer(v[2], n) && n > 0 && s.here());
    const int64_t m = a->size(0), k = a->size(1);
    const std::array<int64_t, 2> sizes{m, n};
    const at::Tensor out = s.empty(sizes, at::kHalf);
    return launch("mi355_w4a16_gemm_prepacked", out,
                  [&, pa = a->data_ptr(), lda = a->stride(0), pw = w->data_ptr(), po = out.data_ptr(), st = s.stream()] {
                      return mi355_w4a16_gemm_prepacked(pa, lda, pw, po, n, m, n, k, st);
                  });
}

// two integers, one for either axis, or up to `most` of 4 for both axes' low and high padding; None leaves what is there
bool read_integers(PyObject* o, Py_ssize_t most, int64_t* to, Py_ssize_t& count)
{
    if(o == Py_None)
        return true;
    if(!PyTuple_CheckExact(o) && !PyList_CheckExact(o))
        return false;
    count = PySequence_Fast_GET_SIZE(o);
    if(count != 2 && count != most)
        return false;
    for(Py_ssize_t i = 0; i < count; i++)
    {
        if(!integer(PySequence_Fast_GET_ITEM(o, i), to[i]))
            return false;
    }
    return true;
}

// (x, w, padding, stride, dilation, group, fp8, scale_x, scale_w, out_dtype, out, workspace): two spatial axes
PyObject* quant_convolution(PyObject* const* v)
{
    site s;
    bool fp8 = false;
    const at::Tensor *xt = nullptr, *wt = nullptr, *sx = nullptr, *sw = nullptr;
    PLAIN_IF(v[10] == Py_None && v[11] == Py_None && truth(v[6], fp8) && s.dense(v[0], xt) && s.dense(v[1], wt));
    const at::Tensor &x = *xt, &w = *wt;
    PLAIN_IF(x.dim() == 4 && w.dim() == 4 && x.scalar_type() == w.scalar_type() &&
             x.scalar_type() == (fp8 ? at::kByte : at::kChar));
    int64_t pad[4] = {0, 0, 0, 0}, stride[2] = {1, 1}, dil[2] = {1, 1};
    Py_ssize_t pads = 2, twos = 2;
    mi355_quant_conv_desc d{};
    PLAIN_IF(read_integers(v[2], 4, pad, pads) && read_integers(v[3], 2, stride, twos) && read_integers(v[4], 2, dil, twos) &&
             integer(v[5], d.group));
    d.n        = x.size(0);
    d.c        = x.size(1);
    d.h        = x.size(2);
    d.w        = x.size(3);
    d.o        = w.size(0);
    d.kh       = w.size(2);
    d.kw       = w.size(3);
    d.pad_h    = pad[0];
    d.pad_w    = pad[1];
    d.pad_h_hi = pads == 4 ? pad[2] : pad[0];
    d.pad_w_hi = pads == 4 ? pad[3] : pad[1];
    d.stride_h = stride[0];
    d.stride_w = stride[1];
    d.dil_h    = dil[0];
    d.dil_w    = dil[1];
    PLAIN_IF(d.group >= 1 && w.size(1) * d.group == d.c && d.o % d.group == 0 && s.vector(v[7], sx) && s.vector(v[8], sw) &&
             one_or(sx, 1) && one_or(sw, d.o));
    const bool dequant = sx != nullptr || sw != nullptr || v[9] != Py_None;
    at::ScalarType type;
    PLAIN_IF(result_type(v[9], dequant, fp8, type, d.out_type));
    d.in_type      = fp8 ? MI355_FP8 : MI355_I8;
    d.dequant      = dequant;
    d.scale_x_mode = sx == nullptr ? MI355_QP_NONE : MI355_QP_PER_TENSOR;
    d.scale_w_mode = sw == nullptr ? MI355_QP_NONE : sw->numel() == 1 ? MI355_QP_PER_TENSOR : MI355_QP_PER_ROW;
    std::array<int64_t, 4> sizes{d.n, d.o, 0, 0};
    size_t need = 0;
    PLAIN_IF(mi355_quant_convolution_dims(&d, &sizes[2], &sizes[3], &need) == MI355_OK && s.here());
    const int64_t bytes[1] = {(int64_t)std::max<size_t>(need, 16)};
    const at::Tensor out   = s.empty(sizes, type);
    const at::Tensor room  = s.empty(bytes, at::kByte);
    return launch("mi355_quant_convolution", out,
                  [&, px = x.data_ptr(), pw = w.data_ptr(), po = out.data_ptr(), fx = at_data<float>(sx),
                   fw = at_data<float>(sw), ws = room.data_ptr(), st = s.stream()] {
                      return mi355_quant_convolution(&d, px, pw, po, fx, fw, ws, need, st);
                  });
}

template <int N, PyObject* (*F)(PyObject* const*)>
PyMethodDef method(const char* name)
{
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<N, F>)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {method<4, quantizelinear>("quantizelinear"),
                         method<4, dequantizelinear>("dequantizelinear"),
                         method<2, int4<true>>("pack_int4"),
                         method<2, int4<false>>("unpack_int4"),
                         method<13, quant_dot>("quant_dot"),
                         method<13, quant_dot_prepacked>("quant_dot_prepacked"),
                         method<8, quant_dot_mx>("quant_dot_mx"),
                         method<8, w4a16_gemm>("w4a16_gemm"),
                         method<4, w4a16_gemm_prepacked>("w4a16_gemm_prepacked"),
                         method<12, quant_convolution>("quant_convolution"),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__torch_calls()
{
    PyObject* capi = PyImport_ImportModule("amdmigraphx_amd.capi");
    if(capi == nullptr)
        return nullptr;
    check_status = PyObject_GetAttrString(capi, "check");
    Py_DECREF(capi);
    return check_status == nullptr ? nullptr : PyModule_Create(&module_def);
}
