// Host path of the grouped n:m products: operand caches, choice of the route, allocation of results
// and workspaces, launch.  A product of a few tokens keeps the GPU busy for 7 to 15 us; the same
// steps in Python (attribute look-ups, ctypes conversions, the generic dispatcher) took 24 to 37 us
// per call, so they bounded every small product whatever its kernel did.  Built as the extension
// module sten_amd._host and linked against libnmg_hip.so, whose C ABI stays the only way to a kernel.
//
// Everything here runs with the GIL held (nothing blocks); that is what makes the operand caches safe
// with several threads.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <map>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/nmg_hip.h"

namespace {

using at::Tensor;

constexpr long kInterface = 2;        // INTERFACE in sten_amd/_host_loader.py
PyObject *g_nmg_error = nullptr;      // sten_amd.native.NmgError

struct NmgError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

template <typename... A>
[[noreturn]] void fail(const A &...parts)
{
    std::ostringstream s;
    (s << ... << parts);
    throw NmgError(s.str());
}

void check(int rc)
{
    if (rc != NMG_OK) fail("nmg call failed with status ", rc, ": ", nmg_last_error());
}

#define HOST_TRY try {
#define HOST_CATCH(ret)                                                       \
    }                                                                         \
    catch (const NmgError &e) { PyErr_SetString(g_nmg_error, e.what()); return ret; } \
    catch (python_error &e) { e.restore(); return ret; }                      \
    catch (const c10::Error &e) { PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace()); return ret; } \
    catch (const std::exception &e) { PyErr_SetString(PyExc_RuntimeError, e.what()); return ret; }

// ---------------------------------------------------------------------------------- small helpers

struct Text {
    PyObject *kernel, *variant, *dense_variant, *slices, *expand, *cache_dense, *container, *dense_shape, *B, *s, *meta, *grad_fmt, *data, *alpha;
    PyObject *arguments[4], *nothing;      // names of __torch_function__'s, ()
} S_;

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return NMG_F32;
    case at::kHalf: return NMG_F16;
    case at::kBFloat16: return NMG_BF16;
    case at::kDouble: return NMG_F64;
    default: fail("unsupported dtype ", t);
    }
}

bool is16(const Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

void require_gpu(const Tensor &t)
{
    if (!t.is_cuda())
        fail("nmg kernels run on the GPU only; got a tensor on ", t.device(), " (move the tensor to an MI355X device)");
}

void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor new_empty(at::IntArrayRef size, const Tensor &like) { return at::empty(size, like.options()); }
Tensor new_empty(at::IntArrayRef size, const Tensor &like, at::ScalarType dt) { return at::empty(size, like.options().dtype(dt)); }

bool aligned16(const Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }
int64_t round_up(int64_t a, int64_t b) { return up(a, b) * b; }

// t (2-D) with contiguous rows that do not overlap: t itself where they lie so, else a copy.
bool rows_lie(const Tensor &t)
{
    const int64_t R = t.size(0), C = t.size(1);
    return (C <= 1 || t.stride(1) == 1) && (R <= 1 || t.stride(0) >= C);
}
Tensor rows_of(const Tensor &t) { return rows_lie(t) ? t : t.contiguous(); }

// t (16-bit, 2-D) as rows of at least `cols` elements that start on 16 bytes, zeros from t's extent on, and at
// least `rows` of them: t itself where it is that already, else a copy.
Tensor padded(const Tensor &t, int64_t rows, int64_t cols)
{
    const int64_t R = t.size(0), C = t.size(1);
    const Tensor s = rows_of(t);
    if (R == rows && C == cols && (R <= 1 || s.stride(0) % 8 == 0) && aligned16(s)) return s;
    Tensor out = new_empty({rows, cols}, t);
    check(nmg_copy_rows16(s.data_ptr(), R, C, R > 1 ? s.stride(0) : C, out.data_ptr(), rows, cols, cols, stream_of(t)));
    return out;
}

// b^T (b [K, N], 16-bit) as rows of Kp >= K elements that start on 16 bytes, zeros from K on.
Tensor transposed(const Tensor &b, int64_t Kp)
{
    const int64_t K = b.size(0), N = b.size(1);
    if (b.stride(0) == 1 && b.stride(1) != 1) return padded(b.t(), N, Kp);
    const Tensor s = rows_of(b);
    Tensor out = new_empty({N, Kp}, b);
    check(nmg_transpose16(s.data_ptr(), K, N, K > 1 ? s.stride(0) : N, out.data_ptr(), Kp, Kp, stream_of(b)));
    return out;
}

int64_t pitch_of(const Tensor &t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

// pitch_of(padded(t, t.size(0), round_up(t.size(1), 8)))
int64_t pitch_of_whole_pieces(const Tensor &t)
{
    const bool kept = rows_lie(t) && t.size(0) > 1 && t.size(1) % 8 == 0 && t.stride(0) % 8 == 0 && aligned16(t);
    return kept ? t.stride(0) : round_up(t.size(1), 8);
}

constexpr int64_t k2G = int64_t(1) << 31;
constexpr int64_t kOstreamMaxTokens = 4;    // nmg_spmm_ostream: the token rows its lanes hold
constexpr int64_t kOstreamAutoTokens = 2;   // ... and up to where it is ahead of the sliced kernel (4096 x 11008: 12.4 / 13.3 / 16.2 against 15.9 / 16.0 / 16.3 us at 1 / 2 / 3 tokens)
constexpr int64_t kGstreamMaxTokens = 16;   // nmg_spmm_gstream: tokens up to which the stream of the weight bounds the product
// Activations whose rows are no whole number of 128-byte lines, a copy in whole K steps of 64 against the rows as they lie: a tile's
// piece of a row then reaches into two lines, and every line tile reads it again, from memory where no cache holds the activations; from some
// size on that costs more than the copy and its launch.  Time with the copy over time as they lie, 29 weights of 520 x 200 to 8200 x 8104
// with 32 to 2000 tokens, 2:4 / 4:8, weights and activations from memory: up to 7.2 Mi weights 1.07 to 1.45 / 1.05 to 1.43 at 100 to 500 tokens,
// up to 64 tokens 1.22 to 1.41 / 1.0 (the kernel for few tokens, either way) to 1.31.  Beyond the line 7.8 to 13.7 Mi weights would still gain
// (1.02 to 1.21 / 1.0 to 1.20), as would more tokens (1.0 to 1.45; 1768 x 4088 x 1000 alone loses, 0.98); 16 Mi and more lose as often as not
// (0.84 to 1.12 / 0.90 to 1.15, most with many outputs and a short reduction: 12000 x 2056 0.84 to 0.94), but up to 64 tokens
// still gain 1.04 to 1.27 / 1.0 to 1.25.  With everything in the caches 1.0 to 1.7 up to 14 Mi, 0.86 to 1.23 beyond.
constexpr int64_t kRaggedMost = 15 << 19;
constexpr int64_t kF32GemmMaxTokens = 65535 * 32;   // one launch of the fp32 GEMM: token tiles of 32 in grid.y

// ------------------------------------------------------------------------------- the tensor's core

struct Geometry {
    int nd = 0, n = 0, m = 0, g = 0, sdim = 0, gdim = 0;
    std::vector<int64_t> dims;
    int64_t G = 0, S = 0, nb = 0, cols = 0, chunks = 0;
};

// What is derived from val and idx for the products; dropped when either changes.
struct Operands {
    bool valid = false;
    uint32_t val_version = 0, idx_version = 0;
    Tensor pk_val, pk_pat, fp_val, fp_idx;      // rowpack, and fragpack where the pattern has one
    Tensor frag[2];                             // densefrag per reduction direction
    std::map<int64_t, Tensor> dense[2];         // dense copies per reduction direction, by row pitch
    Tensor lp_val, lp_pat, gp, op;              // operands of the streamed few-token products
};

struct State {
    Tensor val, idx;
    PyObject *layout = nullptr, *opt = nullptr;
    Geometry geo;
    Operands ops;
    bool slot_valid = false;
    uint32_t slot_version = 0;
    Tensor slot;
};

struct Core {
    PyObject_HEAD
    State *st;
};

PyTypeObject CoreType = {PyVarObject_HEAD_INIT(nullptr, 0)};

State &state_of(PyObject *o)
{
    if (!PyObject_TypeCheck(o, &CoreType)) fail("expected a GroupedNMTensor, got ", Py_TYPE(o)->tp_name);
    return *reinterpret_cast<Core *>(o)->st;
}

State &matmul_state(PyObject *o)
{
    State &w = state_of(o);
    if (w.geo.nd != 2) fail("matmul needs a 2-D grouped n:m tensor");
    return w;
}

// The operands of the present val / idx: an in-place change of either shows in its version.
Operands &operands(State &w)
{
    const uint32_t vv = w.val._version(), iv = w.idx._version();
    if (!w.ops.valid || w.ops.val_version != vv || w.ops.idx_version != iv) {
        w.ops = Operands();
        w.ops.valid = true;
        w.ops.val_version = vv;
        w.ops.idx_version = iv;
    }
    return w.ops;
}

long opt_long(PyObject *d, PyObject *key, long dflt)
{
    PyObject *v = PyDict_GetItemWithError(d, key);
    if (v == nullptr) {
        if (PyErr_Occurred()) throw python_error();
        return dflt;
    }
    PyObject *whole = PyNumber_Long(v);      // what int() takes
    if (whole == nullptr) throw python_error();
    const long r = PyLong_AsLong(whole);
    Py_DECREF(whole);
    if (r == -1 && PyErr_Occurred()) throw python_error();
    return r;
}

bool opt_bool(PyObject *d, PyObject *key, bool dflt)
{
    PyObject *v = PyDict_GetItemWithError(d, key);
    if (v == nullptr) {
        if (PyErr_Occurred()) throw python_error();
        return dflt;
    }
    const int r = PyObject_IsTrue(v);
    if (r < 0) throw python_error();
    return r != 0;
}

struct Options {
    std::string kernel = "auto";
    long variant = -1, dense_variant = -1, slices = -1;      // slices: -1 where none are asked for
    bool expand = true, cache_dense = true;
};

Options options_of(const State &w)
{
    Options o;
    PyObject *k = PyDict_GetItemWithError(w.opt, S_.kernel);
    if (k != nullptr) {
        const char *c = PyUnicode_AsUTF8(k);
        if (c == nullptr) throw python_error();
        o.kernel = c;
    }
    if (PyDict_Size(w.opt) > (k != nullptr ? 1 : 0)) {
        o.variant = opt_long(w.opt, S_.variant, -1);
        o.dense_variant = opt_long(w.opt, S_.dense_variant, -1);
        if (PyDict_Contains(w.opt, S_.slices) == 1) o.slices = std::max(opt_long(w.opt, S_.slices, 0), 0L);
        o.expand = opt_bool(w.opt, S_.expand, true);
        o.cache_dense = opt_bool(w.opt, S_.cache_dense, true);
    }
    return o;
}

// ------------------------------------------------------------------------------- derived operands

void pack(State &w)
{
    Operands &o = operands(w);
    if (o.pk_val.defined()) return;
    const Geometry &q = w.geo;
    require_gpu(w.val);
    const bool narrow = nmg_rowpack_pat_bytes(q.n, q.m) == 1;
    Tensor pk_val = new_empty({q.G, q.nb, q.n}, w.val);
    Tensor pk_pat = new_empty({q.G, q.nb}, w.val, narrow ? at::kByte : at::kShort);
    Tensor fp_val, fp_idx;
    if (is16(w.val) && nmg_fragpack_supported(q.n, q.m)) {
        int64_t ve = 0, iw = 0;
        check(nmg_fragpack_sizes(q.G, q.S, &ve, &iw));
        fp_val = new_empty({ve}, w.val);
        fp_idx = new_empty({iw}, w.val, at::kInt);
    }
    check(nmg_pack_operands(w.val.data_ptr(), (const int16_t *)w.idx.data_ptr(), q.G, q.S, pk_val.data_ptr(), pk_pat.data_ptr(),
                            fp_val.defined() ? fp_val.data_ptr() : nullptr, fp_idx.defined() ? fp_idx.data_ptr() : nullptr,
                            q.n, q.m, q.g, dtype_code(w.val.scalar_type()), stream_of(w.val)));
    o.pk_val = pk_val;
    o.pk_pat = pk_pat;
    o.fp_val = fp_val;
    o.fp_idx = fp_idx;
}

// The weight as the A operand of the dense matrix cores, [outputs, reduction] in fragment order.
Tensor densefrag(State &w, int rd, bool keep)
{
    Operands &o = operands(w);
    if (keep && o.frag[rd].defined()) return o.frag[rd];
    if (!keep) o.frag[0] = o.frag[1] = Tensor();
    pack(w);
    const Geometry &q = w.geo;
    int64_t elems = 0;
    check(nmg_densefrag_elems(q.dims[1 - rd], q.dims[rd], &elems));
    Tensor df = new_empty({elems}, w.val);
    // rowpack lines run along the group dim
    check(nmg_densefrag(o.pk_val.data_ptr(), o.pk_pat.data_ptr(), q.G, q.S, q.gdim == rd ? 1 : 0, df.data_ptr(), q.n, q.m,
                        dtype_code(w.val.scalar_type()), stream_of(w.val)));
    if (keep) o.frag[rd] = df;
    return df;
}

// Dense copy [outputs, reduction] of the weight, rows zero-padded to a multiple of pad_k.
Tensor dense_operand(State &w, int rd, bool keep, int64_t pad_k)
{
    Operands &o = operands(w);
    const Geometry &q = w.geo;
    const int64_t O = q.dims[1 - rd], K = q.dims[rd], Kp = up(K, pad_k) * pad_k;
    if (keep) {
        auto it = o.dense[rd].find(Kp);
        if (it != o.dense[rd].end()) return it->second;
    }
    Tensor out = Kp == K ? new_empty({O, Kp}, w.val) : at::zeros({O, Kp}, w.val.options());
    require_gpu(w.val);
    // Straight from val / idx where two tiles fit the LDS that the scatter has for them, else by way of the rowpack: its two
    // passes cost 21 us for 768 x 3072 2:4:16 in single precision, the scatter 7.5; 74 and 30 for 3712 x 3584 4:8:32.
    if (q.cols * q.m * (int64_t)w.val.element_size() * 2 <= 150 * 1024 && q.nb >= 4) {
        const nmg_view v{1, q.G, q.S, 0, q.gdim == rd ? 1 : Kp, q.sdim == rd ? 1 : Kp};
        check(nmg_to_dense(w.val.data_ptr(), (const int16_t *)w.idx.data_ptr(), out.data_ptr(), &v, q.n, q.m, q.g,
                           dtype_code(w.val.scalar_type()), stream_of(w.val)));
        if (keep) o.dense[rd][Kp] = out;
        return out;
    }
    pack(w);
    check(nmg_rowpack_expand(o.pk_val.data_ptr(), o.pk_pat.data_ptr(), q.G, q.S, out.data_ptr(), Kp, q.gdim == rd ? 1 : 0, q.n,
                             q.m, dtype_code(w.val.scalar_type()), stream_of(w.val)));
    if (keep) o.dense[rd][Kp] = out;      // only an operand that was written is kept
    return out;
}

void lanepack8(State &w)
{
    Operands &o = operands(w);
    if (o.lp_val.defined()) return;
    pack(w);
    const Geometry &q = w.geo;
    int64_t ve = 0, pb = 0;
    check(nmg_lanepack8_sizes(q.G, q.S, q.n, &ve, &pb));
    Tensor lp_val = new_empty({ve}, w.val), lp_pat = new_empty({pb}, w.val, at::kByte);
    check(nmg_lanepack8(o.pk_val.data_ptr(), o.pk_pat.data_ptr(), q.G, q.S, q.n, lp_val.data_ptr(), lp_pat.data_ptr(),
                        dtype_code(w.val.scalar_type()), stream_of(w.val)));
    o.lp_val = lp_val;
    o.lp_pat = lp_pat;
}

template <typename Bytes, typename Pack>
void stream_operand(State &w, Tensor Operands::*slot, Bytes bytes_of, Pack pack_to)
{
    Operands &o = operands(w);
    if ((o.*slot).defined()) return;
    pack(w);
    const Geometry &q = w.geo;
    int64_t bytes = 0;
    check(bytes_of(q.G, q.S, q.n, q.m, &bytes));
    Tensor t = new_empty({std::max<int64_t>(bytes, 16)}, w.val, at::kByte);
    check(pack_to(o.pk_val.data_ptr(), o.pk_pat.data_ptr(), q.G, q.S, q.n, q.m, t.data_ptr(), dtype_code(w.val.scalar_type()),
                  stream_of(w.val)));
    o.*slot = t;
}

void gpack(State &w) { stream_operand(w, &Operands::gp, nmg_gpack_bytes, nmg_gpack); }
void opack(State &w) { stream_operand(w, &Operands::op, nmg_opack_bytes, nmg_opack); }

Tensor slotmap(State &w)
{
    const Geometry &q = w.geo;
    if (q.nd != 2) fail("the slot map needs a 2-D grouped n:m tensor");
    const uint32_t iv = w.idx._version();
    if (w.slot_valid && w.slot_version == iv) return w.slot;
    require_gpu(w.idx);
    Tensor slot = new_empty({q.nb, q.chunks * q.cols}, w.idx, at::kShort);
    check(nmg_slotmap((const int16_t *)w.idx.data_ptr(), q.G, q.S, (int16_t *)slot.data_ptr(), q.n, q.m, q.g, stream_of(w.idx)));
    w.slot = slot;
    w.slot_version = iv;
    w.slot_valid = true;
    return slot;
}

// ------------------------------------------------------------------------------- views of dense data

std::string shape_text(const Tensor &t)
{
    std::ostringstream s;
    s << "(";
    for (int64_t d = 0; d < t.dim(); d++) s << (d ? ", " : "") << t.size(d);
    s << (t.dim() == 1 ? ",)" : ")");
    return s.str();
}

// t as [batch, G, S] with element strides; `t` is replaced by a re-ordered copy where the other dims
// do not collapse into one stride.
nmg_view view_of(Tensor &t, const Geometry &q)
{
    if (t.sizes() != at::IntArrayRef(q.dims)) fail("the dense tensor must have the shape of the layout, got ", shape_text(t));
    if (q.nd == 2) return nmg_view{1, q.G, q.S, 0, t.stride(q.gdim), t.stride(q.sdim)};
    std::vector<int64_t> perm;
    for (int d = 0; d < q.nd; d++)
        if (d != q.sdim && d != q.gdim) perm.push_back(d);
    perm.push_back(q.gdim);
    perm.push_back(q.sdim);
    t = t.permute(perm).reshape({-1, q.G, q.S});     // a view wherever there is one
    return nmg_view{t.size(0), q.G, q.S, t.size(0) > 1 ? t.stride(0) : 0, t.stride(1), t.stride(2)};
}

Tensor gather(State &w, const Tensor &dense)
{
    require_gpu(dense);
    require_gpu(w.val);
    Tensor t = dense.scalar_type() == w.val.scalar_type() ? dense : dense.to(w.val.scalar_type());
    nmg_view v = view_of(t, w.geo);
    Tensor val = at::empty_like(w.val);
    check(nmg_gather(t.data_ptr(), &v, (const int16_t *)w.idx.data_ptr(), val.data_ptr(), w.geo.n, w.geo.m, w.geo.g,
                     dtype_code(val.scalar_type()), stream_of(t)));
    return val;
}

// ---------------------------------------------------------------------------------------- products

const char *dtype_name(const Tensor &t)
{
    switch (t.scalar_type()) {
    case at::kFloat: return "torch.float32";
    case at::kHalf: return "torch.float16";
    case at::kBFloat16: return "torch.bfloat16";
    case at::kDouble: return "torch.float64";
    default: return "another dtype";
    }
}

Tensor workspace(int64_t floats, const Tensor &like) { return new_empty({std::max<int64_t>(floats, 1)}, like, at::kFloat); }

int64_t split_ws(int slices, int64_t T, int64_t O) { return slices * T * up(O, 256) * 256; }

// A product in single precision, operands as they lie (form 0: nmg_gemm_nt, 1: nmg_gemm_nn, 2: nmg_gemm_tn), its reduction in slices where
// its results are too few tiles for the chip.
void product_f32(int form, const Tensor &a, int64_t lda, const Tensor &x, int64_t ldx, Tensor &y, const void *bias, int64_t O, int64_t K, int64_t T)
{
    int slices = 1;
    int64_t bytes = 0;
    check(nmg_gemm_f32_plan(lda, ldx, O, K, T, form, &slices, &bytes));
    Tensor ws;
    if (slices > 1) ws = workspace(bytes / 4, y);
    check(nmg_gemm_f32_splitk(a.data_ptr(), lda, x.data_ptr(), ldx, y.data_ptr(), O, bias, O, K, T, form, slices,
                              slices > 1 ? ws.data_ptr() : nullptr, bytes, stream_of(y)));
}

// The code of the kernel that takes what no other route does; KeyError for a name that there is no kernel of.
int kernel_code(const std::string &name)
{
    static const std::map<std::string, int> codes = {
        {"mfma", NMG_KERNEL_MFMA}, {"expand", NMG_KERNEL_MFMA}, {"densefrag", NMG_KERNEL_MFMA},
        {"smfmac", NMG_KERNEL_SMFMAC}, {"skinny", NMG_KERNEL_SKINNY}, {"gstream", NMG_KERNEL_SKINNY},
        {"sstream", NMG_KERNEL_SKINNY}, {"ostream", NMG_KERNEL_SKINNY}};
    const auto it = codes.find(name);
    if (it != codes.end()) return it->second;
    PyObject *key = PyUnicode_FromString(name.c_str());
    if (key != nullptr) PyErr_SetObject(PyExc_KeyError, key);
    Py_XDECREF(key);
    throw python_error();
}

// Y = X @ op(W): rd = 1 is X [T, C] @ W^T (F.linear forward), rd = 0 is X [T, R] @ W (the input's gradient).
Tensor spmm(State &w, Tensor x, Tensor bias, int rd, const char *kernel)
{
    const Geometry &q = w.geo;
    require_gpu(x);
    require_gpu(w.val);
    if (bias.defined()) require_gpu(bias);
    if (x.scalar_type() != w.val.scalar_type())
        fail("dtype mismatch: activations ", dtype_name(x), ", weight ", dtype_name(w.val));
    const bool reduce_sparse = rd == q.sdim;
    const int64_t K = q.dims[rd], O = q.dims[1 - rd];
    if (x.dim() != 2 || x.size(1) != K) fail("activations must be [tokens, ", K, "], got ", shape_text(x));
    c10::DeviceGuard device(x.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    const int64_t T = x.size(0);
    if (x.stride(1) != 1 || (T > 1 && x.stride(0) < K)) x = x.contiguous();      // (the kernels take no rows that share memory)
    const int64_t ldx = T > 1 ? x.stride(0) : K;      // the stride of a dim of extent 1 means nothing
    Tensor y = new_empty({T, O}, x);
    if (bias.defined()) bias = bias.to(x.scalar_type()).contiguous();
    const Options opt = options_of(w);
    const std::string kname = kernel != nullptr ? kernel : opt.kernel;
    const bool automatic = kname == "auto";
    const int code = automatic ? NMG_KERNEL_AUTO : kernel_code(kname);
    const int dt = dtype_code(x.scalar_type());
    const bool half = is16(x), al = aligned16(x);
    void *const stream = stream_of(x);
    void *const xp = x.data_ptr(), *const yp = y.data_ptr(), *const bp = bias.defined() ? bias.data_ptr() : nullptr;

    if (kname == "skinny" && T > 16) fail("the skinny kernel serves at most 16 tokens");
    // Few tokens on blocks of 8 along the reduction (1:8, 2:8, 4:8): the rowpack operand holds 0.375 /
    // 0.625 / 1.125 bytes per dense weight where the operand of the sparse matrix cores holds 1.125
    // (and 4:8 has none): streamed once, expanded in registers, one kernel.
    if ((automatic || kname == "sstream") && reduce_sparse && T <= 16 && half && nmg_spmm_sstream_supported(q.n, q.m) && K % 256 == 0
        // weights of fewer than 3072 lines with more than 8 tokens: the operand of the sparse matrix
        // cores streams as fast or faster although it is larger (4:8 has none)
        && (!automatic || q.n == 4 || O >= 96 * 32 || T <= 8) && ldx % 8 == 0 && al
        && T * std::max(ldx, K) * 2 < k2G && 32 * (K / 8) * q.n * 2 < k2G) {
        lanepack8(w);
        check(nmg_spmm_sstream(w.ops.lp_val.data_ptr(), w.ops.lp_pat.data_ptr(), O, K, xp, ldx, yp, O, bp, T, q.n, q.m, dt, stream));
        return y;
    }
    if (kname == "sstream")
        fail("the streaming product along the sparse dim needs 16-bit data, at most 16 tokens, "
             "1:8, 2:8 or 4:8 and a reduction extent that is a multiple of 256");
    const bool flat = T * ldx * 2 < k2G;
    // An extent, a pitch or a start that the matrix-core kernels do not read gets a copy of the activations with
    // whole K steps of 64 (nmg_align.hip).  The sparse cores' operand holds whole steps anyway, the dense cores'
    // operand is padded; in both, what lies behind the reduction is zero.  Reductions that are a multiple of 8 but
    // not of 64 go as they lie, from 17 tokens on to the kernels with tiles, which clear the last step's pieces in LDS,
    // but for large weights (kRaggedMost).
    const bool plain8 = K % 8 == 0 && ldx % 8 == 0 && al, plain64 = K % 64 == 0 && plain8;
    const bool pad_ok = half && (automatic || kname == "densefrag") && opt.expand && T * round_up(K, 64) * 2 < k2G && T > 0 && K > 0;
    const bool smf_pad = pad_ok && automatic && opt.variant == -1 && reduce_sparse && (T > 16 ? plain8 && !plain64 : !plain8)
                         && nmg_fragpack_supported(q.n, q.m);
    const bool smf_ok = reduce_sparse && plain8 && half;
    const bool ragged = plain8 && !plain64 && flat && (T <= 64 || (T <= 512 && O * K <= kRaggedMost));
    bool packed = false;
    if (smf_pad) {
        pack(w);
        packed = w.ops.fp_val.defined();
        const int64_t Kp = round_up(K, 64);
        const void *fv = w.ops.fp_val.data_ptr(), *fi = w.ops.fp_idx.data_ptr();
        int slices = 1;
        int64_t bytes = 0;
        if (T > 16) check(nmg_smfmac_plan(O, Kp, T, &slices, &bytes));
        if (ragged) {      // (more than 16 tokens: `smf_pad`)
            Tensor ws;
            if (slices > 1) ws = workspace(split_ws(slices, T, O), x);
            check(nmg_spmm_smfmac_ragged(fv, fi, O, K, xp, ldx, yp, O, bp, T, dt, slices, slices > 1 ? ws.data_ptr() : nullptr, bytes, stream));
            return y;
        }
        const Tensor xq = padded(x, T, Kp);
        if (slices > 1) {
            Tensor ws = workspace(split_ws(slices, T, O), x);
            check(nmg_spmm_smfmac_splitk(fv, fi, O, Kp, xq.data_ptr(), pitch_of(xq), yp, O, bp, T, dt, slices, ws.data_ptr(), ws.numel() * 4, stream));
        } else {
            check(nmg_spmm_smfmac(fv, fi, O, Kp, xq.data_ptr(), pitch_of(xq), yp, O, bp, T, dt, T <= 16 ? 5 : -1, stream));
        }
        return y;
    }
    if (smf_ok && (automatic || kname == "skinny" || kname == "smfmac")) {
        pack(w);
        packed = w.ops.fp_val.defined();
    }
    if (kname == "smfmac" && !packed)
        fail("the sparse-matrix-core kernel needs 16-bit data, a 2-of-4 compatible n:m "
             "pattern along the reduction dim and 16-byte aligned activations");
    if (packed) {
        const void *fv = w.ops.fp_val.data_ptr(), *fi = w.ops.fp_idx.data_ptr();
        long variant = opt.variant;
        if (T <= 16 && kname != "smfmac")
            variant = 5;      // decode shapes: streaming kernel on the same operand
        else if (T <= 24 && automatic && variant == -1 && K % 128 == 0 && flat && opt.slices < 0)
            // 17 .. 24 tokens: the streaming kernel with the second half of its 32 token columns in
            // use is still ahead of the sliced reduction (4096 x 11008: 15.8 / 17.9 against 18.2 /
            // 18.7 us at 17 / 24 tokens; at 32 tokens 20.1 against 19.3)
            variant = 5;
        if (T > 16 && variant == -1 && K % 64 == 0 && flat) {
            // few tiles for the chip: the reduction is cut into slices, summed by a second kernel
            int slices = 1;
            int64_t bytes = 0;
            check(nmg_smfmac_plan(O, K, T, &slices, &bytes));
            if (opt.slices >= 0) slices = (int)opt.slices;
            if (slices > 1) {
                Tensor ws = workspace(split_ws(slices, T, O), x);
                check(nmg_spmm_smfmac_splitk(fv, fi, O, K, xp, ldx, yp, O, bp, T, dt, slices, ws.data_ptr(), ws.numel() * 4, stream));
                return y;
            }
        }
        check(nmg_spmm_smfmac(fv, fi, O, K, xp, ldx, yp, O, bp, T, dt, (int)variant, stream));
        return y;
    }
    // Few tokens as well when the choice is automatic: without a sparse-core operand (another
    // pattern, the reduction along the group dim, fp32) the alternative for <= 16 tokens is the untuned
    // streaming kernel.  4096 x 11008 at 1 / 4 / 16 tokens: 4:8 25 / 25 / 26 us on the dense-core
    // operand with the reduction cut into slices against 63 / 119 / 342; 2:4 reduced along the
    // group dim (the reference's default orientation) 24 / 25 / 26 against 1190 / 1203 / 1286; fp32
    // 65 / 65 / 65 against 70 / 134 / 361.
    const int64_t min_t = automatic ? 1 : 17;
    // Few tokens with the reduction along the group dim (what F.linear does with a weight in the
    // reference's default orientation): the compressed lines are streamed once and expanded in
    // registers -- 51 MB instead of the 90 MB of the dense-core operand for 4096 x 11008 at 2:4.
    // ... and with a handful of tokens at 2:4 every workgroup owns 16 outputs over the whole
    // reduction: one kernel, no sums through memory (the token rows are then read by every
    // workgroup, which is why this is for few of them)
    if (pad_ok && automatic && !reduce_sparse && T <= kGstreamMaxTokens && !plain8 && nmg_spmm_gstream_supported(q.n, q.m)) {
        // the streams take lines in groups of 8; those behind the last are zero in the operand and in the copy
        const int64_t Kp = round_up(K, 8);
        const Tensor xq = padded(x, T, Kp);
        if (T <= kOstreamAutoTokens && nmg_spmm_ostream_supported(q.n, q.m)) {
            opack(w);
            check(nmg_spmm_ostream(w.ops.op.data_ptr(), Kp, O, xq.data_ptr(), pitch_of(xq), yp, O, bp, T, q.n, q.m, dt, stream));
            return y;
        }
        gpack(w);
        int slices = 1;
        int64_t bytes = 0;
        check(nmg_spmm_gstream_plan(Kp, O, T, q.n, q.m, &slices, &bytes));
        Tensor ws = workspace(bytes / 4, x);
        check(nmg_spmm_gstream(w.ops.gp.data_ptr(), Kp, O, xq.data_ptr(), pitch_of(xq), yp, O, bp, T, q.n, q.m, dt, ws.data_ptr(), ws.numel() * 4, stream));
        return y;
    }
    const bool few_ok = !reduce_sparse && half && plain8 && flat;
    if ((automatic || kname == "ostream") && few_ok && T <= (automatic ? kOstreamAutoTokens : kOstreamMaxTokens)
        && nmg_spmm_ostream_supported(q.n, q.m)) {
        opack(w);
        check(nmg_spmm_ostream(w.ops.op.data_ptr(), K, O, xp, ldx, yp, O, bp, T, q.n, q.m, dt, stream));
        return y;
    }
    if (kname == "ostream")
        fail("the product with 16 outputs per workgroup needs 16-bit data, 2:4, the reduction along "
             "the group dim, at most ", kOstreamMaxTokens, " tokens and a reduction extent that is a multiple of 8");
    if ((automatic || kname == "gstream") && few_ok && T <= kGstreamMaxTokens && nmg_spmm_gstream_supported(q.n, q.m)) {
        gpack(w);
        int slices = 1;
        int64_t bytes = 0;
        check(nmg_spmm_gstream_plan(K, O, T, q.n, q.m, &slices, &bytes));
        Tensor ws = workspace(bytes / 4, x);
        check(nmg_spmm_gstream(w.ops.gp.data_ptr(), K, O, xp, ldx, yp, O, bp, T, q.n, q.m, dt, ws.data_ptr(), ws.numel() * 4, stream));
        return y;
    }
    if (kname == "gstream")
        fail("the streaming product along the group dim needs 16-bit data, at most ", kGstreamMaxTokens,
             " tokens, m = 4 or 8 with n = 1 or 2 and a reduction extent that is a multiple of 8");
    const bool dense16 = T >= min_t && half && plain64 && flat;
    if ((automatic || kname == "mfma" || kname == "densefrag") && (dense16 || (pad_ok && T >= min_t)) && nmg_densefrag_supported(q.n, q.m)
        && (kname == "densefrag" || opt.expand)) {
        // "expand, then multiply": one HBM-bound pass writes the weight in the register order of
        // the dense matrix cores into scratch, the pipelined kernel multiplies from there
        Tensor df = densefrag(w, rd, opt.cache_dense);
        if (plain8 && !plain64 && flat && opt.slices < 0 && opt.dense_variant == -1 && nmg_densefrag_few(O, K, T)) {
            // activations as they are: the kernel for few tokens takes a reduction that is no whole number of K steps
            check(nmg_spmm_densefrag_few(df.data_ptr(), O, K, xp, ldx, yp, O, bp, T, dt, stream));
            return y;
        }
        const int64_t Kp = round_up(K, 64);
        if (ragged && opt.slices < 0 && opt.dense_variant == -1) {
            int slices = 1;
            int64_t bytes = 0;
            check(nmg_densefrag_plan(O, Kp, T, &slices, &bytes));
            Tensor ws;
            if (slices > 1) ws = workspace(split_ws(slices, T, O), x);
            check(nmg_spmm_densefrag_ragged(df.data_ptr(), O, K, xp, ldx, yp, O, bp, T, dt, slices, slices > 1 ? ws.data_ptr() : nullptr, bytes, stream));
            return y;
        }
        const Tensor xq = dense16 ? x : padded(x, T, Kp);
        const void *const xp = xq.data_ptr();
        const int64_t ldx = dense16 ? (T > 1 ? x.stride(0) : K) : pitch_of(xq), K = Kp;
        int slices = 1;
        int64_t bytes = 0;
        if (opt.dense_variant == -1) check(nmg_densefrag_plan(O, K, T, &slices, &bytes));
        if (opt.slices >= 0) slices = (int)opt.slices;
        if (slices > 1) {
            // few tiles for the chip: the reduction is cut into slices, summed by a second kernel
            Tensor ws = workspace(split_ws(slices, T, O), x);
            check(nmg_spmm_densefrag_splitk(df.data_ptr(), O, K, xp, ldx, yp, O, bp, T, dt, slices, ws.data_ptr(), ws.numel() * 4, stream));
            return y;
        }
        check(nmg_spmm_densefrag(df.data_ptr(), O, K, xp, ldx, yp, O, bp, T, dt, (int)opt.dense_variant, stream));
        return y;
    }
    if (kname == "densefrag")
        fail("the densefrag route needs 16-bit data, more than 16 tokens, an m that is a power of two or three times one "
             "and a reduction extent that is a multiple of 64");
    if (kname == "expand") {
        if (!(dense16 && O * K * 2 < k2G))
            fail("the expand-then-multiply route needs 16-bit data, more than 16 tokens "
                 "and a reduction extent that is a multiple of 64");
        // the same idea with a plain row-major dense copy of the weight
        Tensor a = dense_operand(w, rd, false, 1);
        check(nmg_gemm_nt(a.data_ptr(), K, xp, ldx, yp, O, bp, O, K, T, dt, stream));
        return y;
    }
    if (x.scalar_type() == at::kFloat && T >= min_t && automatic && opt.expand && T <= kF32GemmMaxTokens) {
        // single precision: "expand, then multiply" as well -- a dense copy of the weight (kept per
        // weight version) and the pipelined fp32 matrix-core kernel; the kernel below, which expands
        // inside its reduction loop, runs at a tenth of that rate
        // One dense copy [R, C] serves both directions: row-major operand of the product that
        // reduces along dim 1, reduction-major operand of the one that reduces along dim 0.
        Tensor a = dense_operand(w, 1, opt.cache_dense, 1);
        product_f32(rd == 1 ? 0 : 1, a, a.stride(0), x, ldx, y, bp, O, K, T);
        return y;
    }
    const int64_t Kp = round_up(K, 64);
    if (half && T >= (reduce_sparse ? 4 : 1) && automatic && opt.expand && O * Kp * 2 < k2G && T * Kp * 2 < k2G) {
        // 16-bit shapes that none of the matrix-core routes above takes (an m such as 5 or 7):
        // a dense copy of the weight with zero-padded rows (kept per weight version) and, where
        // needed, a zero-padded copy of the activations, through the dense 16-bit GEMM -- the
        // kernel below runs at a hundredth of its rate (from 4 tokens on where the reduction runs
        // along the sparse dim: this GEMM does not cut its reduction, and at 1 token the streaming kernel
        // below is ahead, 81 us against 132; along the group dim that kernel takes 470 us at 4096^2)
        Tensor a = dense_operand(w, rd, opt.cache_dense, 64);
        const Tensor xq = plain64 && flat ? x : padded(x.contiguous(), T, Kp);
        check(nmg_gemm_nt(a.data_ptr(), Kp, xq.data_ptr(), pitch_of(xq), yp, O, bp, O, Kp, T, dt, stream));
        return y;
    }
    pack(w);
    check(nmg_spmm(w.ops.pk_val.data_ptr(), w.ops.pk_pat.data_ptr(), q.G, q.S, xp, ldx, yp, O, bp, T, reduce_sparse ? 1 : 0, q.n, q.m,
                   dt, code, stream));
    return y;
}

// op(W) @ B in single precision with B and the result as they lie in memory: the dense copy of the
// weight (kept per weight version; the same one for both directions) as the row operand of the fp32
// matrix-core GEMM, B as its reduction-major operand.  Undefined when the route does not apply.
Tensor mm_f32(State &w, Tensor b, int rd, const Options &opt)
{
    if (b.scalar_type() != at::kFloat || b.size(1) <= 16 || opt.kernel != "auto" || !opt.expand || b.size(1) > kF32GemmMaxTokens)
        return Tensor();
    const Geometry &q = w.geo;
    const int64_t K = q.dims[rd], O = q.dims[1 - rd];
    if (b.stride(1) != 1) b = b.contiguous();
    const int64_t N = b.size(1);
    // the one dense copy [R, C]: row-major row operand of W @ B, reduction-major row operand of W^T @ B
    Tensor wd = dense_operand(w, 1, opt.cache_dense, 1);
    Tensor c = new_empty({O, N}, b);
    product_f32(rd == 1 ? 1 : 2, b, K > 1 ? b.stride(0) : N, wd, wd.stride(0), c, nullptr, N, K, O);
    return c;
}

void check_mm(const State &w, const Tensor &b, int64_t K)
{
    require_gpu(b);
    require_gpu(w.val);
    if (b.dim() != 2 || b.size(0) != K) fail("B must be [", K, ", N], got ", shape_text(b));
    if (b.scalar_type() != w.val.scalar_type()) fail("dtype mismatch: B ", dtype_name(b), ", weight ", dtype_name(w.val));
}

Tensor spmm_tt_dense(State &w, Tensor b, int rd);

// C = op(W) B from a transposed copy of B rather than from B as it lies.  The copy takes about 3.5 + K N / 0.8 * 10^6 us; without it
// the fragments of B are transposing LDS reads, at half the rate of plain ones, which costs nothing on tiles of 256 outputs and 0.1 us a
// step of 64 on tiles of 128 x 128.  us, copy and kernel -> as it lies, sparse / dense cores: 4096 x 4096 x 2048 columns 55 -> 44 /
// 70 -> 62; 1024^3 13 -> 10 / 15 -> 11; 512 x 4096 x 4096 39 -> 33 / 47 -> 39; 512 x 512 x 64 10 -> 6.7 / 10 -> 7.1; 768 x 768 x 512
// 11.6 -> 8.4 / 12.4 -> 9.1; but 744 x 11520 x 272 60, 62 / 65, 72 and 3032 x 13888 x 400 74, 88 / 92, 101.  (57 random
// products of up to 2^36 multiplications: 0.86 / 0.87 of the time.)  Operands that need a padded copy anyway take the transposed one.
bool transposed_pays(int64_t O, int64_t K, int64_t N, bool as_it_lies)
{
    if (N * round_up(K, 64) * 2 >= k2G) return false;
    const bool narrow = up(O, 128) * up(N, 128) <= 256;
    return !as_it_lies || (narrow && (double)up(K, 64) * 0.1 > 3.5 + (double)K * (double)N / 0.8e6);
}

// Whether op(W) B with few columns is better cut along the reduction (as spmm does it, its result transposed
// back) than run whole on the CUs that its tiles occupy.  A reduction step of 64 takes about 0.45 us on the sparse and
// 0.6 us on the dense cores, 0.4 on tiles of 128 x 128; the cut saves the steps of all slices but one and costs about 11 us of launches beside
// the partial sums, written and read once.  us, whole -> cut: sparse cores 4096 x 11008 x 32 columns 81 -> 27, x 512
// 102 -> 58, 4096 x 4096 x 128 31 -> 25 (8 slices), x 512 32 -> 41 (4 slices); dense cores 1024 x 16384 x 128 141 -> 31,
// 4096 x 4096 x 512 46 -> 41, x 1024 50 -> 57.  The kernel for few tokens walks no steps one after the other and has no partial sums: 32
// columns 2048 x 2048 18.8 -> 12.4, 1024 x 4096 28.0 -> 14.4, 4096 x 4096 33.7 -> 20.4, 8192 x 2048 23.1 -> 18.6; 64 columns 1000 x 3000
// 23.2 -> 15.5, 512 x 4096 28.0 -> 15.2.
bool tt_split_pays(const Options &opt, int64_t O, int64_t K, int64_t N, bool sparse)
{
    if (opt.kernel != "auto" || opt.variant != -1 || opt.dense_variant != -1 || opt.slices >= 0 || !opt.expand || N * round_up(K, 64) * 2 >= k2G)
        return false;
    int slices = 1;
    int64_t bytes = 0;
    check(sparse ? nmg_smfmac_plan(O, K, N, &slices, &bytes) : nmg_densefrag_plan(O, round_up(K, 64), N, &slices, &bytes));
    const bool narrow = up(O, 128) * up(N, 128) <= 256;      // (tiles of 128 x 128)
    const double walk = (double)up(K, 64) * (narrow ? 0.4 : sparse ? 0.45 : 0.6);
    if (!sparse && slices == 1 && nmg_densefrag_few(O, round_up(K, 64), N)) return walk > 11.0;
    return slices > 1 && walk * (1.0 - 1.0 / slices) > 11.0 + (double)slices * (double)(N * O) * 8 / 4e6;
}

Tensor tt_split(State &w, const Tensor &b, int rd)
{
    const int64_t K = b.size(0), N = b.size(1);
    const Tensor y = spmm(w, transposed(b, round_up(K, 64)).narrow(1, 0, K), Tensor(), rd, nullptr);
    return N % 8 == 0 ? transposed(y, N) : y.t().contiguous();
}

// The kernels read whole pieces of 8 columns, also in the last row: those of a view whose storage ends before must not be read as they lie.
bool tt_as_it_lies(const Tensor &b)
{
    const int64_t end = b.storage_offset() + (b.size(0) - 1) * b.stride(0) + round_up(b.size(1), 8);
    if (b.size(1) % 8 != 0 && end * b.element_size() > (int64_t)b.storage().nbytes()) return false;
    return b.stride(1) == 1 && b.stride(0) % 8 == 0 && b.stride(0) >= b.size(1) && aligned16(b) && b.stride(0) < (int64_t(1) << 24);
}

// The dense matrix cores take B as it lies, or a copy of it.
bool tt_dense_ok(const State &w, const Tensor &b, const Options &opt)
{
    return is16(b) && b.size(0) > 0 && b.size(1) > 16 && nmg_densefrag_supported(w.geo.n, w.geo.m) && (opt.kernel == "auto" || opt.kernel == "densefrag")
           && opt.expand && round_up(b.size(1), 8) < (int64_t(1) << 24);
}

// C = W @ B (torch.mm): the sparse matrix cores where they can take it, else the dense ones, else the transposed
// operands through spmm.
Tensor spmm_tt(State &w, Tensor b)
{
    const Geometry &q = w.geo;
    const int64_t R = q.dims[0], C = q.dims[1];
    check_mm(w, b, C);
    c10::DeviceGuard device(b.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    const int64_t N = b.size(1);
    const Options opt = options_of(w);
    bool direct = q.sdim == 1 && is16(b) && N > 16 && C > 0 && round_up(N, 8) < (int64_t(1) << 24) && (opt.kernel == "auto" || opt.kernel == "smfmac");
    if (direct && nmg_fragpack_supported(q.n, q.m)) {
        pack(w);
        direct = w.ops.fp_val.defined();
    } else {
        direct = false;
    }
    if (!direct) {
        Tensor c = mm_f32(w, b, 1, opt);
        if (c.defined()) return c;
        if (opt.kernel == "auto" && tt_dense_ok(w, b, opt))
            return spmm_tt_dense(w, b, 1);
        return spmm(w, b.t().contiguous(), Tensor(), 1, nullptr).t();
    }
    // (whole K steps and pieces of 8 columns: see `padded`)
    if (tt_split_pays(opt, R, C, N, true)) return tt_split(w, b, 1);
    const int64_t Cp = round_up(C, 64);
    const bool as_it_lies = tt_as_it_lies(b) && C == Cp;
    Tensor c = new_empty({R, N}, b);
    if (transposed_pays(R, C, N, as_it_lies)) {
        const Tensor bt = transposed(b, Cp);
        check(nmg_spmm_smfmac_ct(w.ops.fp_val.data_ptr(), w.ops.fp_idx.data_ptr(), R, Cp, bt.data_ptr(), pitch_of(bt), c.data_ptr(), N,
                                 nullptr, N, dtype_code(b.scalar_type()), stream_of(b)));
        return c;
    }
    const Tensor bq = as_it_lies ? b : padded(b, Cp, round_up(N, 8));
    check(nmg_spmm_smfmac_tt(w.ops.fp_val.data_ptr(), w.ops.fp_idx.data_ptr(), R, Cp, bq.data_ptr(), bq.stride(0), c.data_ptr(), N, nullptr,
                             N, dtype_code(b.scalar_type()), stream_of(b)));
    return c;
}

// op(W) @ B on the dense matrix cores.
Tensor spmm_tt_dense(State &w, Tensor b, int rd)
{
    const Geometry &q = w.geo;
    const int64_t K = q.dims[rd], O = q.dims[1 - rd];
    check_mm(w, b, K);
    c10::DeviceGuard device(b.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    const int64_t N = b.size(1);
    const Options opt = options_of(w);
    if (!tt_dense_ok(w, b, opt)) {
        Tensor c = mm_f32(w, b, rd, opt);
        if (c.defined()) return c;
        return spmm(w, b.t().contiguous(), Tensor(), rd, nullptr).t();
    }
    if (tt_split_pays(opt, O, K, N, false)) return tt_split(w, b, rd);
    Tensor df = densefrag(w, rd, opt.cache_dense);
    const int64_t Kp = round_up(K, 64);
    const bool as_it_lies = tt_as_it_lies(b) && K == Kp;
    Tensor c = new_empty({O, N}, b);
    if (transposed_pays(O, K, N, as_it_lies)) {
        const Tensor bt = transposed(b, Kp);
        check(nmg_spmm_densefrag_ct(df.data_ptr(), O, Kp, bt.data_ptr(), pitch_of(bt), c.data_ptr(), N, nullptr, N, dtype_code(b.scalar_type()),
                                    stream_of(b)));
        return c;
    }
    const Tensor bq = as_it_lies ? b : padded(b, Kp, round_up(N, 8));
    check(nmg_spmm_densefrag_tt(df.data_ptr(), O, Kp, bq.data_ptr(), bq.stride(0), c.data_ptr(), N, nullptr, N, dtype_code(b.scalar_type()),
                                stream_of(b)));
    return c;
}

// Sum over the rows.  From 4097 rows on the library's sum, which also cuts the rows over workgroups.
Tensor column_sum(const Tensor &g)
{
    const at::ScalarType dt = g.scalar_type();
    if (!g.is_cuda() || !(dt == at::kFloat || is16(g)) || g.size(0) == 0 || g.size(0) > 4096 || g.size(1) == 0) return g.sum(0);
    c10::DeviceGuard device(g.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    const Tensor s = rows_of(g);
    Tensor y = new_empty({g.size(1)}, g);
    check(nmg_colsum(s.data_ptr(), s.size(0), s.size(1), pitch_of(s), y.data_ptr(), dtype_code(dt), stream_of(g)));
    return y;
}

bool masked_product_supported(const State &w, const Tensor &rows, const Tensor &cols, bool last)
{
    const Geometry &q = w.geo;
    if (q.nd != 2 || !is16(w.val) || rows.scalar_type() != w.val.scalar_type() || cols.scalar_type() != w.val.scalar_type()) return false;
    // the pitches that the kernel's 32-bit offsets reach
    return std::max(pitch_of_whole_pieces(rows), pitch_of_whole_pieces(cols)) < (int64_t(1) << (last ? 22 : 25));
}

// val of the kept positions of rows^T @ cols (rows [T, R], cols [T, C]; with `last` rows [R, T], cols [C, T]).
Tensor masked_product(State &w, Tensor rows, Tensor cols, bool last)
{
    const Geometry &q = w.geo;
    if (q.nd != 2) fail("the masked product needs a 2-D grouped n:m tensor");
    const int64_t R = q.dims[0], C = q.dims[1];
    require_gpu(rows);
    require_gpu(cols);
    require_gpu(w.val);
    const int td = last ? 1 : 0, fd = 1 - td;      // token dim / feature dim of the operands
    if (rows.dim() != 2 || cols.dim() != 2 || rows.size(td) != cols.size(td) || rows.size(fd) != R || cols.size(fd) != C) {
        if (last) fail("operands must be [", R, ", T] and [", C, ", T], got ", shape_text(rows), " and ", shape_text(cols));
        fail("operands must be [T, ", R, "] and [T, ", C, "], got ", shape_text(rows), " and ", shape_text(cols));
    }
    if (rows.scalar_type() != w.val.scalar_type() || cols.scalar_type() != w.val.scalar_type())
        fail("dtype mismatch: operands ", dtype_name(rows), " / ", dtype_name(cols), ", weight ", dtype_name(w.val));
    c10::DeviceGuard device(w.val.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    rows = padded(rows, rows.size(0), round_up(rows.size(1), 8));
    cols = padded(cols, cols.size(0), round_up(cols.size(1), 8));
    const Tensor &lines = q.gdim == 0 ? rows : cols, &pos = q.gdim == 0 ? cols : rows;
    const int64_t T = rows.size(td);      // (padded with zeros where the tokens are the fast dim)
    if (T == 0) return at::zeros_like(w.val);
    Tensor slot = slotmap(w);
    Tensor val = at::empty_like(w.val);
    auto entry = last ? nmg_sddmm_nt : nmg_sddmm_padded;
    check(entry(lines.data_ptr(), pitch_of(lines), pos.data_ptr(), pitch_of(pos), T, (const int16_t *)slot.data_ptr(), q.G, q.S,
                val.data_ptr(), q.n, q.m, q.g, dtype_code(val.scalar_type()), stream_of(val)));
    return val;
}

// Dense product on this library's matrix-core kernels, operands as they lie in memory: tn: x [K, T],
// a [K, O] -> x^T @ a;  nt: x [T, K], a [O, K] -> x @ a^T.  fp32 always; 16-bit types where the kernels take
// the shape (extents and pitches that are multiples of 8, 16-byte aligned bases; nt: K a multiple of 64),
// else padded copies of the operands and, tn, a padded result; what lies beyond the 16-bit kernels' 32-bit offsets
// (operands of 2 GiB, rows of 2^24) is widened for the fp32 kernel, the result rounded once.  Undefined where none
// applies (double, more than 2 097 120 rows of the result in fp32).
Tensor dense_product(bool tn, Tensor x, Tensor a)
{
    const at::ScalarType dt = x.scalar_type();
    const int64_t T = x.size(tn ? 1 : 0), K = x.size(tn ? 0 : 1), O = a.size(tn ? 1 : 0);
    const bool f32 = dt == at::kFloat, half = is16(x);
    const bool sound = x.is_cuda() && a.scalar_type() == dt && (f32 || half) && T > 0 && O > 0 && K > 0;
    if (!sound) return Tensor();
    c10::DeviceGuard device(x.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    if (x.stride(1) != 1) x = x.contiguous();
    if (a.stride(1) != 1) a = a.contiguous();
    void *const stream = stream_of(x);
    const int64_t T8 = round_up(T, 8), O8 = round_up(O, 8), K64 = round_up(K, 64);
    const bool reached = tn ? std::max({T8, O8, x.stride(0), a.stride(0)}) < (int64_t(1) << 24)
                            : std::max(O * std::max(K64, a.stride(0)), T * std::max(K64, x.stride(0))) * 2 < k2G;
    if (!half || !reached) {
        if (up(T, 32) > 65535) return Tensor();
        if (half) {
            x = x.to(at::kFloat).contiguous();
            a = a.to(at::kFloat).contiguous();
        }
        Tensor y = new_empty({T, O}, x);
        product_f32(tn ? 2 : 0, a, a.stride(0), x, x.stride(0), y, nullptr, O, K, T);
        return half ? y.to(dt) : y;
    }
    if (tn) {
        x = padded(x, K, T8);
        a = padded(a, K, O8);
        Tensor y = new_empty({T8, O8}, x);
        check(nmg_gemm_tn(a.data_ptr(), pitch_of(a), x.data_ptr(), pitch_of(x), y.data_ptr(), O8, nullptr, O8, K, T8, dtype_code(dt), stream));
        if (O8 == O) return T8 == T ? y : y.narrow(0, 0, T);
        Tensor out = new_empty({T, O}, x);
        check(nmg_copy_rows16(y.data_ptr(), T, O, O8, out.data_ptr(), T, O, O, stream));
        return out;
    }
    x = padded(x, T, K64);
    a = padded(a, O, K64);
    Tensor y = new_empty({T, O}, x);
    check(nmg_gemm_nt(a.data_ptr(), pitch_of(a), x.data_ptr(), pitch_of(x), y.data_ptr(), O, nullptr, O, K64, T, dtype_code(dt), stream));
    return y;
}

// x [T, K] @ dequantised(B, meta, s)^T for at most 16 token rows.
Tensor w4_linear(const Tensor &B, const Tensor &meta, const Tensor &s, int64_t M, int64_t K, Tensor x, Tensor bias)
{
    c10::DeviceGuard device(x.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    const int64_t T = x.size(0);
    if (x.stride(1) != 1 || x.stride(0) % 8 != 0 || !aligned16(x)) x = x.contiguous();
    if (bias.defined()) bias = bias.to(at::kHalf).contiguous();
    Tensor y = new_empty({T, M}, x);
    check(nmg_w4_linear(B.data_ptr(), meta.data_ptr(), s.data_ptr(), M, K, x.data_ptr(), T > 1 ? x.stride(0) : K, y.data_ptr(), M,
                        bias.defined() ? bias.data_ptr() : nullptr, T, stream_of(x)));
    return y;
}

// ------------------------------------------------------------------------------- Python: the core type

PyObject *wrap(const Tensor &t) { return THPVariable_Wrap(t); }

Tensor tensor_arg(PyObject *o, const char *what)
{
    if (!THPVariable_Check(o)) fail(what, " must be a tensor, got ", Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}

Tensor optional_arg(PyObject *o, const char *what) { return o == nullptr || o == Py_None ? Tensor() : tensor_arg(o, what); }

int dim_arg(PyObject *o)
{
    const long d = PyLong_AsLong(o);
    if (d == -1 && PyErr_Occurred()) throw python_error();
    if (d != 0 && d != 1) fail("reduce_dim must be 0 or 1, got ", d);
    return (int)d;
}

PyObject *core_new(PyTypeObject *type, PyObject *, PyObject *)
{
    PyObject *o = type->tp_alloc(type, 0);
    if (o == nullptr) return nullptr;
    State *st = new State();
    st->layout = Py_None;
    Py_INCREF(Py_None);
    st->opt = PyDict_New();
    reinterpret_cast<Core *>(o)->st = st;
    return o;
}

void core_dealloc(PyObject *o)
{
    State *st = reinterpret_cast<Core *>(o)->st;
    if (st != nullptr) {
        Py_XDECREF(st->layout);
        Py_XDECREF(st->opt);
        delete st;
    }
    Py_TYPE(o)->tp_free(o);
}

int64_t int_attr(PyObject *o, const char *name)
{
    PyObject *v = PyObject_GetAttrString(o, name);
    if (v == nullptr) throw python_error();
    const long long r = PyLong_AsLongLong(v);
    Py_DECREF(v);
    if (r == -1 && PyErr_Occurred()) throw python_error();
    return r;
}

void set_layout(State &w, PyObject *layout)
{
    Geometry q;
    PyObject *shape = PyObject_GetAttr(layout, S_.dense_shape);
    if (shape == nullptr) throw python_error();
    PyObject *seq = PySequence_Fast(shape, "dense_shape must be a sequence");
    Py_DECREF(shape);
    if (seq == nullptr) throw python_error();
    q.nd = (int)PySequence_Fast_GET_SIZE(seq);
    for (int d = 0; d < q.nd; d++) q.dims.push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, d)));
    Py_DECREF(seq);
    if (PyErr_Occurred()) throw python_error();
    q.n = (int)int_attr(layout, "n");
    q.m = (int)int_attr(layout, "m");
    q.g = (int)int_attr(layout, "group_size");
    q.sdim = (int)int_attr(layout, "sparse_dim");
    q.gdim = (int)int_attr(layout, "group_dim");
    q.G = q.dims.at(q.gdim);
    q.S = q.dims.at(q.sdim);
    q.nb = up(q.S, q.m);
    q.cols = nmg_chunk(q.n, q.m) * q.g;
    q.chunks = up(q.G, q.cols);
    w.geo = std::move(q);
    Py_INCREF(layout);
    Py_XDECREF(w.layout);
    w.layout = layout;
}

int set_tensor(PyObject *self, PyObject *v, void *slot)
{
    HOST_TRY
    State &w = state_of(self);
    if (v == nullptr) fail("the tensor cannot be deleted");
    (w.*(slot == nullptr ? &State::val : &State::idx)) = tensor_arg(v, slot == nullptr ? "val" : "idx");
    w.ops = Operands();
    if (slot != nullptr) {
        w.slot = Tensor();
        w.slot_valid = false;
    }
    return 0;
    HOST_CATCH(-1)
}

PyObject *get_tensor(PyObject *self, void *slot)
{
    HOST_TRY
    State &w = state_of(self);
    return wrap(slot == nullptr ? w.val : w.idx);
    HOST_CATCH(nullptr)
}

PyObject *get_layout(PyObject *self, void *)
{
    PyObject *l = reinterpret_cast<Core *>(self)->st->layout;
    Py_INCREF(l);
    return l;
}

int put_layout(PyObject *self, PyObject *v, void *)
{
    HOST_TRY
    State &w = state_of(self);
    if (v == nullptr) fail("the layout cannot be deleted");
    set_layout(w, v);
    w.ops = Operands();
    w.slot_valid = false;
    return 0;
    HOST_CATCH(-1)
}

PyObject *get_opt(PyObject *self, void *)
{
    PyObject *d = reinterpret_cast<Core *>(self)->st->opt;
    Py_INCREF(d);
    return d;
}

int put_opt(PyObject *self, PyObject *v, void *)
{
    if (v == nullptr || !PyDict_Check(v)) {
        PyErr_SetString(PyExc_TypeError, "spmm_opt must be a dict");
        return -1;
    }
    State &w = *reinterpret_cast<Core *>(self)->st;
    Py_INCREF(v);
    Py_XDECREF(w.opt);
    w.opt = v;
    return 0;
}

// {reduction direction: operand} of the operands kept for the present val and idx
PyObject *get_frag_cache(PyObject *self, void *)
{
    HOST_TRY
    Operands &o = operands(state_of(self));
    PyObject *d = PyDict_New();
    for (long rd = 0; rd < 2; rd++)
        if (o.frag[rd].defined()) {
            PyObject *k = PyLong_FromLong(rd), *t = wrap(o.frag[rd]);
            PyDict_SetItem(d, k, t);
            Py_DECREF(k);
            Py_DECREF(t);
        }
    return d;
    HOST_CATCH(nullptr)
}

// {reduction direction, or (direction, extent) where the reduction is padded: dense copy, as rows or in fragment order}
PyObject *get_dense_cache(PyObject *self, void *)
{
    HOST_TRY
    State &w = state_of(self);
    Operands &o = operands(w);
    PyObject *d = PyDict_New();
    for (int rd = 0; rd < 2; rd++)
        for (auto &e : o.dense[rd]) {
            PyObject *k = e.first == w.geo.dims[rd] ? PyLong_FromLong(rd) : Py_BuildValue("(iL)", rd, (long long)e.first);
            PyObject *t = wrap(e.second);
            PyDict_SetItem(d, k, t);
            Py_DECREF(k);
            Py_DECREF(t);
        }
    for (int rd = 0; rd < 2; rd++)
        if (o.frag[rd].defined() && w.geo.dims[rd] % 64 != 0) {
            PyObject *k = Py_BuildValue("(iL)", rd, (long long)round_up(w.geo.dims[rd], 64)), *t = wrap(o.frag[rd]);
            PyDict_SetItem(d, k, t);
            Py_DECREF(k);
            Py_DECREF(t);
        }
    return d;
    HOST_CATCH(nullptr)
}

PyObject *pair_or_none(const Tensor &a, const Tensor &b)
{
    if (!a.defined()) Py_RETURN_NONE;
    return Py_BuildValue("(NN)", wrap(a), wrap(b));
}

// a C++ scope for the operand methods: device of the weight, no autograd, a 2-D weight
struct OperandScope {
    State &w;
    c10::DeviceGuard device;
    at::AutoDispatchBelowADInplaceOrView raw;
    explicit OperandScope(PyObject *self) : w(matmul_state(self)), device((require_gpu(w.val), w.val.device())) {}
};

PyObject *py_rowpack(PyObject *self, PyObject *)
{
    HOST_TRY
    OperandScope s(self);
    pack(s.w);
    return pair_or_none(s.w.ops.pk_val, s.w.ops.pk_pat);
    HOST_CATCH(nullptr)
}

PyObject *py_fragpack(PyObject *self, PyObject *)
{
    HOST_TRY
    OperandScope s(self);
    pack(s.w);
    return pair_or_none(s.w.ops.fp_val, s.w.ops.fp_idx);
    HOST_CATCH(nullptr)
}

PyObject *py_densefrag(PyObject *self, PyObject *arg)
{
    HOST_TRY
    OperandScope s(self);
    return wrap(densefrag(s.w, dim_arg(arg), options_of(s.w).cache_dense));
    HOST_CATCH(nullptr)
}

PyObject *py_dense_operand(PyObject *self, PyObject *args, PyObject *kwargs)
{
    HOST_TRY
    static const char *names[] = {"reduce_dim", "cached", "pad_k", nullptr};
    PyObject *rd = nullptr;
    int cached = 0;
    long long pad_k = 1;
    if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O|pL", const_cast<char **>(names), &rd, &cached, &pad_k)) return nullptr;
    OperandScope s(self);
    return wrap(dense_operand(s.w, dim_arg(rd), cached && options_of(s.w).cache_dense, pad_k));
    HOST_CATCH(nullptr)
}

PyObject *py_lanepack8(PyObject *self, PyObject *)
{
    HOST_TRY
    OperandScope s(self);
    lanepack8(s.w);
    return pair_or_none(s.w.ops.lp_val, s.w.ops.lp_pat);
    HOST_CATCH(nullptr)
}

PyObject *py_gpack(PyObject *self, PyObject *)
{
    HOST_TRY
    OperandScope s(self);
    gpack(s.w);
    return wrap(s.w.ops.gp);
    HOST_CATCH(nullptr)
}

PyObject *py_opack(PyObject *self, PyObject *)
{
    HOST_TRY
    OperandScope s(self);
    opack(s.w);
    return wrap(s.w.ops.op);
    HOST_CATCH(nullptr)
}

PyObject *py_slotmap(PyObject *self, PyObject *)
{
    HOST_TRY
    State &w = state_of(self);
    c10::DeviceGuard device(w.idx.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    return wrap(slotmap(w));
    HOST_CATCH(nullptr)
}

PyObject *py_drop(PyObject *self, PyObject *)
{
    reinterpret_cast<Core *>(self)->st->ops = Operands();
    Py_RETURN_NONE;
}

// A tensor of the same class, pattern and options with other values.
PyObject *with_val(PyObject *self, const Tensor &val)
{
    State &w = state_of(self);
    PyObject *o = core_new(Py_TYPE(self), nullptr, nullptr);
    if (o == nullptr) throw python_error();
    State &n = *reinterpret_cast<Core *>(o)->st;
    n.val = val;
    n.idx = w.idx;
    n.geo = w.geo;
    Py_INCREF(w.layout);
    Py_DECREF(n.layout);
    n.layout = w.layout;
    Py_DECREF(n.opt);
    n.opt = PyDict_Copy(w.opt);
    return o;
}

PyObject *py_gather(PyObject *self, PyObject *arg)
{
    HOST_TRY
    State &w = state_of(self);
    Tensor t = tensor_arg(arg, "the dense tensor");
    require_gpu(t);
    c10::DeviceGuard device(t.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    return with_val(self, gather(w, t));
    HOST_CATCH(nullptr)
}

PyObject *py_to_dense(PyObject *self, PyObject *)
{
    HOST_TRY
    State &w = state_of(self);
    const Geometry &q = w.geo;
    require_gpu(w.val);
    c10::DeviceGuard device(w.val.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    Tensor out = new_empty(q.dims, w.val), t = out;
    nmg_view v = view_of(t, q);
    check(nmg_to_dense(w.val.data_ptr(), (const int16_t *)w.idx.data_ptr(), t.data_ptr(), &v, q.n, q.m, q.g,
                       dtype_code(w.val.scalar_type()), stream_of(w.val)));
    if (t.storage().data_ptr().get() != out.storage().data_ptr().get()) {
        std::vector<int64_t> perm, sizes;
        for (int d = 0; d < q.nd; d++)
            if (d != q.sdim && d != q.gdim) perm.push_back(d);
        perm.push_back(q.gdim);
        perm.push_back(q.sdim);
        for (int64_t d : perm) sizes.push_back(q.dims[d]);
        std::vector<int64_t> inv(q.nd);
        for (int i = 0; i < q.nd; i++) inv[perm[i]] = i;
        out = t.view(sizes).permute(inv).contiguous();
    }
    return wrap(out);
    HOST_CATCH(nullptr)
}

PyObject *py_masked_product(PyObject *self, PyObject *args)
{
    HOST_TRY
    PyObject *r, *c;
    int last = 0;
    if (!PyArg_ParseTuple(args, "OOp", &r, &c, &last)) return nullptr;
    State &w = state_of(self);
    const Tensor rows = tensor_arg(r, "rows_op"), cols = tensor_arg(c, "cols_op");
    if (last && rows.dim() == 2 && rows.size(1) % 8 != 0)      // (the backward of torch.mm pads its operands)
        fail("reduction-contiguous operands need a token count that is a multiple of 8, got ", rows.size(1));
    return with_val(self, masked_product(w, rows, cols, last != 0));
    HOST_CATCH(nullptr)
}

PyObject *py_masked_product_supported(PyObject *self, PyObject *args)
{
    HOST_TRY
    PyObject *r, *c;
    int last = 0;
    if (!PyArg_ParseTuple(args, "OOp", &r, &c, &last)) return nullptr;
    const Tensor rows = tensor_arg(r, "rows_op"), cols = tensor_arg(c, "cols_op");
    return PyBool_FromLong(masked_product_supported(state_of(self), rows, cols, last != 0) && !(last && rows.size(1) % 8 != 0));
    HOST_CATCH(nullptr)
}

PyGetSetDef core_getset[] = {
    {"val", get_tensor, set_tensor, "kept values [outer, c, g, n]", nullptr},
    {"idx", get_tensor, set_tensor, "int16 column positions [outer, c, g, 1]", (void *)1},
    {"layout", get_layout, put_layout, "NMGLayout", nullptr},
    {"spmm_opt", get_opt, put_opt, "options of the products", nullptr},
    {"_densefrag", get_frag_cache, nullptr, "dense-core operands kept for the present values", nullptr},
    {"_dense_operand", get_dense_cache, nullptr, "dense copies kept for the present values", nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyMethodDef core_methods[] = {
    {"rowpack", py_rowpack, METH_NOARGS,
     "(pk_val [G, nb, n], pk_pat [G, nb]) -- per line of the group dim and block of the sparse dim, the kept\n"
     "values and the pattern number; cached until ``val`` changes."},
    {"fragpack", py_fragpack, METH_NOARGS,
     "Operand of the sparse-matrix-core kernel (values + 2-bit positions in instruction register order);\n"
     "``None`` when the n:m pattern does not fit 2-of-4 groups or the dtype is not 16-bit.  Cached until ``val`` changes."},
    {"densefrag", py_densefrag, METH_O,
     "densefrag(reduce_dim): the weight as the A operand of the dense matrix cores, [outputs, reduction] in\n"
     "fragment order, expanded from the rowpack operand.  It is as large as the dense weight.  It is kept until\n"
     "``val`` changes (one copy per reduction direction), so a frozen weight, or the forward and backward of one\n"
     "training step, pay the expansion once; ``spmm_opt[\"cache_dense\"] = False`` rebuilds it per call instead and\n"
     "keeps the memory of the compressed format."},
    {"dense_operand", (PyCFunction)(void (*)(void))py_dense_operand, METH_VARARGS | METH_KEYWORDS,
     "dense_operand(reduce_dim, cached=False, pad_k=1): dense copy [outputs, reduction] of the weight (transposed\n"
     "when the reduction runs along dim 0), expanded from the rowpack operand into fresh scratch.  ``cached``: kept\n"
     "until ``val`` changes, like the densefrag operand (``spmm_opt[\"cache_dense\"] = False`` turns that off).\n"
     "``pad_k``: the rows are padded with zeros to a multiple of it."},
    {"lanepack8", py_lanepack8, METH_NOARGS,
     "Operand of the streaming product on blocks of 8 along the reduction (1:8, 2:8, 4:8 with at most 16 tokens):\n"
     "the rowpack values and pattern bytes in the order in which the lanes of ``nmg_spmm_sstream`` take them; as\n"
     "large as the rowpack operand (0.625 bytes per dense weight at 2:8), kept until ``val`` changes."},
    {"gpack", py_gpack, METH_NOARGS,
     "Operand of the streaming product along the group dim (at most 16 tokens, m = 4 or 8 with n = 1 or 2): the\n"
     "rowpack operand in tiles of 32 lines x 256 outputs, each one contiguous run in the order in which the lanes\n"
     "of ``nmg_spmm_gstream`` take it, pattern numbers in 4 bits where there are at most 16; kept until ``val`` changes."},
    {"opack", py_opack, METH_NOARGS,
     "Operand of ``nmg_spmm_ostream`` (a handful of tokens, 2:4, reduction along the group dim): the rowpack operand\n"
     "per span of 16 outputs and set of 256 lines in the order in which the lanes fetch it, pattern numbers in 4\n"
     "bits; kept until ``val`` changes."},
    {"slotmap", py_slotmap, METH_NOARGS,
     "int16 [num_blocks, Gpad]: for every line of the (padded) group dim and block of the sparse dim, the slot that\n"
     "holds it -- the inverse of ``idx``.  Operand of the masked weight-gradient kernel; depends on the pattern\n"
     "only, cached until ``idx`` changes."},
    {"to_dense", py_to_dense, METH_NOARGS, "The dense tensor, zeros at the positions that are not kept."},
    {"_gather", py_gather, METH_O, nullptr},
    {"_masked_product", py_masked_product, METH_VARARGS, nullptr},
    {"_masked_product_supported", py_masked_product_supported, METH_VARARGS, nullptr},
    {"_drop_operands", py_drop, METH_NOARGS, "Forget every operand derived from ``val`` (in-place updates call this)."},
    {nullptr, nullptr, 0, nullptr}};

// ---------------------------------------------------------------------------------- Python: functions

PyObject *py_sparsify(PyObject *, PyObject *args)
{
    HOST_TRY
    PyObject *self, *dense;
    if (!PyArg_ParseTuple(args, "OO", &self, &dense)) return nullptr;
    State &w = state_of(self);      // layout set, val and idx not yet
    const Geometry &q = w.geo;
    Tensor t = tensor_arg(dense, "the dense tensor");
    require_gpu(t);
    c10::DeviceGuard device(t.device());
    at::AutoDispatchBelowADInplaceOrView raw;
    nmg_view v = view_of(t, q);
    const int64_t outer = v.batch * q.chunks * q.nb, c = nmg_chunk(q.n, q.m);
    Tensor val = new_empty({outer, c, q.g, q.n}, t), idx = new_empty({outer, c, q.g, 1}, t, at::kShort);
    check(nmg_sparsify(t.data_ptr(), &v, val.data_ptr(), (int16_t *)idx.data_ptr(), q.n, q.m, q.g, dtype_code(t.scalar_type()),
                       stream_of(t)));
    w.val = val;
    w.idx = idx;
    Py_RETURN_NONE;
    HOST_CATCH(nullptr)
}

const char *kernel_arg(PyObject *o)
{
    if (o == nullptr || o == Py_None) return nullptr;
    const char *c = PyUnicode_AsUTF8(o);
    if (c == nullptr) throw python_error();
    return *c != 0 ? c : nullptr;
}

PyObject *py_spmm(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HOST_TRY
    if (n != 5) fail("spmm takes 5 arguments");
    return wrap(spmm(matmul_state(a[0]), tensor_arg(a[1], "the activations"), optional_arg(a[2], "the bias"), dim_arg(a[3]), kernel_arg(a[4])));
    HOST_CATCH(nullptr)
}

PyObject *py_column_sum(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HOST_TRY
    if (n != 1) fail("column_sum takes 1 argument");
    const Tensor x = tensor_arg(a[0], "x");
    if (x.dim() != 2) fail("column_sum takes a matrix");
    return wrap(column_sum(x));
    HOST_CATCH(nullptr)
}

PyObject *py_spmm_tt(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HOST_TRY
    if (n != 2) fail("spmm_tt takes 2 arguments");
    return wrap(spmm_tt(matmul_state(a[0]), tensor_arg(a[1], "B")));
    HOST_CATCH(nullptr)
}

PyObject *py_spmm_tt_dense(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HOST_TRY
    if (n != 3) fail("spmm_tt_dense takes 3 arguments");
    return wrap(spmm_tt_dense(matmul_state(a[0]), tensor_arg(a[1], "B"), dim_arg(a[2])));
    HOST_CATCH(nullptr)
}

PyObject *py_dense_product(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HOST_TRY
    if (n != 3) fail("dense_product takes 3 arguments");
    Tensor y = dense_product(PyObject_IsTrue(a[0]) == 1, tensor_arg(a[1], "x"), tensor_arg(a[2], "a"));
    if (!y.defined()) Py_RETURN_NONE;
    return wrap(y);
    HOST_CATCH(nullptr)
}

PyObject *py_w4_linear(PyObject *, PyObject *args)
{
    HOST_TRY
    PyObject *B, *meta, *s, *x, *bias;
    long long M, K;
    if (!PyArg_ParseTuple(args, "OOOLLOO", &B, &meta, &s, &M, &K, &x, &bias)) return nullptr;
    return wrap(w4_linear(tensor_arg(B, "B"), tensor_arg(meta, "meta"), tensor_arg(s, "s"), M, K, tensor_arg(x, "the activations"),
                          optional_arg(bias, "the bias")));
    HOST_CATCH(nullptr)
}

// --------------------------------------------------------------------- the dispatch of wrapped tensors

// `__torch_function__` of a dispatch module.  The operators that have a native route and the accessors that an
// optimizer or a module touches on every step are served here; everything else, and whatever the native
// route does not know (another format, a registered replacement, sparse outputs, other gradient formats),
// goes to the module's own Python dispatcher.
struct Dispatch {
    PyObject *slow;        // (func, types, args, kwargs)
    PyObject *failed;      // (func, exception): the dispatcher's warning before an exception leaves it
    PyObject *plain;       // set: functions that run on the wrapper's own placeholder
    PyObject *native;      // operator -> {format: [forward, dense gradient, pattern gradient: bit per arity, place of the weight]}
    PyObject *grad_of;     // (wrapped, dtype and device of this tensor) -> wrapper of a weight gradient
    PyObject *add_;        // torch.Tensor.add_
    PyObject *keep_all, *dense_tensor, *tensor;      // the module's KeepAll and DenseTensor, torch.Tensor
};

Dispatch *dispatch_of(PyObject *capsule) { return (Dispatch *)PyCapsule_GetPointer(capsule, nullptr); }

// The list that holds what a wrapper wraps; nullptr where `o` is no wrapper.
PyObject *container_of(PyObject *o)
{
    PyObject **d = _PyObject_GetDictPtr(o);
    if (d == nullptr || *d == nullptr) return nullptr;
    PyObject *c = PyDict_GetItem(*d, S_.container);
    return c != nullptr && PyList_CheckExact(c) && PyList_GET_SIZE(c) == 1 ? c : nullptr;
}

bool plain_tensor(PyObject *o) { return THPVariable_CheckExact(o); }

bool has_bit(PyObject *masks, Py_ssize_t slot, int arity)
{
    const long m = PyLong_AsLong(PyList_GET_ITEM(masks, slot));
    return (m >> arity & 1) != 0;
}

// The format of the weight gradient where the native backward knows it: 1 dense, 2 the weight's pattern, else 0.
int grad_kind(const Dispatch &d, PyObject *weight, PyObject *wrapped)
{
    PyObject **dict = _PyObject_GetDictPtr(weight);
    PyObject *f = dict != nullptr && *dict != nullptr ? PyDict_GetItem(*dict, S_.grad_fmt) : nullptr;
    if (f == nullptr || !PyTuple_Check(f) || PyTuple_GET_SIZE(f) != 4) return 0;
    if ((PyObject *)Py_TYPE(PyTuple_GET_ITEM(f, 0)) != d.keep_all || (PyObject *)Py_TYPE(PyTuple_GET_ITEM(f, 2)) != d.keep_all) return 0;
    PyObject *tmp = PyTuple_GET_ITEM(f, 1), *out = PyTuple_GET_ITEM(f, 3);
    if (tmp == d.tensor && out == d.dense_tensor) return 1;
    if (tmp == (PyObject *)Py_TYPE(wrapped) && out == tmp) return 2;
    return 0;
}

// val-layout gradient: the kept positions of lhs^T @ rhs (lhs [T, rows of W], rhs [T, columns of W]).  16-bit weights
// take the fused kernel, which never stores the dense product; fp32 goes through the dense product and the
// same-pattern gather.
Tensor masked_weight_grad(State &w, const Tensor &lhs, Tensor rhs)
{
    if (rhs.scalar_type() != w.val.scalar_type()) rhs = rhs.to(w.val.scalar_type());
    if (masked_product_supported(w, lhs, rhs, false)) return masked_product(w, lhs, rhs, false);
    Tensor g = dense_product(true, lhs, rhs);
    if (!g.defined()) g = at::mm(lhs.t(), rhs);
    return gather(w, g);
}

// Backward of F.linear(x, W[, b]) (weight at place 1) and of torch.mm(W, B) (weight at place 0).
struct ProductNode : public torch::autograd::Node {
    torch::autograd::SavedVariable dense;      // x or B
    PyObject *container = nullptr, *owner = nullptr;
    int place = 1, kind = 1;
    bool released = false;

    ~ProductNode() override
    {
        if (!Py_IsInitialized()) return;
        pybind11::gil_scoped_acquire gil;
        Py_XDECREF(container);
        Py_XDECREF(owner);
    }
    std::string name() const override { return place == 1 ? "SparseLinearBackward" : "SparseMmBackward"; }
    void release_variables() override
    {
        dense.reset_data();
        released = true;
    }

    Tensor weight_grad(PyObject *wrapped, const Tensor &g)
    {
        PyObject *payload = kind == 2 ? with_val(wrapped, g) : wrap(g);
        PyObject *like = wrap(state_of(wrapped).val);
        PyObject *r = PyObject_CallFunctionObjArgs(dispatch_of(owner)->grad_of, payload, like, kind == 2 ? Py_True : Py_False, nullptr);
        Py_DECREF(payload);
        Py_DECREF(like);
        if (r == nullptr) throw python_error();
        Tensor t = THPVariable_Unpack(r);
        Py_DECREF(r);
        return t;
    }

    void linear(PyObject *wrapped, const Tensor &gy, torch::autograd::variable_list &out)
    {
        State &w = matmul_state(wrapped);
        Tensor x = dense.unpack();
        Tensor g = gy.dim() == 2 ? gy : gy.reshape({-1, gy.size(-1)});
        Tensor x2 = x.dim() == 2 ? x : x.reshape({-1, x.size(-1)});
        if (g.scalar_type() != w.val.scalar_type()) g = g.to(w.val.scalar_type());
        if (task_should_compute_output(0)) {
            Tensor gx = spmm(w, g.contiguous(), Tensor(), 0, nullptr);
            out[0] = x.dim() == 2 ? gx : gx.reshape(x.sizes());
        }
        if (task_should_compute_output(1)) {
            Tensor gw;
            if (kind == 2) {
                gw = masked_weight_grad(w, g, x2);
            } else {
                // the dense weight gradient dY^T X from the operands as they lie (both token-major)
                const Tensor r = x2.scalar_type() == g.scalar_type() ? x2 : x2.to(g.scalar_type());
                gw = dense_product(true, g, r);
                if (!gw.defined()) gw = at::mm(g.t(), r);
            }
            out[1] = weight_grad(wrapped, gw);
        }
        if (out.size() > 2 && task_should_compute_output(2)) out[2] = column_sum(g);
    }

    void mm(PyObject *wrapped, Tensor gc, torch::autograd::variable_list &out)
    {
        State &w = matmul_state(wrapped);
        Tensor b = dense.unpack();
        if (gc.scalar_type() != w.val.scalar_type()) gc = gc.to(w.val.scalar_type());
        if (task_should_compute_output(1)) out[1] = spmm_tt_dense(w, gc, 0);      // W^T @ grad_out
        if (!task_should_compute_output(0)) return;
        Tensor gw;
        const Tensor r = b.scalar_type() == gc.scalar_type() ? b : b.to(gc.scalar_type());
        if (kind == 2 && masked_product_supported(w, gc, b, true)) {
            // grad_out [R, N] and B [C, N] are reduction-contiguous as they lie: no transposing copies
            gw = masked_product(w, gc, b, true);
        } else if (kind == 2 && !(gc.scalar_type() == at::kFloat && b.scalar_type() == at::kFloat)) {
            gw = masked_weight_grad(w, gc.t(), b.t());
        } else {
            gw = dense_product(false, gc, r);      // grad_out @ B^T
            if (!gw.defined()) gw = at::mm(gc, r.t());
            if (kind == 2) gw = gather(w, gw);
        }
        out[0] = weight_grad(wrapped, gw);
    }

    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override
    {
        torch::autograd::variable_list out(next_edges().size());
        TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
        if (!grads[0].defined()) return out;
        c10::AutoGradMode no_grad(false);
        pybind11::gil_scoped_acquire gil;
        try {
            c10::DeviceGuard device(grads[0].device());
            PyObject *wrapped = PyList_GetItem(container, 0);
            if (wrapped == nullptr) throw python_error();
            Py_INCREF(wrapped);
            std::unique_ptr<PyObject, void (*)(PyObject *)> hold(wrapped, [](PyObject *o) { Py_DECREF(o); });
            if (place == 1) linear(wrapped, grads[0], out);
            else mm(wrapped, grads[0], out);
        } catch (const NmgError &e) {
            PyErr_SetString(g_nmg_error, e.what());
            python_error err;
            err.persist();
            throw std::move(err);
        } catch (python_error &e) {
            e.persist();
            throw;
        }
        return out;
    }
};

std::shared_ptr<ProductNode> new_node(PyObject *capsule, PyObject *container, int place, int kind, const Tensor &dense,
                                      torch::autograd::edge_list edges)
{
    std::shared_ptr<ProductNode> node(new ProductNode(), torch::autograd::deleteNode);
    Py_INCREF(container);
    Py_INCREF(capsule);
    node->container = container;
    node->owner = capsule;
    node->place = place;
    node->kind = kind;
    node->dense = torch::autograd::SavedVariable(dense, false);
    node->set_next_edges(std::move(edges));
    return node;
}

// A tensor with a forward-mode tangent or inside a function transform (vmap, grad): what the Python dispatcher's
// autograd.Function refuses must reach it, the kernels see neither.
bool transformed(const Tensor &t)
{
    return t.defined()
           && (t._fw_grad(0).defined()
               || t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                           c10::DispatchKey::Functionalize})));
}

// A new reference to the result, or nullptr without an error where the native route does not apply.
PyObject *native_product(PyObject *capsule, PyObject *formats, PyObject *args)
{
    // torch.jit.trace records the allocation of the result but no launch: the graph would return memory that nothing
    // has written.  The Python dispatcher's autograd.Function is recorded whole.
    if (torch::jit::tracer::isTracing()) return nullptr;
    Dispatch &d = *dispatch_of(capsule);
    const Py_ssize_t n = PyTuple_GET_SIZE(args);
    if (n < 2 || n > 3) return nullptr;
    PyObject *a0 = PyTuple_GET_ITEM(args, 0), *a1 = PyTuple_GET_ITEM(args, 1);
    const int guess = plain_tensor(a0) ? 1 : 0;      // where the weight would be
    PyObject *pw = guess == 1 ? a1 : a0, *px = guess == 1 ? a0 : a1;
    if (plain_tensor(pw) || !plain_tensor(px)) return nullptr;
    PyObject *container = container_of(pw);
    if (container == nullptr) return nullptr;
    PyObject *wrapped = PyList_GET_ITEM(container, 0);
    PyObject *masks = PyDict_GetItem(formats, (PyObject *)Py_TYPE(wrapped));
    if (masks == nullptr || PyLong_AsLong(PyList_GET_ITEM(masks, 3)) != guess) return nullptr;
    PyObject *pb = n == 3 ? PyTuple_GET_ITEM(args, 2) : Py_None;
    if (pb != Py_None && !plain_tensor(pb)) return nullptr;
    const int arity = pb == Py_None ? 2 : 3;
    if (!has_bit(masks, 0, arity) || (guess == 0 && n != 2)) return nullptr;
    const Tensor &x = THPVariable_Unpack(px), &wt = THPVariable_Unpack(pw);
    Tensor bias = pb == Py_None ? Tensor() : THPVariable_Unpack(pb);
    if (transformed(x) || transformed(wt) || transformed(bias)) return nullptr;
    const bool grad = c10::GradMode::is_enabled() && (x.requires_grad() || wt.requires_grad() || (bias.defined() && bias.requires_grad()));
    if (x.dim() < 2 && !(guess == 1 && x.dim() == 1)) return nullptr;
    if (!PyObject_TypeCheck(wrapped, &CoreType)) {      // the int4 format: generation without gradients
        if (grad || guess != 1 || !x.is_cuda() || x.scalar_type() != at::kHalf) return nullptr;
        Tensor t[3];
        PyObject *names[3] = {S_.B, S_.meta, S_.s};
        for (int i = 0; i < 3; i++) {
            PyObject *o = PyObject_GetAttr(wrapped, names[i]);
            if (o == nullptr) throw python_error();
            t[i] = tensor_arg(o, "a part of the int4 weight");
            Py_DECREF(o);
        }
        PyObject *shape = PyObject_GetAttr(wrapped, S_.dense_shape);
        if (shape == nullptr) throw python_error();
        long long M = 0, K = 0;
        const int ok = PyArg_ParseTuple(shape, "LL", &M, &K);
        Py_DECREF(shape);
        if (!ok) throw python_error();
        if (x.size(-1) != K || x.numel() > 16 * K) return nullptr;
        Tensor y = w4_linear(t[0], t[1], t[2], M, K, x.dim() == 2 ? x : x.reshape({-1, K}), bias);
        if (x.dim() != 2) {
            std::vector<int64_t> size(x.sizes().begin(), x.sizes().end());
            size.back() = M;
            y = y.reshape(size);
        }
        return wrap(y);
    }
    int kind = 0;
    if (grad) {
        kind = grad_kind(d, pw, wrapped);
        if (kind == 0 || !has_bit(masks, kind, arity)) return nullptr;
    }
    State &w = matmul_state(wrapped);
    Tensor y;
    if (guess == 1) {
        Tensor x2 = x;
        {
            at::AutoDispatchBelowADInplaceOrView raw;
            if (x.dim() != 2) x2 = x.reshape({-1, x.size(-1)});
            y = spmm(w, x2, bias, 1, nullptr);
            if (x.dim() != 2) {
                std::vector<int64_t> size(x.sizes().begin(), x.sizes().end());
                size.back() = y.size(-1);
                y = y.reshape(size);
            }
        }
    } else {
        y = spmm_tt(w, x);
    }
    if (grad) {
        torch::autograd::edge_list edges = guess == 0 ? torch::autograd::collect_next_edges(wt, x)
                                           : arity == 3 ? torch::autograd::collect_next_edges(x, wt, bias)
                                                        : torch::autograd::collect_next_edges(x, wt);
        torch::autograd::set_history(y, new_node(capsule, container, guess, kind, x, std::move(edges)));
    }
    return wrap(y);
}

bool same_tensor(const Tensor &a, const Tensor &b)
{
    return a.unsafeGetTensorImpl() == b.unsafeGetTensorImpl() || (a.data_ptr() == b.data_ptr() && a.sizes() == b.sizes());
}

// weight.add_(gradient, alpha=...): the step of an optimizer.  nullptr without an error where it is another call.
PyObject *native_add_(const Dispatch &d, PyObject *args, PyObject *kwargs)
{
    if (PyTuple_GET_SIZE(args) != 2) return nullptr;
    PyObject *alpha = nullptr;
    if (kwargs != nullptr && PyDict_Size(kwargs) > 0) {
        alpha = PyDict_GetItem(kwargs, S_.alpha);
        if (alpha == nullptr || PyDict_Size(kwargs) != 1 || !(PyFloat_CheckExact(alpha) || PyLong_CheckExact(alpha))) return nullptr;
    }
    PyObject *cw = container_of(PyTuple_GET_ITEM(args, 0)), *cg = container_of(PyTuple_GET_ITEM(args, 1));
    if (cw == nullptr || cg == nullptr) return nullptr;
    PyObject *pw = PyList_GET_ITEM(cw, 0), *pg = PyList_GET_ITEM(cg, 0);
    if (!PyObject_TypeCheck(pw, &CoreType)) return nullptr;
    State &w = state_of(pw);
    at::Scalar a = 1;
    if (alpha != nullptr) {
        if (PyFloat_CheckExact(alpha)) a = PyFloat_AS_DOUBLE(alpha);
        else a = (int64_t)PyLong_AsLongLong(alpha);
    }
    if (PyObject_TypeCheck(pg, &CoreType)) {
        State &g = state_of(pg);
        if (g.layout != w.layout || !same_tensor(g.idx, w.idx)) return nullptr;
        w.val.add_(g.val, a);
    } else if ((PyObject *)Py_TYPE(pg) == d.dense_tensor) {
        PyObject *o = PyObject_GetAttr(pg, S_.data);
        if (o == nullptr) throw python_error();
        const bool plain = plain_tensor(o);
        Tensor t = plain ? THPVariable_Unpack(o) : Tensor();
        Py_DECREF(o);
        if (!plain || !t.is_cuda() || t.device() != w.val.device() || t.sizes() != at::IntArrayRef(w.geo.dims)) return nullptr;
        c10::DeviceGuard device(t.device());
        Tensor kept;
        {
            at::AutoDispatchBelowADInplaceOrView raw;
            kept = gather(w, t);
        }
        w.val.add_(kept, a);
    } else {
        return nullptr;
    }
    w.ops = Operands();
    PyObject *self = PyTuple_GET_ITEM(args, 0);
    Py_INCREF(self);
    return self;
}

// The dispatcher's warning in front of the error that is set; the error stays, or the one that the warning became.
void warn_of_failure(const Dispatch &d, PyObject *func)
{
    if (!PyErr_ExceptionMatches(PyExc_Exception)) return;
    PyObject *type, *value, *trace;
    PyErr_Fetch(&type, &value, &trace);
    PyErr_NormalizeException(&type, &value, &trace);
    if (trace != nullptr) PyException_SetTraceback(value, trace);
    PyObject *done = PyObject_CallFunctionObjArgs(d.failed, func, value, nullptr);
    if (done != nullptr) {
        Py_DECREF(done);
        PyErr_Restore(type, value, trace);
        return;
    }
    Py_XDECREF(type);
    Py_XDECREF(value);
    Py_XDECREF(trace);
}

// __torch_function__(func, types, args=(), kwargs=None), by position or by name
PyObject *torch_function(PyObject *capsule, PyObject *const *a, Py_ssize_t n, PyObject *names)
{
    PyObject *given[4] = {nullptr, nullptr, nullptr, nullptr};
    bool known = n <= 4;
    for (Py_ssize_t i = 0; i < n && known; i++) given[i] = a[i];
    for (Py_ssize_t k = 0; names != nullptr && k < PyTuple_GET_SIZE(names) && known; k++) {
        int i = 0;
        while (i < 4 && PyUnicode_Compare(PyTuple_GET_ITEM(names, k), S_.arguments[i]) != 0) i++;
        known = i < 4 && given[i] == nullptr;
        if (known) given[i] = a[n + k];
    }
    if (!known || given[0] == nullptr || given[1] == nullptr) {
        PyErr_SetString(PyExc_TypeError, "__torch_function__(func, types, args=(), kwargs=None)");
        return nullptr;
    }
    Dispatch &d = *dispatch_of(capsule);
    PyObject *func = given[0], *args = given[2] != nullptr ? given[2] : S_.nothing;
    PyObject *kwargs = given[3] != Py_None ? given[3] : nullptr;
    pybind11::object own_args, own_kwargs;      // any sequence and any mapping will do
    if (!PyTuple_Check(args)) {
        own_args = pybind11::reinterpret_steal<pybind11::object>(PySequence_Tuple(args));
        if (!own_args) return nullptr;
        args = own_args.ptr();
    }
    if (kwargs != nullptr && !PyDict_Check(kwargs)) {
        own_kwargs = pybind11::reinterpret_steal<pybind11::object>(PyDict_New());
        if (!own_kwargs || PyDict_Update(own_kwargs.ptr(), kwargs) < 0) return nullptr;
        kwargs = own_kwargs.ptr();
    }
    const int plain = PySet_Contains(d.plain, func);
    if (plain < 0) return nullptr;
    if (plain) {
        const auto before = at::impl::PythonTorchFunctionTLS::get_disabled_state();
        at::impl::PythonTorchFunctionTLS::set_disabled_state(at::impl::TorchFunctionDisabledState::SUBCLASSES_DISABLED);
        PyObject *r = PyObject_Call(func, args, kwargs);
        at::impl::PythonTorchFunctionTLS::set_disabled_state(before);
        if (r == nullptr) warn_of_failure(d, func);
        return r;
    }
    PyObject *r = nullptr;
    bool bad = false;
    try {
        PyObject *formats = PyDict_GetItem(d.native, func);
        if (formats != nullptr && (kwargs == nullptr || PyDict_Size(kwargs) == 0)) r = native_product(capsule, formats, args);
        else if (func == d.add_) r = native_add_(d, args, kwargs);
    }
    catch (const NmgError &e) { PyErr_SetString(g_nmg_error, e.what()); bad = true; }
    catch (python_error &e) { e.restore(); bad = true; }
    catch (const c10::Error &e) { PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace()); bad = true; }
    catch (const std::exception &e) { PyErr_SetString(PyExc_RuntimeError, e.what()); bad = true; }
    if (bad) {
        warn_of_failure(d, func);
        return nullptr;
    }
    if (r != nullptr) return r;
    return PyObject_CallFunctionObjArgs(d.slow, func, given[1], args, kwargs != nullptr ? kwargs : Py_None, nullptr);
}

PyMethodDef torch_function_def = {"__torch_function__", (PyCFunction)(void (*)(void))torch_function, METH_FASTCALL | METH_KEYWORDS, nullptr};

PyObject *py_make_torch_function(PyObject *, PyObject *args)
{
    Dispatch d;
    if (!PyArg_ParseTuple(args, "OOO!O!OOOOO", &d.slow, &d.failed, &PySet_Type, &d.plain, &PyDict_Type, &d.native, &d.grad_of, &d.add_,
                          &d.keep_all, &d.dense_tensor, &d.tensor))
        return nullptr;
    Py_INCREF(args);      // a dispatch module lives as long as the process; so does what its callable refers to
    PyObject *capsule = PyCapsule_New(new Dispatch(d), nullptr, nullptr);
    if (capsule == nullptr) return nullptr;
    PyObject *f = PyCFunction_New(&torch_function_def, capsule);
    Py_DECREF(capsule);
    return f;
}

PyObject *py_init(PyObject *, PyObject *arg)
{
    Py_INCREF(arg);
    Py_XDECREF(g_nmg_error);
    g_nmg_error = arg;
    Py_RETURN_NONE;
}

PyMethodDef functions[] = {
    {"init", py_init, METH_O, "init(error class)"},
    {"make_torch_function", py_make_torch_function, METH_VARARGS,
     "make_torch_function(slow, failed, plain, native, grad_of, add_, KeepAll, DenseTensor, Tensor)"},
    {"sparsify", py_sparsify, METH_VARARGS, "sparsify(core, dense): fills val and idx of a core whose layout is set"},
    {"spmm", (PyCFunction)(void (*)(void))py_spmm, METH_FASTCALL, "spmm(weight, x, bias, reduce_dim, kernel)"},
    {"column_sum", (PyCFunction)(void (*)(void))py_column_sum, METH_FASTCALL, "column_sum(x): sum over the rows"},
    {"spmm_tt", (PyCFunction)(void (*)(void))py_spmm_tt, METH_FASTCALL, "spmm_tt(weight, b)"},
    {"spmm_tt_dense", (PyCFunction)(void (*)(void))py_spmm_tt_dense, METH_FASTCALL, "spmm_tt_dense(weight, b, reduce_dim)"},
    {"dense_product", (PyCFunction)(void (*)(void))py_dense_product, METH_FASTCALL, "dense_product(tn, x, a), None where no kernel takes it"},
    {"w4_linear", py_w4_linear, METH_VARARGS, "w4_linear(B, meta, s, M, K, x, bias)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Native host path of the grouped n:m products.", -1, functions};

}  // namespace

PyMODINIT_FUNC PyInit__host()
{
    CoreType.tp_name = "sten_amd._host.Core";
    CoreType.tp_doc = "Values, indices, geometry and cached operands of a grouped n:m tensor.";
    CoreType.tp_basicsize = sizeof(Core);
    CoreType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    CoreType.tp_new = core_new;
    CoreType.tp_dealloc = core_dealloc;
    CoreType.tp_getset = core_getset;
    CoreType.tp_methods = core_methods;
    if (PyType_Ready(&CoreType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module_def);
    if (m == nullptr) return nullptr;
    g_nmg_error = PyExc_RuntimeError;
    Py_INCREF(g_nmg_error);
    S_ = {PyUnicode_InternFromString("kernel"), PyUnicode_InternFromString("variant"), PyUnicode_InternFromString("dense_variant"),
          PyUnicode_InternFromString("slices"), PyUnicode_InternFromString("expand"), PyUnicode_InternFromString("cache_dense"),
          PyUnicode_InternFromString("_wrapped_tensor_container"), PyUnicode_InternFromString("dense_shape"),
          PyUnicode_InternFromString("B"), PyUnicode_InternFromString("s"), PyUnicode_InternFromString("meta"),
          PyUnicode_InternFromString("grad_fmt"), PyUnicode_InternFromString("data"), PyUnicode_InternFromString("alpha"),
          {PyUnicode_InternFromString("func"), PyUnicode_InternFromString("types"), PyUnicode_InternFromString("args"),
           PyUnicode_InternFromString("kwargs")},
          PyTuple_New(0)};
    if (PyModule_AddIntConstant(m, "INTERFACE", kInterface) < 0) return nullptr;
    Py_INCREF(&CoreType);
    if (PyModule_AddObject(m, "Core", (PyObject *)&CoreType) < 0) return nullptr;
    return m;
}
