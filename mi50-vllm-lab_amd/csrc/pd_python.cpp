// pd_native: the Python face of libpthdec.so's operator calls (pth_dec.py, vllm_shim.py) in C++. A call
// fills the pd_tensor descriptors from its torch tensors, takes torch's current stream and calls
// the C entry whose address it is given; the entry does every check and reports its message.
// In Python with ctypes that work took 20-30 us per call, and the split plans, which are evaluated on every
// call too, 50-100 us: more than a decode layer of one user takes on the GPU. One eager layer step
// (cache write, routing, decode; 4,096 keys) 116 -> 19 us, a 16-token cache write 18.6 -> 3.7.
//
// The module holds no state: the library that is active is pth_dec.load_library()'s business.
#include <Python.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <exception>
#include <functional>
#include <queue>
#include <vector>

#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include "pd_plan.hpp"
#include "pth_dec.h"

namespace {

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kChar: return PD_DTYPE_INT8;
        case at::kHalf: return PD_DTYPE_FP16;
        case at::kFloat: return PD_DTYPE_FP32;
        case at::kInt: return PD_DTYPE_INT32;
        case at::kBFloat16: return PD_DTYPE_BF16;
        case at::kLong: return PD_DTYPE_INT64;
        default: return 0;
    }
}

// Descriptor of a tensor argument; false with a Python error set.
bool describe(PyObject* o, pd_tensor& d) {
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
        return false;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.dim() > PD_MAX_DIMS) {
        PyErr_Format(PyExc_RuntimeError, "tensor rank %lld exceeds %d", (long long)t.dim(), PD_MAX_DIMS);
        return false;
    }
    d = pd_tensor{};
    d.data = t.data_ptr();
    d.dtype = dtype_code(t.scalar_type());
    d.ndim = (int)t.dim();
    for (int i = 0; i < d.ndim; ++i) {
        d.sizes[i] = t.size(i);
        d.strides[i] = t.stride(i);
    }
    return true;
}

bool describe_all(PyObject* const* o, pd_tensor* d, int n) {
    for (int i = 0; i < n; ++i)
        if (!describe(o[i], d[i])) return false;
    return true;
}

// torch's current stream on a tensor's device, with that device current while this object lives.
class OnDevice {
public:
    explicit OnDevice(PyObject* o) {
        const c10::Device dev = THPVariable_Unpack(o).device();
        if (!dev.is_cuda()) return;  // the entry gets no further than its checks
        before_ = c10::hip::current_device();
        const c10::DeviceIndex index = dev.has_index() ? dev.index() : before_;
        if (index != before_) c10::hip::set_device(index);
        now_ = index;
        stream = c10::hip::getCurrentHIPStream(index).stream();
    }
    ~OnDevice() {
        try {
            if (now_ != before_) c10::hip::set_device(before_);
        } catch (...) {  // the call itself has already been made
        }
    }
    OnDevice(const OnDevice&) = delete;
    hipStream_t stream = nullptr;

private:
    c10::DeviceIndex before_ = -1, now_ = -1;
};

bool as_int64(PyObject* o, int64_t& v) {
    v = PyLong_AsLongLong(o);
    return !(v == -1 && PyErr_Occurred());
}
bool as_double(PyObject* o, double& v) {
    v = PyFloat_AsDouble(o);
    return !(v == -1.0 && PyErr_Occurred());
}
template <class F>
bool entry(PyObject* o, F& f) {
    f = reinterpret_cast<F>(PyLong_AsVoidPtr(o));
    return f != nullptr || (PyErr_Occurred() ? false : (PyErr_SetString(PyExc_ValueError, "null entry point"), false));
}
bool count_is(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return false;
}
PyObject* done(int rc, const char* err) {
    if (rc == 0) Py_RETURN_NONE;
    PyErr_SetString(PyExc_RuntimeError, err);
    return nullptr;
}
// No C++ exception crosses into Python (torch's accessors throw for tensors without storage).
template <class F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

// decode(entry, q, key_cache, value_cache, k_scale, v_scale, block_table, seq_lens, query_start_loc, out, scale,
//        part_o, part_m, part_l, num_seqs, qmax, nsplit, window, causal)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        decltype(&pth_dec_decode) fn;
        pd_tensor t[9], p[3];
        double scale;
        int64_t v[5];
        if (!count_is(n, 19) || !entry(a[0], fn) || !describe_all(a + 1, t, 9) || !as_double(a[10], scale) ||
            !describe_all(a + 11, p, 3))
            return nullptr;
        for (int i = 0; i < 5; ++i)
            if (!as_int64(a[14 + i], v[i])) return nullptr;
        char err[256] = "";
        OnDevice dev(a[1]);
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6], &t[7], &t[8], scale, &p[0], &p[1], &p[2], v[0], v[1],
                v[2], v[3], v[4], dev.stream, err, (int)sizeof err);
        Py_END_ALLOW_THREADS;
        return done(rc, err);
    });
}

// prefill(entry, q, key_cache, value_cache, block_table, seq_lens, scale, q_abs_offset, out)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        decltype(&pth_fa_forward) fn;
        pd_tensor t[5], p[2];
        double scale;
        if (!count_is(n, 9) || !entry(a[0], fn) || !describe_all(a + 1, t, 5) || !as_double(a[6], scale) ||
            !describe_all(a + 7, p, 2))
            return nullptr;
        char err[256] = "";
        OnDevice dev(a[1]);
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(&t[0], &t[1], &t[2], &t[3], &t[4], scale, &p[0], &p[1], dev.stream, err, (int)sizeof err);
        Py_END_ALLOW_THREADS;
        return done(rc, err);
    });
}

// prefill_split(entry, q, key_cache, value_cache, block_table, seq_lens, scale, q_abs_offset, out, workspace, nsplit, exact)
PyObject* prefill_split(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        decltype(&pth_fa_forward_split) fn;
        pd_tensor t[5], p[3];
        double scale;
        int64_t nsplit, exact;
        if (!count_is(n, 12) || !entry(a[0], fn) || !describe_all(a + 1, t, 5) || !as_double(a[6], scale) ||
            !describe_all(a + 7, p, 3) || !as_int64(a[10], nsplit) || !as_int64(a[11], exact))
            return nullptr;
        char err[256] = "";
        OnDevice dev(a[1]);
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(&t[0], &t[1], &t[2], &t[3], &t[4], scale, &p[0], &p[1], &p[2], nsplit, exact, dev.stream, err,
                (int)sizeof err);
        Py_END_ALLOW_THREADS;
        return done(rc, err);
    });
}

// prefill_balanced(entry, workspace entry, q, key_cache, value_cache, block_table, seq_lens, scale, q_abs_offset, out,
//                  query_start, max_keys, nsplit, exact): pth_fa_forward_balanced with its workspace from torch's allocator.
// query_start None: the batch form, with q_abs_offset; a list of row numbers: the rows form. False, with nothing
// launched, if the entry does not take such a call or its workspace cannot be had.
PyObject* prefill_balanced(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        decltype(&pth_fa_forward_balanced) fn;
        decltype(&pth_fa_balanced_workspace) need;
        pd_tensor t[5], qa{}, od, wd{};
        double scale;
        int64_t max_keys, nsplit, exact;
        if (!count_is(n, 14) || !entry(a[0], fn) || !entry(a[1], need) || !describe_all(a + 2, t, 5) ||
            !as_double(a[7], scale) || (a[8] != Py_None && !describe(a[8], qa)) || !describe(a[9], od) ||
            !as_int64(a[11], max_keys) || !as_int64(a[12], nsplit) || !as_int64(a[13], exact))
            return nullptr;
        int starts[33];
        int64_t seqs = 0;
        const bool rows = a[10] != Py_None;
        if (rows) {
            if (!PyList_Check(a[10]) || PyList_GET_SIZE(a[10]) < 2) {
                PyErr_SetString(PyExc_TypeError, "query_start must be a list of at least two row numbers");
                return nullptr;
            }
            seqs = PyList_GET_SIZE(a[10]) - 1;
            if (seqs > 32) Py_RETURN_FALSE;
            for (int64_t i = 0; i <= seqs; ++i) {
                int64_t v;
                if (!as_int64(PyList_GET_ITEM(a[10], i), v)) return nullptr;
                starts[i] = (int)std::max<int64_t>(-1, std::min<int64_t>(v, INT32_MAX));
            }
        }
        const bool shaped = t[0].ndim == (rows ? 3 : 4) && t[1].ndim == 4 && t[3].ndim == 2;
        OnDevice dev(a[2]);
        int64_t floats = 0;
        if (shaped && nsplit == 0)
            floats = need(rows ? seqs : t[0].sizes[0], rows ? starts : nullptr, rows ? 0 : t[0].sizes[2], t[0].sizes[1],
                          t[1].sizes[2], max_keys, t[3].sizes[1] * t[1].sizes[1]);
        else if (shaped && rows)
            floats = nsplit > 1 ? (starts[1] - starts[0]) * t[0].sizes[1] * nsplit * 258 : 4;
        if (floats <= 0) Py_RETURN_FALSE;
        at::Tensor ws;
        try {
            ws = at::empty({floats}, THPVariable_Unpack(a[2]).options().dtype(at::kFloat));
        } catch (const c10::OutOfMemoryError&) {
            Py_RETURN_FALSE;
        }
        wd.data = ws.data_ptr();
        wd.dtype = PD_DTYPE_FP32;
        wd.ndim = 1;
        wd.sizes[0] = floats;
        wd.strides[0] = 1;
        char err[256] = "";
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(&t[0], &t[1], &t[2], &t[3], &t[4], scale, a[8] == Py_None ? nullptr : &qa, rows ? starts : nullptr, seqs, &od,
                &wd, max_keys, nsplit, exact, dev.stream, err, (int)sizeof err);
        Py_END_ALLOW_THREADS;
        if (rc != 0) return done(rc, err);
        Py_RETURN_TRUE;
    });
}

// cache_write(entry, key, value, key_cache, value_cache, k_scale, v_scale, slot_mapping)
PyObject* cache_write(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        decltype(&pth_cache_write) fn;
        pd_tensor t[7];
        if (!count_is(n, 8) || !entry(a[0], fn) || !describe_all(a + 1, t, 7)) return nullptr;
        char err[256] = "";
        OnDevice dev(a[1]);
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(&t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6], dev.stream, err, (int)sizeof err);
        Py_END_ALLOW_THREADS;
        return done(rc, err);
    });
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The lengths of a batch on the host: a contiguous int32 or int64 CPU tensor.
class Lengths {
public:
    // false with a Python error set
    bool take(PyObject* o, int64_t num_seqs, int64_t max_q, int64_t window) {
        if (!THPVariable_Check(o)) {
            PyErr_SetString(PyExc_TypeError, "lens must be a tensor");
            return false;
        }
        const at::Tensor& lens = THPVariable_Unpack(o);
        wide_ = lens.scalar_type() == at::kLong;
        if (!lens.device().is_cpu() || !lens.is_contiguous() || (!wide_ && lens.scalar_type() != at::kInt)) {
            PyErr_SetString(PyExc_ValueError, "lens must be a contiguous int32 or int64 CPU tensor");
            return false;
        }
        data_ = lens.const_data_ptr();
        count = std::min<int64_t>(lens.numel(), num_seqs);
        most_ = window > 0 ? window + max_q : INT64_MAX;
        return true;
    }
    // visible keys of sequence i in 32-key tiles (+ 1: alignment)
    int64_t tiles(int64_t i) const {
        const int64_t len = std::min<int64_t>(wide_ ? static_cast<const int64_t*>(data_)[i] : static_cast<const int32_t*>(data_)[i], most_);
        return len > 0 ? ceil_div(len, 32) + 1 : 0;
    }
    int64_t count = 0;

private:
    const void* data_ = nullptr;
    bool wide_ = false;
    int64_t most_ = INT64_MAX;
};

// plan_decode(lens, num_seqs, num_kv_heads, rows, max_q, window, cap, cus, tile_us, fixed_us, empty_us, merge_us_per_mb,
//             row_bytes): vllm_shim.decode_splits' makespan model.
PyObject* plan_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t num_seqs, hkv, rows, max_q, window, cap, cus;
        double tile_us, fixed_us, empty_us, merge_us, row_bytes;
        if (!count_is(n, 13) || !as_int64(a[1], num_seqs) || !as_int64(a[2], hkv) || !as_int64(a[3], rows) ||
            !as_int64(a[4], max_q) || !as_int64(a[5], window) || !as_int64(a[6], cap) || !as_int64(a[7], cus) ||
            !as_double(a[8], tile_us) || !as_double(a[9], fixed_us) || !as_double(a[10], empty_us) ||
            !as_double(a[11], merge_us) || !as_double(a[12], row_bytes))
            return nullptr;
        Lengths lens;
        if (!lens.take(a[0], num_seqs, max_q, window)) return nullptr;
        bool live = false;
        for (int64_t i = 0; i < lens.count; ++i) live = live || lens.tiles(i) > 0;
        if (!live) return PyLong_FromLong(1);
        int64_t best_s = cap;
        double best_t = HUGE_VAL;
        for (int64_t s = 1;; s = s * 2 < cap ? s * 2 : cap) {  // powers of two, and the cap
            double total = 0.0, longest = 0.0;
            for (int64_t i = 0; i < lens.count; ++i) {
                const int64_t t = lens.tiles(i), per = std::max<int64_t>(ceil_div(t, s), 1);
                const int64_t filled = t > 0 ? ceil_div(t, per) : 0;  // splits holding tiles
                const double us = fixed_us + tile_us * (double)ceil_div(per, 4);
                total += (double)filled * us + (double)(s - filled) * empty_us;
                if (t > 0) longest = std::max(longest, us);
            }
            const double span = std::max((double)hkv * total / (double)cus, longest) +
                                merge_us * (double)rows * (double)s * row_bytes / 1e6;
            if (span < best_t - 1e-9) best_s = s, best_t = span;
            if (s >= cap) break;
        }
        return PyLong_FromLongLong(best_s);
    });
}

// deal_pays(lens, num_seqs, num_kv_heads, max_q, window, cus): whether pd_balanced_kernel is rated faster than one unsplit
// workgroup per (sequence, kv head), of which there are more than CUs. In tiles (a workgroup's set-up and
// merge are kSegmentUnits = 12): the workgroups run in order on the CU that is free first, the kv heads of a
// sequence side by side; the deal takes an equal share and, measured, 15 % and 8 tiles more (a share's ends, its second
// segment, the planning on the device). us, unsplit against dealt (24 q / 4 kv heads), with the two ratings: 100 x 512
// keys 34.8 / 38.1 (58 : 60), 160 x 1,024 91.7 / 91.7 (135 : 137), 96 x 2,048 100 / 94 (154 : 141), 256 of 16 to 4,096
// 289 / 248, 70 x 8,192 316 / 228.
PyObject* deal_pays(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t num_seqs, hkv, max_q, window, cus;
        if (!count_is(n, 6) || !as_int64(a[1], num_seqs) || !as_int64(a[2], hkv) || !as_int64(a[3], max_q) ||
            !as_int64(a[4], window) || !as_int64(a[5], cus))
            return nullptr;
        Lengths lens;
        if (!lens.take(a[0], num_seqs, max_q, window)) return nullptr;
        constexpr int64_t kSegment = 12;
        const int64_t lanes = std::max<int64_t>(1, cus / std::max<int64_t>(1, hkv));
        std::priority_queue<int64_t, std::vector<int64_t>, std::greater<int64_t>> busy;  // until when, of each lane
        int64_t total = 0, span = 0;
        for (int64_t i = 0; i < lens.count; ++i) {
            const int64_t t = lens.tiles(i);
            if (t == 0) continue;
            int64_t at = t + kSegment;
            total += at;
            if ((int64_t)busy.size() == lanes) {
                at += busy.top();
                busy.pop();
            }
            busy.push(at);
            span = std::max(span, at);
        }
        const double share = (double)total * (double)hkv / (double)cus;
        return PyBool_FromLong((double)span > 1.15 * share + 8.0);
    });
}

// plan_prefill(work_items, rows, max_keys, block_size, cus, wg_us, mb_us, merge_us, max_splits, min_tiles, max_workspace,
//              lds_table, global_factor, sq, tok_per_wg, rows per kv head, exact): pth_dec.prefill_splits' makespan model, with
// the tile times of pd_plan.hpp. With sq > 0 (the chunk's query tokens, the last of max_keys keys) the 256-row kernel, at the
// counts where the launch takes it, is rated as well, and the result is 0 where the balanced launch is rated
// faster. Equal query tiles (the kernel's aligned split) stay with the splits, whose kernel takes less per tile.
PyObject* plan_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t items, rows, max_keys, block_size, cus, max_splits, min_tiles, max_workspace, lds_table, sq, tok, head_rows, exact;
        double wg_us, mb_us, merge_us, factor;
        if (!count_is(n, 17) || !as_int64(a[0], items) || !as_int64(a[1], rows) || !as_int64(a[2], max_keys) ||
            !as_int64(a[3], block_size) || !as_int64(a[4], cus) || !as_double(a[5], wg_us) || !as_double(a[6], mb_us) ||
            !as_double(a[7], merge_us) || !as_int64(a[8], max_splits) || !as_int64(a[9], min_tiles) ||
            !as_int64(a[10], max_workspace) || !as_int64(a[11], lds_table) || !as_double(a[12], factor) || !as_int64(a[13], sq) ||
            !as_int64(a[14], tok) || !as_int64(a[15], head_rows) || !as_int64(a[16], exact))
            return nullptr;
        const pd::FaTimes& times = pd::fa_times(exact != 0);
        const int64_t keys = std::max<int64_t>(0, max_keys), bs = std::max<int64_t>(1, block_size), tiles = ceil_div(keys, 32);
        // `count` workgroups per split, of which each takes `tile_us` per tile
        auto cost = [&](int64_t count, int64_t s, double tile_us) {
            const int64_t rounds = ceil_div(count * s, cus), per = ceil_div(tiles, s);
            const bool in_lds = block_size % 16 == 0 ? 2 * per <= lds_table : ceil_div(keys, bs) <= lds_table;
            double t = (double)rounds * ((double)per * (tile_us * (in_lds ? 1.0 : factor)) + wg_us);
            if (s > 1) t += merge_us + mb_us * (double)rows * (double)s * 1032 / 1e6;
            return t;
        };
        const int64_t top = std::max<int64_t>(1, std::min(max_splits, tiles / min_tiles));
        auto fits = [&](int64_t s) { return s == 1 || rows * s * 1032 <= max_workspace; };
        int64_t best = 1;
        double best_t = cost(items, 1, times.tile);
        for (int64_t s = 2; s <= top && fits(s); ++s) {
            const double t = cost(items, s, times.tile);
            if (t < best_t) best = s, best_t = t;
        }
        if (sq > 0 && items > 0) {
            const int64_t nqt = ceil_div(sq, std::max<int64_t>(1, tok)), heads = items / nqt;
            const int64_t wide_items = ceil_div(head_rows, 256) * heads;
            auto wide = [&](int64_t s) { return pd::fa_wide_saves(ceil_div(wide_items * s, cus), ceil_div(items * s, cus), exact != 0); };
            for (int64_t s = 1; s <= top && fits(s); ++s) {
                if (!wide(s)) continue;
                const double t = cost(wide_items, s, times.wide_tile);
                if (t < best_t) best = s, best_t = t;
            }
            // key tiles that a workgroup whose last token is `last` - 1 sees
            auto seen = [&](int64_t last) { return ceil_div(std::max<int64_t>(0, keys - sq) + std::min(sq, last), 32); };
            // A launch of s splits as the hardware runs it (pd_prefill_kernel's order): each of the 8 XCDs has a contiguous
            // part of the workgroups, a query tile's splits apart and the tiles ascending, and starts the next one on
            // the CU that is free first. The workgroups' lengths differ by the causal triangle, which the rounds above do
            // not see: 3 chunks of 1,000 fresh tokens run 109 us unsplit (114 here, 137 in rounds) and 133 dealt.
            auto ordered = [&](int64_t s, int64_t sequences) {
                const bool w = wide(s);
                const int64_t nq = w ? ceil_div(head_rows, 256) : nqt, group = std::max<int64_t>(1, head_rows / sq);
                const int64_t total = nq * s * sequences, lanes = std::max<int64_t>(1, cus / 8);
                if (total > 64 * cus) return 0.0;  // many rounds: as even as dealt
                double span = 0.0;
                for (int64_t xcd = 0, i = 0; xcd < 8; ++xcd) {
                    std::priority_queue<double, std::vector<double>, std::greater<double>> busy;
                    for (const int64_t end = i + total / 8 + (xcd < total % 8 ? 1 : 0); i < end; ++i) {
                        const int64_t x = i % (nq * s), q = x % nq, split = x / nq;
                        const int64_t t = seen(w ? std::min((q + 1) * 256 - 1, head_rows - 1) / group + 1 : (q + 1) * tok);
                        const int64_t per = ceil_div(t, s), mine = std::max<int64_t>(0, std::min(per, t - split * per));
                        double at = (double)mine * (w ? times.wide_tile : times.tile) + wg_us;
                        if ((int64_t)busy.size() == lanes) {
                            at += busy.top();
                            busy.pop();
                        }
                        busy.push(at);
                        span = std::max(span, at);
                    }
                }
                return s > 1 ? span + merge_us + mb_us * (double)rows * (double)s * 1032 / 1e6 : span;
            };
            int64_t units = 0;
            for (int64_t q = 0; q < nqt; ++q) units += seen((q + 1) * tok) + pd::kFaSegmentUnits;
            const int64_t share = std::max<int64_t>(pd::kFaMinShare, ceil_div(units * heads, cus)), ns = items <= cus ? cus / items : 0;
            const bool aligned = ns > 0 && ceil_div(tiles, ns) <= share + share / pd::kFaAlignedPart;
            const double dealt = times.deal_unit * (double)(share + pd::kFaDealSpareUnits) + pd::kFaDealFixedUs;
            if (!aligned && dealt < pd::kFaDealMargin * best_t && dealt < pd::kFaDealMargin * ordered(best, heads)) best = 0;
        }
        return PyLong_FromLongLong(best);
    });
}

#define PD_METHOD(f, doc) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, doc}
PyMethodDef methods[] = {
    PD_METHOD(decode, "pth_dec_decode on torch tensors"),
    PD_METHOD(prefill, "pth_fa_forward / pth_fa_forward_exact on torch tensors"),
    PD_METHOD(prefill_split, "pth_fa_forward_split on torch tensors"),
    PD_METHOD(prefill_balanced, "pth_fa_forward_balanced on torch tensors"),
    PD_METHOD(cache_write, "pth_cache_write on torch tensors"),
    PD_METHOD(plan_decode, "split count of a decode batch"),
    PD_METHOD(deal_pays, "whether a batch of unsplit sequences is dealt instead"),
    PD_METHOD(plan_prefill, "key splits of a prefill launch"),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "pd_native", "operator calls of libpthdec.so on torch tensors", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_pd_native() { return PyModule_Create(&module); }
