// Host path of the sparse convolution calls: everything between the Python modules and the C ABI of
// libsphconv_hip.so (include/sphconv_hip.h) that runs once per call.
//
// A layer of a LiDAR network is one to three launches of 5 to 50 us, so what the host does around them decides the
// smaller calls: through Python and ctypes a layer took 35 us of host time (allocations 1.8 us each, a ctypes call with
// its argument conversions 3 to 5 us, struct building 2.5 us), and a single scan's encoder pass waited for its host for
// more than half of its time.  Here a call allocates its outputs, fills the structs and launches in one step.  Policy
// (which kernel form a book takes, what is kept) stays in Python; this file holds no state beyond pinned words.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <memory>
#include <mutex>
#include <optional>
#include <unordered_map>
#include <vector>

#include "../../include/sphconv_hip.h"
#include "outcoords.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

PyObject *g_error = nullptr; // the package's SphconvError

[[noreturn]] void raise(const std::string &msg, PyObject *type = nullptr)
{
    PyErr_SetString(type ? type : g_error ? g_error : PyExc_RuntimeError, msg.c_str());
    throw py::error_already_set();
}
void check(int rc)
{
    if (rc) raise("libsphconv_hip: " + std::string(sph_last_error()) + " (status " + std::to_string(rc) + ")");
}

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return SPH_F32;
    case at::kHalf: return SPH_F16;
    case at::kBFloat16: return SPH_BF16;
    case at::kChar: return SPH_I8;
    default: raise("unsupported element type " + std::string(toString(t)) + " (float32, float16, bfloat16, int8)");
    }
}
// device address of a contiguous GPU tensor
template <typename T = void> T *ptr(const Tensor &t)
{
    if (!t.is_cuda()) raise("expected a GPU tensor, got device " + t.device().str());
    if (!t.is_contiguous()) raise("expected a contiguous tensor");
    return (T *)t.data_ptr();
}
template <typename T = void> T *ptr(const OptTensor &t) { return t ? ptr<T>(*t) : nullptr; }

// The device of a call's tensors, current while the call allocates and launches, and torch's current stream on it.  A
// kernel is launched on a stream that came from here and nowhere else: torch's own operations follow their tensors'
// device, so a launch on the stream of whatever device happens to be current would not be ordered with what made its inputs.
struct OnDevice {
    c10::OptionalDeviceGuard guard; // (empty where the device is current anyway: leaving a guard sets the device again)
    hipStream_t stream;
    explicit OnDevice(const Tensor &t)
    {
        if (!t.is_cuda()) raise("expected a GPU tensor, got device " + t.device().str());
        if (t.device().index() != c10::hip::current_device()) guard.reset_device(t.device());
        stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    }
};

// The default stream (handle 0) cannot be recorded and is not asked: while another stream that waits for it is recorded, the question
// alone is an error.  A stream that cannot say counts as recorded, and leaves no error for the next launch to report.
bool being_recorded(hipStream_t st)
{
    if (!st) return false;
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &s) == hipSuccess) return s != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

Tensor bytes(size_t n, const Tensor &like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte).requires_grad(false)); }
Tensor ints(int64_t n, const Tensor &like) { return at::empty({n}, like.options().dtype(at::kInt).requires_grad(false)); }

// ---- pinned words the GPU writes and the host waits for -----------------------------------------
// One 8-byte word per wait in flight, from pages of pinned memory that live as long as the process (pinning costs a
// system call, and the GPU may still write to a word whose owner is gone: such a word is not handed out again).
class PinnedWords {
    std::mutex m;
    std::vector<Tensor> pages;
    std::vector<int64_t *> free_;

public:
    int64_t *take()
    {
        std::lock_guard<std::mutex> lock(m);
        if (free_.empty()) {
            pages.push_back(at::empty({64}, at::TensorOptions().dtype(at::kLong).pinned_memory(true)));
            int64_t *p = pages.back().data_ptr<int64_t>();
            for (int i = 63; i >= 0; i--) free_.push_back(p + i);
        }
        int64_t *w = free_.back();
        free_.pop_back();
        return w;
    }
    void give(int64_t *w)
    {
        std::lock_guard<std::mutex> lock(m);
        free_.push_back(w);
    }
};
PinnedWords &pinned()
{
    static PinnedWords *p = new PinnedWords; // never destroyed: the GPU's memory goes before static objects do
    return *p;
}

// A word set to -1 that a kernel on `st` will overwrite.  wait() returns as soon as the store arrives, without an
// event (recording one costs 4.6 us) and without waiting for what was enqueued behind that kernel; should the store
// not arrive within 20 ms the stream is waited for instead, which also reports an error it holds.
class HostWord {
    int64_t *w;
    hipStream_t st;
    bool seen = false;

public:
    explicit HostWord(const OnDevice &here) : w(pinned().take()), st(here.stream) { __atomic_store_n(w, (int64_t)-1, __ATOMIC_SEQ_CST); }
    HostWord(const HostWord &) = delete;
    HostWord &operator=(const HostWord &) = delete;
    ~HostWord()
    {
        if (seen) pinned().give(w);
    }
    int32_t *address() { return (int32_t *)w; }
    // the word, to an owner who gives it back once the store has arrived; only where wait() has not returned
    int64_t *leave() const { return w; }
    // no kernel was given its address
    void unused() { seen = true; }
    hipStream_t on() const { return st; }
    // both: the two 32-bit halves are written by one store; otherwise only the low half is written
    int64_t wait(bool both)
    {
        const int64_t none = -1;
        auto ready = [&]() {
            if (both) return __atomic_load_n(w, __ATOMIC_ACQUIRE) != none;
            return __atomic_load_n((int32_t *)w, __ATOMIC_ACQUIRE) != (int32_t)-1;
        };
        if (!ready()) {
            py::gil_scoped_release nogil;
            const auto t0 = std::chrono::steady_clock::now();
            int spin = 0;
            while (!ready()) {
                if (++spin % 64) {
                    __builtin_ia32_pause();
                    continue;
                }
                if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) {
                    const hipError_t e = hipStreamSynchronize(st);
                    if (e != hipSuccess) {
                        py::gil_scoped_acquire gil;
                        raise(std::string("waiting for the GPU: ") + hipGetErrorString(e));
                    }
                    break;
                }
            }
        }
        if (!ready()) raise("the kernel that reports a count has not run");
        seen = true;
        return both ? __atomic_load_n(w, __ATOMIC_ACQUIRE) : (int64_t) __atomic_load_n((int32_t *)w, __ATOMIC_ACQUIRE);
    }
};

// ---- cells on the GPU that a count adds to --------------------------------------------------------
// Zeros before and after a count, so a count in flight has cells of its own and the next one needs no launch that clears them.
// Pages of 64 counts' cells (139 KB) for each device, as many as there were counts in flight at once; like the pinned words they
// live as long as the process.  A count that nobody waited for (its layer did not run, or raised, the call that starts the count
// itself among them) leaves its cells with its word, and both are handed out again once the word says that the count has ended.
class CountCells {
    std::mutex m;
    std::vector<Tensor> pages;
    std::unordered_map<int, std::vector<uint64_t *>> free_;
    struct Left { int device; uint64_t *cells; int64_t *word; };
    std::vector<Left> left;
    void collect()
    {
        size_t kept = 0;
        for (const Left &l : left)
            if (__atomic_load_n((int32_t *)l.word, __ATOMIC_ACQUIRE) == (int32_t)-1) left[kept++] = l;
            else {
                free_[l.device].push_back(l.cells);
                pinned().give(l.word);
            }
        left.resize(kept);
    }

public:
    // null: no page can be had just now (the stream that would clear it cannot be waited for)
    uint64_t *take(const OnDevice &here, const Tensor &like)
    {
        const int device = like.device().index();
        std::lock_guard<std::mutex> lock(m);
        if (!left.empty()) collect();
        std::vector<uint64_t *> &f = free_[device];
        if (f.empty()) {
            const int words = sph_outcoords2_cell_words();
            Tensor page = at::zeros({64, words}, like.options().dtype(at::kLong).requires_grad(false));
            // another stream's count may be the first to use them
            if (hipStreamSynchronize(here.stream) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
            pages.push_back(page);
            for (int i = 63; i >= 0; i--) f.push_back((uint64_t *)page.data_ptr<int64_t>() + (int64_t)i * words);
        }
        uint64_t *c = f.back();
        f.pop_back();
        return c;
    }
    void give(int device, uint64_t *c)
    {
        std::lock_guard<std::mutex> lock(m);
        free_[device].push_back(c);
    }
    void leave(int device, uint64_t *c, int64_t *word)
    {
        std::lock_guard<std::mutex> lock(m);
        left.push_back(Left{device, c, word});
    }
};
CountCells &count_cells()
{
    static CountCells *p = new CountCells; // never destroyed, as the pinned words
    return *p;
}

// A count's cells, beside the word it reports to: given back with the count's end, whichever way its owner ends.
class HeldCells {
    HostWord &word;
    uint64_t *cells = nullptr;
    int device = 0;
    bool adding = false; // a kernel may add to them

public:
    explicit HeldCells(HostWord &w) : word(w) {}
    HeldCells(const HeldCells &) = delete;
    HeldCells &operator=(const HeldCells &) = delete;
    ~HeldCells()
    {
        if (!cells) return;
        if (adding) count_cells().leave(device, cells, word.leave());
        else {
            count_cells().give(device, cells);
            word.unused();
        }
    }
    bool take(const OnDevice &here, const Tensor &like)
    {
        device = like.device().index();
        cells = count_cells().take(here, like);
        return cells != nullptr;
    }
    uint64_t *get() const { return cells; }
    void launched() { adding = true; }
    // the word has arrived: all zeros again
    void done()
    {
        if (cells) count_cells().give(device, cells);
        cells = nullptr;
    }
};

// ---- geometry and books -------------------------------------------------------------------------
struct Geometry {
    sph_geom g;
    Geometry(int batch, const std::vector<int> &in, const std::vector<int> &out, const std::vector<int> &kernel,
             const std::vector<int> &stride, const std::vector<int> &padding, const std::vector<int> &dilation)
    {
        for (auto *v : {&in, &out, &kernel, &stride, &padding, &dilation})
            if (v->size() < 3) raise("a geometry has three axes");
        g.B = batch;
        for (int d = 0; d < 3; d++) {
            g.S[d] = in[d]; g.O[d] = out[d]; g.K[d] = kernel[d];
            g.stride[d] = stride[d]; g.pad[d] = padding[d]; g.dil[d] = dilation[d];
        }
    }
    uintptr_t address() const { return (uintptr_t)&g; }
    // whether the compressed coordinates of a tensor are what the rule kernels take on this geometry
    bool takes(const Tensor &z_idx, const Tensor &z_ptr) const
    {
        return z_idx.scalar_type() == at::kInt && z_ptr.scalar_type() == at::kInt && z_idx.dim() == 1 && z_ptr.dim() == 3 &&
               z_ptr.size(0) == g.B && z_ptr.size(1) == g.S[0] && z_ptr.size(2) == g.S[1] && z_idx.is_contiguous() &&
               z_ptr.is_contiguous() && z_idx.is_cuda() && z_ptr.is_cuda();
    }
};

// Device arrays of one book, carved out of one allocation.
struct BookBuffers {
    Tensor storage;
    sph_book book;
    int rows, kv, ntiles, cap;
    bool by_row, groups;
    size_t off[6], size[6];
    BookBuffers(int rows_, int kv_, const c10::Device &dev, bool by_row_, bool groups_)
        : rows(rows_), kv(kv_), ntiles(sph_book_tiles(rows_)), cap(sph_book_cap(kv_)), by_row(by_row_), groups(groups_ || !by_row_)
    {
        const size_t nt = ntiles > 0 ? ntiles : 1, g = groups ? 1 : 0;
        const size_t sizes[6] = {nt * 4, nt * (kv + 1) * 2, g * nt * cap * 4, g * nt * cap * SPH_GROUP * 4,
                                 g * nt * cap * SPH_GROUP * 4, by_row ? nt * kv * SPH_TILE_ROWS * 4 : 0};
        size_t total = 0;
        for (int i = 0; i < 6; i++) {
            off[i] = total;
            size[i] = sizes[i];
            total += (sizes[i] + 255) & ~(size_t)255;
        }
        storage = at::empty({(int64_t)total}, at::TensorOptions().dtype(at::kByte).device(dev));
        char *p = (char *)storage.data_ptr();
        book.tile_ngrp = (int32_t *)(p + off[0]);
        book.tile_koff = (uint16_t *)(p + off[1]);
        book.grp_k = groups ? (int32_t *)(p + off[2]) : nullptr;
        book.grp_gather = groups ? (int32_t *)(p + off[3]) : nullptr;
        book.grp_owner = groups ? (int32_t *)(p + off[4]) : nullptr;
        book.rows = rows;
        book.KV = kv;
        book.tile_nbr = by_row ? (int32_t *)(p + off[5]) : nullptr;
        book.middle_run = 0;
    }
    uintptr_t address() const { return (uintptr_t)&book; }
};

// A table of the rows' columns, or null when there is none (or it does not fit).
const int32_t *row_table(const OptTensor &t, int rows)
{
    if (!t || !t->is_cuda() || t->scalar_type() != at::kInt || !t->is_contiguous() || t->dim() != 1 || t->size(0) != rows) return nullptr;
    return (const int32_t *)t->data_ptr();
}

// ---- weights ------------------------------------------------------------------------------------
// weight [KV,a,b] -> description of its fragment-ordered copy in element type dt, for the contraction over a
// (transpose: over b, W[k]^T; reverse: offsets from the last to the first); allocates the copy.
sph_pack_desc describe_pack(const Tensor &w, bool transpose, bool reverse, int dt, Tensor &packed)
{
    if (w.dim() != 3) raise("weight must be a GPU tensor [KV,iC,oC]");
    const int kv = (int)w.size(0), a = (int)w.size(1), b = (int)w.size(2);
    sph_pack_desc d;
    d.dt = (sph_dtype)dt;
    const int src = dtype_code(w.scalar_type());
    if (src != dt && src != SPH_F32) raise("a packed weight keeps the weight's type, or narrows float32");
    d.w_f32 = src == SPH_F32 && dt != SPH_F32;
    d.KV = kv;
    d.kdim = transpose ? b : a;
    d.ndim = transpose ? a : b;
    d.stride_k = (long)a * b;
    d.stride_kk = transpose ? 1 : b;
    d.stride_n = transpose ? b : 1;
    d.w = ptr(w);
    if (reverse) {
        d.w = (const char *)d.w + (size_t)(kv - 1) * a * b * w.element_size();
        d.stride_k = -d.stride_k;
    }
    const size_t n = sph_weight_packed_bytes((sph_dtype)dt, kv, d.kdim, d.ndim);
    if (n == 0)
        raise("cannot pack weight of shape (" + std::to_string(kv) + ", " + std::to_string(a) + ", " + std::to_string(b) + ")");
    packed = bytes(n, w);
    d.packed = packed.data_ptr();
    return d;
}

Tensor pack_weight(const Tensor &w, bool transpose, bool reverse, int dt)
{
    const OnDevice here(w);
    Tensor packed;
    const sph_pack_desc d = describe_pack(w, transpose, reverse, dt, packed);
    check(sph_weight_packs(&d, 1, here.stream));
    return packed;
}

// the copies for the forward pass and for dgrad in one launch
std::pair<Tensor, Tensor> pack_weight_both(const Tensor &w, bool reverse, int dt)
{
    const OnDevice here(w);
    Tensor f, t;
    const sph_pack_desc d[2] = {describe_pack(w, false, false, dt, f), describe_pack(w, true, reverse, dt, t)};
    check(sph_weight_packs(d, 2, here.stream));
    return {f, t};
}

// ---- rules --------------------------------------------------------------------------------------
void rules_build(const Tensor &z_idx, const Tensor &z_ptr, const Tensor &oz_idx, const Tensor &oz_ptr, const Geometry &geom,
                 bool transposed, BookBuffers &buf, const OptTensor &row_cols)
{
    const OnDevice here(z_ptr);
    const int in_rows = (int)z_idx.size(0), out_rows = (int)oz_idx.size(0);
    check(sph_rules_build((const int32_t *)z_idx.data_ptr(), (const int32_t *)z_ptr.data_ptr(), in_rows, (const int32_t *)oz_idx.data_ptr(),
                          (const int32_t *)oz_ptr.data_ptr(), out_rows, &geom.g, transposed, &buf.book,
                          row_table(row_cols, transposed ? in_rows : out_rows), here.stream));
}

// ... with one weight (kind 0: as it is; 1: transposed) or both forms (2; reverse: dgrad's offsets mirrored) packed by
// the same launch
py::object rules_build_pack(const Tensor &z_idx, const Tensor &z_ptr, const Tensor &oz_idx, const Tensor &oz_ptr, const Geometry &geom,
                            bool transposed, BookBuffers &buf, const OptTensor &row_cols, const Tensor &weight, int kind, bool reverse,
                            int dt)
{
    const OnDevice here(z_ptr);
    const int in_rows = (int)z_idx.size(0), out_rows = (int)oz_idx.size(0);
    Tensor p[2];
    sph_pack_desc d[2];
    const int n = kind == 2 ? 2 : 1;
    d[0] = describe_pack(weight, kind == 1, false, dt, p[0]);
    if (n == 2) d[1] = describe_pack(weight, true, reverse, dt, p[1]);
    check(sph_rules_build_packs((const int32_t *)z_idx.data_ptr(), (const int32_t *)z_ptr.data_ptr(), in_rows,
                                (const int32_t *)oz_idx.data_ptr(), (const int32_t *)oz_ptr.data_ptr(), out_rows, &geom.g, transposed,
                                &buf.book, row_table(row_cols, transposed ? in_rows : out_rows), d, n, here.stream));
    if (n == 2) return py::make_tuple(p[0], p[1]);
    return py::cast(p[0]);
}

// Output coordinates of a strided layer.  start(): the count is enqueued, and behind it already the
// kernel that writes the coordinates, into arrays of the most rows the layer can reach -- prod ceil(K / stride) per input
// row -- so that the GPU has work while the host learns the row count and enqueues what needs it.  What is handed out is
// then the leading part of arrays that may be several times its size and live as long as it does, so this is done where
// the two arrays hold at most kAheadBytes; beyond, the coordinates are written after the wait, into arrays of their size.
// Two launches, or three (a scan between them) for deep or very large grids and where a stream is being recorded.
struct OutCoords {
    static constexpr double kAheadBytes = 16 << 20;
    Tensor z_idx, z_ptr, oz_ptr, scratch, oz_idx, cols;
    const Geometry *geom;
    py::object geom_owner;
    HostWord total;
    HeldCells cells{total}; // of a count in two launches (destroyed before the word)
    bool two;
    long bound;
    bool filled = false;
    OutCoords(const OnDevice &here, Tensor zi, Tensor zp, py::object g)
        : z_idx(std::move(zi)), z_ptr(std::move(zp)), geom(g.cast<const Geometry *>()), geom_owner(g), total(here)
    {
        const sph_geom &q = geom->g;
        int n = sph_outcoords2_scratch_ints(&q);
        if (n < 0) check(n);
        two = n > 0 && !being_recorded(here.stream) && cells.take(here, z_ptr);
        if (!two) {
            n = sph_outcoords_scratch_ints(&q);
            if (n < 0) check(n);
        }
        oz_ptr = at::empty({q.B, q.O[0], q.O[1]}, z_ptr.options());
        scratch = ints(n + (n & 1) + 2, z_ptr);
        const int rows = (int)z_idx.size(0);
        double most = rows;
        for (int d = 0; d < 3; d++) most *= (q.K[d] + q.stride[d] - 1) / q.stride[d];
        most = std::min(most, (double)q.B * q.O[0] * q.O[1] * q.O[2]);
        if (two) {
            const int32_t *zi = ptr<int32_t>(z_idx), *zp = ptr<int32_t>(z_ptr);
            int32_t *sc = ptr<int32_t>(scratch);
            const int rc = sph_outcoords2_count(zi, zp, rows, &q, sc, cells.get(), total.address(), total.on());
            if (rc != SPH_ERR_ARG) cells.launched(); // (also where a launch is said to have failed: such cells are not handed out again)
            check(rc);
        } else
            check(sph_outcoords_count(ptr<int32_t>(z_idx), ptr<int32_t>(z_ptr), rows, &q, ptr<int32_t>(oz_ptr), ptr<int32_t>(scratch),
                                      total.address(), total.on()));
        if (most * 8 <= kAheadBytes) {
            bound = (long)most;
            fill(here, bound);
        }
    }
    OutCoords(const OutCoords &) = delete;
    OutCoords &operator=(const OutCoords &) = delete;
    // (on the stream of the count, which `here`'s device is that of)
    void fill(const OnDevice &here, long rows)
    {
        oz_idx = ints(rows, z_ptr);
        cols = ints(rows, z_ptr);
        if (two)
            check(sph_outcoords2_fill(&geom->g, ptr<int32_t>(scratch), ptr<int32_t>(oz_ptr), ptr<int32_t>(oz_idx), (int)rows, ptr<int32_t>(cols),
                                      total.on()));
        else
            check(sph_outcoords_fill(ptr<int32_t>(z_idx), ptr<int32_t>(z_ptr), (int)z_idx.size(0), &geom->g, ptr<int32_t>(scratch),
                                     ptr<int32_t>(oz_ptr), ptr<int32_t>(oz_idx), (int)rows, ptr<int32_t>(cols), total.on()));
        filled = true;
    }
    uintptr_t on() const { return (uintptr_t)total.on(); }
    // -> oz_idx, oz_ptr, columns of the output rows; the one wait of a strided layer
    std::tuple<Tensor, Tensor, Tensor> finish()
    {
        const long rows = (long)total.wait(false);
        cells.done();
        if (rows < 0 || (filled && rows > bound)) raise("the output coordinates of a strided layer are inconsistent");
        if (!filled) fill(OnDevice(z_ptr), rows);
        else if (rows < bound) {
            oz_idx = oz_idx.narrow(0, 0, rows);
            cols = cols.narrow(0, 0, rows);
        }
        scratch = Tensor();
        return {oz_idx, oz_ptr, cols};
    }
};

// ---- convolution --------------------------------------------------------------------------------
const sph_epilogue *epilogue(sph_epilogue &e, const OptTensor &scale, const OptTensor &shift, bool relu, int ndim)
{
    for (const OptTensor *t : {&scale, &shift}) // the kernels read one float per output channel
        if (*t && ((*t)->scalar_type() != at::kFloat || (*t)->numel() < ndim))
            raise("scale and shift must be float32 with one value per output channel (" + std::to_string(ndim) + ")");
    e.scale = ptr<const float>(scale);
    e.shift = ptr<const float>(shift);
    e.relu = relu;
    return &e;
}

// the kernels take the rows to be as wide as the weight says
void check_rows(const Tensor &feature, int kdim)
{
    if (feature.dim() != 2 || feature.size(1) != kdim)
        raise("feature [N,iC] / weight [KV,iC,oC] mismatch: iC = " + std::to_string(kdim) + ", rows of " +
              std::to_string(feature.dim() ? feature.size(-1) : 0));
}

Tensor conv_apply(const Tensor &feature_, const Tensor &packed, int kdim, int ndim, BookBuffers &buf, const OptTensor &scale,
                  const OptTensor &shift, bool relu)
{
    check_rows(feature_, kdim);
    const OnDevice here(feature_);
    const Tensor feature = feature_.contiguous();
    const Tensor out = at::empty({buf.book.rows, ndim}, feature.options().requires_grad(false));
    sph_epilogue e;
    check(sph_conv_apply((sph_dtype)dtype_code(feature.scalar_type()), ptr(feature), (int)feature.size(0), kdim, packed.data_ptr(), ndim,
                         &buf.book, epilogue(e, scale, shift, relu, ndim), out.data_ptr(), here.stream));
    return out;
}

// pairs and forward pass in one launch, or None where the library has no such kernel for the call
py::object rules_conv(const Tensor &z_idx, const Tensor &z_ptr, const Tensor &oz_idx, const Tensor &oz_ptr, const Geometry &geom,
                      BookBuffers &buf, int flags, const OptTensor &row_cols, const Tensor &feature_, const Tensor &packed, int kdim,
                      int ndim, const OptTensor &scale, const OptTensor &shift, bool relu)
{
    check_rows(feature_, kdim);
    const OnDevice here(feature_);
    const Tensor feature = feature_.contiguous();
    if (feature.size(0) != z_idx.size(0)) raise("the rows and their coordinates differ in number");
    const int out_rows = (int)oz_idx.size(0);
    const Tensor out = at::empty({out_rows, ndim}, feature.options().requires_grad(false));
    sph_epilogue e;
    const int rc = sph_rules_conv((const int32_t *)z_idx.data_ptr(), (const int32_t *)z_ptr.data_ptr(), (int)z_idx.size(0),
                                  (const int32_t *)oz_idx.data_ptr(), (const int32_t *)oz_ptr.data_ptr(), out_rows, &geom.g, &buf.book,
                                  flags, row_table(row_cols, out_rows), (sph_dtype)dtype_code(feature.scalar_type()), ptr(feature), kdim,
                                  packed.data_ptr(), ndim, epilogue(e, scale, shift, relu, ndim), out.data_ptr(), here.stream);
    if (rc == SPH_ERR_UNSUPPORTED) return py::none();
    check(rc);
    return py::cast(out);
}

Tensor conv_wgrad(const Tensor &feature_, const Tensor &d_out_, BookBuffers &buf, bool transposed, bool f32)
{
    const OnDevice here(feature_);
    const Tensor feature = feature_.contiguous(), d_out = d_out_.contiguous();
    const int ic = (int)feature.size(1), oc = (int)d_out.size(1);
    // the kernel checks the rows that a book's groups gather, and takes those the book is stationary on as given
    if ((transposed ? feature : d_out).size(0) < buf.book.rows) raise("fewer rows than the rule book holds");
    const int64_t n = (int64_t)sph_wgrad_partial_elems(buf.kv, ic, oc, buf.book.rows);
    const Tensor partial = at::empty({n > 0 ? n : 1}, feature.options().dtype(at::kFloat).requires_grad(false));
    const Tensor dw = at::empty({buf.kv, ic, oc}, feature.options().dtype(f32 ? at::kFloat : feature.scalar_type()).requires_grad(false));
    const sph_dtype dt = (sph_dtype)dtype_code(feature.scalar_type());
    if (transposed)
        check(sph_conv_wgrad_transposed(dt, ptr(feature), ic, ptr(d_out), (int)d_out.size(0), oc, &buf.book, (float *)partial.data_ptr(),
                                        dw.data_ptr(), f32, here.stream));
    else
        check(sph_conv_wgrad(dt, ptr(feature), (int)feature.size(0), ic, ptr(d_out), oc, &buf.book, (float *)partial.data_ptr(),
                             dw.data_ptr(), f32, here.stream));
    return dw;
}

// ---- tensors ------------------------------------------------------------------------------------
// -> out feature, z_idx, z_ptr, permutation, row_cols, coordinates outside the grid, duplicated coordinates
py::tuple init_tensor(const Tensor &feature_, const Tensor &indices_, int B, int S0, int S1, int S2)
{
    if (indices_.scalar_type() != at::kInt || indices_.dim() != 2 || indices_.size(1) != 4)
        raise("indices must be int32 [NNZ,4] (b,s0,s1,s2)", PyExc_ValueError);
    if (feature_.dim() != 2 || feature_.size(0) != indices_.size(0)) raise("feature must be [NNZ,C]", PyExc_ValueError);
    const OnDevice here(indices_);
    const Tensor indices = indices_.contiguous(), feature = feature_.contiguous();
    const int n = (int)indices.size(0);
    const size_t nbytes = sph_init_tensor_workspace(n, B, S0, S1, S2);
    if (nbytes == 0)
        raise("bad batch size / spatial shape [" + std::to_string(B) + ", " + std::to_string(S0) + ", " + std::to_string(S1) + ", " +
              std::to_string(S2) + "]");
    Tensor z_idx = ints(n, indices), perm = ints(n, indices), cols = ints(n, indices), status = ints(2, indices);
    Tensor z_ptr = at::empty({B, S0, S1}, indices.options());
    Tensor out = at::empty_like(feature, feature.options().requires_grad(false));
    const Tensor work = bytes(nbytes, indices);
    HostWord word(here);
    check(sph_init_tensor_rows(ptr<int32_t>(indices), n, B, S0, S1, S2, ptr(feature),
                               (int)(feature.size(1) * feature.element_size()), ptr<int32_t>(z_idx), ptr<int32_t>(z_ptr), ptr<int32_t>(perm),
                               ptr<int32_t>(cols), ptr(out), ptr<int32_t>(status), word.address(), ptr(work), nbytes, word.on()));
    const int64_t s = word.wait(true);
    return py::make_tuple(out, z_idx, z_ptr, perm, cols, (int)(int32_t)(s & 0xffffffff), (int)(int32_t)(s >> 32));
}

Tensor to_dense_channels_first(const Tensor &feature_, const Tensor &z_idx, const Tensor &z_ptr, int B, int C, int S0, int S1, int S2)
{
    const OnDevice here(feature_);
    const Tensor feature = feature_.contiguous();
    if (feature.size(1) != C || z_ptr.numel() != (int64_t)B * S0 * S1) raise("rows and pointers do not match the dense shape");
    if (z_idx.scalar_type() != at::kInt || z_ptr.scalar_type() != at::kInt || z_idx.numel() < feature.size(0))
        raise("z_idx and z_ptr must be int32, with an entry of z_idx per row");
    const Tensor out = at::empty({B, C, S0, S1, S2}, feature.options().requires_grad(false));
    check(sph_to_dense_channels_first(ptr(feature), ptr<int32_t>(z_idx), ptr<int32_t>(z_ptr), (int)feature.size(0), B * S0 * S1, S0 * S1,
                                      S2, C, (int)feature.element_size(), out.data_ptr(), here.stream));
    return out;
}

// ---- points -------------------------------------------------------------------------------------
// -> voxels, mask, coordinates, points per voxel, number of voxels
py::tuple points_to_voxel(const Tensor &points, int system, const std::vector<double> &lo, const std::vector<double> &vs,
                          const std::vector<int> &grid, int max_points, int max_voxels, int append_mode, const OptTensor &cells,
                          const OptTensor &cell_out)
{
    const OnDevice here(points);
    const int n = (int)points.size(0), nfeat = (int)points.size(1), width = append_mode == 1 ? nfeat + 3 : nfeat;
    const size_t nbytes = sph_points_to_voxel_workspace(n, grid[0], grid[1], grid[2]);
    if (nbytes == 0)
        raise("bad resolution [" + std::to_string(grid[0]) + ", " + std::to_string(grid[1]) + ", " + std::to_string(grid[2]) +
              "], or more than 2^29 points (" + std::to_string(n) + ")");
    Tensor voxels = at::empty({max_voxels, max_points, width}, points.options());
    Tensor mask = at::empty({max_voxels, max_points, 1}, points.options());
    Tensor coors = at::empty({max_voxels, 3}, points.options().dtype(at::kInt));
    Tensor num = at::empty({max_voxels}, points.options().dtype(at::kInt));
    const Tensor work = bytes(nbytes, points);
    HostWord word(here);
    check(sph_points_to_voxel(n ? ptr<float>(points) : nullptr, n, nfeat, system, (float)lo[0], (float)lo[1], (float)lo[2], (float)vs[0],
                              (float)vs[1], (float)vs[2], grid[0], grid[1], grid[2], max_points, max_voxels, append_mode,
                              ptr<float>(voxels), ptr<float>(mask), ptr<int32_t>(coors), ptr<int32_t>(num), word.address(),
                              ptr<const long long>(cells), ptr<long long>(cell_out), ptr(work), nbytes, word.on()));
    return py::make_tuple(voxels, mask, coors, num, (int)word.wait(false));
}

Tensor voxel_mean(const Tensor &voxels, const Tensor &num, int nf)
{
    const OnDevice here(voxels);
    const Tensor out = at::empty({voxels.size(0), nf}, voxels.options());
    check(sph_voxel_mean(ptr<float>(voxels), ptr<int32_t>(num), (int)voxels.size(0), (int)voxels.size(1), (int)voxels.size(2), nf,
                         (float *)out.data_ptr(), here.stream));
    return out;
}

Tensor batch_coordinates(const std::vector<Tensor> &parts)
{
    if (parts.empty()) raise("no coordinates to join");
    const OnDevice here(parts[0]);
    std::vector<const int32_t *> p;
    std::vector<int32_t> rows;
    int64_t total = 0;
    for (auto &t : parts) {
        p.push_back(ptr<const int32_t>(t));
        rows.push_back((int32_t)t.size(0));
        total += t.size(0);
    }
    const Tensor out = at::empty({total, 4}, parts[0].options());
    check(sph_batch_coordinates(p.data(), rows.data(), (int)parts.size(), (int32_t *)out.data_ptr(), here.stream));
    return out;
}

} // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("set_error", [](py::object e) { Py_XINCREF(e.ptr()); g_error = e.ptr(); });
    m.def("abi_version", []() { return sph_abi_version(); });
    py::class_<Geometry>(m, "Geometry")
        .def(py::init<int, const std::vector<int> &, const std::vector<int> &, const std::vector<int> &, const std::vector<int> &,
                      const std::vector<int> &, const std::vector<int> &>())
        .def("takes", &Geometry::takes)
        .def_property_readonly("address", &Geometry::address);
    py::class_<BookBuffers>(m, "BookBuffers")
        .def(py::init([](int rows, int kv, py::object dev, bool by_row, bool groups) {
            return new BookBuffers(rows, kv, py::cast<c10::Device>(dev), by_row, groups);
        }))
        .def_readonly("storage", &BookBuffers::storage)
        .def_readonly("ntiles", &BookBuffers::ntiles)
        .def_readonly("cap", &BookBuffers::cap)
        .def_property("rows", [](const BookBuffers &b) { return b.book.rows; },
                      [](BookBuffers &b, int rows) {
                          if (rows < 0 || rows > b.rows) raise("a book does not grow");
                          b.book.rows = rows;
                      })
        .def_property("middle_run", [](const BookBuffers &b) { return b.book.middle_run; }, [](BookBuffers &b, int v) { b.book.middle_run = v; })
        .def_property_readonly("address", &BookBuffers::address)
        .def("range", [](const BookBuffers &b, int i) { return std::make_pair(b.off[i], b.size[i]); });
    py::class_<OutCoords>(m, "OutCoords")
        .def(py::init([](Tensor z_idx, Tensor z_ptr, py::object geometry) {
            const OnDevice here(z_ptr);
            return new OutCoords(here, std::move(z_idx), std::move(z_ptr), std::move(geometry));
        }))
        .def_property_readonly("stream", &OutCoords::on)
        .def("finish", &OutCoords::finish);
    m.def("pack_weight", &pack_weight);
    m.def("pack_weight_both", &pack_weight_both);
    m.def("rules_build", &rules_build);
    m.def("rules_build_pack", &rules_build_pack);
    m.def("conv_apply", &conv_apply);
    m.def("rules_conv", &rules_conv);
    m.def("conv_wgrad", &conv_wgrad);
    m.def("init_tensor", &init_tensor);
    m.def("to_dense_channels_first", &to_dense_channels_first);
    m.def("points_to_voxel", &points_to_voxel);
    m.def("voxel_mean", &voxel_mean);
    m.def("batch_coordinates", &batch_coordinates);
}
