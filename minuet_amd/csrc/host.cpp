// The host side of a layer call, as a Python extension module.
//
// A layer of a network is one or two kernel launches of 5 to 30 us, and a
// launch costs the host about 3 us.  Written in Python, everything around
// them (checks, cache lookups, the output tensor, a ctypes call of 17 to 29
// arguments) took 15 to 25 us more per layer, which left the GPU waiting in
// every network but the largest.  This module does the same work in about
// 2 us: a Layer holds what depends on the module alone (weights, their packed
// copy, widths, tunables), a MapEntry what depends on the kernel map, and
// Layer.run checks that both still describe the call at hand.  Whatever is
// not exactly as it was when the two were made sends the caller (None is
// returned) through the Python code that makes them.
//
// Every entry point that touches a tensor stands between HANDLE_TH_ERRORS and
// END_HANDLE_TH_ERRORS: what torch throws (no memory left, a tensor without
// storage) reaches the caller as the Python exception it is, and no further.
// What such a function owns meanwhile it holds in a Ref.
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPEvent.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdint>
#include <memory>

namespace {

// ------------------------------------------------------- the library's calls ----

using ImplicitFn = int (*)(const void *, const void *, const int32_t *, int64_t, int64_t, int64_t, int64_t, int64_t,
                           int, const float *, const float *, const void *, int, float, const void *, void *, void *);
using GroupsFn = int (*)(const void *, const void *, const int32_t *, const int32_t *, const int32_t *,
                         const int32_t *, int64_t, int64_t, int64_t, int64_t, int, const float *, const float *,
                         const void *, int, float, void *, void *);
using TablesFn = int (*)(int64_t, int64_t, int, int64_t, int, double, const void *, const void *, const void *,
                         const void *, const void *, const void *, const int64_t *, int64_t, int64_t, int64_t,
                         int64_t, int64_t, int, int, const int32_t *, const float *, const float *, const void *,
                         int, float, const void *, const int64_t *, void *, void *);
using TiledFn = int (*)(const void *, const void *, const int32_t *, int64_t, int64_t, int64_t, int64_t, int64_t, int,
                        const float *, const float *, const void *, int, float, void *, void *);
using PiecesFn = int (*)(const void *, const void *, int64_t, int64_t, int64_t, int64_t, const float *, const float *,
                         const void *, int, float, void *, void *);
using PadFn = int (*)(const void *, int64_t, int64_t, int64_t, int, void *, void *);
using TilesFn = int (*)(const int32_t *, int64_t, int64_t, int32_t *, void *);
using TilesSizeFn = int (*)(int64_t, int64_t, int64_t *);
using TilesShareFn = double (*)(int64_t, int64_t, int64_t, int64_t, int);
using ErrorFn = const char *(*)();

ImplicitFn g_implicit = nullptr;
GroupsFn g_groups = nullptr;
TablesFn g_tables = nullptr;
TiledFn g_tiled = nullptr;
PiecesFn g_pieces = nullptr;
TiledFn g_single = nullptr;
PadFn g_pad = nullptr;
TilesFn g_tiles = nullptr;
TilesSizeFn g_tiles_size = nullptr;
TilesShareFn g_tiles_share = nullptr;
ErrorFn g_error = nullptr;

// ------------------------------------------------------------ Python objects ----

// What the Python side hands over once (bind): classes and modules' dicts.
PyTypeObject *g_sparse_tensor = nullptr;          // minuet_amd.SparseTensor
PyObject *g_conv_types = nullptr;                 // tuple of the exact convolution classes
PyObject *g_norm_types = nullptr;                 // tuple of the exact BatchNorm classes
PyObject *g_activations = nullptr;                // dict: exact activation class -> activation code
PyObject *g_global_hooks = nullptr;               // tuple of torch's global module hook dicts
PyObject *g_conv_namespace = nullptr;             // dict of minuet_amd.nn.convolutions.SparseConv at bind time
PyObject *g_forward = nullptr;                    // SparseConv.forward at bind time
PyObject *g_no_arguments = nullptr;               // an empty tuple

#define MNT_NAMES(X)                                                                                        \
  X(_features) X(_coordinates) X(_stride) X(_batch_dims) X(_parameters) X(_buffers) X(kernel) X(bias)        \
  X(_kernel_map_cache) X(_tunable_config) X(_tuning_data) X(stride) X(dilation) X(kernel_size) X(_fast)      \
  X(_fast_maps) X(dataflow) X(threshold) X(gather_tile_size) X(scatter_tile_size) X(scale) X(shift)          \
  X(residual) X(activation) X(negative_slope) X(_forward_hooks) X(_forward_pre_hooks) X(_backward_hooks)     \
  X(_backward_pre_hooks) X(_compiled_call_impl) X(forward) X(training) X(weight) X(running_mean)             \
  X(running_var) X(eps) X(_minuet_affine) X(_identity_map) X(relu) X(leaky_relu) X(relu6)
#define MNT_DECLARE(name) PyObject *s_##name = nullptr;
MNT_NAMES(MNT_DECLARE)
#undef MNT_DECLARE

// The instance dictionary of an object (borrowed), or null.
inline PyObject *dict_of(PyObject *object) {
  PyObject **at = _PyObject_GetDictPtr(object);
  return at == nullptr ? nullptr : *at;
}

// Borrowed lookup; null when the key is missing (no exception set).
inline PyObject *look(PyObject *dict, PyObject *key) { return PyDict_GetItem(dict, key); }

// An owned reference.
struct Ref {
  PyObject *object;
  explicit Ref(PyObject *o = nullptr) : object(o) {}
  Ref(const Ref &) = delete;
  Ref &operator=(const Ref &) = delete;
  ~Ref() { Py_XDECREF(object); }
  PyObject *release() {
    PyObject *o = object;
    object = nullptr;
    return o;
  }
};

inline bool is_none(PyObject *o) { return o == nullptr || o == Py_None; }

inline const at::Tensor *tensor_of(PyObject *o) {
  return o != nullptr && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}

inline int64_t version_of(const at::Tensor &t) {
  return t.is_inference() ? -1 : static_cast<int64_t>(t.unsafeGetTensorImpl()->version_counter().current_version());
}

// A tensor that derived data was made from: unchanged while the object under
// its name is the same one, with the same storage and version counter.
struct Watched {
  PyObject *object = nullptr;      // owned
  const void *data = nullptr;
  int64_t version = 0;

  void set(PyObject *o) {
    if (const at::Tensor *t = tensor_of(o)) {
      data = t->const_data_ptr();
      version = version_of(*t);
    }
    Py_XINCREF(o);
    Py_XDECREF(object);
    object = o;
  }
  bool same(PyObject *o) const {
    if (o != object) return false;
    const at::Tensor *t = tensor_of(o);
    return t == nullptr || (t->const_data_ptr() == data && version_of(*t) == version);
  }
  void clear() { Py_CLEAR(object); }
};

// --------------------------------------------------------------- MapEntry ----

enum Kind { kImplicit = 0, kGroups = 1, kTables = 2, kPointwise = 3, kPieces = 4 };

// One kernel map as one kind of layer reads it: the coordinates its output
// carries and the device addresses of its tables (`keep` holds their owners).
struct MapEntry {
  PyObject_HEAD
  PyObject *coordinates, *stride, *batch_dims, *keep;
  int kind;
  int device;
  int index_code;
  int64_t num_sources, num_targets;
  const void *at[8];       // kind's own pointers, in the order of the entry point's arguments
  // Of a map built ahead of the layer that asks for it: the source coordinates
  // it was built from (null: the cache serves it to whoever asks), and whether
  // any layer has used it.
  const void *built_from;
  char used;
  // Tiles of the map (kind kImplicit; null until they are made) and what they
  // would have saved so far, over what making them takes (below 0: never).
  PyObject *tiles;
  double tiles_credit;
  double tiles_saved;      // what they saved or would have saved all the layers that have run
  // The stream that makes the tiles, the end of that work, and whether the host
  // has seen it ended.
  void *tiles_stream;
  at::cuda::CUDAEvent *tiles_made;
  char tiles_ready;
};

void map_entry_dealloc(PyObject *self) {
  MapEntry *e = reinterpret_cast<MapEntry *>(self);
  Py_XDECREF(e->coordinates);
  Py_XDECREF(e->stride);
  Py_XDECREF(e->batch_dims);
  Py_XDECREF(e->keep);
  Py_XDECREF(e->tiles);
  delete e->tiles_made;
  Py_TYPE(self)->tp_free(self);
}

PyObject *hold(PyObject *o) {
  Py_INCREF(o);
  return o;
}

void swap_in(PyObject *&held, PyObject *o) {
  PyObject *before = held;
  held = hold(o);
  Py_XDECREF(before);
}

// Tiles that the current stream of the map's device has made; false with a
// Python error.
bool take_tiles(MapEntry *e, PyObject *tiles) {
  if (tensor_of(tiles) == nullptr) {
    PyErr_SetString(PyExc_TypeError, "tiles are a tensor");
    return false;
  }
  try {
    const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(e->device));
    std::unique_ptr<at::cuda::CUDAEvent> made(new at::cuda::CUDAEvent());
    made->record(c10::hip::HIPStreamMasqueradingAsCUDA(stream));
    e->tiles_stream = stream.stream();
    e->tiles_made = made.release();
  } catch (const std::exception &error) {
    PyErr_SetString(PyExc_RuntimeError, error.what());
    return false;
  }
  e->tiles = hold(tiles);
  return true;
}

struct MapArgs {
  PyObject *coordinates, *stride, *batch_dims, *keep, *tiles;
  int kind, device, index_code;
  long long num_sources, num_targets;
  unsigned long long built_from;
  const void *at[8];
};

bool parse_map(PyObject *args, MapArgs *a) {
  PyObject *pointers;
  a->built_from = 0;
  a->tiles = Py_None;                         // those the current stream of `device` has made already
  if (!PyArg_ParseTuple(args, "iOOOOiiLLO!|KO", &a->kind, &a->coordinates, &a->stride, &a->batch_dims, &a->keep,
                        &a->device, &a->index_code, &a->num_sources, &a->num_targets, &PyTuple_Type, &pointers,
                        &a->built_from, &a->tiles)) {
    return false;
  }
  for (Py_ssize_t i = 0; i < 8; ++i) {
    a->at[i] = nullptr;
    if (i < PyTuple_GET_SIZE(pointers) && !is_none(PyTuple_GET_ITEM(pointers, i))) {
      a->at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(pointers, i));
    }
  }
  return PyErr_Occurred() == nullptr;
}

PyObject *map_entry_new(PyTypeObject *type, PyObject *args, PyObject *) {
  MapArgs a;
  if (!parse_map(args, &a)) return nullptr;
  MapEntry *e = reinterpret_cast<MapEntry *>(type->tp_alloc(type, 0));       // (all zeros)
  if (e == nullptr) return nullptr;
  e->coordinates = hold(a.coordinates);
  e->stride = hold(a.stride);
  e->batch_dims = hold(a.batch_dims);
  e->keep = hold(a.keep);
  e->kind = a.kind;
  e->device = a.device;
  e->index_code = a.index_code;
  e->num_sources = a.num_sources;
  e->num_targets = a.num_targets;
  e->built_from = reinterpret_cast<const void *>(static_cast<uintptr_t>(a.built_from));
  std::copy(a.at, a.at + 8, e->at);
  if (a.tiles != Py_None && !take_tiles(e, a.tiles)) {
    Py_DECREF(e);
    return nullptr;
  }
  return reinterpret_cast<PyObject *>(e);
}

// renew(the constructor's arguments): this entry as the constructor would make
// it, but with its tiles and what is known about them; False, and nothing done,
// where it is of another map.
PyObject *map_entry_renew(PyObject *self, PyObject *args) {
  MapEntry *e = reinterpret_cast<MapEntry *>(self);
  MapArgs a;
  if (!parse_map(args, &a)) return nullptr;
  if (e->kind != a.kind || e->device != a.device || e->index_code != a.index_code ||
      e->num_sources != a.num_sources || e->num_targets != a.num_targets || !std::equal(a.at, a.at + 8, e->at)) {
    Py_RETURN_FALSE;
  }
  if (a.tiles != Py_None && e->tiles == nullptr && !take_tiles(e, a.tiles)) return nullptr;
  swap_in(e->coordinates, a.coordinates);
  swap_in(e->stride, a.stride);
  swap_in(e->batch_dims, a.batch_dims);
  swap_in(e->keep, a.keep);
  e->built_from = reinterpret_cast<const void *>(static_cast<uintptr_t>(a.built_from));
  Py_RETURN_TRUE;
}

// tiles_of(address, stream): the tiles of the map at that address, if this entry
// has them and that stream made them.
PyObject *map_entry_tiles_of(PyObject *self, PyObject *args) {
  MapEntry *e = reinterpret_cast<MapEntry *>(self);
  unsigned long long address, stream;
  if (!PyArg_ParseTuple(args, "KK", &address, &stream)) return nullptr;
  if (e->tiles == nullptr || reinterpret_cast<uintptr_t>(e->at[0]) != address ||
      reinterpret_cast<uintptr_t>(e->tiles_stream) != stream) {
    Py_RETURN_NONE;
  }
  return hold(e->tiles);
}

PyObject *py_reduce(PyObject *, PyObject *);

PyMethodDef map_entry_methods[] = {{"__reduce__", py_reduce, METH_NOARGS, "Copies as None."},
                                   {"renew", map_entry_renew, METH_VARARGS, "Describes the same map anew."},
                                   {"tiles_of", map_entry_tiles_of, METH_VARARGS, "The tiles a stream has made."},
                                   {nullptr, nullptr, 0, nullptr}};

PyObject *map_entry_used(PyObject *self, void *) {
  return PyBool_FromLong(reinterpret_cast<MapEntry *>(self)->used);
}

PyObject *map_entry_tiles_saved(PyObject *self, void *) {
  return PyFloat_FromDouble(reinterpret_cast<MapEntry *>(self)->tiles_saved);
}

PyGetSetDef map_entry_getset[] = {{"used", map_entry_used, nullptr, "Whether a layer has run with this map.", nullptr},
                                  {"tiles_saved", map_entry_tiles_saved, nullptr,
                                   "What tiles saved, or would have saved, the layers that ran with this map, over "
                                   "what making them takes.", nullptr},
                                  {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject MapEntryType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ------------------------------------------------------------------ Layer ----

// A convolution module as it was when its last call went through the Python code.
struct Layer {
  PyObject_HEAD
  Watched kernel, bias;
  PyObject *weights, *packed;                 // what is multiplied by (padded where rows are), its packed copy
  PyObject *stride, *dilation, *kernel_size;  // the module's settings, by identity
  PyObject *shape_id;                         // key of this layer's map inside the cache's _fast_maps
  PyObject *dataflow, *threshold, *gather_tile, *scatter_tile;
  int kind, float_code, device;
  int shortcut, has_threshold;
  double threshold_value;
  int64_t gather_tile_value, scatter_tile_value;
  int64_t num_offsets, in_channels, out_channels;
  int64_t item_size;
  // The source rows for which this kind is the one to take, and a Layer of the
  // module for others, if it has run on such a cloud, which names the next (null,
  // and 0 to the most there are, where the choice does not depend on rows).
  int64_t rows_from, rows_to;
  PyObject *other;
};

// Layers that a module keeps: a kind may be the one to take over several ranges
// of rows (an fp32 layer multiplies hits, writes product rows, multiplies hits
// again and, where features are past 32-bit offsets, writes product rows).
constexpr int kMostLayers = 4;

void layer_dealloc(PyObject *self) {
  Layer *l = reinterpret_cast<Layer *>(self);
  l->kernel.clear();
  l->bias.clear();
  for (PyObject **o : {&l->weights, &l->packed, &l->stride, &l->dilation, &l->kernel_size, &l->shape_id,
                       &l->dataflow, &l->threshold, &l->gather_tile, &l->scatter_tile, &l->other}) {
    Py_CLEAR(*o);
  }
  Py_TYPE(self)->tp_free(self);
}

PyTypeObject LayerType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// Layer(module, kind, weights, packed, shape_id, shortcut, rows_from, rows_to, other);
// shortcut: of kind TABLES whether the centre offset may take one, of kind
// IMPLICIT whether a target of the map has one source, of kind PIECES whether
// autocast has a say (the layer would be torch.mm otherwise)
PyObject *layer_new(PyTypeObject *type, PyObject *args, PyObject *) {
  HANDLE_TH_ERRORS
  PyObject *module, *weights, *packed, *shape_id;
  PyObject *other = Py_None;
  int kind, shortcut;
  long long rows_from = 0, rows_to = INT64_MAX;
  if (!PyArg_ParseTuple(args, "OiOOOi|LLO", &module, &kind, &weights, &packed, &shape_id, &shortcut, &rows_from,
                        &rows_to, &other)) {
    return nullptr;
  }
  PyObject *d = dict_of(module);
  const at::Tensor *w = tensor_of(weights);
  PyObject *parameters = d == nullptr ? nullptr : look(d, s__parameters);
  PyObject *config = d == nullptr ? nullptr : look(d, s__tunable_config);
  // (a pruned, normalised or parametrised kernel or bias is no parameter of the
  // module but made anew from others: nothing here would see it change)
  if (parameters == nullptr || config == nullptr || w == nullptr || w->dim() != 3 || tensor_of(packed) == nullptr ||
      !w->is_contiguous() || tensor_of(look(parameters, s_kernel)) == nullptr || look(parameters, s_bias) == nullptr) {
    PyErr_SetString(PyExc_ValueError, "Layer needs a convolution module whose kernel and bias are its own parameters, "
                                      "its weights and their packed copy");
    return nullptr;
  }
  Ref made(type->tp_alloc(type, 0));
  if (made.object == nullptr) return nullptr;
  Layer *l = reinterpret_cast<Layer *>(made.object);
  new (&l->kernel) Watched();
  new (&l->bias) Watched();
  l->kernel.set(look(parameters, s_kernel));
  l->bias.set(look(parameters, s_bias));
  auto hold = [](PyObject *o) {
    o = o == nullptr ? Py_None : o;
    Py_INCREF(o);
    return o;
  };
  l->weights = hold(weights);
  l->packed = hold(packed);
  l->stride = hold(look(d, s_stride));
  l->dilation = hold(look(d, s_dilation));
  l->kernel_size = hold(look(d, s_kernel_size));
  l->shape_id = hold(shape_id);
  l->dataflow = hold(look(config, s_dataflow));
  l->threshold = hold(look(config, s_threshold));
  l->gather_tile = hold(look(config, s_gather_tile_size));
  l->scatter_tile = hold(look(config, s_scatter_tile_size));
  l->rows_from = rows_from;
  l->rows_to = rows_to;
  l->kind = kind;
  l->shortcut = shortcut;
  l->device = w->device().index();
  l->float_code = w->scalar_type() == at::kFloat ? 0 : w->scalar_type() == at::kHalf ? 1 : 2;
  l->item_size = static_cast<int64_t>(w->element_size());
  l->num_offsets = w->size(0);
  l->in_channels = w->size(1);
  l->out_channels = w->size(2);
  l->has_threshold = l->threshold == Py_None ? 0 : 1;
  l->threshold_value = l->has_threshold ? PyFloat_AsDouble(l->threshold) : 0.0;
  l->gather_tile_value = l->gather_tile == Py_None ? 0 : PyLong_AsLongLong(l->gather_tile);
  l->scatter_tile_value = l->scatter_tile == Py_None ? 0 : PyLong_AsLongLong(l->scatter_tile);
  if (PyErr_Occurred()) return nullptr;
  // the module's Layers so far: those for other rows stay, the latest first
  Layer *last = l;
  PyObject *next = Py_TYPE(other) == &LayerType ? hold(other) : nullptr;
  for (int count = 1; next != nullptr && count < kMostLayers;) {
    const Ref before(next);
    Layer *b = reinterpret_cast<Layer *>(next);
    next = b->other;                                     // (taken from it)
    b->other = nullptr;
    if (b->rows_to < l->rows_from || b->rows_from > l->rows_to) {
      last->other = hold(before.object);
      last = b;
      ++count;
    }
  }
  Py_XDECREF(next);
  return made.release();
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------- runs ----

struct EpilogueArgs {
  PyObject *scale = nullptr, *shift = nullptr, *residual = nullptr;
  int activation = 0;
  float slope = 0.0f;
};

// fp32 [channels] on `device`, contiguous: the form the kernels read.
inline bool vector_fits(const at::Tensor *t, int64_t channels, int device) {
  return t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == channels && t->is_contiguous() &&
         t->is_cuda() && t->device().index() == device;
}

// The tiles of a layer's map, or null where the layer runs without.  Tiles cost
// one or more forwards to make and are kept with the map.  A wide layer, which
// loses half its time without, makes them at once (a share of kTilesCredit); the
// others' are made once
// the forwards that have run over it would have saved twice their price: a map
// that a network reads a few times and drops does not pay for them there (a
// pass that is built ahead makes them for less, from what the pass before it
// would have saved), one that is read on and on soon does.  Layers of all widths and types share a map, so
// whether this one can use tiles (a share of 0: it cannot) is asked first.
constexpr double kTilesCredit = 2.0;
constexpr int64_t kTilesMostInts = int64_t{1} << 29;

bool make_tiles(MapEntry *map, const Layer *l, int64_t T, const at::Device &device, const c10::hip::HIPStream &stream) {
  int64_t ints = 0;
  if (g_tiles_size(T, l->num_offsets, &ints) != 0 || ints > kTilesMostInts) return false;
  at::Tensor tiles;
  try {
    tiles = at::detail::empty_cuda({ints}, at::kInt, device, std::nullopt);
  } catch (const std::exception &) {                     // no room: the layer runs without
    return false;
  }
  if (g_tiles(static_cast<const int32_t *>(map->at[0]), T, l->num_offsets,
              static_cast<int32_t *>(tiles.mutable_data_ptr()), stream.stream()) != 0) {
    return false;
  }
  std::unique_ptr<at::cuda::CUDAEvent> made(new at::cuda::CUDAEvent());
  made->record(c10::hip::HIPStreamMasqueradingAsCUDA(stream));
  map->tiles = THPVariable_Wrap(std::move(tiles));
  if (map->tiles == nullptr) {
    PyErr_Clear();
    return false;
  }
  map->tiles_stream = stream.stream();
  map->tiles_made = made.release();
  return true;
}

// A call on the stream that makes the tiles comes after that work by itself.
// One on another stream takes them once the host has seen the work ended: the
// two streams owe each other nothing because of tiles, which no caller asked
// for and none can wait for, and until then the layer without them gives the
// same rows.  (The event is not asked during a capture, which forbids it.)  The
// allocator is told of the other stream, which may still read the tiles when
// the cache has dropped them.
const at::Tensor *tiles_of(MapEntry *map, const Layer *l, int64_t T, const at::Device &device,
                           const c10::hip::HIPStream &stream) {
  const double share = g_tiles_share(T, l->num_offsets, l->in_channels, l->out_channels, l->float_code);
  if (share == 0.0) return nullptr;
  map->tiles_saved += share;
  if (map->tiles == nullptr) {
    if (map->tiles_credit < 0.0) return nullptr;
    map->tiles_credit += share;
    if (map->tiles_credit < kTilesCredit) return nullptr;
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return nullptr;
    map->tiles_credit = -1.0;
    if (!make_tiles(map, l, T, device, stream)) return nullptr;
  }
  const at::Tensor *tiles = tensor_of(map->tiles);
  if (map->tiles_stream == stream.stream()) return tiles;
  if (map->tiles_ready == 0) {
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return nullptr;
    if (!map->tiles_made->query()) return nullptr;
    map->tiles_ready = 1;
  }
  tiles->record_stream(c10::hip::HIPStreamMasqueradingAsCUDA(stream));
  return tiles;
}

PyObject *none() { Py_RETURN_NONE; }

// Whether nothing but the operand's value counts (plain in _C.py): it is of no
// class of its own, records no gradient, carries no tangent and wraps nothing.
bool plain(PyObject *o) {
  if (is_none(o)) return true;
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor &t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet kWrapped{c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Python};
  return !t.key_set().has_any(kWrapped) && !(c10::GradMode::is_enabled() && t.requires_grad()) &&
         !t._fw_grad(/*level=*/0).defined();
}

// A 1 x 1 x 1 layer has derivatives, batching rules and a trace through
// torch.mm: whether it may go past that, for these operands and here.
bool stands_in(const Layer *l, PyObject *features, const EpilogueArgs &ep) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::tracer::impl::is_dispatch_enabled() ||
      (l->kind == kPieces && l->shortcut != 0 && at::autocast::is_autocast_enabled(at::kCUDA))) {
    return false;
  }
  for (PyObject *o : {features, l->kernel.object, l->bias.object, ep.scale, ep.shift, ep.residual}) {
    if (!plain(o)) return false;
  }
  return true;
}

// The layer on `inputs`; None when anything is not as the Layer describes it.
PyObject *run_layer(Layer *l, PyObject *module_dict, PyObject *inputs, const EpilogueArgs &ep) {
  // the one of the module's Layers that is for so many rows
  if (Py_TYPE(inputs) != g_sparse_tensor) return none();
  PyObject *in = dict_of(inputs);
  const at::Tensor *x = in == nullptr ? nullptr : tensor_of(look(in, s__features));
  if (x == nullptr || x->dim() != 2) return none();
  const int64_t S = x->size(0);
  while (S < l->rows_from || S > l->rows_to) {
    if (l->other == nullptr) return none();
    l = reinterpret_cast<Layer *>(l->other);
  }
  Py_INCREF(l);
  const Ref keep(reinterpret_cast<PyObject *>(l));
  if ((l->kind == kPointwise || l->kind == kPieces) && !stands_in(l, look(in, s__features), ep)) return none();
  // the module: same parameters, same settings, not being tuned
  PyObject *parameters = look(module_dict, s__parameters);
  PyObject *config = look(module_dict, s__tunable_config);
  if (parameters == nullptr || config == nullptr || !l->kernel.same(look(parameters, s_kernel)) ||
      !l->bias.same(look(parameters, s_bias)) || look(module_dict, s_stride) != l->stride ||
      look(module_dict, s_dilation) != l->dilation || look(module_dict, s_kernel_size) != l->kernel_size ||
      look(config, s_dataflow) != l->dataflow || look(config, s_threshold) != l->threshold ||
      look(config, s_gather_tile_size) != l->gather_tile || look(config, s_scatter_tile_size) != l->scatter_tile ||
      !is_none(look(module_dict, s__tuning_data))) {
    return none();
  }
  const at::Tensor &kernel = THPVariable_Unpack(l->kernel.object);
  if (c10::GradMode::is_enabled()) {
    const at::Tensor *b = tensor_of(l->bias.object);
    if (kernel.requires_grad() || (b != nullptr && b->requires_grad())) return none();
  }
  // the input
  PyObject *coordinates = look(in, s__coordinates), *stride = look(in, s__stride);
  PyObject *batch_dims = look(in, s__batch_dims);
  if (coordinates == nullptr || stride == nullptr || batch_dims == nullptr) return none();
  // (rows that the layer pads have the kernel's channels, its weights the padded row's)
  const int64_t channels = l->kind == kImplicit ? kernel.size(1) : l->in_channels;
  if (x->size(1) != channels || x->scalar_type() != kernel.scalar_type() || !x->is_cuda() ||
      x->device().index() != l->device || !x->is_contiguous() || (c10::GradMode::is_enabled() && x->requires_grad())) {
    return none();
  }
  const void *source = x->const_data_ptr();
  if (reinterpret_cast<uintptr_t>(source) % 16 != 0 || c10::hip::current_device() != l->device) return none();
  // its kernel map
  PyObject *out_coordinates = coordinates, *out_stride = stride, *out_batch_dims = batch_dims;
  int64_t T = S;
  MapEntry *map = nullptr;
  const at::Tensor *identity = nullptr;
  if (l->kind == kPointwise || l->kind == kPieces) {
    // 1 x 1 x 1: every row is its own source
    if (l->kind == kPointwise) {
      identity = tensor_of(look(module_dict, s__identity_map));
      if (identity == nullptr || identity->dim() != 2 || identity->size(1) < S || identity->device() != x->device()) {
        return none();
      }
    }
    if (batch_dims != Py_None) {
      const at::Tensor *dims = tensor_of(batch_dims);
      if (dims == nullptr || dims->dim() != 1 || dims->size(0) <= 2) return none();
    }
  } else {
    PyObject *cache = look(module_dict, s__kernel_map_cache);
    PyObject *cache_dict = is_none(cache) ? nullptr : dict_of(cache);
    PyObject *maps = cache_dict == nullptr ? nullptr : look(cache_dict, s__fast_maps);
    PyObject *by_stride = maps == nullptr ? nullptr : look(maps, l->shape_id);
    PyObject *found = by_stride == nullptr ? nullptr : look(by_stride, stride);
    if (found == nullptr || Py_TYPE(found) != &MapEntryType) return none();
    map = reinterpret_cast<MapEntry *>(found);
    if (map->kind != l->kind || map->num_sources != S || map->device != l->device) return none();
    if (map->built_from != nullptr) {
      const at::Tensor *rows = tensor_of(coordinates);
      if (rows == nullptr || rows->const_data_ptr() != map->built_from) return none();
    }
    map->used = 1;
    T = map->num_targets;
    out_coordinates = map->coordinates;
    out_stride = map->stride;
    out_batch_dims = map->batch_dims;
  }
  // the epilogue; a bias is one more per-channel shift where there is none yet
  const at::Tensor *scale = nullptr, *shift = nullptr, *residual = nullptr;
  if (!is_none(ep.scale)) {
    scale = tensor_of(ep.scale);
    if (scale == nullptr || !vector_fits(scale, l->out_channels, l->device)) return none();
  }
  at::Tensor bias;
  if (!is_none(l->bias.object)) {
    if (!is_none(ep.scale) || !is_none(ep.shift)) return none();
    // (read at every call: a write through .data leaves no mark on the parameter)
    bias = THPVariable_Unpack(l->bias.object);
    if (bias.scalar_type() != at::kFloat) bias = bias.to(at::kFloat);
    shift = &bias;
  } else if (!is_none(ep.shift)) {
    shift = tensor_of(ep.shift);
  }
  if (shift != nullptr || !is_none(ep.shift)) {
    if (shift == nullptr || !vector_fits(shift, l->out_channels, l->device)) return none();
  }
  if (!is_none(ep.residual)) {
    residual = tensor_of(ep.residual);
    if (residual == nullptr || residual->scalar_type() != kernel.scalar_type() || residual->dim() != 2 ||
        residual->size(0) != T || residual->size(1) != l->out_channels || !residual->is_contiguous() ||
        !residual->is_cuda() || residual->device().index() != l->device ||
        reinterpret_cast<uintptr_t>(residual->const_data_ptr()) % 16 != 0) {
      return none();
    }
  }
  at::Tensor out = at::detail::empty_cuda({T, l->out_channels}, kernel.scalar_type(), kernel.device(), std::nullopt);
  const c10::hip::HIPStream current = c10::hip::getCurrentHIPStream(l->device);
  void *stream = current.stream();
  auto data = [](const at::Tensor *t) -> const void * { return t == nullptr ? nullptr : t->const_data_ptr(); };
  const float *scale_at = static_cast<const float *>(data(scale));
  const float *shift_at = static_cast<const float *>(data(shift));
  const void *weights_at = THPVariable_Unpack(l->weights).const_data_ptr();
  const void *packed_at = THPVariable_Unpack(l->packed).const_data_ptr();
  int status = 0;
  at::Tensor padded;
  if (channels != l->in_channels) {
    padded = at::detail::empty_cuda({S, l->in_channels}, kernel.scalar_type(), kernel.device(), std::nullopt);
    // (of 32-bit values as of twice as many of 16 bits)
    const int halves = l->item_size == 4 ? 2 : 1;
    status = g_pad(source, S, halves * channels, halves * l->in_channels, halves == 2 ? 1 : l->float_code,
                   padded.mutable_data_ptr(), stream);
    if (status != 0) {
      PyErr_SetString(PyExc_RuntimeError, g_error());
      return nullptr;
    }
    source = padded.const_data_ptr();
  }
  switch (l->kind) {
    case kImplicit:
      if (l->shortcut != 0) {                              // a target has one source
        status = g_single(source, packed_at, static_cast<const int32_t *>(map->at[0]), S, T, l->num_offsets,
                          l->in_channels, l->out_channels, l->float_code, scale_at, shift_at, data(residual),
                          ep.activation, ep.slope, out.mutable_data_ptr(), stream);
        break;
      }
      if (const at::Tensor *tiles = tiles_of(map, l, T, kernel.device(), current)) {
        status = g_tiled(source, packed_at, static_cast<const int32_t *>(tiles->const_data_ptr()), S, T,
                         l->num_offsets, l->in_channels, l->out_channels, l->float_code, scale_at, shift_at,
                         data(residual), ep.activation, ep.slope, out.mutable_data_ptr(), stream);
        break;
      }
      status = g_implicit(source, weights_at, static_cast<const int32_t *>(map->at[0]), S, T, l->num_offsets,
                          l->in_channels, l->out_channels, l->float_code, scale_at, shift_at, data(residual),
                          ep.activation, ep.slope, packed_at, out.mutable_data_ptr(), stream);
      break;
    case kGroups:
      status = g_groups(source, packed_at, static_cast<const int32_t *>(map->at[0]),
                        static_cast<const int32_t *>(map->at[1]), static_cast<const int32_t *>(map->at[2]),
                        static_cast<const int32_t *>(map->at[3]), S, T, l->in_channels, l->out_channels,
                        l->float_code, scale_at, shift_at, data(residual), ep.activation, ep.slope,
                        out.mutable_data_ptr(), stream);
      break;
    case kTables:
      // source_masks, target_masks, order, sizes, sizes on the host, order on the host, pair list
      status = g_tables(l->gather_tile_value, l->scatter_tile_value, l->shortcut, 4, l->has_threshold,
                        l->threshold_value, source, weights_at, map->at[0], map->at[1], map->at[2], map->at[3],
                        static_cast<const int64_t *>(map->at[4]), S, T, l->num_offsets, l->in_channels,
                        l->out_channels, map->index_code, l->float_code, static_cast<const int32_t *>(map->at[6]),
                        scale_at, shift_at, data(residual), ep.activation, ep.slope, packed_at,
                        static_cast<const int64_t *>(map->at[5]), out.mutable_data_ptr(), stream);
      break;
    case kPieces: {
      // the input channels in pieces, which the wavefronts of a workgroup share
      const int64_t pieces = THPVariable_Unpack(l->packed).size(0);
      status = g_pieces(source, weights_at, S, pieces, l->in_channels / pieces, l->out_channels, scale_at, shift_at,
                        data(residual), ep.activation, ep.slope, out.mutable_data_ptr(), stream);
      break;
    }
    default:
      status = g_implicit(source, weights_at, static_cast<const int32_t *>(identity->const_data_ptr()), S, T, 1,
                          l->in_channels, l->out_channels, l->float_code, scale_at, shift_at, data(residual),
                          ep.activation, ep.slope, packed_at, out.mutable_data_ptr(), stream);
      break;
  }
  if (status != 0) {
    PyErr_SetString(PyExc_RuntimeError, g_error());
    return nullptr;
  }
  // the result: a SparseTensor like the ones SparseTensor.like makes
  Ref result(g_sparse_tensor->tp_new(g_sparse_tensor, g_no_arguments, nullptr));
  if (result.object == nullptr) return nullptr;
  const Ref features(THPVariable_Wrap(std::move(out)));
  const bool ok = features.object != nullptr && PyObject_SetAttr(result.object, s__features, features.object) == 0 &&
                  PyObject_SetAttr(result.object, s__coordinates, out_coordinates) == 0 &&
                  PyObject_SetAttr(result.object, s__stride, out_stride) == 0 &&
                  PyObject_SetAttr(result.object, s__batch_dims, out_batch_dims) == 0;
  return ok ? result.release() : nullptr;
}

// The Layer a module keeps, or null.
Layer *layer_of(PyObject *module_dict) {
  PyObject *fast = look(module_dict, s__fast);
  return fast != nullptr && Py_TYPE(fast) == &LayerType ? reinterpret_cast<Layer *>(fast) : nullptr;
}

int activation_code(PyObject *name) {
  if (is_none(name)) return 0;
  if (name == s_relu) return 1;
  if (name == s_leaky_relu) return 2;
  if (name == s_relu6) return 3;
  if (!PyUnicode_Check(name)) return -1;
  if (PyUnicode_Compare(name, s_relu) == 0) return 1;
  if (PyUnicode_Compare(name, s_leaky_relu) == 0) return 2;
  if (PyUnicode_Compare(name, s_relu6) == 0) return 3;
  return -1;
}

// run(module, inputs, epilogue): the module's forward, or None.
PyObject *py_run(PyObject *, PyObject *const *args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 3) {
    PyErr_SetString(PyExc_TypeError, "run(module, inputs, epilogue)");
    return nullptr;
  }
  PyObject *d = dict_of(args[0]);
  Layer *l = d == nullptr ? nullptr : layer_of(d);
  if (l == nullptr) return none();
  EpilogueArgs ep;
  Ref held[5];
  if (args[2] != Py_None) {
    PyObject *names[5] = {s_scale, s_shift, s_residual, s_activation, s_negative_slope};
    for (int i = 0; i < 5; ++i) {
      held[i].object = PyObject_GetAttr(args[2], names[i]);
      if (held[i].object == nullptr) return nullptr;
    }
    ep.scale = held[0].object;
    ep.shift = held[1].object;
    ep.residual = held[2].object;
    ep.activation = activation_code(held[3].object);
    ep.slope = static_cast<float>(PyFloat_AsDouble(held[4].object));
    if (PyErr_Occurred()) return nullptr;
  }
  if (ep.activation < 0) return none();
  return run_layer(l, d, args[1], ep);
  END_HANDLE_TH_ERRORS
}

// ----------------------------------------------------------------- Affine ----

// scale and shift of a BatchNorm in evaluation mode, and the tensors they were made from.
struct Affine {
  PyObject_HEAD
  Watched mean, var, weight, bias;
  PyObject *eps;
  PyObject *scale, *shift;
};

void affine_dealloc(PyObject *self) {
  Affine *a = reinterpret_cast<Affine *>(self);
  for (Watched *w : {&a->mean, &a->var, &a->weight, &a->bias}) w->clear();
  Py_CLEAR(a->eps);
  Py_CLEAR(a->scale);
  Py_CLEAR(a->shift);
  Py_TYPE(self)->tp_free(self);
}

// Affine(norm, scale, shift)
PyObject *affine_new(PyTypeObject *type, PyObject *args, PyObject *) {
  HANDLE_TH_ERRORS
  PyObject *norm, *scale, *shift;
  if (!PyArg_ParseTuple(args, "OOO", &norm, &scale, &shift)) return nullptr;
  PyObject *d = dict_of(norm);
  PyObject *buffers = d == nullptr ? nullptr : look(d, s__buffers);
  PyObject *parameters = d == nullptr ? nullptr : look(d, s__parameters);
  if (buffers == nullptr || parameters == nullptr) {
    PyErr_SetString(PyExc_ValueError, "Affine needs a module with buffers and parameters");
    return nullptr;
  }
  Ref made(type->tp_alloc(type, 0));
  if (made.object == nullptr) return nullptr;
  Affine *a = reinterpret_cast<Affine *>(made.object);
  for (Watched *w : {&a->mean, &a->var, &a->weight, &a->bias}) new (w) Watched();
  a->mean.set(look(buffers, s_running_mean));
  a->var.set(look(buffers, s_running_var));
  a->weight.set(look(parameters, s_weight));
  a->bias.set(look(parameters, s_bias));
  PyObject *eps = look(d, s_eps);
  a->eps = eps == nullptr ? Py_None : eps;
  a->scale = scale;
  a->shift = shift;
  Py_INCREF(a->eps);
  Py_INCREF(scale);
  Py_INCREF(shift);
  return made.release();
  END_HANDLE_TH_ERRORS
}

PyTypeObject AffineType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// The valid Affine of a BatchNorm module in evaluation mode, or null.
Affine *affine_of(PyObject *norm) {
  PyObject *d = dict_of(norm);
  if (d == nullptr || look(d, s_training) != Py_False) return nullptr;
  PyObject *kept = look(d, s__minuet_affine);
  PyObject *buffers = look(d, s__buffers), *parameters = look(d, s__parameters);
  if (kept == nullptr || !PyTuple_Check(kept) || buffers == nullptr || parameters == nullptr) return nullptr;
  PyObject *last = PyTuple_GET_ITEM(kept, PyTuple_GET_SIZE(kept) - 1);
  if (Py_TYPE(last) != &AffineType) return nullptr;
  Affine *a = reinterpret_cast<Affine *>(last);
  return a->mean.same(look(buffers, s_running_mean)) && a->var.same(look(buffers, s_running_var)) &&
                 a->weight.same(look(parameters, s_weight)) && a->bias.same(look(parameters, s_bias)) &&
                 look(d, s_eps) == a->eps
             ? a
             : nullptr;
}

inline bool exact_type_in(PyObject *object, PyObject *types) {
  PyObject *type = reinterpret_cast<PyObject *>(Py_TYPE(object));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(types); ++i) {
    if (PyTuple_GET_ITEM(types, i) == type) return true;
  }
  return false;
}

inline bool empty_dict(PyObject *d) { return d == nullptr || (PyDict_Check(d) && PyDict_GET_SIZE(d) == 0); }

// conv_norm_act(conv, norm, act, x, residual): conv -> norm -> (+ residual) ->
// act as one call of the library, or None.  The module is called around
// torch's Module.__call__, so it must be one whose call is its forward alone:
// no hooks on it, none global, nothing overridden.
PyObject *py_conv_norm_act(PyObject *, PyObject *const *args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 5) {
    PyErr_SetString(PyExc_TypeError, "conv_norm_act(conv, norm, act, x, residual)");
    return nullptr;
  }
  PyObject *conv = args[0], *norm = args[1], *act = args[2];
  if (!exact_type_in(conv, g_conv_types)) return none();
  PyObject *d = dict_of(conv);
  Layer *l = d == nullptr ? nullptr : layer_of(d);
  if (l == nullptr) return none();
  if (!empty_dict(look(d, s__forward_hooks)) || !empty_dict(look(d, s__forward_pre_hooks)) ||
      !empty_dict(look(d, s__backward_hooks)) || !empty_dict(look(d, s__backward_pre_hooks)) ||
      !is_none(look(d, s__compiled_call_impl)) || look(d, s_forward) != nullptr ||
      look(g_conv_namespace, s_forward) != g_forward) {
    return none();
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(g_global_hooks); ++i) {
    if (!empty_dict(PyTuple_GET_ITEM(g_global_hooks, i))) return none();
  }
  EpilogueArgs ep;
  if (norm != Py_None) {
    if (!exact_type_in(norm, g_norm_types)) return none();
    Affine *a = affine_of(norm);
    if (a == nullptr) return none();
    ep.scale = a->scale;
    ep.shift = a->shift;
  }
  if (act != Py_None) {
    PyObject *code = look(g_activations, reinterpret_cast<PyObject *>(Py_TYPE(act)));
    if (code == nullptr) return none();
    ep.activation = static_cast<int>(PyLong_AsLong(code));
    if (ep.activation == 2) {
      PyObject *ad = dict_of(act);
      PyObject *slope = ad == nullptr ? nullptr : look(ad, s_negative_slope);
      if (slope == nullptr || !PyFloat_Check(slope)) return none();
      ep.slope = static_cast<float>(PyFloat_AS_DOUBLE(slope));
    }
  }
  ep.residual = args[4];
  return run_layer(l, d, args[3], ep);
  END_HANDLE_TH_ERRORS
}

// bind(addresses: dict name -> int, sparse_tensor, conv_types, norm_types, activations, global_hooks)
PyObject *py_bind(PyObject *, PyObject *args) {
  PyObject *addresses, *sparse_tensor, *conv_types, *norm_types, *activations, *hooks;
  if (!PyArg_ParseTuple(args, "O!O!O!O!O!O!", &PyDict_Type, &addresses, &PyType_Type, &sparse_tensor, &PyTuple_Type,
                        &conv_types, &PyTuple_Type, &norm_types, &PyDict_Type, &activations, &PyTuple_Type, &hooks)) {
    return nullptr;
  }
  auto address = [&](const char *name) -> void * {
    PyObject *value = PyDict_GetItemString(addresses, name);
    if (value == nullptr) {
      PyErr_Format(PyExc_KeyError, "no address for %s", name);
      return nullptr;
    }
    return PyLong_AsVoidPtr(value);
  };
  g_implicit = reinterpret_cast<ImplicitFn>(address("mnt_sparse_convolution_forward_implicit"));
  g_groups = reinterpret_cast<GroupsFn>(address("mnt_sparse_convolution_forward_groups"));
  g_tables = reinterpret_cast<TablesFn>(address("mnt_sparse_convolution_forward_fused"));
  g_tiled = reinterpret_cast<TiledFn>(address("mnt_sparse_convolution_forward_tiled"));
  g_pieces = reinterpret_cast<PiecesFn>(address("mnt_sparse_convolution_forward_pieces"));
  g_single = reinterpret_cast<TiledFn>(address("mnt_sparse_convolution_forward_single"));
  g_pad = reinterpret_cast<PadFn>(address("mnt_pad_rows"));
  g_tiles = reinterpret_cast<TilesFn>(address("mnt_kernel_map_tiles"));
  g_tiles_size = reinterpret_cast<TilesSizeFn>(address("mnt_kernel_map_tiles_size"));
  g_tiles_share = reinterpret_cast<TilesShareFn>(address("mnt_kernel_map_tiles_share"));
  g_error = reinterpret_cast<ErrorFn>(address("mnt_last_error"));
  if (PyErr_Occurred()) return nullptr;
  g_sparse_tensor = reinterpret_cast<PyTypeObject *>(sparse_tensor);
  g_conv_types = conv_types;
  g_norm_types = norm_types;
  g_activations = activations;
  g_global_hooks = hooks;
  for (PyObject *o : {sparse_tensor, conv_types, norm_types, activations, hooks}) Py_INCREF(o);
  PyTypeObject *base = reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(conv_types, 0));
  g_conv_namespace = base->tp_dict;
  g_forward = look(g_conv_namespace, s_forward);
  Py_XINCREF(g_forward);
  Py_RETURN_NONE;
}

// A copied or unpickled module keeps None in the place of these objects and
// makes its own at its first call.
PyObject *py_reduce(PyObject *, PyObject *) {
  return Py_BuildValue("(O())", reinterpret_cast<PyObject *>(Py_TYPE(Py_None)));
}

PyMethodDef object_methods[] = {{"__reduce__", py_reduce, METH_NOARGS, "Copies as None."},
                                {nullptr, nullptr, 0, nullptr}};

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, "Takes the library's addresses and the package's classes."},
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_run)), METH_FASTCALL,
     "run(module, inputs, epilogue) -> SparseTensor, or None where the Python code has to look."},
    {"conv_norm_act", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_conv_norm_act)), METH_FASTCALL,
     "conv_norm_act(conv, norm, act, x, residual) -> SparseTensor, or None where the Python code has to look."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "minuet_host", "Host side of layer calls.", -1, methods};

bool ready(PyTypeObject &type, const char *name, size_t size, destructor dealloc, newfunc make) {
  type.tp_name = name;
  type.tp_basicsize = static_cast<Py_ssize_t>(size);
  type.tp_flags = Py_TPFLAGS_DEFAULT;
  type.tp_dealloc = dealloc;
  type.tp_new = make;
  if (type.tp_methods == nullptr) type.tp_methods = object_methods;
  return PyType_Ready(&type) == 0;
}

}  // namespace

PyMODINIT_FUNC PyInit_minuet_host() {
#define MNT_INTERN(name) s_##name = PyUnicode_InternFromString(#name);
  MNT_NAMES(MNT_INTERN)
#undef MNT_INTERN
  MapEntryType.tp_getset = map_entry_getset;
  MapEntryType.tp_methods = map_entry_methods;
  if (!ready(MapEntryType, "minuet_host.MapEntry", sizeof(MapEntry), map_entry_dealloc, map_entry_new) ||
      !ready(LayerType, "minuet_host.Layer", sizeof(Layer), layer_dealloc, layer_new) ||
      !ready(AffineType, "minuet_host.Affine", sizeof(Affine), affine_dealloc, affine_new)) {
    return nullptr;
  }
  g_no_arguments = PyTuple_New(0);
  PyObject *module = PyModule_Create(&module_def);
  if (module == nullptr) return nullptr;
  Py_INCREF(&MapEntryType);
  Py_INCREF(&LayerType);
  Py_INCREF(&AffineType);
  PyModule_AddObject(module, "MapEntry", reinterpret_cast<PyObject *>(&MapEntryType));
  PyModule_AddObject(module, "Layer", reinterpret_cast<PyObject *>(&LayerType));
  PyModule_AddObject(module, "Affine", reinterpret_cast<PyObject *>(&AffineType));
  PyModule_AddIntConstant(module, "IMPLICIT", kImplicit);
  PyModule_AddIntConstant(module, "GROUPS", kGroups);
  PyModule_AddIntConstant(module, "TABLES", kTables);
  PyModule_AddIntConstant(module, "POINTWISE", kPointwise);
  PyModule_AddIntConstant(module, "PIECES", kPieces);
  return module;
}
