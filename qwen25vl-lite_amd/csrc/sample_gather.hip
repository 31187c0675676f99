// Host code: the settings of a sampler call's rows, from the requests' Python objects into the block of 32-bit words that goes to
// the device.  A loop over 64 requests and 3,100 generated ids in Python takes longer than the sampler's kernels (90 us on the host of
// an MI355X for 64 requests, this 12).  Whatever is not the usual kind (settings that are no numbers, ids in
// other containers than lists and tuples or other than Python's integers) is left to the caller's Python.
#include <Python.h>

#include <cstdint>
#include <cstring>

namespace {

struct Row {                    // as the sampler's kernels read it
  float temperature, top_p, min_p, u, repetition, presence, frequency;
  int32_t top_k, prev_begin, prev_end;
  uint32_t seed;
  int32_t seeded;
};
constexpr long ROW_WORDS = sizeof(Row) / 4;

PyObject* name_of(int i) {
  static const char* const names[] = {"temperature", "top_p", "min_p", "repetition_penalty", "presence_penalty", "frequency_penalty",
                                      "top_k", "seed"};
  static PyObject* interned[8] = {};      // made once, under the interpreter's lock
  if (!interned[i]) interned[i] = PyUnicode_InternFromString(names[i]);
  return interned[i];
}
bool number(PyObject* object, int name, double& out) {
  PyObject* key = name_of(name);
  PyObject* v = key ? PyObject_GetAttr(object, key) : nullptr;
  if (!v) return false;
  const bool ok = PyFloat_CheckExact(v) || PyLong_CheckExact(v);
  if (ok) out = PyFloat_AsDouble(v);
  Py_DECREF(v);
  return ok && !PyErr_Occurred();
}
// 0: no such integer, 1: one, 2: None
int integer(PyObject* v, long long& out) {
  if (v == Py_None) return 2;
  if (!PyLong_CheckExact(v)) return 0;
  int over = 0;
  out = PyLong_AsLongLongAndOverflow(v, &over);
  return over || PyErr_Occurred() ? 0 : 1;
}
int integer_of(PyObject* object, int name, long long& out) {
  PyObject* key = name_of(name);
  PyObject* v = key ? PyObject_GetAttr(object, key) : nullptr;
  if (!v) return 0;
  const int kind = integer(v, out);
  Py_DECREF(v);
  return kind;
}
// Numbers from 0 to 2^30 - 1 have one digit at most, which this interpreter's header shows.
bool one_digit(PyObject* v, long& out) {
#if PY_VERSION_HEX < 0x030C0000
  const Py_ssize_t digits = Py_SIZE(v);
  out = digits ? (long)reinterpret_cast<PyLongObject*>(v)->ob_digit[0] : 0;
  return digits == 0 || digits == 1;
#else
  (void)v;
  (void)out;
  return false;
#endif
}
bool items(PyObject* s) { return PyList_CheckExact(s) || PyTuple_CheckExact(s); }

long gather(PyObject* params, PyObject* prev, PyObject* steps, long M, long vocab, int32_t* out, long room, int32_t* flags,
            int32_t* more) {
  if (!items(params) || !items(prev) || !items(steps)) return -1;
  if (M * ROW_WORDS + 1 > room) return -(M * ROW_WORDS + 1);
  Row* rows = reinterpret_cast<Row*>(out);
  int32_t* ids = out + M * ROW_WORDS;
  const long id_room = room - M * ROW_WORDS;
  long count = 0;
  bool draws = false, scores = false, top_k = false, top_p = false, cut = false, whole = false;
  int32_t unseeded = 0;
  for (long i = 0; i < M; ++i) {
    if (PySequence_Fast_GET_SIZE(params) != M || PySequence_Fast_GET_SIZE(prev) != M || PySequence_Fast_GET_SIZE(steps) != M) return -1;
    PyObject* p = PySequence_Fast_GET_ITEM(params, i);
    Py_INCREF(p);
    double v[6];
    bool ok = true;
    for (int a = 0; a < 6 && ok; ++a) ok = number(p, a, v[a]);
    long long k = 0, seed = 0;
    ok = ok && integer_of(p, 6, k) == 1 && k >= INT32_MIN && k <= INT32_MAX;
    const int seed_kind = ok ? integer_of(p, 7, seed) : 0;
    Py_DECREF(p);
    if (!ok || seed_kind == 0) return -1;
    Row& r = rows[i];
    r.temperature = (float)v[0];
    r.top_p = (float)v[1];
    r.min_p = (float)v[2];
    r.u = 0.f;
    r.repetition = (float)v[3];
    r.presence = (float)v[4];
    r.frequency = (float)v[5];
    r.top_k = k ? (int32_t)k : -1;
    r.seed = 0;
    r.seeded = 0;
    r.prev_begin = (int32_t)count;
    if (v[0] > 0 && seed_kind == 2 && more) {
      r.seeded = -1;        // the caller's to fill in
      ++unseeded;
    } else if (v[0] > 0) {
      // the generator's seed: the request's and the number of its tokens
      if (PySequence_Fast_GET_SIZE(steps) != M) return -1;
      long long step = 0;
      if (seed_kind != 1 || integer(PySequence_Fast_GET_ITEM(steps, i), step) != 1) return -1;
      if (seed < -(1ll << 61) || seed > (1ll << 61) || step < 0 || step > (1ll << 60)) return -1;
      r.seed = (uint32_t)(uint64_t)(seed + step);
      r.seeded = 1;
    }
    if (v[3] != 1.0 || v[4] != 0.0 || v[5] != 0.0) {
      if (PySequence_Fast_GET_SIZE(prev) != M) return -1;
      PyObject* tokens = PySequence_Fast_GET_ITEM(prev, i);
      if (!items(tokens)) return -1;
      const long n = PySequence_Fast_GET_SIZE(tokens);
      PyObject** item = PySequence_Fast_ITEMS(tokens);
      if (count + n > (1l << 30)) return -1;
      for (long j = 0; j < n; ++j) {        // (no other code runs meanwhile: the items are whole numbers or the loop ends)
        if (!PyLong_CheckExact(item[j])) return -1;
        long t;
        if (!one_digit(item[j], t)) {
          int over = 0;
          t = PyLong_AsLongAndOverflow(item[j], &over);
          if (over || t < INT32_MIN || t > INT32_MAX) return -1;
        }
        if (count + j < id_room) ids[count + j] = (int32_t)t;
      }
      count += n;
    }
    r.prev_end = (int32_t)count;
    if (r.temperature > 0.f) {
      draws = true;
      scores |= r.prev_end > r.prev_begin;
      const bool k_cut = r.top_k > 0 && r.top_k < vocab, p_cut = r.top_p < 1.f, any = k_cut || p_cut || r.min_p > 0.f;
      top_k |= k_cut;
      top_p |= p_cut;
      cut |= any;
      whole |= !any;
    }
  }
  if (count > id_room) return -(M * ROW_WORDS + count);
  if (count == 0) ids[count++] = 0;
  flags[0] = draws;
  flags[1] = scores;
  flags[2] = top_k;
  flags[3] = top_p;
  if (more) {
    more[0] = cut;
    more[1] = whole;
    more[2] = unseeded;
  }
  return M * ROW_WORDS + count;
}

}  // namespace

// Called with the interpreter's lock held.  out: `room` 32-bit words: M rows, then the generated ids of rows with penalties (one zero
// if there are none).  flags: whether any row draws, draws with ids, cuts by top-k, by top-p; more (or null): draws
// with any cut, with none, and how many draw without a seed (`seeded` is -1 in these; without `more` they are not taken).  Returns the words written;
// -1: not taken; -n below that: n words are needed.  No exception is left behind.
extern "C" long qvl_sample_gather(PyObject* params, PyObject* prev, PyObject* steps, long M, long vocab, void* out, long room, void* flags,
                                  void* more) {
  const long n = M < 1 ? -1 : gather(params, prev, steps, M, vocab, (int32_t*)out, room, (int32_t*)flags, (int32_t*)more);
  if (PyErr_Occurred()) PyErr_Clear();
  return n;
}
