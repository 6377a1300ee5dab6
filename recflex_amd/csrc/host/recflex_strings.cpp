// The text front end on Python's own strings: sample lines of every feature (lists of str) -> packed
// buffer, without joining and encoding them first (a thousand features of 64 lines, 3.7 MB of text: 1.5
// of the call's 2.8 ms).  Python's objects are only read, through macros that touch memory and need no
// symbol of the interpreter; the caller holds the interpreter's lock for the call, so nothing changes
// them, and the threads that share the work live within it.  What is not plain (other containers,
// strings that are not ASCII, line ends inside a line, numbers beyond int32) is left to the caller's
// other path, which also knows the errors.
#define PY_SSIZE_T_CLEAN
#ifndef NDEBUG
#define NDEBUG
#endif
#include <Python.h>

#include "recflex_hip.h"

#include <atomic>
#include <cstring>
#include <thread>

namespace {

constexpr int NOT_PLAIN = 1;

// The str at place `line` of a list or tuple, or null.
struct Text { const char *at; int64_t len; };
inline bool text_of(PyObject *lines, Py_ssize_t line, Text *t) {
  PyObject *s = PyList_Check(lines) ? PyList_GET_ITEM(lines, line) : PyTuple_GET_ITEM(lines, line);
  if (!s || !PyUnicode_Check(s) || !PyUnicode_IS_READY(s) || !PyUnicode_IS_COMPACT_ASCII(s)) return false;
  t->at = static_cast<const char *>(static_cast<void *>(reinterpret_cast<PyASCIIObject *>(s) + 1));
  t->len = reinterpret_cast<PyASCIIObject *>(s)->length;
  return true;
}

inline PyObject *item(PyObject *seq, Py_ssize_t i) {
  return PyList_Check(seq) ? PyList_GET_ITEM(seq, i) : PyTuple_GET_ITEM(seq, i);
}
inline Py_ssize_t size_of(PyObject *seq) {         // -1: neither a list nor a tuple
  if (!seq) return -1;
  return PyList_Check(seq) ? PyList_GET_SIZE(seq) : (PyTuple_Check(seq) ? PyTuple_GET_SIZE(seq) : -1);
}

inline uint64_t load8(const char *p) {
  uint64_t w;
  std::memcpy(&w, p, 8);
  return w;
}
// bit 7 of every byte that is no digit; w has ASCII bytes only
inline uint64_t not_digits(uint64_t w) {
  return ((w ^ 0x3030303030303030ull) + 0x7676767676767676ull) & 0x8080808080808080ull;
}

// indices of a line: one per separator and one for what comes last, none in an empty line
int64_t count_line(const Text &t) {
  int64_t n = t.len > 0, i = 0;
  for (; i + 8 <= t.len; i += 8) n += __builtin_popcountll(not_digits(load8(t.at + i)));
  for (; i < t.len; ++i) n += t.at[i] < '0' || t.at[i] > '9';
  return n;
}

// The indices of a line to out[0 .. n); false: not plain, or another number of them.
bool parse_line(const Text &t, int32_t *out, int64_t n) {
  const char *p = t.at, *const end = p + t.len;
  int64_t at = 0;
  // numbers of up to seven digits and their separator, eight bytes at a time
  while (end - p >= 8) {
    const uint64_t w = load8(p), stops = not_digits(w);
    if (stops == 0) break;
    const int digits = __builtin_ctzll(stops) >> 3;
    if (p[digits] == '\n' || at >= n) return false;
    uint32_t value = 0;
    if (digits > 0) {
      uint64_t d = (w ^ 0x3030303030303030ull) << (64 - 8 * digits);    // the first digits read 0
      d = (d * 10 + (d >> 8)) & 0x00ff00ff00ff00ffull;
      d = (d * 100 + (d >> 16)) & 0x0000ffff0000ffffull;
      value = static_cast<uint32_t>(d * 10000 + (d >> 32));
    }
    out[at++] = static_cast<int32_t>(value);
    p += digits + 1;
  }
  int64_t value = 0;
  for (; p < end; ++p) {
    if (*p >= '0' && *p <= '9') {
      value = value * 10 + (*p - '0');
      if (value > INT32_MAX) return false;
      continue;
    }
    if (*p == '\n' || at >= n) return false;
    out[at++] = static_cast<int32_t>(value);
    value = 0;
  }
  if (t.len > 0) {
    if (at >= n) return false;
    out[at++] = static_cast<int32_t>(value);
  }
  return at == n;
}

// body(f) for every feature, on a few threads that live for the call, this one among them; one for every 4 096
// lines (a thread takes some 20 us to start, a line some 50 ns to find and read)
template <typename Body> void for_all_features(int32_t num_features, int64_t lines, Body body) {
  constexpr int kMaxThreads = 8;
  constexpr int64_t kLinesPerThread = 4096;
  int64_t want = 1 + lines / kLinesPerThread;
  const int64_t cpus = static_cast<int64_t>(std::thread::hardware_concurrency());
  if (want > kMaxThreads) want = kMaxThreads;
  if (want > cpus) want = cpus > 0 ? cpus : 1;
  std::atomic<int32_t> next(0);
  auto work = [&]() {
    for (int32_t f; (f = next.fetch_add(8, std::memory_order_relaxed)) < num_features;)
      for (int32_t g = f; g < f + 8 && g < num_features; ++g) body(g);
  };
  std::thread others[kMaxThreads];
  int started = 0;
  try {
    for (; started < want - 1; ++started) others[started] = std::thread(work);
  } catch (...) {
    // no more threads to be had: those that run share the work
  }
  work();
  for (int t = 0; t < started; ++t) others[t].join();
}

} // namespace

extern "C" {

// The interpreter whose objects this was built to read: PY_MAJOR_VERSION * 256 + PY_MINOR_VERSION, and 65536
// more where objects begin with the links of Py_TRACE_REFS.
int recom_host_strings_python() {
#ifdef Py_TRACE_REFS
  constexpr int links = 65536;
#else
  constexpr int links = 0;
#endif
  return links + PY_MAJOR_VERSION * 256 + PY_MINOR_VERSION;
}

// raw: num_features lists (or tuples) of `batch` str each, in one.  num_indices_out[f]: the indices
// of feature f.  0, or 1 where something is not plain.
int recom_host_count_strings(void *raw, int32_t num_features, int32_t batch, int64_t *num_indices_out) {
  PyObject *features = static_cast<PyObject *>(raw);
  if (num_features < 0 || batch < 0 || !num_indices_out || size_of(features) != num_features) return NOT_PLAIN;
  std::atomic<bool> plain(true);
  for_all_features(num_features, static_cast<int64_t>(num_features) * batch, [&](int32_t f) {
    PyObject *lines = item(features, f);
    int64_t n = 0;
    Text t;
    bool ok = size_of(lines) == batch;
    for (int32_t b = 0; ok && b < batch; ++b) {
      ok = text_of(lines, b, &t);
      if (ok) n += count_line(t);
    }
    if (!ok || n > INT32_MAX) plain.store(false, std::memory_order_relaxed);
    num_indices_out[f] = n;
  });
  return plain.load() ? 0 : NOT_PLAIN;
}

// The same lines into a packed buffer (recom_host_pack's layout) of the size that num_indices asks for;
// byte_offsets_out[num_features + 1].  0, 1 where something is not plain or no longer as it was counted.
int recom_host_parse_strings(void *raw, int32_t num_features, int32_t batch, const int64_t *num_indices, void *dst,
                             int64_t dst_capacity, int64_t *byte_offsets_out) {
  PyObject *features = static_cast<PyObject *>(raw);
  if (num_features < 0 || batch < 0 || !num_indices || !dst || !byte_offsets_out ||
      size_of(features) != num_features)
    return NOT_PLAIN;
  byte_offsets_out[0] = 0;
  for (int32_t f = 0; f < num_features; ++f)
    byte_offsets_out[f + 1] = byte_offsets_out[f] + recom_host_packed_size(batch, num_indices[f]);
  if (byte_offsets_out[num_features] > dst_capacity) return NOT_PLAIN;
  const int64_t off_bytes = (static_cast<int64_t>(batch) + 1) * 4, off_pad = recom_host_alignmem(off_bytes);
  std::atomic<bool> plain(true);
  for_all_features(num_features, static_cast<int64_t>(num_features) * batch, [&](int32_t f) {
    PyObject *lines = item(features, f);
    char *out = static_cast<char *>(dst) + byte_offsets_out[f];
    int32_t *offsets = reinterpret_cast<int32_t *>(out), *indices = reinterpret_cast<int32_t *>(out + off_pad);
    const int64_t total = num_indices[f];
    int64_t n = 0;
    Text t;
    bool ok = size_of(lines) == batch;
    offsets[0] = 0;
    for (int32_t b = 0; ok && b < batch; ++b) {
      ok = text_of(lines, b, &t);
      if (!ok) break;
      const int64_t here = count_line(t);
      ok = here <= total - n && parse_line(t, indices + n, here);
      n += here;
      offsets[b + 1] = static_cast<int32_t>(n);
    }
    if (!ok || n != total) {
      plain.store(false, std::memory_order_relaxed);
      return;
    }
    std::memset(out + off_bytes, 0, off_pad - off_bytes);
    std::memset(out + off_pad + n * 4, 0, recom_host_alignmem(n * 4) - n * 4);
  });
  return plain.load() ? 0 : NOT_PLAIN;
}

} // extern "C"
