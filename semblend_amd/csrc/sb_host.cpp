// Host conversion of Python index lists (libsemblend_host.so, called through ctypes.PyDLL with
// the GIL held). The callers hold positions and (source, target) pairs as Python lists; walking
// them in Python costs 0.1 us or more per number (1.1 ms for the 8192 pairs of an 8K-token
// permutation, whose launches take 0.35 ms), here about 5 ns.
//
// Only exact lists of exact ints (or of 2-tuples / 2-lists of them) are taken; for anything else
// the functions return -1 without an exception set, and the caller converts in Python, which
// also raises its errors.

#include <Python.h>

#include <cstdint>
#include <limits>
#include <new>
#include <vector>

namespace {

// The value of an exact int within [lo, hi]; false otherwise.
bool exact_int(PyObject* o, int64_t lo, int64_t hi, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || v < lo || v > hi) return false;
  *out = v;
  return true;
}

constexpr int64_t kI32Min = std::numeric_limits<int32_t>::min();
constexpr int64_t kI32Max = std::numeric_limits<int32_t>::max();

}  // namespace

// The interpreter ABI (sysconfig's SOABI) this library was built for. It reads list, tuple and int
// objects through that interpreter's macros, so the loader compares it before any other call.
#ifndef SB_HOST_SOABI
#error "SB_HOST_SOABI must name the interpreter ABI"
#endif
extern "C" const char* sb_host_soabi() { return SB_HOST_SOABI; }

// first[i], second[i] of the n pairs of `pairs`. Returns n, or -1.
extern "C" int64_t sb_host_pairs(PyObject* pairs, int64_t n, int32_t* first, int32_t* second) {
  if (!PyList_CheckExact(pairs) || PyList_GET_SIZE(pairs) != n) return -1;
  for (int64_t i = 0; i < n; ++i) {
    PyObject* p = PyList_GET_ITEM(pairs, i);
    PyObject *a, *b;
    if (PyTuple_CheckExact(p) && PyTuple_GET_SIZE(p) == 2) {
      a = PyTuple_GET_ITEM(p, 0);
      b = PyTuple_GET_ITEM(p, 1);
    } else if (PyList_CheckExact(p) && PyList_GET_SIZE(p) == 2) {
      a = PyList_GET_ITEM(p, 0);
      b = PyList_GET_ITEM(p, 1);
    } else {
      return -1;
    }
    int64_t x, y;
    if (!exact_int(a, kI32Min, kI32Max, &x) || !exact_int(b, kI32Min, kI32Max, &y)) return -1;
    first[i] = static_cast<int32_t>(x);
    second[i] = static_cast<int32_t>(y);
  }
  return n;
}

// The distinct logical positions of `positions` (n entries) in order of first occurrence, and
// how often each occurs: positions whose block lies past the table are skipped, negative ones
// count blocks from the end of the table. keys / counts hold up to n entries, *num_keys of them
// filled. Returns the number of positions processed, or -1 (also where a block lies before the
// table's start, which the caller reports).
extern "C" int64_t sb_host_rotation_counts(PyObject* positions, int64_t n, int64_t block_size,
                                           int64_t num_blocks, int32_t* keys, int32_t* counts,
                                           int64_t* num_keys) {
  if (!PyList_CheckExact(positions) || PyList_GET_SIZE(positions) != n) return -1;
  if (block_size <= 0 || num_blocks < 0 || num_blocks > kI32Max / block_size) return -1;
  const int64_t end = num_blocks * block_size;
  uint64_t cap = 16;
  while (cap < 2 * static_cast<uint64_t>(n)) cap *= 2;
  // open addressing: slot -> index into keys, -1 free
  int32_t small[1024];
  std::vector<int32_t> large;
  int32_t* slots = small;
  if (cap > 1024) {
    try {
      large.resize(cap);
    } catch (const std::bad_alloc&) {
      return -1;
    }
    slots = large.data();
  }
  for (uint64_t s = 0; s < cap; ++s) slots[s] = -1;
  int64_t used = 0, processed = 0;
  for (int64_t i = 0; i < n; ++i) {
    int64_t p;
    if (!exact_int(PyList_GET_ITEM(positions, i), -(int64_t{1} << 62), int64_t{1} << 62, &p))
      return -1;
    if (p >= end) continue;
    if (p < -end) return -1;
    if (p < 0) p += end;
    uint64_t h = (static_cast<uint64_t>(p) * 0x9E3779B97F4A7C15ull) >> 32 & (cap - 1);
    while (slots[h] >= 0 && keys[slots[h]] != p) h = (h + 1) & (cap - 1);
    if (slots[h] < 0) {
      slots[h] = static_cast<int32_t>(used);
      keys[used] = static_cast<int32_t>(p);
      counts[used++] = 1;
    } else {
      ++counts[slots[h]];
    }
    ++processed;
  }
  *num_keys = used;
  return processed;
}
