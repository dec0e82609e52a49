// The loops over pages of the cache manager's bookkeeping (hfee_amd/cache/manager.py), on its own Python objects.
//
// A request of 400 tokens has 24 pages, and its admission and its release looked at each of them in Python: 35 + 16 us a
// request, 3.3 ms for 64 of them, and the GPU waits for every one.  What bounds it is the interpreter, a microsecond a page, and
// numpy's reading of a list of numbers, 14 us for 384.  The objects stay what they were (an ordered dict of the kept pages,
// lists of owners, bytes of tokens), so that every rule of the manager is still in one place, and only the walks are here.
// us of the host for admitting and releasing, before and now: 64 requests of 385 tokens with 24 kept pages each 3,290 -> 2,250, 40 of
// 367 to 1,099 3,710 -> 2,370, two of 8,193 1,470 -> 670.
//
// Called with the interpreter's lock held (ctypes.PyDLL).  A function that returns an object returns null with a Python
// exception set.
#include <Python.h>

#include <cstdint>
#include <cstring>

#define HFEE_API extern "C" __attribute__((visibility("default")))

// The numbers of a list as int64, one after the other, in bytes; None where one is no plain int (the caller then goes by way
// of an array); OverflowError where one does not fit.
HFEE_API PyObject* hfee_token_bytes(PyObject* tokens) {
  if (!PyList_CheckExact(tokens)) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(tokens);
  PyObject* out = PyBytes_FromStringAndSize(nullptr, n * 8);
  if (out == nullptr) return nullptr;
  char* to = PyBytes_AS_STRING(out);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* item = PyList_GET_ITEM(tokens, i);
    if (!PyLong_CheckExact(item)) {
      Py_DECREF(out);
      Py_RETURN_NONE;
    }
    const long long value = PyLong_AsLongLong(item);
    if (value == -1 && PyErr_Occurred()) {
      Py_DECREF(out);
      return nullptr;
    }
    const int64_t word = value;
    std::memcpy(to + 8 * i, &word, 8);
  }
  return out;
}

// Follows a chain of kept pages.  kept: digest -> (pages, the page's tokens as bytes, the digest of the page behind it).  From
// byte `at` of data on, as long as the entry under `following` holds the next page_bytes of data: it leaves `kept`, its digest is added to
// `digests` and its pages to `taken`.  Returns (the byte that it came to, the digest that is followed there).
HFEE_API PyObject* hfee_follow_chain(PyObject* kept, PyObject* data, Py_ssize_t page_bytes, Py_ssize_t at, PyObject* following,
                                     PyObject* digests, PyObject* taken) {
  if (!PyDict_Check(kept) || !PyBytes_CheckExact(data) || !PyList_CheckExact(digests) || !PyList_CheckExact(taken) || page_bytes < 1 || at < 0) {
    PyErr_SetString(PyExc_TypeError, "follow_chain: a dict, bytes and lists");
    return nullptr;
  }
  const Py_ssize_t size = PyBytes_GET_SIZE(data);
  const char* bytes = PyBytes_AS_STRING(data);
  Py_INCREF(following);
  for (; following != Py_None && at + page_bytes <= size; at += page_bytes) {
    PyObject* entry = PyDict_GetItemWithError(kept, following);
    if (entry == nullptr) {
      if (PyErr_Occurred()) goto failed;
      break;
    }
    PyObject* own = PyTuple_Check(entry) && PyTuple_GET_SIZE(entry) == 3 ? PyTuple_GET_ITEM(entry, 1) : nullptr;
    if (own == nullptr || !PyBytes_CheckExact(own) || PyBytes_GET_SIZE(own) != page_bytes ||
        std::memcmp(PyBytes_AS_STRING(own), bytes + at, (size_t)page_bytes) != 0)
      break;
    Py_INCREF(entry);
    const bool ok = PyObject_DelItem(kept, following) == 0 && PyList_Append(digests, following) == 0 &&
                    PyList_Append(taken, PyTuple_GET_ITEM(entry, 0)) == 0;
    PyObject* behind = PyTuple_GET_ITEM(entry, 2);
    Py_INCREF(behind);
    Py_DECREF(entry);
    Py_DECREF(following);
    following = behind;
    if (!ok) goto failed;
  }
  {
    PyObject* out = Py_BuildValue("(nO)", at, following);
    Py_DECREF(following);
    return out;
  }
failed:
  Py_DECREF(following);
  return nullptr;
}

// Leaves the first `n` pages of a request behind in `kept`, the deepest first.  tables: a list of page lists, one a group;
// digests and data: as above.  Returns (the pages of those that stay, the pages of those that were kept already), a list a group each.
HFEE_API PyObject* hfee_keep_pages(PyObject* kept, PyObject* digests, PyObject* tables, PyObject* data, Py_ssize_t page_bytes, Py_ssize_t n) {
  bool fits = PyDict_Check(kept) && PyList_CheckExact(digests) && PyList_CheckExact(tables) && PyBytes_CheckExact(data) && page_bytes > 0 && n >= 0 &&
              PyList_GET_SIZE(digests) >= n && PyBytes_GET_SIZE(data) / page_bytes >= n;
  const Py_ssize_t groups = fits ? PyList_GET_SIZE(tables) : 0;
  for (Py_ssize_t g = 0; g < groups; ++g)
    fits = fits && PyList_CheckExact(PyList_GET_ITEM(tables, g)) && PyList_GET_SIZE(PyList_GET_ITEM(tables, g)) >= n;
  if (!fits) {
    PyErr_SetString(PyExc_ValueError, "keep_pages: fewer digests, pages or tokens than pages to keep");
    return nullptr;
  }
  PyObject *stays = PyList_New(0), *twice = PyList_New(0), *behind = Py_None, *out = nullptr;
  bool ok = stays != nullptr && twice != nullptr;
  for (Py_ssize_t g = 0; ok && g < 2 * groups; ++g) {
    PyObject* list = PyList_New(0);
    ok = list != nullptr && PyList_Append(g < groups ? stays : twice, list) == 0;
    Py_XDECREF(list);
  }
  for (Py_ssize_t b = n - 1; ok && b >= 0; --b) {
    PyObject* digest = PyList_GET_ITEM(digests, b);
    const int there = PyDict_Contains(kept, digest);
    ok = there >= 0;
    if (ok && there == 0) {
      PyObject* pages = PyTuple_New(groups);
      for (Py_ssize_t g = 0; pages != nullptr && g < groups; ++g) {
        PyObject* page = PyList_GET_ITEM(PyList_GET_ITEM(tables, g), b);
        Py_INCREF(page);
        PyTuple_SET_ITEM(pages, g, page);
      }
      PyObject* own = PyBytes_FromStringAndSize(PyBytes_AS_STRING(data) + b * page_bytes, page_bytes);
      PyObject* entry = pages != nullptr && own != nullptr ? PyTuple_Pack(3, pages, own, behind) : nullptr;
      ok = entry != nullptr && PyObject_SetItem(kept, digest, entry) == 0;
      Py_XDECREF(pages);
      Py_XDECREF(own);
      Py_XDECREF(entry);
    }
    for (Py_ssize_t g = 0; ok && g < groups; ++g)
      ok = PyList_Append(PyList_GET_ITEM(there == 0 ? stays : twice, g), PyList_GET_ITEM(PyList_GET_ITEM(tables, g), b)) == 0;
    behind = digest;                                // (lives in `digests`)
  }
  if (ok) out = PyTuple_Pack(2, stays, twice);
  Py_XDECREF(stays);
  Py_XDECREF(twice);
  return out;
}

// owners[page] <- new_owner for every page of a list, as long as it is `owner`'s.  Returns None, or the first page that is not
// (those in front of it are handed over).
HFEE_API PyObject* hfee_hand_over(PyObject* owners, PyObject* pages, PyObject* owner, PyObject* new_owner) {
  if (!PyList_CheckExact(owners) || !PyList_CheckExact(pages)) {
    PyErr_SetString(PyExc_TypeError, "hand_over: lists of owners and pages");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(pages); ++i) {
    PyObject* number = PyList_GET_ITEM(pages, i);
    Py_INCREF(number);
    Py_ssize_t page = PyNumber_AsSsize_t(number, PyExc_IndexError);      // (whatever a list takes for an index)
    if (page < 0 && !PyErr_Occurred()) page += PyList_GET_SIZE(owners);      // (as a list's own index does)
    PyObject* other = nullptr;                      // whether somebody else has it
    if (!PyErr_Occurred()) {
      if (page < 0 || page >= PyList_GET_SIZE(owners)) {
        PyErr_SetString(PyExc_IndexError, "list index out of range");
      } else {
        PyObject* now = PyList_GET_ITEM(owners, page);
        Py_INCREF(now);
        other = PyObject_RichCompare(now, owner, Py_NE);
        Py_DECREF(now);
      }
    }
    const int is_other = other == nullptr ? -1 : PyObject_IsTrue(other);
    Py_XDECREF(other);
    if (is_other > 0 || (is_other == 0 && (owner == Py_None || new_owner == Py_None))) return number;
    Py_DECREF(number);
    if (is_other < 0) return nullptr;
    Py_INCREF(new_owner);
    if (PyList_SetItem(owners, page, new_owner) != 0) return nullptr;        // (takes the reference)
  }
  Py_RETURN_NONE;
}
