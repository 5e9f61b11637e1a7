// host_pair.h -- two parts of one call at the same time; no GPU needed, so host
// tests compile it by itself.
#pragma once
#include <exception>
#include <functional>
#include <new>
#include <string>
#include <thread>

namespace dvc {

// part() with an exception (host memory that is not to be had) turned into
// `failed` and its text: one that left a thread's function would end the process,
// as would one that passed a thread still running.
template <class Part>
int caught(Part &part, int failed, std::string &what) noexcept {
  try {
    return part();
  } catch (const std::bad_alloc &) {
    what = "out of memory";  // short enough to need none itself
  } catch (const std::exception &e) {
    try {
      what = e.what();
    } catch (...) {
    }
  } catch (...) {
    what = "exception";
  }
  return failed;
}

// first() on a thread of its own, or on this one before second() when there is
// none to be had, and second() on this one.  rc[k] and what[k]: each part's result
// and, if it threw, `failed` and the exception's text.
template <class First, class Second>
void run_pair(First first, Second second, int failed, int rc[2], std::string what[2]) {
  std::thread other;
  try {
    other = std::thread([&] { rc[0] = caught(first, failed, what[0]); });
  } catch (...) {
  }
  if (!other.joinable()) rc[0] = caught(first, failed, what[0]);
  rc[1] = caught(second, failed, what[1]);
  if (other.joinable()) other.join();
}

}  // namespace dvc
