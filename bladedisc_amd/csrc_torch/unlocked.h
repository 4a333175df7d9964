// Work without Python's interpreter lock.
#ifndef DQ8_UNLOCKED_H_
#define DQ8_UNLOCKED_H_

#define PY_SSIZE_T_CLEAN
#include <Python.h>

namespace dq8 {

// Gives the lock up for a scope and takes it again however the scope is left:
// Py_BEGIN / Py_END_ALLOW_THREADS would leave the thread without it when something throws, and
// the next use of Python's C API then takes the process down.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};

// f(args...) without the lock.  What reads a tensor (its pointer, its strides) can throw -- a
// tensor without storage under torch.vmap, a dimension it does not have -- and so belongs into
// the arguments, which are evaluated while the lock is still held.
template <typename R, typename... P, typename... A>
R call_unlocked(R (*f)(P...), A... args) {
  const Unlocked unlocked;
  return f(args...);
}

}  // namespace dq8

#endif  // DQ8_UNLOCKED_H_
