// Exceptions end at the C-ABI: every entry point that can allocate or throws
// on purpose runs its body in guarded(), which turns whatever leaves it into
// a status and the text of lblg_last_error.
#pragma once
#include <new>
#include <stdexcept>

#include "lblg.h"

namespace lblg {

void set_last_error(const char* what);  // capi_numeric.cpp (lblg_last_error)

template <typename F>
auto guarded(F f) noexcept -> decltype(f()) {
  try {
    return f();
  } catch (const std::bad_alloc&) {
    set_last_error("allocation failed");
    return LBLG_ERR_NOMEM;
  } catch (const std::length_error& e) {  // a size no allocation can have
    set_last_error(e.what());
    return LBLG_ERR_NOMEM;
  } catch (const std::invalid_argument& e) {
    set_last_error(e.what());
    return LBLG_ERR_ARG;
  } catch (const std::exception& e) {
    set_last_error(e.what());
    return LBLG_ERR_DEVICE;
  } catch (...) {
    set_last_error("unknown exception");
    return LBLG_ERR_DEVICE;
  }
}

}  // namespace lblg
