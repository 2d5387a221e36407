// Exceptions inside the host entry points of the C-ABI: operator new is
// replaced (the library resolves it here) and throws at the k-th allocation
// of an entry, k = 1, 2, ... until the call no longer reaches it.  Every
// such call must return a status below zero, and the same call without the
// failure must then succeed on the same handle.
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <new>
#include <stdexcept>
#include <vector>

#include "lblg.h"

static long g_left = 0;  // allocations until the failure (0: none)
static int g_kind = 0;
static bool g_thrown = false;

static void* take(std::size_t n) {
  if (g_left > 0 && --g_left == 0) {
    g_thrown = true;
    if (g_kind == 0) throw std::bad_alloc();
    if (g_kind == 1) throw std::length_error("length");
    if (g_kind == 2) throw std::runtime_error("runtime");
    throw 7;
  }
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void* operator new(std::size_t n) { return take(n); }
void* operator new[](std::size_t n) { return take(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
void operator delete[](void* p, std::size_t) noexcept { std::free(p); }

static int failures = 0;
static void check(bool ok, const char* what, int kind, long k, int rc) {
  if (ok) return;
  ++failures;
  std::printf("FAIL %s kind %d allocation %ld status %d\n", what, kind, k, rc);
}

// call: runs the entry on a state made by `fresh`
static void sweep(const char* what, const std::function<void()>& fresh, const std::function<int()>& call) {
  for (int kind = 0; kind < 4; ++kind) {
    long k = 1;
    for (;; ++k) {
      fresh();
      std::printf("case %s kind %d allocation %ld\n", what, kind, k);
      std::fflush(stdout);
      g_kind = kind;
      g_thrown = false;
      g_left = k;
      int rc = call();
      g_left = 0;
      if (!g_thrown) {
        check(rc == LBLG_OK, what, kind, k, rc);
        break;
      }
      check(rc < 0, what, kind, k, rc);
      rc = call();
      check(rc == LBLG_OK, what, kind, -k, rc);
      if (k >= 200) k += k / 10;  // late allocations of long calls: a sample
    }
  }
}

int main() {
  // a 12 x 12 grid Laplacian's lower half
  const int g = 12, n = g * g;
  std::vector<int> Ap(1, 0), Ai;
  std::vector<double> Ax;
  for (int j = 0; j < n; ++j) {
    Ai.push_back(j);
    Ax.push_back(5.0);
    if (j % g != g - 1) {
      Ai.push_back(j + 1);
      Ax.push_back(-1.0);
    }
    if (j + g < n) {
      Ai.push_back(j + g);
      Ax.push_back(-1.0);
    }
    Ap.push_back((int)Ai.size());
  }
  lblg_settings st;
  lblg_default_settings(&st);
  lblg_handle* h = nullptr;
  auto drop = [&] {
    lblg_destroy(h);
    h = nullptr;
  };
  auto made = [&] {
    drop();
    lblg_create(&h, n, Ap.data(), Ai.data(), Ax.data());
  };
  auto analyzed = [&] {
    made();
    lblg_analyze(h, &st, nullptr, nullptr);
  };
  sweep("create", drop, [&] {
    drop();
    return lblg_create(&h, n, Ap.data(), Ai.data(), Ax.data());
  });
  sweep("analyze", made, [&] { return lblg_analyze(h, &st, nullptr, nullptr); });
  std::vector<int> perm(n);
  sweep("order_nd", [] {}, [&] { return lblg_order_nd(n, Ap.data(), Ai.data(), perm.data()); });
  std::vector<int64_t> idx;
  std::vector<double> val;
  for (int j = 0; j < n; j += 3) {
    idx.push_back(Ap[j]);
    val.push_back(6.0);
  }
  sweep("update_values", analyzed, [&] { return lblg_update_values(h, (int64_t)idx.size(), idx.data(), val.data()); });
  for (int which = 0; which < 12; ++which)
    sweep("symbolic_ints", analyzed, [&] { return lblg_symbolic_ints(h, which, nullptr) >= 0 ? LBLG_OK : -1; });
  drop();

  const int count = 3;
  const int ns[count] = {n, n, n};
  const int* P[count] = {Ap.data(), Ap.data(), Ap.data()};
  const int* I[count] = {Ai.data(), Ai.data(), Ai.data()};
  const double* X[count] = {Ax.data(), Ax.data(), Ax.data()};
  auto batch = [&] {
    drop();
    return lblg_batch_create(&h, count, ns, P, I, X);
  };
  sweep("batch_create", drop, batch);
  sweep("batch_analyze", [&] { batch(); }, [&] { return lblg_batch_analyze(h, &st); });
  std::vector<double> B(count * n, 1.0), err(count);
  sweep("batch_backward_errors", [&] { batch(); }, [&] {
    return lblg_batch_backward_errors(h, 1, B.data(), count * n, B.data(), count * n, err.data());
  });
  drop();

  // min 1/2 x'Hx + q'x, x_0 + x_1 = 1, x_i <= 1/2 (the rows of the identity)
  std::vector<double> q(n, -1.0), b(n, 0.5);
  const double a[1] = {1.0};
  std::vector<int> Ep(n + 1, 2), Bp(n + 1), Bi(n);
  std::vector<double> Bx(n, 1.0);
  Ep[0] = 0;
  Ep[1] = 1;
  const int Ei[2] = {0, 0};
  const double Ex[2] = {1.0, 1.0};
  for (int j = 0; j < n; ++j) {
    Bp[j + 1] = j + 1;
    Bi[j] = j;
  }
  lblg_qp* qp = nullptr;
  auto qp_drop = [&] {
    lblg_qp_destroy(qp);
    qp = nullptr;
  };
  auto qp_make = [&] {
    qp_drop();
    return lblg_qp_create(&qp, n, Ap.data(), Ai.data(), Ax.data(), q.data(), 1, Ep.data(), Ei, Ex, a, n, Bp.data(),
                          Bi.data(), Bx.data(), b.data());
  };
  sweep("qp_create", qp_drop, qp_make);
  sweep("kkt_analyze", [&] { qp_make(); }, [&] { return lblg_kkt_analyze(qp, &st); });
  std::vector<int> rows(n);
  for (int i = 0; i < n; ++i) rows[i] = i;
  sweep("kkt_edit", [&] {
    qp_make();
    lblg_kkt_analyze(qp, &st);
  }, [&] { return lblg_kkt_edit(qp, 1, n, rows.data()); });
  qp_drop();
  std::printf("failures %d\n", failures);
  return failures != 0;
}
