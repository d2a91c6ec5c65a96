// Host check of what handles, batches and servers allocate (fake_hip.hpp):
//   capture  a captured first step allocates nothing, on grids of every
//            shell-sum path
//   handle   where the expansion's work fields find no room, a handle takes
//            the direct sums, up to the bytes those need
//   batch    the same for a batch
//   slots    a batch of expanded systems needs no more than they do alone
//   tune     tuning an expanded handle or batch tries no splits of the direct
//            sums' back-projection, which would allocate their rows again
//   layout   a batch clears S where a step's layout of it differs from the last
// Prints "ok" and returns 0, or one line per failure.
#include "fake_hip.hpp"
#include "glst_batch.h"
#include "glst_hip.h"

#include <cstdio>
#include <string>
#include <vector>

using fake::st;

namespace {

int failures = 0;
#define CHECK(cond, ...)                                          \
  do {                                                            \
    if (!(cond)) {                                                \
      std::printf("FAIL %s:%d: %s: ", __FILE__, __LINE__, #cond); \
      std::printf(__VA_ARGS__);                                   \
      std::printf("\n");                                          \
      ++failures;                                                 \
    }                                                             \
  } while (0)

// the launches are stand-ins: any addresses do for the caller's arrays
const double *arr(int i) { return reinterpret_cast<const double *>(4096 * (i + 1)); }

struct Sys {
  uint32_t n;
  double box[3], rcut, tol;
};

void capture() {
  const Sys cases[] = {{262000, {144, 144, 342}, 9, 1e-4},
                       {400000, {144, 144, 297}, 9, 1e-4},
                       {200000, {144, 144, 216}, 9, 1e-4},
                       {400000, {189, 189, 189}, 9, 1e-4},
                       {100000, {135, 135, 135}, 9, 1e-4},
                       {10000, {54, 54, 54}, 9, 1e-5},
                       {30000, {90, 90, 90}, 9, 1e-4}};
  for (const Sys &c : cases)
    for (int ct : {GLST_CT_FLOAT, GLST_CT_DOUBLE})
      for (int shape : {4, 0, 3, 2}) {
        glst_handle_t h = nullptr;
        CHECK(glst_create(ct, c.n, c.tol, c.box[0], c.box[1], c.box[2], c.rcut,
                          nullptr, &h) == GLST_OK, "%s",
              glst_global_last_error());
        if (!h) continue;
        glst_set_option(h, "graph", 1);
        glst_set_option(h, "rmt_shape", shape);
        st.refused_in_capture = 0;
        st.reset();
        const glst_status_t s =
            glst_calc_ener_force(h, arr(0), arr(1), arr(2), arr(3));
        CHECK(s == GLST_OK && st.refused_in_capture == 0,
              "box %g %g %g ct %d shape %d: %s", c.box[0], c.box[1], c.box[2],
              ct, shape, glst_last_error(h));
        CHECK(st.steps == 1 && st.harm + (st.direct > 0) == 1,
              "%ld steps, %ld expanded, %ld direct launches", st.steps, st.harm,
              st.direct);
        glst_destroy(h);
      }
}

void handle() {
  const Sys cases[] = {{400000, {189, 189, 189}, 9, 1e-4},
                       {100000, {135, 135, 135}, 9, 1e-4},
                       {10000, {54, 54, 54}, 9, 1e-5}};
  for (const Sys &c : cases)
    for (int ct : {GLST_CT_FLOAT, GLST_CT_DOUBLE}) {
      auto run = [&](size_t limit, size_t *peak) {
        st.limit = limit;
        st.peak = st.used;
        glst_handle_t h = nullptr;
        st.reset();
        glst_status_t s = glst_create(ct, c.n, c.tol, c.box[0], c.box[1],
                                      c.box[2], c.rcut, nullptr, &h);
        if (s == GLST_OK)
          s = glst_calc_ener_force(h, arr(0), arr(1), arr(2), arr(3));
        *peak = st.peak;
        const int route = s != GLST_OK ? 0 : st.harm ? 1 : 2;
        if (h) glst_destroy(h);
        st.limit = SIZE_MAX;
        CHECK(st.used == 0, "%zu bytes left", st.used);
        return route;
      };
      size_t full = 0, less = 0;
      CHECK(run(SIZE_MAX, &full) == 1, "box %g", c.box[0]);
      CHECK(run(full - 1, &less) == 2, "box %g ct %d: %zu bytes", c.box[0], ct,
            full - 1);
    }
}

size_t batch_run(int ct, const std::vector<Sys> &v, size_t limit, int *route) {
  std::vector<uint32_t> n;
  std::vector<double> box, rcut;
  for (const Sys &s : v) {
    n.push_back(s.n);
    box.insert(box.end(), s.box, s.box + 3);
    rcut.push_back(s.rcut);
  }
  st.limit = limit;
  st.peak = st.used;
  st.reset();
  glst_batch_t b = nullptr;
  glst_status_t s =
      glst_batch_create(ct, static_cast<uint32_t>(n.size()), n.data(),
                        box.data(), rcut.data(), v[0].tol, nullptr, &b);
  if (s == GLST_OK)
    s = glst_batch_calc_ener_force(b, arr(0), arr(1), arr(2), arr(3));
  const size_t peak = st.peak;
  *route = s != GLST_OK ? 0 : st.harm ? 1 : 2;
  if (b) glst_batch_destroy(b);
  st.limit = SIZE_MAX;
  CHECK(st.used == 0, "%zu bytes left", st.used);
  return peak;
}

void batch() {
  const std::vector<Sys> v = {{100000, {135, 135, 135}, 9, 1e-4},
                              {30000, {66.9, 66.9, 66.9}, 9, 1e-4},
                              {10000, {54, 54, 54}, 9, 1e-4}};
  for (int ct : {GLST_CT_FLOAT, GLST_CT_DOUBLE}) {
    int route = 0;
    const size_t full = batch_run(ct, v, SIZE_MAX, &route);
    CHECK(route == 1, "route %d", route);
    batch_run(ct, v, full - 1, &route);
    CHECK(route == 2, "ct %d: route %d with %zu bytes", ct, route, full - 1);
    batch_run(ct, v, full / 4, &route);
    CHECK(route == 0, "ct %d: route %d with %zu bytes", ct, route, full / 4);
  }
}

void slots() {
  const std::vector<Sys> v = {{288000, {142, 142, 142}, 9, 1e-4},
                              {30000, {66.9, 66.9, 66.9}, 9, 1e-4},
                              {30000, {66.9, 66.9, 66.9}, 9, 1e-4},
                              {30000, {66.9, 66.9, 66.9}, 9, 1e-4}};
  for (int ct : {GLST_CT_FLOAT, GLST_CT_DOUBLE}) {
    auto bytes = [&](const std::vector<Sys> &w) {
      std::vector<uint32_t> n;
      std::vector<double> box, rcut;
      for (const Sys &s : w) {
        n.push_back(s.n);
        box.insert(box.end(), s.box, s.box + 3);
        rcut.push_back(s.rcut);
      }
      size_t b = 0;
      CHECK(glst_batch_device_bytes(ct, static_cast<uint32_t>(n.size()),
                                    n.data(), box.data(), rcut.data(),
                                    w[0].tol, &b) == GLST_OK, "sizing");
      return b;
    };
    size_t alone = 0;
    for (const Sys &s : v) alone += bytes({s});
    const size_t all = bytes(v);
    CHECK(all <= alone, "ct %d: %zu bytes, %zu alone", ct, all, alone);
    int route = 0;
    batch_run(ct, v, SIZE_MAX, &route);  // (and the buffers of every slot)
    CHECK(route == 1, "route %d", route);
  }
}

void tune() {
  const double box[] = {135, 135, 135}, rcut = 9;
  for (uint32_t n : {100000u, 20000u}) {  // expanded, and dilute
    glst_handle_t h = nullptr;
    CHECK(glst_create(GLST_CT_DOUBLE, n, 1e-4, 135, 135, 135, 9, nullptr, &h) ==
              GLST_OK, "%s", glst_global_last_error());
    long before = st.allocations;
    double ms = 0.0;
    st.reset();
    CHECK(glst_autotune(h, arr(0), arr(1), arr(2), arr(3), 2, &ms) == GLST_OK,
          "%s", glst_last_error(h));
    CHECK((st.harm > 0) == (n == 100000), "%u charges", n);
    CHECK((st.allocations == before) == (st.harm > 0), "%ld allocations",
          st.allocations - before);
    glst_destroy(h);
    glst_batch_t b = nullptr;
    CHECK(glst_batch_create(GLST_CT_DOUBLE, 1, &n, box, &rcut, 1e-4, nullptr,
                            &b) == GLST_OK, "%s", glst_global_last_error());
    before = st.allocations;
    st.reset();
    CHECK(glst_batch_autotune(b, arr(0), arr(1), arr(2), arr(3), 2, &ms) ==
              GLST_OK, "%s", glst_batch_last_error(b));
    CHECK((st.allocations == before) == (st.harm > 0), "batch: %ld allocations",
          st.allocations - before);
    glst_batch_destroy(b);
  }
}

// fused 0 expands, the other launch modes do not
void layout() {
  const uint32_t n = 100000;
  const double box[] = {135, 135, 135}, rcut = 9;
  glst_batch_t b = nullptr;
  CHECK(glst_batch_create(GLST_CT_FLOAT, 1, &n, box, &rcut, 1e-4, nullptr,
                          &b) == GLST_OK, "%s", glst_global_last_error());
  int last = -1;
  for (int graph : {0, 1})
    for (int fused : {0, 0, 1, 1, 0, 2, 0, 3, 2, 0}) {
      glst_batch_set_option(b, "graph", graph);
      CHECK(glst_batch_set_option(b, "fused", fused) == GLST_OK, "%s",
            glst_batch_last_error(b));
      st.reset();
      CHECK(glst_batch_calc_ener_force(b, arr(0), arr(1), arr(2), arr(3)) ==
                GLST_OK, "%s", glst_batch_last_error(b));
      const int now = fused == 0;
      CHECK((st.harm > 0) == (now == 1), "fused %d", fused);
      // S: more than the 4 n doubles of the accumulators
      CHECK((st.filled > 4 * n) == (last >= 0 && now != last),
            "fused %d graph %d: %zu doubles filled", fused, graph, st.filled);
      last = now;
    }
  glst_batch_destroy(b);
}

}  // namespace

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "capture") capture();
  else if (what == "handle") handle();
  else if (what == "batch") batch();
  else if (what == "slots") slots();
  else if (what == "tune") tune();
  else if (what == "layout") layout();
  else return 2;
  if (failures || st.failures) return 1;
  std::printf("ok\n");
  return 0;
}
