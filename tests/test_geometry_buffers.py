"""Host side of the geometry on a stand-in runtime.  After a shape gradient that ran out of memory half
way through growing its work buffers, a later call with fewer corners has buffers of the sizes it
needs; and a call that fails with copies of the caller's arrays under way waits for them, as its
buffers' hipFree did, before it returns."""
import host_build

HEAD = r"""
#include "host_runtime.hpp"
#include "lsx_geometry_host.hpp"

using host_runtime::room;
static int corners = 0;

namespace lsx { namespace geo {
void level_set(const double*, const double*, const double*, int, int, int, Box, Body, double*, hipStream_t) {}
int oscillation_fix(const double*, double*, double*, unsigned char*, int*, int, int, int, Box, hipStream_t) { return 1; }
void alpha(const double*, int, int, int, Box, double*, double*, double*, hipStream_t) {}
void types(const double*, int, int, int, Box, int*, int*, int*, int*, hipStream_t) {}
void theta(const double*, const double*, const double*, const int*, const int*, const int*, int, int, int, Box, double*,
           double*, double*, hipStream_t) {}
void vof(const int*, const double*, const double*, const double*, const double*, const double*, const double*,
         const double*, const double*, const double*, int, int, int, double*, hipStream_t) {}
int active_blocks(long) { return 1; }
void count_nodes(const double*, const double*, const unsigned char*, unsigned char*, int, int, int, int, Box, double,
                 int* count, hipStream_t) {
  CHECK(room(count) >= active_counts(0) * sizeof(int));
  count[1] = corners;
  count[2] = 0;
}
void list_nodes(const double*, const double*, const unsigned char*, int, int, int, int, Box, double, int*, int* list,
                hipStream_t) {
  CHECK(room(list) >= corners * sizeof(int));
}
void corner_gradient(const GeoBase&, const int*, int, const unsigned char*, const int*, int, const double*,
                     const double*, const double*, const double*, int, int, int, Box, int, const double*, const double*,
                     int, const RhsArgs*, double, double*, hipStream_t) {}
void bezier_chain(const double*, const int*, int count, const double*, const double*, const double*, int, int, Body,
                  int* hf, double* huv, double* hw, double* out, hipStream_t) {
  CHECK(room(hf) >= count * sizeof(int));
  CHECK(room(huv) >= 2 * count * sizeof(double));
  CHECK(room(hw) >= 3 * count * sizeof(double));
  CHECK(room(out) >= 288 * sizeof(double));
}
} }

"""

GROWTH = HEAD + r"""
int main() {
  const int N = 8;
  const double w[N] = {1, 1, 1, 1, 1, 1, 1, 1};
  const std::vector<double> v(N * N * N, 1.0), ctrl(288, 0.5);
  double out[288];
  const size_t list = 100 + 100 / 4;  // what a list of 100 corners grows to
  for (size_t size : {list * sizeof(int), 2 * list * sizeof(double), 3 * list * sizeof(double)}) {
    lsx::Geometry g(N, N, N, w, w, w, 0, 0, 0, nullptr);
    g.build(lsx::geo::Body{lsx::geo::BODY_BEZIER6, {4, 4, 4}, {1, 1, 1}}, lsx::geo::Box{1, N - 1, 1, N - 1}, ctrl.data());
    auto gradient = [&](int n) {
      corners = n;
      g.shape_gradient(v.data(), v.data(), lsx::geo::OBJ_DRAG_X, nullptr, 1, 1e-7, nullptr, out, LSX_MEM_DEVICE);
    };
    gradient(10);
    host_runtime::fail_size = size;
    bool failed = false;
    try {
      gradient(100);
    } catch (const lsx::Error&) {
      failed = true;
    }
    CHECK(failed);
    (void)hipGetLastError();
    host_runtime::fail_size = 0;
    for (int n : {50, 10, 100, 0, 101}) gradient(n);
  }
  std::printf("ok\n");
}
"""

FAILURE = HEAD + r"""
int main() {
  const int N = 8;
  const double w[N] = {1, 1, 1, 1, 1, 1, 1, 1};
  std::vector<double> v(N * N * N, 1.0), b(N * N * N);
  lsx::Geometry g(N, N, N, w, w, w, 0, 0, 0, nullptr);
  g.build(lsx::geo::Body{lsx::geo::BODY_SPHERE, {4, 4, 4}, {1, 1, 1}}, lsx::geo::Box{1, N - 1, 1, N - 1});
  lsx_flow_bc bc{};
  bc.outflow = 1;
  for (int round = 0; round < 2; ++round) {  // with new blocks, then with kept ones
    host_runtime::allowed = round == 0 ? 5 : 0;  // u, v, w, west, b; the outflow's copy comes after their copies
    const long before = host_runtime::syncs;
    bool failed = false;
    try {
      g.pressure_rhs(v.data(), v.data(), v.data(), v.data(), v.data(), bc, b.data(), LSX_MEM_HOST);
    } catch (const lsx::Error&) {
      failed = true;
    }
    CHECK(failed);
    CHECK(host_runtime::syncs > before);
  }
  std::printf("ok\n");
}
"""


def test_buffers_after_a_failed_growth(tmp_path):
    host_build.run(tmp_path, GROWTH, ["lsx_geometry_host.cpp"])


def test_failed_call_waits_for_its_copies(tmp_path):
    host_build.run(tmp_path, FAILURE, ["lsx_geometry_host.cpp"])
