"""Device blocks kept for a handle's next call, on a stand-in runtime."""
import host_build

HEAD = r"""
#include "host_runtime.hpp"
#include "lsx_solver.hpp"
using lsx::BlockPool;
using lsx::DevBuf;
namespace hr = host_runtime;
"""

OUT_OF_MEMORY = HEAD + r"""
// leaves `count` idle blocks of `bytes` in a pool
static void fill(BlockPool& pool, int count, size_t bytes) {
  BlockPool::Scope s(pool);
  std::vector<DevBuf<char>> b(count);
  for (auto& q : b) q.alloc(bytes);
}
int main() {
  hr::limit = 1000;
  {  // an allocation outside any call's scope, as a solve's staging buffers are
    BlockPool a;
    fill(a, 3, 300);
    CHECK(hr::live == 900);
    DevBuf<char> x;
    x.alloc(500);
    CHECK(hr::live == 500 && hipGetLastError() == hipSuccess);
  }
  CHECK(hr::live == 0);
  {  // another handle's call, with blocks of its own and of a third one
    BlockPool a, b, c;
    fill(a, 2, 200);
    fill(b, 1, 100);
    fill(c, 1, 100);
    BlockPool::Scope s(b);
    DevBuf<char> x;
    x.alloc(900);
    CHECK(hr::live == 900);
  }
  {  // a pool that is gone is not asked
    BlockPool a;
    { BlockPool b; fill(b, 1, 600); }
    fill(a, 1, 600);
    DevBuf<char> x;
    x.alloc(1000);
  }
  {  // nothing idle: the error is reported
    BlockPool a;
    DevBuf<char> x, y;
    x.alloc(600);
    bool failed = false;
    try {
      y.alloc(600);
    } catch (const lsx::Error& e) {
      failed = e.code == LSX_ERR_HIP;
    }
    CHECK(failed && !y.p && y.n == 0);
  }
  CHECK(hr::live == 0);
  std::printf("ok\n");
}
"""

# a set-up: work blocks of a size, given back at its end
OTHER_SIZES = HEAD + r"""
static long setup(BlockPool& pool, int count, size_t bytes) {  // allocations it made
  const long before = hr::mallocs;
  BlockPool::Scope s(pool);
  std::vector<DevBuf<char>> b(count);
  for (auto& q : b) q.alloc(bytes);
  return hr::mallocs - before;
}
int main() {
  const size_t mb = size_t(1) << 20;
  {  // two sizes in turn: both are kept
    BlockPool a;
    setup(a, 3, 100);
    setup(a, 4, 300);
    for (int k = 0; k < 40; ++k) CHECK(setup(a, 3, 100) == 0 && setup(a, 4, 300) == 0);
    CHECK(hr::live == 1500);
  }
  CHECK(hr::live == 0);
  {  // blocks of a size that is asked for no more go, in calls
    BlockPool a;
    setup(a, 5, 700);
    for (int k = 0; k < BlockPool::idle_calls; ++k) setup(a, 1, 100);
    CHECK(hr::live == 3600);
    setup(a, 1, 100);
    CHECK(hr::live == 100);
  }
  {  // and so do those of a size that is asked for less often than there are blocks
    BlockPool a;
    setup(a, 5, 700);
    for (int k = 0; k <= BlockPool::idle_calls; ++k) setup(a, 2, 700);
    CHECK(hr::live == 1400);
  }
  {  // a full pool makes room for the present call's sizes, never beyond its bound
    BlockPool a;
    setup(a, 4, 64 * mb);
    CHECK(hr::live == 256 * mb);
    setup(a, 5, 40 * mb);
    CHECK(hr::live <= BlockPool::bound);
    CHECK(setup(a, 5, 40 * mb) == 0);
    setup(a, 8, 40 * mb);
    CHECK(hr::live <= BlockPool::bound);
    setup(a, 1, 300 * mb);
    CHECK(hr::live <= BlockPool::bound);
  }
  {  // a call inside a call is one call
    BlockPool a;
    setup(a, 1, 700);
    for (int k = 0; k < BlockPool::idle_calls - 1; ++k) {
      BlockPool::Scope s(a);
      setup(a, 1, 100);
    }
    CHECK(setup(a, 1, 700) == 0);
  }
  CHECK(hr::live == 0);
  std::printf("ok\n");
}
"""


def test_out_of_memory_takes_every_handles_idle_blocks(tmp_path):
    host_build.run(tmp_path, OUT_OF_MEMORY)


def test_blocks_of_other_sizes_go(tmp_path):
    host_build.run(tmp_path, OTHER_SIZES)
