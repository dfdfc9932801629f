"""The counter of a tile whose windows share its finishing (wq_gemm_stream.hip): what the built kernels do to it."""
import os
import re
import subprocess

import pytest

from tests.test_lds_requests_cpu import CSRC, listing


def shared_split_kernels(name, tmp_path):
    """{kernel: its instructions} of the builds of an object that split K over workgroups on tiles of 128 columns and 64 rows or more."""
    if not os.path.exists(os.path.join(CSRC, name)):
        subprocess.run(["make", "-C", CSRC, name], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    kernels, here = {}, None
    for line in listing(os.path.join(CSRC, name), tmp_path):
        label = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if label:
            shape = re.search(r"wq_gemm_stream_kernelILi\dELi(\d)ELi(\d)ELi(\d)E(?:Li\d+E){5}Lb[01]ELi1ELb[01]E", label[1])
            shares = shape and int(shape[1]) >= 2 and int(shape[2]) * int(shape[3]) == 4
            here = kernels.setdefault(label[1], []) if shares else None
        elif here is not None:
            here.append(re.sub(r"\s*//.*", "", line).strip())
    return kernels


@pytest.mark.parametrize("name", ["wq_gemm_stream4.o", "wq_gemm_stream8.o"])
def test_every_access_to_the_counter_but_its_return_to_zero_is_an_add(name, tmp_path):
    """Arrive, look, resign and account are each an add that returns what was there, so that all of them are in one order.  (A look
    that adds a zero which the compiler sees becomes a load.)  The two stores: the counter's return to zero, and the host's mark."""
    kernels = shared_split_kernels(name, tmp_path)
    assert len(kernels) == 6, "two tiles: tile-major, scales in pieces, scales by macro step"
    for kernel, code in kernels.items():
        accesses = [i.split()[0] for i in code if re.match(r"(global|flat)_", i)]
        assert sorted(accesses) == ["global_atomic_add"] * 4 + ["global_store_dword"] * 2, (kernel, accesses)
        assert all("sc0" in i for i in code if i.startswith("global_atomic_add")), kernel


PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>
#include "%s/wq_split_share.h"
using namespace wq;
#define CHECK(c) do { if (!(c)) { std::printf("line %%d: %%s (%%d windows, %%d looks)\\n", __LINE__, #c, windows, looks); std::exit(1); } } while (0)

static int windows, looks;

// What is shared, and of every workgroup what its accesses to memory so far have returned.
struct State {
  uint32_t counter = 0, returned = 0, finished = 0, shared = 0, written[8] = {};
  std::vector<uint32_t> seen[8];
  bool ended[8] = {};
};

struct Stop {};

// Workgroup w from its beginning again, what it did before answered from `seen`, up to and with one more access to memory.
static void step(State& s, int w) {
  size_t at = 0;
  bool moved = false;
  auto access = [&](auto&& f) -> uint32_t {
    if (at < s.seen[w].size()) return s.seen[w][at++];
    if (moved) throw Stop{};
    moved = true;
    s.seen[w].push_back(f());
    return s.seen[w][at++];
  };
  try {
    const uint32_t parts = split_parts(
        windows, w, looks, [&](uint32_t p) { access([&] { return s.written[w] |= p & ((1u << windows) - 1); }); }, [&](auto&& f) { return f(); },
        [&](uint32_t by) {
          return access([&] {
            CHECK(!s.returned);  // nobody touches the counter once it is back at zero
            const uint32_t before = s.counter;
            s.counter += by;
            return before;
          });
        },
        [&](auto&& if_last) { if (if_last()) access([&] { return s.counter = 0, ++s.returned; }); });
    access([&] {
      CHECK(!(parts & s.finished));  // no part by two workgroups
      for (int v = 0; v < windows; ++v) CHECK(v == w || (s.written[v] & parts) == parts);  // nor read before it was written
      s.finished |= parts;
      if (parts & ~(1u << w)) s.shared |= 1;  // somebody finished another's part
      if (parts == 0) s.shared |= 2;          // somebody left his own
      return 0u;
    });
    s.ended[w] = true;
  } catch (Stop) {
  }
}

static bool over(const State& s) {
  for (int w = 0; w < windows; ++w)
    if (!s.ended[w]) return false;
  CHECK(s.finished == (1u << windows) - 1 && s.counter == 0 && s.returned == 1);
  return true;
}

static std::set<std::vector<uint32_t>> been;
static uint32_t ends, shared;

static void every_order(const State& s) {
  std::vector<uint32_t> key{s.counter, s.returned, s.finished, s.shared};
  for (int w = 0; w < windows; ++w) {
    key.push_back(s.written[w]), key.push_back(0xFFFFFFFFu);
    key.insert(key.end(), s.seen[w].begin(), s.seen[w].end());
  }
  if (!been.insert(key).second) return;
  if (over(s)) {
    ++ends, shared |= s.shared;
    return;
  }
  for (int w = 0; w < windows; ++w)
    if (!s.ended[w]) {
      State next = s;
      step(next, w);
      every_order(next);
    }
}

int main(int argc, char** argv) {
  windows = std::atoi(argv[1]), looks = std::atoi(argv[2]);
  if (argc == 3) {
    every_order(State{});
    std::printf("%%u ends, shared %%u\\n", ends, shared);
    return 0;
  }
  std::mt19937 rng(windows);
  for (int run = 0; run < 3000; ++run) {
    State s;
    const uint32_t late = rng() %% 100;
    while (!over(s)) {
      int w = rng() %% 100 < late ? 0 : rng() %% windows;
      while (s.ended[w]) w = (w + 1) %% windows;
      step(s, w);
    }
    ++ends, shared |= s.shared;
  }
  std::printf("%%u ends, shared %%u\\n", ends, shared);
  return 0;
}
"""


@pytest.fixture(scope="module")
def orders(tmp_path_factory):
    d = tmp_path_factory.mktemp("orders")
    (d / "orders.cpp").write_text(PROGRAM % CSRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-Wno-attributes", "-o", str(d / "orders"), str(d / "orders.cpp")], check=True)
    return lambda *args: subprocess.run([str(d / "orders")] + [str(a) for a in args], stdout=subprocess.PIPE, text=True)


@pytest.mark.parametrize("windows,looks", [(2, 0), (2, 1), (2, 2), (2, 8), (3, 0), (3, 1), (3, 2), (4, 0)])
def test_every_part_is_finished_once_in_every_order_of_the_kernels_own_steps(orders, windows, looks):
    """wq_split_share.h, which the kernel runs, one access to memory at a time."""
    r = orders(windows, looks)
    assert r.returncode == 0 and r.stdout.endswith("shared 3\n"), r.stdout


@pytest.mark.parametrize("windows", [3, 5, 8])
@pytest.mark.parametrize("looks", [0, 2, 8])
def test_every_part_is_finished_once_in_random_orders_of_the_kernels_own_steps(orders, windows, looks):
    r = orders(windows, looks, "random")
    assert r.returncode == 0 and r.stdout == "3000 ends, shared 3\n", r.stdout
