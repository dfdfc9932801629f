"""The ownership of the library's workspaces (wq_slots.h), compiled as host code with made-up streams."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "relax_amd", "csrc")

PROGRAM = """
#include <cstdio>
#include "%s/wq_slots.h"
using namespace wq;
static hipStream_t at(long a) { return (hipStream_t)a; }
#define CHECK(c) do { if (!(c)) { std::printf("line %%d: %%s\\n", __LINE__, #c); return 1; } } while (0)
static uint32_t done[4][kSlotTiles];
static SlotOwners<4> o;
static int index_of(Slot* s) { return s == nullptr ? -1 : (int)(s - o.slot); }
// a launch of `tiles` tiles on `s`: -1 without a slot
static int launch(hipStream_t s, int tiles) {
  Slot* const slot = o.take(s);
  if (slot == nullptr) return -1;
  slot->done = done[slot - o.slot];
  ++slot->launch;
  slot->tiles = tiles;
  return index_of(slot);
}
static void finish(int i, int from, int to) {
  for (int t = from; t < to; ++t) done[i][t] = o.slot[i].launch;
}
int main() {
  // a slot each, the same one again -- the null stream is a stream like others -- whether or not the launches have ended
  for (long s = 0; s < 4; ++s) CHECK(launch(at(s), 40) == s && launch(at(s), 40 + (int)s) == s);
  // all taken and busy: none, and every owner keeps its own
  CHECK(launch(at(9), 40) == -1);
  for (long s = 0; s < 4; ++s) CHECK(index_of(o.take(at(s))) == s);
  // busy until the last tile has ended, also with an earlier launch's numbers there
  finish(2, 0, 41);
  CHECK(launch(at(9), 40) == -1);
  finish(2, 41, 42);
  CHECK(launch(at(9), 10) == 2);
  CHECK(launch(at(2), 40) == -1);  // the former owner has to ask again
  finish(2, 1, 10);
  CHECK(launch(at(2), 40) == -1);
  finish(2, 0, 1);
  CHECK(launch(at(2), 40) == 2);
  // streams that are gone hold nothing back: any number of streams may come and go
  for (int i = 0; i < 4; ++i) finish(i, 0, o.slot[i].tiles);
  for (long s = 100; s < 1000; ++s) {
    const int i = launch(at(s), (int)(s %% kSlotTiles));
    CHECK(i >= 0 && i < 4);
    finish(i, 0, (int)(s %% kSlotTiles));
  }
  // launch numbers wrap
  o.slot[0].launch = 0xFFFFFFFFu;
  const int i = launch(o.slot[0].stream, 3);
  CHECK(i == 0 && o.slot[0].launch == 0 && !o.slot[0].idle());
  finish(0, 0, 3);
  CHECK(o.slot[0].idle());
  // calls of up to 16 rows: more streams than slots for larger calls, each busy, each with a slot
  static SlotOwners<kDecodeSlots> decode;
  static uint32_t never[kSlotTiles];
  static_assert(kDecodeSlots >= 3 * kSlots, "as many as a program has streams");
  for (long s = 0; s < kDecodeSlots; ++s) {
    Slot* const slot = decode.take(at(1000 + s));
    CHECK(slot == &decode.slot[s]);
    slot->done = never, slot->launch = 1, slot->tiles = 80;
  }
  CHECK(decode.take(at(5000)) == nullptr);
  std::printf("ok\\n");
  return 0;
}
"""


def test_slots_pass_on_once_the_last_launch_has_ended(tmp_path):
    (tmp_path / "slots.cpp").write_text(PROGRAM % CSRC)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", str(tmp_path / "slots"),
                    str(tmp_path / "slots.cpp")], check=True)
    r = subprocess.run([str(tmp_path / "slots")], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_the_library_never_asks_about_another_callers_stream():
    """A stream that owns a workspace may have been destroyed, and HIP reads through the handle it is given.  The host part makes
    calls about the calling stream (p.stream, or the parameter it was passed as) only."""
    import re

    text = re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, "wq_gemm_stream_host.hip")).read() + open(os.path.join(CSRC, "wq_slots.h")).read())
    calls = re.findall(r"\bhip(?:Stream|Event)\w+\(([^)]*)\)", text)
    assert calls and all(c.split(",")[0].strip() == "s" for c in calls), calls
    assert re.search(r"bool capturing\(hipStream_t s\)", text) and re.findall(r"capturing\(([^)]*)\)", text)[1:] == ["p.stream"]
