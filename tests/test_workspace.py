"""The growing device buffers (csrc/workspace.hpp), compiled for the host with
an allocator that counts and can fail: a failed growth leaves nothing that a
later call would take for a buffer or free again, and whoever holds the old
address is told before it goes."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "workspace.hpp"
#include <cstdio>
#include <cstdlib>
#include <set>
static std::set<void*> live;
static bool full = false, held = false;
static int frees = 0, moves = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
int main()
{
  Work w;
  auto moving = [&]() { moves++; CHECK(!w.p || live.count(w.p)); held = false; return 0; };
  auto alloc = [](void** p, size_t n) { if (full) return 3; *p = std::malloc(n); live.insert(*p); return 0; };
  auto release = [](void* p) { CHECK(live.erase(p) == 1); CHECK(!held); frees++; std::free(p); };
  auto grow = [&](size_t n) { return work_grow(w, n, moving, alloc, release); };
  CHECK(grow(64) == 0 && w.p && w.bytes == 64 && frees == 0);
  void* p = w.p;
  held = true;  // a captured graph has the address
  moves = 0;
  CHECK(grow(64) == 0 && grow(8) == 0 && w.p == p && moves == 0);
  CHECK(grow(128) == 0 && w.bytes == 128 && live.size() == 1 && frees == 1 && moves == 1);
  // no memory: an error now and again, nothing kept, nothing freed twice
  full = true;
  CHECK(grow(256) == 3);
  CHECK(!w.p && w.bytes == 0 && live.empty() && frees == 2);
  CHECK(grow(256) == 3 && grow(1) == 3 && frees == 2);
  full = false;
  CHECK(grow(32) == 0 && w.p && w.bytes == 32 && live.count(w.p));
  // a refusal to move keeps the buffer
  p = w.p;
  CHECK(work_grow(w, 512, []() { return 7; }, alloc, release) == 7 && w.p == p && w.bytes == 32 && live.count(p));
  std::puts("ok");
}
"""


def test_growth_failure_and_move(tmp_path):
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(SRC)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "miniafqmc_amd", "csrc"),
                           str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_every_growing_buffer_goes_through_it():
    """No buffer of the context keeps a size beside its pointer by hand."""
    import re
    src = open(os.path.join(ROOT, "miniafqmc_amd", "csrc", "ctx.hip")).read()
    assert not re.findall(r"\b\w+_bytes\s*=\s*(?:need|bytes|ybytes)\b", src)
    assert src.count("work_grow(") == 1
