"""The device arena of plans, compiled with the host compiler against a stand-in allocator: what it
reports is what it took from the device, blocks of small tables included, and all of it goes back."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "holoflow_amd", "csrc")

HIP = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
inline std::map<void *, size_t> g_held;
inline size_t g_total = 0, g_limit = (size_t)1 << 40;
inline hipError_t g_last = hipSuccess;
inline hipError_t hipMalloc(void **p, size_t n) {
  if (g_total + n > g_limit) return g_last = hipErrorOutOfMemory;
  *p = std::malloc(n < 64 ? 64 : n);
  g_held[*p] = n;
  g_total += n;
  return hipSuccess;
}
inline hipError_t hipFree(void *p) {
  if (!g_held.count(p)) std::abort();
  g_total -= g_held[p];
  g_held.erase(p);
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
"""

PRELUDE = r"""
#include <cstdio>
#include "dev_arena.hh"
namespace hfx { std::string g_err; void set_last_error(const std::string &m) { g_err = m; } }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
"""


def _run(tmp_path, body):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    src = tmp_path / "arena.cpp"
    src.write_text(PRELUDE + "int main() {\n" + body + "\n  return 0;\n}\n")
    exe = tmp_path / "arena"
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-I", str(tmp_path), "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def test_reported_bytes_are_the_bytes_held(tmp_path):
    _run(tmp_path, r"""
  {
    hfx::DevArena a;
    float *p[40];
    float *big;
    char *c;
    CHECK(a.alloc(&p[0], 0) == HFX_OK);                     // an empty table opens the first block
    CHECK(a.bytes == g_total && a.bytes == a.kBlock);
    for (int i = 1; i < 40; ++i) {
      CHECK(a.alloc(&p[i], 1000 + i) == HFX_OK);            // 4 KB each: several blocks
      CHECK(a.bytes == g_total);
      CHECK(((size_t)((char *)p[i] - a.block) & 255) == 0);
    }
    CHECK(a.ptrs.size() == 2);
    CHECK(a.alloc(&big, 1 << 20) == HFX_OK && a.bytes == g_total);
    CHECK(a.alloc(&c, a.kSmall) == HFX_OK && a.alloc(&c, a.kSmall + 1) == HFX_OK && a.bytes == g_total);
    g_limit = g_total;
    CHECK(a.alloc(&big, 1 << 20) == HFX_E_NOMEM && a.bytes == g_total && !hfx::g_err.empty());
  }
  CHECK(g_total == 0 && g_held.empty());""")


def test_a_full_device_gets_one_window(tmp_path):
    """Creation where the library's windows do not fit, and where not even one does; a caller's own
    count and other failures stand."""
    _run(tmp_path, r"""
  int calls = 0;
  auto create = [&](const hfx_plan_desc &d) -> hfx_status {
    ++calls;
    hfx::DevArena a;
    char *tiny, *planes;
    hfx_status rc = a.alloc(&tiny, 16);
    if (rc == HFX_OK) rc = a.alloc(&planes, (size_t)(d.batch_windows ? d.batch_windows : 32) << 20);
    return rc != HFX_OK ? rc : d.height > 0 ? HFX_OK : HFX_E_INVALID;
  };
  hfx_plan_desc d{};
  d.height = 8;
  g_limit = 8 << 20;
  CHECK(hfx::create_or_one_window(d, create) == HFX_OK && calls == 2 && g_last == hipSuccess);
  d.batch_windows = 9;
  CHECK(hfx::create_or_one_window(d, create) == HFX_E_NOMEM && calls == 3);
  d.batch_windows = 0;
  g_limit = 1 << 20;
  CHECK(hfx::create_or_one_window(d, create) == HFX_E_NOMEM && calls == 5);
  g_limit = 1 << 30;
  CHECK(hfx::create_or_one_window(d, create) == HFX_OK && calls == 6);
  d.height = 0;
  CHECK(hfx::create_or_one_window(d, create) == HFX_E_INVALID && calls == 7);
  CHECK(g_total == 0 && g_held.empty());""")
