"""The codecs' pool of device blocks (vkdt_amd/csrc/scratch_pool.h) over a
counted memory of two devices, on the CPU: every block freed once, failures
leave nothing behind, idle blocks bounded, given back and kept apart by
device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "scratch_pool.h"
#include <map>
#include <stdio.h>
#include <string.h>

// memory: live addresses, a limit per device, failures on demand
static std::map<void *, size_t> dev_live, pin_live;
static int cur_device, dev_allocs, pin_allocs, bad_frees, fail_pin, fail_dev, last_error;
static size_t limit = (size_t)1 << 40, next_addr = 4096;
enum { OOM = 2, OTHER = 7 };

struct mem
{
  static size_t used() { size_t s = 0; for(auto &k : dev_live) s += k.second; return s; }
  static int device(int *d) { *d = cur_device; return 0; }
  static int dev_alloc(void **p, size_t n)
  {
    dev_allocs++;
    if(fail_dev) { last_error = fail_dev; return fail_dev; }
    if(used() + n > limit) { last_error = OOM; return OOM; }
    *p = (void *)next_addr; next_addr += n; dev_live[*p] = n;
    return 0;
  }
  static int pin_alloc(void **p, size_t n)
  {
    pin_allocs++;
    if(fail_pin && pin_live.size() >= (size_t)fail_pin - 1) { last_error = OOM; return OOM; }
    *p = (void *)next_addr; next_addr += n; pin_live[*p] = n;
    return 0;
  }
  static void dev_free(void *p) { if(!dev_live.erase(p)) bad_frees++; }
  static void pin_free(void *p) { if(!pin_live.erase(p)) bad_frees++; }
  static bool oom(int e) { return e == OOM; }
  static void forget() { last_error = 0; }
};

typedef scratch_pool<mem> pool_t;
static const size_t MB = (size_t)1 << 20;
#define CHECK(x) do { if(!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while(0)

// a block whose second allocation fails is freed once, and the caller may put
// back what it was given
static int pinned_failure()
{
  pool_t p;
  scratch_t s;
  fail_pin = 1;
  CHECK(p.get(s, 3 * MB, true) == OOM);
  CHECK(!s.dev && !s.pin && dev_live.empty());
  p.put(s, false);
  p.put(s, true);
  CHECK(bad_frees == 0);
  return 0;
}

// an allocation that succeeds at the second try, without the idle blocks, and
// one that fails altogether leave no error for a later check to find
static int last_error_is_cleared()
{
  pool_t p;
  scratch_t s;
  limit = 10 * MB;
  CHECK(p.get(s, 6 * MB, false) == 0);
  p.put(s, true);
  CHECK(p.get(s, 1 * MB, false) == 0);          // too small for the idle block
  CHECK(last_error == 0);
  p.put(s, true);
  void *q = nullptr;
  CHECK(p.alloc(mem::dev_alloc, &q, 8 * MB) == 0 && q && last_error == 0);
  CHECK(dev_live.size() == 1);           // the idle blocks went
  CHECK(p.get(s, 6 * MB, false) == OOM && !s.dev && last_error == 0);
  mem::dev_free(q);
  fail_dev = OTHER;                      // no lack of memory: nothing is given back for it
  CHECK(p.get(s, 6 * MB, false) == OTHER && last_error == 0);
  fail_dev = 0;
  fail_pin = 1;
  CHECK(p.get(s, 6 * MB, true) == OOM && last_error == 0 && dev_live.empty() && bad_frees == 0);
  return 0;
}

// pinned memory that is short comes from the idle blocks too
static int pinned_from_idle()
{
  pool_t p;
  scratch_t a, b;
  CHECK(p.get(a, 2 * MB, true) == 0);
  p.put(a, true);
  fail_pin = 2;                          // one pinned buffer at a time
  CHECK(p.get(b, 20 * MB, true) == 0 && b.pin && dev_live.size() == 1 && pin_live.size() == 1 && last_error == 0);
  p.put(b, true);
  void *q = nullptr;
  CHECK(p.alloc(mem::pin_alloc, &q, MB) == 0 && q && dev_live.empty() && bad_frees == 0);
  return 0;
}

// a pinned buffer is made where one is asked for, and stays with its block
static int pinned_where_used()
{
  pool_t p;
  scratch_t s;
  CHECK(p.get(s, 5 * MB, false) == 0 && !s.pin && pin_allocs == 0);
  uint8_t *first = s.dev;
  p.put(s, true);
  CHECK(p.get(s, 5 * MB, true) == 0 && s.dev == first && s.pin && pin_allocs == 1);
  p.put(s, true);
  CHECK(p.get(s, 5 * MB, true) == 0 && pin_allocs == 1);
  p.put(s, false);
  CHECK(dev_live.empty() && pin_live.empty() && bad_frees == 0);
  return 0;
}

// a block that failed comes back to the driver, a good one to the next caller
static int reuse()
{
  pool_t p;
  scratch_t a, b;
  CHECK(p.get(a, 5 * MB, false) == 0 && a.size >= 5 * MB);
  uint8_t *first = a.dev;
  p.put(a, true);
  CHECK(!a.dev && dev_live.size() == 1);
  CHECK(p.get(b, 4 * MB, false) == 0 && b.dev == first && dev_allocs == 1);
  p.put(b, false);
  CHECK(dev_live.empty() && bad_frees == 0);
  // not a block of more than twice the size, nor a smaller one
  CHECK(p.get(a, 20 * MB, false) == 0);
  p.put(a, true);
  CHECK(p.get(b, 4 * MB, false) == 0 && b.size < 10 * MB);
  p.put(b, true);
  CHECK(p.get(b, 8 * MB, false) == 0 && dev_allocs == 4);
  p.put(b, true);
  CHECK(p.trim() && dev_live.empty() && pin_live.empty() && !p.trim() && bad_frees == 0);
  return 0;
}

// the blocks of a 9504x6336 export in 4:4:4 (130 bytes a block of coefficients,
// three times a stream of 4 bits a coefficient) serve the next one
static int large_export()
{
  const size_t blocks = (size_t)3 * (9504 / 8) * (6336 / 8);
  pool_t p;
  for(int k = 0; k < 3; k++)
  {
    scratch_t a, b;
    CHECK(p.get(a, 130 * blocks, true) == 0 && p.get(b, 96 * blocks, false) == 0);
    p.put(a, true);
    p.put(b, true);
  }
  CHECK(dev_allocs == 2 && pin_allocs == 1);
  return 0;
}

static int devices()
{
  pool_t p;
  scratch_t a, b;
  CHECK(p.get(a, 5 * MB, false) == 0);
  uint8_t *first = a.dev;
  p.put(a, true);
  cur_device = 1;
  CHECK(p.get(b, 5 * MB, false) == 0 && b.dev != first && b.device == 1);
  p.put(b, true);
  cur_device = 0;
  CHECK(p.get(a, 5 * MB, false) == 0 && a.dev == first);
  p.put(a, true);
  return 0;
}

// the oldest idle blocks go where the bound, in bytes or blocks, is passed
static int bounded()
{
  pool_t p;
  scratch_t s[4], t[SCRATCH_SLOTS + 3];
  for(int k = 0; k < 4; k++) CHECK(p.get(s[k], SCRATCH_KEEP / 3 - 2 * MB, false) == 0);
  uint8_t *first = s[0].dev, *second = s[1].dev;
  for(int k = 0; k < 4; k++) p.put(s[k], true);
  CHECK(mem::used() <= SCRATCH_KEEP && dev_live.size() == 3 && !dev_live.count(first) && dev_live.count(second));
  CHECK(p.get(s[0], SCRATCH_KEEP + MB, false) == 0);
  p.put(s[0], true);
  CHECK(mem::used() <= SCRATCH_KEEP && dev_live.size() == 3);
  p.trim();
  for(auto &b : t) CHECK(p.get(b, 1, false) == 0);
  for(auto &b : t) p.put(b, true);
  CHECK(dev_live.size() == SCRATCH_SLOTS && bad_frees == 0);
  return 0;
}

int main(int, char **v)
{
#define RUN(f) if(!strcmp(v[1], #f)) return f()
  @RUN@
  return 2;
}
"""
NAMES = ["pinned_failure", "last_error_is_cleared", "pinned_from_idle", "pinned_where_used", "reuse", "large_export", "devices", "bounded"]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "pool.cpp").write_text(SRC.replace("@RUN@", " ".join(f"RUN({n});" for n in NAMES)))
    try:
        subprocess.run(["g++", "--version"], check=True, capture_output=True)
    except (OSError, subprocess.CalledProcessError) as e:
        pytest.skip(f"no C++ compiler: {e}")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I" + os.path.join(ROOT, "vkdt_amd", "csrc"),
                    "-o", str(d / "pool"), str(d / "pool.cpp")], check=True)
    return str(d / "pool")


@pytest.mark.parametrize("name", NAMES)
def test_pool(exe, name):
    r = subprocess.run([exe, name], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
