"""The pool that lends multi-token calls their chunk buffers
(catena-models_amd/csrc/workspace.h), compiled for the host over a counted
allocator: blocks are lent again, a larger need replaces a smaller idle block,
at most eight stay idle, a failed allocation takes the idle ones back first,
the last model gives everything back, threads never share a block, and fewer
rows are taken where a new block would take an eighth of the free memory or is
not to be had."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "workspace.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>
using namespace cq35;

static std::atomic<long> held{0}, blocks{0};
static long limit = 1l << 40;
struct Counted {
  static void* allocate(size_t bytes) {
    if (held + (long)bytes > limit) return nullptr;
    held += (long)bytes;
    ++blocks;
    size_t* p = (size_t*)malloc(sizeof(size_t) + bytes);
    *p = bytes;
    return p + 1;
  }
  static void release(void* p) {
    size_t* q = (size_t*)p - 1;
    held -= (long)*q;
    --blocks;
    free(q);
  }
};
using Pool = BlockPool<Counted>;
static DeviceBlock lend(Pool& pool, size_t bytes) {
  DeviceBlock b = pool.idle(bytes);
  return b.p ? b : pool.allocate(bytes);
}
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main(int, char** argv) {
  Pool pool;
  pool.enter();
  if (!strcmp(argv[1], "again")) {  // sessions one after another: one block
    for (int i = 0; i < 100; ++i) pool.give(lend(pool, 1000 + i % 7 * 100));
    CHECK(blocks == 1 && held == 1600);
    DeviceBlock small = lend(pool, 10), large = lend(pool, 2000);
    CHECK(small.bytes == 1600 && large.bytes == 2000 && blocks == 2);
    pool.give(small), pool.give(large);
    CHECK(pool.idle(1500).bytes == 1600 || !"the smallest that fits");
  } else if (!strcmp(argv[1], "most")) {
    std::vector<DeviceBlock> b;
    for (int i = 0; i < 20; ++i) b.push_back(lend(pool, 100));
    CHECK(blocks == 20);
    for (auto& x : b) pool.give(x);
    CHECK(blocks == Pool::kMostIdle && held == 100 * Pool::kMostIdle);
  } else if (!strcmp(argv[1], "short")) {
    limit = 1000;
    DeviceBlock a = lend(pool, 300), b = lend(pool, 300);
    pool.give(a), pool.give(b);
    a = lend(pool, 900);  // only with both back
    CHECK(a.p && blocks == 1 && held == 900);
    CHECK(!lend(pool, 200).p && blocks == 1);
    pool.give(a);
    CHECK(pool.trim() && !pool.trim() && held == 0);
  } else if (!strcmp(argv[1], "last")) {
    pool.enter();
    DeviceBlock out = lend(pool, 10);
    pool.give(lend(pool, 20));
    pool.leave();
    CHECK(blocks == 2);
    pool.leave();
    CHECK(blocks == 1);
    pool.give(out);  // no model left: not kept
    CHECK(blocks == 0);
  } else if (!strcmp(argv[1], "rows")) {
    size_t room = 1 << 20;
    int asked = 0;
    auto bytes = [](long m) { return (size_t)m * 10; };
    auto room_left = [&] { return ++asked, room; };
    long rows = 1000;
    DeviceBlock b = lend_rows(pool, &rows, 200, bytes, room_left);
    CHECK(rows == 1000 && b.bytes == 10000 && asked == 1);
    pool.give(b);
    room = 79999;  // an eighth is less than a block of 1000 rows: an idle one will do, a new one not
    b = lend_rows(pool, &rows, 200, bytes, room_left);
    CHECK(rows == 1000 && asked == 1);
    DeviceBlock c = lend_rows(pool, &rows, 200, bytes, room_left);
    CHECK(rows == 200 && c.bytes == 2000 && asked == 2);
    pool.give(b), pool.give(c);
    b = lend_rows(pool, &(rows = 5000), 200, bytes, room_left);  // an idle block of more than the few rows
    CHECK(rows == 200 && b.bytes == 2000);
    pool.give(b);
    room = 1 << 20;
    limit = 30000;
    b = lend_rows(pool, &(rows = 5000), 200, bytes, room_left);  // no such block to be had
    CHECK(rows == 200 && b.p);
    pool.give(b);
    limit = 0;
    CHECK(!lend_rows(pool, &(rows = 5000), 4000, bytes, room_left).p);
    rows = 16;
    limit = 1 << 20;
    room = 0;
    CHECK(lend_rows(pool, &rows, 16, bytes, room_left).p && rows == 16);
  } else {  // threads: a lent block is written and read by its holder alone
    std::atomic<int> wrong{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 12; ++t)
      threads.emplace_back([&, t] {
        for (int i = 0; i < 2000; ++i) {
          DeviceBlock b = lend(pool, 64 + (t * 31 + i) % 5 * 64);
          memset(b.p, t, b.bytes);
          std::this_thread::yield();
          for (size_t k = 0; k < b.bytes; ++k) wrong += ((unsigned char*)b.p)[k] != t;
          pool.give(b);
        }
      });
    for (auto& t : threads) t.join();
    CHECK(wrong == 0 && blocks <= Pool::kMostIdle);
    pool.leave();
    CHECK(held == 0);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    src = d / "pool.cpp"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "catena-models_amd", "csrc"),
                    str(src), "-o", str(d / "pool")], check=True)
    return str(d / "pool")


@pytest.mark.parametrize("what", ["again", "most", "short", "last", "rows", "threads"])
def test_pool(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
