"""The pool of freed tensors' blocks (csrc/tensor_pool.h), compiled and run on
the host."""
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>

#include "tensor_pool.h"

#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)

using vh::TensorPool;

int main() {
    TensorPool pool;
    std::set<uintptr_t> freed;
    auto release = [&](void *p) { CHECK(freed.insert((uintptr_t)p).second); };
    auto keep = [&](uintptr_t p, size_t bytes) { return pool.keep((void *)p, bytes, release); };
    const size_t mb = (size_t)1 << 20;

    // Of one size the last block back is the first out; none of another size.
    CHECK(keep(1, 512) && keep(2, 512));
    CHECK(!pool.take(1024) && pool.take(512) == (void *)2 && pool.take(512) == (void *)1 && !pool.take(512));
    CHECK(pool.held() == 0);

    // A block above the limit stays the caller's.
    CHECK(!keep(3, TensorPool::kMaxBlock + 1) && freed.empty() && keep(3, TensorPool::kMaxBlock));
    CHECK(pool.take(TensorPool::kMaxBlock) == (void *)3);

    // Sizes that never come back fill the pool; the next ones are still kept,
    // and the oldest go back in their order.
    for (uintptr_t i = 0; i < 100; i++) {
        CHECK(keep(100 + i, 16 * mb + 512 * i));
        CHECK(pool.held() <= TensorPool::kMaxHeld);
        for (uintptr_t j = 0; j < i; j++)
            CHECK(freed.count(100 + j) || !freed.count(100 + j + 1));
    }
    CHECK(!freed.empty() && freed.size() >= 100 - 32 && !freed.count(199));
    CHECK(keep(500, 4096) && pool.take(4096) == (void *)500);
    // One that is used again and again does not wait, so it stays.
    for (uintptr_t i = 0; i < 100; i++) {
        CHECK(keep(600, 4096) && keep(1000 + i, 32 * mb + 512 * i));
        CHECK(pool.take(4096) == (void *)600);
    }
    // All of them, or, where they may still be in use, none.
    const size_t held = pool.held(), before = freed.size();
    pool.give_back([] { return false; }, release);
    CHECK(held > 0 && pool.held() == held && freed.size() == before);
    pool.give_back([] { return true; }, release);
    CHECK(pool.held() == 0 && !pool.take(16 * mb + 512 * 99) && freed.count(199) && freed.count(1099));

    // Freed from several threads.
    TensorPool shared;
    std::thread threads[4];
    for (int t = 0; t < 4; t++)
        threads[t] = std::thread([&, t] {
            for (int i = 0; i < 20000; i++)
                if (!shared.take(512 * (1 + i % 7)))
                    shared.keep((void *)(uintptr_t)(1 + t), 512 * (1 + i % 7), [](void *) { std::exit(2); });
        });
    for (auto &t : threads) t.join();
    shared.give_back([] { return true; }, [](void *) {});
    CHECK(shared.held() == 0);
    return 0;
}
"""


def test_pool_keeps_makes_room_and_gives_back(tmp_path):
    (tmp_path / "pool.cpp").write_text(PROGRAM)
    include = ROOT / "vestra-kernels_amd" / "csrc"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-fsanitize=undefined", f"-I{include}",
                    str(tmp_path / "pool.cpp"), "-o", str(tmp_path / "pool")], check=True)
    done = subprocess.run([str(tmp_path / "pool")], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout
