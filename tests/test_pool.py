"""The memory pool of factors and plans (hss_pool.h), on the CPU with a counted allocator: held
blocks never keep an allocation of the device from fitting, in whichever pool they are; a block handed
out is at most a sixteenth and an eighth above the request, and its size is reported; `exact`
requests get no more than their pages; the oldest held block goes first at a limit."""
import pathlib
import shutil
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "hssmatrices.jl_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "hss_pool.h"
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
struct Mem {  // a card of `room` bytes
    static size_t room, out, count;
    static std::map<void*, size_t> live;
    static void* alloc(size_t b) {
        if (out + b > room) return nullptr;
        void* p = reinterpret_cast<void*>(++count * 64);
        live[p] = b;
        out += b;
        return p;
    }
    static void release(void* p) {
        out -= live.at(p);
        live.erase(p);
    }
};
size_t Mem::room = size_t(8) << 30, Mem::out = 0, Mem::count = 0;
std::map<void*, size_t> Mem::live;
using Pool = hss::BlockPool<Mem>;
constexpr size_t MB = size_t(1) << 20;

int main() {
    {
        Pool a, b, other;
        a.attach(0);
        b.attach(0);
        other.attach(1);
        // sizes: new blocks, held blocks, exact ones
        for (size_t n : {size_t(1), size_t(4096), size_t(100001), 3 * MB + 7, 777 * MB}) {
            size_t got = 0, again = 0;
            void* p = a.get(0, n, false, &got);
            CHECK(p && got >= n && got <= n + n / 16 + Pool::kPage && Mem::live.at(p) == got);
            a.put(p);
            void* q = a.get(0, n, false, &again);
            CHECK(q == p && again == got);
            a.put(q);
            size_t ex = 0;
            void* e = a.get(0, n, true, &ex);
            CHECK(e && ex >= n && ex < n + Pool::kPage);
            a.put(e);
            a.trim();
        }
        CHECK(Mem::out == 0);
        size_t got = 0;
        void* big = a.get(0, 64 * MB);
        a.put(big);
        void* half = a.get(0, 33 * MB, false, &got);  // half the size is not taken
        CHECK(half != big && got < 36 * MB);
        a.put(half);
        void* near = a.get(0, 60 * MB, false, &got);
        CHECK(near == big && got == Mem::live.at(big));
        void* ex = a.get(0, 60 * MB, true);
        CHECK(ex != big);
        a.put(near);
        a.put(ex);
        a.trim();
        CHECK(Mem::out == 0);

        // what any pool of the device holds does not keep an allocation from fitting
        void* pa = a.get(0, 1500 * MB);
        void* pb = b.get(0, 1500 * MB);
        void* po = other.get(1, 100 * MB);
        a.put(pa);
        b.put(pb);
        other.put(po);
        CHECK(Mem::out > 3000 * MB);
        void* all = Pool::allocate(0, Mem::room - 200 * MB);
        CHECK(all);
        CHECK(Mem::out <= Mem::room && other.trim());  // the other device's pool was left alone
        Mem::release(all);
        pa = a.get(0, 1500 * MB);
        a.put(pa);
        void* most = b.get(0, Mem::room - 64 * MB, true);
        CHECK(most);
        b.put(most);  // larger than a pool holds: freed
        CHECK(Mem::out == 0);
        // the last of the memory, without the rounding
        void* last = a.get(0, Mem::room);
        CHECK(last && Mem::out == Mem::room);
        CHECK(!b.get(0, 1) && !Pool::allocate(0, 1));
        a.put(last);

        // limits: the oldest goes
        std::vector<void*> v;
        for (int i = 0; i < 5; ++i) v.push_back(a.get(0, (500 + 100 * i) * MB, true));
        for (void* p : v) a.put(p);  // 3500 MB in all
        CHECK(Mem::out <= Pool::kHeldMax);
        CHECK(a.get(0, 900 * MB, true) == v[4] && a.get(0, 800 * MB, true) == v[3]);
        a.put(v[4]);
        a.put(v[3]);
        a.trim();
        v.clear();
        for (size_t i = 0; i < Pool::kHeldBlocks + 3; ++i) v.push_back(a.get(0, Pool::kPage * (i + 1), true));
        for (void* p : v) a.put(p);
        CHECK(Mem::live.size() == Pool::kHeldBlocks && !Mem::live.count(v[2]) && Mem::live.count(v[3]));
    }
    CHECK(Mem::out == 0 && Mem::live.empty());  // destroyed pools have given everything back
    std::puts("ok");
    return 0;
}
"""


def test_pool(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src = tmp_path / "pool.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "pool"
    subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-Wall", "-I", str(CSRC), str(src), "-o", str(exe), "-pthread"], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.strip() == "ok", p.stdout + p.stderr


def test_every_device_allocation_goes_through_the_pools():
    """hipMalloc is called in one place, the one that makes the pools give back."""
    calls = [(f.name, i) for f in sorted(CSRC.glob("hss_*.*")) if f.suffix in (".hip", ".h")
             for i, line in enumerate(f.read_text().splitlines(), 1)
             if "hipMalloc(" in line.split("//")[0]]
    assert len(calls) == 1 and calls[0][0] == "hss_runtime.hip", calls
