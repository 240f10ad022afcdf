"""The host side of the bulk transfers (csrc/kge_transfer.h) without a device: slots filled and emptied by
hand, through any number of copy threads, with every byte compared."""

import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "distributed-kge-poplar_amd" / "csrc"

# argv: threads that pthread_create grants, threads asked for, total, chunk, slots, offset of the array,
# milliseconds that every slot takes
PROGRAM = r"""
#include "kge_transfer.h"
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <pthread.h>
#include <sys/resource.h>

static int granted;
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    if (granted-- <= 0) return EAGAIN;
    return ((Fn)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}
static double cpu_seconds() {
    rusage u;
    getrusage(RUSAGE_SELF, &u);
    return u.ru_utime.tv_sec + u.ru_stime.tv_sec + 1e-6 * (u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

int main(int, char** argv) {
    granted = atoi(argv[1]);
    const int expect = std::min(granted, atoi(argv[2]));
    const size_t total = atol(argv[3]), chunk = atol(argv[4]);
    const int n_slots = atoi(argv[5]), offset = atoi(argv[6]), ms = atoi(argv[7]);
    kge::CopyThreads threads(atoi(argv[2]));
    if (threads.size() != expect) { printf("%d threads\n", threads.size()); return 1; }
    std::vector<char> array_v(total + offset + 64, 0x5a), slots(n_slots * chunk), device(total);
    char* const array = array_v.data() + offset;
    for (size_t i = 0; i < total; ++i) array[i] = (char)(i * 2654435761u >> 13);
    const std::vector<char> want(array, array + total);
    const double cpu0 = cpu_seconds();
    auto slot_work = [&] { if (ms) std::this_thread::sleep_for(std::chrono::milliseconds(ms)); };
    {
        kge::SlottedCopy copy(array, slots.data(), total, chunk, n_slots, true, &threads);
        for (size_t k = 0; k < copy.n_chunks(); ++k) {
            slot_work();
            copy.allow(k);
            copy.wait(k);
            std::memcpy(device.data() + k * chunk, slots.data() + k % n_slots * chunk, std::min(chunk, total - k * chunk));
        }
    }
    if (device != want) return printf("to the slots\n"), 1;
    std::memset(array, 0, total);
    {
        kge::SlottedCopy copy(array, slots.data(), total, chunk, n_slots, false, &threads);
        for (size_t k = 0; k < copy.n_chunks(); ++k) {
            std::memcpy(slots.data() + k % n_slots * chunk, device.data() + k * chunk, std::min(chunk, total - k * chunk));
            slot_work();
            copy.allow(k);
            copy.wait(k);
        }
    }
    if (std::memcmp(array, want.data(), total)) return printf("from the slots\n"), 1;
    for (int i = 0; i < 64; ++i)
        if (array[total + i] != 0x5a) return printf("behind the array\n"), 1;
    {  // given up half way (a launch that fails): the threads come back, asleep or not
        kge::SlottedCopy copy(array, slots.data(), total, chunk, n_slots, true, &threads);
        copy.allow(0);
        slot_work();
    }
    printf("cpu %.3f\n", cpu_seconds() - cpu0);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("transfer")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-pthread", f"-I{CSRC}", "-o", os.fspath(d / "t"),
                    os.fspath(d / "t.cpp"), "-ldl"], check=True)
    return d / "t"


def _run(program, *args):
    r = subprocess.run([os.fspath(program), *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    return float(r.stdout.split()[1])


# one byte; less than a page; chunks that end on no page; many times round the slots
@pytest.mark.parametrize("total,chunk,n_slots,offset", [(1, 16, 1, 0), (5000, 5008, 1, 13), (1 << 20, 100_000, 4, 4095),
                                                        (3_000_001, 65_536, 4, 1), (1 << 22, 1 << 20, 2, 4096)])
@pytest.mark.parametrize("threads", [0, 1, 7])
def test_every_byte_arrives(program, total, chunk, n_slots, offset, threads):
    _run(program, threads, threads, total, chunk, n_slots, offset, 0)


@pytest.mark.parametrize("granted", [0, 3])
def test_a_system_without_threads(program, granted):
    """The system refuses a thread: the copies go on with those there are."""
    _run(program, granted, 7, 3_000_001, 65_536, 4, 1, 0)


def test_waiting_threads_sleep(program):
    """Ten chunks of 20 ms each way, seven threads: they look on for 0.2 ms of each wait and sleep for
    the rest (all of them on a core for the whole time would be 7 x 0.42 s where there are the cores)."""
    assert _run(program, 7, 7, 1 << 20, 110_000, 4, 0, 20) < 0.2
