"""parallel_copy (ncnn_amd/host/ncnn/hostcopy.cpp), the host side of large uploads: what its helper threads mean for the
process around them.  Compiled with a small driver; every run is bounded in time."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "ncnn_amd", "host", "ncnn")

DRIVER = r'''
#include "hostcopy.h"
#include <atomic>
#include <cerrno>
#include <csignal>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>
#include <dlfcn.h>
#include <pthread.h>
#include <sys/wait.h>
#include <unistd.h>

static bool copies(size_t bytes)
{
    std::vector<unsigned char> a(bytes), b(bytes + 1, 0);
    for (size_t i = 0; i < bytes; i++) a[i] = (unsigned char)(i * 7 + (i >> 11));
    ncnn::parallel_copy(b.data(), a.data(), bytes);
    return memcmp(a.data(), b.data(), bytes) == 0 && b[bytes] == 0;
}

// a process at its limit of threads: every creation from the allowed number on fails
static std::atomic<int> threads_left(1 << 30);
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* attr, void* (*start)(void*), void* arg)
{
    typedef int (*create)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const create real = (create)dlsym(RTLD_NEXT, "pthread_create");
    return threads_left.fetch_sub(1) > 0 ? real(t, attr, start, arg) : EAGAIN;
}

int main(int argc, char** argv)
{
    const char* what = argv[1];
    if (!strncmp(what, "limit", 5)) threads_left = atoi(what + 5);
    for (size_t bytes : {(size_t)1, (size_t)1 << 20, (size_t)(3 << 20) + 5, (size_t)8 << 20})
        if (!copies(bytes)) return 2;
    if (!strcmp(what, "fork")) // the child copies and leaves through exit()
    {
        const pid_t child = fork();
        if (child == 0) exit(copies((size_t)8 << 20) ? 0 : 3);
        int status = 0;
        for (int tenths = 0; tenths < 100; tenths++)
        {
            if (waitpid(child, &status, WNOHANG) == child)
            {
                if (!WIFEXITED(status) || WEXITSTATUS(status) != 0) return 4;
                return copies((size_t)8 << 20) ? 0 : 2; // the parent's helpers are untouched
            }
            usleep(100000);
        }
        kill(child, SIGKILL);
        waitpid(child, &status, 0);
        return 5;
    }
    if (!strcmp(what, "busy")) // another thread is copying when the process leaves
    {
        static std::atomic<int> rounds(0);
        std::thread([] { for (;;) { if (!copies((size_t)4 << 20)) _exit(2); rounds++; } }).detach();
        while (rounds < 3) usleep(1000);
    }
    return 0;
}
'''


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("hostcopy")
    (d / "driver.cpp").write_text(DRIVER)
    exe = str(d / "driver")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", "-Wno-unused-parameter", "-I", HOST, str(d / "driver.cpp"),
                           os.path.join(HOST, "hostcopy.cpp"), "-o", exe, "-lpthread", "-ldl"])
    return exe


@pytest.mark.parametrize("what", ["plain", "fork", "busy"])
def test_the_process_leaves(driver, what):
    """A forked child that leaves through exit() has the pool's object and none of its threads."""
    assert subprocess.run([driver, what], timeout=60).returncode == 0


@pytest.mark.parametrize("threads", [0, 1, 2])
def test_a_process_at_its_limit_of_threads_copies_with_those_it_gets(driver, threads):
    p = subprocess.run([driver, "limit%d" % threads], timeout=60, capture_output=True, text=True)
    assert p.returncode == 0, (p.returncode, p.stderr)
