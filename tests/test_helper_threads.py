"""Host threads of the staged prefill where the system refuses one: the caller goes on with those that exist (no GPU needed)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyre_amd", "csrc")
# the program's own pthread_create refuses after `allowed` threads, as a process limit does
PROGRAM = r"""
#include "workers.h"
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <pthread.h>
static int allowed, made;
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  if (made >= allowed) return EAGAIN;
  ++made; return ((int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*))dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, x);
}
int main(int, char** v) {
  const int n = atoi(v[1]); allowed = atoi(v[2]);
  std::atomic<int> todo{1000}, done{0}; auto work = [&](int) { while (todo.fetch_sub(1) > 0) ++done; };
  std::vector<std::thread> th; start_helpers(th, n, work);
  work(0);
  for (auto& x : th) x.join();
  cpu_set_t one; CPU_ZERO(&one); CPU_SET(sched_getcpu(), &one);
  const int all = helper_count(1 << 20); const bool alone = sched_setaffinity(0, sizeof one, &one) == 0 && helper_count(4) == 0;
  printf("%d %d %d %d\n", (int)th.size(), done.load(), all < (1 << 20) && helper_count(-1) == 0, (int)alone);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("threads"); src, exe = str(d / "t.cpp"), str(d / "t")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D_GNU_SOURCE", "-I", CSRC, src, "-o", exe, "-rdynamic", "-pthread", "-ldl"], check=True)
    return exe


@pytest.mark.parametrize("n,allowed", [(0, 9), (5, 9), (5, 5), (5, 3), (5, 0), (-1, 9)])
def test_refused_threads_leave_the_work_to_the_others(program, n, allowed):
    r = subprocess.run([program, str(n), str(allowed)], capture_output=True, text=True, timeout=30)
    assert r.returncode == 0 and r.stdout.split() == [str(max(0, min(n, allowed))), "1000", "1", "1"], (r.returncode, r.stdout, r.stderr)
