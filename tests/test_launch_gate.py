"""Ordering of persistent launches across streams and threads: the bookkeeping (csrc/launch_gate.h) on the CPU, step by
step through the interleavings that matter, and real launches from several threads on the GPU."""
import os
import subprocess
import threading

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashlstm_poc_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "launch_gate.h"
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    enum : int { kPerThread = 2, X = 10, Y = 11, Z = 12 };
    typedef flstm_hip::LaunchGate<int> Gate;
    {   // one stream: nothing waits; another one does until the first has been waited for
        Gate g(kPerThread);
        CHECK(!g.must_wait(X) && !g.must_wait(kPerThread));
        g.launched(X, false);
        CHECK(!g.must_wait(X) && g.must_wait(Y) && g.last() == X && !g.recorded());
        g.waited(Y, g.launches());
        CHECK(g.must_wait(Y));
        g.waited(X, g.launches());
        CHECK(!g.must_wait(Y));
    }
    {   // a second thread launches on the stream that the first is waiting for: the wait says nothing about that launch
        Gate g(kPerThread);
        g.launched(X, false);
        const unsigned long first = g.launches();
        g.launched(X, false);
        const unsigned long second = g.launches();
        g.waited(X, first);
        CHECK(g.must_wait(Y));
        g.waited(X, second);
        CHECK(!g.must_wait(Y));
    }
    {   // a chain over three streams: the end of an early one clears nothing, the end of the last one everything
        Gate g(kPerThread);
        g.launched(X, false);
        const unsigned long at_x = g.launches();
        g.launched(Y, false);
        g.waited(X, at_x);
        CHECK(g.must_wait(Z) && g.must_wait(X) && g.last() == Y);
        g.waited(Y, g.launches());
        CHECK(!g.must_wait(Z) && !g.must_wait(X));
    }
    {   // a launch on one stream between a wait for another and what it says: X, Y (waited for), X again, then "Y is over"
        Gate g(kPerThread);
        g.launched(Y, false);
        const unsigned long at_y = g.launches();
        g.launched(X, false);
        g.waited(Y, at_y);
        CHECK(g.must_wait(Y));
    }
    {   // the per-thread handle names another stream in every thread: a stranger to itself, and never known to be over
        Gate g(kPerThread);
        CHECK(g.wants_event(kPerThread) && !g.wants_event(X));
        g.launched(kPerThread, true);
        CHECK(g.must_wait(kPerThread) && g.must_wait(X) && g.recorded());
        g.waited(kPerThread, g.launches());
        CHECK(g.must_wait(kPerThread) && g.must_wait(X));
        g.launched(X, false);
        CHECK(!g.must_wait(X) && !g.recorded());
        g.waited(X, g.launches());
        CHECK(!g.must_wait(kPerThread));
    }
    std::printf("ok\n");
    return 0;
}
"""


def test_gate_bookkeeping(tmp_path):
    src, exe = tmp_path / "gate.cpp", tmp_path / "gate"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", str(exe)])
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


# whole-chip recurrences from three threads, two of them on one stream: none of them may find its workgroups waiting for
# another's (a launch that did would give up and be counted as a fallback); 96 rows of 1024 units take every CU.  Or all
# three through the one handle (2) that names another stream in every thread
@pytest.mark.gpu
@pytest.mark.parametrize("T,B,H,per_thread", [(40, 96, 1024, False), (24, 20, 2560, False), (30, 16, 2048, False), (40, 96, 1024, True)])
def test_persistent_launches_of_several_threads_and_streams(T, B, H, per_thread, monkeypatch):
    import torch
    from helpers import make_problem
    from flashlstm_poc_amd import LstmCore
    p = {k: v.cuda() for k, v in make_problem(T, B, 64, H, seed=H).items()}
    x, dy = p["x"].half(), p["dy"].half()
    h0, c0 = p["h0"].half(), p["c0"].half()

    def one_pass(core):
        return (*core.forward(x, h0, c0), *core.backward(x, dy))

    cores = [LstmCore(B, 64, H) for _ in range(3)]
    for core in cores:
        core.pack(p["w_ih"], p["w_hh"], p["b_ih"], p["b_hh"])
    want = [t.clone() for t in one_pass(cores[0])]
    torch.cuda.synchronize()
    assert cores[0].info("persistent_fwd") == 1 and cores[0].info("persistent_bwd") == 1
    shared, other = torch.cuda.Stream(), torch.cuda.Stream()
    if per_thread:
        monkeypatch.setattr(LstmCore, "_stream", staticmethod(lambda: 2))
        shared = other = torch.cuda.default_stream()
    wrong = []

    def work(core, stream):
        try:
            with torch.cuda.stream(stream):
                for n in range(12):
                    got = one_pass(core)
                    wrong.extend((n, k) for k, (a, b) in enumerate(zip(got, want)) if not torch.equal(a, b))
        except Exception as e:   # (an exception in a thread would otherwise pass unseen)
            wrong.append(repr(e))

    threads = [threading.Thread(target=work, args=a) for a in zip(cores, (shared, shared, other))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not wrong, wrong[:5]
    assert [core.info("fallbacks") for core in cores] == [0, 0, 0]
    for core in cores:
        core.close()
