"""Two contexts on two devices driven by one thread: every entry point selects
its context's device before it allocates, launches, fills or synchronises,
whatever device the calls before it left current.

Runs in a child process against tests/fake_hip.c, which stands in for the HIP
runtime and notes each such call made with another device current."""
import ctypes as C
import os
import re
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def counter_slots():
    """Counter name -> slot, from the library's own enumeration."""
    text = open(os.path.join(ROOT, "dynoplan_amd", "csrc", "dp_internal.h")).read()
    body = re.search(r"enum \{([^}]*DPC_COUNT[^}]*)\}", text).group(1)
    names = [n.split("=")[0].strip() for n in body.split(",") if n.strip()]
    return {n: k for k, n in enumerate(names)}


CASES = ["novel append past the capacity", "few nodes", "many nodes", "window overflow", "radius", "select",
         "surrogate", "batch", "settings"]


@pytest.fixture(scope="module")
def fake_runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-std=c11", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")],
                   check=True)
    return so


@pytest.mark.parametrize("case", CASES)
def test_device_is_selected(fake_runtime, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake_runtime, case], cwd=ROOT, text=True,
                       capture_output=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "checked" in r.stdout


class Driver:
    """A context on `device`; each call runs with the other device current."""

    def __init__(self, fake, device, w):
        from dynoplan_amd import expander as E
        self.fake, self.device = fake, device
        self.calls = 0
        fake.hipSetDevice(1 - device)
        fake.fake_expect(device)
        self.ex = E.GpuExpander(w.desc, device)
        self.note("create")
        self.call("upload_primitives", w.offsets, w.states, w.actions)
        self.call("upload_world", w.lo, w.hi, w.boxes, w.spheres)

    def note(self, what):
        buf = C.create_string_buffer(65536)
        n = self.fake.fake_notes(buf, len(buf))
        self.fake.fake_expect(-1)
        self.calls += 1
        if n:
            raise SystemExit(f"{what}, context on device {self.device}:\n{buf.value.decode()}")

    def call(self, name, *args, fails=False, **kw):
        from dynoplan_amd import _native as N
        self.fake.hipSetDevice(1 - self.device)
        self.fake.fake_expect(self.device)
        try:
            return getattr(self.ex, name)(*args, **kw)
        except N.DynoplanError:
            if not fails:
                raise
        finally:
            self.note(name)


def main(lib, case):
    fake = C.CDLL(lib, mode=C.RTLD_GLOBAL)  # ahead of the runtime the library links
    fake.fake_allocations.restype = C.c_longlong
    fake.fake_counter.argtypes = [C.c_int, C.c_longlong, C.c_int]
    sys.path.insert(0, ROOT)
    from dynoplan_amd import _native as N
    from dynoplan_amd import expander as E
    from dynoplan_amd import synth
    slots = counter_slots()
    quad = case == "window overflow"
    if quad:
        w = synth.quadrotor(seed=3, P=64, N_nodes=8, n_visited=1)
    elif case == "select":
        w = synth.unicycle2_small(seed=5)
    else:
        w = synth.unicycle1_small(seed=1, P=64, N_nodes=8, n_visited=0)
    pair = [Driver(fake, d, w) for d in (0, 1)]
    nodes, g, p = w.nodes, w.g_parent, w.params
    n1, g1 = nodes[:1], g[:1]
    if case == "novel append past the capacity":
        for round_ in range(3):  # each append is past the capacity before
            for d in pair:
                fake.fake_counter(slots["DPC_PAIRS"], 4000, 1)
                fake.fake_counter(slots["DPC_NOVEL"], 1500 << round_, 1)
                d.call("expand", n1 if round_ else nodes, g1 if round_ else g, p)
            for d in pair:
                before = [fake.fake_allocations(k) for k in (0, 1)]
                d.call("visited_append_novel")
                after = [fake.fake_allocations(k) for k in (0, 1)]
                assert after[d.device] > before[d.device] and after[1 - d.device] == before[1 - d.device]
    elif case in ("few nodes", "many nodes"):
        n, gg = (n1, g1) if case == "few nodes" else (nodes, g)
        for d in pair:
            d.call("visited_append", np.repeat(nodes, 200, axis=0))
            d.call("expand", n, gg, p)
            d.call("counts")
            d.call("fetch")
            d.call("upload_nodes", n, gg)
            d.call("expand_async", p)
            d.call("counts")
            d.call("fetch")
            d.call("timing")
            d.call("timing_detail")
            d.call("health")
            d.call("visited_append", nodes)
            d.call("visited_reset")
            d.call("expand", n, gg, p)
            d.call("search", w.nodes[0], w.nodes[1], max_expands=3)
    elif quad:
        p.fp32_rollout = 1
        for slot in ("DPC_WINDOW_OVF", "DPC_NODES_LEFT"):
            for d in pair:
                # read with the batch and still fresh when counts() finds them
                # and has the batch completed
                fake.fake_counter(slots[slot], 1, 1)
                d.call("upload_nodes", n1, g1)
                fake.hipSetDevice(1 - d.device)
                N.check(d.ex.lib.dp_expand_batch(d.ex.ctx, E._dptr(n1), E._dptr(g1), 1, C.byref(p), None))
                d.call("counts")
                d.call("expand", n1, g1, p)
    elif case == "radius":
        for d in pair:
            d.call("visited_append", nodes)
            d.call("visited_radius", nodes, 0.2, idx_cap=4)
            buf = (C.c_int64 * 4096)()
            q = np.ascontiguousarray(nodes)
            fake.hipSetDevice(1 - d.device)
            fake.fake_expect(d.device)
            N.check(d.ex.lib.dp_visited_radius_noalloc(d.ex.ctx, q.ctypes.data, q.shape[0], 0.2, C.addressof(buf),
                                                       C.addressof(buf), 8, None))
            d.note("visited_radius_noalloc")
            d.call("visited_append", np.repeat(nodes, 300, axis=0))
            d.call("visited_radius", nodes, 0.3, idx_cap=4)
    elif case == "select":
        for d in pair:
            for n in (1, 8):
                d.call("expand_select", w.nodes[:n], w.g_parent[:n], w.nodes[:n], 0.4, list(w.nodes[0]))
    elif case == "surrogate":
        for d in pair:
            d.call("surrogate_init")
            d.call("surrogate_train", nodes, p, epochs=1, batch=8, fails=True)  # no pair: no kernel ran
            d.call("surrogate_calibrate", nodes, p)
            p2 = type(p).from_buffer_copy(p)
            p2.use_surrogate = 2
            d.call("expand", nodes, g, p2)
            d.call("surrogate_scores", 4)
    elif case == "batch":
        for d in pair:
            d.call("upload_nodes", nodes, g)
        for mode in (N.BATCH_GRAPH, N.BATCH_STREAMS):
            for d in pair:
                fake.hipSetDevice(1 - d.device)
                fake.fake_expect(d.device)
                b = E.GpuBatch([d.ex], mode)
                d.note("batch create")
                for _ in range(2):
                    fake.hipSetDevice(1 - d.device)
                    fake.fake_expect(d.device)
                    b.expand_async([p])
                    b.latency_ms()
                    d.note("batch expand")
                d.call("counts")
                b.close()
    else:
        for d in pair:
            order = np.arange(w.offsets.size - 1, dtype=np.int32)[::-1].copy()
            d.call("set_order", order)
            d.call("set_order", None)
            d.call("set_constraints", np.array([0.5]), nodes[:1])
            d.call("reserve", 64, 100000)
            d.call("upload_nodes", nodes, g)
            d.call("autotune", p)
            d.call("expand", nodes, g, p)
    print("checked", sum(d.calls for d in pair), "calls")


if __name__ == "__main__":
    main(sys.argv[1], sys.argv[2])
