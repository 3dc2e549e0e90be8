"""Runs of elementwise launches that a recorded graph issues as one printed
kernel: every output of every launch byte for byte as the launches give it
one by one, infinities and NaN among the inputs (of a NaN only that it is one
in FAST mode: its sign is that of whichever operand the compiler put first).  The runs are formed and
broken where they can go wrong: rows broadcast, a value read twice or by a
later launch, an earlier output read at another index (a row of it), buffers
that a later launch overwrites, runs longer than one kernel takes, an overflow
flag, a last axis that is no whole vector, element counts below the
vectorised nests'."""
import ctypes

import numpy as np
import pytest

from presk_amd import hip
from presk_amd import lower as L
from presk_amd.program import BYTES
from tests import fmt

A, O = L.ax, L.Operand


def runs(r, c):
    """name -> [(lowered nest of (r, c), input names, output name)]"""
    m, row, col = A(("batch", r), ("model", c)), A(("model", c)), A(("batch", r))

    def two(op, x, y, o, ay=m):
        return lambda dt: (L.elementwise_binary(op, [O(m), O(ay)], dt), [x, y], o)

    def one(op, x, o):
        return lambda dt: (L.unary(op, [O(m)], dt), [x], o)

    def sums(x, o):
        return lambda dt: (L.reduce_axis("sum", "model", [O(m)], dt), [x], o)

    return {
        "chain": [two("add", "x", "y", "a"), one("neg", "a", "b"), two("mul", "b", "a", "c"), two("sub", "c", "row", "d", row)],
        "columns": [two("add", "x", "col", "a", col), one("exp", "a", "b"), two("div", "b", "x", "c"), two("mul", "a", "c", "d")],
        "apart": [two("add", "x", "y", "a"), one("neg", "y", "b"), two("mul", "b", "a", "c"), sums("c", "s"),
                  two("sub", "c", "s", "d", col), one("gelu", "d", "e")],
        # the next launch reads elements another thread wrote
        "shifted": [two("add", "x", "y", "a"), two("mul", "x", "a", "b", row), one("neg", "b", "c")],
        # a later launch writes what an earlier one read, or wrote
        "reused": [two("add", "x", "y", "a"), one("neg", "a", "b"), two("mul", "b", "b", "a"), two("sub", "a", "b", "y2"),
                   one("sqrt", "y2", "b")],
        # three runs of one graph, the first two the same kernels
        "thrice": [two("add", "x", "y", "a"), one("neg", "a", "b"), two("add", "y", "x", "c"), one("neg", "c", "d"),
                   two("mul", "x", "y", "e"), two("sub", "e", "row", "f", row)],
        "long": [one("neg", "x", "a0")] + [two("add", f"a{j}", "y", f"a{j + 1}") for j in range(9)],
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name,r,c,dt,mode", [
    ("chain", 1024, 520, "f32", hip.FAST), ("chain", 1027, 512, "bf16", hip.FAST), ("chain", 4096, 136, "f16", hip.FAST),
    ("chain", 1024, 520, "f32", hip.EXACT), ("chain", 2000, 131, "f32", hip.FAST), ("chain", 16, 8, "f32", hip.FAST),
    ("columns", 1024, 520, "f32", hip.FAST), ("columns", 1027, 512, "bf16", hip.EXACT), ("columns", 1027, 512, "f16", hip.FAST),
    ("apart", 1027, 512, "bf16", hip.FAST), ("apart", 1024, 520, "f32", hip.EXACT), ("shifted", 1027, 512, "f32", hip.FAST),
    ("shifted", 1100, 512, "bf16", hip.FAST), ("reused", 1027, 512, "f32", hip.FAST), ("reused", 1100, 512, "f16", hip.FAST),
    ("thrice", 1024, 520, "f32", hip.FAST), ("thrice", 1027, 512, "f16", hip.FAST),
    ("long", 1024, 520, "f32", hip.FAST), ("long", 1027, 512, "bf16", hip.FAST)])
def test_a_recorded_run_of_elementwise_launches(name, r, c, dt, mode):
    print(f"[chain] {name} {r} x {c} {dt} mode {mode}", flush=True)
    rng = np.random.default_rng(7)
    special = name != "columns" or dt != "f16"
    sizes = {"x": r * c, "y": r * c, "row": c, "col": r}
    host = {}
    for q, n in sizes.items():
        v = rng.standard_normal(n).astype(np.float32)
        if special:
            v[rng.integers(0, n, 3)] = np.nan, np.inf, -np.inf
        elif q == "col":
            v[: r // 2] = 12.0    # exp past f16's largest value: the overflow flag is raised
        host[q] = fmt.encode(v, dt)
    steps = [f(dt) for f in runs(r, c)[name]]
    # a launch that reads the first row of an earlier output reads c elements of it
    dev = {q: hip.DeviceBuffer(h.nbytes) for q, h in host.items()}
    for q, h in host.items():
        dev[q].upload(h)
    for low, ins, out in steps:
        n = int(np.prod([a.len for a in low.out_axes]))
        if out not in dev:
            dev[out] = hip.DeviceBuffer(n * BYTES[dt])
    flag = hip.DeviceBuffer(4)
    kept, tables, outs = [], [], []
    for low, ins, out in steps:
        k = hip.Compiled(low.text, dt, mode=mode)
        ptrs = [dev[q].ptr for q in ins] + [dev[out].ptr] + ([flag.ptr] if k.guarded else [])
        kept.append(k)
        tables.append((ctypes.c_void_p * len(ptrs))(*ptrs))
        outs.append(out)

    def scribble(byte):
        for o in set(outs):
            dev[o].upload(np.full(dev[o].nbytes, byte, np.uint8))
        flag.zero()
        hip.sync()

    def read():
        hip.sync()
        words = {o: dev[o].download(np.uint32 if dt == "f32" else np.uint16) for o in set(outs)}
        if mode == hip.FAST:
            for o, w in words.items():
                w[np.isnan(fmt.decode(w.view(np.float32) if dt == "f32" else w, dt))] = 0xFFFF
        return {o: w.tobytes() for o, w in words.items()}, int(flag.download(np.uint32)[0])

    scribble(0xA5)
    for k, t in zip(kept, tables):
        hip.check(hip.lib().presk_hip_run(k.handle, t, 0, max(k.split_bound, 0), None))
    want = read()
    b = ctypes.c_void_p()
    hip.check(hip.lib().presk_hip_batch_create(ctypes.byref(b)))
    try:
        for k, t in zip(kept, tables):
            hip.check(hip.lib().presk_hip_batch_add(b, k.handle, t, 0, max(k.split_bound, 0)))
        hip.check(hip.lib().presk_hip_batch_graph(b))
        for rep in range(3):
            scribble(0x5A + rep)
            hip.check(hip.lib().presk_hip_batch_run(b, None))
            got = read()
            bad = [o for o in want[0] if want[0][o] != got[0][o]]
            assert not bad, f"replay {rep}: {bad}"
            assert got[1] == want[1]
    finally:
        hip.lib().presk_hip_batch_release(b)
    if not special and kept[1].guarded:
        assert want[1], "exp past the largest f16 raises the flag"


UNARY = ["neg", "exp", "log", "tanh", "sqrt", "sin", "cos", "abs", "gelu", "gelu_deriv", "relu", "heaviside", "sign", "sigmoid",
         "pow2", "pow3", "pow4", "pow5", "pow6"]


@pytest.mark.gpu
def test_more_runs_than_a_kernel_keeps():
    """Every graph begins with the same kernel; those past the sixteenth run
    that it keeps are launched kernel by kernel, with the same results, and
    recording an earlier one again finds its run."""
    hip.init(0)
    r, c, dt = 1024, 512, "f32"
    m = A(("batch", r), ("model", c))
    rng = np.random.default_rng(3)
    x = np.abs(rng.standard_normal(r * c)).astype(np.float32)
    bx, b0 = hip.DeviceBuffer.of(x), hip.DeviceBuffer(4 * r * c)
    first = hip.Compiled(L.unary("abs", [O(m)], dt).text, dt, mode=hip.FAST)

    def table(*bufs):
        return (ctypes.c_void_p * len(bufs))(*[b.ptr for b in bufs])
    made = []
    for op in UNARY + UNARY[:2]:
        print(f"[chain] abs, {op}", flush=True)
        k, out = hip.Compiled(L.unary(op, [O(m)], dt).text, dt, mode=hip.FAST), hip.DeviceBuffer(4 * r * c)
        steps = [(first, table(bx, b0)), (k, table(b0, out))]
        for q, t in steps:
            hip.check(hip.lib().presk_hip_run(q.handle, t, 0, max(q.split_bound, 0), None))
        hip.sync()
        want = out.download(np.uint32)
        out.upload(np.full(4 * r * c, 0x5A, np.uint8))
        b = ctypes.c_void_p()
        hip.check(hip.lib().presk_hip_batch_create(ctypes.byref(b)))
        made.append((b, steps, k))
        for q, t in steps:
            hip.check(hip.lib().presk_hip_batch_add(b, q.handle, t, 0, max(q.split_bound, 0)))
        hip.check(hip.lib().presk_hip_batch_graph(b))
        for _ in range(2):
            hip.check(hip.lib().presk_hip_batch_run(b, None))
            hip.sync()
            assert np.array_equal(out.download(np.uint32), want), op
    for b, _, _ in made:
        hip.lib().presk_hip_batch_release(b)
