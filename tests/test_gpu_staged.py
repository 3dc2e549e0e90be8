"""Contractions staged through registers (gemm_stage.hpp).

16-bit operands whose vectors are not whole, and few rows (gemm_ragged.hip):
the same 32x32x16 MFMAs over the same k-steps as the 128 x 128 tiles, so the
same bits as those give under PRESK_HIP_GEMM_TILE, at the same k-split.

Integer weights (gemm_quant.hip): s sum_k x_k q_k, the products exact in f32
(three of them a k for f32 activations), against the float64 sum of
x_k f32(q_k) s: within 2 gamma_K sum|x w| (one f32 order of K products; the
scale's and the weights' own roundings are 2^-24 each) plus one unit of the
storage type for the sum and for the result."""
import numpy as np
import pytest

from presk_amd import hip
from presk_amd import lower as L
from presk_amd import quant as Q
from tests import fmt

A, O = L.ax, L.Operand
UNIT = {"f32": 2.0 ** -23, "bf16": 2.0 ** -7, "f16": 2.0 ** -10}


def nest(kind, m, n, k, dt):
    if kind == "nn":
        return L.dot([O(A(("batch", m), k)), O(A(k, n))], dt)
    if kind == "bias":
        return L.dot([O(A(("batch", m), k)), O(A(k, n)), O(A(n))], dt, epilogue=(True, A(("batch", m), n)))
    if kind == "nt":
        return L.dot_vjp_l([O(A(("batch", m), k)), O(A(n, k))], dt)
    if kind == "tn":
        return L.dot_vjp_r([O(A(("batch", k), m)), O(A(("batch", k), n))], dt)
    if kind == "tt":
        return L.ein([O(A(("k", k), ("m", m))), O(A(("n", n), ("k", k)))], [["k", "m"], ["n", "k"]], ["m", "n"], dt)
    return L.ein([O(A(("b", 3), ("m", m), ("k", k))), O(A(("b", 3), ("k", k), ("n", n)))],
                 [["b", "m", "k"], ["b", "k", "n"]], ["b", "m", "n"], dt)


def call(c, ins, nbytes, lo=0, hi=None, out=None):
    out = hip.DeviceBuffer(nbytes) if out is None else out
    flag = hip.DeviceBuffer(4)
    flag.zero()
    ptrs = [b.ptr for b in ins[:c.n_inputs]] + [out.ptr] + [b.ptr for b in ins[c.n_inputs:]] + ([flag.ptr] if c.guarded else [])
    c.run(ptrs, lo, hi)
    hip.sync()
    return out, int(flag.download(np.uint32)[0])


# one past and one short of a tile (128, 64, 32 rows or columns) and of a
# k-block, ragged in rows, columns or k alone, the few-row tiles whole and
# ragged, split plans, and sizes below a vector
SIZES = [(129, 65, 77), (127, 193, 129), (1000, 72, 1021), (264, 100, 63), (300, 40, 2050), (5, 136, 520), (32, 1032, 1100),
         (31, 129, 4100), (3, 7, 5), (65, 257, 64), (300, 5, 1100)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("kind,dt,scale", [("nn", "bf16", 1.0), ("nn", "f16", 1.0), ("bias", "bf16", 1.0), ("nt", "bf16", 1.0),
                                           ("tn", "bf16", 1.0), ("tn", "f16", 1.0), ("tt", "bf16", 1.0), ("batched", "bf16", 1.0),
                                           ("bias", "f16", 60.0)])
def test_ragged_and_few_rows_equal_the_tiles(kind, dt, scale, m, n, k, monkeypatch):
    from oracle import kernel_text as kt
    hip.init(0)
    print(f"[staged] {kind} {dt} {m}x{n}x{k}", flush=True)
    low = nest(kind, m, n, k, dt)
    kn = kt.parse_kernel(low.text)
    rng = np.random.default_rng(m + n + k)
    ins = [hip.DeviceBuffer.of(fmt.encode(fmt.roundtrip(scale * rng.standard_normal(b.dims, dtype=np.float32), dt), dt))
           for b in kn.inputs]
    c = hip.Compiled(low.text, dt, low.lanes, hip.FAST)
    assert c.kind == "gemm" and c.order.startswith("mfma-k16"), (c.kind, c.order)
    splits = c.order.split("-split")[1] if "-split" in c.order else "1"
    monkeypatch.setenv("PRESK_HIP_GEMM_TILE", f"128x128/{splits}")
    t = hip.Compiled(low.text, dt, low.lanes, hip.FAST)
    assert t.order == c.order
    poison = np.full(2 * kn.output.numel, 0xFF, np.uint8)
    outs = []
    for kernel in (c, t):
        out = hip.DeviceBuffer(poison.size)
        out.upload(poison)
        outs.append((call(kernel, ins, poison.size, out=out)[0].download(np.uint16), call(kernel, ins, poison.size)[1]))
    assert outs[0][1] == outs[1][1]
    differ = np.count_nonzero(outs[0][0] != outs[1][0])
    assert differ == 0, f"{differ} of {outs[0][0].size} outputs differ from the 128 x 128 tiles'"


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("axes", ["columns", "all", "none"])
@pytest.mark.parametrize("m,n,k", [(130, 66, 97), (70, 67, 130), (129, 193, 97), (65, 191, 96), (257, 384, 97), (40, 1, 33), (5, 2, 70),
                                   (129, 3, 65), (64, 6, 77), (33, 132, 600)])
def test_the_bias_of_the_last_columns(axes, dt, m, n, k):
    """A bias by columns is read in runs of four that end inside it: columns
    at the end of a run's, a tile's and the operand's, and fewer than four."""
    hip.init(0)
    print(f"[staged] bias {axes} {dt} {m}x{n}x{k}", flush=True)
    out_axes = A(("batch", m), n)
    b = {"columns": A(n), "all": out_axes, "none": A()}[axes]
    low = L.dot([O(A(("batch", m), k)), O(A(k, n)), O(b)], dt, epilogue=(True, out_axes))
    rng = np.random.default_rng(m + n + k)
    # small integers: every product and sum is exact, each output's rounding the storage's
    x, w = rng.integers(-3, 4, (m, k)).astype(np.float32), rng.integers(-2, 3, (k, n)).astype(np.float32)
    bias = rng.integers(-64, 65, [a.len for a in b] or [1]).astype(np.float32) / 8
    c = hip.Compiled(low.text, dt, low.lanes, hip.FAST)
    esz = 4 if dt == "f32" else 2
    out, _ = call(c, [hip.DeviceBuffer.of(fmt.encode(v, dt)) for v in (x, w, bias)], esz * m * n)
    got = fmt.decode(out.download(np.float32 if dt == "f32" else np.uint16), dt).reshape(m, n)
    want = fmt.roundtrip(fmt.roundtrip(x @ w, dt) + bias.reshape(bias.shape if axes != "none" else ()), dt)
    assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(140, 70, 77), (129, 71, 1021), (66, 131, 97)])
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("kind", ["nn", "nt", "tn", "tt"])
def test_what_follows_a_ragged_row_reaches_no_other_output(kind, dt, m, n, k):
    """Vectors past a row's end hold the next row's elements: infinities and
    NaN there give NaN in their own rows and columns alone."""
    hip.init(0)
    print(f"[staged] {kind} {dt} {m}x{n}x{k} with NaN", flush=True)
    from oracle import kernel_text as kt
    low = nest(kind, m, n, k, dt)
    rng = np.random.default_rng(m + n + k)
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    rows, cols = [1, m // 2, m - 1], [2, n - 2]
    x[rows[0], 0], x[rows[1], : 3], x[rows[2], k - 1] = np.nan, np.inf, -np.inf
    w[0, cols[0]], w[k - 1, cols[1]] = np.nan, np.inf
    stored = {"nn": (x, w), "nt": (x, w.T), "tn": (x.T, w), "tt": (x.T, w.T)}[kind]
    dims = [tuple(b.dims) for b in kt.parse_kernel(low.text).inputs]
    assert dims == [q.shape for q in stored], dims
    c = hip.Compiled(low.text, dt, low.lanes, hip.FAST)
    out, _ = call(c, [hip.DeviceBuffer.of(fmt.encode(np.ascontiguousarray(q), dt)) for q in stored], (4 if dt == "f32" else 2) * m * n)
    got = fmt.decode(out.download(np.float32 if dt == "f32" else np.uint16), dt).reshape(m, n)
    with np.errstate(invalid="ignore"):
        want = fmt.roundtrip(x, dt).astype(np.float64) @ fmt.roundtrip(w, dt).astype(np.float64)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    assert np.array_equal(np.isnan(got), np.isnan(want))


# name -> (nest, the weights' stored axes, the axis their scales run over, the
# operand marked, its view's axes)
def weights(name, dt, bits, m, k, n):
    if name == "dot":
        return nest("nn", m, n, k, dt), (k, n), 0, (k, n), lambda x, w: x @ w
    if name == "dot+add":
        return nest("bias", m, n, k, dt), (k, n), 0, (k, n), lambda x, w: x @ w
    if name == "dot_vjp_l":
        return nest("nt", m, n, k, dt), (n, k), 1, (n, k), lambda x, w: x @ w.T
    # grouped projections: batch axes of the weights' own, scales a column of each
    low = L.ein([O(A(("batch", 1), ("seq", m), ("model", k))), O(A(("model", k), ("groups", 2), ("hd", n)))],
                [["batch", "seq", "model"], ["model", "groups", "hd"]], ["batch", "groups", "seq", "hd"], dt)
    return low, (k, 2, n), 0, (k, 2, n), lambda x, w: np.einsum("sk,kgn->gsn", x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["dot", "dot+add", "dot_vjp_l", "grouped"])
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("m,k,n", [(8, 512, 256), (1, 1030, 129), (130, 257, 33), (256, 2048, 40)])
def test_integer_weights_against_float64(name, dt, bits, m, k, n):
    hip.init(0)
    print(f"[staged] int{bits} {name} {dt} {m}x{k}x{n}", flush=True)
    low, dims, over, view, product = weights(name, dt, bits, m, k, n)
    rng = np.random.default_rng(m + k + n + bits)
    qt = Q.quantize(rng.standard_normal(dims), dims, Q.Quant(bits, over))
    text = Q.mark(low.text, 1, Q.of_quant(qt, view))
    x = fmt.roundtrip(rng.standard_normal((m, k), dtype=np.float32), dt)
    bias = fmt.roundtrip(rng.standard_normal(n, dtype=np.float32), dt)
    c = hip.Compiled(text, dt, low.lanes, hip.FAST)
    assert c.kind == "gemm" and c.order.startswith("mfma-f32x3-k16" if dt == "f32" else "mfma-k16"), c.order
    ins = [hip.DeviceBuffer.of(fmt.encode(x, dt)), hip.DeviceBuffer.of(qt.data)]
    if name == "dot+add":
        ins.append(hip.DeviceBuffer.of(fmt.encode(bias, dt)))
    ins.append(hip.DeviceBuffer.of(qt.scales))
    w = qt.dequantize().astype(np.float64).reshape(dims)
    want, S = product(x.astype(np.float64), w), product(np.abs(x).astype(np.float64), np.abs(w))
    if name == "dot+add":
        want = (fmt.roundtrip(want.astype(np.float32), dt).astype(np.float64) if dt != "f32" else want) + bias
    esz = 4 if dt == "f32" else 2
    out, _ = call(c, ins, esz * want.size)
    raw = out.download(np.float32 if dt == "f32" else np.uint16)
    got = fmt.decode(raw, dt).astype(np.float64).reshape(want.shape)
    gamma = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    bound = 2 * gamma * S + UNIT[dt] * (S + 2 * np.maximum(np.abs(want), np.abs(got))) + 1e-30
    err = np.abs(got - want)
    assert np.all(err <= bound), f"{np.count_nonzero(~(err <= bound))} outputs outside the band"
    assert np.median(err / bound) < 1 / 16
    # the split loop's pieces give the whole call's bytes
    if c.split_bound > 1:
        part = hip.DeviceBuffer(esz * want.size)
        part.upload(np.full(esz * want.size, 0xFF, np.uint8))
        for t in range(3):
            call(c, ins, 0, c.split_bound * t // 3, c.split_bound * (t + 1) // 3, out=part)
        assert part.download(raw.dtype).tobytes() == raw.tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("name", ["dot", "dot_vjp_l"])
@pytest.mark.parametrize("m,k,n", [(5, 65, 33), (40, 131, 34), (33, 64, 35), (129, 193, 37), (8, 520, 39), (130, 72, 602)])
def test_int4_vectors_from_the_middle_of_a_byte(name, dt, m, k, n):
    """Rows of odd and of even lengths, none a whole vector of eight: vectors
    that start at either half of a byte, and the operand's last ones."""
    test_integer_weights_against_float64(name, dt, 4, m, k, n)


@pytest.mark.gpu
def test_integer_weights_of_infinite_and_large_activations():
    """An infinity or a NaN gives what the loads' own products give, and a
    finite sum stays finite where x q alone passes f32's range."""
    hip.init(0)
    m, k, n, dt = 64, 512, 128, "bf16"
    rng = np.random.default_rng(3)
    qt = Q.quantize(rng.standard_normal((k, n)) * 1e-4, (k, n), Q.Quant(8, 0))
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3, 5], x[7, 9], x[11, 100], x[11, 101] = np.inf, np.nan, 3e38, -3e38
    x = fmt.roundtrip(x, dt)
    low = nest("nn", m, n, k, dt)
    c = hip.Compiled(Q.mark(low.text, 1, Q.of_quant(qt, (k, n))), dt, low.lanes, hip.FAST)
    ins = [hip.DeviceBuffer.of(fmt.encode(x, dt)), hip.DeviceBuffer.of(qt.data), hip.DeviceBuffer.of(qt.scales)]
    got = fmt.decode(call(c, ins, 2 * m * n)[0].download(np.uint16), dt).reshape(m, n)
    w = qt.dequantize().reshape(k, n)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32))
    fin = np.isfinite(want)
    assert np.all(np.isfinite(got[fin])) and fin[11].all()
    rest = np.delete(np.arange(m), [3, 7, 11])
    assert np.allclose(got[rest], want[rest], rtol=2e-2, atol=1e-4) and np.allclose(got[11], want[11], rtol=2e-2, atol=1e33)


def test_rule():
    """Where each path begins: 16-bit sizes off eight, at most 32 rows at K
    of 512 and 128 columns; integer weights from 32 columns to 2 048 rows."""
    def order(m, k, n, dt, bits=0):
        low = nest("nn", m, n, k, dt)
        text = Q.mark(low.text, 1, Q.of_quant_dims(bits, 0, (k, n), (k, n))) if bits else low.text
        return hip.Compiled(text, dt, low.lanes, hip.FAST).order
    for bits in (8, 4):
        assert order(2048, 512, 32, "bf16", bits).startswith("mfma-k16")
        assert order(2048, 512, 32, "f32", bits).startswith("mfma-f32x3-k16")
        for m, n in ((2049, 256), (512, 31)):
            assert order(m, 512, n, "bf16", bits).startswith("mfma-f32-k4")
        assert order(64, 512, 64, "e8m15", bits).startswith("mfma-f32-k4")
    assert order(8, 4096, 4096, "bf16") == "mfma-k16-split8"
    assert order(1999, 1021, 777, "f16") == "mfma-k16"


def test_named_tiles_reach_integer_weights(monkeypatch):
    """PRESK_HIP_GEMM_TILE puts integer weights on the tiles it names, on the
    f32 MFMAs that have them, as it does f32 operands."""
    low = nest("nn", 256, 256, 2048, "bf16")
    text = Q.mark(low.text, 1, Q.of_quant_dims(8, 0, (2048, 256), (2048, 256)))
    assert hip.Compiled(text, "bf16", low.lanes, hip.FAST).order.startswith("mfma-k16")
    monkeypatch.setenv("PRESK_HIP_GEMM_TILE", "128x64/4")
    assert hip.Compiled(text, "bf16", low.lanes, hip.FAST).order == "mfma-f32-k4-split4"
    monkeypatch.setenv("PRESK_HIP_GEMM_TILE", "256x96")
    assert hip.Compiled(text, "bf16", low.lanes, hip.FAST).order == "mfma-f32-k4"
