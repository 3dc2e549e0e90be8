"""f32 contractions on the bf16 matrix cores (gemm_split.hip: each operand
element as three bf16 parts, six exact products a k).

Every output against the float64 product: a sum of K products, each off by
at most 2^-25 |x w| (the dropped parts), accumulated 16 at a time in f32
(K/16 roundings of the running sum, and as many of the five small terms'
2^-8 smaller one), so it lies within 2 gamma_K sum|x w| plus one unit of the
result -- the f32 tiles' own band -- and the bulk far inside it.  Sizes at the
edges of the tiles (128 rows, 192 / 128 / 64 columns, 16- and 32-deep
blocks), in each operand layout, with and without whole vectors, batched,
split in K, with the bias.  Operands with infinities, NaNs and values past
bf16's largest give what the f32 MFMAs give."""
import numpy as np
import pytest

from presk_amd import hip
from presk_amd import lower as L

A, O = L.ax, L.Operand


def nest(kind, m, n, k, batch=1):
    if kind == "nn":
        return L.dot([O(A(("batch", m), k)), O(A(k, n))], "f32")
    if kind == "bias":
        return L.dot([O(A(("batch", m), k)), O(A(k, n)), O(A(n))], "f32", epilogue=(True, A(("batch", m), n)))
    if kind == "nt":
        return L.dot_vjp_l([O(A(("batch", m), k)), O(A(n, k))], "f32")
    if kind == "tn":
        return L.dot_vjp_r([O(A(("batch", k), m)), O(A(("batch", k), n))], "f32")
    if kind == "tt":
        return L.ein([O(A(("k", k), ("m", m))), O(A(("n", n), ("k", k)))], [["k", "m"], ["n", "k"]], ["m", "n"], "f32")
    return L.ein([O(A(("b", batch), ("m", m), ("k", k))), O(A(("b", batch), ("k", k), ("n", n)))],
                 [["b", "m", "k"], ["b", "k", "n"]], ["b", "m", "n"], "f32")


def operands(kind, m, n, k, batch, rng):
    shapes = {"nn": [(m, k), (k, n)], "bias": [(m, k), (k, n), (n,)], "nt": [(m, k), (n, k)], "tn": [(k, m), (k, n)],
              "tt": [(k, m), (n, k)], "batched": [(batch, m, k), (batch, k, n)]}[kind]
    return [rng.standard_normal(s, dtype=np.float32) for s in shapes]


def f64(kind, v):
    a, b = v[0].astype(np.float64), v[1].astype(np.float64)
    a = a.swapaxes(-1, -2) if kind in ("tn", "tt") else a
    b = b.swapaxes(-1, -2) if kind in ("nt", "tt") else b
    return a @ b + (v[2].astype(np.float64) if kind == "bias" else 0.0), np.abs(a) @ np.abs(b)


def run(low, v, want_order="mfma-f32x3-k16"):
    c = hip.Compiled(low.text, "f32", low.lanes, hip.FAST)
    assert c.kind == "gemm" and c.order.startswith(want_order), (c.kind, c.order)
    n = 1
    for a in low.out_axes:
        n *= a.len
    out = hip.DeviceBuffer(4 * n)
    out.upload(np.full(4 * n, 0xFF, np.uint8))
    bufs = [hip.DeviceBuffer.of(x) for x in v]
    c.run([b.ptr for b in bufs] + [out.ptr])
    hip.sync()
    return out.download(np.float32), c


# (rows, columns, K, batch): whole tiles, one past and one short of a tile,
# ragged vectors, the shortest K, K off the blocks, the split plans
SIZES = [(128, 192, 96, 1), (129, 193, 97, 1), (127, 191, 128, 1), (130, 66, 1021, 1), (65, 65, 65 * 2, 1),
         (512, 388, 200, 1), (16384, 384, 100, 1), (384, 384, 4096, 1), (100, 72, 2056, 1), (2048, 1000, 72, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,batch", SIZES)
@pytest.mark.parametrize("kind", ["nn", "bias", "nt", "tn", "tt", "batched"])
def test_product_against_float64(kind, m, n, k, batch):
    hip.init(0)
    batch = 3 if kind == "batched" else 1
    print(f"[split3] {kind} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    v = operands(kind, m, n, k, batch, rng)
    got, _ = run(nest(kind, m, n, k, batch), v)
    want, S = f64(kind, v)
    err = np.abs(got.astype(np.float64).reshape(want.shape) - want)
    gamma = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    bound = 2 * gamma * S + 2.0 ** -23 * (S + np.abs(want))
    assert np.all(err <= bound), f"{np.count_nonzero(~(err <= bound))} outputs outside the band"
    assert np.median(err / bound) < 1 / 64


@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,n,k", [("nn", 256, 384, 256), ("tn", 130, 131, 2050), ("nt", 256, 192, 513)])
def test_infinities_and_nans_as_the_f32_tiles_give_them(kind, m, n, k, monkeypatch):
    hip.init(0)
    print(f"[split3] specials {kind}", flush=True)
    rng = np.random.default_rng(5)
    v = operands(kind, m, n, k, 1, rng)
    flat = v[0].reshape(-1)
    # an infinity, a NaN, values that round past bf16's largest, a zero row's worth of denormals
    flat[rng.integers(0, flat.size, 6)] = [np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-40]
    low = nest(kind, m, n, k)
    got, _ = run(low, v)
    monkeypatch.setenv("PRESK_HIP_GEMM_TILE", "128x128/1")
    want, _ = run(low, v, "mfma-f32-k4")
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(got[np.isinf(got)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert np.count_nonzero(~fin) > 0 and np.allclose(got[fin], want[fin], rtol=1e-4, atol=1e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,n,k", [("nn", 256, 384, 512), ("tn", 130, 131, 2050), ("nt", 200, 130, 513)])
@pytest.mark.parametrize("size", [1e-30, 1e-33, 1e-35, 1e-37, 1e-39, 1e-42])
@pytest.mark.parametrize("small", [0, 1])
@pytest.mark.parametrize("up", [False, True])
def test_small_operands_keep_their_bits(kind, m, n, k, size, small, up):
    """One operand down to f32's subnormals, whose steps bf16 has not, the
    other near one or scaled up to give results near one: the band of the
    sizes above, and for results that are themselves subnormal the rounding
    of each split's sum and of their total to steps of 2^-149."""
    hip.init(0)
    print(f"[split3] {kind} {m}x{n}x{k} at {size} {small} {up}", flush=True)
    rng = np.random.default_rng(m + n + k)
    v = operands(kind, m, n, k, 1, rng)
    v[small] = (v[small] * size).astype(np.float32)
    if up:
        v[1 - small] = (v[1 - small] * min(1 / size, 1e37)).astype(np.float32)
    got, c = run(nest(kind, m, n, k), v)
    want, S = f64(kind, v)
    splits = int(c.order.split("-split")[1]) if "-split" in c.order else 1
    gamma = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    bound = 2 * gamma * S + 2.0 ** -23 * (S + np.abs(want)) + (splits + 1) * 2.0 ** -149
    err = np.abs(got.astype(np.float64).reshape(want.shape) - want)
    assert np.all(err <= bound), f"{np.count_nonzero(~(err <= bound))} outputs outside the band, {np.max(err / bound):.3g} of it"


@pytest.mark.gpu
@pytest.mark.parametrize("kind,m,n,k", [("nn", 256, 384, 512), ("tn", 130, 131, 2050), ("bias", 200, 130, 513)])
@pytest.mark.parametrize("sizes", [(2.0 ** 47, 2.0 ** 47), (2.0 ** 50, 2.0 ** 50), (2.0 ** 110, 1.0), (1.0, 2.0 ** 112), (2.0 ** 123, 2.0 ** -60)])
def test_large_operands_and_sums(kind, m, n, k, sizes):
    """Elements on both sides of 2^112 and sums of 2^96, past which the split
    operands' own sums are not finite and the f32 MFMAs' stand in."""
    hip.init(0)
    print(f"[split3] {kind} {m}x{n}x{k} at {sizes}", flush=True)
    rng = np.random.default_rng(m + n + k)
    v = operands(kind, m, n, k, 1, rng)
    for i in range(2):
        v[i] = (v[i] * np.float32(sizes[i])).astype(np.float32)
    if kind == "bias":
        v[2] = (v[2] * np.float32(sizes[0] * sizes[1])).astype(np.float32)
    got, _ = run(nest(kind, m, n, k), v)
    want, S = f64(kind, v)
    gamma = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    bound = 2 * gamma * S + 2.0 ** -23 * (S + np.abs(want))
    err = np.abs(got.astype(np.float64).reshape(want.shape) - want)
    assert np.all(np.isfinite(got)) and np.all(err <= bound), f"{np.count_nonzero(~(err <= bound))} outputs outside the band"


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("size", [1e-33, 1e-37, 1e-41])
@pytest.mark.parametrize("scale", [1.0, 1e30])
def test_small_activations_of_integer_weights(bits, size, scale):
    """f32 activations are split the same way; the weights' scales multiply
    the finished sum (a rounding each, and one of the sum before them)."""
    from presk_amd import quant as Q
    hip.init(0)
    print(f"[split3] int{bits} at {size} scales {scale}", flush=True)
    m, k, n = 64, 513, 130
    rng = np.random.default_rng(bits)
    qt = Q.quantize(rng.standard_normal((k, n)), (k, n), Q.Quant(bits, 0))
    scales = (qt.scales * scale).astype(np.float32)
    x = (rng.standard_normal((m, k)) * size).astype(np.float32)
    low = nest("nn", m, n, k)
    c = hip.Compiled(Q.mark(low.text, 1, Q.of_quant(qt, (k, n))), "f32", low.lanes, hip.FAST)
    assert c.order.startswith("mfma-f32x3-k16"), c.order
    out = hip.DeviceBuffer(4 * m * n)
    ins = [hip.DeviceBuffer.of(x), hip.DeviceBuffer.of(qt.data), out, hip.DeviceBuffer.of(scales)]
    c.run([b.ptr for b in ins])
    hip.sync()
    got = out.download(np.float32).astype(np.float64).reshape(m, n)
    w = qt.dequantize().astype(np.float64).reshape(k, n) * scale
    want, S = x.astype(np.float64) @ w, np.abs(x).astype(np.float64) @ np.abs(w)
    splits = int(c.order.split("-split")[1]) if "-split" in c.order else 1
    gamma = k * 2.0 ** -24 / (1 - k * 2.0 ** -24)
    # (dequantize rounds q s to f32, and the scaled scales are rounded: 2^-23 of S)
    bound = 2 * gamma * S + 2.0 ** -22 * (S + np.abs(want)) + (splits + 1) * 2.0 ** -149
    err = np.abs(got - want)
    assert np.all(err <= bound), f"{np.count_nonzero(~(err <= bound))} outputs outside the band, {np.max(err / bound):.3g} of it"


def test_rule():
    """Which products take the split operands: more than 64 rows and columns,
    K from 96 (65 at 128 columns); named tiles, other types and integer
    weights keep theirs."""
    def order(m, n, k, dt="f32"):
        low = L.dot([O(A(("batch", m), k)), O(A(k, n))], dt)
        return hip.Compiled(low.text, dt, low.lanes, hip.FAST).order
    for m, n, k in [(65, 65, 96), (65, 128, 65), (4096, 1024, 1024), (1999, 777, 1021)]:
        assert order(m, n, k).startswith("mfma-f32x3-k16"), (m, n, k)
    for m, n, k in [(64, 4096, 4096), (4096, 64, 4096), (4096, 1024, 64), (4096, 65, 95), (4096, 127, 95)]:
        assert order(m, n, k).startswith("mfma-f32-k4"), (m, n, k)
    assert order(4096, 1024, 1024, "bf16") == "mfma-k16"
    assert order(4096, 1024, 1024, "e8m15") == "mfma-f32-k4"
