"""EXACT mode's tiled contractions (gemm_seq.hip): the interpreter's bits.

Each output is its products' running sum in index order, so the device must
equal the oracle's run of the nest byte for byte -- at the edges of the 32 and
64 wide tiles and of the 32-deep k-blocks, in every operand layout and storage
type, batched, with the bias, with infinities, NaNs and subnormal products.
Nests whose sums run in another order (a realization's `interleaved` or
`chunked`), and small ones, stay with the printer."""
import numpy as np
import pytest

from oracle import cexec
from presk_amd import hip
from presk_amd import lower as L
from tests import fmt

A, O = L.ax, L.Operand


def nests(dt):
    x = O(A(("batch", 5), ("seq", 131), 97))
    w = O(A(97, 160))
    d = L.dot([x, w], dt)
    out = {"dot": d, "dot+add": L.dot([x, w, O(A(160))], dt, epilogue=(True, d.out_axes))}
    x = O(A(("batch", 1030), 130))
    out["dot-odd"] = L.dot([x, O(A(130, 65))], dt)                      # (row-wise in f32)
    out["dot+add-odd"] = L.dot([x, O(A(130, 65)), O(A(65))], dt, epilogue=(True, A(("batch", 1030), 65)))
    out["dot-wide"] = L.dot([O(A(("batch", 2049), 33)), O(A(33, 1536))], dt)   # 64 x 64 tiles
    out["dot_vjp_l"] = L.dot_vjp_l([O(A(("batch", 3), ("seq", 257), 129)), O(A(96, 129))], dt)
    out["dot_vjp_r"] = L.dot_vjp_r([O(A(("batch", 7), ("seq", 150), 95)), O(A(("batch", 7), ("seq", 150), 100))], dt)
    q = O(A(("batch", 2), ("heads", 3), ("seq", 150), ("hd", 64)))
    k = O(A(("batch", 2), ("heads", 3), ("seq2", 150), ("hd", 64)))
    s = O(A(("batch", 2), ("heads", 3), ("seq", 150), ("seq2", 150)))
    lq, lk, ls = ["batch", "heads", "seq", "hd"], ["batch", "heads", "seq2", "hd"], ["batch", "heads", "seq", "seq2"]
    out["ein-qk"] = L.ein([q, k], [lq, lk], ls, dt)
    out["ein-av"] = L.ein([s, k], [ls, lk], lq, dt)
    out["ein-swapped"] = L.ein([q, s], [lq, ls], lk, dt)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("name", list(nests("f32")))
@pytest.mark.parametrize("special", [False, True])
def test_bits_equal_the_interpreter(name, dt, special):
    from oracle import kernel_text as kt
    low = nests(dt)[name]
    print(f"[seqdot] {name} {dt} special {special}", flush=True)
    k = kt.parse_kernel(low.text)
    rng = np.random.default_rng(17)
    vals = [rng.standard_normal(b.numel).astype(np.float32) for b in k.inputs]
    if special:
        for v in vals[:2]:
            # infinities, a NaN, the largest, products below the smallest normal
            at = rng.integers(0, v.size, 8)
            v[at] = [np.inf, -np.inf, np.nan, 3e38, -3e38, 1e-30, -1e-39, 0.0]
    ins = [fmt.encode(v, dt) for v in vals]
    want, flag = cexec.run(low.text, dt, ins, lanes=low.lanes)
    hip.init(0)
    c = hip.Compiled(low.text, dt, low.lanes, hip.EXACT)
    assert (c.kind, c.order) == ("seqdot", "sequential")
    bufs = [hip.DeviceBuffer.of(a) for a in ins]
    out = hip.DeviceBuffer(want.nbytes)
    out.upload(np.full(want.nbytes, 0xFF, np.uint8))
    f = hip.DeviceBuffer(4)
    f.zero()
    c.run([b.ptr for b in bufs] + [out.ptr] + ([f.ptr] if c.guarded else []))
    hip.sync()
    got = out.download(want.dtype)
    if c.guarded:
        assert bool(f.download(np.uint32, 1)[0]) == flag
    g, r = fmt.decode(got, dt), fmt.decode(want, dt)
    nan = np.isnan(r)
    assert np.array_equal(np.isnan(g), nan)
    # (which operand's NaN a product of two keeps is the instruction's choice)
    assert np.array_equal(got[~nan], want[~nan])


def test_rule():
    """Taken: the nests above in each type; not taken: another order's sums,
    a narrow type's row-wise nest (it rounds at every k), small products."""
    for dt in ("f32", "bf16", "f16"):
        for name, low in nests(dt).items():
            assert hip.Compiled(low.text, dt, low.lanes, hip.EXACT).kind == "seqdot", (name, dt)
    x, w = O(A(("batch", 1024), 512)), O(A(512, 1024))

    def kind(low, dt="f32", text=None):
        return hip.Compiled(text or low.text, dt, low.lanes, hip.EXACT).kind
    assert kind(L.dot([x, w], "f32")) == "seqdot"
    assert kind(L.dot([x, w], "f32", order=("interleaved", 4))) == "generic"
    assert kind(L.dot_vjp_l([x, O(A(1024, 512))], "f32", order=("chunked", 64))) == "generic"
    assert kind(L.dot([O(A(("batch", 240), 96)), O(A(96, 136))], "f32")) == "generic"
    assert kind(L.dot([x, w], "f64"), "f64") == "generic"
    assert kind(L.dot([x, w], "e8m15"), "e8m15") == "generic"
    row_wise = L.dot([O(A(("batch", 2048), 384)), O(A(384, 65))], "f32")
    assert "= 0\n" in row_wise.text and kind(row_wise) == "seqdot"
    narrow = row_wise.text.replace(": f32[", ": bf16[")
    assert kind(row_wise, "bf16", narrow) == "generic"
