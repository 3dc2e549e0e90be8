"""EXACT mode's tiled contractions (gemm_seq.hip): the interpreter's bits.

Each output is its products' running sum in index order, so the device must
equal the oracle's run of the nest byte for byte -- at the edges of the 16, 32 and
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
    out["dot-mid"] = L.dot([O(A(("batch", 1001), 70)), O(A(70, 328))], dt)     # 32 x 32 ones, the others 16 x 16
    out["dot_vjp_l-mid"] = L.dot_vjp_l([O(A(("batch", 1030), 97)), O(A(193, 97))], dt)
    out["dot_vjp_r-mid"] = L.dot_vjp_r([O(A(("batch", 65), 385)), O(A(("batch", 65), 545))], dt)
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


def edits():
    """(name, text, lanes, type) of nests under a contraction's name that do
    not compute it, or not in its loops: one edit each of what the lowering
    writes, at equal sizes wherever that lets the edit stay in bounds."""
    n = 512

    def each(title, low, dt, changes):
        for what, *pairs in changes:
            text = low.text
            for old, new in pairs:
                assert old in text, (title, what, old, text)
                text = text.replace(old, new)
            assert text != low.text
            yield f"{title}: {what}", text, low.lanes, dt
    sum_loop, rows, columns = "for i2 in 0..512", "for i0 in 0..512", "for i1 in 0..512"
    yield from each("dot_vjp_l", L.dot_vjp_l([O(A(("batch", n), n)), O(A(n, n))], "f32"), "f32", [
        ("half the sum", (sum_loop, "for i2 in 0..256")),
        ("half the rows", (rows, "for i0 in 0..256")),
        ("half the columns", (columns, "for i1 in 0..256")),
        ("one row of %0", ("%0[i0, i2]", "%0[0, i2]")),
        ("one row of %1", ("%1[i1, i2]", "%1[0, i2]")),
        ("one k of %1", ("%1[i1, i2]", "%1[i1, 0]")),
        ("rows exchanged", ("%0[i0, i2]", "%0[i1, i2]"), ("%1[i1, i2]", "%1[i0, i2]")),
        ("%0 transposed", ("%0[i0, i2]", "%0[i2, i0]")),
        ("%1 transposed", ("%1[i1, i2]", "%1[i2, i1]")),
        ("the diagonal of %0", ("%0[i0, i2]", "%0[i0, i0]")),
        ("store transposed", ("%2[i0, i1]", "%2[i1, i0]")),
        ("store of a row's first", ("%2[i0, i1]", "%2[i0, 0]")),
        ("zero above the columns", ("      s0 = 0\n", ""), ("    for i1 in", "    s0 = 0\n    for i1 in")),
        ("from one", ("s0 = 0\n", "s0 = 1\n")),
        # (columns outermost: a partial range of the split loop is of columns)
        ("loops exchanged", (rows, "for iX in 0..512"), (columns, rows), ("for iX in", "for i1 in")),
    ])
    x, w = O(A(("batch", n), n)), O(A(n, n))
    yield from each("dot", L.dot([x, w], "f32"), "f32", [
        ("stores exchanged", ("<v= v0", "<v= vX"), ("<v= v1", "<v= v0"), ("<v= vX", "<v= v1")),
        ("one sum stored twice", ("<v= v1", "<v= v0")),
        ("one column run stored twice", ("%2[i0, ((i1 * 8) + 4)]", "%2[i0, ((i1 * 8) + 0)]")),
        ("columns of %1 exchanged", ("((i1 * 8) + 0)]<v>", "((i1 * 8) + X)]<v>"), ("((i1 * 8) + 4)]<v>", "((i1 * 8) + 0)]<v>"),
         ("((i1 * 8) + X)]<v>", "((i1 * 8) + 4)]<v>")),
        ("half the columns", ("for i1 in 0..64", "for i1 in 0..32")),
        ("overlapping columns", ("(i1 * 8)", "(i1 * 4)")),
        ("one sum twice", ("        s0 = %0[i0, i2]\n        v0", "        s0 = %0[i0, i2]\n        v1 = (v1 + (splat(s0) * %1[i2, ((i1 * 8) + 4)]<v>)<v>)<v>\n        v0")),
        ("one sum not zeroed", ("      v1 = splat(0)\n", "")),
        ("half the sum", (sum_loop, "for i2 in 0..256")),
        ("one k of %0", ("%0[i0, i2]", "%0[i0, 0]")),
    ])
    b = O(A(n))
    yield from each("dot+add f32", L.dot([x, w, b], "f32", epilogue=(True, A(("batch", n), n))), "f32", [
        ("first biases", ("%2[((i1 * 8) + 0)]", "%2[0]"), ("%2[((i1 * 8) + 4)]", "%2[4]")),
        ("a row's bias", ("%2[((i1 * 8) + 0)]<v>", "splat(%2[i0])")),
        ("biases exchanged", ("%2[((i1 * 8) + 0)]", "%2[((i1 * 8) + X)]"), ("%2[((i1 * 8) + 4)]", "%2[((i1 * 8) + 0)]"),
         ("%2[((i1 * 8) + X)]", "%2[((i1 * 8) + 4)]")),
        ("one bias twice", ("v1 = (v1 + %2[((i1 * 8) + 4)]<v>)<v>", "v0 = (v0 + %2[((i1 * 8) + 4)]<v>)<v>")),
    ])
    yield from each("dot+add bf16", L.dot([x, w, b], "bf16", epilogue=(True, A(("batch", n), n))), "bf16", [
        ("a bias elsewhere", ("%2[((i1 * 8) + 3)]", "%2[((i1 * 8) + 2)]")),
        ("a bias twice", ("%3[i0, ((i1 * 8) + 3)] = (%3[i0, ((i1 * 8) + 3)] + %2[((i1 * 8) + 3)])",
                          "%3[i0, ((i1 * 8) + 2)] = (%3[i0, ((i1 * 8) + 2)] + %2[((i1 * 8) + 2)])")),
        ("a column left", ("%3[i0, ((i1 * 8) + 3)] = s3", "%3[i0, ((i1 * 8) + 2)] = s3")),
    ])
    m, j, k = 1030, 65, 130
    low = L.dot([O(A(("batch", m), k)), O(A(k, j)), O(A(j))], "f32", epilogue=(True, A(("batch", m), j)))
    zero = "    for i2 in 0..65 {\n      %3[i0, i2] = 0\n    }\n"
    yield from each("row-wise", low, "f32", [
        ("half the sum", ("for i1 in 0..130", "for i1 in 0..65")),
        ("half the rows", ("for i0 in 0..1030", "for i0 in 0..515")),
        ("half zeroed", ("for i2 in 0..65 {\n      %3[i0, i2] = 0", "for i2 in 0..32 {\n      %3[i0, i2] = 0")),
        ("one row zeroed", ("%3[i0, i2] = 0", "%3[0, i2] = 0")),
        ("one k of %0", ("%0[i0, i1]", "%0[i0, 0]")),
        ("%0 by column", ("%0[i0, i1]", "%0[i1, i1]")),
        ("one k of %1", ("%1[i1, i2]", "%1[0, i2]")),
        ("one bias", ("%2[i2]", "%2[0]")),
        ("one column twice", ("(%3[i0, i2] + (s0", "(%3[i0, 0] + (s0")),
        ("zeroed after", (zero, "    }\n"), ("  for i0 in 0..1030 {\n    }\n", "  for i0 in 0..1030 {\n"),
         ("    for i2 in 0..65 {\n      %3[i0, i2] = (%3[i0, i2] + %2", zero + "    for i2 in 0..65 {\n      %3[i0, i2] = (%3[i0, i2] + %2")),
    ])
    q, kk = O(A(("heads", 2), ("seq", n), ("hd", n))), O(A(("heads", 2), ("seq2", n), ("hd", n)))
    yield from each("ein", L.ein([q, kk], [["heads", "seq", "hd"], ["heads", "seq2", "hd"]], ["heads", "seq", "seq2"], "f32"), "f32", [
        ("half the sum", ("for i3 in 0..512", "for i3 in 0..256")),
        ("half the rows", ("for i1 in 0..512", "for i1 in 0..256")),
        ("half the columns", ("for i2 in 0..512", "for i2 in 0..256")),
        ("one batch entry", ("for i0 in 0..2", "for i0 in 0..1")),
    ])


def test_edited_nests_keep_their_own_loops():
    """A nest is taken for what it computes and not for its name: each of
    these runs as printed."""
    taken = [name for name, text, lanes, dt in edits() if hip.Compiled(text, dt, lanes, hip.EXACT).kind != "generic"]
    assert not taken, taken
