"""The streaming GEMMs' products from three-part bf16 operands (mx_pw_*), at
the edges of every form: tiles whose waves share X in fours and twos (_s4, _s2),
each wave its own, the split reduction (_k4) with whole and half chunks of 32
k's, both layouts, ragged columns and rows.

- Against a float64 product: each of the six products of 32 k's is added with
  one rounding of the running sum, so after K / 32 chunks the sum has had at
  most 6 K / 32 roundings of 2^-24 relative to sum |w x|, what the split drops
  is below 3 * 2^-24 of it, and the split reduction and bias add 4 more: the
  bound is (6 ceil(K / 32) + 7) 2^-24 (|W| |X| + |b|). Roundings of random
  data cancel, so the 2-norm of the error is held to 3e-8 sqrt(K) of the
  result's as well, twice the 1.5e-8 sqrt(K) measured: losing the low part of
  one operand gives 2.5e-6 at any K, losing the three smallest of the six
  products 4.4e-6, against 6.8e-7 at the longest reduction here.
- Operands the split cannot hold (infinities, NaN, the largest floats) and
  sums that overflow give what fp32 arithmetic gives: the same infinities and
  NaNs as the CPU path, and the finite outputs within the bound; the outputs
  that they do not reach keep every bit.
- Small operands, subnormal ones too, keep all their bits.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # op, shape, the form expected
    ("conv", (64, 128, 208, 320), "ch2_s4"),   # two stages, four waves share
    ("conv", (32, 64, 180, 364), "ch2_s2"),    # one stage, two waves share, a ragged column tile
    ("conv", (96, 64, 180, 364), "ch2_s2"),    # three stages
    ("conv", (64, 32, 180, 364), "ch2"),       # each wave its own X
    ("conv", (48, 24, 180, 364), "ch2"),       # an odd superstep: half a chunk of zeros
    ("conv", (16, 12, 33, 36), "ch1"),         # half a chunk, a partial weight tile
    ("conv", (64, 40, 13, 20), "ch2_k4"),      # split: a quarter is half a chunk
    ("conv", (192, 40, 13, 20), "ch2_k4"),     # split: quarters of three supersteps, half chunks at either end
    ("conv", (512, 128, 9, 12), "ch2_k4"),     # split: four chunks a quarter
    ("gate0", (32, 256, 280), "chb2_s4"),      # GateMm over tokens, a folded batch
    ("gate0", (33, 64, 1000), "chb2_s2"),      # the same, an odd channel count
    ("gate0", (32, 256, 96), "chb2_k4"),
    ("gate1", (32, 258, 256), "rw2_s4"),       # GateMm over cells, ragged rows
    ("gate1", (16, 2100, 64), "rw2_s2"),
    ("gate1", (3, 37, 64), "rw2_k4"),
]


def _run(op, shape, poison=None, bias=None):
    from maxim_amd import hip as H
    from maxim_amd import plan as P
    rng = np.random.default_rng(sum(shape))
    if op == "conv":
        ci, co, h, w = shape
        x = rng.standard_normal((ci, h, w)).astype(np.float32)
        wt = rng.standard_normal((co, ci)).astype(np.float32)
        b = rng.standard_normal(co).astype(np.float32)
        o = P.make_op(P.CONV1X1, dst=1, src=0, w=0, bias=1, c_in=ci, c_out=co, h=h, wd=w)
        bufs = [(ci, h, w), (co, h, w)]
    else:
        c, outer, inner = shape
        mode = int(op[-1])
        k = outer if mode == 0 else inner
        x = rng.standard_normal((c, outer, inner)).astype(np.float32)
        wt = rng.standard_normal((k, k)).astype(np.float32)
        b = rng.standard_normal(k).astype(np.float32)
        o = P.make_op(P.GATE_MM, dst=1, src=0, w=0, bias=1, c=c, mode=mode, p=[outer, inner])
        bufs = [x.shape, x.shape]
    if poison is not None:
        poison(x, wt, rng)
    b = b if bias is None else bias
    cp = P.CustomPlan(bufs, [o], [wt, b], input=0, output=1)
    gpu = H.Gpu(cp)
    gpu.write_buf(0, x)
    gpu.run_ops(0, 1)
    got = gpu.read_buf(1).reshape(bufs[1])
    kernel = gpu.launches()[0][1]
    gpu.close()
    return x, wt, b, got, kernel


def _sums(op, x, wt, b):
    """The op on float64 (or whatever x and wt are)."""
    with np.errstate(all="ignore"):
        if op == "conv":
            return (wt @ x.reshape(x.shape[0], -1)).reshape(wt.shape[0], *x.shape[1:]) + b[:, None, None]
        if op == "gate0":
            return np.stack([wt @ c for c in x]) + b[:, None]
        return x @ wt.T + b


@pytest.mark.parametrize("op,shape,form", CASES)
def test_split_products_against_64_bits(gpu_ok, op, shape, form):
    x, wt, b, got, kernel = _run(op, shape)
    print(op, shape, kernel, flush=True)
    assert kernel.startswith("mx_pw_" + form), kernel
    want = _sums(op, x.astype(np.float64), wt.astype(np.float64), b.astype(np.float64))
    size = _sums(op, np.abs(x).astype(np.float64), np.abs(wt).astype(np.float64), np.abs(b).astype(np.float64))
    k = wt.shape[1]
    bound = (6 * -(-k // 32) + 7) * 2.0 ** -24 * size
    worst = float((np.abs(got - want) / bound).max())
    rel = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    print("worst share of the bound %.3f, relative error %.1e" % (worst, rel))
    assert worst <= 1.0
    assert rel <= 3e-8 * np.sqrt(k)


@pytest.mark.parametrize("op,shape,form", CASES)
def test_operands_the_split_cannot_hold(gpu_ok, op, shape, form):
    big = np.float32(3.4e38)  # finite, but rounds to infinity in bf16

    def poison(x, wt, rng):
        # [streamed][k]; one poisoned operand per streamed element, so that no
        # sum meets two infinities; one sign of weight, so an infinite input
        # is an infinite sum
        k = wt.shape[1]
        v = x.reshape(k, -1).T if op == "conv" else x.transpose(0, 2, 1).reshape(-1, k) if op == "gate0" else x.reshape(-1, k)
        v = v.copy()
        wt[:] = np.abs(wt) + np.float32(0.5)
        wt[-1, -1] = np.float32(3e38)
        v[:, -1] = np.clip(v[:, -1], -0.5, 0.5)
        bad = [np.inf, -np.inf, np.nan, big, -big, 2e38, 1e30, -1e30]
        at = rng.choice(len(v), 2 * len(bad) + 2, replace=False)
        for n, val in enumerate(bad + bad):
            v[at[n], rng.integers(k - 1)] = np.float32(val)
        v[at[-2], -1], v[at[-1], -1] = 10, -10  # overflows with the last weight
        if op == "conv":
            x[:] = v.T.reshape(x.shape)
        elif op == "gate0":
            x[:] = v.reshape(x.shape[0], x.shape[2], k).transpose(0, 2, 1)
        else:
            x[:] = v.reshape(x.shape)

    x, wt, b, got, kernel = _run(op, shape, poison)
    print(op, shape, kernel, flush=True)
    want = _sums(op, x.astype(np.float64), wt.astype(np.float64), b.astype(np.float64))
    size = _sums(op, np.abs(x).astype(np.float64), np.abs(wt).astype(np.float64), np.abs(b).astype(np.float64))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    # where every partial sum is certainly in range the same value; a sum
    # certainly past the range is infinite; between the two fp32 may do either
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf].astype(np.float32))
    top = float(np.finfo(np.float32).max)
    safe = np.isfinite(want) & (size < 0.5 * top)
    bound = (6 * -(-wt.shape[1] // 32) + 7 + wt.shape[1]) * 2.0 ** -24 * size[safe]
    assert np.isfinite(got[safe]).all() and (np.abs(got[safe] - want[safe]) <= bound).all()
    over = np.isfinite(want) & (np.abs(want) > 1.01 * top) & (np.abs(want) >= 0.9 * size)
    assert over.any() and np.isinf(got[over]).all()


def _columns(op, x):
    """x as [streamed element][k] (a copy)."""
    k = x.shape[0] if op == "conv" else x.shape[1] if op == "gate0" else x.shape[2]
    v = x.reshape(k, -1).T if op == "conv" else x.transpose(0, 2, 1).reshape(-1, k) if op == "gate0" else x.reshape(-1, k)
    return v.copy()


def _put(op, x, v):
    """The inverse of _columns, into x."""
    x[:] = v.T.reshape(x.shape) if op == "conv" else \
        v.reshape(x.shape[0], x.shape[2], -1).transpose(0, 2, 1) if op == "gate0" else v.reshape(x.shape)


def _rows(op, y):
    """An output as [streamed element][weight row]."""
    return y.reshape(y.shape[0], -1).T if op == "conv" else \
        y.transpose(0, 2, 1).reshape(-1, y.shape[1]) if op == "gate0" else y.reshape(-1, y.shape[2])


@pytest.mark.parametrize("op,shape,form", CASES)
def test_sums_that_are_not_finite_leave_the_others(gpu_ok, op, shape, form):
    """Infinite, NaN and overflowing operands change the outputs that they
    reach and no bit of any other, whatever tile it shares with them."""
    def poison(x, wt, rng):
        v = _columns(op, x)
        for n, val in enumerate((np.inf, np.nan, 3.4e38, -np.inf)):
            v[3 + n * 11, n] = val
        wt[2, 1] = np.float32(np.inf)
        _put(op, x, v)

    clean = _run(op, shape)[3]
    got, kernel = _run(op, shape, poison)[3:]
    print(op, shape, kernel, flush=True)
    assert kernel.startswith("mx_pw_" + form), kernel
    a, b = (_rows(op, y).copy() for y in (clean, got))
    hit = np.zeros(a.shape, bool)
    hit[[3, 14, 25, 36]], hit[:, 2] = True, True
    assert not np.isfinite(b[:, 2]).any() and not np.isfinite(b[[3, 14, 36]]).any()
    assert np.array_equal(a[~hit].view(np.uint32), b[~hit].view(np.uint32))


@pytest.mark.parametrize("which", ["x", "w"])
@pytest.mark.parametrize("e", [-70, 100, 120])
@pytest.mark.parametrize("op,shape,form", CASES)
def test_operands_of_any_size(gpu_ok, op, shape, form, e, which):
    """2^-e times the inputs (or weights) and the bias give 2^-e times the
    outputs, down to subnormal operands: the same bits, but for the rounding of
    sums (and of the four partial sums of a split reduction) that are
    subnormal floats themselves, each within half of 2^-149."""
    def grid(a, bits):  # whole numbers of 2^-bits, which stay floats at every e
        return np.round(np.clip(a, -8, 8) * np.float32(2.0 ** bits)) * np.float32(2.0 ** -bits)

    def scaled(s):
        def poison(x, wt, rng):
            x[:], wt[:] = grid(x, 20), grid(wt, 20)
            (x if which == "x" else wt)[:] *= np.float32(s)
        return poison

    rng = np.random.default_rng(sum(shape))
    b = grid(rng.standard_normal({"conv": shape[1], "gate0": shape[1], "gate1": shape[2]}[op]).astype(np.float32), 20)
    base = _run(op, shape, scaled(1.0), b)[3]
    got, kernel = _run(op, shape, scaled(2.0 ** -e), b * np.float32(2.0 ** -e))[3:]
    print(op, shape, kernel, flush=True)
    assert kernel.startswith("mx_pw_" + form), kernel
    diff = np.abs(got.astype(np.float64) * 2.0 ** e - base).max()
    print("largest difference %.1e" % diff)
    assert np.abs(base).max() > 1 and diff <= 5 * 2.0 ** (e - 150)


@pytest.mark.parametrize("kind,ci,co,h,w,form", [
    ("add", 64, 32, 256, 256, "ch1_s2_f"),      # 16-wide tiles, 32-wide when unfused
    ("mul", 64, 32, 256, 256, "ch1_s2_mul_f"),
    ("mul", 128, 128, 128, 160, "ch2_s4_mul_f"),
    ("mul", 128, 64, 20, 28, "ch2_k4_mul_f"),
    ("ln", 64, 128, 180, 364, "ch2_s4_ln_f"),
    ("ln", 48, 24, 256, 260, "ch1_ln_f"),       # an odd superstep
    ("ln", 128, 256, 20, 28, "ch2_k4_ln_f"),
    ("t", 64, 32, 100, 200, "ch2_s4_t"),
    ("t", 128, 16, 20, 28, "ch2_k4_t"),
])
def test_folded_operands_the_split_cannot_hold(gpu_ok, monkeypatch, kind, ci, co, h, w, form):
    """Infinite, NaN and overflowing inputs where the streamed operand is formed
    on the way in (a Mul, a LayerNorm) or the epilogue takes other tiles: the
    unfused ops' bits. The transposed convolution: the CPU path's infinities and
    NaNs, and its other values within the GEMM bar."""
    from maxim_amd import hip as H
    from maxim_amd import plan as P
    from test_gpu_pointwise import fam, he, oracle_plan
    monkeypatch.setenv("MAXIM_PLAN_ORDER", "1")  # fused = unfused to the bit
    rng = np.random.default_rng(ci + co + h)
    n = co * h * w
    x = rng.standard_normal((ci, h, w)).astype(np.float32)
    flat = x.reshape(ci, -1)
    for k, val in enumerate((np.inf, -np.inf, np.nan, 3.4e38, -3e38, 1e35, 1e25)):
        flat[rng.integers(ci), rng.choice(h * w, 2, replace=False)] = np.float32(val)
    b = (rng.standard_normal(co) * 0.1).astype(np.float32)
    X, F, M, T, R, Y = range(6)
    bufs = [x.shape, x.shape, x.shape, (co, h, w), (co, h, w), (co, h, w)]
    conv = dict(dst=T, src=X, w=0, bias=1, c_in=ci, c_out=co, h=h, wd=w)
    add = P.make_op(P.ADD, dst=Y, src=T, src2=R, n=n)
    ws = [he(rng, (co, ci), ci), b]
    if kind == "t":
        bufs, ws = [x.shape, (co, 2 * h, 2 * w)], [he(rng, (ci, co, 2, 2), ci), b]
        ops, Y = [P.make_op(P.CONVT2X2, **dict(conv, dst=1))], 1
    elif kind == "add":
        ops = [P.make_op(P.CONV1X1, **conv), add]
    elif kind == "mul":
        ops = [P.make_op(P.MUL, dst=M, src=X, src2=F, n=x.size), P.make_op(P.CONV1X1, **dict(conv, src=M)), add]
    else:
        ws += [np.ones(ci, np.float32), np.zeros(ci, np.float32)]
        ops = [P.make_op(P.CHAN_LN, dst=M, src=X, scale=2, bias=3, c=ci, hw=h * w),
               P.make_op(P.CONV1X1, **dict(conv, src=M)), add]
    cp = P.CustomPlan(bufs, ops, ws, input=X, output=Y)
    inputs = {X: x}
    if kind != "t":
        inputs.update({F: rng.standard_normal(x.shape).astype(np.float32),
                       R: rng.standard_normal((co, h, w)).astype(np.float32)})
    outs = []
    for fused in (True, False):
        gpu = H.Gpu(cp)
        gpu.set_fusion(fused)
        for k, v in inputs.items():
            gpu.write_buf(k, v)
        gpu.run_ops(0, len(ops))
        outs.append(gpu.read_buf(Y).reshape(cp.bufs[Y]))
        if fused:
            names = [fam(k) for _, k in gpu.launches()]
        gpu.close()
    got, plain = outs
    print(kind, ci, co, h, w, names, "%d not finite" % (~np.isfinite(got)).sum(), flush=True)
    assert "mx_pw_" + form in names
    assert not np.isfinite(got).all() and np.isfinite(got).any()
    assert np.array_equal(np.isnan(got), np.isnan(plain))
    ok = ~np.isnan(got)
    assert np.array_equal(got[ok].view(np.uint32), plain[ok].view(np.uint32))
    if kind == "t":
        with np.errstate(all="ignore"):
            want = oracle_plan(cp, inputs, Y)
        fin = np.isfinite(want)
        assert np.array_equal(got[~fin & ok], want[~fin & ok]) and np.array_equal(np.isnan(got), np.isnan(want))
        small = fin & (np.abs(want) < 1e3)
        assert np.abs(got[small] - want[small]).max() <= 1e-4 * np.abs(want[small]).max()
