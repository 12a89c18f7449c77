"""The any-width Winograd 3x3 convolution (mx_wino3_t16_u) and its three-part
bf16 products: chunks of 16 input channels with a half at the end, partial
output blocks, rows and columns that end inside a block, at odd, even and
4-aligned widths.

Against float64: each of an output's nine groups of transformed sums carries the
transforms' own roundings and at most 6 ceil(ci / 16) of its running sum, each
2^-24; as 2-norms over random data that stays under 3e-8 sqrt(9 ci) of the
result, three times the 8.5e-9 to 1.1e-8 sqrt(9 ci) measured (1.0e-6 at 128
channels; losing the low part of one operand alone gives 2.4e-6 or more).
Operands the parts cannot hold: the block forms direct nine-tap sums instead, so
the largest floats give finite, right outputs and an infinity is an infinity in
the outputs that read it and nothing in the others.
"""

import numpy as np
import pytest

from test_gpu_conv import unfused
from test_gpu_pointwise import check, he, oracle_plan, run_plan

pytestmark = pytest.mark.gpu

CASES = [
    (16, 32, 64, 51, "mx_wino3_t16_u"),
    (40, 33, 90, 31, "mx_wino3_t16_u"),
    (24, 40, 47, 61, "mx_wino3_t16_u"),
    (32, 32, 46, 62, "mx_wino3_t16_u"),
    (128, 64, 37, 60, "mx_wino3_t16_u"),
]


def conv64(x, wt, b):
    co, ci = wt.shape[:2]
    h, w = x.shape[1:]
    p = np.pad(x.astype(np.float64), ((0, 0), (1, 1), (1, 1)))
    y = np.zeros((co, h * w))
    for ky in range(3):
        for kx in range(3):
            y += wt[:, :, ky, kx].astype(np.float64) @ p[:, ky:ky + h, kx:kx + w].reshape(ci, -1)
    return y.reshape(co, h, w) + b[:, None, None].astype(np.float64)


def make(ci, co, h, w):
    from maxim_amd import plan as P
    rng = np.random.default_rng(ci + co + h + w)
    x = rng.standard_normal((ci, h, w)).astype(np.float32)
    wt = he(rng, (co, ci, 3, 3), 9 * ci)
    b = (rng.standard_normal(co) * 0.1).astype(np.float32)
    ops = [P.make_op(P.CONV3X3, dst=1, src=0, w=0, bias=1, c_in=ci, c_out=co, h=h, wd=w),
           P.make_op(P.LRELU, dst=2, src=1, n=co * h * w, slope=0.2)]
    bufs = [(ci, h, w), (co, h, w), (co, h, w)]
    plain = P.CustomPlan(bufs[:2], ops[:1], [wt, b], input=0, output=1)
    act = P.CustomPlan(bufs, ops, [wt, b], input=0, output=2)
    return x, wt, b, plain, act


@pytest.mark.parametrize("ci,co,h,w,kernel", CASES)
def test_against_64_bits(gpu_ok, ci, co, h, w, kernel):
    x, wt, b, plain, act = make(ci, co, h, w)
    got, steps = run_plan(plain, {0: x}, 1)
    want = conv64(x, wt, b)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(steps, "relative error %.2e" % err, flush=True)
    assert steps[0][2] == kernel
    assert err <= 3e-8 * np.sqrt(9 * ci)
    assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max()
    got, steps = run_plan(act, {0: x}, 2)
    assert len(steps) == 1 and steps[0][2] == kernel + "_f_e16"
    assert np.array_equal(got.view(np.uint32), unfused(act, {0: x}, 2).view(np.uint32))


@pytest.mark.parametrize("ci,co,h,w,kernel", CASES)
@pytest.mark.parametrize("bad", [np.float32(3.4e38), np.float32(-3.4e38), np.float32(np.inf), np.float32(np.nan)])
def test_operands_the_parts_cannot_hold(gpu_ok, ci, co, h, w, kernel, bad):
    x, wt, b, plain, _ = make(ci, co, h, w)
    c, r, q = ci - 1, h - 2, w - 3
    x[c, r, q] = bad
    got, _ = run_plan(plain, {0: x}, 1)
    clean = x.copy()
    clean[c, r, q] = 0
    want = conv64(clean, wt, b)
    near = np.zeros((h, w), bool)
    near[max(r - 3, 0):r + 4, max(q - 3, 0):q + 4] = True  # the 2x2 tiles whose 4x4 patches hold it
    assert np.abs(got - want)[:, ~near].max() <= 1e-4 * np.abs(want).max()
    if np.isfinite(bad):
        want = conv64(x, wt, b)
        top = 3.4e38 * np.abs(wt).max()
        assert np.isfinite(got).all() and np.abs(got - want)[:, near].max() <= 1e-5 * top
    else:
        assert not np.isfinite(got[:, r - 1:r + 2, q - 1:q + 2]).any()


@pytest.mark.parametrize("ci,co,h,w,kernel", CASES)
def test_infinities_and_the_largest_floats_as_direct_sums(gpu_ok, ci, co, h, w, kernel):
    """What nine-tap sums give: an infinity is that infinity times a weight in
    the outputs that read it and nothing in the others, opposite infinities and
    NaNs are NaN, and neighbours of opposite sign past half the float range
    (whose difference overflows) leave finite sums finite, within 9 ci roundings
    of 2^-24 of the sum of magnitudes."""
    x, wt, b, plain, _ = make(ci, co, h, w)
    inf = np.float32(np.inf)
    x[0, 3, 5], x[ci - 1, 3, 12], x[1, 3, 13] = inf, -inf, inf  # columns 11..14 read both of the last two
    x[2, 20, 7] = np.nan
    x[3, 30, 9], x[3, 30, 11], x[4, 30, 10] = 3e38, -3e38, 2.9e38
    x[5, 0, 0], x[ci - 2, h - 1, w - 1] = -inf, inf
    got, steps = run_plan(plain, {0: x}, 1)
    assert steps[0][2] == kernel
    with np.errstate(all="ignore"):
        # (no zero weights, and padding is left out: no 0 * inf)
        assert (wt != 0).all()
        want = conv64(np.where(np.isfinite(x), x, 0), wt, b)
        size = conv64(np.where(np.isfinite(x), np.abs(x), 0), np.abs(wt), np.abs(b))
        kinds = [(conv64(m.astype(np.float32), np.where(s, wt > 0, wt < 0).astype(np.float32), 0 * b) +
                  conv64(n.astype(np.float32), np.where(s, wt < 0, wt > 0).astype(np.float32), 0 * b)) > 0
                 for m, n, s in ((x == inf, x == -inf, True), (x == inf, x == -inf, False))]
        nan = conv64(np.isnan(x).astype(np.float32), np.ones_like(wt), 0 * b) > 0
    nan |= kinds[0] & kinds[1]
    want = np.where(nan, np.nan, np.where(kinds[0], np.inf, np.where(kinds[1], -np.inf, want)))
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~nan], want[~fin & ~nan].astype(np.float32))
    # the tiles beside the poisoned ones are Winograd sums, their own products'
    # roundings through the transforms: 1e-4 of the largest ordinary output
    near = size > 1e6
    far, near = fin & ~near, fin & near
    assert (np.abs(got[near] - want[near]) <= (9 * ci + 2) * 2.0 ** -24 * size[near]).all()
    assert np.abs(got[far] - want[far]).max() <= 1e-4 * np.abs(want[far]).max()


@pytest.mark.parametrize("which", ["x", "w"])
@pytest.mark.parametrize("e", [-60, 100, 120])
@pytest.mark.parametrize("ci,co,h,w,kernel", CASES)
def test_operands_of_any_size(gpu_ok, ci, co, h, w, kernel, e, which):
    """2^-e times the input (or the filters) and the bias give 2^-e times the
    outputs, down to subnormal operands: the same bits, but for the rounding of
    outputs that are subnormal floats themselves."""
    from maxim_amd import plan as P
    x, wt, b, plain, _ = make(ci, co, h, w)
    # whole numbers of 2^-18, which stay floats at every e, as do their transforms
    x, wt, b = (np.round(np.clip(a, -8, 8) * np.float32(2 ** 18)) * np.float32(2.0 ** -18) for a in (x, wt, b))
    bufs, ops = [(ci, h, w), (co, h, w)], [P.Op.from_buffer_copy(plain.ops[0])]
    s = np.float32(2.0 ** -e)
    base, _ = run_plan(P.CustomPlan(bufs, ops, [wt, b], input=0, output=1), {0: x}, 1)
    x, wt = (x * s, wt) if which == "x" else (x, wt * s)
    got, steps = run_plan(P.CustomPlan(bufs, ops, [wt, b * s], input=0, output=1), {0: x}, 1)
    assert steps[0][2] == kernel
    diff = np.abs(got.astype(np.float64) * 2.0 ** e - base).max()
    print("largest difference %.1e" % diff, flush=True)
    assert np.abs(base).max() > 1 and diff <= 2.0 ** (e - 150)


@pytest.mark.parametrize("ci,co,h,w,kernel", [
    # few input channels against the implicit GEMM's smallest tile: by the
    # waves of one block per CU (256) of either
    (24, 96, 37, 60, "mx_conv3x3_m32_t4"),    # 60 blocks against 120
    (40, 96, 37, 60, "mx_conv3x3_m32_t4"),
    (24, 320, 52, 100, "mx_conv3x3_m32_t4"),  # 520 (three waves) against 910 (four)
    (24, 160, 33, 92, "mx_wino3_t16_u"),      # 135 against 270 (two)
    (24, 64, 37, 60, "mx_wino3_t16_u"),       # another tile
    (32, 96, 37, 60, "mx_wino3_t16_u"),       # as many input channels as are computed
    (48, 96, 37, 60, "mx_wino3_t16_u"),
])
def test_the_choice_for_few_input_channels(gpu_ok, ci, co, h, w, kernel):
    x, wt, b, plain, _ = make(ci, co, h, w)
    got, steps = run_plan(plain, {0: x}, 1)
    want = conv64(x, wt, b)
    assert steps[0][2] == kernel
    assert np.linalg.norm(got - want) <= 8e-8 * np.sqrt(9 * ci) * np.linalg.norm(want)


@pytest.mark.parametrize("misalign", [0, 1])
@pytest.mark.parametrize("kind", ["add", "gate"])
@pytest.mark.parametrize("ci,co,h,w,kernel", CASES)
def test_fused_epilogues(gpu_ok, ci, co, h, w, kernel, kind, misalign):
    """Conv3x3 -> Add, and Conv3x3 -> Sigmoid -> Mul -> Add (an attention
    gate), as one step of the run-time epilogue: paired operand reads where the
    width is a multiple of 4 and all operands are aligned, one by one at other
    widths, at a right edge that cuts a pair and with the residual one float
    off (misalign). The unfused ops' bits, and the CPU path's values."""
    from maxim_amd import plan as P
    x, wt, b, _, _ = make(ci, co, h, w)
    rng = np.random.default_rng(ci + co + h + w + 1)
    n, y = co * h * w, (co, h, w)
    odd = lambda size: (1, 1, 4 - size % 4)  # up to the next multiple of 4
    X, F, R, OUT = 0, 2, 4, 6
    # all but R start on multiples of 4 floats; R one further with misalign
    bufs = [(ci, h, w), odd(ci * h * w), y, odd(n), y, odd(n + misalign), y, odd(n), y, odd(n), y]
    if misalign:
        bufs[3] = (1, 1, bufs[3][2] + 1)
    T, S = 8, 10
    ops = [P.make_op(P.CONV3X3, dst=T, src=X, w=0, bias=1, c_in=ci, c_out=co, h=h, wd=w)]
    if kind == "add":
        ops += [P.make_op(P.ADD, dst=OUT, src=T, src2=R, n=n)]
    else:
        bufs += [odd(n), y]
        ops += [P.make_op(P.SIGMOID, dst=S, src=T, n=n), P.make_op(P.MUL, dst=12, src=S, src2=F, n=n),
                P.make_op(P.ADD, dst=OUT, src=12, src2=R, n=n)]
    cp = P.CustomPlan(bufs, ops, [wt, b], input=X, output=OUT, align=1)
    assert [int(cp.offs[i]) % 4 for i in (X, F, R, OUT, T)] == [0, 0, misalign, 0, 0]
    inputs = {X: x, F: rng.standard_normal(y).astype(np.float32), R: rng.standard_normal(y).astype(np.float32)}
    got, steps = run_plan(cp, inputs, OUT)
    assert len(steps) == 1 and steps[0][2] == kernel + "_f", steps
    assert np.array_equal(got.view(np.uint32), unfused(cp, inputs, OUT).view(np.uint32))
    check(got, oracle_plan(cp, inputs, OUT), "%s %d->%d @%dx%d" % (kind, ci, co, h, w))
