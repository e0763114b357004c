"""GPU parity of the FP32 path (Projection::columns_tiled, tensor.rs:206-269)
that Projection::apply_quantized takes for non-finite inputs (tensor.rs:197-201):
dq8_linear_fp32 (the path itself), dq8_apply (the device picks the path) and the
FFN chain's down projection on a non-finite h.  Finite results are bit-exact
against the oracle; NaN positions must match (NaN payloads are not compared)."""
import numpy as np
import pytest
import torch

import dq8
import dq8o

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def same(got, want):
    got, want = np.asarray(got), np.asarray(want)
    nan = np.isnan(want)
    return got.shape == want.shape and np.array_equal(np.isnan(got), nan) and \
        got[~nan].tobytes() == want[~nan].tobytes()


def oracle_fp32(x, v, s, bias=None, a=None, b=None, scale=0.0, result=None, epilogue=0):
    """columns_tiled over dequantized weights, adapter, store (composed from pinned parts)."""
    vals = dq8o.linear_f32(x, dq8o.dequantize_weights(v, s), bias=bias, threads=8)
    if a is not None:
        delta = dq8o.linear_f32(dq8o.lora_mid(x, a, threads=8), b, threads=8)
        vals = (vals + (np.float32(scale) * delta).astype(np.float32)).astype(np.float32)
    if epilogue == 0:
        return vals
    base = np.asarray(result, np.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        if epilogue == 1:
            return (base + vals).astype(np.float32)
    return np.array([dq8o.silu(o) * e for o, e in zip(base.ravel(), vals.ravel())], np.float32).reshape(vals.shape)


def case(rng, m, k, n, rank=0):
    x = (rng.standard_normal((m, k)) * 2).astype(np.float32)
    v, s = dq8o.quantize_weights((rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    bias = rng.standard_normal(n).astype(np.float32)
    a = b = None
    if rank:
        a = (rng.standard_normal((rank, k)) * 0.05).astype(np.float32)
        b = (rng.standard_normal((n, rank)) * 0.05).astype(np.float32)
    return x, v, s, bias, a, b


SHAPES = [(1, 1, 1, 0), (5, 7, 3, 0), (33, 100, 70, 3), (70, 131, 65, 0), (24, 2048, 96, 16), (130, 257, 200, 8),
          (3, 64, 300, 1), (64, 6144, 40, 0)]


@pytest.mark.parametrize("m,k,n,rank", SHAPES)
@pytest.mark.parametrize("ep", [dq8.WRITE, dq8.ADD, dq8.SWIGLU])
def test_linear_fp32_is_columns_tiled(ctx, m, k, n, rank, ep):
    rng = np.random.default_rng(m * 13 + k + n + rank + ep)
    x, v, s, bias, a, b = case(rng, m, k, n, rank)
    h = ctx.weights_from_quantized(dev(v), dev(s))
    base = (rng.standard_normal((m, n)) * 2).astype(np.float32)
    lora = dq8.Lora(ctx.lora_mid(dev(x), dev(a)), dev(b), 0.75) if rank else None
    got = host(ctx.linear_fp32(h, dev(x), out=dev(base.copy()), bias=dev(bias), lora=lora, epilogue=ep))
    want = oracle_fp32(x, v, s, bias, a, b, 0.75, base, ep)
    assert got.tobytes() == want.tobytes()


def test_linear_fp32_columns_layout(ctx):
    rng = np.random.default_rng(2)
    x, v, s, bias, _, _ = case(rng, 37, 300, 90)
    h = ctx.weights_from_quantized(dev(v), dev(s))
    got = host(ctx.linear_fp32(h, dev(x), bias=dev(bias), layout=dq8.COLUMNS))
    assert got.tobytes() == np.ascontiguousarray(oracle_fp32(x, v, s, bias).T).tobytes()


@pytest.mark.parametrize("m,k,n,rank", [(24, 2048, 96, 0), (130, 257, 200, 8), (48, 6144, 64, 16), (3, 131, 31, 0)])
@pytest.mark.parametrize("bad", [None, np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("ep", [dq8.WRITE, dq8.ADD])
def test_apply_takes_the_path_the_crate_takes(ctx, m, k, n, rank, bad, ep):
    rng = np.random.default_rng(m + k + n + rank)
    x, v, s, bias, a, b = case(rng, m, k, n, rank)
    if bad is not None:
        x[m // 2, k // 3] = bad
    h = ctx.weights_from_quantized(dev(v), dev(s))
    base = rng.standard_normal((m, n)).astype(np.float32)
    lora = dq8.Lora(ctx.lora_mid(dev(x), dev(a)), dev(b), 0.5) if rank else None
    got = host(ctx.apply(h, dev(x), out=dev(base.copy()), bias=dev(bias), lora=lora, epilogue=ep))
    want, fp32 = dq8o.apply(x, v, s, bias=bias, a=a, b=b, scale=0.5, result=base, epilogue=ep, threads=8)
    assert fp32 == (bad is not None)
    assert same(got, want)
    # the same call again (the context flag is reset per call)
    got2 = host(ctx.apply(h, dev(x), out=dev(base.copy()), bias=dev(bias), lora=lora, epilogue=ep))
    assert got2.tobytes() == got.tobytes()


# h from the skinny pair (24 and 130 rows), the mid pair and the wide pair; each
# call twice, with finite calls before and between
@pytest.mark.parametrize("m,inter", [(24, 384), (130, 384), (600, 384), (600, 2048)])
def test_ffn_with_a_non_finite_h_takes_the_fp32_down(ctx, m, inter):
    # qwen.rs:486-492 with h overflowing to infinity: the crate's down
    # projection finds QuantizedInputs::new(h) = None and runs columns_tiled.
    hidden = 256
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, hidden)).astype(np.float32)
    gv, gs = dq8o.quantize_weights((rng.standard_normal((inter, hidden)) * 0.05).astype(np.float32))
    uv, us = dq8o.quantize_weights((rng.standard_normal((inter, hidden)) * 0.05).astype(np.float32))
    dv, ds = dq8o.quantize_weights((rng.standard_normal((hidden, inter)) * 0.05).astype(np.float32))
    gb = np.zeros(inter, np.float32)
    ub = np.zeros(inter, np.float32)
    gb[7], ub[7] = 1e30, 1e30  # column 7 of h: silu(~1e30) * ~1e30 = inf
    G, U, D = (ctx.weights_from_quantized(dev(v), dev(s)) for v, s in ((gv, gs), (uv, us), (dv, ds)))
    q, s = ctx.quantize(dev(x))
    resid0 = rng.standard_normal((m, hidden)).astype(np.float32)
    resid = dev(resid0.copy())
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    h = host(ctx.ffn(G, U, D, q, s, resid, biases=(dev(gb), dev(ub), None), nonfinite=flag))
    gate = dq8o.linear(x, gv, gs, bias=gb, threads=4)
    want_h = dq8o.linear(x, uv, us, bias=ub, result=gate, epilogue=2, threads=4)
    assert np.isinf(want_h[:, 7]).all()
    assert same(h, want_h)
    want_r, fp32 = dq8o.apply(want_h, dv, ds, result=resid0, epilogue=1, threads=8)
    assert fp32
    assert same(host(resid), want_r)
    assert int(host(flag)[0]) == 1
    # finite and non-finite calls after it: each follows its own h
    fh = dq8o.linear(x, uv, us, result=dq8o.linear(x, gv, gs, threads=4), epilogue=2, threads=4)
    fr, fp32 = dq8o.apply(fh, dv, ds, result=resid0, epilogue=1, threads=8)
    assert not fp32
    for bad in (False, True, True, False):
        resid, flag = dev(resid0.copy()), torch.zeros(1, dtype=torch.int32, device="cuda")
        ctx.ffn(G, U, D, q, s, resid, biases=(dev(gb), dev(ub), None) if bad else (None, None, None), nonfinite=flag)
        assert same(host(resid), want_r if bad else fr) and int(host(flag)[0]) == bad


# dq8_apply of a few rows in one launch (quantization and the choice of path
# inside its blocks): the bounds of each instance (rows, chunks, groups, outputs)
# and just past them, a partial last group, widths of no whole vector, an
# unaligned x, the columns layout.
@pytest.mark.parametrize("m,k,n,rank", [(1, 2048, 100, 0), (2, 2048, 33, 16), (4, 2048, 33, 16), (5, 2048, 33, 16),
                                        (8, 512, 40, 0), (9, 64, 40, 0), (3, 1, 1, 0), (5, 67, 17, 3), (2, 2049, 16, 0),
                                        (1, 6144, 40, 5), (1, 6145, 20, 0), (3, 1500, 4100, 0), (2, 1111, 4100, 2)])
@pytest.mark.parametrize("bad", [False, True])
def test_apply_few_rows(ctx, m, k, n, rank, bad):
    rng = np.random.default_rng(m + k + n + rank)
    x, v, s, bias, a, b = case(rng, m, k, n, rank)
    if bad:
        x[m - 1, k - 1] = np.nan
    h = ctx.weights_from_quantized(dev(v), dev(s))
    base = rng.standard_normal((m, n)).astype(np.float32)
    store = torch.empty(m * k + 1, device="cuda")
    for off in (0, 1):
        xd = store[off:off + m * k].view(m, k)
        xd.copy_(dev(x))
        lora = dq8.Lora(ctx.lora_mid(xd, dev(a)), dev(b), 0.5) if rank else None
        for ep in (dq8.WRITE, dq8.ADD, dq8.SWIGLU):
            got = host(ctx.apply(h, xd, out=dev(base.copy()), bias=dev(bias), lora=lora, epilogue=ep))
            want, fp32 = dq8o.apply(x, v, s, bias=bias, a=a, b=b, scale=0.5, result=base, epilogue=ep, threads=8)
            assert fp32 == bad
            assert same(got, want)
        cols = host(ctx.apply(h, xd, bias=dev(bias), lora=lora, layout=dq8.COLUMNS))
        want, _ = dq8o.apply(x, v, s, bias=bias, a=a, b=b, scale=0.5, result=base, epilogue=0, threads=8)
        assert same(cols, np.ascontiguousarray(want.T))


# Columns layout as row chunks (each chunk's rows inside the whole output's columns),
# up to their limit and past it.
@pytest.mark.parametrize("m,k,n", [(40, 2048, 200), (333, 1000, 130), (70, 6144, 33), (81, 256, 7000),
                                   (81, 256, 11100), (319, 130, 2700), (40, 4096, 2300)])
@pytest.mark.parametrize("bad", [False, True])
def test_apply_columns_in_row_chunks(ctx, m, k, n, bad):
    rng = np.random.default_rng(m + k + n)
    x, v, s, bias, a, b = case(rng, m, k, n, 16)
    if bad:
        x[m - 1, 0] = np.inf
    h = ctx.weights_from_quantized(dev(v), dev(s))
    lora = dq8.Lora(ctx.lora_mid(dev(x), dev(a)), dev(b), 0.5)
    got = host(ctx.apply(h, dev(x), bias=dev(bias), lora=lora, layout=dq8.COLUMNS))
    want, fp32 = dq8o.apply(x, v, s, bias=bias, a=a, b=b, scale=0.5, result=np.zeros((m, n), np.float32), epilogue=0,
                            threads=8)
    assert fp32 == bad
    assert same(got, np.ascontiguousarray(want.T))


# The FP32 path inside the blocks of the skinny, posting and mid kernels, finite
# and non-finite inputs in turn: short K with 2, 3, 5, 6 and 7 units of 16 columns
# per block (FP32 tiles of 32 and 64 columns, partial ones and the last block's
# included), one and two row tiles, row chunks; 4-wave blocks of one and two row
# tiles and of 33 to 64 groups; the posting kernel's; the mid kernel's 64 x 64.
@pytest.mark.parametrize("m,k,n,rank", [(24, 2048, 5200, 0), (12, 512, 5200, 16), (16, 70, 8230, 0), (20, 64, 17001, 0),
                                        (17, 72, 20800, 3), (9, 64, 28011, 0), (128, 2048, 2050, 0), (65, 64, 5203, 16),
                                        (24, 4096, 300, 5), (10, 2112, 33, 0), (33, 2304, 100, 16), (24, 512, 300, 0),
                                        (30, 6145, 70, 16), (12, 4224, 40, 0), (100, 512, 300, 5), (513, 96, 65, 16)])
def test_apply_non_finite_inside_the_int8_kernels(ctx, m, k, n, rank):
    rng = np.random.default_rng(m + k + n + rank)
    x, v, s, bias, a, b = case(rng, m, k, n, rank)
    h = ctx.weights_from_quantized(dev(v), dev(s))
    base = rng.standard_normal((m, n)).astype(np.float32)
    bad = x.copy()
    bad[m - 1, k - 1] = np.nan  # the other rows stay finite: the FP32 path's own sums
    for inp in (x, bad, x, bad):
        lora = dq8.Lora(ctx.lora_mid(dev(inp), dev(a)), dev(b), 0.5) if rank else None
        got = host(ctx.apply(h, dev(inp), out=dev(base.copy()), bias=dev(bias), lora=lora, epilogue=dq8.ADD))
        want, fp32 = dq8o.apply(inp, v, s, bias=bias, a=a, b=b, scale=0.5, result=base, epilogue=1, threads=8)
        assert fp32 == (inp is bad)
        assert same(got, want)


# out sharing memory with a finite x: in place, shifted by rows or by part of a
# row, and reaching into x from either side, at the rows that k_apply_few would
# otherwise take and just past them.
@pytest.mark.parametrize("m", [1, 2, 4, 8, 9, 24])
@pytest.mark.parametrize("k,n", [(512, 512), (2048, 2048), (256, 1024), (1024, 96)])
def test_apply_out_overlapping_x(ctx, m, k, n):
    rng = np.random.default_rng(m + k + n)
    x, v, s, bias, _, _ = case(rng, m, k, n)
    h = ctx.weights_from_quantized(dev(v), dev(s))
    want, fp32 = dq8o.apply(x, v, s, bias=bias, result=np.zeros((m, n), np.float32), epilogue=0, threads=8)
    assert not fp32
    for shift in (0, k, -n, 17, -33, (m * k - 1), -(m * n - 1)):  # out starts `shift` floats after x
        lo, hi = min(0, shift), max(m * k, shift + m * n)
        store = torch.zeros(hi - lo, device="cuda")
        xd = store[-lo:m * k - lo].view(m, k)
        out = store[shift - lo:shift - lo + m * n].view(m, n)
        xd.copy_(dev(x))
        ctx.apply(h, xd, out=out, bias=dev(bias))
        assert host(out).tobytes() == want.tobytes(), shift
    if k == n:  # a residual: x + W x into x
        xd = dev(x)
        ctx.apply(h, xd, out=xd, bias=dev(bias), epilogue=dq8.ADD)
        assert host(xd).tobytes() == (x + want).astype(np.float32).tobytes()
