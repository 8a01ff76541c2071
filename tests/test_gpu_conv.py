"""Every convolution kernel of the warm-start network with every input and
epilogue that the network gives it, against the same sums in float64: plain or
upsampled-and-joined input; bias and ReLU, with a 2x2 average; the data
gradient's ReLU mask, and its split into a 2x2-summed and a plain part.  And the
weight and bias gradients on both of their tiles.

Bounds, from the arithmetic: a product that passes through n additions in fp32
contributes an error of at most n 2^-23 of its size (room for truncation in the
matrix unit); n is at most 9 Cin for an output, and 512 for a weight gradient (32 in
a matrix instruction, 8 per tile of a split, the row sets and the splits).  A
value rounded to bf16 is off by 2^-8 of it."""
import ctypes as C

import pytest

# (Cin, Cout, level, channels of the upsampled input) of the network's layers
LAYERS = [(32, 32, 0, 0), (32, 32, 0, 0), (32, 64, 1, 0), (64, 64, 1, 0), (64, 96, 2, 0),
          (96, 96, 2, 0), (96, 128, 3, 0), (128, 128, 3, 0), (224, 96, 2, 128), (96, 96, 2, 0),
          (160, 64, 1, 96), (64, 64, 1, 0), (96, 32, 0, 64), (32, 32, 0, 0)]
POOLED = {1, 3, 5}
UNMASKED = {2, 4, 6}           # the input is a pooled map, masked when it is unpooled
# (side, images): between them, all that the network reaches
RUNS = [(256, 1), (256, 4), (256, 16), (8, 3), (40, 13), (40, 256), (8, 128)]


def calls():
    """(Cin, Cout, level, kind, extra) of every convolution call; extra: the
    channels of the upsampled input, or of the summed part of the output"""
    out = []
    for l, (ci, co, lv, up) in enumerate(LAYERS):
        out.append((ci, co, lv, "pool" if l in POOLED else "join" if up else "relu", up))
        if l:
            out.append((co, ci, lv, "split" if up else "none" if l in UNMASKED else "mask", up))
    return sorted(set(out))


def kernel_of(n, side, ci, co):
    import cvtamd
    return cvtamd.lib()._ZN3cvt17nn_conv3x3_kernelEiiiii(n, side, side, ci, co)


def reached(r, n):
    return {(kernel_of(n, r >> lv, ci, co), ci, co, kind) for ci, co, lv, kind, _ in calls()}


def test_runs_hold_all_that_the_network_reaches():
    want = set()
    for r in range(8, 1025, 8):
        for n in list(range(1, 17)) + [24, 32, 64, 128, 256]:
            want |= reached(r, n)
    have = set().union(*(reached(r, n) for r, n in RUNS))
    assert want <= have, sorted(want - have)
    assert {k[0] for k in want} == set(range(9))


class NnConv(C.Structure):
    _fields_ = [("in0", C.c_void_p), ("c0", C.c_int), ("up", C.c_int), ("in1", C.c_void_p),
                ("w", C.c_void_p), ("bias", C.c_void_p), ("relu", C.c_int), ("out", C.c_void_p),
                ("pool", C.c_void_p), ("low", C.c_void_p), ("c_low", C.c_int),
                ("mask", C.c_void_p)]


def ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def conv64(x, w):
    """[tap][Cout][Cin] convolution of (N, H, W, Cin) in float64"""
    import torch
    n, h, wd, ci = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = 0
    for t in range(9):
        y = y + xp[:, t // 3:t // 3 + h, t % 3:t % 3 + wd].reshape(-1, ci) @ w[t].t().contiguous()
    return y.view(n, h, wd, -1)


def sum2(x):
    return x[:, 0::2, 0::2] + x[:, 1::2, 0::2] + x[:, 0::2, 1::2] + x[:, 1::2, 1::2]


GUARD = 4096


def out_buffer(*shape):
    """NaN everywhere, with a guard behind it"""
    import torch
    n = 1
    for s in shape:
        n *= s
    b = torch.full((n + GUARD,), float("nan"), dtype=torch.bfloat16, device="cuda")
    return b, b[:n].view(*shape)


def inputs(g, n, side, ci, up, positive):
    """(in0, in1, the joined input in float64)"""
    import torch

    def make(s, c):
        x = torch.randn(n, s, s, c, device="cuda", generator=g)
        return (x.relu() if positive else x).bfloat16()
    if not up:
        x = make(side, ci)
        return x, None, x.double()
    lo, hi = make(side // 2, up), make(side, ci - up)
    both = torch.cat([lo.repeat_interleave(2, 1).repeat_interleave(2, 2), hi], 3)
    return lo, hi, both.double()


def near(got, ref, err, what):
    d = (got.double() - ref).abs()
    bad = ~(d <= err + 1e-30)                      # (NaN is bad)
    assert not bool(bad.any()), (what, int(bad.sum()), float(d[bad].max()))


@pytest.mark.gpu
@pytest.mark.parametrize("r,n", RUNS)
def test_convolutions(gpu, r, n):
    import torch
    import cvtamd
    lib = cvtamd.lib()
    g = torch.Generator(device="cuda").manual_seed(r * 1000 + n)
    for ci, co, lv, kind, extra in calls():
        side = r >> lv
        what = (n, side, ci, co, kind, "kernel", kernel_of(n, side, ci, co))
        print(what, flush=True)
        forward = kind in ("relu", "pool", "join")
        x0, x1, x = inputs(g, n, side, ci, extra if kind == "join" else 0, forward)
        # the layer's master: [9][its Cout][its Cin], exact in bf16
        lci, lco = (ci, co) if forward else (co, ci)
        w = (torch.randn(9, lco, lci, device="cuda", generator=g) / (9 * ci) ** 0.5).bfloat16().float()
        wf = torch.empty(9 * ci * co, dtype=torch.bfloat16, device="cuda")
        wb = torch.empty_like(wf)
        lib._ZN3cvt15nn_weights_bf16EP12ihipStream_tPKfiiPtS4_(None, ptr(w), lci, lco, ptr(wf), ptr(wb))
        w64 = w.double() if forward else w.double().flip(0).transpose(1, 2)
        bias = torch.randn(co, device="cuda", generator=g) if forward else None
        cl = extra if kind == "split" else 0
        raw, out = out_buffer(n, side, side, co - cl)
        raws = [raw]
        pool = low = mask = None
        if kind == "pool":
            raw, pool = out_buffer(n, side // 2, side // 2, co)
            raws.append(raw)
        if cl:
            raw, low = out_buffer(n, side // 2, side // 2, cl)
            raws.append(raw)
        if kind in ("mask", "split"):
            like = low if cl else out
            mask = torch.randn(like.shape, device="cuda", generator=g).bfloat16()
            mask[..., ::5] = 0.0
        p = NnConv(ptr(x0), extra if kind == "join" else ci, int(kind == "join"), ptr(x1),
                   ptr(wf if forward else wb), ptr(bias), int(forward), ptr(out), ptr(pool),
                   ptr(low), cl, ptr(mask))
        lib._ZN3cvt10nn_conv3x3EP12ihipStream_tRKNS_6NnConvEiiiii(None, C.byref(p), n, side, side,
                                                                   ci, co)
        torch.cuda.synchronize()
        v, s = conv64(x, w64), conv64(x.abs(), w64.abs())
        if forward:
            v, s = (v + bias.double()).relu(), s + bias.double().abs()
        e = 9 * ci * 2.0 ** -23 * s
        full = e + 2.0 ** -8 * (v.abs() + e)       # of a value rounded to bf16
        if kind == "mask":
            keep = mask > 0
            v, full = v * keep, full * keep
        near(out, v[..., cl:], full[..., cl:], what)
        if pool is not None:
            pe = 0.25 * sum2(full) + 2.0 ** -22 * sum2(v.abs())
            pv = 0.25 * sum2(v)
            near(pool, pv, pe + 2.0 ** -8 * (pv.abs() + pe), what)
        if low is not None:
            keep = mask > 0
            pe = sum2(full[..., :cl]) + 2.0 ** -22 * sum2(v[..., :cl].abs())
            pv = sum2(v[..., :cl])
            near(low, pv * keep, (pe + 2.0 ** -8 * (pv.abs() + pe)) * keep, what)
        for raw in raws:
            assert bool(raw[-GUARD:].isnan().all()), what


@pytest.mark.gpu
@pytest.mark.parametrize("r,n", RUNS)
def test_weight_gradients(gpu, r, n):
    import torch
    import cvtamd
    lib = cvtamd.lib()
    g = torch.Generator(device="cuda").manual_seed(r * 1000 + n + 1)
    for ci, co, lv, up in sorted(set(LAYERS)):
        side = r >> lv
        what = (n, side, ci, co, up)
        print(what, flush=True)
        x0, x1, x = inputs(g, n, side, ci, up, True)
        gr = torch.randn(n, side, side, co, device="cuda", generator=g).bfloat16()
        size = co * (9 * ci + 1)
        out = torch.full((size + GUARD,), float("nan"), device="cuda")
        work = torch.empty(lib._ZN3cvt16nn_dw_max_splitsEii(ci, co) * size, device="cuda")
        p = NnConv(ptr(x0), up if up else ci, int(up > 0), ptr(x1))
        lib._ZN3cvt13nn_conv3x3_dwEP12ihipStream_tRKNS_6NnConvEPKtPfS7_iiiii(
            None, C.byref(p), ptr(gr), ptr(out), ptr(work), n, side, side, ci, co)
        torch.cuda.synchronize()
        g2 = gr.double().reshape(-1, co).t().contiguous()
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        for t in range(9):
            xt = xp[:, t // 3:t // 3 + side, t % 3:t % 3 + side].reshape(-1, ci).contiguous()
            near(out[t * co * ci:(t + 1) * co * ci].view(co, ci), g2 @ xt,
                 512 * 2.0 ** -23 * (g2.abs() @ xt.abs()), (what, t))
        near(out[9 * co * ci:size], g2.sum(1), 512 * 2.0 ** -23 * g2.abs().sum(1), (what, "bias"))
        assert bool(out[size:].isnan().all()), what
