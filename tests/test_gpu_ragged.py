"""Shapes that are no whole number of 16-byte vectors, and addresses off a
16-byte boundary, on the vector paths: every byte against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gpu_util import activation, bits, f32_equal, say

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "bf16": torch.bfloat16}


def _codec_equals_the_oracle(oracle, x, fmt):
    from elysium_wan_amd import fp8

    raw = bits(x) if x.dtype == torch.bfloat16 else bits(x).astype(np.float32)
    name = "bf16" if x.dtype == torch.bfloat16 else "f32"
    same = np.array_equal if name == "bf16" else f32_equal
    q, k = fp8.quantize(x, fmt)
    oq, ok = oracle.quantize(raw, fmt)
    assert np.array_equal(bits(k).reshape(-1), ok.reshape(-1)), "exponents"
    assert np.array_equal(bits(q).reshape(-1), oq.reshape(-1)), "fp8 bytes"
    assert same(bits(fp8.roundtrip(x, fmt)).reshape(-1), oracle.roundtrip(raw, fmt).reshape(-1)), "round trip"
    for out in ("f32", "bf16"):
        got, want = bits(fp8.dequantize(q, k, DT[out])).reshape(-1), oracle.dequantize(oq, ok, fmt, out).reshape(-1)
        assert (np.array_equal if out == "bf16" else f32_equal)(got, want), f"dequantize {out}"


# one vector and its neighbours, a lane's and a wave's last vector, the edges
# of each kernel's row lengths, and rows past the registers
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("dname", ["bf16", "f32"])
@pytest.mark.parametrize("cols", [3, 4, 5, 7, 8, 9, 15, 17, 255, 511, 513, 1023, 1025, 1601, 3071, 3073, 4095, 4097, 8191, 8193, 12001, 16383, 16385, 24577, 32767, 32769])
def test_rows_of_any_width_equal_the_oracle(oracle, fmt, dname, cols):
    rows = 9 + 2048 // cols
    base = activation((rows * cols + 3,), seed=cols % 89, dtype=DT[dname])
    for off in (0, 1, 3):  # elements off the allocation's boundary
        x = base[off : off + rows * cols].reshape(rows, cols).clone() if off == 0 else base[off : off + rows * cols].reshape(rows, cols)
        if off == 1:  # rows outside the instruction path beside rows inside it
            x[1] = 0.0
            x[2, cols - 1] = float("nan")
            x[3, cols // 2] = float("-inf")
            x[4] *= 2.0**-120
            x[5] *= 2.0**115
        say("fp8 ragged rows", fmt, dname, rows, cols, "offset", off)
        _codec_equals_the_oracle(oracle, x, fmt)


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("cols", [8, 9, 13, 100, 1000, 1025, 1601, 2053])
def test_ragged_dequantize_with_a_distinct_exponent_per_row(oracle, fmt, cols):
    """Every code, neighbouring rows' exponents different and some outside
    the instruction path, so that a vector holding the end of one row and the
    start of the next shows a wrong one; q off its boundary too."""
    _ragged_dequantize_equals_the_oracle(oracle, fmt, cols, max(3, (5 * 1024 + 7) // cols))


# both sides of the number of rows up to which narrow fp32 results go row by row
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("cols", [8, 9, 13, 31, 100, 255, 256, 257])
@pytest.mark.parametrize("rows", [1, 3, 33, 2048, 2049])
def test_ragged_dequantize_of_few_and_of_many_rows(oracle, fmt, cols, rows):
    _ragged_dequantize_equals_the_oracle(oracle, fmt, cols, rows)


def _ragged_dequantize_equals_the_oracle(oracle, fmt, cols, rows):
    from elysium_wan_amd import fp8

    rng = np.random.default_rng(cols)
    codes = ((np.arange(rows * cols, dtype=np.int64) * 37 + 11) % 256).astype(np.uint8)
    kk = rng.integers(-140, 141, rows).astype(np.int32)
    kk[1:][kk[1:] == kk[:-1]] += 1
    for off in (0, 1):
        buf = torch.empty(rows * cols + off, dtype=torch.uint8, device="cuda")
        buf[off:] = torch.from_numpy(codes).cuda()
        q = buf[off:].view(fp8.FORMATS[fmt][0]).reshape(rows, cols)
        k = torch.from_numpy(kk.reshape(rows, 1)).cuda()
        for out in ("f32", "bf16"):
            say("fp8 ragged dequantize", fmt, cols, out, "offset", off)
            d = bits(fp8.dequantize(q, k, DT[out])).reshape(-1)
            od = oracle.dequantize(codes.reshape(rows, cols), kk, fmt, out).reshape(-1)
            assert f32_equal(d, od) if out == "f32" else np.array_equal(d, od)


# per tensor around a vector, a segment (2,048 elements), one block's and every
# block's share of the |x|max launch, and past the sampled guess's 64 MiB
@pytest.mark.parametrize("dname", ["bf16", "f32"])
@pytest.mark.parametrize("n", [32777, 40 * 2048 + 1, 64 * 2048 - 3, 2048 * 2048 + 2047, 2049 * 2048 + 6])
def test_per_tensor_of_any_length_equals_the_oracle(oracle, dname, n):
    base = activation((n + 1,), seed=n % 97, dtype=DT[dname])
    for off in (0, 1):
        x = base[off : off + n]
        say("fp8 ragged per tensor", dname, n, "offset", off)
        _codec_equals_the_oracle(oracle, x.reshape(1, n), "e4m3" if off else "e5m2")


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("dname", ["bf16", "f32"])
@pytest.mark.parametrize("off", [0, 3])
def test_a_ragged_tensor_past_the_guess_size_equals_torch(dname, fmt, off):
    """An odd length of over 64 MiB, its largest value (infinities and NaN
    too) in the vector that overlaps the last whole segment, which the guess
    does not sample, against torch's own ops on this GPU."""
    from elysium_wan_amd import fp8

    dt, (f8, e) = DT[dname], fp8.FORMATS[fmt]
    n = (1 << (25 if dname == "bf16" else 24)) + 2048 + 5
    assert (n // 2048 - 1) % 61 != 0 and (n // 2048) % 61 != 0
    g = torch.Generator(device="cuda").manual_seed(off)
    x = torch.randn(n + off, generator=g, device="cuda").to(dt)[off:]
    for top in (None, 1e4, float("inf"), float("-inf"), float("nan"), "rising"):
        if top == "rising":  # every segment that the guess does not sample exceeds those it does
            x[: n // 2048 * 2048].view(-1, 2048)[::61] *= 2.0**-5
            x[n - 2] = 0.25
        elif top is not None:
            x[n - 2] = top
        say("fp8 ragged guess", dname, fmt, off, top)
        q, k = fp8.quantize(x, fmt, per_tensor=True)
        back = fp8.roundtrip(x, fmt, per_tensor=True)
        amax = x.abs().max().float().cpu()
        # frexp's exponent of an infinity is 0; a NaN maximum scales by 1 (model/fp8.py:36-38)
        kref = 0 if amax.isnan() else -e if amax.isinf() else int(torch.frexp(amax).exponent) - e
        assert int(k) == kref
        qref = (x * torch.tensor(2.0**-kref, dtype=dt, device="cuda")).to(f8)
        assert torch.equal(q.view(torch.uint8), qref.view(torch.uint8))
        want = qref.to(dt) * torch.tensor(2.0**kref, dtype=dt, device="cuda")
        assert torch.equal(torch.nan_to_num(back, nan=7.0), torch.nan_to_num(want, nan=7.0)) and torch.equal(back.isnan(), want.isnan())


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 4099])
def test_cast_fold_and_widen_at_any_address(n):
    """Views off the 16-byte (fp32) and 8-byte (bf16) boundary against torch's
    own cast and adds, and nothing written beside them."""
    from elysium_wan_amd import pieces

    g = torch.Generator(device="cuda").manual_seed(n)
    for off in (0, 1, 2, 3):
        say("pieces at any address", n, off)
        x = torch.randn(n + 8, generator=g, device="cuda")
        h = torch.randn(n + 8, generator=g, device="cuda").bfloat16()
        assert torch.equal(pieces.cast_piece(x[off : off + n], torch.bfloat16), x[off : off + n].bfloat16())
        assert torch.equal(pieces.fold_start(h[off : off + n]), h[off : off + n].float())
        for acc, part in ((x, h), (x, x.flip(0)), (h, x), (h, h.flip(0))):
            got, want = acc.clone(), acc.clone()
            # torch's in-place add into bf16 is the fp32 sum rounded once
            want[off : off + n] = (acc[off : off + n].float() + part[1 : n + 1].float()).to(acc.dtype)
            pieces.fold_add(got[off : off + n], part[1 : n + 1])
            assert torch.equal(got, want)


# lengths around a quad, a wave's step, an 8-element group, both norm tiles
LENGTHS = [1, 2, 3, 4, 5, 7, 8, 9, 63, 255, 256, 257, 511, 513, 4095, 4096, 4097, 12291, 16385]


def _lay(values, packed):
    """The values as views of one buffer, back to back from element 1 on, or
    each in memory of its own."""
    if not packed:
        return [v.clone() for v in values]
    flat = torch.empty(1 + sum(v.numel() for v in values), dtype=values[0].dtype, device="cuda")
    out, o = [], 1
    for v in values:
        out.append(flat[o : o + v.numel()])
        out[-1].copy_(v)
        o += v.numel()
    return out


@pytest.mark.parametrize("gdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("order,fold", [("host", False), ("torch", True)])
def test_packed_step_equals_the_step_over_separate_tensors(gdt, order, fold):
    """Neighbours in one buffer: a lane past its tensor's end would change
    the next tensor's values."""
    from elysium_wan_amd import optim

    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda scale: [torch.randn(n, generator=g, device="cuda") * scale for n in LENGTHS]  # noqa: E731
    p, acc, gr = rnd(0.02), rnd(1e-3), [t.to(gdt) for t in rnd(1e-1)]
    got = []
    for packed in (False, True):
        say("packed step", gdt, order, fold, packed)
        ps = [t.requires_grad_(True) for t in _lay(p, packed)]
        copies = _lay([torch.zeros(n, dtype=torch.bfloat16, device="cuda") for n in LENGTHS], packed)
        opt = optim.FusedAdamW(ps, lr=3e-4, weight_decay=0.1, order=order, max_norm=1.0, working_copy=copies)
        for _ in range(2):
            opt.step(grads=_lay(gr, packed), acc=_lay(acc, packed) if fold else None)
        got.append([t.detach() for t in ps] + copies + [opt.state[i][k] for i in range(len(ps)) for k in ("exp_avg", "exp_avg_sq")] + [opt.grad_norm()])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("gdt", [torch.bfloat16, torch.float32])
def test_packed_clip_equals_the_clip_over_separate_tensors(gdt):
    from elysium_wan_amd import optim

    g = torch.Generator(device="cuda").manual_seed(9)
    values = [(torch.randn(n, generator=g, device="cuda") * 0.1).to(gdt) for n in LENGTHS * 3]  # past the argument table too
    got = []
    for packed in (False, True):
        say("packed clip", gdt, packed)
        ps = [torch.zeros_like(v) for v in values]
        for t, v in zip(ps, _lay(values, packed)):
            t.grad = v
        got.append([optim.clip_grad_norm_(ps, 1.0)] + [t.grad for t in ps])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [1, 3, 7, 8, 9, 255, 511, 513, 1025, 1601])
def test_tied_fold_at_any_width_equals_the_dense_fold(dtype, d):
    """Widths around a vector, a wave's piece and its last, against the dense
    fold in torch's ops; a row's elements past its last vector are folded
    once."""
    from elysium_wan_amd.accumulate import TiedRowFold

    n, m, t = 67, 4, 9
    g = torch.Generator(device="cuda").manual_seed(d)
    hs = [torch.randn(n, d, generator=g, device="cuda").to(dtype) for _ in range(m)]
    ids = [torch.randperm(n, generator=g, device="cuda")[:t].sort().values for _ in range(m)]
    es = [torch.randn(t, d, generator=g, device="cuda").to(dtype) for _ in range(m)]
    say("tied fold width", dtype, d)
    fold = TiedRowFold(n, range(m))
    want = None
    for k in range(m):
        fold.add_head(k, hs[k], ids[k])
        if k:
            fold.add_embed(k - 1, es[k - 1])
        e = torch.zeros(n, d, dtype=dtype, device="cuda")
        e[ids[k]] = es[k]
        want = hs[k] + e if want is None else want + (hs[k] + e)
    fold.add_embed(m - 1, es[m - 1])
    assert torch.equal(fold.result(), want)


# rows of vectors around each block shape's, in lists on both sides of the
# shapes' row counts; 3 more elements leave a tail
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [300, 700, 1100])
@pytest.mark.parametrize("vecs", [1, 63, 64, 65, 128, 129, 256, 257, 448, 449, 512, 513, 768, 769])
def test_tied_fold_in_every_block_shape_equals_the_dense_fold(dtype, n, vecs):
    epv = 8 if dtype == torch.bfloat16 else 4
    for d in (vecs * epv, vecs * epv + 3):
        _tied_fold_equals_the_dense_fold(dtype, n, d)


# past 32 MB, and past the size from which launches stream
@pytest.mark.parametrize("dtype,n,d", [(torch.bfloat16, 9000, 2048), (torch.bfloat16, 17000, 1001), (torch.float32, 9000, 2050), (torch.float32, 9000, 1025),
                                       (torch.float32, 16500, 2051), (torch.bfloat16, 33000, 2053)])
def test_tied_fold_of_large_tables_equals_the_dense_fold(dtype, n, d):
    _tied_fold_equals_the_dense_fold(dtype, n, d)


def _tied_fold_equals_the_dense_fold(dtype, n, d):
    from elysium_wan_amd.accumulate import TiedRowFold

    g = torch.Generator(device="cuda").manual_seed(d)
    t = n - 90
    hs = [torch.randn(n, d, generator=g, device="cuda").to(dtype) for _ in range(2)]
    ids = [torch.randperm(n, generator=g, device="cuda")[:t].sort().values for _ in range(2)]
    es = [torch.randn(t, d, generator=g, device="cuda").to(dtype) for _ in range(2)]
    say("tied fold shapes", dtype, n, d)
    fold = TiedRowFold(n, range(2))
    for k in range(2):
        fold.add_head(k, hs[k], ids[k])
    for k in range(2):
        fold.add_embed(k, es[k])
    parts = []
    for k in range(2):
        e = torch.zeros(n, d, dtype=dtype, device="cuda")
        e[ids[k]] = es[k]
        parts.append(hs[k] + e)
    assert torch.equal(fold.result(), parts[0] + parts[1])
