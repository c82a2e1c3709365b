"""Packed encoder attention (vfl_encoder_attention) against fp64 softmax attention."""

import pytest
import torch

from vflorence_amd import decoder_ops, hip_attn
from vflorence_amd.layers.bart import BartEncoderSelfAttention

pytestmark = pytest.mark.gpu


def reference(qkv, segments, heads):
    """(attention, attention of |v|) per prompt in fp64; rows outside every run are zero."""
    n, d = qkv.shape[0], qkv.shape[1] // 3
    out = torch.zeros(2, n, d, dtype=torch.float64, device=qkv.device)
    for start, count, length in segments:
        for at in range(start, start + count * length, max(length, 1)):
            q, k, v = (t.double().view(length, heads, 64).transpose(0, 1)
                       for t in qkv[at:at + length].chunk(3, dim=-1))
            p = torch.softmax(q @ k.transpose(1, 2).contiguous() / 8, -1)
            for i, x in enumerate((v, v.abs())):
                out[i, at:at + length] = (p @ x.contiguous()).transpose(0, 1).reshape(length, d)
    return out


def check(out, qkv, segments, heads):
    ref, size = reference(qkv, segments, heads)
    # each weight and each output is rounded once, by at most u = 2^-p for p significant
    # bits (8 in bf16, 11 in fp16); fp16 weights below 2^-14 of the
    # largest lose at most 2^-25 each; 2e-5 for the fp32 scores and sums
    u = 2.0**-8 if qkv.dtype == torch.bfloat16 else 2.0**-11
    tiny = max(n for _, _, n in segments) * 2.0**-25 * float(qkv.abs().max())
    bound = 1.05 * u * (size + ref.abs()) + 2e-5 * size + tiny + 1e-6
    err = (out.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads, runs", [
    (1, [(1, 1)]),                                   # one key
    (3, [(2, 31), (1, 32), (1, 33), (3, 64)]),       # edges of the query and key tiles
    (12, [(1, 590)]),                                # two key groups
    (1, [(1, 65)]), (2, [(1, 200)]),                 # as many key groups as key tiles; four
    (2, [(1, 600)]),                                 # four key groups, three steps, the last ragged
    (1, [(1, 1000), (1, 5), (2, 70)]),               # four, of which some see no key
    (12, [(1, 590), (2, 20)]),                       # two, of which one sees no key
    (16, [(4, 129), (1, 127), (2, 128)]),            # two key groups
    (16, [(8, 1000), (0, 7), (5, 65), (3, 0)]),      # one key group; empty runs
    (2, [(1, 1 + 3 * i) for i in range(150)]),       # more runs than one launch holds
])
def test_packed_prompts(dtype, heads, runs):
    g = torch.Generator(device="cuda").manual_seed(heads)
    segments, at = [], 3  # three rows before the first run
    for count, length in runs:
        segments.append((at, count, length))
        at += count * length
    # strided rows; rows that no run names hold NaN, which nothing may read
    qkv = torch.randn(at + 5, 3 * heads * 64 + 8, generator=g, device="cuda").to(dtype)
    qkv = qkv[:, :3 * heads * 64].mul_(2)
    qkv[:3], qkv[at:] = float("nan"), float("nan")
    out = torch.full((at + 5, heads * 64), 7.0, dtype=dtype, device="cuda")
    assert hip_attn.encoder_attention_fits(qkv, out, heads, 0.125)
    hip_attn.encoder_attention(qkv, segments, out, heads, 0.125)
    assert bool((out[:3] == 7).all()) and bool((out[at:] == 7).all())
    check(out[3:at], qkv[3:at], [(s - 3, c, n) for s, c, n in segments], heads)


def test_layer_forms():
    """The layer's three callers agree, and a call with a gradient keeps torch's path."""
    torch.manual_seed(0)
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    x = torch.randn(3, 45, 128, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        a = layer(x)
        b = layer(x.view(-1, 128), [(0, 3, 45)]).view_as(a)
    assert torch.equal(a, b)
    c = layer(x)
    c.float().sum().backward()
    assert layer.qkv_proj.weight.grad is not None
    c = c.detach()
    assert float((a - c).float().norm() / c.float().norm()) < 1e-2  # two bf16 roundings


@pytest.mark.parametrize("third", [0, 1, 2])
def test_output_over_the_projections(third):
    """An output that overlaps q, k or v keeps torch's path: its rows are complete before
    any is stored."""
    g = torch.Generator(device="cuda").manual_seed(third)
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    qkv = torch.randn(700, 384, generator=g, device="cuda").to(torch.bfloat16)
    want, runs = torch.empty(700, 128, dtype=qkv.dtype, device="cuda"), [(0, 1, 600), (600, 2, 50)]
    out = qkv[:, 128 * third:128 * (third + 1)]
    with torch.no_grad():
        assert hip_attn.encoder_attention_fits(qkv, want, 2, 0.125)
        assert not hip_attn.encoder_attention_fits(qkv, out, 2, 0.125)
        before = qkv.clone()
        layer.attend(qkv, runs, out)
    check(out.clone(), before, runs, 2)


def test_tensors_of_another_device(monkeypatch):
    """Neither the attention nor the projections launch their own kernels for tensors of a
    device that is not current."""
    layer = BartEncoderSelfAttention(256, 4).cuda().to(torch.bfloat16)
    x = torch.randn(40, 256, device="cuda").to(torch.bfloat16)
    calls = lambda: (hip_attn.encoder_attention_fits(layer.qkv_proj(x), None, 4, 0.125),  # noqa: E731
                     decoder_ops.linear_rows_fits(x, layer.out_proj.weight, layer.out_proj.bias))
    with torch.no_grad():
        assert calls() == (True, True)
        monkeypatch.setattr(torch.cuda, "current_device", lambda: x.get_device() + 1)
        assert calls() == (False, False)


def test_function_modes_see_the_call():
    from torch.overrides import TorchFunctionMode

    class Names(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.names = set()

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.add(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    layer = BartEncoderSelfAttention(256, 4).cuda().to(torch.bfloat16)
    x = torch.randn(2, 40, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad(), Names() as seen:
        layer(x)
        assert {"linear", "scaled_dot_product_attention"} <= seen.names
        seen.names.clear()
        layer(x.view(-1, 256), [(0, 2, 40)])
        assert {"linear", "scaled_dot_product_attention"} <= seen.names


def test_overlapping_rows():
    """Projections whose rows overlap (expanded, or a window that slides by less than a
    row) keep torch's path instead of the kernel's refusal."""
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    flat = torch.randn(384 * 40, device="cuda").to(torch.bfloat16)
    for qkv in (flat[:384].expand(40, 384), flat.as_strided((40, 384), (8, 1))):
        out = torch.empty(40, 128, dtype=qkv.dtype, device="cuda")
        with torch.no_grad():
            assert not hip_attn.encoder_attention_fits(qkv, out, 2, 0.125)
            layer.attend(qkv, [(0, 1, 40)], out)
        check(out, qkv.contiguous(), [(0, 1, 40)], 2)


def test_empty_run_of_a_long_length():
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    qkv = torch.randn(40, 384, device="cuda").to(torch.bfloat16)
    out = torch.empty(40, 128, dtype=qkv.dtype, device="cuda")
    with torch.no_grad():
        layer.attend(qkv, [(0, 1, 30), (30, 0, 1000), (30, 1, 10)], out)
    check(out, qkv, [(0, 1, 30), (30, 1, 10)], 2)


def test_autocast_type():
    """Under autocast to another type the attention runs in that type, as torch's does."""
    qkv = torch.randn(40, 384, device="cuda").to(torch.float16)
    for dtype in (torch.float16, torch.bfloat16):
        with torch.autocast("cuda", dtype=dtype):
            assert hip_attn.encoder_attention_fits(qkv, None, 2, 0.125) == (dtype == qkv.dtype)


def test_in_place_rules():
    """The write counts as one in place: a tensor saved for a gradient is known to have
    changed, and an inference tensor is written in inference mode only."""
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    qkv, runs = torch.randn(40, 384, device="cuda").to(torch.bfloat16), [(0, 1, 40)]
    w = torch.ones(40, 128, dtype=qkv.dtype, device="cuda", requires_grad=True)
    out = torch.zeros_like(qkv[:, :128])
    y = (w * out).sum()
    with torch.no_grad():
        assert hip_attn.encoder_attention_fits(qkv, out, 2, 0.125)
        layer.attend(qkv, runs, out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    with torch.inference_mode():
        out = torch.zeros_like(out)
        layer.attend(qkv, runs, out)
    check(out.clone(), qkv, runs, 2)
    with torch.no_grad(), pytest.raises(RuntimeError, match="[Ii]nference"):
        layer.attend(qkv, runs, out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads, length", [(1, 40), (2, 70), (2, 300), (12, 300), (16, 700)])
def test_infinities_and_nan(dtype, heads, length):
    """Infinite and NaN queries, keys and values come out where softmax attention has them,
    and stay within their prompt and head; a query whose scores are all -inf is NaN."""
    g = torch.Generator(device="cuda").manual_seed(length)
    # weights far above the least 16-bit number, so that none is 0 against an infinite value
    qkv = (torch.randn(6 * length, 3 * heads * 64, generator=g, device="cuda") / 2).to(dtype)
    inf, nan, d = float("inf"), float("nan"), heads * 64
    at = [slice(i * length, (i + 1) * length) for i in range(6)]
    last = length - 1
    qkv[at[0]][last, 2 * d + 3] = inf            # a value
    qkv[at[1]][0, 2 * d + 5] = nan
    qkv[at[2]][last, d + 1] = inf                # a key: scores of both signs
    qkv[at[3]][1, 2] = nan                       # a query
    qkv[at[4]][:, 0] = 1 + qkv[at[4]][:, 0].abs()
    qkv[at[4]][:, d] = -inf                      # every score of the first head
    segments = [(0, 6, length)]
    out = torch.empty(6 * length, d, dtype=dtype, device="cuda")
    assert hip_attn.encoder_attention_fits(qkv, out, heads, 0.125)
    hip_attn.encoder_attention(qkv, segments, out, heads, 0.125)
    ref, size = reference(qkv, segments, heads)
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    assert torch.equal(out[ref.isinf()] > 0, ref[ref.isinf()] > 0)
    assert bool(ref[at[4]][:, :64].isnan().all()) and bool(ref[at[5]].isfinite().all())
    u = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11  # the bound of check(), finite |v| <= 4
    bound = 1.05 * u * (size + ref.abs()) + 2e-5 * size + length * 2.0**-25 * 4 + 1e-6
    fine = ref.isfinite()
    assert bool(((out.double() - ref).abs()[fine] <= bound[fine]).all())


def test_replays_of_a_captured_launch():
    g = torch.Generator(device="cuda").manual_seed(7)
    layer = BartEncoderSelfAttention(256, 4).cuda().to(torch.bfloat16)
    x, runs = torch.zeros(500, 256, dtype=torch.bfloat16, device="cuda"), [(0, 1, 300), (300, 4, 50)]
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x, runs)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, runs)
        for _ in range(4):
            x.copy_(torch.randn(500, 256, generator=g, device="cuda"))
            want = layer(x, runs)
            torch.cuda.synchronize()
            graph.replay()
            assert torch.equal(out, want)


def test_runs_that_keep_torchs_path():
    """Runs out of order, or that overlap, are taken in the order given."""
    layer = BartEncoderSelfAttention(128, 2).cuda().to(torch.bfloat16)
    qkv = torch.randn(90, 384, device="cuda").to(torch.bfloat16)
    for runs in ([(30, 1, 60), (0, 2, 15)], [(0, 1, 50), (40, 1, 50)]):
        out = torch.empty(90, 128, dtype=qkv.dtype, device="cuda")
        with torch.no_grad():
            assert hip_attn.encoder_attention_fits(qkv, out, 2, 0.125)
            layer.attend(qkv, runs, out)
        check(out, qkv, runs, 2)
