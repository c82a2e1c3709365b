"""vfl_encoder_attention's argument checks and the calls that keep torch's path (CPU)."""

import ctypes
from types import SimpleNamespace

import pytest
import torch

from vflorence_amd import hip_attn
from vflorence_amd._lib import lib
from vflorence_amd.layers.bart import BartEncoderSelfAttention, _runs_fit


def call(segments=((0, 1, 4),), heads=2, dim=64, stride=384, scale=0.125, dtype=1, tokens=4,
         base=1 << 20, out=1 << 21):
    flat = [x for s in segments for x in s]
    return lib.vfl_encoder_attention(base, base + 256, base + 512, stride, out, 128, tokens,
                                     (ctypes.c_int64 * len(flat))(*flat), len(segments), heads,
                                     dim, scale, dtype, None)


@pytest.mark.parametrize("bad", [
    dict(dtype=0), dict(dim=128), dict(heads=0), dict(scale=0.0), dict(stride=100),
    dict(stride=388), dict(base=8), dict(out=(1 << 21) + 4),
    dict(segments=((0, 1, 5),)), dict(segments=((1, 1, 4),)), dict(segments=((-1, 1, 2),)),
    dict(segments=((0, 2, 3),)), dict(segments=((0, 1 << 62, 4),)), dict(segments=((0, -1, 2),)),
])
def test_refused_calls(bad):
    assert call(**bad) < 0 and lib.vfl_last_error()


def test_runs_and_plain_calls():
    assert _runs_fit([(0, 2, 3), (6, 0, 5), (6, 1, 4)], 10)
    assert not _runs_fit([(0, 2, 3)], 5) and not _runs_fit([(3, 1, 2), (0, 1, 2)], 9)
    assert not hip_attn.encoder_attention_fits(torch.zeros(4, 384, dtype=torch.bfloat16), None, 2,
                                               0.125)


def test_runs_given_once(monkeypatch):
    """Runs from a one-shot iterable reach the kernel as the same runs in a list do."""
    seen = []
    monkeypatch.setattr(hip_attn, "encoder_attention_fits", lambda *a: True)
    monkeypatch.setattr(hip_attn, "encoder_attention",
                        lambda qkv, segments, *a: seen.append([tuple(r) for r in segments]))
    runs = [(0, 2, 3), (6, 1, 4)]
    layer, qkv, out = BartEncoderSelfAttention(128, 2), torch.zeros(10, 384), torch.zeros(10, 128)
    layer.attend(qkv, runs, out)
    layer.attend(qkv, iter(runs), out)
    layer.attend(qkv, zip(*zip(*runs)), out)
    layer.attend(qkv, (map(int, r) for r in runs), out)
    assert seen == [runs] * 4


def test_shared_memory_is_seen():
    rows = torch.zeros(12, 512, dtype=torch.bfloat16)
    other = torch.zeros(12, 128, dtype=torch.bfloat16)
    meet = hip_attn._spans_meet
    assert meet(rows[:, :384], rows[:, 128:256]) and meet(rows[:, 256:384], rows[:, :384])
    assert meet(rows[:6, :384], rows[4:, 384:]) and meet(rows[:1], rows[:1])
    assert not meet(rows[:6], rows[6:]) and not meet(rows[6:], rows[:6])
    assert not meet(rows, other) and not meet(other, rows)


def test_current_device(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    for index in (0, 1):
        assert hip_attn.on_current_device(SimpleNamespace(get_device=lambda: index)) == index


def test_modes_are_not_passed_by():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    assert hip_attn.plain_eager()
    with torch.device("cpu"):  # a default device: a function mode that takes no operator
        assert hip_attn.plain_eager()
    for mode in (TorchFunctionMode, TorchDispatchMode):
        with mode():
            assert not hip_attn.plain_eager()
    seen = []
    torch.vmap(lambda x: seen.append(hip_attn.plain_eager()) or x)(torch.zeros(2))
    with torch.autograd.forward_ad.dual_level():
        seen.append(hip_attn.plain_eager())
    assert seen == [False, False] and hip_attn.plain_eager()


def test_runs_of_no_tokens(monkeypatch):
    """A run of no prompts may state any length, as torch's path allows."""
    seen = []
    fake = SimpleNamespace(vfl_encoder_attention=lambda *a: seen.append(a[7][:3 * a[8]]) or 0)
    monkeypatch.setattr(hip_attn, "lib", fake)
    monkeypatch.setattr(hip_attn, "_stream", lambda device: 0)
    qkv, out = torch.zeros(10, 384).bfloat16(), torch.zeros(10, 128).bfloat16()
    runs = [(0, 2, 3), (6, 0, 1000), (6, 1, 4), (10, 0, 1 << 70), (10, 5, 0)]
    assert _runs_fit(runs, 10)
    hip_attn.encoder_attention(qkv, runs, out, 2, 0.125)
    assert seen == [[0, 2, 3, 6, 1, 4]] and out._version == 1  # written in place
    with pytest.raises(TypeError):  # as a slice by it is
        hip_attn.encoder_attention(qkv, [(0, 1, 4.5)], out, 2, 0.125)


@pytest.mark.parametrize("dtype, count, length, kernel", [
    (torch.bfloat16, 64, 16, True), (torch.bfloat16, 65, 16, False), (torch.bfloat16, 65, 17, True),
    (torch.float16, 170, 1, True), (torch.float16, 171, 1, False), (torch.float16, 342, 17, False),
    (torch.float16, 342, 33, True), (torch.bfloat16, 342, 17, True),
])
def test_many_short_prompts(monkeypatch, dtype, count, length, kernel):
    """12 heads: one run of many short prompts keeps torch's path, two runs do not."""
    seen = []
    monkeypatch.setattr(hip_attn, "encoder_attention_fits", lambda *a: True)
    monkeypatch.setattr(hip_attn, "encoder_attention", lambda *a: seen.append(a))
    layer, rows = BartEncoderSelfAttention(768, 12).to(dtype), count * length
    qkv, out = torch.zeros(rows + 1, 2304, dtype=dtype), torch.zeros(rows + 1, 768, dtype=dtype)
    layer.attend(qkv, [(0, count, length), (rows, 0, 9)], out)
    assert len(seen) == kernel
    layer.attend(qkv, [(0, count, length), (rows, 1, 1)], out)
    assert len(seen) == kernel + 1
    if length == 1:
        with torch.no_grad():
            layer.attention(torch.zeros(count, length, 768, dtype=dtype))
        assert len(seen) == 2 * kernel + 1
