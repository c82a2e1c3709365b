"""Linear layers on a weight in its own layout (the encoder's small eager projections): the
same bits as the packed kernel, which the other tests check against float64, at the edges
of its tiles; and the calls that stay with torch."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def rand(shape, g, dtype, scale=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 16, 17, 65, 127, 257, 455, 590, 1024])
@pytest.mark.parametrize("out_f,in_f", [(768, 768), (2304, 768), (1024, 1024), (3072, 1024),
                                        (64, 256)])
def test_equals_the_packed_kernel(dtype, rows, out_f, in_f):
    from vflorence_amd import decoder_ops as ops

    g = torch.Generator(device="cuda").manual_seed(rows + out_f)
    x = rand((rows, in_f + 8), g, dtype)[:, :in_f]  # rows with a stride of their own
    w, b = rand((out_f, in_f), g, dtype, in_f**-0.5), rand((out_f,), g, dtype)
    packed = ops.pack_linear_weight(w)
    for bias in (b, None):
        if rows * out_f <= ops.LINEAR_ROWS_MAX_OUTPUTS:
            assert ops.linear_rows_fits(x, w, bias)
        assert torch.equal(ops.linear_rows(x, w, bias), ops.linear(x, packed, bias, out_f))


def test_calls_that_stay_with_torch():
    from vflorence_amd import decoder_ops as ops
    from vflorence_amd.layers.bart import EncoderLinear

    g = torch.Generator(device="cuda").manual_seed(1)
    layer = EncoderLinear(256, 128, device="cuda", dtype=torch.bfloat16)
    wide = rand((40, 264), g, torch.bfloat16)
    x = wide[:, :256]
    fits = lambda t: ops.linear_rows_fits(t, layer.weight, layer.bias)  # noqa: E731
    assert not fits(x)  # the weight's gradient
    assert layer(x).requires_grad
    with torch.no_grad():
        assert fits(x)
        assert not fits(wide[:, 1:257])                     # unaligned rows
        assert not fits(x.t()[:40].t().contiguous().t())    # not rows of the weight's depth
        assert not fits(x.float()) and not fits(x[:0]) and not fits(x[None])
        with torch.autocast("cuda", dtype=torch.float16):
            assert not fits(x) and layer(x).dtype == torch.float16
        for t in (x, wide[:, 1:257], x[None], x[:0]):
            want = F.linear(t, layer.weight, layer.bias)
            got = layer(t)
            assert got.shape == want.shape
            # one rounding apart at most: both sum in 32 bits and round once
            torch.testing.assert_close(got, want, rtol=2**-7, atol=1e-4)
        # vmap rounds the product (below 2 in size here) before it adds the bias: up to
        # half a unit of bf16's last place at 2 more, 2**-8
        mapped = torch.vmap(layer)(x[None])
        torch.testing.assert_close(mapped[0], layer(x), rtol=2**-7, atol=2**-8)
        graph = torch.jit.trace(layer, x).graph
        assert "linear" in str(graph)


@pytest.mark.parametrize("rows, out_f, in_f, kernel", [
    (224, 2304, 768, True), (225, 2304, 768, False), (590, 2304, 768, False),
    (672, 768, 768, True), (673, 768, 768, False), (1024, 768, 768, False),
    (1024, 1024, 1024, True), (320, 3072, 1024, True), (321, 3072, 1024, False),
    (455, 3072, 1024, False), (672, 1536, 512, True), (673, 1536, 512, False),
    (1025, 64, 256, False),
])
def test_sizes_of_the_kernel(rows, out_f, in_f, kernel):
    from vflorence_amd import decoder_ops as ops

    x, w = (torch.empty(n, in_f, dtype=torch.bfloat16, device="cuda") for n in (rows, out_f))
    assert ops.linear_rows_fits(x, w, None) == kernel


@pytest.mark.parametrize("shape", [(3, 45, 256), (2, 3, 7, 256), (1, 1, 256), (0, 4, 256)])
def test_shapes_of_the_same_rows(shape):
    """Equal tokens have equal bits in every shape of the call: prompts of equal length as
    [prompts, tokens, d] and as packed rows."""
    from vflorence_amd import decoder_ops as ops
    from vflorence_amd.layers.bart import BartEncoderSelfAttention

    g = torch.Generator(device="cuda").manual_seed(2)
    layer = BartEncoderSelfAttention(256, 4).cuda().to(torch.bfloat16)
    x, lin = rand(shape, g, torch.bfloat16), layer.out_proj
    rows = x.view(-1, 256)
    with torch.no_grad():
        assert ops.linear_rows_fits(x, lin.weight, lin.bias) == bool(x.numel())
        assert not ops.linear_rows_fits(x.transpose(0, 1), lin.weight, lin.bias) or shape[0] < 2
        assert torch.equal(lin(x), lin(rows).view(shape))
        if len(shape) == 3 and x.numel():
            packed = layer(rows, [(0, *shape[:2])])
            assert torch.equal(layer(x), packed.view(shape))
