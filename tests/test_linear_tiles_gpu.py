"""The decode-step linear kernels' output tiles: a call's rows have the same bits whatever
tile its size selects, so each call equals the same rows taken 32 (and 16) at a time, the
smaller tiles, whose results the other tests check against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def rand(shape, g, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 129, 161, 193, 255, 257, 321, 385, 449, 512])
@pytest.mark.parametrize("out_f,in_f", [(3072, 1024), (4096, 1024), (3072, 768), (2304, 768),
                                        (1024, 1024), (768, 3072), (1024, 4096), (96, 2560),
                                        (5120, 1280), (1280, 5120)])
@pytest.mark.parametrize("step", [32, 16])
def test_rows_do_not_depend_on_the_tile(dtype, rows, out_f, in_f, step):
    from vflorence_amd import decoder_ops as ops

    g = torch.Generator(device="cuda").manual_seed(rows + out_f)
    x = rand((rows, in_f), g, dtype=dtype)
    w = ops.pack_linear_weight(rand((out_f, in_f), g, in_f**-0.5, dtype))
    bias, res = rand((out_f,), g, dtype=dtype), rand((rows, out_f), g, dtype=dtype)
    gamma, beta = rand((out_f,), g, dtype=dtype), rand((out_f,), g, dtype=dtype)
    u, fb = (torch.randn(out_f, device="cuda", generator=g) for _ in range(2))
    x_stats = torch.rand(rows, in_f // 32, 2, device="cuda", generator=g)
    r_stats = torch.rand(rows, out_f // 32, 2, device="cuda", generator=g)

    def unpack(packed, count):
        t = packed.view(-1, out_f // 32, 4, 16, 8).permute(0, 3, 1, 2, 4)
        return t.reshape(-1, out_f)[:count]

    def calls(at):
        n = x[at].shape[0]
        gelu = ops.LINEAR_GELU | ops.LINEAR_Y_PACKED
        packed_x = torch.zeros((n + 31) // 32 * 32, in_f, dtype=x.dtype, device="cuda")
        packed_x[:n] = x[at]
        packed_x = ops.pack_linear_weight(packed_x)
        residual = (bias, res[at], r_stats[at], gamma, beta, 1e-5, out_f)
        return [ops.linear(x[at], w, bias, out_f), unpack(ops.linear(x[at], w, bias, out_f,
                                                                     flags=gelu), n),
                ops.linear_norm(x[at], x_stats[at], 1e-5, w, u, fb, out_f),
                unpack(ops.linear_norm(x[at], x_stats[at], 1e-5, w, u, fb, out_f, gelu), n),
                *ops.linear_residual(x[at], w, *residual),
                *ops.linear_residual(packed_x, w, *residual, n, ops.LINEAR_X_PACKED)]

    parts = [calls(slice(at, at + step)) for at in range(0, rows, step)]
    for whole, *pieces in zip(calls(slice(0, rows)), *parts):
        assert torch.equal(whole, torch.cat(pieces))
