"""Decode attention over fp32 caches: row groups sharing a table, with and without slot
descriptors, and the fused K/V write, both of the vector kernel, against 64-bit softmax
attention of the same pages, at the edges of blocks, wave splits, group sizes and tables."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BS = 16


def pools(g, blocks, heads, dim):
    return [torch.randn(blocks, heads, BS, dim, device="cuda", generator=g) for _ in range(2)]


def attend(q, k, v, scale):
    """q [rows, heads, D] over one sequence's k, v [heads, tokens, D], in 64 bits."""
    s = torch.einsum("rhd,htd->hrt", q.double(), k.double()) * scale
    return torch.einsum("hrt,htd->rhd", torch.softmax(s, -1), v.double())


def gather(pool, ids, length):
    return pool[ids.long()].transpose(0, 1).flatten(1, 2)[:, :length]


def close(got, want):
    # 32-bit sums over at most 1000 tokens and 128 dims, values of order 1
    torch.testing.assert_close(got.double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("waves", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("descriptors", [False, True])
def test_shared_table_groups(dim, waves, descriptors):
    from vflorence_amd import hip_attn

    g = torch.Generator(device="cuda").manual_seed(dim + waves)
    heads, lens, sizes = 3, [1, 15, 16, 17, 33, 64, 257, 1000, 0], [3, 8, 4, 5, 7, 1, 2, 8, 3]
    rows, width = sum(sizes), 63
    starts = torch.tensor([sum(sizes[:i]) for i in range(len(sizes) + 1)], dtype=torch.int32)
    count = width * len(lens)
    k, v = pools(g, count, heads, dim)
    place = torch.randperm(count, device="cuda", generator=g).int().view(len(lens), width)
    # what a kernel must not read into its results: tokens past the length, unlisted blocks
    for pages, n in zip(place, lens):
        if n % BS:
            for pool in (k, v):
                pool[pages[n // BS].long(), :, n % BS:] = float("nan")
        pages[-(-n // BS):] = -1
    place[7, 3], place[7, 40] = -1, count  # ids outside the pool are skipped
    group = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes)).cuda()
    table = place[group].contiguous()
    seq = torch.tensor(lens, dtype=torch.int32).cuda()[group].contiguous()
    q = torch.randn(rows, heads, dim, device="cuda", generator=g)
    order = torch.tensor([7, 6, 5, 4, 3, 2, 1, 0, 8], dtype=torch.int32)
    desc = None
    if descriptors:
        desc = hip_attn.build_slot_descriptors(table.cpu(), seq.cpu(), starts,
                                               group_order=order).to("cuda")
    meta = hip_attn.get_scheduler_metadata(
        num_reqs=rows, num_heads=heads, num_kv_heads=heads, head_dim=dim, dtype=torch.float32,
        block_size=BS, group_start=starts.cuda(), group_order=order.cuda(), max_group_size=8,
        waves_per_workgroup=waves, slot_descriptors=desc)
    out = torch.full_like(q, float("nan"))
    hip_attn.attention_with_kv_cache(q, k, v, out, torch.arange(rows + 1, dtype=torch.int32,
                                                                device="cuda"),
                                     seq, scale=dim**-0.5, causal=False, block_table=table,
                                     scheduler_metadata=meta)
    for i, n in enumerate(lens):
        a, b = starts[i], starts[i + 1]
        if n == 0:
            assert (out[a:b] == 0).all()
            continue
        ids = place[i][:-(-n // BS)]
        listed = ((ids >= 0) & (ids < count)).repeat_interleave(BS)[:n]
        kk, vv = (gather(p, ids.clamp(0, count - 1), n)[:, listed] for p in (k, v))
        close(out[a:b], attend(q[a:b], kk, vv, dim**-0.5))


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("longest", [40, 900])
def test_fused_write(dim, grouped, longest):
    """The op's fused write equals the separate write followed by attention: the caches bit
    for bit, with new tokens at block edges, rows without a slot and slots elsewhere."""
    from vflorence_amd import hip_attn

    g = torch.Generator(device="cuda").manual_seed(dim + longest)
    heads, lens = 4, [1, 2, 15, 16, 17, 32, 33, longest, longest - 1, 0, 20, 31]
    rows, width = len(lens), -(-longest // BS)
    count = rows * width + 2
    k, v = pools(g, count, heads, dim)
    place = torch.randperm(count, device="cuda", generator=g).int()
    table = place[:rows * width].view(rows, width).contiguous()
    seq = torch.tensor(lens, dtype=torch.int32, device="cuda")
    slots = torch.tensor([int(table[r, max(n - 1, 0) // BS]) * BS + max(n - 1, 0) % BS
                          for r, n in enumerate(lens)], device="cuda")
    slots[9] = int(place[-1]) * BS + 3  # an empty row: a slot that no row reads
    slots[10] = -1                      # nothing to write
    slots[11] = int(place[-2]) * BS     # not the row's last position
    # strided views of a fused projection, as the decoder passes them
    qkv = torch.randn(rows, 3 * heads * dim + 4, device="cuda", generator=g)[:, 1:-3]
    q, kn, vn = (t.view(rows, heads, dim) for t in qkv.chunk(3, dim=-1))
    extra = dict(group_start=torch.arange(0, rows + 1, 4, dtype=torch.int32, device="cuda"),
                 max_group_size=4, own_tables=True) if grouped else {}
    common = dict(num_reqs=rows, num_heads=heads, num_kv_heads=heads, head_dim=dim,
                  dtype=torch.float32, block_size=BS)
    k2, v2, out = k.clone(), v.clone(), torch.full((rows, heads, dim), float("nan"),
                                                   device="cuda")
    hip_attn.self_attention_with_kv_write(
        q, kn, vn, k2, v2, out, seq, slots, scale=dim**-0.5, block_table=table,
        scheduler_metadata=hip_attn.get_scheduler_metadata(fuse_kv_write=True, **common,
                                                           **extra))
    hip_attn.reshape_and_cache(kn, vn, k, v, slots)
    assert torch.equal(k2, k) and torch.equal(v2, v)
    for r, n in enumerate(lens):
        if n == 0:
            assert (out[r] == 0).all()
            continue
        ids = table[r, :-(-n // BS)]
        close(out[r:r + 1], attend(q[r:r + 1], gather(k, ids, n), gather(v, ids, n), dim**-0.5))
