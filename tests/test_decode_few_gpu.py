"""Decode attention of a few sequences: steps dealt out to workgroups and wavefronts, against float64 and around every edge of the plan.

Bar: weights of the values are rounded to bfloat16 (2^-9 each, of either sign) and the result once more (2^-9)."""
import pytest
import torch

from infer_amd import ops, qwen3
from infer_amd.context import reset_context, set_context

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _inputs(gen, lens, hq, hkv, block, columns=None):
    per = columns or max(1, -(-max(lens) // block))
    blocks = len(lens) * per + 2
    k, v = (torch.randn(blocks, block, hkv, 128, generator=gen).to(BF16).cuda() for _ in range(2))
    table = torch.full((len(lens), per), -1, dtype=torch.int32)
    order = torch.randperm(blocks, generator=gen).to(torch.int32)
    for i, n in enumerate(lens):
        used = -(-n // block)
        table[i, :used] = order[i * per:i * per + used]
    return torch.randn(len(lens), hq, 128, generator=gen).to(BF16).cuda(), k, v, table.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()


def _reference(q, k, v, table, lens, scale):
    out, group = torch.zeros(q.shape, dtype=torch.float64), q.shape[1] // k.shape[2]
    for i, n in enumerate(lens):
        if n == 0:
            continue
        pages = table[i].clamp(min=0).long()
        kk, vv = (t[pages].flatten(0, 1)[:n].double().cpu().repeat_interleave(group, 1) for t in (k, v))
        w = torch.softmax(torch.einsum("hd,nhd->hn", q[i].double().cpu(), kk) * scale, -1)
        out[i] = torch.einsum("hn,nhd->hd", w, vv)
    return out


def _check(q, k, v, table, ctx, lens, scale=128 ** -0.5):
    out = torch.full_like(q, float("nan"))
    ops.paged_attn_decode(q, k, v, table, ctx, scale, out)
    want = _reference(q, k, v, table, lens, scale)
    for i in range(len(lens)):
        err = (out[i].double().cpu() - want[i]).norm() / max(want[i].norm().item(), 1e-9)
        assert err <= 2.0 ** -8, (i, lens[i], float(err))
    return out


@pytest.mark.parametrize("lens,hq,hkv,block", [
    ([1], 16, 8, 256), ([31, 32, 33, 0], 16, 8, 256), ([1023, 1024, 1025, 1057], 32, 8, 256), ([4095, 4097, 4128], 16, 8, 256),
    ([0, 2081, 37, 2048, 640, 5, 991, 4096], 32, 8, 256), ([300, 1, 64, 500, 97, 33, 1300], 8, 8, 32), ([129] * 6, 48, 8, 96),
    ([9000], 16, 1, 64), ([2049, 8193], 6, 2, 128), ([777] * 64, 4, 1, 512), ([1, 70, 3000], 5, 5, 256),
])
def test_against_float64(gpu, lens, hq, hkv, block):
    gen = torch.Generator().manual_seed(sum(lens) + hq)
    _check(*_inputs(gen, lens, hq, hkv, block), lens)


def test_batches_on_either_side_of_the_rule_agree(gpu):
    """Rows of a batch that takes the general kernel, and the same rows by themselves."""
    gen = torch.Generator().manual_seed(5)
    lens = [1500, 20, 700, 333, 1, 900, 64, 1200, 256, 31, 2000, 511]
    q, k, v, table, ctx = _inputs(gen, lens, 16, 8, 256)
    whole = _check(q, k, v, table, ctx, lens)
    for i in range(0, 12, 3):
        part = _check(q[i:i + 3], k, v, table[i:i + 3], ctx[i:i + 3], lens[i:i + 3])
        assert (part.float() - whole[i:i + 3].float()).norm() <= 2.0 ** -8 * whole[i:i + 3].float().norm()
    # eight sequences of a table for more than 4096 tokens are the general kernel's
    wide = _inputs(gen, lens[:8], 16, 8, 256, columns=17)
    _check(*wide, lens[:8])


@pytest.mark.parametrize("hq,hkv,most", [(16, 8, 1024), (8, 8, 1024), (8, 4, 2048), (24, 12, 1024), (32, 16, 1024)])
def test_one_sequence_has_the_bits_of_the_general_kernels(gpu, hq, hkv, most):
    """Up to a wavefront per step of 32 tokens both leave the same partial results, and add them up in one order with the same roundings."""
    gen = torch.Generator().manual_seed(hq + hkv)
    for length in (1, 32, 33, 64, 65, 127, 129, 250, 257, 700, most - 31, most):
        q, k, v, table, ctx = _inputs(gen, [length], hq, hkv, 256)
        got, want, ws = torch.empty_like(q), torch.empty_like(q), ops.decode_workspace(q.device, 1, hq, hkv, 128)
        ops.paged_attn_decode(q, k, v, table, ctx, 0.09, got)
        ops.paged_attn_decode_split(q, k, v, table, ctx, 0.09, ws)
        ops.paged_attn_decode_merge(want, ctx, hkv, ws)
        assert torch.equal(got, want), length


def test_what_lies_behind_the_end_is_not_looked_at(gpu):
    """Stale NaN in keys and values behind a length, ids out of range behind the last block, a length beyond the table."""
    gen = torch.Generator().manual_seed(6)
    lens = [40, 300, 512]
    q, k, v, table, ctx = _inputs(gen, lens, 16, 8, 256)
    want = _check(q, k, v, table, ctx, lens)
    for i, n in enumerate(lens):
        if n % 256:
            for t in (k, v):
                t[table[i, n // 256], n % 256:] = float("nan")
    table[0, 1] = 1 << 30
    ctx[2] = 5000
    got = torch.empty_like(q)
    ops.paged_attn_decode(q, k, v, table, ctx, 128 ** -0.5, got)
    assert torch.equal(got, want)


def test_captured_and_replayed_with_other_lengths(gpu):
    gen = torch.Generator().manual_seed(7)
    lens = [900, 10, 2000, 450]
    q, k, v, table, ctx = _inputs(gen, lens, 16, 8, 256)
    table = table.clamp(min=0)
    out, ws = torch.empty_like(q), ops.decode_workspace(q.device, 64, 16, 8, 128).clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        ops.paged_attn_decode(q, k, v, table, ctx, 128 ** -0.5, out, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.paged_attn_decode(q, k, v, table, ctx, 128 ** -0.5, out, workspace=ws)
    for now in ([900, 10, 2000, 450], [1, 0, 33, 2048], [1024, 700, 64, 0]):
        ctx.copy_(torch.tensor(now, dtype=torch.int32))
        out.fill_(float("nan"))
        graph.replay()
        want = _reference(q, k, v, table, now, 128 ** -0.5)
        assert (out.double().cpu() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("lens,hq,hkv,block", [
    ([1], 16, 8, 256), ([31, 32, 33, 0], 16, 8, 256), ([1024, 1025, 2049], 32, 8, 256), ([700, 64, 257, 4096, 1, 96, 128, 3000], 32, 8, 256),
    ([9000], 16, 1, 64), ([129] * 6, 48, 8, 96), ([33, 65], 5, 5, 32), ([65, 70], 4, 1, 64),
])
def test_with_the_front_as_in_two_launches(gpu, lens, hq, hkv, block):
    """Norms, rotary positions and the append inside: the bits of the launches one after the other, in the caches and in the result.  Stale
    NaN lies where the new rows belong; one row's slot is elsewhere, one has none, one has a slot and no tokens."""
    gen = torch.Generator().manual_seed(sum(lens) + hkv)
    _, k, v, table, ctx = _inputs(gen, lens, hq, hkv, block)
    n, spare = len(lens), (k.shape[0] - 1) * block
    slots = [int(table[i, (m - 1) // block]) * block + (m - 1) % block if m else -1 for i, m in enumerate(lens)]
    free = sorted(set(range(k.shape[0])) - set(table.flatten().tolist()))
    for i, s in enumerate(slots):
        if s >= 0:
            for t in (k, v):
                t.view(-1, hkv, 128)[s] = float("nan")
    if n > 2:
        slots[1] = free[0] * block + 3                    # elsewhere: what the cache has there is attended
        k.view(-1, hkv, 128)[int(table[1, (lens[1] - 1) // block]) * block + (lens[1] - 1) % block] = 1.0
        v.view(-1, hkv, 128)[int(table[1, (lens[1] - 1) // block]) * block + (lens[1] - 1) % block] = 1.0
        if lens[-1] == 0:
            slots[-1] = free[0] * block + 5
    slots = torch.tensor(slots, dtype=torch.int32).cuda()
    qkv = (3 * torch.randn(n, (hq + 2 * hkv) * 128 + 64, generator=gen)).to(BF16).cuda()[:, 64:]
    q, kn, vn = (t.view(n, -1, 128) for t in qkv.split([hq * 128, hkv * 128, hkv * 128], -1))
    wq, wk = ((1 + 0.3 * torch.randn(128, generator=gen)).to(BF16).cuda() for _ in range(2))
    cs = torch.randn(max(lens) + 9, 128, generator=gen).to(BF16).cuda()
    positions = torch.tensor([max(m - 1, 0) + 5 * (i % 2) for i, m in enumerate(lens)]).cuda()
    k2, v2, kept = k.clone(), v.clone(), qkv.clone()
    out = ops.few_decode_with_front(q, kn, vn, positions, wq, wk, 1e-6, cs, k2, v2, slots, table, ctx, 0.09)
    assert torch.equal(qkv, kept)
    ops.qk_norm_rope_store_kvcache(q, kn, vn, positions, wq, wk, 1e-6, cs, k, v, slots, write_key=False)
    want = torch.empty_like(out)
    ops.paged_attn_decode(q, k, v, table, ctx, 0.09, want)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert same(k, k2) and same(v, v2)
    assert torch.isfinite(out.float()).all() and torch.equal(out, want)


@pytest.mark.parametrize("rows,hq,hkv,block", [
    ([(0, 33), (0, 34)], 16, 8, 256), ([(0, 32), (0, 33)], 16, 8, 256), ([(0, 1), (0, 2), (0, 3)], 5, 5, 32), ([(0, 700 + i) for i in range(6)], 32, 8, 64),
    ([(0, 66), (1, 40), (0, 65), (1, 41), (0, 64)], 48, 8, 32), ([(0, 4096), (0, 4097)], 16, 1, 256), ([(i % 2, 1 + 9 * i) for i in range(64)], 4, 1, 64),
])
@pytest.mark.parametrize("moved", [False, True])
def test_rows_that_see_each_other(gpu, rows, hq, hkv, block, moved):
    """Rows (sequence, length) of the same sequences: each attends to the new tokens of those in front of it, as behind an append of all.  Stale NaN
    lies where the new rows belong.  ``moved``: the first row's slot lies in the middle of its own context, and a row without tokens has its slot in it, too."""
    gen = torch.Generator().manual_seed(sum(m for _, m in rows) + hkv)
    longest = [max([m for s, m in rows if s == i] or [1]) for i in range(2)]
    _, k, v, table, _ = _inputs(gen, longest, hq, hkv, block)
    lens, place = [m for _, m in rows], lambda s, m: int(table[s, (m - 1) // block]) * block + (m - 1) % block
    slots, table = [place(s, m) for s, m in rows], table[[s for s, _ in rows]].contiguous()
    if moved:
        slots[0] = place(rows[0][0], (lens[0] + 1) // 2)
        slots[-1], lens[-1] = place(rows[0][0], 1), 0
        if slots[0] == slots[-1]:
            slots[0] = -1
    n = len(rows)
    for t in (k, v):
        t.view(-1, hkv, 128)[[s for s in slots if s >= 0]] = float("nan")
    slots, ctx = (torch.tensor(x, dtype=torch.int32).cuda() for x in (slots, lens))
    q, kn, vn = (3 * torch.randn(n, h, 128, generator=gen).to(BF16).cuda() for h in (hq, hkv, hkv))
    wq, wk = ((1 + 0.3 * torch.randn(128, generator=gen)).to(BF16).cuda() for _ in range(2))
    cs, positions = torch.randn(max(lens) + 9, 128, generator=gen).to(BF16).cuda(), torch.tensor([max(m - 1, 0) + 3 * (i % 2) for i, m in enumerate(lens)]).cuda()
    k2, v2 = k.clone(), v.clone()
    out = ops.few_decode_with_front(q, kn, vn, positions, wq, wk, 1e-6, cs, k2, v2, slots, table, ctx, 0.09)
    ops.qk_norm_rope_store_kvcache(q, kn, vn, positions, wq, wk, 1e-6, cs, k, v, slots, write_key=False)
    want = torch.empty_like(out)
    ops.paged_attn_decode(q, k, v, table, ctx, 0.09, want)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert same(k, k2) and same(v, v2)
    assert torch.isfinite(want.float()).all() and same(out, want)


@pytest.mark.parametrize("length,hq,hkv,hidden", [(0, 16, 8, 1024), (1, 16, 8, 1024), (33, 16, 8, 1024), (260, 16, 8, 1000), (4097, 16, 8, 520),
                                                  (700, 32, 8, 512), (9000, 32, 16, 248), (300, 24, 8, 768), (300, 12, 12, 744), (64, 16, 8, 4096), (64, 4, 1, 512),
                                                  (700, 16, 8, 1024), (1024, 16, 8, 1024), (230, 16, 8, 1024)])
def test_with_the_product_behind_it(gpu, length, hq, hkv, hidden):
    """The pieces of a sequence's attention added up by the product's workgroups: the bits of attention and split product, again in replays of
    a graph; not where a workgroup would have more than four heads, there are more workgroups than compute units, or pieces are many."""
    gen = torch.Generator().manual_seed(length + hidden)
    _, k, v, table, ctx = _inputs(gen, [length], hq, hkv, 256)
    slots = torch.tensor([int(table[0, (length - 1) // 256]) * 256 + (length - 1) % 256 if length else -1], dtype=torch.int32).cuda()
    qkv = (3 * torch.randn(1, (hq + 2 * hkv) * 128, generator=gen)).to(BF16).cuda()
    q, kn, vn = (t.view(1, -1, 128) for t in qkv.split([hq * 128, hkv * 128, hkv * 128], -1))
    wq, wk = ((1 + 0.3 * torch.randn(128, generator=gen)).to(BF16).cuda() for _ in range(2))
    cs, positions = torch.randn(length + 9, 128, generator=gen).to(BF16).cuda(), torch.tensor([max(length - 1, 0)]).cuda()
    weight = (0.02 * torch.randn(hidden, hq * 128, generator=gen)).to(BF16).cuda()
    args = q, kn, vn, positions, wq, wk, 1e-6, cs, k, v, slots, table, ctx, 0.09
    out = ops.few_decode_with_front(*args)
    want = ops.linear(out.view(1, -1), weight, defer=True)
    if isinstance(want, ops.SplitKSum):
        splits, want = want.partial.shape[0], want.materialize()
    else:
        splits = 1
    got = ops.few_decode_with_front(*args, weight)
    if splits == 1 or hq // splits > 4 or hkv < 8 or -(-hidden // 16) * splits > 256:
        assert torch.equal(got, out)
        return
    assert isinstance(got, ops.SplitKSum) and got.partial.shape == (splits, 1, hidden)
    assert torch.equal(got.materialize(), want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.few_decode_with_front(*args, weight).materialize()
    for _ in range(3):
        got.fill_(float("nan"))
        graph.replay()
        ops.few_decode_with_front(*args, weight)
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_batches_that_are_not_small_are_left_alone(gpu):
    gen = torch.Generator().manual_seed(9)
    q, k, v, table, ctx = _inputs(gen, [64] * 9, 16, 8, 256)
    rows, w = torch.zeros(9, 8, 128, dtype=BF16, device="cuda"), torch.ones(128, dtype=BF16, device="cuda")
    cs, at = torch.ones(64, 128, dtype=BF16, device="cuda"), torch.zeros(9, dtype=torch.int64, device="cuda")
    kept = k.clone()
    assert ops.few_decode_with_front(q, rows, rows, at, w, w, 1e-6, cs, k, v, at.int(), table, ctx, 0.1) is None
    assert torch.equal(k, kept)


def test_one_length_for_the_whole_batch(gpu):
    """A decode step's context may hold one number instead of the lengths, as decode attention takes it."""
    gen = torch.Generator().manual_seed(10)
    _, k, v, table, ctx = _inputs(gen, [300, 300], 16, 8, 256)
    slots, positions = (table[:, 1] * 256 + 299 % 256).to(torch.int32), torch.tensor([299, 299]).cuda()
    layer = qwen3.QwenAttention(256, 16, 8, max_position=512).to(device="cuda", dtype=BF16)
    for p in (layer.qkv_proj.weight, layer.o_proj.weight):
        p.data.copy_(0.05 * torch.randn(p.shape, generator=gen))
    x, out = torch.randn(2, 256, generator=gen).to(BF16).cuda(), []
    for lens in (ctx, 300):
        layer.attn.k_cache, layer.attn.v_cache = k.clone(), v.clone()
        set_context(False, slot_mapping=slots, context_lens=lens, block_tables=table)
        y = layer(positions, x)
        out.append((y.materialize() if isinstance(y, ops.SplitKSum) else y, layer.attn.k_cache, layer.attn.v_cache))
    reset_context()
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][2], out[1][2])
    assert (out[0][0].float() - out[1][0].float()).norm() <= 2.0 ** -7 * out[1][0].float().norm()
