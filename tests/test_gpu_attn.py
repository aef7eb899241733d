"""GPU parity: decode paged attention, KV append and length advance vs the CPU oracle.

Tolerance: attention outputs within 2e-2 absolute in fp16/bf16 (fp32 softmax and accumulation on
both sides; the reference's flash-attn rounds the probabilities to the storage dtype before the PV
product, this kernel keeps them in fp32).
"""
import pytest
import torch

from fastcache_amd import _lib, ops, synth
from oracle import attention as oattn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens", [
    (4, 4, [1, 255, 256, 257, 700]),
    (8, 2, [33, 1024, 513]),
    (14, 2, [300, 17]),
    (16, 1, [129, 0, 600]),
    (6, 2, [77, 260]),          # a group of 3 in a tile of 4
    (10, 2, [513]),             # a group of 5 in a tile of 8
])
def test_decode_attention(dev, dtype, Hq, Hkv, lens):
    L, B = 2, len(lens)
    case = synth.make_paged_case(seed=21, num_layers=L, batch=B, num_kv_heads=Hkv, seq_lens=[max(n, 1) for n in lens],
                                 dtype=dtype, reserve_tokens=8)
    g = torch.Generator().manual_seed(5)
    q = torch.randn(L, B, Hq, 128, generator=g).to(dtype)
    width = max(len(t) for t in case.block_tables) + 2
    tables = case.table_tensor("cpu", width)
    lens_t = torch.tensor(lens, dtype=torch.int32)
    scale = 128 ** -0.5

    pool = case.kv_cache.to(dev)
    tab_d, len_d = tables.to(dev), lens_t.to(dev)
    max_len = width * 256
    kview = _lib.paged_view(pool[0], tab_d, None, max_len)
    vview = _lib.paged_view(pool[1], tab_d, None, max_len)
    ws = ops.decode_attn_workspace(B, Hq, max_len, dev)
    for layer in range(L):
        ref = oattn.decode_attention(q[layer], case.kv_cache[0, layer], case.kv_cache[1, layer], lens_t, tables, scale)
        got = ops.decode_attn(kview, vview, layer, q[layer].to(dev), len_d, scale, ws)
        torch.cuda.synchronize()
        torch.testing.assert_close(got.cpu().float(), ref.float(), atol=2e-2, rtol=0)
        # much tighter in practice: fp32 math on both sides, one rounding at the end
        assert float((got.cpu().float() - ref.float()).abs().max()) < 4e-3


@pytest.mark.parametrize("block_size", [16, 32, 48, 64])
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (8, 2)])
def test_decode_attention_small_and_odd_pages(dev, block_size, Hq, Hkv):
    """Pages smaller than a 32-token tile or of a size that is no power of two take the per-row
    addressing path; pages of 32 and 64 tokens take the tile path with several pages per chunk."""
    dtype, lens = torch.bfloat16, [1, 31, 32, 33, 255, 256, 257, 530]
    B = len(lens)
    case = synth.make_paged_case(seed=8, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype,
                                 block_size=block_size)
    q = torch.randn(B, Hq, 128, generator=torch.Generator().manual_seed(6)).to(dtype)
    tables, lens_t = case.table_tensor("cpu"), torch.tensor(lens, dtype=torch.int32)
    ref = oattn.decode_attention(q, case.kv_cache[0, 0], case.kv_cache[1, 0], lens_t, tables, 128 ** -0.5)
    pool, tab_d = case.kv_cache.to(dev), tables.to(dev)
    max_len = tables.shape[1] * block_size
    kview, vview = (_lib.paged_view(pool[i], tab_d, None, max_len) for i in range(2))
    ws = ops.decode_attn_workspace(B, Hq, max_len, dev)
    got = ops.decode_attn(kview, vview, 0, q.to(dev), lens_t.to(dev), 128 ** -0.5, ws).cpu()
    assert float((got.float() - ref.float()).abs().max()) < 4e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_decode_attention_dense_view(dev, dtype):
    """A HuggingFace-layout cache [B, Hkv, S, D] gives the same output as the same rows in pages."""
    Hq, Hkv, lens = 8, 4, [700, 64, 385]
    B, S = len(lens), max(lens)
    case = synth.make_paged_case(seed=4, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype,
                                 keep_dense=True)
    q = torch.randn(B, Hq, 128, generator=torch.Generator().manual_seed(7)).to(dtype).to(dev)
    lens_d = torch.tensor(lens, dtype=torch.int32, device=dev)
    dk, dv = case.dense_k[0].to(dev), case.dense_v[0].to(dev)    # rows past a sequence's length hold other data
    ws = ops.decode_attn_workspace(B, Hq, S, dev)
    got = ops.decode_attn(_lib.dense_view(dk), _lib.dense_view(dv), 0, q, lens_d, 128 ** -0.5, ws).cpu()
    pool, tab = case.kv_cache.to(dev), case.table_tensor(dev)
    ws2 = ops.decode_attn_workspace(B, Hq, tab.shape[1] * 256, dev)
    paged = ops.decode_attn(_lib.paged_view(pool[0], tab, None, tab.shape[1] * 256),
                            _lib.paged_view(pool[1], tab, None, tab.shape[1] * 256), 0, q, lens_d, 128 ** -0.5, ws2).cpu()
    assert torch.equal(got, paged)
    ref = oattn.decode_attention(q.cpu(), case.kv_cache[0, 0], case.kv_cache[1, 0], lens_d.cpu(), tab.cpu(), 128 ** -0.5)
    assert float((got.float() - ref.float()).abs().max()) < 4e-3


def test_block_permutation_invariance(dev):
    """Moving the pages around (with the table following) leaves the output bit-identical."""
    dtype, Hq, Hkv, lens = torch.float16, 8, 4, [900, 300, 77]
    case = synth.make_paged_case(seed=2, num_layers=1, batch=3, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype)
    nb = case.kv_cache.shape[2]
    perm = torch.randperm(nb, generator=torch.Generator().manual_seed(1))
    pool2 = torch.empty_like(case.kv_cache)
    pool2[:, :, perm] = case.kv_cache                       # block i moves to perm[i]
    tables1 = case.table_tensor("cpu")
    tables2 = torch.where(tables1 >= 0, perm[tables1.clamp_min(0).long()].int(), tables1)
    q = torch.randn(3, Hq, 128, generator=torch.Generator().manual_seed(3)).to(dtype).to(dev)
    lens_d = torch.tensor(lens, dtype=torch.int32, device=dev)
    outs = []
    for pool, tab in ((case.kv_cache, tables1), (pool2, tables2)):
        p, t = pool.to(dev), tab.to(dev)
        kv = [_lib.paged_view(p[i], t, None, t.shape[1] * 256) for i in range(2)]
        ws = ops.decode_attn_workspace(3, Hq, t.shape[1] * 256, dev)
        outs.append(ops.decode_attn(kv[0], kv[1], 0, q, lens_d, 128 ** -0.5, ws).cpu())
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_store_kv_and_advance(dev, dtype):
    L, B, Hkv = 3, 4, 2
    lens = [5, 255, 256, 511]
    case = synth.make_paged_case(seed=9, num_layers=L, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype,
                                 reserve_tokens=4)
    g = torch.Generator().manual_seed(1)
    k_new = torch.randn(L, B, Hkv, 128, generator=g).to(dtype)
    v_new = torch.randn(L, B, Hkv, 128, generator=g).to(dtype)
    ref = case.kv_cache.clone()
    for layer in range(L):
        slots = torch.tensor([oattn.decode_slot(case.block_tables[b], lens[b]) for b in range(B)])
        oattn.store_kv(ref[0, layer], ref[1, layer], k_new[layer], v_new[layer], slots)

    pool = case.kv_cache.to(dev)
    tab = case.table_tensor(dev)
    len_d = torch.tensor(lens, dtype=torch.int32, device=dev)
    max_len = tab.shape[1] * 256
    kview = _lib.paged_view(pool[0], tab, None, max_len)
    vview = _lib.paged_view(pool[1], tab, None, max_len)
    ops.store_kv(kview, vview, k_new.to(dev), v_new.to(dev), len_d)
    ops.advance_lens(len_d, 1)
    torch.cuda.synchronize()
    assert torch.equal(pool.cpu().view(torch.uint8), ref.view(torch.uint8))
    assert len_d.cpu().tolist() == [n + 1 for n in lens]


def test_multi_step_decode_graph_matches_eager_and_oracle(dev):
    """T steps in one HIP graph: every replay equals the eager launches bit for bit, and both follow
    the oracle (store, advance, attend) across a block boundary."""
    from fastcache_amd.engine.decode_graph import DecodeGraph
    dtype, L, B, Hq, Hkv, T = torch.float16, 2, 3, 4, 2, 6
    lens = [254, 100, 511]                       # two sequences cross a 256-token block boundary
    case = synth.make_paged_case(seed=13, num_layers=L, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype,
                                 reserve_tokens=T + 1)
    g = torch.Generator().manual_seed(2)
    q = torch.randn(T, L, B, Hq, 128, generator=g).to(dtype)
    kn = torch.randn(T, L, B, Hkv, 128, generator=g).to(dtype)
    vn = torch.randn(T, L, B, Hkv, 128, generator=g).to(dtype)
    tables = case.table_tensor("cpu")
    scale = 128 ** -0.5

    # oracle
    ref_pool = case.kv_cache.clone()
    ref_out = torch.empty_like(q)
    cur = list(lens)
    for t in range(T):
        for layer in range(L):
            slots = torch.tensor([oattn.decode_slot(case.block_tables[b], cur[b]) for b in range(B)])
            oattn.store_kv(ref_pool[0, layer], ref_pool[1, layer], kn[t, layer], vn[t, layer], slots)
        cur = [n + 1 for n in cur]
        for layer in range(L):
            ref_out[t, layer] = oattn.decode_attention(q[t, layer], ref_pool[0, layer], ref_pool[1, layer],
                                                       torch.tensor(cur, dtype=torch.int32), tables, scale)

    def fresh():
        pool = case.kv_cache.to(dev)
        lens_d = torch.tensor(lens, dtype=torch.int32, device=dev)
        return DecodeGraph(pool, tables.to(dev), lens_d, q.to(dev), kn.to(dev), vn.to(dev), scale), pool, lens_d

    dg, pool, lens_d = fresh()
    eager = dg.run_eager().clone()
    torch.cuda.synchronize()
    assert lens_d.tolist() == [n + T for n in lens]
    assert torch.equal(pool.cpu().view(torch.uint8), ref_pool.view(torch.uint8))
    torch.testing.assert_close(eager.cpu().float(), ref_out.float(), atol=2e-2, rtol=0)

    dg2, pool2, lens2 = fresh()
    dg2.capture()
    assert lens2.tolist() == lens
    for rep in range(3):
        lens2.copy_(torch.tensor(lens, dtype=torch.int32))
        dg2.out.zero_()
        torch.cuda.synchronize()
        out = dg2.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {rep} differs from eager"
        assert lens2.tolist() == [n + T for n in lens]
        _ = (pool2.float().sum()).item()          # unrelated eager work between replays
    assert torch.equal(pool2, pool)


def test_bucketed_decode_graphs_match_eager_layers(dev):
    """One captured step per batch bucket, static buffers patched per step: every replay equals the eager
    Attention layers bit for bit (outputs and pool), for batches that fill a bucket exactly and that do not."""
    from fastcache_amd.engine.decode_graph import BucketedDecodeGraphs
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    dtype, L, Hq, Hkv, D, steps = torch.float16, 2, 8, 2, 128, 3
    max_bs, scale = 40, 128 ** -0.5
    all_lens = [100 + 37 * i for i in range(21)]
    all_lens[4] = 255                                            # crosses a block boundary during the steps
    case = synth.make_paged_case(seed=21, num_layers=L, batch=21, num_kv_heads=Hkv, seq_lens=all_lens, dtype=dtype,
                                 reserve_tokens=steps + 1)
    tables_all = case.table_tensor("cpu")

    def make_layers(pool):
        layers = []
        for l in range(L):
            a = Attention(Hq, D, scale, Hkv)
            a.k_cache, a.v_cache = pool[0, l], pool[1, l]
            layers.append(a)
        return layers

    pool_g, pool_e = case.kv_cache.to(dev), case.kv_cache.to(dev)
    graphs = BucketedDecodeGraphs(make_layers(pool_g), max_bs, tables_all.shape[1], dtype, dev)
    graphs.capture_cudagraph()
    assert graphs.graph_bs == [1, 2, 4, 8, 16, 32, 40]
    pool_g.copy_(case.kv_cache)                                  # capture warm-ups wrote nothing (slots are -1)
    eager_layers = make_layers(pool_e)
    g = torch.Generator().manual_seed(6)
    for bs in (3, 21, 16):
        lens = list(all_lens[:bs])
        tables = tables_all[:bs].to(dev)
        for t in range(steps):
            q = torch.randn(L, bs, Hq * D, generator=g).to(dtype).to(dev)
            k = torch.randn(L, bs, Hkv * D, generator=g).to(dtype).to(dev)
            v = torch.randn(L, bs, Hkv * D, generator=g).to(dtype).to(dev)
            slots = torch.tensor([oattn.decode_slot(case.block_tables[b], lens[b]) for b in range(bs)],
                                 dtype=torch.int32, device=dev)
            lens = [n + 1 for n in lens]
            ctx_lens = torch.tensor(lens, dtype=torch.int32, device=dev)
            set_context(False, slot_mapping=slots, context_lens=ctx_lens, block_tables=tables)
            out_g = graphs.run(q, k, v).clone()
            out_e = torch.stack([eager_layers[l](q[l], k[l], v[l]) for l in range(L)])
            reset_context()
            torch.cuda.synchronize()
            assert torch.equal(out_g, out_e), f"bs={bs} step={t}"
            assert torch.equal(pool_g, pool_e)
        # restore the prefixes for the next batch size
        pool_g.copy_(case.kv_cache)
        pool_e.copy_(case.kv_cache)


def test_decode_attention_empty_rows(dev):
    """Rows with no cached token give zeros, whatever their table row holds; their neighbours are unaffected."""
    dtype, Hq, Hkv = torch.bfloat16, 8, 2
    case = synth.make_paged_case(seed=3, num_layers=1, batch=3, num_kv_heads=Hkv, seq_lens=[300, 1, 5], dtype=dtype)
    q = torch.randn(3, Hq, 128, generator=torch.Generator().manual_seed(2)).to(dtype).to(dev)
    pool, tab = case.kv_cache.to(dev), case.table_tensor(dev)
    max_len = tab.shape[1] * 256
    kview, vview = _lib.paged_view(pool[0], tab, None, max_len), _lib.paged_view(pool[1], tab, None, max_len)
    ws = ops.decode_attn_workspace(3, Hq, max_len, dev)
    full = ops.decode_attn(kview, vview, 0, q, torch.tensor([300, 1, 5], dtype=torch.int32, device=dev), 128 ** -0.5, ws).cpu()
    some = ops.decode_attn(kview, vview, 0, q, torch.tensor([300, 0, 0], dtype=torch.int32, device=dev), 128 ** -0.5, ws).cpu()
    assert torch.equal(some[0], full[0]) and bool((some[1:] == 0).all())
    none = ops.decode_attn(kview, vview, 0, q, torch.zeros(3, dtype=torch.int32, device=dev), 128 ** -0.5, ws).cpu()
    assert bool((none == 0).all())


@pytest.mark.parametrize("dtype,Hq,Hkv,lens,slot_at", [
    (torch.bfloat16, 28, 4, [300, 900, 1, 0, 31, 32, 33, 255, 256, 257, 511, 513], 0),   # the new row right behind the context
    (torch.bfloat16, 8, 2, [1, 2, 32, 33, 256, 257, 512, 900], -1),                      # the new row is the last attended one
    (torch.float16, 4, 4, [2047, 5, 1024], -1),
    (torch.float16, 32, 2, [700, 130], -2),                                              # 16 heads a group; a row inside the context
    (torch.bfloat16, 40, 2, [300, 77], -1),                                              # 20 heads a group: rows go in first
    (torch.bfloat16, 8, 2, [2500, 40], -1),                                              # too long for one workgroup a column
    # many columns: ranges of 512 tokens and more, on both sides of their ends, and of a wavefront's second tile
    (torch.bfloat16, 16, 2, ([1023, 511, 512, 513, 1, 256, 257, 767] * 5)[:33], -1),
    (torch.float16, 2, 2, ([900, 511, 512, 1023, 40] * 7)[:33], 0),
    (torch.bfloat16, 8, 2, ([1700, 767, 768, 769, 1535, 1536, 33] * 6)[:40], -1),        # 4 heads a group: 768
    (torch.float16, 8, 1, ([3900, 1535, 1536, 1537, 100, 3072, 3073] * 10)[:65], -1),    # 8 heads a group: 1536
    (torch.bfloat16, 32, 4, ([700, 511, 512, 1, 600] * 14)[:70], -1),                    # two rounds of whole columns
    (torch.float16, 8, 8, ([1200, 1030, 257, 1279, 64, 1025, 800, 1] * 4)[:28], -1),      # 5 tiles a wavefront, whole columns
    (torch.bfloat16, 8, 4, ([2700, 2815, 1407, 1408, 1409, 1] * 6)[:32], 0),               # two heads a group, chunks that append
])
def test_attention_layer_appends_and_attends(dev, dtype, Hq, Hkv, lens, slot_at):
    """``Attention.forward`` of a decode step against the oracle on a cache the oracle appended to: every launch form the
    layer picks (append inside the attention's launch or before it), rows behind, at and inside the attended range, a
    sequence without context and a padded one (slot -1)."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    B = len(lens)
    case = synth.make_paged_case(seed=31, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables, lens_t = case.table_tensor("cpu"), torch.tensor(lens, dtype=torch.int32)
    pos = [max(0, n + slot_at) for n in lens]
    slots = torch.tensor([case.block_tables[b][p // 256] * 256 + p % 256 for b, p in enumerate(pos)], dtype=torch.int32)
    slots[-1] = -1
    pool = case.kv_cache[:, 0].clone()
    for p, new in ((0, k), (1, v)):
        for b in range(B - 1):
            pool[p].view(-1, Hkv, 128)[int(slots[b])] = new[b].view(Hkv, 128)
    ref = oattn.decode_attention(q.view(B, Hq, 128), pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    layer = Attention(Hq, 128, 128 ** -0.5, Hkv)
    on_gpu = case.kv_cache[:, 0].to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    set_context(False, slot_mapping=slots.to(dev), context_lens=lens_t.to(dev), block_tables=tables.to(dev))
    try:
        got = layer(q.to(dev), k.to(dev), v.to(dev)).cpu().view(B, Hq, 128)
    finally:
        reset_context()
    assert torch.equal(on_gpu.cpu(), pool)
    assert float((got.float() - ref.float()).abs().max()) < 4e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,max_pages", [([200, 33, 64], 1), ([700, 300], 3)])     # one workgroup a column; several
def test_keys_of_infinite_distance_weigh_nothing(dev, dtype, lens, max_pages):
    """Keys whose logit is -inf (here the first ones of every context, whole 32-key tiles and, in the longer contexts, a
    whole workgroup's range) take no weight, as in a softmax over the whole row."""
    from fastcache_amd.layers.attention import decode_attention
    Hq, Hkv, B = 8, 2, len(lens)
    case = synth.make_paged_case(seed=5, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype)
    pool = case.kv_cache[:, 0].clone()
    for b, n in enumerate(lens):
        for p in range(n // 2):
            pool[0, case.block_tables[b][p // 256], p % 256, :, 0] = -float("inf")
    q = torch.randn(B, Hq, 128, generator=torch.Generator().manual_seed(1)).to(dtype)
    q[..., 0] = q[..., 0].abs() + 0.5
    tables, lens_t = case.table_tensor("cpu"), torch.tensor(lens, dtype=torch.int32)
    assert tables.shape[1] == max_pages
    ref = oattn.decode_attention(q, pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    assert bool(torch.isfinite(ref).all())
    on_gpu = pool.to(dev)
    got = decode_attention(q.to(dev), on_gpu[0], on_gpu[1], lens_t.to(dev), tables.to(dev), 128 ** -0.5).cpu()
    assert float((got.float() - ref.float()).abs().max()) < 4e-3      # as for finite keys above


@pytest.mark.parametrize("dtype,Hq,Hkv,lens,pages", [
    (torch.bfloat16, 28, 4, [300, 0, 1, 255, 256, 257, 511], 2),
    (torch.float16, 8, 8, [2048, 2047, 700], 8),                # ranges read eight at a time: one group of them, one more
    (torch.bfloat16, 8, 2, [2049, 1], 9),
    (torch.float16, 32, 2, [3584, 513], 14),                    # 16 heads a group; the most ranges the last workgroup merges
    (torch.bfloat16, 7, 1, [3600], 15),                         # one more: a launch merges
    (torch.bfloat16, 14, 2, ([1000, 512, 513, 0, 80] * 7)[:33], 4),     # ranges of 512
])
def test_last_workgroup_merges_as_the_merge_launch(dev, dtype, Hq, Hkv, lens, pages):
    """A column's ranges merged by its last workgroup (streams of torch, outside capture) against the launch that merges
    (inside a captured graph, and on streams whose handle torch does not own): which kernels ran, and the same bits, launch
    after launch, with two streams at work at once, and the oracle's values.  Outputs lie where NaN was: a launch that found
    its counters not at zero would leave them."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    B = len(lens)
    case = synth.make_paged_case(seed=51, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables = case.table_tensor("cpu")
    tables = torch.cat([tables, tables[:, :1].expand(-1, max(0, pages - tables.shape[1]))], 1)[:, :pages].contiguous()
    lens_t = torch.tensor(lens, dtype=torch.int32)
    slots = torch.full((B,), -1, dtype=torch.int32)
    pool = case.kv_cache[:, 0]
    ref = oattn.decode_attention(q.view(B, Hq, 128), pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    layer = Attention(Hq, 128, 128 ** -0.5, Hkv)
    on_gpu = pool.to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    set_context(False, slot_mapping=slots.to(dev), context_lens=lens_t.to(dev), block_tables=tables.to(dev))

    def call():
        torch.full((B, Hq * 128), float("nan"), dtype=dtype, device=dev)       # freed: the output's memory
        return layer(q, k, v)

    def kernels(fn, of_graph=False):
        """(whether its columns merge themselves, launches of decode_merge_kernel) of the one decode layer in ``fn``; None for a
        graph of whose launches the profile holds none, as happens now and then"""
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA], acc_events=True) as prof:
            fn()
            torch.cuda.synchronize()
        names = [e.name for e in prof.events()]
        column = [n for n in names if "decode_column_kernel<" in n]
        if of_graph and not any("decode_" in n for n in names):
            return None
        assert len(column) == 1, names
        return column[0].split(">")[0].endswith("true"), sum("decode_merge_kernel" in n for n in names)

    last, launch = (True, 0), (False, 1)
    eager = last if pages <= 14 else launch
    try:
        side = [torch.cuda.Stream(), torch.cuda.Stream()]
        foreign = torch.cuda.ExternalStream(torch.cuda.Stream().cuda_stream)
        torch.cuda.synchronize()
        outs = [call() for _ in range(3)]
        assert kernels(lambda: outs.append(call())) == eager
        for _ in range(4):                                       # two streams at once
            for s in side:
                with torch.cuda.stream(s):
                    outs.append(call())
        torch.cuda.synchronize()
        with torch.cuda.stream(side[1]):
            assert kernels(lambda: outs.append(call())) == eager
        with torch.cuda.stream(foreign):
            merged = call()
            assert kernels(lambda: outs.append(call())) == launch
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            held = layer(q, k, v)
        assert kernels(graph.replay, of_graph=True) in (launch, None)
        for _ in range(3):
            held.zero_()
            graph.replay()
            outs.append(call())
            torch.cuda.synchronize()
            assert torch.equal(held.view(torch.int16), merged.view(torch.int16))
    finally:
        reset_context()
    for o in outs:
        assert torch.equal(o.view(torch.int16), merged.view(torch.int16))
    assert float((merged.cpu().view(B, Hq, 128).float() - ref.float()).abs().max()) < 4e-3


@pytest.mark.parametrize("copies,lens,block_size", [
    (3, [300, 40], 256),            # one workgroup a column
    (2, [254, 700], 256),           # several; the second copy's row is the first of a page
    (5, [30, 64, 255], 32),
    (35, [260, 90], 64),            # more sequences than a wavefront has lanes
])
def test_new_rows_are_seen_by_every_sequence_that_reads_their_page(dev, copies, lens, block_size):
    """The same table listed several times with lengths one apart: several tokens of one sequence in one step, each
    attending the rows of those before it, which other rows of the batch append (attention.py:62-79 stores all rows
    before any sequence is attended)."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    dtype, Hq, Hkv = torch.bfloat16, 2, 1
    case = synth.make_paged_case(seed=41, num_layers=1, batch=len(lens), num_kv_heads=Hkv, seq_lens=[n + copies for n in lens],
                                 dtype=dtype, block_size=block_size)
    rows = [(s, j) for j in range(copies) for s in range(len(lens))]        # copies of a sequence far apart in the batch
    B = len(rows)
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables = case.table_tensor("cpu")[[s for s, _ in rows]].contiguous()
    lens_t = torch.tensor([lens[s] + j + 1 for s, j in rows], dtype=torch.int32)
    pos = [lens[s] + j for s, j in rows]
    slots = torch.tensor([case.block_tables[s][p // block_size] * block_size + p % block_size for (s, _), p in zip(rows, pos)],
                         dtype=torch.int32)
    pool = case.kv_cache[:, 0].clone()
    for p, new in ((0, k), (1, v)):
        pool[p].view(-1, Hkv, 128)[slots.long()] = new.view(B, Hkv, 128)
    ref = oattn.decode_attention(q.view(B, Hq, 128), pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    layer = Attention(Hq, 128, 128 ** -0.5, Hkv)
    on_gpu = case.kv_cache[:, 0].to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    set_context(False, slot_mapping=slots.to(dev), context_lens=lens_t.to(dev), block_tables=tables.to(dev))
    try:
        got = layer(q.to(dev), k.to(dev), v.to(dev)).cpu().view(B, Hq, 128)
    finally:
        reset_context()
    assert torch.equal(on_gpu.cpu(), pool)
    assert float((got.float() - ref.float()).abs().max()) < 4e-3      # as above


@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (4, 2), (8, 2), (14, 2)])
@pytest.mark.parametrize("lens,table", [([64, 250], 1), ([700, 300], 3),     # one workgroup a column; several
                                        ([64, 250, 700], 70)])                # a table too wide for that kernel
@pytest.mark.parametrize("below", [12, 20, 26])
def test_small_fp16_probabilities_keep_their_bits(dev, Hq, Hkv, lens, table, below):
    """Of every 32 keys one has the largest logit and a value of zero, the others 2^-below of its weight: the output is what
    those add, and its error stays within the output's own rounding (2^-11 of an element) and 2^-13 for the logits in
    fp32 (26 times 2^-24 and an exponential: below 2^-18 of a weight; the sum over equal weights adds no more).  An fp16
    operand with its subnormal step of 2^-24 has no bits left for such weights."""
    from fastcache_amd.layers.attention import decode_attention
    dtype, B, scale = torch.float16, len(lens), 128 ** -0.5
    case = synth.make_paged_case(seed=6, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype)
    pool, tables = case.kv_cache[:, 0].clone(), case.table_tensor("cpu", table)
    g = torch.Generator().manual_seed(8)
    pool[0] = 0
    pool[0, ..., 0] = -below * 0.6931471805599453 / scale / 16                # the query's first element is 16
    pool[1] = (512 + 512 * torch.rand(pool[1].shape, generator=g)).to(dtype)
    for at in range(0, 256, 32):
        pool[:, :, at] = 0
    q = torch.zeros(B, Hq, 128, dtype=dtype)
    q[..., 0] = 16
    on_gpu, lens_t = pool.to(dev), torch.tensor(lens, dtype=torch.int32)
    got = decode_attention(q.to(dev), on_gpu[0], on_gpu[1], lens_t.to(dev), tables.to(dev), scale).cpu().double()
    for b, n in enumerate(lens):
        pages = tables[b, :(n + 255) // 256].long()
        k, v = (pool[p, pages].reshape(-1, Hkv, 128)[:n].double().repeat_interleave(Hq // Hkv, 1) for p in range(2))
        w = torch.softmax(torch.einsum("hd,nhd->hn", q[b].double(), k) * scale, dim=-1)
        ref = torch.einsum("hn,nhd->hd", w, v)
        # 2^-25: half of fp16's smallest step, for outputs below its normal range
        assert bool(((got[b] - ref).abs() <= (2.0 ** -11 + 2.0 ** -13) * ref.abs() + 2.0 ** -25).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,n", [(16, 16, 3), (16, 8, 32), (16, 4, 33), (12, 4, 250)])
def test_probabilities_of_up_to_four_heads_keep_24_bits(dev, dtype, Hq, Hkv, n):
    """One key of weight x = 2^-e, and two of weight 1 whose values are minus x's first 8 bits and minus the next 8: what the
    output holds is the rest of x, at most 2^6 of its last places, so that dropping one place changes it by 2^-6.  Sums of
    the three are multiples of that place below 2^24 of them, which fp32 holds in any order; the weights' sum and the
    division may round differently, and then the output by one step, against the kernel that multiplies probabilities in
    fp32 (taken for wide tables)."""
    from fastcache_amd.layers.attention import decode_attention
    B, scale, up = 16, 0.6931471805599453, 2.0 ** 15        # this scale times log2 e is 1 in fp32: exponents are exact
    case = synth.make_paged_case(seed=6, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n] * B, dtype=dtype)
    tables, wide = case.table_tensor("cpu"), case.table_tensor("cpu", 70)
    e = torch.randint(1, 256, (B, Hkv), generator=torch.Generator().manual_seed(9)) / 64
    pool, first = case.kv_cache[:, 0].clone(), tables[:, 0].long()
    pool[0] = 0
    pool[0, ..., 0] = -20                                   # the query's first element is 16: 2^-320 for the other keys
    rest = torch.exp2(-e.double()).float().double()
    for i, t in enumerate([0, n // 2, n - 1]):
        pool[0, first, t, :, 0] = (-e / 16).to(dtype) if i == 0 else 0
        part = torch.full_like(rest, -1.0) if i == 0 else rest.bfloat16().double()
        pool[1, first, t] = (-part * up).to(dtype).unsqueeze(-1)
        rest = rest if i == 0 else rest - part
    q = torch.zeros(B, Hq, 128, dtype=dtype)
    q[..., 0] = 16
    on_gpu, lens_t = pool.to(dev), torch.full((B,), n, dtype=torch.int32)
    got, fp32 = (decode_attention(q.to(dev), on_gpu[0], on_gpu[1], lens_t.to(dev), t.to(dev), scale).cpu().double()
                 for t in (tables, wide))
    assert float((fp32 != 0).double().mean()) > 0.9 and float(fp32.abs().max()) <= 2.0 ** -18 * up
    assert bool(((got - fp32).abs() <= torch.finfo(dtype).eps * fp32.abs()).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,wide", [(2, 2, 0), (4, 2, 0), (6, 2, 0), (8, 2, 0),
                                         (2, 2, 70), (8, 2, 70)])     # a table too wide for the column kernel
@pytest.mark.parametrize("lens", [[64, 250], [700, 300], [1500, 40] * 15])      # one workgroup a column; several; tiles per wavefront
def test_infinite_values_stay_infinite(dev, dtype, Hq, Hkv, wide, lens):
    """Groups of up to 4 heads: an infinity in V reaches the outputs of its dimension, with its sign and as that, whatever its
    key weighs above nothing: the largest weight, those of the other keys, 2^-60; two of different sign and NaN give NaN; the other dimensions
    are those of a cache without."""
    from fastcache_amd.layers.attention import decode_attention
    B, scale = len(lens), 128 ** -0.5
    case = synth.make_paged_case(seed=12, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=lens, dtype=dtype)
    pool, tables = case.kv_cache[:, 0].clone(), case.table_tensor("cpu", wide or None)
    q = torch.randn(B, Hq, 128, generator=torch.Generator().manual_seed(1)).to(dtype)
    q[..., 0] = 16
    pool[0, ..., 0] = 0
    inf, at = float("inf"), lambda b, t: (case.block_tables[b][t // 256], t % 256)
    for b, n in enumerate(lens):
        pool[(0, *at(b, 9))][:, 0], pool[(0, *at(b, n // 2))][:, 0] = 8, -32       # about 2^16 and 2^-65 of the others' weight
        v = [pool[(1, *at(b, t))] for t in (9, n // 2, 3, n - 2)]
        v[0][:, 5], v[0][:, 6], v[1][:, 7], v[1][:, 8], v[2][:, 64], v[3][:, 127] = inf, -inf, inf, -inf, inf, -inf
        v[0][:, 30], v[1][:, 30], v[2][:, 31] = inf, -inf, float("nan")
    tables_d, lens_t = tables.to(dev), torch.tensor(lens, dtype=torch.int32)
    got = decode_attention(q.to(dev), pool[0].to(dev), pool[1].to(dev), lens_t.to(dev), tables_d, scale).cpu().float()
    special = [5, 6, 7, 8, 30, 31, 64, 127]
    assert bool((got[..., [5, 7, 64]] == inf).all()) and bool((got[..., [6, 8, 127]] == -inf).all())
    assert bool(got[..., [30, 31]].isnan().all())
    finite = pool.clone()
    finite[1, ..., special] = 0
    ref = oattn.decode_attention(q, finite[0], finite[1], lens_t, tables, scale).float()
    rest = [d for d in range(128) if d not in special]
    # one key carries nearly all of the weight: outputs are as large as values, and both sides round theirs once (a step of
    # the type apart where the fp32 results, 1e-5 apart at most, lie on two sides of a middle)
    assert bool(((got - ref)[..., rest].abs() <= torch.finfo(dtype).eps * ref[..., rest].abs() + 1e-5).all())


def _launches(run, *names):
    """Names of the launches of ``run`` that contain one of ``names``.  A profile now and then holds nothing: the next one is
    asked.  That none holds any fails, unless none held the launch made beside them either: then there is nothing to look at."""
    works = False
    for _ in range(8):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA], acc_events=True) as prof:
            run()
            torch.ones(1, device="cuda")
            torch.cuda.synchronize()
        seen = [e.name for e in prof.events()]
        found = [n for n in seen if any(name in n for name in names)]
        if found:
            return found
        works |= any("FillFunctor" in n for n in seen)
    if works:
        pytest.fail(f"no profile holds any of {names}")
    pytest.skip("the profiler holds no launches in this process")


@pytest.mark.parametrize("Hq,Hkv,lens,plain,merges", [
    (14, 2, [700, 0, 255, 513], True, 0),         # columns of several ranges: their last workgroup merges
    (4, 2, [100, 256, 31], True, 0),              # one range a column
    (7, 1, [3600, 40], True, 2),                  # more ranges than the last workgroup takes
    (14, 2, [700, 0, 255, 513], False, 0),        # a layer of its own class: what it returns is copied
])
def test_bucket_graphs_hold_one_launch_per_layer(dev, Hq, Hkv, lens, plain, merges):
    """What a bucket's graph launches, and the layers' results in the static output, replay after replay with eager steps on
    the same layers between (which share the workspace and the counters)."""
    from fastcache_amd.engine.decode_graph import BucketedDecodeGraphs
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context

    class Doubled(Attention):
        def forward(self, q, k, v):
            return super().forward(q, k, v) * 2

    L, B, dtype = 2, len(lens), torch.bfloat16
    case = synth.make_paged_case(seed=61, num_layers=L, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    pool, tables = case.kv_cache.to(dev), case.table_tensor(dev)
    layers = [(Attention if plain else Doubled)(Hq, 128, 128 ** -0.5, Hkv) for _ in range(L)]
    for l, a in enumerate(layers):
        a.k_cache, a.v_cache = pool[0, l], pool[1, l]
    graphs = BucketedDecodeGraphs(layers, B, tables.shape[1], dtype, dev)
    graphs.capture_cudagraph()
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(L, B, h * 128, generator=g).to(dtype).to(dev) for h in (Hq, Hkv, Hkv))
    set_context(False, slot_mapping=torch.full((B,), -1, dtype=torch.int32, device=dev),
                context_lens=torch.tensor(lens, dtype=torch.int32, device=dev), block_tables=tables)
    try:
        got, kinds = [], ("decode_column_kernel", "decode_attn_kernel", "decode_merge_kernel")
        step = torch.empty_like(q)                   # the calls a capture records, made eagerly
        names = _launches(lambda: graphs._model(q, k, v, step), *kinds)
        assert [sum(kind in n for n in names) for kind in kinds] == [L, 0, merges]
        got.append(step)
        for _ in range(3):        # and the graph's launches, of which a profile may hold nothing, but never others
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA], acc_events=True) as prof:
                got.append(graphs.run(q, k, v).clone())
                torch.cuda.synchronize()
            held = [sum(kind in e.name for e in prof.events()) for kind in kinds]
            assert held[0] <= L and held[1] == 0 and held[2] <= merges
        for _ in range(3):
            with torch.inference_mode():
                graphs.graph_vars["outputs"].fill_(float("nan"))
            eager = torch.stack([a(q[l], k[l], v[l]) for l, a in enumerate(layers)])
            got.append(graphs.run(q, k, v).clone())
            torch.cuda.synchronize()
    finally:
        reset_context()
    for o in got:
        assert torch.equal(o.view(torch.int16), eager.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,lens,pages", [
    (14, 2, [384, 385, 257, 383, 0, 512], 2),           # the first workgroup's alone, or two ranges merged, either side of the border
    (2, 2, [384, 385, 641, 700], 3),
    (8, 2, ([640, 641, 513, 768] * 12)[:46], 3),        # ranges of 512
])
def test_sequences_that_reach_a_little_into_a_second_range(dev, dtype, Hq, Hkv, lens, pages):
    """Merged by the last workgroup, by a launch, or one workgroup's alone: the oracle's values, and the same bits whoever
    merges."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    B = len(lens)
    case = synth.make_paged_case(seed=71, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables, lens_t = case.table_tensor("cpu")[:, :pages].contiguous(), torch.tensor(lens, dtype=torch.int32)
    pool = case.kv_cache[:, 0]
    ref = oattn.decode_attention(q.view(B, Hq, 128), pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    layer, on_gpu = Attention(Hq, 128, 128 ** -0.5, Hkv), pool.to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    set_context(False, slot_mapping=torch.full((B,), -1, dtype=torch.int32, device=dev), context_lens=lens_t.to(dev),
                block_tables=tables.to(dev))
    try:
        eager = layer(q, k, v)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            held = layer(q, k, v)
        for _ in range(3):
            held.zero_()
            graph.replay()
            again = layer(q, k, v)
            torch.cuda.synchronize()
            assert torch.equal(held.view(torch.int16), eager.view(torch.int16))
            assert torch.equal(again.view(torch.int16), eager.view(torch.int16))
    finally:
        reset_context()
    assert float((eager.cpu().view(B, Hq, 128).float() - ref.float()).abs().max()) < 4e-3      # as above


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,B,most,launches", [
    (32, 32, 9, 256, 1), (32, 32, 17, 512, 1), (32, 32, 10, 768, 1), (32, 32, 17, 1024, 1), (32, 32, 9, 1025, 2), (32, 16, 70, 1025, 2), (6, 3, 128, 1300, 2), (6, 3, 129, 1300, 3),
    (32, 16, 33, 256, 1), (32, 16, 40, 900, 1),
    (32, 8, 64, 512, 1), (24, 8, 65, 768, 1), (32, 8, 33, 1024, 2),             # of 1024 tokens two workgroups do not fit
    (28, 4, 66, 768, 1), (32, 4, 129, 256, 2), (16, 8, 128, 256, 1), (32, 4, 129, 512, 3), (40, 4, 129, 256, 2)])      # 10 heads a group: two workgroups, which do not append
def test_more_columns_than_compute_units(dev, dtype, Hq, Hkv, B, most, launches):
    """Columns held whole by one workgroup each, which append the step's rows and write the output, or chunks that append (of up
    to 4 heads a group) and a merge: the launches of a layer, the caches' bytes and the oracle's values, an empty sequence among them, a row that belongs to no
    sequence and one that lies inside another sequence's range."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    lens = [(most * (i + 1)) // B - 1 for i in range(B)]
    lens[B // 2] = 0
    case = synth.make_paged_case(seed=81, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables, lens_t = case.table_tensor("cpu"), torch.tensor(lens, dtype=torch.int32)
    slots = torch.tensor([t[n // 256] * 256 + n % 256 for t, n in zip(case.block_tables, lens)], dtype=torch.int32)
    slots[1] = -1
    slots[2] = case.block_tables[B - 1][0] * 256 + 40
    pool = case.kv_cache[:, 0].clone()
    keep = slots >= 0
    for p, new in ((0, k), (1, v)):
        pool[p].view(-1, Hkv, 128)[slots[keep].long()] = new.view(B, Hkv, 128)[keep]
    ref = oattn.decode_attention(q.view(B, Hq, 128), pool[0], pool[1], lens_t, tables, 128 ** -0.5)
    ref[B // 2] = 0
    layer, on_gpu = Attention(Hq, 128, 128 ** -0.5, Hkv), case.kv_cache[:, 0].to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    set_context(False, slot_mapping=slots.to(dev), context_lens=lens_t.to(dev), block_tables=tables.to(dev))
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    try:
        got = [layer(q, k, v).cpu()]
        names = _launches(lambda: got.append(layer(q, k, v)), "decode_", "store_slots")
        assert len(names) == launches, names
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            held = layer(q, k, v)
        for _ in range(3):
            held.fill_(float("nan"))
            graph.replay()
            got.append(held.clone())
        torch.cuda.synchronize()
    finally:
        reset_context()
    assert torch.equal(on_gpu.cpu(), pool)
    for o in got:
        assert torch.equal(o.cpu().view(torch.int16), got[0].view(torch.int16))
    assert float((got[0].view(B, Hq, 128).float() - ref.float()).abs().max()) < 4e-3      # as above


def test_graphs_keep_their_scratch_when_the_layers_are_captured_again(dev):
    """Two sets of bucketed graphs over the same layers, the second capture of which replaces the layers' scratch: the first
    set still owns what its kernels write, and a ``forward`` set on one layer object is called as it was set."""
    from fastcache_amd.engine.decode_graph import BucketedDecodeGraphs
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    L, Hq, Hkv, lens, dtype = 2, 7, 1, [700, 1000], torch.bfloat16
    case = synth.make_paged_case(seed=62, num_layers=L, batch=2, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    pool, tables = case.kv_cache.to(dev), case.table_tensor(dev)
    layers = [Attention(Hq, 128, 128 ** -0.5, Hkv) for _ in range(L)]
    for l, a in enumerate(layers):
        a.k_cache, a.v_cache = pool[0, l], pool[1, l]
    plain = layers[1].forward
    layers[1].forward = lambda q, k, v: plain(q, k, v)
    sets = []
    for _ in range(2):
        sets.append(BucketedDecodeGraphs(layers, 2, tables.shape[1], dtype, dev))
        sets[-1].capture_cudagraph()
    a, b = (s._scratch for s in sets)
    assert layers[0].workspace is b[0] and a[0].data_ptr() != b[0].data_ptr() and a[1].data_ptr() != b[1].data_ptr()
    others = [torch.full_like(a[0], 255) for _ in range(8)]
    g = torch.Generator().manual_seed(8)
    q, k, v = (torch.randn(L, 2, h * 128, generator=g).to(dtype).to(dev) for h in (Hq, Hkv, Hkv))
    set_context(False, slot_mapping=torch.full((2,), -1, dtype=torch.int32, device=dev),
                context_lens=torch.tensor(lens, dtype=torch.int32, device=dev), block_tables=tables)
    try:
        outs = [s.run(q, k, v).clone() for s in sets for _ in range(3)]
    finally:
        reset_context()
    assert all(torch.equal(o.view(torch.int16), outs[0].view(torch.int16)) for o in outs)
    assert all(bool((t == 255).all()) for t in others)


def test_eager_calls_on_captured_layers_leave_the_graphs_counters_alone(dev):
    """The layers of bucketed graphs called eagerly, with a batch of the graphs' size and with a larger one, whose partial
    results do not fit the graphs' workspace: both may run beside a replay, so neither may count on the graphs' words (which hold
    numbers here that would have no workgroup of a column merge it)."""
    from fastcache_amd.engine.decode_graph import BucketedDecodeGraphs
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    Hq, Hkv, lens, dtype = 14, 2, [700, 513, 600, 900, 257, 800], torch.bfloat16
    case = synth.make_paged_case(seed=63, num_layers=1, batch=6, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    pool, tables = case.kv_cache.to(dev), case.table_tensor(dev)
    layers = [Attention(Hq, 128, 128 ** -0.5, Hkv) for _ in range(2)]
    for a in layers:
        a.k_cache, a.v_cache = pool[0, 0], pool[1, 0]
    fresh, layer = layers
    graphs = BucketedDecodeGraphs([layer], 2, tables.shape[1], dtype, dev)
    graphs.capture_cudagraph()
    workspace, arrivals = graphs._scratch
    assert bool((arrivals == 0).all()) and layer.workspace is workspace
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(6, h * 128, generator=g).to(dtype).to(dev) for h in (Hq, Hkv, Hkv))
    with torch.inference_mode():
        arrivals.fill_(1 << 20)
    try:
        for given in (None, arrivals):          # by the layer as it is, and handed to it
            for n in (2, 6):
                if given is not None and n == 2:
                    continue                    # counters that come with the workspace they are for are counted on
                layer.arrivals = given
                set_context(False, slot_mapping=torch.full((n,), -1, dtype=torch.int32, device=dev),
                            context_lens=torch.tensor(lens[:n], dtype=torch.int32, device=dev), block_tables=tables[:n])
                got, want = layer(q[:n], k[:n], v[:n]), fresh(q[:n], k[:n], v[:n])
                torch.cuda.synchronize()
                assert torch.equal(got.view(torch.int16), want.view(torch.int16))
                assert bool((arrivals == 1 << 20).all())
                to = torch.empty_like(want)
                assert fresh(q[:n], k[:n], v[:n], out=to) is to and torch.equal(to.view(torch.int16), want.view(torch.int16))
        layer.arrivals = None
        with torch.inference_mode():
            arrivals.zero_()
        set_context(False, slot_mapping=torch.full((2,), -1, dtype=torch.int32, device=dev),
                    context_lens=torch.tensor(lens[:2], dtype=torch.int32, device=dev), block_tables=tables[:2])
        for _ in range(3):
            replayed = graphs.run(q[None, :2], k[None, :2], v[None, :2]).clone()
            assert torch.equal(replayed[0].view(torch.int16), layer(q[:2], k[:2], v[:2]).view(torch.int16))
        assert bool((arrivals == 0).all())
    finally:
        reset_context()


@pytest.mark.parametrize("Hq,Hkv,B,pages,column", [
    (32, 32, 4, 6, True), (32, 32, 4, 7, False), (32, 32, 2, 18, False),      # ranges of 3 tiles for all compute units; of 4, 5
    (8, 8, 4, 20, True), (8, 8, 5, 18, False), (16, 8, 5, 18, True),          # 7 ranges of 3 tiles; 6, one and two heads a group
    (8, 8, 4, 32, True), (8, 8, 4, 28, False), (16, 8, 4, 28, True), (16, 8, 16, 11, False),      # 8 and 7 ranges of 4 tiles; 2 of 6
    (32, 32, 6, 6, True), (32, 32, 8, 6, False), (32, 16, 16, 6, True),       # whole columns of 6 tiles
    (32, 8, 12, 7, False), (32, 8, 12, 8, True), (32, 8, 12, 5, True), (32, 8, 16, 7, True)])
def test_which_kernel_takes_columns_of_several_tiles(dev, Hq, Hkv, B, pages, column):
    """Ranges of 3 and more tiles a wavefront for groups of up to 4 heads, on both sides of the rule between the column and
    the split kernel: which of them runs, and the oracle's values."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    dtype, hi = torch.bfloat16, pages * 256 - 1
    lens = [hi - (hi * 9 * b) // (10 * B) for b in range(B)]
    case = synth.make_paged_case(seed=91, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[n + 1 for n in lens], dtype=dtype)
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn(B, h * 128, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    tables, lens_t = case.table_tensor("cpu"), torch.tensor(lens, dtype=torch.int32)
    slots = torch.tensor([t[n // 256] * 256 + n % 256 for t, n in zip(case.block_tables, lens)], dtype=torch.int32)
    ref = oattn.decode_attention(q.view(B, Hq, 128), case.kv_cache[0, 0], case.kv_cache[1, 0], lens_t, tables, 128 ** -0.5)
    layer, on_gpu = Attention(Hq, 128, 128 ** -0.5, Hkv), case.kv_cache[:, 0].to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    set_context(False, slot_mapping=slots.to(dev), context_lens=lens_t.to(dev), block_tables=tables.to(dev))
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    try:
        got = layer(q, k, v).cpu()
        names = _launches(lambda: layer(q, k, v), "decode_column_kernel<", "decode_attn_kernel<")
    finally:
        reset_context()
    assert ["decode_column_kernel<" in n for n in names] == [column]
    assert float((got.view(B, Hq, 128).float() - ref.float()).abs().max()) < 4e-3      # as above


@pytest.mark.parametrize("Hq,Hkv,B", [(32, 32, 17), (32, 16, 33), (24, 8, 65)])     # 1, 2 and 3 heads a group; of 3, 768 tokens
def test_whole_columns_are_summed_as_accurately_as_chunks(dev, Hq, Hkv, B):
    """Columns that one workgroup holds whole, on values whose sums grow for half of the context and cancel in the other half,
    so that the errors of the fp32 sums show in the rounded result.  A tile's products are summed by themselves: 0.54 to 0.60 of
    the distance from 64 bits that fp32 sums of 256 tokens at a time, merged, have (0.82 to 1.0 as one sum over all tiles of a
    wavefront, which on values that do not cancel is up to 1.1 of it); the bound lies between."""
    from fastcache_amd.layers import Attention
    from fastcache_amd.utils.context import reset_context, set_context
    S = 768 if Hq // Hkv == 3 else 1024
    lens, dtype, half = [S, S] + [8] * (B - 2), torch.float16, S // 2
    case = synth.make_paged_case(seed=95, num_layers=1, batch=B, num_kv_heads=Hkv, seq_lens=[S, S] + [8] * (B - 2), dtype=dtype)
    g = torch.Generator().manual_seed(4)
    kd = torch.randn(2, S, Hkv, 128, generator=g).to(dtype)
    kd[:, half:] = kd[:, :half]                                         # the second half weighs what the first does
    vd = torch.empty(2, S, Hkv, 128, dtype=dtype)
    vd[:, :half] = (torch.randn(2, half, Hkv, 128, generator=g) * 256).to(dtype)
    vd[:, half:] = -vd[:, :half] + (0.25 * torch.randint(-1, 2, (2, half, Hkv, 128), generator=g)).to(dtype)
    pool = case.kv_cache[:, 0]
    for b in range(2):
        for t in range(0, S, 256):
            pool[0, case.block_tables[b][t // 256]], pool[1, case.block_tables[b][t // 256]] = kd[b, t:t + 256], vd[b, t:t + 256]
    q, k, v = ((torch.randn(B, h * 128, generator=g) * 0.5).to(dtype) for h in (Hq, Hkv, Hkv))
    layer, on_gpu = Attention(Hq, 128, 128 ** -0.5, Hkv), pool.to(dev)
    layer.k_cache, layer.v_cache = on_gpu[0], on_gpu[1]
    set_context(False, slot_mapping=torch.full((B,), -1, dtype=torch.int32, device=dev),
                context_lens=torch.tensor(lens, dtype=torch.int32, device=dev), block_tables=case.table_tensor(dev))
    q_d, k_d, v_d = q.to(dev), k.to(dev), v.to(dev)
    try:
        got = layer(q_d, k_d, v_d).cpu()[:2].view(2, Hkv, Hq // Hkv, 128).double()
        names = _launches(lambda: layer(q_d, k_d, v_d), "decode_")
    finally:
        reset_context()
    assert len(names) == 1 and "decode_attn_kernel" in names[0]
    logits = torch.matmul(q[:2].view(2, Hkv, Hq // Hkv, 128).double(), kd.permute(0, 2, 3, 1).contiguous().double()) * 128 ** -0.5
    p64 = logits.softmax(-1)
    exact = torch.matmul(p64, vd.permute(0, 2, 1, 3).contiguous().double())
    e = (logits - logits.amax(-1, keepdim=True)).exp().float()           # chunks of 256: one sum a token slot of 16, then those
    acc = torch.zeros(2, Hkv, Hq // Hkv, 128)
    for c in range(0, S, 256):
        slots = torch.zeros(16, 2, Hkv, Hq // Hkv, 128)
        for t in range(256):
            s = (t // 32 % 4) * 4 + t % 4
            slots[s] = (slots[s].double() + e[..., c + t, None].double() * vd[:, c + t, :, None].double()).float()       # one rounding
        part = torch.zeros_like(acc)
        for s in slots:
            part += s
        acc += part
    chunks = (acc / e.double().sum(-1, keepdim=True).float()).to(dtype).double()
    err, ref = float((got - exact).norm()), float((chunks - exact).norm())
    # what rounding the result leaves is the same for all: the rest of the errors is compared
    last = float((exact.to(dtype).double() - exact).norm()) ** 2
    ratio = ((err ** 2 - last) / (ref ** 2 - last)) ** 0.5
    assert ratio < 0.7, ratio


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 12])                                                  # a workgroup a column; several
@pytest.mark.parametrize("Hq,Hkv,B,apart", [(8, 8, 33, 1), (32, 8, 33, 32), (56, 8, 33, 2),          # 1, 4 and 7 heads a group
                                            (4, 4, 66, 65), (4, 4, 130, 129), (4, 4, 200, 128)])
def test_sequences_that_share_a_prefix_read_what_copies_of_it_hold(dev, dtype, width, Hq, Hkv, B, apart):
    """The split kernel loads ranges of a prefix that two tables name in another way than those of one sequence alone: the
    same bits as from a private copy of the pages, for sequences next to each other in the batch and up to its other end,
    and with tables padded by entries that look like another sequence's page."""
    g = torch.Generator().manual_seed(B)
    lens = [40 + 7 * b % 300 for b in range(B)]
    lens[0], lens[apart] = 700, 600
    q = torch.randn(B, Hq, 128, generator=g).to(dtype).to(dev)
    pages = sum(-(-n // 256) for n in lens)
    pool = torch.randn(2, 1, pages + 2, 256, Hkv, 128, generator=g).to(dtype).to(dev)
    tables, at = torch.full((B, width), -1, dtype=torch.int32), 0
    for b, n in enumerate(lens):
        for i in range(-(-n // 256)):
            tables[b, i], at = at, at + 1
    lens_d = torch.tensor(lens, dtype=torch.int32, device=dev)
    shared = tables.clone()
    shared[apart, :2] = shared[0, :2]                                   # two of three pages in common
    copied = tables.clone()
    copied[apart, :2] = torch.tensor([pages, pages + 1], dtype=torch.int32)
    for i in range(2):
        pool[:, :, pages + i] = pool[:, :, int(shared[0, i])]
    decoys = copied.clone()
    decoys[decoys < 0] = int(copied[0, 0])
    ws = ops.decode_attn_workspace(B, Hq, width * 256, dev)

    def run(t):
        t = t.to(dev)
        kv = [_lib.paged_view(pool[p], t, None, width * 256) for p in range(2)]
        return ops.decode_attn(*kv, 0, q, lens_d, 128 ** -0.5, ws).cpu()

    assert all("decode_attn_kernel<" in n for n in _launches(lambda: run(shared), "decode_column_kernel<", "decode_attn_kernel<"))
    want = run(copied)
    assert torch.equal(run(shared).view(torch.int16), want.view(torch.int16))
    assert torch.equal(run(decoys).view(torch.int16), want.view(torch.int16))
    ref = oattn.decode_attention(q.cpu(), pool[0, 0].cpu(), pool[1, 0].cpu(), lens_d.cpu(), shared, 128 ** -0.5)
    assert float((want.float() - ref.float()).abs().max()) < 4e-3      # as above
