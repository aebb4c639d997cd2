"""The KV write folded into the attention launch (bf16 and E4M3FN pools).

``forward_mixed`` and ``Attention.forward`` run the library's own store inside
the attention launch: the launch writes the step's new K/V rows to their slots
and reads the new tokens from those rows instead of the pool.  The reference
order is store first, then attend (nanovllm/layers/mixed_attention.py:33-34,
nanovllm/layers/attention.py:66-67); these tests check that the folded launch
gives the same output and the same pool bytes, bit for bit, as that order run
as two launches (a ``store_fn`` that is not the library's own store takes the
two-launch path), on the benchmark workloads (decode rows, prefill rows with
and without history) and through the V0 branches, including slot -1 padding.
"""
import pytest
import torch

from slo_attn import (Attention, MixedAttentionContext, forward_mixed, reserve_workspace, reset_context,
                      set_context, store_kvcache)
import workloads
from slo_attn import _lib
from slo_attn.ops import paged_attention, workspace_events
from types import SimpleNamespace

pytestmark = pytest.mark.gpu


def _two_launch_store(*args):
    store_kvcache(*args)


@pytest.mark.parametrize("index", [0, 1, 2, 3])
def test_forward_mixed_folded_store_equals_store_then_attend(device, index):
    w = workloads.config(index)
    d = workloads.to_device(w, device)
    ctx = SimpleNamespace(mixed=d["meta"], slot_mapping=d["slot_mapping"])
    q, k, v = d["q"], d["k"], d["v"]
    kc0, vc0 = w.k_cache.to(device), w.v_cache.to(device)
    if w.num_decode:
        reserve_workspace(device, w.num_decode, max(len(t) for t in w.decode_tables) * w.block_size, 32, 8, 128)
    kc1, vc1 = kc0.clone(), vc0.clone()
    ref = forward_mixed(q, k, v, kc0, vc0, ctx, w.scale, _two_launch_store)
    got = forward_mixed(q, k, v, kc1, vc1, ctx, w.scale, store_kvcache)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(kc1.view(torch.int16), kc0.view(torch.int16))
    assert torch.equal(vc1.view(torch.int16), vc0.view(torch.int16))


def _fp8_pools(w, device):
    """E4M3FN codes and scales of the workload's bf16 pool, written by the store kernel."""
    base_k, base_v = w.k_cache.to(device), w.v_cache.to(device)
    nblk, bs, hkv, dh = base_k.shape
    kc = torch.empty(nblk, bs, hkv, dh, dtype=torch.uint8, device=device)
    vc = torch.empty_like(kc)
    ks = torch.empty(nblk, bs, hkv, dtype=torch.float32, device=device)
    vs = torch.empty_like(ks)
    slots = torch.arange(nblk * bs, dtype=torch.int32, device=device)
    store_kvcache(base_k.view(-1, hkv, dh), base_v.view(-1, hkv, dh), kc, vc, slots, ks, vs)
    return kc, vc, ks, vs


def _fp8_fold_matches_store_then_attend(device, meta, slots, q, k, v, pools, scale, history):
    """The folded E4M3FN launch against the store kernel followed by the same
    launch: outputs, codes and scales bit for bit."""
    d = meta.num_decode
    nr = (meta.prefill_cu_q.numel() - 1) if meta.num_prefill_tokens else 0
    p1 = tuple(t.clone() for t in pools)

    def launch(kc, vc, ks, vs, **store):
        return paged_attention(
            q, kc, vc, scale, num_kv_heads=k.shape[1], k_scale=ks, v_scale=vs, num_decode=d,
            decode_lens=meta.decode_lens, decode_tables=meta.decode_tables, num_prefill=nr,
            prefill_cu_q=meta.prefill_cu_q, prefill_cu_k=meta.prefill_cu_k, max_q=meta.max_q, max_k=meta.max_k,
            prefill_tables=meta.prefill_tables if history else None, k=None if history else k[d:],
            v=None if history else v[d:], **store)
    store_kvcache(k, v, pools[0], pools[1], slots, pools[2], pools[3])
    ref = launch(*pools)
    got = launch(*p1, store_slot_mapping=slots, new_k=k, new_v=v)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    for a_, b_ in zip(p1, pools):
        assert torch.equal(a_.view(torch.uint8), b_.view(torch.uint8))


@pytest.mark.parametrize("index", [0, 1, 2, 3, 4])
def test_folded_fp8_store_equals_store_then_attend(device, index):
    # E4M3FN pool: the launch quantises the new rows as the store kernel does
    # (decode rows' newest tokens, prefill tiles of new tokens, the tile that
    # straddles a prefix, the write at the end) -- same codes, scales and
    # outputs, bit for bit, as the store kernel followed by the launch; with
    # the rows reading the pool (history) and, where the workload allows,
    # without.  forward_mixed folds pure decode steps.
    w = workloads.config(index)
    d = workloads.to_device(w, device)
    if w.num_decode:
        reserve_workspace(device, w.num_decode, max(len(t) for t in w.decode_tables) * w.block_size, 32, 8, 128)
    for history in ((True, False) if not w.has_history else (True,)):
        _fp8_fold_matches_store_then_attend(device, d["meta"], d["slot_mapping"], d["q"], d["k"], d["v"],
                                            _fp8_pools(w, device), w.scale, history)
    if not w.prefill_q:  # a pure decode step: forward_mixed takes the folded launch
        ctx = SimpleNamespace(mixed=d["meta"], slot_mapping=d["slot_mapping"])
        p0, p1 = _fp8_pools(w, device), _fp8_pools(w, device)
        ref = forward_mixed(d["q"], d["k"], d["v"], p0[0], p0[1], ctx, w.scale, _two_launch_store, p0[2], p0[3])
        got = forward_mixed(d["q"], d["k"], d["v"], p1[0], p1[1], ctx, w.scale, store_kvcache, p1[2], p1[3])
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
        for a_, b_ in zip(p1, p0):
            assert torch.equal(a_.view(torch.uint8), b_.view(torch.uint8))


def test_folded_fp8_store_on_small_blocks_and_straddled_prefixes(device):
    # 64-token blocks, prefixes inside a key tile (100, 700: the tile holding
    # the prefix end is written to the pool by each item before it is read)
    # and decode rows whose newest token sits at a 16/32-token step edge.
    from attn_cases import Case
    case = Case([31, 63, 300, 1000], [100, 700, 0], [45, 90, 33], bs=64, seed=21, kv_fp8=True)
    kc, vc = case.cpu_pools()
    codes, scales = case.fp8_pools(kc, vc)
    pools = tuple(torch.from_numpy(x.copy()).to(device) for x in (*codes, *scales))
    slots = torch.tensor(case.slots, dtype=torch.int32, device=device)
    _fp8_fold_matches_store_then_attend(device, case.meta(device), slots, case.q.to(device), case.k.to(device),
                                        case.v.to(device), pools, case.scale, True)


def test_folded_store_skips_padding_slots_and_matches_explicit_launch(device):
    # Decode rows of a captured batch: real rows, then padding rows (slot -1,
    # length 0).  The folded launch must leave every byte but the real slots
    # alone and give the outputs of store + attend.
    g = torch.Generator().manual_seed(9)
    hq, hkv, dh, bs, nblk = 32, 8, 128, 256, 6
    pool_k = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    pool_v = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    lens = [300, 1, 257, 0, 0]
    tables = torch.tensor([[0, 1, -1], [2, -1, -1], [3, 4, -1], [-1, -1, -1], [5, 5, 5]],
                          dtype=torch.int32, device=device)
    slots = torch.tensor([bs + 43, 2 * bs, 4 * bs + 0, -1, -1], dtype=torch.int32, device=device)
    B = len(lens)
    q = torch.randn(B, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k = torch.randn(B, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    v = torch.randn(B, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    dl = torch.tensor(lens, dtype=torch.int32, device=device)
    reserve_workspace(device, B, 3 * bs, hq, hkv, dh)
    kc0, vc0 = pool_k.clone(), pool_v.clone()
    store_kvcache(k, v, kc0, vc0, slots)
    ref = paged_attention(q, kc0, vc0, dh ** -0.5, num_kv_heads=hkv, num_decode=B, decode_lens=dl,
                          decode_tables=tables)
    kc1, vc1 = pool_k.clone(), pool_v.clone()
    got = paged_attention(q, kc1, vc1, dh ** -0.5, num_kv_heads=hkv, num_decode=B, decode_lens=dl,
                          decode_tables=tables, store_slot_mapping=slots, new_k=k, new_v=v)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(kc1.view(torch.int16), kc0.view(torch.int16))
    assert torch.equal(vc1.view(torch.int16), vc0.view(torch.int16))


def test_v0_branches_fold_the_store(device):
    # Cold prefill, prefix-cache prefill and decode through Attention.forward
    # (bf16 pool: folded) against the same calls with the store run first and
    # kv_stored=True (two launches).
    g = torch.Generator().manual_seed(11)
    hq, hkv, dh, bs, nblk = 32, 8, 128, 256, 8
    a1 = Attention(hq, dh, dh ** -0.5, hkv)
    a2 = Attention(hq, dh, dh ** -0.5, hkv)
    base_k = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    base_v = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    a1.k_cache, a1.v_cache = base_k.clone(), base_v.clone()
    a2.k_cache, a2.v_cache = base_k.clone(), base_v.clone()

    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device=device)

    def both(q, k, v, **ctx):
        set_context(**ctx)
        try:
            got = a1(q, k, v)
            store_kvcache(k, v, a2.k_cache, a2.v_cache, ctx["slot_mapping"])
            ref = a2(q, k, v, kv_stored=True)
        finally:
            reset_context()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
        assert torch.equal(a1.k_cache.view(torch.int16), a2.k_cache.view(torch.int16))
        assert torch.equal(a1.v_cache.view(torch.int16), a2.v_cache.view(torch.int16))

    # cold prefill: two prompts of 100 and 300 tokens in blocks 0 and 1-2
    lq = [100, 300]
    T = sum(lq)
    q = torch.randn(T, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k = torch.randn(T, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    v = torch.randn(T, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    slots = list(range(0, 100)) + list(range(bs, bs + 300))
    both(q, k, v, is_prefill=True, cu_seqlens_q=i32([0, 100, T]), cu_seqlens_k=i32([0, 100, T]),
         max_seqlen_q=300, max_seqlen_k=300, slot_mapping=i32(slots))
    # prefix-cache prefill: row 0 has 256 cached tokens (block 3) + 60 new (block 4)
    q = torch.randn(60, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k = torch.randn(60, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    v = torch.randn(60, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    both(q, k, v, is_prefill=True, cu_seqlens_q=i32([0, 60]), cu_seqlens_k=i32([0, 316]),
         max_seqlen_q=60, max_seqlen_k=316, slot_mapping=i32(list(range(4 * bs, 4 * bs + 60))),
         block_tables=i32([[3, 4]]))
    # decode: the two prompts' next tokens plus a padded row
    q = torch.randn(3, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k = torch.randn(3, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    v = torch.randn(3, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    reserve_workspace(device, 3, 2 * bs, hq, hkv, dh)
    both(q, k, v, is_prefill=False, slot_mapping=i32([100, bs + 300, -1]), context_lens=i32([101, 301, 0]),
         block_tables=i32([[0, -1], [1, 2], [-1, -1]]))


def test_fold_rejects_wide_fp8_groups_and_bad_rows(device):
    # An E4M3FN pool with more than 8 query heads per kv head cannot carry the
    # write (forward_mixed then runs the store kernel first).
    hq, hkv, dh, bs = 16, 1, 128, 256
    q = torch.zeros(2, hq, dh, dtype=torch.bfloat16, device=device)
    k = torch.zeros(2, hkv, dh, dtype=torch.bfloat16, device=device)
    kc = torch.zeros(2, bs, hkv, dh, dtype=torch.uint8, device=device)
    sc = torch.ones(2, bs, hkv, device=device)
    dl = torch.tensor([1, 1], dtype=torch.int32, device=device)
    tb = torch.tensor([[0], [1]], dtype=torch.int32, device=device)
    slots = torch.tensor([0, bs], dtype=torch.int32, device=device)
    with pytest.raises(ValueError):
        paged_attention(q, kc, kc.clone(), 1.0, num_kv_heads=hkv, k_scale=sc, v_scale=sc.clone(), num_decode=2,
                        decode_lens=dl, decode_tables=tb, store_slot_mapping=slots, new_k=k, new_v=k)
    hq, hkv = 8, 2
    q = torch.zeros(2, hq, dh, dtype=torch.bfloat16, device=device)
    k = torch.zeros(2, hkv, dh, dtype=torch.bfloat16, device=device)
    kb = torch.zeros(2, bs, hkv, dh, dtype=torch.bfloat16, device=device)
    with pytest.raises(ValueError):
        paged_attention(q, kb, kb.clone(), 1.0, num_kv_heads=hkv, num_decode=2, decode_lens=dl, decode_tables=tb,
                        store_slot_mapping=slots[:1].contiguous(), new_k=k[:1], new_v=k[:1])


@pytest.mark.parametrize("prefixes", [(300, 77, 0), (64, 511, 1000)])
def test_folded_store_with_prefixes_inside_a_key_tile(device, prefixes):
    # Prefill rows whose cached prefix ends inside a 64-key tile (a chunked
    # prompt): that tile mixes pool keys and new keys; plus decode rows.  The
    # folded launch must equal the store followed by the attention launch.
    g = torch.Generator().manual_seed(13)
    hq, hkv, dh, bs, nblk = 32, 8, 128, 256, 24
    pool_k = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    pool_v = torch.randn(nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    perm = torch.randperm(nblk, generator=g).tolist()
    chunks = [130, 45, 200]
    dec_lens = [700, 33]
    rows, tables, slots, nxt = [], [], [], 0

    def take(n_tokens):
        nonlocal nxt
        nb = (n_tokens + bs - 1) // bs
        t = perm[nxt:nxt + nb]
        nxt += nb
        return t

    dec_tables = []
    for L in dec_lens:
        t = take(L)
        dec_tables.append(t)
        slots.append(t[(L - 1) // bs] * bs + (L - 1) % bs)
    pf_tables = []
    for pfx, n in zip(prefixes, chunks):
        t = take(pfx + n)
        pf_tables.append(t)
        slots += [t[j // bs] * bs + j % bs for j in range(pfx, pfx + n)]
    width = max(len(t) for t in dec_tables + pf_tables)

    def pad(ts):
        return torch.tensor([t + [-1] * (width - len(t)) for t in ts], dtype=torch.int32, device=device)

    T = len(dec_lens) + sum(chunks)
    q = torch.randn(T, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k = torch.randn(T, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    v = torch.randn(T, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    cu_q = [0]
    cu_k = [0]
    for pfx, n in zip(prefixes, chunks):
        cu_q.append(cu_q[-1] + n)
        cu_k.append(cu_k[-1] + pfx + n)
    meta = MixedAttentionContext(len(dec_lens), sum(chunks), torch.tensor(dec_lens, dtype=torch.int32, device=device),
                                 pad(dec_tables), torch.tensor(cu_q, dtype=torch.int32, device=device),
                                 torch.tensor(cu_k, dtype=torch.int32, device=device), pad(pf_tables), max(chunks),
                                 max(p + n for p, n in zip(prefixes, chunks)), True)
    ctx = SimpleNamespace(mixed=meta, slot_mapping=torch.tensor(slots, dtype=torch.int32, device=device))
    reserve_workspace(device, len(dec_lens), width * bs, hq, hkv, dh)
    kc0, vc0 = pool_k.clone(), pool_v.clone()
    kc1, vc1 = pool_k.clone(), pool_v.clone()
    ref = forward_mixed(q, k, v, kc0, vc0, ctx, dh ** -0.5, _two_launch_store)
    got = forward_mixed(q, k, v, kc1, vc1, ctx, dh ** -0.5, store_kvcache)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(kc1.view(torch.int16), kc0.view(torch.int16))
    assert torch.equal(vc1.view(torch.int16), vc0.view(torch.int16))
    # strided new rows (a view of a fused projection) take the two-launch path
    wide = torch.randn(T, 3, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    ks, vs = wide[:, 1], wide[:, 2]
    kc2, vc2 = pool_k.clone(), pool_v.clone()
    kc3, vc3 = pool_k.clone(), pool_v.clone()
    ref2 = forward_mixed(q, ks, vs, kc2, vc2, ctx, dh ** -0.5, _two_launch_store)
    got2 = forward_mixed(q, ks, vs, kc3, vc3, ctx, dh ** -0.5, store_kvcache)
    torch.cuda.synchronize()
    assert torch.equal(got2.view(torch.int16), ref2.view(torch.int16))
    assert torch.equal(kc3.view(torch.int16), kc2.view(torch.int16))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("rows,hi,hkv", [(1, 700, 8), (5, 300, 4), (40, 4000, 8), (150, 4096, 8)])
def test_decode_folds_views_of_the_qkv_projection(device, fp8, rows, hi, hkv):
    # Decode steps fold K/V rows that are views of the fused projection's
    # output (row stride larger than a pool row), bf16 and E4M3FN, in the
    # direct kernel and (150 long rows) the work lists: output and pool bytes
    # of the store kernel followed by the attention launch, through
    # Attention.forward's V0 decode branch and through forward_mixed.
    g = torch.Generator().manual_seed(rows + hkv)
    hq, dh, bs = 4 * hkv, 128, 256
    lens = torch.randint(1, hi + 1, (rows,), generator=g).tolist()
    lens[0] = hi
    per = [(n + bs - 1) // bs for n in lens]
    nblk, width = sum(per) + 1, max(per)
    perm = torch.randperm(nblk, generator=g).tolist()
    tables, at = [], 0
    for n in per:
        tables.append(perm[at:at + n])
        at += n
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    slots = i32([t[(n - 1) // bs] * bs + (n - 1) % bs for t, n in zip(tables, lens)])
    padded, dl = i32([t + [-1] * (width - len(t)) for t in tables]), i32(lens)
    qkv = torch.randn(rows, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, k, v = (t.view(rows, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q = q.contiguous()
    reserve_workspace(device, rows, width * bs, hq, hkv, dh)
    base = torch.randn(2, nblk, bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)

    def pools():
        if not fp8:
            return [base[0].clone(), base[1].clone()]
        p = [torch.empty(nblk, bs, hkv, dh, dtype=torch.uint8, device=device) for _ in range(2)]
        s = [torch.empty(nblk, bs, hkv, device=device) for _ in range(2)]
        every = torch.arange(nblk * bs, dtype=torch.int32, device=device)
        store_kvcache(base[0].view(-1, hkv, dh), base[1].view(-1, hkv, dh), *p, every, *s)
        return p + s

    ctx = SimpleNamespace(mixed=MixedAttentionContext(rows, 0, dl, padded, None, None, None, 0, 0),
                          slot_mapping=slots)
    ref_pools, got_pools, v0_pools = pools(), pools(), pools()
    ref = forward_mixed(q, k, v, ref_pools[0], ref_pools[1], ctx, dh ** -0.5, _two_launch_store, *ref_pools[2:])
    got = forward_mixed(q, k, v, got_pools[0], got_pools[1], ctx, dh ** -0.5, store_kvcache, *got_pools[2:])
    attn = Attention(hq, dh, dh ** -0.5, hkv)
    attn.k_cache, attn.v_cache = v0_pools[:2]
    if fp8:
        attn.k_scale, attn.v_scale = v0_pools[2:]
    set_context(False, slot_mapping=slots, context_lens=dl, block_tables=padded)
    v0 = attn(q, k, v).squeeze(1)
    reset_context()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
    assert torch.equal(v0.view(torch.int16), ref.view(torch.int16))
    for a_, b_, c_ in zip(ref_pools, got_pools, v0_pools):
        assert torch.equal(a_.view(torch.uint8), b_.view(torch.uint8))
        assert torch.equal(a_.view(torch.uint8), c_.view(torch.uint8))
    # Without the flag for strided rows the launch refuses them, as it does
    # beside prefill rows.
    if rows > 1:
        with pytest.raises(RuntimeError):
            paged_attention(q, got_pools[0], got_pools[1], dh ** -0.5, num_kv_heads=hkv,
                            k_scale=got_pools[2] if fp8 else None, v_scale=got_pools[3] if fp8 else None,
                            num_decode=rows, decode_lens=dl, decode_tables=padded, store_slot_mapping=slots,
                            new_k=k, new_v=v)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens,hq,hkv", [([1], 32, 8), ([31, 33, 1, 64, 100], 8, 8), ([700, 257], 64, 8),
                                         ([1813, 346, 16], 32, 8)])
def test_cold_prefill_items_write_the_new_rows(device, fp8, lens, hq, hkv):
    # A launch of cold prefill rows reads no pool: its items write their own
    # blocks' tokens (all kv heads, head groups once), and new rows outside
    # every prefill row follow (here three padding tokens, one with a slot).
    # Views of the QKV projection and contiguous rows, through
    # Attention.forward's V0 branch and forward_mixed, against the store kernel
    # followed by the launch: outputs and pool bytes.
    g = torch.Generator().manual_seed(sum(lens) + hq)
    dh, bs, n = 128, 256, sum(lens)
    total, nblk = n + 3, (n + 3 + 255) // 256 + 2
    slot = torch.randperm(nblk * bs, generator=g)[:total].to(torch.int32)
    slot[n], slot[n + 2], slot[0] = -1, nblk * bs, -1  # skipped: -1 and past the pool
    slots = slot.to(device)
    qkv = torch.randn(total, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, k, v = (t.view(total, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q = q.contiguous()
    cu = [0]
    for x in lens:
        cu.append(cu[-1] + x)
    cu = torch.tensor(cu, dtype=torch.int32, device=device)
    reserve_workspace(device, 0, 0, hq, hkv, dh)

    def pools():
        if not fp8:
            return [torch.full((nblk, bs, hkv, dh), x, dtype=torch.bfloat16, device=device) for x in (3.0, -3.0)]
        return ([torch.full((nblk, bs, hkv, dh), 7, dtype=torch.uint8, device=device) for _ in range(2)]
                + [torch.full((nblk, bs, hkv), 9.0, device=device) for _ in range(2)])

    meta = MixedAttentionContext(0, total, None, None, cu, cu, None, max(lens), max(lens), False)
    ctx = SimpleNamespace(mixed=meta, slot_mapping=slots)
    for kk, vv in ((k, v), (k.contiguous(), v.contiguous())):
        a, b, c = pools(), pools(), pools()
        ref = forward_mixed(q, kk, vv, a[0], a[1], ctx, dh ** -0.5, _two_launch_store, *a[2:])
        got = forward_mixed(q, kk, vv, b[0], b[1], ctx, dh ** -0.5, store_kvcache, *b[2:])
        attn = Attention(hq, dh, dh ** -0.5, hkv)
        attn.k_cache, attn.v_cache = c[:2]
        if fp8:
            attn.k_scale, attn.v_scale = c[2:]
        set_context(True, cu, cu, max(lens), max(lens), slots)
        v0 = attn(q, kk, vv)
        reset_context()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
        assert torch.equal(v0.view(torch.int16), ref.view(torch.int16))
        for x, y, z in zip(a, b, c):
            assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
            assert torch.equal(x.view(torch.uint8), z.view(torch.uint8))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("strided", [False, True])
def test_decode_launch_stores_every_new_row(device, fp8, strided):
    # One decode row and 900 query rows, all with a slot: the launch's small
    # grid (64 workgroups) takes the new rows in several turns.  Pool bytes of
    # the store kernel, and zeros in the output rows past the decode row.
    g = torch.Generator().manual_seed(3)
    rows, hq, hkv, dh, bs, nblk = 900, 32, 8, 128, 256, 6
    slots = torch.randperm((nblk - 1) * bs, generator=g)[:rows].to(torch.int32)
    slots[0] = (nblk - 1) * bs + 69
    slots, dl = slots.to(device), torch.tensor([70], dtype=torch.int32, device=device)
    table = torch.tensor([[nblk - 1]], dtype=torch.int32, device=device)
    qkv = torch.randn(rows, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, k, v = (t.view(rows, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q = q.contiguous()
    if not strided:
        k, v = k.contiguous(), v.contiguous()
    ctx = SimpleNamespace(mixed=MixedAttentionContext(1, 0, dl, table, None, None, None, 0, 0), slot_mapping=slots)
    outs, pools = [], []
    for store in (_two_launch_store, store_kvcache):
        if fp8:
            pool = [torch.full((nblk, bs, hkv, dh), 7, dtype=torch.uint8, device=device) for _ in range(2)]
            pool += [torch.full((nblk, bs, hkv), 9.0, device=device) for _ in range(2)]
        else:
            pool = [torch.full((nblk, bs, hkv, dh), x, dtype=torch.bfloat16, device=device) for x in (3.0, -3.0)]
        outs.append(forward_mixed(q, k, v, pool[0], pool[1], ctx, dh ** -0.5, store, *pool[2:]))
        pools.append(pool)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)) and not outs[1][1:].any()
    for a, b in zip(*pools):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("head,length,rows", [(0, 40, 1500), (70, 33, 200), (31, 1, 65), (33, 0, 40)])
def test_cold_launch_writes_rows_outside_every_prefill_row(device, fp8, head, length, rows):
    # A cold prefill row at [head, head + length) of `rows` new rows: the rows
    # before and after it are written in blocks of 32, at the edges of a block
    # and with blocks whose slots are all -1 or past the pool, in part or not
    # at all.  Pool bytes of the store kernel; the attention output is that of
    # the launch without the write.
    g = torch.Generator().manual_seed(head + rows)
    hq, hkv, dh, bs, nblk = 16, 4, 128, 256, 7
    slot = torch.randperm(nblk * bs, generator=g)[:rows].to(torch.int32)
    slot[head + length:head + length + 32] = -1
    slot[-40:-1] = -1
    slot[head // 2:head // 2 + 3] = nblk * bs
    slots = slot.to(device)
    q = torch.randn(rows, hq, dh, generator=g).to(torch.bfloat16).to(device)
    k, v = (torch.randn(rows, hkv, dh, generator=g).to(torch.bfloat16).to(device) for _ in range(2))
    cu = torch.tensor([head, head + length], dtype=torch.int32, device=device)
    reserve_workspace(device, 0, 0, hq, hkv, dh)
    a, b = [], []
    for pool in (a, b):
        if fp8:
            pool += [torch.full((nblk, bs, hkv, dh), 7, dtype=torch.uint8, device=device) for _ in range(2)]
            pool += [torch.full((nblk, bs, hkv), 9.0, device=device) for _ in range(2)]
        else:
            pool += [torch.full((nblk, bs, hkv, dh), x, dtype=torch.bfloat16, device=device) for x in (3.0, -3.0)]
    common = dict(num_kv_heads=hkv, num_prefill=1, prefill_cu_q=cu, prefill_cu_k=cu, max_q=length, max_k=length, k=k, v=v)
    store_kvcache(k, v, a[0], a[1], slots, *a[2:])
    outs = [torch.zeros(rows, hq, dh, dtype=torch.bfloat16, device=device) for _ in range(2)]
    paged_attention(q, None, None, dh ** -0.5, out=outs[0], **common)
    paged_attention(q, b[0], b[1], dh ** -0.5, out=outs[1], k_scale=b[2] if fp8 else None,
                    v_scale=b[3] if fp8 else None, store_slot_mapping=slots, new_k=k, new_v=v, **common)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens", [[1], [64, 65], [128, 129, 256, 257], [255, 1, 512, 513, 640, 2, 768, 769, 1025],
                                  [37 * i % 300 + 1 for i in range(70)]])
@pytest.mark.parametrize("views", ["v", "k", ""])
def test_decode_folds_at_the_edges_of_a_step(device, fp8, lens, views):
    # The workgroups that carry the write skip the waits of their first two
    # steps: rows of one, two, three and more steps, one token short of a step,
    # at it and past it.  As Qwen3 hands them over, K is contiguous and V a view
    # of the QKV projection ("v"); the other way round ("k") the strides differ
    # as well.  Output and pool bytes of the store kernel followed by the launch.
    g = torch.Generator().manual_seed(len(lens))
    rows, hq, hkv, dh, bs = len(lens), 32, 8, 128, 256
    per = [(n + bs - 1) // bs for n in lens]
    nblk = sum(per) + 1
    perm = torch.randperm(nblk, generator=g).tolist()
    tables, at = [], 0
    for n in per:
        tables.append(perm[at:at + n] + [-1] * (max(per) - n))
        at += n
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    slots = i32([t[(n - 1) // bs] * bs + (n - 1) % bs for t, n in zip(tables, lens)])
    padded, dl = i32(tables), i32(lens)
    qkv = torch.randn(rows, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, k, v = (t.view(rows, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q, k, v = q.contiguous(), k if views == "k" else k.contiguous(), v if views == "v" else v.contiguous()
    reserve_workspace(device, rows, max(per) * bs, hq, hkv, dh)
    base = torch.randn(2, nblk * bs, hkv, dh, generator=g).to(torch.bfloat16).to(device)
    ctx = SimpleNamespace(mixed=MixedAttentionContext(rows, 0, dl, padded, None, None, None, 0, 0), slot_mapping=slots)
    outs, pools = [], []
    for store in (_two_launch_store, store_kvcache):
        if fp8:
            pool = [torch.empty(nblk, bs, hkv, dh, dtype=torch.uint8, device=device) for _ in range(2)]
            pool += [torch.empty(nblk, bs, hkv, device=device) for _ in range(2)]
            every = torch.arange(nblk * bs, dtype=torch.int32, device=device)
            store_kvcache(base[0], base[1], pool[0], pool[1], every, *pool[2:])
        else:
            pool = [base[i].clone().view(nblk, bs, hkv, dh) for i in range(2)]
        outs.append(forward_mixed(q, k, v, pool[0], pool[1], ctx, dh ** -0.5, store, *pool[2:]))
        pools.append(pool)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    for a, b in zip(*pools):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("case", ["tail queries", "more new rows than decode rows", "merged heads"])
def test_v0_steps_that_no_launch_carries(device, fp8, case):
    # V0 steps with views of the QKV projection that keep the store kernel's own
    # launch: the queries of a cold prompt's last tokens beside the keys of all
    # of it, decode steps with more new rows than query rows, and a cold step on
    # a pool view of merged heads.  Output and pool bytes of the store kernel
    # followed by the attention launch.
    g = torch.Generator().manual_seed(17)
    hq, hkv, dh, bs, nblk, n = 32, 8, 128, 256, 3, 100
    qkv = torch.randn(n, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, k, v = (t.view(n, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q = q.contiguous()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    slots = torch.randperm(nblk * bs, generator=g)[:n].to(torch.int32).to(device)
    decode = case.startswith("more")
    rows = 100 if case.startswith("merged") else 20
    q = q[-rows:]
    lens, tables = i32([5 + i for i in range(rows)]), i32([[i % nblk] for i in range(rows)])
    cu_q, cu_k = i32([0, rows]), i32([0, n])
    outs, pools = [], []
    for fold in (False, True):
        if fp8:
            pool = [torch.full((nblk, bs, hkv, dh), 7, dtype=torch.uint8, device=device) for _ in range(2)]
            pool += [torch.full((nblk, bs, hkv), 0.5, device=device) for _ in range(2)]
        else:
            pool = [torch.full((nblk, bs, hkv, dh), x, dtype=torch.bfloat16, device=device) for x in (3.0, -3.0)]
        if not fold:
            store_kvcache(k, v, pool[0], pool[1], slots, *pool[2:])
            where = (dict(num_decode=rows, decode_lens=lens, decode_tables=tables, k_scale=pool[2] if fp8 else None,
                          v_scale=pool[3] if fp8 else None) if decode else
                     dict(num_prefill=1, prefill_cu_q=cu_q, prefill_cu_k=cu_k, max_q=rows, max_k=n, k=k, v=v))
            outs.append(paged_attention(q, pool[0] if decode else None, pool[1] if decode else None, dh ** -0.5,
                                        num_kv_heads=hkv, **where))
        else:
            attn = Attention(hq, dh, dh ** -0.5, hkv)
            merged = case.startswith("merged")
            attn.k_cache, attn.v_cache = (p.view(nblk, bs, -1) if merged else p for p in pool[:2])
            if fp8:
                attn.k_scale, attn.v_scale = pool[2:]
            if decode:
                set_context(False, slot_mapping=slots, context_lens=lens, block_tables=tables)
            else:
                set_context(True, cu_q, cu_k, rows, n, slots)
            outs.append(attn(q, k, v).view(rows, hq, dh))
            reset_context()
        pools.append(pool)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    for a, b in zip(*pools):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _cold_launch_against_store(device, fp8, cu_q, cu_k, hq, hkv, seed, views="v"):
    """A cold prefill launch with the KV write (keys from the contiguous rows
    k/v, which may be longer than the new rows) against the store kernel and
    the same launch without it."""
    g = torch.Generator().manual_seed(seed)
    dh, bs, n, keys = 128, 256, cu_q[-1], cu_k[-1]
    nblk = (n + bs - 1) // bs + 2
    slots = torch.randperm(nblk * bs, generator=g)[:n].to(torch.int32).to(device)
    qkv = torch.randn(n, (hq + 2 * hkv) * dh, generator=g).to(torch.bfloat16).to(device)
    q, nk, nv = (t.view(n, -1, dh) for t in qkv.split([hq * dh, hkv * dh, hkv * dh], -1))
    q, nk, nv = q.contiguous(), nk if views == "k" else nk.contiguous(), nv if views == "v" else nv.contiguous()
    k, v = nk, nv
    if keys != n:
        k, v = (torch.randn(keys, hkv, dh, generator=g).to(torch.bfloat16).to(device) for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    lq = [b - a for a, b in zip(cu_q, cu_q[1:])]
    lk = [b - a for a, b in zip(cu_k, cu_k[1:])]
    common = dict(num_kv_heads=hkv, num_prefill=len(lq), prefill_cu_q=i32(cu_q), prefill_cu_k=i32(cu_k), max_q=max(lq),
                  max_k=max(lk), k=k, v=v)
    reserve_workspace(device, 0, 0, hq, hkv, dh)
    outs, pools = [], []
    for fold in (False, True):
        if fp8:
            pool = [torch.full((nblk, bs, hkv, dh), 7, dtype=torch.uint8, device=device) for _ in range(2)]
            pool += [torch.full((nblk, bs, hkv), 9.0, device=device) for _ in range(2)]
        else:
            pool = [torch.full((nblk, bs, hkv, dh), x, dtype=torch.bfloat16, device=device) for x in (3.0, -3.0)]
        if fold:
            outs.append(paged_attention(q, pool[0], pool[1], dh ** -0.5, k_scale=pool[2] if fp8 else None,
                                        v_scale=pool[3] if fp8 else None, store_slot_mapping=slots, new_k=nk, new_v=nv,
                                        phases=_lib.PHASE_ALL | _lib.NEW_ROWS_STRIDED, **common))
        else:
            store_kvcache(nk, nv, pool[0], pool[1], slots, *pool[2:])
            outs.append(paged_attention(q, None, None, dh ** -0.5, **common))
        pools.append(pool)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    for a, b in zip(*pools):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    return q, k, v, outs[1], lq, lk


def _cu(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


def _plain_prefill(q, k, v, lq, lk):
    out, a, b = [], 0, 0
    for m, n in zip(lq, lk):
        s = torch.einsum("qhd,khd->hqk", q[a:a + m].float().cpu(),
                         k[b:b + n].float().cpu().repeat_interleave(q.shape[1] // k.shape[1], 1)) * q.shape[2] ** -0.5
        s.masked_fill_(torch.arange(n) > torch.arange(m)[:, None] + n - m, float("-inf"))
        out.append(torch.einsum("hqk,khd->qhd", s.softmax(-1),
                                v[b:b + n].float().cpu().repeat_interleave(q.shape[1] // v.shape[1], 1)))
        a, b = a + m, b + n
    return torch.cat(out)


# The item orders of a cold launch: ranked units up to 128 rows, 1,024 units and
# 16,384 units x rows, row order past each of these, and a row split in two key
# ranges (more keys than queries, 32-position blocks whose second part stores
# nothing).  Empty rows and ties between equal rows among them.
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("name,lens,hist,hkv", [
    ("128 rows", [(5 * i) % 33 for i in range(128)], 0, 4),
    ("129 rows", [(5 * i) % 33 for i in range(129)], 0, 4),
    ("140 equal and empty rows", [0, 33] * 70, 0, 4),
    ("128 rows, more than 16,384 units x rows", [(7 * i) % 41 for i in range(128)], 0, 4),
    ("1,021 units of 16 positions", [4096] + [816] * 15, 0, 1),
    ("1,036 units of 16 positions", [4096] + [832] * 15, 0, 1),
    ("split row", [96, 40], 1500, 4),
    ("split row of 33 queries", [33, 1, 64], 2100, 4),
])
def test_cold_write_in_every_item_order(device, fp8, name, lens, hist, hkv):
    # Qwen3's pair: K contiguous, V a view of the projection.
    cu_q = _cu(lens)
    cu_k = _cu([n + (hist if i == 0 else 0) for i, n in enumerate(lens)])
    q, k, v, out, lq, lk = _cold_launch_against_store(device, fp8, cu_q, cu_k, 4 * hkv, hkv, 5)
    if hist:
        assert workspace_events(device)["split_prefill_merges"] > 0
    want = _plain_prefill(q, k, v, lq, lk)
    assert (out.float().cpu() - want).abs().max() <= 2e-2


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("views", ["v", "k", ""])
@pytest.mark.parametrize("lens,hq,hkv", [([1], 32, 8), ([31, 33, 1, 64, 100], 8, 8), ([700, 257], 64, 8)])
def test_cold_write_with_different_k_and_v_strides(device, fp8, views, lens, hq, hkv):
    _cold_launch_against_store(device, fp8, _cu(lens), _cu(lens), hq, hkv, 9, views)
