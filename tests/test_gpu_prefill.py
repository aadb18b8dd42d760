"""GPU parity of prefill-with-parent-context (packed ragged chunks, bottom-right
causal over scattered parent slots) against the CPU oracle."""
import ctypes
import dataclasses

import pytest
import torch

from oracle.ref_ops import ref_cos_sin_cache, ref_prefill_with_parent, ref_rope_neox

pytestmark = pytest.mark.gpu

TOL = {torch.float16: dict(atol=2e-3, rtol=1e-2), torch.bfloat16: dict(atol=1e-2, rtol=2e-2)}


def prefill_plan(q_lens, ctx_lens, H, D, dtype, workspace_bytes=None):
    """(queries per workgroup, parts per context) of a call of these sizes; the workspace it asks for by default"""
    from parrotserve_amd import _lib

    lib, tile, parts = _lib.load(), ctypes.c_int32(), ctypes.c_int32()
    code = _lib.PH_F16 if dtype == torch.float16 else _lib.PH_BF16
    if workspace_bytes is None:
        workspace_bytes = lib.ph_prefill_workspace_bytes(sum(q_lens), H, D, code, max(ctx_lens))
    assert lib.ph_prefill_plan(sum(q_lens), len(q_lens), H, D, code, max(ctx_lens), sum(ctx_lens), workspace_bytes,
                               ctypes.byref(tile), ctypes.byref(parts)) == _lib.PH_OK
    return tile.value, parts.value


def run_prefill_case(case, dev, fused_path=True):
    """RoPE on new q/k -> append -> attention, on the GPU; returns (out, oracle_out)."""
    from parrotserve_amd import kernels, synth

    T, H, D = case.q.shape
    cache = ref_cos_sin_cache(int(case.positions.max()) + 1, D, case.theta, case.dtype)
    # oracle: rotate with the reference kernel's arithmetic, then attention over parents || own
    rq, rk = ref_rope_neox(case.positions, case.q.reshape(T, -1), case.k_new.reshape(T, -1), cache, D,
                           elem_rounding=True)
    rq, rk = rq.view(T, H, D), rk.view(T, H, D)
    k_all = torch.cat([case.k_rows, rk])
    v_all = torch.cat([case.v_rows, case.v_new])
    ctx = [torch.cat([p, n]) for p, n in zip(case.parent_lists, case.new_lists)]
    ref = ref_prefill_with_parent(rq, k_all, v_all, case.q_lens, ctx)

    kc, vc = synth.pool_to_device(case.k_rows, case.v_rows, case.used_slots, case.pool_slots, dev)
    q, k, v = case.q.to(dev), case.k_new.to(dev), case.v_new.to(dev)
    kernels.vllm_rotary_emb(case.positions.to(dev), q.view(T, -1), k.view(T, -1), cache.to(dev), D)
    new_slots = torch.cat([case.used_slots[n] for n in case.new_lists]).to(torch.int32).to(dev)
    kernels.vllm_reshape_and_cache(k, v, kc, vc, new_slots)
    tables = kernels.PrefillTables.build(case.q_lens, [case.used_slots[c].tolist() for c in ctx], dev)
    out = kernels.prefill_attention(q, kc, vc, tables)
    torch.cuda.synchronize()
    return out.cpu(), ref


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q_lens,parent,H", [([5, 1, 70, 33], 100, 4), ([64, 128, 17], 0, 8), ([200], 333, 2),
                                             ([1, 1, 1], 50, 40)])
def test_prefill_small(dev, dtype, q_lens, parent, H):
    from parrotserve_amd import synth

    case = synth.make_prefill_case("p", 21 + parent, dtype, q_lens, parent, H, 128, 1 << 13)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[dtype])


def test_config4_scaled(dev):
    """Config 4's recipe (bf16, 40x128, ragged chunks over 2048-token parents, RoPE theta 1e4, seed 3)
    on 4 of the 16 chunks with chunk lengths U[64,256]."""
    from parrotserve_amd import synth

    case = synth.config4(chunks=4, lo=64, hi=256, parent=2048, pool_slots=1 << 15)
    assert case.dtype == torch.bfloat16 and case.q.shape[1:] == (40, 128)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_prefill_tile_boundaries(dev, dtype):
    """Chunk lengths around the 64-query tile and 32-token KV tile sizes, with and without parents."""
    from parrotserve_amd import synth

    for parent, q_lens in ((0, [63, 64, 65, 1, 129]), (31, [64, 33]), (96, [2, 127, 128]), (1, [300])):
        case = synth.make_prefill_case("b", 77 + parent, dtype, q_lens, parent, 3, 128, 1 << 12)
        out, ref = run_prefill_case(case, dev)
        torch.testing.assert_close(out.float(), ref.float(), **TOL[dtype])


def test_config4_full_size_property(dev):
    """Config 4 at full size (16 chunks U[64,1024] over 2048-token parents, 40x128, bf16, seed 3): a query
    row of the prefill equals a decode request over exactly the keys it may see (q_len == 1 reduction),
    checked on the GPU for 512 sampled rows, plus oracle parity on the first and on the longest chunk."""
    from parrotserve_amd import kernels, synth

    case = synth.config4()
    T, H, D = case.q.shape
    assert len(case.q_lens) == 16 and H == 40 and case.dtype == torch.bfloat16
    kc, vc = synth.pool_to_device(case.k_rows, case.v_rows, case.used_slots, case.pool_slots, dev)
    cache = ref_cos_sin_cache(int(case.positions.max()) + 1, D, case.theta, case.dtype)
    q, k, v = case.q.to(dev), case.k_new.to(dev), case.v_new.to(dev)
    kernels.vllm_rotary_emb(case.positions.to(dev), q.view(T, -1), k.view(T, -1), cache.to(dev), D)
    new_slots = torch.cat([case.used_slots[n] for n in case.new_lists]).to(torch.int32).to(dev)
    kernels.vllm_reshape_and_cache(k, v, kc, vc, new_slots)
    ctx = [case.used_slots[torch.cat([p, n])].tolist() for p, n in zip(case.parent_lists, case.new_lists)]
    tables = kernels.PrefillTables.build(case.q_lens, ctx, dev)
    out = kernels.prefill_attention(q, kc, vc, tables)

    g = torch.Generator().manual_seed(0)
    rows = torch.randperm(T, generator=g)[:512].sort().values.tolist()
    starts = [0]
    for n in case.q_lens:
        starts.append(starts[-1] + n)
    lists = []
    for r in rows:
        c = max(i for i in range(16) if starts[i] <= r)
        n = case.q_lens[c]
        vis = len(ctx[c]) - n + (r - starts[c]) + 1
        lists.append(ctx[c][:vis])
    dt = kernels.DecodeTables.build([], [], lists, dev)
    ridx = torch.tensor(rows, device=dev)
    dec = kernels.decode_attention(q[ridx].contiguous(), kc, vc, dt)
    torch.testing.assert_close(out[ridx].float(), dec.float(), **TOL[torch.bfloat16])

    # oracle parity on the first chunk and on the longest one (the chunk that runs every tile form; its queries
    # and keys only)
    longest = max(range(16), key=case.q_lens.__getitem__)
    for c in sorted({0, longest}):
        a, n = starts[c], case.q_lens[c]
        rq, rk = ref_rope_neox(case.positions[a:a + n], case.q[a:a + n].reshape(n, -1),
                               case.k_new[a:a + n].reshape(n, -1), cache, D, elem_rounding=True)
        k_all = torch.cat([case.k_rows[case.parent_lists[c]], rk.view(n, H, D)])
        v_all = torch.cat([case.v_rows[case.parent_lists[c]], case.v_new[a:a + n]])
        ref_c = ref_prefill_with_parent(rq.view(n, H, D), k_all, v_all, [n], [torch.arange(k_all.shape[0])])
        torch.testing.assert_close(out[a:a + n].cpu().float(), ref_c.float(), **TOL[torch.bfloat16])


@pytest.mark.parametrize("q_lens,parent", [([260], 9000),          # average 260 -> 256-query tiles
                                           ([40, 300], 5000),      # average 170 -> 128-query tiles
                                           ([30, 64, 20], 4200)])  # average 38 -> 64-query tiles
def test_prefill_long_parents_all_tile_sizes(dev, q_lens, parent):
    """Parents longer than the 4096-token slot window the kernel keeps on chip (the window slides while the
    staging ring runs ahead), for each of the three query-tile sizes the launcher picks by average chunk length."""
    from parrotserve_amd import synth

    case = synth.make_prefill_case("w", 5 + parent, torch.float16, q_lens, parent, 2, 128, 1 << 15)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.float16])


@pytest.mark.parametrize("n,tile", [(61, 64), (125, 128), (255, 256)])
@pytest.mark.parametrize("ctx", [512, 513, 4032, 4095, 4097])
def test_prefill_window_filled_in_part(dev, n, tile, ctx):
    """The slot window is filled 512 entries at a time as far as the tile's steps reach (64 or 128 tokens a step): contexts
    that end on, before and behind an edge of either, and at the window's own end, with query rows missing from the last
    block (its rows are staged as whole 32-row blocks).  More than four rounds of workgroups, so that none is
    cut into parts."""
    from parrotserve_amd import synth

    q_lens, H = [n] * 32, 40
    assert prefill_plan(q_lens, [ctx] * 32, H, 128, torch.float16) == (tile, 1)
    case = synth.make_prefill_case("win", ctx + n, torch.float16, q_lens[:2], ctx - n, 2, 128, 1 << 14)
    k_all, v_all = torch.cat([case.k_rows, case.k_new]), torch.cat([case.v_rows, case.v_new])
    lists = [torch.cat([p, m]) for p, m in zip(case.parent_lists, case.new_lists)]
    from parrotserve_amd import kernels

    kc, vc = synth.pool_to_device(k_all, v_all, case.used_slots, case.pool_slots, dev)
    # the two chunks sixteen times each, their two heads twenty times
    tables = kernels.PrefillTables.build(q_lens, [case.used_slots[lists[i % 2]].tolist() for i in range(32)], dev)
    q = case.q.view(2, n, 2, 128).repeat(16, 1, 20, 1).view(32 * n, H, 128)
    wide = lambda t: t.repeat(1, 20, 1).contiguous()  # noqa: E731
    out = kernels.prefill_attention(q.to(dev), wide(kc), wide(vc), tables)
    torch.cuda.synchronize()
    ref = ref_prefill_with_parent(case.q, k_all, v_all, q_lens[:2], lists)
    got = out.cpu().view(16, 2 * n, 20, 2, 128)
    assert (got == got[:1, :, :1]).all()
    torch.testing.assert_close(got[0, :, 0].float(), ref.float(), **TOL[torch.float16])


@pytest.mark.parametrize("q_lens", [[1], [3], [4], [5], [33], [36, 1, 4], [65, 96, 97], [100, 128]])
def test_prefill_query_rows_up_to_the_last_live_one(dev, q_lens):
    """Short Fills on the 64- and 128-query tiles: only the loads of query rows that hold a live one are issued."""
    from parrotserve_amd import synth

    case = synth.make_prefill_case("rows", 40 + sum(q_lens), torch.bfloat16, q_lens, 100, 4, 128, 1 << 12)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.bfloat16])


def test_prefill_heads_not_multiple_of_eight_and_tail_tiles(dev):
    """Head counts that leave part of the padded head axis empty, chunks that end inside every tile size."""
    from parrotserve_amd import synth

    for H, q_lens, parent in ((5, [257, 511, 193], 70), (9, [129, 100, 95], 33), (3, [65, 31, 96, 1], 200)):
        case = synth.make_prefill_case("h", 900 + H, torch.bfloat16, q_lens, parent, H, 128, 1 << 13)
        out, ref = run_prefill_case(case, dev)
        torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.bfloat16])


@pytest.mark.parametrize("D,H", [(64, 6), (64, 5), (256, 2), (80, 5), (96, 3), (112, 2)])
def test_prefill_other_head_sizes(dev, D, H):
    """The other head sizes the reference dispatches: 80, 96 and 112 run on the matrix-core kernel as short heads
    on its 128-wide tile, 64 on head pairs (even head counts); 256 and 64 with an odd head count run every query
    row through the per-request kernel over its visible slots.  Same results."""
    from parrotserve_amd import synth

    case = synth.make_prefill_case("hd", 300 + D, torch.float16, [33, 5, 70], 41, H, D, 1 << 12)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.float16])


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("seed", range(8))
def test_randomized_prefill_shapes(dev, seed, D):
    """Seeded random chunk sets: 1-6 chunks of 1-400 new tokens over parents of 0-700 tokens, odd head counts,
    both element types (covers every query-tile size and partial tiles on both axes).  64-wide heads run as
    halves of head pairs on the same matrix-core kernel when the head count is even, through the per-request
    kernel when it is odd."""
    from parrotserve_amd import synth

    g = torch.Generator().manual_seed(2000 + seed)
    ri = lambda lo, hi: int(torch.randint(lo, hi + 1, (1,), generator=g))  # noqa: E731
    dtype = torch.float16 if seed % 2 else torch.bfloat16
    chunks = ri(1, 6)
    hi = [30, 120, 400][seed % 3]
    q_lens = [ri(1, hi) for _ in range(chunks)]
    case = synth.make_prefill_case("rnd", 2000 + seed, dtype, q_lens, ri(0, 700), ri(1, 6), D, 1 << 13)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [80, 96, 112])
def test_prefill_short_heads_on_the_wide_tile(dev, D, dtype):
    """Head sizes 80 / 96 / 112 on the 128-wide matrix-core tile, every query-tile form (chunks averaging 270, 130
    and 40 tokens), partial tiles on both axes, parents longer than a tile; the last head of the last slot row
    included (its padding lanes must stay inside the pool)."""
    from parrotserve_amd import synth

    for q_lens, parent, H in (([300, 240], 600, 3), ([129, 131], 257, 5), ([33, 64, 20, 41], 90, 2)):
        case = synth.make_prefill_case("sh", 500 + D + H, dtype, q_lens, parent, H, D, 1 << 11)
        out, ref = run_prefill_case(case, dev)
        torch.testing.assert_close(out.float(), ref.float(), **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q_lens,parent,H,D,plan", [
    ([61], 1987, 4, 128, (64, 16)),      # many parts of one 64-query tile
    ([1], 1100, 3, 128, (64, 9)),        # nine steps: the last of several parts is empty
    ([16, 5], 900, 5, 128, (64, 8)),     # two chunks of different visible lengths
    ([33], 1500, 2, 96, (64, 12)),       # short heads
    ([40, 7], 800, 4, 64, (64, 7)),      # head pairs
    ([700], 5000, 2, 64, (256, 9)),      # head pairs on more than one tile, parts beyond the slot window's length
    ([300], 6100, 9, 128, (64, 3)),      # several tiles, the last one partly filled
    ([200], 3000, 40, 128, (128, 3)),    # the 128-query tile
    ([1000], 5000, 8, 128, (256, 8)),    # the 256-query tile on whole heads
])
def test_prefill_long_contexts_in_parts(dev, q_lens, parent, H, D, plan, dtype):
    """Few queries over long contexts: every tile's visible tokens are cut into parts folded afterwards.  A call with
    only the smallest workspace takes the same chunks in one part per tile."""
    from parrotserve_amd import _lib, kernels, synth

    case = synth.make_prefill_case("parts", 70 + parent + H, dtype, q_lens, parent, H, D, 1 << 13)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[dtype])

    lib, T = _lib.load(), sum(q_lens)
    shape = (T, H, D, _lib.PH_F16 if dtype == torch.float16 else _lib.PH_BF16, parent + max(q_lens))
    least = lib.ph_prefill_workspace_min_bytes(*shape)
    assert lib.ph_prefill_workspace_bytes(*shape) > least
    ctx_lens = [parent + n for n in q_lens]
    assert prefill_plan(q_lens, ctx_lens, H, D, dtype) == plan
    assert prefill_plan(q_lens, ctx_lens, H, D, dtype, least)[1] == 1
    kc, vc = synth.pool_to_device(torch.cat([case.k_rows, case.k_new]), torch.cat([case.v_rows, case.v_new]),
                                  case.used_slots, case.pool_slots, dev)
    q = case.q.to(dev)
    ctx = [case.used_slots[torch.cat([p, n])].tolist() for p, n in zip(case.parent_lists, case.new_lists)]
    tabs = kernels.PrefillTables.build(q_lens, ctx, dev)
    whole, small = kernels.prefill_attention(q, kc, vc, tabs), torch.empty_like(q)
    ws = torch.empty(least, dtype=torch.uint8, device=dev)
    args = (q.data_ptr(), kc.data_ptr(), vc.data_ptr(), T, len(q_lens), H, D, shape[3], H * D, H * D, H * D, D ** -0.5,
            tabs.q_cu.data_ptr(), tabs.kv_cu.data_ptr(), tabs.ctx_slots.data_ptr(), tabs.ctx_slots.numel(), shape[4])
    assert lib.ph_prefill_attention(small.data_ptr(), *args, ws.data_ptr(), least, kernels._stream()) == 0
    torch.testing.assert_close(whole.float(), small.float(), **TOL[dtype])
    assert lib.ph_prefill_attention(small.data_ptr(), *args, ws.data_ptr(), least - 1, kernels._stream()) == \
        _lib.PH_ERR_WORKSPACE


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bad", ["key nan", "key inf", "query nan", "query inf", "value nan"])
@pytest.mark.parametrize("T,parent,H,D,tile", [
    (61, 1987, 4, 128, 64),    # parts of one 64-query tile
    (300, 3000, 4, 128, 64),   # parts of several tiles
    (200, 3000, 40, 128, 128),
    (1000, 5000, 8, 128, 256),
    (33, 1500, 4, 96, 64),     # short heads
])
def test_prefill_in_parts_keeps_non_finite_values(dev, T, parent, H, D, tile, bad, dtype):
    """A non-finite key, value or query in a prefill in parts: NaN wherever the same attention in plain fp32 has it,
    the other heads and queries as without it."""
    from parrotserve_amd import kernels

    head, n = 1, parent + T
    used, parts = prefill_plan([T], [n], H, D, dtype)
    assert used == tile and parts > 1
    g = torch.Generator().manual_seed(77 + T)
    q, k, v = (torch.randn(m, H, D, generator=g).to(dtype) for m in (T, n, n))
    what, value = bad.split()
    {"key": k, "value": v, "query": q}[what][T // 2 if what == "query" else parent // 2, head, 5] = float(value)
    qf, kf, vf = (x.float().transpose(0, 1).contiguous() for x in (q, k, v))
    s = (qf @ kf.transpose(1, 2).contiguous()) * D ** -0.5
    s.masked_fill_(torch.arange(n)[None, None, :] > parent + torch.arange(T)[None, :, None], -float("inf"))
    ref = (torch.softmax(s, dim=-1) @ vf).transpose(0, 1)
    assert ref.isnan().any() and not ref[:, 0].isnan().any()

    tables = kernels.PrefillTables.build([T], [list(range(n))], dev)
    out = kernels.prefill_attention(q.to(dev), k.to(dev), v.to(dev), tables).cpu().float()
    assert out[ref.isnan()].isnan().all()
    others = torch.arange(H) != head
    torch.testing.assert_close(out[:, others], ref[:, others], **TOL[dtype])
    if what == "query":
        queries = torch.arange(T) != T // 2
        torch.testing.assert_close(out[queries], ref[queries], **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q_lens,ctx_lens,D", [
    ([16] * 4, [8192, 64, 64, 64], 128),               # eight parts made for one long context: the others fill one
    ([64, 3, 64, 1], [512, 4100, 64, 1], 128),         # the long one in the middle, a chunk of one token
    ([61] * 6, [100, 200, 400, 800, 1600, 3200], 96),
    ([256, 40], [6256, 40], 64),
])
def test_prefill_contexts_of_different_lengths(dev, q_lens, ctx_lens, D, dtype):
    """Chunks over contexts of very different lengths in one launch against plain fp32 attention."""
    from parrotserve_amd import kernels

    H = 8
    assert prefill_plan(q_lens, ctx_lens, H, D, dtype)[1] > 1
    g = torch.Generator().manual_seed(5 + sum(ctx_lens))
    n = sum(ctx_lens)
    q, k, v = (torch.randn(m, H, D, generator=g).to(dtype) for m in (sum(q_lens), n, n))
    slots, ref, lists, at = torch.randperm(n, generator=g), [], [], 0
    for new, length in zip(q_lens, ctx_lens):
        lists.append(slots[sum(ctx_lens[:len(lists)]):][:length])
        qf, kf, vf = (x.float().transpose(0, 1).contiguous() for x in (q[at:at + new], k[lists[-1]], v[lists[-1]]))
        s = (qf @ kf.transpose(1, 2).contiguous()) * D ** -0.5
        s.masked_fill_(torch.arange(length)[None, None, :] > length - new + torch.arange(new)[None, :, None], -float("inf"))
        ref.append((torch.softmax(s, dim=-1) @ vf).transpose(0, 1))
        at += new
    tables = kernels.PrefillTables.build(q_lens, [x.tolist() for x in lists], dev)
    out = kernels.prefill_attention(q.to(dev), k.to(dev), v.to(dev), tables)
    torch.testing.assert_close(out.cpu().float(), torch.cat(ref), **TOL[dtype])


@pytest.mark.parametrize("chunks", [64, 65, 130, 256, 257])
def test_prefill_chunk_counts_around_the_tile_search(dev, chunks):
    """Chunk counts at the edges of the in-kernel tile search (64 chunks a round, a pre-pass beyond 256)."""
    from parrotserve_amd import synth

    q_lens = [1 + (7 * i) % 5 + (66 if i % 50 == 3 else 0) for i in range(chunks)]
    case = synth.make_prefill_case("many", 40 + chunks, torch.bfloat16, q_lens, 9, 2, 128, 1 << 13)
    out, ref = run_prefill_case(case, dev)
    torch.testing.assert_close(out.float(), ref.float(), **TOL[torch.bfloat16])


def test_more_tile_rows_than_the_grid_holds(dev):
    """70,000 one-token chunks without parents: more tile rows than a grid's y extent (65,535), so workgroups stride
    over them.  A query that sees exactly one key returns that key's value row."""
    from parrotserve_amd import kernels

    C, H, D = 70000, 2, 128
    g = torch.Generator(device=dev).manual_seed(12)
    k = torch.randn((C, H, D), generator=g, device=dev, dtype=torch.bfloat16)
    v = torch.randn((C, H, D), generator=g, device=dev, dtype=torch.bfloat16)
    q = torch.randn((C, H, D), generator=g, device=dev, dtype=torch.bfloat16)
    perm = torch.randperm(C, generator=torch.Generator().manual_seed(12))
    tabs = kernels.PrefillTables.build([1] * C, [[int(s)] for s in perm.tolist()], dev)
    out = kernels.prefill_attention(q, k, v, tabs)
    torch.cuda.synchronize()
    assert torch.equal(out, v[perm.to(dev)])


@pytest.mark.parametrize("warm", ["the call", "a larger call", "a call of one part"])
def test_prefill_in_parts_replays_from_a_captured_graph(dev, warm):
    """A prefill that is cut into parts, recorded after an eager run of itself, of a longer call that takes no parts, or
    of a call whose scratch holds none (the recorded call then stays in one part): every replay, with eager work between
    them, gives what the eager call with the same workspace gives."""
    from parrotserve_amd import kernels

    H, D, T, n = 32, 128, 61, 2048
    g = torch.Generator(device=dev).manual_seed(41)
    rand = lambda rows: torch.randn(rows, H, D, generator=g, device=dev, dtype=torch.bfloat16)
    k, v, q = rand(4096), rand(4096), rand(T)
    build = lambda new, length: kernels.PrefillTables.build([new], [list(range(length))], dev)
    tables, out = build(T, n), torch.empty_like(q)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        if warm == "the call":
            kernels.prefill_attention(q, k, v, tables)
        elif warm == "a larger call":
            kernels.prefill_attention(rand(4096), k, v, build(4096, 4096))
        else:
            kernels.prefill_attention(rand(1), k, v, build(1, 1))
        room = kernels._workspaces[(dev.index or 0, side.cuda_stream)].numel()
    torch.cuda.synchronize()
    parts = prefill_plan([T], [n], H, D, torch.bfloat16, room)[1]
    assert parts > 1 or warm == "a call of one part"  # (a stream used before may hold more)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        kernels.prefill_attention(q, k, v, tables, out=out)
    for rep in range(3):
        q.copy_(rand(T))
        out.zero_()
        eager = kernels.prefill_attention(q, k, v, tables)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        if parts > 1:
            assert torch.equal(out, eager), f"replay {rep} differs from the eager result"
        torch.testing.assert_close(out.float(), eager.float(), **TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rises", [
    {0: 0.0},                                                # one level throughout
    {0: 0.0, 64: 13.0, 128: 26.0, 192: 39.0},                # past the limit at every step, in its first 32 tokens
    {0: 0.0, 96: 13.0, 160: 26.0, 288: 39.0},                # in its second 32 tokens
    {0: 0.0, 64: 11.0, 96: 13.5, 128: 9.0, 353: 25.0},       # within the limit, then past it; a single later token
    {0: -200.0, 65: 200.0, 66: 0.0},                         # beyond what an fp32 exponential holds
    {0: 40.0, 32: 0.0, 320: -90.0},                          # falling: the reference stays
])
def test_prefill_scores_that_outgrow_the_exponent_reference(dev, rises, dtype):
    """256-query tiles over scores whose level (as a power of two) changes at the given tokens.  The oracle scales and
    rounds the queries as the kernel does, so what is left is the rounding of the 16-bit probabilities and outputs."""
    from parrotserve_amd import kernels

    T, parent, H, D = 300, 2000, 40, 128  # a query sees 2150 tokens on average
    n = parent + T
    assert prefill_plan([T] * 12, [n] * 12, H, D, dtype) == (256, 1)
    g = torch.Generator().manual_seed(5)
    sign = torch.where(torch.rand(D, generator=g) < 0.5, -1.0, 1.0)
    q = (8.0 * sign).expand(T, H, D) + 0.05 * torch.randn(T, H, D, generator=g)
    level = torch.zeros(n)
    for at, value in sorted(rises.items()):
        level[at:] = value
    per_unit = 8.0 * D * D ** -0.5 * 1.4426950408889634      # exponent per unit of a key along `sign`
    k = (level / per_unit)[:, None, None] * sign + 0.1 * torch.randn(n, H, D, generator=g)
    q, k, v = q.to(dtype), k.to(dtype), torch.randn(n, H, D, generator=g).to(dtype)
    scaled = (q.float() * (D ** -0.5 * 1.4426950408889634)).to(dtype).double().transpose(0, 1)
    s = scaled @ k.double().permute(1, 2, 0).contiguous() * 0.6931471805599453
    s.masked_fill_(torch.arange(n)[None, None, :] > parent + torch.arange(T)[None, :, None], -float("inf"))
    ref = (torch.softmax(s, dim=-1) @ v.double().transpose(0, 1)).transpose(0, 1)
    slots = list(range(n))
    tables = kernels.PrefillTables.build([T] * 12, [slots] * 12, dev)
    out = kernels.prefill_attention(q.repeat(12, 1, 1).to(dev), k.to(dev), v.to(dev), tables).cpu().double()
    for c in range(12):
        torch.testing.assert_close(out[c * T:(c + 1) * T], ref, **TOL[dtype])


@pytest.mark.parametrize("D,dtype", [(80, torch.float16), (96, torch.bfloat16), (112, torch.float16), (128, torch.float16),
                                     (128, torch.bfloat16)])
@pytest.mark.parametrize("rises", [
    {0: 0.0, 1920: 13.0, 1952: 26.0, 1984: 39.0, 2016: 52.0},  # in the last whole steps of the waves whose diagonal follows
    {0: 0.0, 1300: 12.5, 1345: 25.0, 1440: 38.0, 1499: 60.0},  # as far as the last token, across the tiles' forms
    {0: 0.0, 1408: 50.0, 1409: 0.0, 2005: 30.0},               # one token far above all others, one inside the diagonal
])
def test_prefill_outgrown_references_in_unequal_chunks_and_short_heads(dev, rises, D, dtype):
    """The same over chunks of different lengths and contexts, without a parent (tiles of both forms in one chunk), with a
    tile of a few queries, and with heads shorter than the tile's 128 dims."""
    from parrotserve_amd import kernels

    q_lens, parents, H, heads = [300, 1500, 40, 777], [2000, 0, 2000, 1300], 40, [0, 17, 39]
    ctx = [n + p for n, p in zip(q_lens, parents)]
    assert prefill_plan(q_lens, ctx, H, D, dtype) == (256, 1)
    g = torch.Generator().manual_seed(6)
    sign = torch.where(torch.rand(D, generator=g) < 0.5, -1.0, 1.0)
    q = ((8.0 * sign).expand(sum(q_lens), H, D) + 0.05 * torch.randn(sum(q_lens), H, D, generator=g)).to(dtype)
    level = torch.zeros(max(ctx))
    for at, value in sorted(rises.items()):
        level[at:] = value
    per_unit = 8.0 * D * D ** -0.5 * 1.4426950408889634
    k = torch.cat([(level[:n] / per_unit)[:, None, None] * sign for n in ctx]) + 0.1 * torch.randn(sum(ctx), H, D, generator=g)
    k, v = k.to(dtype), torch.randn(sum(ctx), H, D, generator=g).to(dtype)
    tables = kernels.PrefillTables.build(q_lens, [list(range(sum(ctx[:c]), sum(ctx[:c + 1]))) for c in range(4)], dev)
    out = kernels.prefill_attention(q.to(dev), k.to(dev), v.to(dev), tables).cpu()[:, heads].double()
    scaled = (q[:, heads].float() * (D ** -0.5 * 1.4426950408889634)).to(dtype).double().transpose(0, 1)
    for c, (n, p) in enumerate(zip(q_lens, parents)):
        rows, keys = slice(sum(q_lens[:c]), sum(q_lens[:c + 1])), slice(sum(ctx[:c]), sum(ctx[:c + 1]))
        s = scaled[:, rows] @ k[keys][:, heads].double().permute(1, 2, 0).contiguous() * 0.6931471805599453
        s.masked_fill_(torch.arange(n + p)[None, None, :] > p + torch.arange(n)[None, :, None], -float("inf"))
        ref = (torch.softmax(s, dim=-1) @ v[keys][:, heads].double().transpose(0, 1)).transpose(0, 1)
        torch.testing.assert_close(out[rows], ref, **TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bad", ["key nan", "key inf", "query nan", "query inf", "value nan"])
def test_prefill_whole_tiles_keep_non_finite_values(dev, bad, dtype):
    """The same in one part per tile of 256 queries: NaN where plain fp32 attention has it and there alone, in the head
    that holds it and in the others."""
    from parrotserve_amd import kernels

    T, parent, H, D, head = 300, 2000, 40, 128, 1
    n = parent + T
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(m, H, D, generator=g).to(dtype) for m in (T, n, n))
    what, value = bad.split()
    {"key": k, "value": v, "query": q}[what][T // 2 if what == "query" else 100, head, 5] = float(value)
    qf, kf, vf = (x.float().transpose(0, 1).contiguous() for x in (q, k, v))
    s = (qf @ kf.transpose(1, 2).contiguous()) * D ** -0.5
    s.masked_fill_(torch.arange(n)[None, None, :] > parent + torch.arange(T)[None, :, None], -float("inf"))
    ref = (torch.softmax(s, dim=-1) @ vf).transpose(0, 1)
    assert prefill_plan([T] * 12, [n] * 12, H, D, dtype) == (256, 1)
    tables = kernels.PrefillTables.build([T] * 12, [list(range(n))] * 12, dev)
    out = kernels.prefill_attention(q.repeat(12, 1, 1).to(dev), k.to(dev), v.to(dev), tables).cpu().float()[:T]
    assert ref.isnan().any() and torch.equal(out.isnan(), ref.isnan())
    torch.testing.assert_close(out, ref, equal_nan=True, **TOL[dtype])


def _random_prefill(dev, q_lens, parents, H=40, D=128):
    from parrotserve_amd import kernels

    g = torch.Generator().manual_seed(11)
    ctx = [n + p for n, p in zip(q_lens, parents)]
    q, k, v = (torch.randn(n, H, D, generator=g).half().to(dev) for n in (sum(q_lens), sum(ctx), sum(ctx)))
    slots = torch.randperm(sum(ctx), generator=g).tolist()
    lists = [slots[sum(ctx[:c]):sum(ctx[:c + 1])] for c in range(len(ctx))]
    return q, k, v, lists, kernels.PrefillTables.build(q_lens, lists, dev)


def test_a_longer_slot_list_does_not_change_the_kernel(dev):
    """The slot list may be longer than the contexts (a buffer kept for the largest call): to the bit the same result."""
    from parrotserve_amd import kernels

    assert prefill_plan([600] * 3, [640] * 3, 40, 128, torch.float16) == (256, 1)
    q, k, v, _, tables = _random_prefill(dev, [600] * 3, [40] * 3)
    out = kernels.prefill_attention(q, k, v, tables)
    room = torch.zeros(15000, dtype=torch.int32, device=dev)
    longer = dataclasses.replace(tables, ctx_slots=torch.cat([tables.ctx_slots, room]))
    assert torch.equal(kernels.prefill_attention(q, k, v, longer), out)


def test_a_chunk_takes_the_kernel_form_of_its_own_length(dev):
    """Chunks over long contexts beside more of them without any, and the other way round: to the bit what each gives in
    a call of its own kind (the form of the tile loop follows from the tile, not from the call's mean)."""
    from parrotserve_amd import kernels

    long, short = [(300, 2000)] * 12, [(300, 0)] * 24
    for chunks in (long, short, long + short):
        q_lens = [n for n, _ in chunks]
        assert prefill_plan(q_lens, [n + p for n, p in chunks], 40, 128, torch.float16) == (256, 1)
    q, k, v, lists, tables = _random_prefill(dev, [300] * 36, [2000] * 12 + [0] * 24)
    together = kernels.prefill_attention(q, k, v, tables)
    for first, last in ((0, 12), (12, 36)):
        part = kernels.PrefillTables.build([300] * (last - first), lists[first:last], dev)
        rows = slice(300 * first, 300 * last)
        assert torch.equal(kernels.prefill_attention(q[rows], k, v, part), together[rows])
