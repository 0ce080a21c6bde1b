"""Fused indexer + top-k (dsa_indexer_topk) on the GPU.

The fused call must select exactly what topk_transform selects over the
logits of indexer_logits on the same inputs (same logits bit for bit, so the
comparison is exact), for plain decode, MTP rows (next_n = 2), short rows and
both top-k sizes, and also when the page sample misleads the threshold and the
list select has to redo a row from its full logits."""
import numpy as np
import pytest
import torch

from nanoengine_amd import ops, synth

pytestmark = pytest.mark.gpu


def _inputs(lens, n, seed):
    inp = synth.make_indexer_inputs(lens, next_n=n, seed=seed, device="cuda")
    ctx = inp.context_lens.to(torch.int32)
    if n == 1:
        cl = ctx.view(-1, 1)
    else:  # causal lengths of the draft tokens: L - (n-1-j)
        offs = torch.arange(n - 1, -1, -1, dtype=torch.int32, device="cuda")
        cl = (ctx[:, None] - offs).clamp_min(1).contiguous()
    max_ctx = inp.block_tables.shape[1] * 64
    return inp, cl, max_ctx


def _unfused(inp, cl, max_ctx, k, n):
    B = cl.shape[0]
    logits = ops.indexer_logits(inp.q_fp8.view(B, n, 64, 128), inp.cache, inp.weights, cl, inp.block_tables,
                                max_ctx)
    pt = inp.block_tables.repeat_interleave(n, dim=0).contiguous()
    phys = torch.empty(B * n, k, dtype=torch.int32, device="cuda")
    logi = torch.empty_like(phys)
    ops.topk_transform(logits, cl.reshape(-1).contiguous(), pt, phys, 64, k, logi)
    torch.cuda.synchronize()
    return phys.cpu().numpy(), logi.cpu().numpy()


def _fused(inp, cl, max_ctx, k, n):
    B = cl.shape[0]
    phys = torch.full((B * n, k), 7, dtype=torch.int32, device="cuda")
    logi = torch.full_like(phys, 7)
    ops.indexer_topk(inp.q_fp8.view(B, n, 64, 128), inp.cache, inp.weights, cl, inp.block_tables, max_ctx, k,
                     phys, logi)
    torch.cuda.synchronize()
    return phys.cpu().numpy(), logi.cpu().numpy()


@pytest.mark.parametrize("lens,n,k", [
    ([1024, 2048, 3000, 4096], 1, 2048),
    ([65536, 40000, 100, 5000], 1, 2048),
    ([20000, 70000, 3000], 2, 2048),              # MTP verify rows
    ([9000, 5000, 300], 1, 512),
    ([262144, 3000], 1, 2048),                    # the longest row: its page table does not fit in LDS
])
def test_fused_matches_indexer_then_topk(cuda, lens, n, k):
    inp, cl, max_ctx = _inputs(lens, n, seed=sum(lens) + n + k)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, k, n)
    g_phys, g_logi = _fused(inp, cl, max_ctx, k, n)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


def test_misleading_sample_takes_the_repair_path(cuda):
    """Row 0: the sampled pages (every 32nd) score 16x higher, so the threshold
    lands above almost every other token and the list is too short. Row 1: the
    sampled pages score 16x lower, so nearly every token passes and the list
    overflows. Both rows must come out exact through the in-place repair."""
    lens = [65536, 65536, 30000]
    inp, cl, max_ctx = _inputs(lens, 1, seed=5)
    scales = inp.cache[:, 64 * 128:].view(torch.float32)  # [pages, 64] per-token key scales
    bt = inp.block_tables.cpu().numpy()
    for row, factor in ((0, 16.0), (1, 1.0 / 16.0)):
        pages = torch.from_numpy(bt[row, 0:1024:32].astype(np.int64)).to("cuda")
        scales[pages] *= factor
    e_phys, e_logi = _unfused(inp, cl, max_ctx, 2048, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, 2048, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


def test_workspace_and_argument_checks(cuda):
    assert ops.indexer_topk_workspace_bytes(128, 1, 65536) > 128 * 65536 * 4
    inp, cl, max_ctx = _inputs([3000], 1, seed=1)
    out = torch.empty(1, 2048, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError):
        ops.indexer_topk(inp.q_fp8.view(1, 1, 64, 128), inp.cache, inp.weights, cl, inp.block_tables, max_ctx,
                         1000, torch.empty(1, 1000, dtype=torch.int32, device="cuda"))
    with pytest.raises(RuntimeError, match="workspace"):
        ops.indexer_topk(inp.q_fp8.view(1, 1, 64, 128), inp.cache, inp.weights, cl, inp.block_tables, max_ctx,
                         2048, out, workspace=torch.empty(16, dtype=torch.uint8, device="cuda"))


def test_fused_batch_at_the_persistent_limit(cuda):
    """4096 entries, the largest batch the persistent filter pass takes: its
    LDS page prefix is at its largest (two workgroups per CU), and every
    wave's page range crosses several batch entries; the selection is still
    exactly topk_transform over indexer_logits."""
    B, L, k = 4096, 2100, 2048
    print(f"fused batch at the persistent limit B={B} L={L}", flush=True)
    inp, cl, max_ctx = _inputs([L - (i % 64) for i in range(B)], 1, seed=4096)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, k, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, k, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


def test_fused_large_batch_takes_the_per_workgroup_filter(cuda):
    """Batches above 4096 entries do not fit the persistent filter pass's LDS
    page prefix (two workgroups per CU) and take the one-workgroup-per-24-pages
    filter instead; the
    selection is still exactly topk_transform over indexer_logits."""
    B, L, k = 8200, 2100, 2048
    print(f"fused large batch B={B} L={L}", flush=True)
    inp, cl, max_ctx = _inputs([L] * B, 1, seed=8200)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, k, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, k, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


def test_fused_max_context_below_some_rows(cuda):
    """max_context_len = 6000 (not a page multiple) with rows of 7000 and 9000
    tokens: every stage clamps a row to max_context_len, as the unfused
    operators do (the logits stop at max_context_len)."""
    print("fused max_context below rows", flush=True)
    inp, cl, _ = _inputs([7000, 5000, 9000, 2500], 1, seed=6000)
    max_ctx, k = 6000, 2048
    e_phys, e_logi = _unfused(inp, cl, max_ctx, k, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, k, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


@pytest.mark.parametrize("lens,n", [
    ([28672, 28673, 2048, 2049, 1, 70000], 1),  # last row whose marks are bytes, first with bits, rows at top-k
    ([131072, 8192, 6000, 2047], 1),           # each row is sampled by its own length
    ([131072, 2048, 2049, 7000], 2),           # entries with one row at or below top-k and one above
    ([2048, 5, 2047], 1),                      # no page is scored
])
def test_ragged_batches_sample_each_row_by_its_length(cuda, lens, n):
    print(f"ragged fused lens={lens} n={n}", flush=True)
    inp, cl, max_ctx = _inputs(lens, n, seed=sum(lens) + n)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, 2048, n)
    g_phys, g_logi = _fused(inp, cl, max_ctx, 2048, n)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


@pytest.mark.parametrize("length,pages,one_score", [
    (65536, 2, False),     # 512 copies of each score: the threshold bin is too crowded to rank by counting
    (20000, 30, False),    # about ten copies: ranked by counting, ties by position
    (10000, 1, True),      # one score: the list fits, its threshold bin does not fit in LDS
    (40000, 1, True),      # one score: the list overflows
])
def test_repeated_scores_select_the_lowest_positions(cuda, length, pages, one_score):
    print(f"repeated scores length={length} pages={pages}", flush=True)
    inp, cl, max_ctx = _inputs([length, 3000, 70000], 1, seed=length)  # the longest row: lists, not whole rows
    width = inp.block_tables.shape[1]
    inp.block_tables[0] = inp.block_tables[0, torch.arange(width, device="cuda") % pages]
    if one_score:
        page = inp.cache[int(inp.block_tables[0, 0])]
        page[:64 * 128] = page[:128].repeat(64)
        page[64 * 128:] = page[64 * 128:64 * 128 + 4].repeat(64)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, 2048, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, 2048, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


@pytest.mark.parametrize("lens,n,k", [
    ([16384, 16383, 4097, 4096, 2049, 2048, 1], 1, 2048),   # the longest short row; 4 and 8 keys a thread; around top-k
    ([16384, 2049, 2048, 2], 2, 2048),                      # MTP rows: one token of an entry at top-k, one above
    ([513, 512, 511, 577, 64], 1, 512),
    ([8193, 700, 513], 2, 512),
    ([100, 7], 1, 2048),                                    # nothing to score
    ([32768, 32767, 20481, 16385, 9000], 1, 2048),          # 32K contexts: 8 chunks
    ([65536, 61441], 1, 2048),                              # two rows of 64K: 16 chunks
])
def test_short_contexts_select_whole_rows(cuda, lens, n, k):
    print(f"short fused lens={lens} n={n} k={k}", flush=True)
    inp, cl, max_ctx = _inputs(lens, n, seed=sum(lens) + n + k)
    assert max_ctx <= 65536
    e_phys, e_logi = _unfused(inp, cl, max_ctx, k, n)
    g_phys, g_logi = _fused(inp, cl, max_ctx, k, n)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


@pytest.mark.parametrize("length,pages,one_score,max_ctx", [
    (16384, 1, False, 16384),  # 256 copies of each score
    (16000, 50, False, 16000), # about five copies: the threshold bin is ranked by counting
    (16384, 1, True, 16384),   # one score: radix levels down to the position bits
    (7000, 3, False, 3001),    # max_context_len below the row, not a page multiple
])
def test_short_contexts_with_repeated_scores(cuda, length, pages, one_score, max_ctx):
    print(f"short repeated length={length} pages={pages}", flush=True)
    inp, cl, _ = _inputs([length, 2500], 1, seed=length + pages)
    width = inp.block_tables.shape[1]
    inp.block_tables[0] = inp.block_tables[0, torch.arange(width, device="cuda") % pages]
    if one_score:
        page = inp.cache[int(inp.block_tables[0, 0])]
        page[:64 * 128] = page[:128].repeat(64)
        page[64 * 128:] = page[64 * 128:64 * 128 + 4].repeat(64)
    e_phys, e_logi = _unfused(inp, cl, max_ctx, 2048, 1)
    g_phys, g_logi = _fused(inp, cl, max_ctx, 2048, 1)
    assert np.array_equal(g_logi, e_logi)
    assert np.array_equal(g_phys, e_phys)


def _list_flags(workspace, rows):
    """(candidates, redone) of each row's candidate list: 16-byte header, 16384 keys and positions."""
    head = workspace.view(torch.int32)[: rows * (4 + 2 * 16384)].view(rows, -1)[:, :4].cpu()
    return head[:, 1], head[:, 2]


def _long_rows(rows, length, seed):
    """Decode rows over one shared context: queries of their own, the same pages."""
    one = synth.make_indexer_inputs([length], next_n=1, seed=seed, device="cuda")
    many = synth.make_indexer_inputs([64] * rows, next_n=1, seed=seed + 1, device="cuda")
    width = max(one.block_tables.shape[1], 2048)  # a context limit of 128K: lists, not whole rows
    bt = torch.zeros(rows, width, dtype=torch.int32, device="cuda")
    bt[:, : one.block_tables.shape[1]] = one.block_tables
    one.q_fp8, one.weights, one.block_tables = many.q_fp8, many.weights, bt
    cl = torch.full((rows, 1), length, dtype=torch.int32, device="cuda")
    return one, cl, width * 64


@pytest.mark.parametrize("kind", ["normal", "outlier", "inf", "tail", "near", "ties"])
@pytest.mark.parametrize("length", [131072, 6000])
def test_long_lists_of_crowded_scores_are_not_redone(cuda, kind, length):
    """Lists past 6144 entries (hot keys that the sample does not see), positive
    ones and ones that cross zero, whose scores carry an outlier, an infinity, a
    long tail, or lie close together: selected exactly from the list, without
    the one-workgroup redo from the row's logits."""
    print(f"long lists {kind} {length}", flush=True)
    rows = 8
    inp, cl, max_ctx = _long_rows(rows, length, seed=5)
    # the key scales: a hot key's scores grow, whatever their sign
    pages = inp.block_tables[0, : -(-length // 64)].long()
    raw = inp.cache[pages]
    scale = raw[:, 64 * 128:].contiguous().view(torch.float32)
    g = torch.Generator(device="cuda").manual_seed(3)
    step = max(1, -(-pages.numel() // 16))
    unseen = (torch.arange(pages.numel(), device="cuda") % step != 0)[:, None]
    if length > 100000:
        scale = torch.where(unseen & (torch.rand(scale.shape, generator=g, device="cuda") < 0.06), scale * 16, scale)
    if kind in ("outlier", "inf"):
        scale[3, 7:40] *= 1e9 if kind == "outlier" else 1e36  # the product with some scores overflows
    if kind == "tail":
        scale = scale * torch.exp(4 * torch.randn(scale.shape, generator=g, device="cuda"))
    if kind in ("near", "ties"):  # one key everywhere: scores 1e-6 apart, or the same
        raw[:, : 64 * 128] = raw[0, :128].repeat(64)
        spread = torch.rand(scale.shape, generator=g, device="cuda") if kind == "near" else torch.zeros_like(scale)
        scale = scale[0, 0] * (1 + 1e-6 * spread)
        # most keys score nothing, so that lists of 2048 to 16384 remain
        scale = torch.where(torch.rand(scale.shape, generator=g, device="cuda") < min(1.0, 8000 / length), scale, 0.0)
    raw[:, 64 * 128:] = scale.contiguous().view(torch.uint8)
    inp.cache[pages] = raw
    e_phys, e_logi = _unfused(inp, cl, max_ctx, 2048, 1)
    ws = torch.zeros(ops.indexer_topk_workspace_bytes(rows, 1, max_ctx), dtype=torch.uint8, device=cuda)
    phys = torch.full((rows, 2048), 7, dtype=torch.int32, device=cuda)
    logi = torch.full_like(phys, 7)
    ops.indexer_topk(inp.q_fp8.view(rows, 1, 64, 128), inp.cache, inp.weights, cl, inp.block_tables, max_ctx, 2048,
                     phys, logi, workspace=ws)
    torch.cuda.synchronize()
    count, redone = _list_flags(ws, rows)
    print(kind, length, count.tolist(), redone.tolist(), flush=True)
    assert np.array_equal(logi.cpu().numpy(), e_logi)
    assert np.array_equal(phys.cpu().numpy(), e_phys)
    usable = (count >= 2048) & (count <= 16384)
    assert torch.equal(redone != 0, ~usable)
    if kind not in ("near", "ties"):
        assert usable.all() and (length < 100000 or (count > 6144).any())
