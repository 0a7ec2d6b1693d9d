"""The whole decode layer step on the GPU (trnrt_amd.kernels.dsa_layer -> dsa_decode_layer) against the oracle:
scores within 1e-2 (row-relative), top-k indices bit-exact against the oracle's selection OF THE KERNEL'S SCORES, the
bf16 output within 2e-2 of the oracle attention over the kernel's selection; at the full ragged and 1M shapes the
indexer is checked on a sample of positions per row (the oracle is exact per position) and everything else in full."""

import pytest
import torch

from oracle import dsa_oracle as O
from tests._helpers import assert_attention_close, row_rel_err, say
from trnrt_amd import workloads as W
from trnrt_amd.kernels.dsa_layer import DecodeLayer

pytestmark = pytest.mark.gpu


def _layer(g):
    cfg = g.cfg
    L = DecodeLayer(cfg.B, cfg.Hi, cfg.H, g.max_pages, cfg.page_size, g.num_pages, cfg.keep, cfg.scale,
                    max_len=max(g.lengths))
    L.step(g.q_idx, g.w_k, g.k_cache, g.k_scale, g.q, g.kv_cache, g.kv_scale, g.table, g.ctx_len)
    torch.cuda.synchronize()
    return L


def _attention_check(g, L, rows=None):
    """Oracle attention over the kernel's own selection (rows: which batch rows to check)."""
    cfg = g.cfg
    rows = range(cfg.B) if rows is None else rows
    idx, cnt = L.idx.cpu(), L.cnt.cpu()
    for b in rows:
        slots = O.token_slots(g.table[b].cpu(), idx[b].long(), cfg.page_size).to(g.kv_cache.device)
        K = O.dequant(g.kv_cache[slots].cpu(), g.kv_scale[slots].cpu())
        bias = torch.where(torch.arange(cfg.keep) < int(cnt[b]), 0.0, O.NEG_INF)
        ro, rl = O.sparse_mla_rows_ref(g.q[b].cpu(), K, bias, cfg.scale)
        assert_attention_close(L.out[b].cpu(), ro)
        torch.testing.assert_close(L.lse[b].cpu(), rl, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("c", [1, 2])
def test_layer_full_oracle(c):
    say(f"layer config {c}")
    inp = W.make_inputs(W.CONFIGS[c], seed=0)
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, 64, sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    ri, rc = O.topk_ref(sc, inp.cfg.keep, inp.ctx_len)
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)
    _attention_check(inp, L)


def test_layer_rows_of_8192_one_kernel_selection():
    """Rows of 4,097 .. 8,192 scores: the fused indexer's first-level histogram feeds the one-workgroup-per-row
    selection, which also writes the cache rows through the page table (128 pages a row); ragged lengths, every
    stage against the oracle."""
    say("layer rows of 8192")
    cfg = W.Config("layer-8k", B=4, L=8192, H=64, Hi=64)
    inp = W.make_inputs(cfg, seed=5, lengths=[8192, 8000, 4097, 6001])
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, 64, sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)
    _attention_check(inp, L)


@pytest.mark.parametrize("ps,L", [(32, 8192), (128, 8192), (32, 20000)])
def test_layer_other_page_sizes(ps, L):
    """Pages of 32 and 128 tokens (a 32-key indexer tile is one page, or a quarter of one): the indexer's page reads,
    the selection's cache rows through the table (page shift 5 and 7) and the attention's gather, against the oracle;
    ragged lengths, rows of 8,192 (the one-workgroup selection) and 20,000 scores (the chunked one)."""
    say(f"layer page_size={ps} L={L}")
    cfg = W.Config(f"layer-ps{ps}", B=3, L=L, H=64, Hi=64, page_size=ps)
    inp = W.make_inputs(cfg, seed=ps + L, lengths=[L, L - 5, L // 2 + 3])
    g = inp.to("cuda")
    layer = _layer(g)
    sc = layer.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, ps, sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(layer.idx.cpu().long(), ri) and torch.equal(layer.cnt.cpu().long(), rc)
    _attention_check(inp, layer)


def test_layer_long_ragged_many_short_rows():
    """A batch with one row past 32,768 tokens (the separate kernels with the long-row indexer and selection) and many
    short rows, empty tiles and short histograms beside a long one; every stage against the oracle."""
    lengths = [40000, 1, 2, 3, 500, 2047, 2048, 2049, 33, 7, 9000, 1, 64, 4095, 100, 31]
    say(f"layer long ragged batch of {len(lengths)} rows")
    cfg = W.Config("layer-long-ragged", B=len(lengths), L=40000, H=64, Hi=64)
    inp = W.make_inputs(cfg, seed=17, lengths=lengths)
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, cfg.page_size,
                        sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    assert torch.all(sc[ref <= -1e29] < -1e29)
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)
    _attention_check(inp, L)


@pytest.mark.parametrize("H, lengths", [
    # 21 rows: XCDs 0-4 hold three (two rows at once, then one row by all 32 workgroups), XCDs 5-7 two at once
    (64, [40000, 1, 33000, 2048, 2049, 7, 36000, 100, 4095, 34000, 0, 50, 39000, 2000, 17, 3000, 33, 38000, 1024, 9,
          35000]),
    # one head group of 32 heads: the rows of an XCD one at a time
    (32, [40000, 3, 33000, 2048, 5000, 37000, 1, 64, 39000, 2047]),
])
def test_layer_long_rows_paired(H, lengths):
    """The long-row launch with two or three rows an XCD: two rows take 16 workgroups each (each workgroup's row's
    selection once, then both head groups of one split), a third row all 32; with one head group the rows go one at a
    time. Short, empty and tied-free ragged rows; every stage against the oracle."""
    say(f"layer long rows paired: H={H}, {len(lengths)} rows")
    cfg = W.Config("layer-long-paired", B=len(lengths), L=max(lengths), H=H, Hi=64)
    inp = W.make_inputs(cfg, seed=53 + H, lengths=lengths)
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, cfg.page_size,
                        sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    assert torch.all(sc[ref <= -1e29] < -1e29)
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.cnt.cpu().long(), rc)
    assert torch.equal(L.idx.cpu().long(), ri)
    _attention_check(inp, L)
    assert L.status()["gave_up"] == 0


@pytest.mark.parametrize("tied", [False, True])
def test_layer_long_rows_mixed_forms(tied):
    """Rows past 32,768 tokens in a small batch (the long-row indexer and the chunked long-row selection) beside rows
    of at most keep keys (every visible key selected), a row whose selection crowds into its first 4,096 positions
    (key scales raised a thousandfold there) and, with `tied`, rows whose scores take two values (the keep-th largest
    tied with thousands of keys). Every stage against the oracle, then a second step on the same workspace."""
    lengths = [100000, 40000, 1500, 33000, 2048, 70000]
    say(f"layer long rows, mixed forms, tied={tied}")
    cfg = W.Config("layer-long-mixed", B=len(lengths), L=100000, H=64, Hi=64)
    inp = W.make_inputs(cfg, seed=23 + tied, lengths=lengths)
    ps = cfg.page_size
    pos = torch.arange(4096)
    slots = inp.table[5, pos // ps].long() * ps + pos % ps
    inp.k_scale[slots] *= 1000.0
    if tied:  # rows 1 and 3: two key patterns, so two score values a row
        for b in (1, 3):
            n = inp.lengths[b]
            p = torch.arange(n)
            sl = inp.table[b, p // ps].long() * ps + p % ps
            inp.k_cache[sl] = inp.k_cache[64 + (p % 2)]
            inp.k_scale[sl] = inp.k_scale[64 + (p % 2)]
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, cfg.page_size,
                        sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    if tied:
        for b in (1, 3):
            assert len(torch.unique(sc[b, :inp.lengths[b]])) <= 2
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.cnt.cpu().long(), rc)
    assert torch.equal(L.idx.cpu().long(), ri)
    _attention_check(inp, L)
    # a second step on the same workspace (the histograms cleared by the first)
    L.step(g.q_idx, g.w_k, g.k_cache, g.k_scale, g.q, g.kv_cache, g.kv_scale, g.table, g.ctx_len)
    torch.cuda.synchronize()
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)


def test_layer_long_tied_row_every_tile_read():
    """A row of 300,000 tokens whose scores take two values: every 32-key tile's maximum is the row's largest score,
    so the one-launch long-row selection reads every tile of every block (296 a block: more than one round of 256
    tile loads) and lists every key; beside it a row of 50,000 with distinct scores. The selection bit-exact on the
    kernel's scores (ties to the lowest positions), the attention against the oracle."""
    lengths = [300000, 50000]
    say("layer long tied row, every tile read")
    cfg = W.Config("layer-long-tied", B=len(lengths), L=300000, H=64, Hi=64)
    inp = W.make_inputs(cfg, seed=41, lengths=lengths)
    ps = cfg.page_size
    n = lengths[0]
    p = torch.arange(n)
    sl = inp.table[0, p // ps].long() * ps + p % ps
    inp.k_cache[sl] = inp.k_cache[64 + (p % 2)]
    inp.k_scale[sl] = inp.k_scale[64 + (p % 2)]
    g = inp.to("cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    assert len(torch.unique(sc[0, :n])) <= 2
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.cnt.cpu().long(), rc)
    assert torch.equal(L.idx.cpu().long(), ri)
    _attention_check(inp, L)


@pytest.mark.parametrize("H, lengths, attend", [
    # 17 and 18 rows: past the 16 of the one-launch layer; the even indexer split past 8,192 tokens, a workgroup per 512
    # positions below; empty, one-token and full-keep rows; 64 heads in 8 splits (17 rows), all in one row block
    (64, [12000, 0, 1, 2047, 2048, 2049, 9000, 31, 33, 64, 4095, 100, 11999, 8192, 8193, 500, 7], "wide"),
    (64, [4097, 0, 1, 2047, 2048, 2049, 4096, 31, 33, 64, 4095, 100, 3000, 8000, 8192, 500, 7, 8191], "wide"),
    # 128 heads (two workgroups a row and split): the many-row attention from 5 rows on
    (128, [6000, 0, 2500, 1, 5999], "wide"),
    # the one-workgroup selection's last length and its edges (groups of 4,096), and the chunked pair's first
    (128, [16384, 0, 12289, 4096, 16383], "wide"),
    (128, [8193, 2049, 1, 8192, 8191], "wide"),
    (128, [16385, 16384, 2047, 0, 12288], "wide"),
    # 32 heads: the XCD-local attention launch over three rows an XCD
    (32, [9000, 0, 1, 2047, 2048, 2049, 8999, 31, 33, 64, 4095, 100, 3000, 8193, 8192, 500, 7], "xcd"),
])
def test_layer_batch_of_many_rows(H, lengths, attend):
    """Batches that take the separate kernels: every stage against the oracle, the selection bit-exact, the histograms
    left zero for the next call (two steps on one workspace)."""
    from tests._helpers import launched_kernels
    say(f"layer batch of {len(lengths)} rows, H={H}")
    cfg = W.Config("layer-batch", B=len(lengths), L=max(lengths), H=H, Hi=48)
    inp = W.make_inputs(cfg, seed=71 + H, lengths=lengths)
    g = inp.to("cuda")
    L = _layer(g)
    names = launched_kernels(lambda: L.step(g.q_idx, g.w_k, g.k_cache, g.k_scale, g.q, g.kv_cache, g.kv_scale, g.table,
                                            g.ctx_len))
    torch.cuda.synchronize()
    assert names[-1 if attend == "xcd" else -2] == ("decode_attend_kernel" if attend == "xcd" else
                                                    "sparse_mla_wide_kernel"), names
    sc = L.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, cfg.page_size,
                        sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    assert torch.all(sc[ref <= -1e29] < -1e29)
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)
    _attention_check(inp, L)
    assert L.status()["gave_up"] == 0


@pytest.mark.parametrize("Hi, L, even", [(33, 8192, False), (33, 8193, True), (32, 16384, False), (32, 16385, True)])
def test_layer_batch_indexer_split(Hi, L, even):
    """The indexer of a batch of 17 ragged rows at the lengths where it changes from a workgroup per 512 positions to the
    even split (later at 32 indexer heads and fewer), against the oracle, and the selection that its histogram feeds."""
    from tests._helpers import launched_kernels
    say(f"layer batch indexer split Hi={Hi} L={L}")
    lengths = [L, 0, 1, 31, 33, 512, 513, 2048, 2049, L - 1, L // 2, 4095, 4097, 8000, 100, 7, 3000]
    cfg = W.Config("layer-even", B=len(lengths), L=L, H=16, Hi=Hi)
    inp = W.make_inputs(cfg, seed=Hi + L, lengths=lengths)
    g = inp.to("cuda")
    layer = _layer(g)
    names = launched_kernels(lambda: layer.step(g.q_idx, g.w_k, g.k_cache, g.k_scale, g.q, g.kv_cache, g.kv_scale,
                                                g.table, g.ctx_len))
    assert names[0] == ("indexer_decode_long_kernel" if even else "indexer_decode_kernel"), names
    torch.cuda.synchronize()
    sc = layer.scores.cpu()
    ref = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, 64, sc.shape[1])
    assert row_rel_err(sc, ref, ref > -1e29) <= 1e-2
    assert torch.all(sc[ref <= -1e29] < -1e29)
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(layer.idx.cpu().long(), ri) and torch.equal(layer.cnt.cpu().long(), rc)


@pytest.mark.parametrize("H, B", [(64, 17), (128, 5)])
def test_layer_batch_scores_far_from_zero(H, B):
    """The many-row attention of a batch step with heads whose scores all lie far from 0 (as trained heads' do): a key
    dim of 2 for every token and query values that put head h's scores around (h % 8 - 5) x 400 in natural units."""
    say(f"layer batch, scores far from zero, H={H}")
    lengths = ([6000, 1, 64, 65, 2047, 3000, 5999] + [100 * i for i in range(1, 11)])[:B]
    cfg = W.Config("layer-levels", B=B, L=max(lengths), H=H, Hi=16)
    inp = W.make_inputs(cfg, seed=H, lengths=lengths)
    inp.kv_scale.fill_(2.0 ** -7)
    inp.kv_cache.view(torch.uint8)[:, 0] = torch.tensor([256.0]).to(W.FP8).view(torch.uint8)
    inp.q[:, :, 0] = ((torch.arange(H) % 8 - 5) * (200.0 / cfg.scale)).to(torch.bfloat16)
    L = _layer(inp.to("cuda"))
    _attention_check(inp, L)


def _sampled_indexer_check(g, sc, nsample=4096, seed=0):
    cfg = g.cfg
    gen = torch.Generator().manual_seed(seed)
    for b in range(cfg.B):
        Lb = g.lengths[b]
        pos = torch.randint(0, Lb, (nsample,), generator=gen)
        pos[:2] = torch.tensor([0, Lb - 1])
        slots = O.token_slots(g.table[b].cpu(), pos, cfg.page_size).to(g.k_cache.device)
        K = O.dequant(g.k_cache[slots].cpu(), g.k_scale[slots].cpu())
        ref = torch.einsum("h,ht->t", g.w_k[b].cpu(), torch.relu(torch.einsum("hd,td->ht", g.q_idx[b].cpu().float(), K)))
        got = sc[b, pos]
        assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2
        assert (sc[b, Lb:] < -1e29).all()


@pytest.mark.parametrize("c", [3, 4])
def test_layer_full_size(c):
    """Configs 3 (12 ragged rows of 8K-128K) and 4 (4 rows of 1M) at full size: config 3's indexer against the oracle
    on every position of every row, config 4's on 4,096 sampled positions per row (with the first and last); the
    selection bit-exact on the kernel's own scores; the attention of every row against the oracle."""
    say(f"layer config {c} (full size)")
    g = W.make_inputs(W.CONFIGS[c], seed=0, device="cuda")
    L = _layer(g)
    sc = L.scores.cpu()
    if c == 3:
        c_in = g.to("cpu")
        ref = O.indexer_ref(c_in.q_idx, c_in.w_k, c_in.k_cache, c_in.k_scale, c_in.table, c_in.ctx_len,
                            g.cfg.page_size, sc.shape[1])
        err = row_rel_err(sc, ref, ref > -1e29)
        say(f"  config 3 indexer rel err {err:.3e} (every position)")
        assert err <= 1e-2
        assert torch.all(sc[ref <= -1e29] < -1e29)
    else:
        _sampled_indexer_check(g, sc)
    ri, rc = O.topk_ref(sc, g.cfg.keep, g.lengths)
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.cnt.cpu().long(), rc)
    _attention_check(g, L, rows=range(g.cfg.B))


def test_layer_long_rows_two_launches():
    """A batch with rows past 32,768 tokens is two launches: the long-row indexer (scores and each row's first-level
    histogram), then the selection, attention and combine in one XCD-local launch (decode_long_attend_kernel);
    12 rows (two rows on four XCDs) of ragged lengths, every stage against the oracle, the workspace's histograms
    left zero (a second step gives the same results)."""
    from tests._helpers import launched_kernels

    lengths = [40000, 131072, 8192, 65536, 33000, 100000, 50000, 9000, 120000, 32769, 70000, 16384]
    say("layer long rows, two launches")
    cfg = W.Config("layer-long-2", B=len(lengths), L=131072, H=64, Hi=64)
    inp = W.make_inputs(cfg, seed=31, lengths=lengths)
    g = inp.to("cuda")
    L = DecodeLayer(cfg.B, cfg.Hi, cfg.H, g.max_pages, cfg.page_size, g.num_pages, cfg.keep, cfg.scale,
                    max_len=max(g.lengths))
    step = lambda: L.step(g.q_idx, g.w_k, g.k_cache, g.k_scale, g.q, g.kv_cache, g.kv_scale, g.table,  # noqa: E731
                          g.ctx_len)
    names = launched_kernels(step)
    assert names == ["indexer_decode_long_kernel", "decode_long_attend_kernel"], names
    torch.cuda.synchronize()
    sc = L.scores.cpu()
    ri, rc = O.topk_ref(sc, cfg.keep, inp.ctx_len)
    assert torch.equal(L.cnt.cpu().long(), rc)
    assert torch.equal(L.idx.cpu().long(), ri)
    _attention_check(inp, L)
    out0 = L.out.clone()
    step()
    torch.cuda.synchronize()
    assert torch.equal(L.idx.cpu().long(), ri) and torch.equal(L.out, out0)
    assert L.status()["gave_up"] == 0
