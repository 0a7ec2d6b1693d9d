"""GPU parity of the sparse MLA decode attention (trnrt_amd.kernels.dsa_decode -> dsa_sparse_mla_decode) against
the oracle (oracle/dsa_oracle.py sparse_mla_ref, trnrt/kernels/dsa_decode.py:26-37 + trnrt/kernels/dsa_slots.py:
48-65) on the same seeded inputs and selections; bound: bf16 output within 2e-2 abs/rel (the north star), lse within
1e-3 abs."""

import pytest
import torch

from oracle import dsa_oracle as O
from tests._helpers import assert_attention_close, say
from trnrt_amd import _lib
from trnrt_amd import workloads as W
from trnrt_amd.kernels import dsa_decode

pytestmark = pytest.mark.gpu


def _selection(inp, keep=None):
    cfg = inp.cfg
    keep = cfg.keep if keep is None else keep
    sc = O.indexer_ref(inp.q_idx, inp.w_k, inp.k_cache, inp.k_scale, inp.table, inp.ctx_len, cfg.page_size,
                       inp.max_pages * cfg.page_size)
    return O.topk_ref(sc, keep, inp.ctx_len)


def _run(inp, idx, cnt, splits=0, out_dtype=torch.bfloat16):
    g = inp.to("cuda")
    o, lse = dsa_decode.attend_tokens(g.q, g.kv_cache, g.kv_scale, idx.cuda(), cnt.cuda(), g.table,
                                      inp.cfg.page_size, inp.cfg.scale, out_dtype=out_dtype, splits=splits)
    torch.cuda.synchronize()
    return o.cpu(), lse.cpu()


def _ref(inp, idx, cnt):
    return O.sparse_mla_ref(inp.q, inp.kv_cache, inp.kv_scale, idx, cnt, inp.table, inp.cfg.page_size, inp.cfg.scale)


@pytest.mark.parametrize("splits", [0, 1, 5])
def test_config1(splits):
    say(f"attention config 1 splits={splits}")
    inp = W.make_inputs(W.CONFIGS[1], seed=0)
    idx, cnt = _selection(inp)
    o, lse = _run(inp, idx, cnt, splits)
    ro, rl = _ref(inp, idx, cnt)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse, rl, atol=1e-3, rtol=1e-4)


def test_config2_full():
    say("attention config 2")
    inp = W.make_inputs(W.CONFIGS[2], seed=0)
    idx, cnt = _selection(inp)
    o, lse = _run(inp, idx, cnt)
    ro, rl = _ref(inp, idx, cnt)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse, rl, atol=1e-3, rtol=1e-4)


def test_counts_below_keep_and_zero():
    """cnt < keep masks the tail slots; cnt 0 attends position 0 alone with lse NEG_INF (the reference's fully
    masked row over slots that all read position 0)."""
    say("attention short counts")
    cfg = W.Config("short", B=4, L=3000, H=32, Hi=16, keep=2048)
    inp = W.make_inputs(cfg, seed=5, lengths=[3000, 100, 1, 2500])
    idx, cnt = _selection(inp)
    cnt[2] = 0
    idx[2] = 0
    for splits in (0, 1, 3):
        o, lse = _run(inp, idx, cnt, splits, out_dtype=torch.float32)
        ro, rl = _ref(inp, idx, cnt)
        assert_attention_close(o, ro)
        torch.testing.assert_close(lse[[0, 1, 3]], rl[[0, 1, 3]], atol=1e-3, rtol=1e-4)
        assert (lse[2] < -1e29).all()


def test_row_form_equals_token_form():
    say("attention row form vs token form")
    cfg = W.Config("rows", B=2, L=4096, H=16, Hi=16, keep=1000)
    inp = W.make_inputs(cfg, seed=6)
    idx, cnt = _selection(inp, keep=1000)
    cnt[1] = 333
    idx[1, 333:] = 0
    rows = torch.stack([O.token_slots(inp.table[b], idx[b], 64) for b in range(2)])
    bias = torch.where(torch.arange(1000).view(1, -1) < cnt.view(2, 1), 0.0, O.NEG_INF)
    g = inp.to("cuda")
    o_row, l_row = dsa_decode.attend(g.q, g.kv_cache.view(-1, 1, 576), rows.cuda(), bias.cuda().unsqueeze(-1),
                                     cfg.scale, kc_scale=g.kv_scale, lse=True)
    o_tok, l_tok = _run(inp, idx, cnt, out_dtype=torch.float32)
    ro, rl = _ref(inp, idx, cnt)
    assert_attention_close(o_row.cpu(), ro)
    torch.testing.assert_close(o_row.cpu(), o_tok, atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(l_row.cpu(), l_tok, atol=1e-5, rtol=1e-5)


def test_fully_masked_row_form_is_uniform():
    say("attention fully masked row form")
    cfg = W.Config("mask", B=1, L=512, H=16, Hi=16, keep=100)
    inp = W.make_inputs(cfg, seed=8)
    rows = torch.randint(64, 64 * 9, (1, 100), generator=torch.Generator().manual_seed(1))
    bias = torch.full((1, 100), O.NEG_INF)
    g = inp.to("cuda")
    o, lse = dsa_decode.attend(g.q, g.kv_cache, rows.cuda(), bias.cuda(), cfg.scale, kc_scale=g.kv_scale, lse=True)
    ro, rl = O.sparse_mla_slots_ref(inp.q, inp.kv_cache, inp.kv_scale, rows, bias, cfg.scale)
    assert_attention_close(o.cpu(), ro)
    assert (lse.cpu() < -1e29).all()


def test_wrong_scale_is_caught():
    """Positive control: per-token value scales shuffled between tokens must break the tolerance."""
    say("attention positive control")
    inp = W.make_inputs(W.CONFIGS[1], seed=9)
    idx, cnt = _selection(inp)
    bad = W.Inputs(**{**inp.__dict__, "kv_scale": inp.kv_scale[torch.randperm(inp.kv_scale.numel())]})
    o, _ = _run(bad, idx, cnt, out_dtype=torch.float32)
    ro, _ = _ref(inp, idx, cnt)
    assert (o - ro).abs().max() > 2e-2 * (1 + ro.abs().max())


@pytest.mark.parametrize("dqk", [576, 512])
def test_many_row_form_vs_oracle(dqk):
    """The many-row form (64-head workgroups, one per query row, pipelined gather: sparse_mla_wide_kernel), taken
    when one split suffices and the rows fill the GPU: ragged counts (0, 1, one chunk, a chunk and one slot, every
    slot, random), 64 heads, both row widths, against the oracle."""
    from tests._helpers import launched_kernels
    g = torch.Generator().manual_seed(dqk + 7)
    B, H, L, ps, keep = 300, 64, 1024, 64, 320
    say(f"attention many-row form dqk={dqk} B={B} keep={keep}")
    npg = L // ps
    num_pages = 1 + B * npg
    kv, ks = W.quantize_rows(torch.randn(num_pages * ps, dqk, generator=g))
    table = (torch.randperm(num_pages - 1, generator=g)[: B * npg] + 1).view(B, npg).to(torch.int32)
    q = torch.randn(B, H, dqk, generator=g).to(torch.bfloat16)
    cnt = torch.randint(0, keep + 1, (B,), generator=g)
    cnt[:6] = torch.tensor([0, 1, 64, 65, keep, 63])
    idx = torch.zeros(B, keep, dtype=torch.int64)
    for b in range(B):
        n = int(cnt[b])
        idx[b, :n] = torch.randperm(L, generator=g)[:n].sort().values
    qg, kvg, ksg, tg = q.cuda(), kv.cuda(), ks.cuda(), table.cuda()
    res = {}

    def step():
        res["o"], res["lse"] = dsa_decode.attend_tokens(qg, kvg, ksg, idx.cuda(), cnt.cuda(), tg, ps, 192 ** -0.5,
                                                        out_dtype=torch.float32)

    names = launched_kernels(step)
    assert names == ["sparse_mla_wide_kernel"], names
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, 192 ** -0.5)
    assert_attention_close(res["o"], ro)
    live = cnt > 0
    torch.testing.assert_close(res["lse"].cpu()[live], rl[live], atol=1e-3, rtol=1e-4)
    assert (res["lse"].cpu()[~live] < -1e29).all()


@pytest.mark.parametrize("B,H,keep", [(9, 64, 2048), (43, 64, 2048), (5, 128, 4160), (70, 64, 192), (140, 128, 64)])
def test_many_row_form_in_splits(B, H, keep):
    """The many-row form in splits (from 9 workgroups' rows on; 8, 5, 8, 1 and 1 of them here), counts that leave the
    last splits empty (0, 1, one chunk, a chunk and one slot, all), against the oracle; slots of one 4,224-token context."""
    g = torch.Generator().manual_seed(B + keep)
    say(f"attention many-row form in splits B={B} H={H} keep={keep}")
    L, ps = 4224, 64
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    cnt = torch.randint(0, keep + 1, (B,), generator=g)
    cnt[:5] = torch.tensor([0, 1, 64, min(65, keep), keep])
    idx = torch.zeros(B, keep, dtype=torch.int64)
    for b in range(B):
        n = int(cnt[b])
        idx[b, :n] = torch.randperm(L, generator=g)[:n].sort().values
    o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps,
                                      192 ** -0.5)
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, 192 ** -0.5)
    live = cnt > 0
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu()[live], rl[live], atol=1e-3, rtol=1e-4)
    assert (lse.cpu()[~live] < -1e29).all()


@pytest.mark.parametrize("keep, splits, form", [
    (2048, 3, "wide"), (2048, 2, "wide"), (2048, 0, "wide"),  # all its splits, fewer, one
    (4160, 3, "wide"), (4160, 2, "wide"), (4160, 0, "split"),  # one split is longer than its slot lists: the split form
])
def test_many_row_form_within_the_workspace(keep, splits, form):
    """70 rows, 3 splits where the workspace holds them: a workspace of the split outputs of fewer (a byte short of one
    more), or of none, is taken as the split form's own needs are (none here), and gives the same result."""
    from tests._helpers import launched_kernels
    B, H, L, ps = 70, 64, 4224, 64
    g = torch.Generator().manual_seed(keep + splits)
    say(f"attention many-row form keep={keep} in a workspace for {splits} splits")
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    cnt = torch.randint(1, keep + 1, (B,), generator=g)
    cnt[:2] = torch.tensor([keep, 1])
    idx = torch.stack([torch.randperm(L, generator=g)[:keep] for _ in range(B)])
    size = B * (splits + 1) * H * (512 * 4 + 8) + 256 - 1 if splits else 256
    args = (q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps, 192 ** -0.5)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    names = launched_kernels(lambda: dsa_decode.attend_tokens(*args, workspace=ws))
    kernel = "sparse_mla_wide_kernel" if form == "wide" else "sparse_mla_kernel"
    assert names == [kernel] + ["combine_splits_kernel"] * (splits > 0), names
    o, lse = dsa_decode.attend_tokens(*args, workspace=ws)
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, 192 ** -0.5)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu(), rl, atol=1e-3, rtol=1e-4)


@pytest.mark.parametrize("rows_form", [False, True])
@pytest.mark.parametrize("dqk", [576, 512])
def test_many_row_form_moving_maxima(dqk, rows_form):
    """The many-row form on rows whose scores keep rising along the selection (kv scales growing 3,000-fold, so the
    running maximum moves, and the output is rescaled, in most chunks), and falling (it moves once), with 128 heads,
    pages of 48 (no power of two) and the rows + count form; bf16 outputs against the oracle. The bound is the file's
    2e-2: the largest scale is 1, so a value is at most about 4.6, and the weights' rounding to bf16 (2^-9 of sum p |v|)
    and the output's (2^-9 of it) are at most 0.009 each."""
    g = torch.Generator().manual_seed(dqk + rows_form)
    B, H, L, ps, keep = 130, 128, 480, 48, 448
    say(f"attention many-row form, moving maxima dqk={dqk} rows={rows_form}")
    npg = L // ps
    num_pages = 1 + npg
    kv = torch.randn(num_pages * ps, dqk, generator=g).to(W.FP8)
    table = (torch.randperm(npg, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    up = torch.logspace(-3.5, 0.0, L)  # by position
    scale_of = torch.ones(num_pages * ps)
    slot = O.token_slots(table[0], torch.arange(L), ps)
    scale_of[slot] = up
    q = torch.randn(B, H, dqk, generator=g).to(torch.bfloat16)
    cnt = torch.randint(1, keep + 1, (B,), generator=g)
    cnt[:5] = torch.tensor([keep, 0, 1, 65, 128])
    idx = torch.zeros(B, keep, dtype=torch.int64)
    for b in range(B):
        n = int(cnt[b])
        idx[b, :n] = torch.randperm(L, generator=g)[:n].sort(descending=bool(b & 1)).values
    if rows_form:
        from trnrt_amd.kernels import dsa_slots_c
        rows = torch.stack([O.token_slots(table[b], idx[b], ps) for b in range(B)])
        bias = torch.where(torch.arange(keep).view(1, -1) < cnt.view(-1, 1), 0.0, -1e30)
        o, lse = dsa_slots_c.attend(q.cuda(), kv.cuda(), rows.int().cuda(), bias.cuda(), 0.6, lse=True,
                                    kc_scale=scale_of.cuda())
        ro, rl = O.sparse_mla_ref(q, kv, scale_of, idx, cnt, table, ps, 0.6)
        live = cnt > 0
        o, ro = o[live.cuda()], ro[live]
    else:
        o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), scale_of.cuda(), idx.cuda(), cnt.cuda(), table.cuda(),
                                          ps, 0.6)
        ro, rl = O.sparse_mla_ref(q, kv, scale_of, idx, cnt, table, ps, 0.6)
        live = cnt > 0
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu()[live], rl[live], atol=1e-3, rtol=1e-4)
    assert (lse.cpu()[~live] < -1e29).all()


LEVELS = (0.0, -40.0, -89.0, -100.0, -500.0, -2000.0, 100.0, 2000.0)  # scaled scores (natural units), by head


def _leveled(B, H, dqk, L, ps, low, seed):
    """Queries and a cache of one L-token context whose heads' scores lie within a few units of LEVELS (heads in turn),
    those of the positions `low` 1,000 below that for every other group of 8 heads. Dims 0 and 1 carry the two: 8 in the
    keys (dim 1: in the low positions' alone), level x 2 in the queries, times the softmax scale 1/16 (all exact)."""
    g = torch.Generator().manual_seed(seed)
    kv = torch.randn(L + ps, dqk, generator=g)
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32)
    kv[:, 0] = 8.0
    kv[:, 1] = 0.0
    kv[O.token_slots(table, low, ps), 1] = 8.0
    q = torch.randn(B, H, dqk, generator=g)
    h = torch.arange(H)
    q[:, :, 0] = 2.0 * torch.tensor(LEVELS)[h % 8]
    q[:, :, 1] = torch.where(h // 8 % 2 == 1, -2000.0, 0.0)
    return q.to(torch.bfloat16), kv.to(W.FP8), torch.ones(L + ps), table.expand(B, -1).contiguous(), 1.0 / 16


@pytest.mark.parametrize("form", ["tokens", "rows"])
@pytest.mark.parametrize("B, keep, dqk", [(9, 2048, 576), (9, 2048, 512), (300, 256, 576), (300, 256, 512)])
def test_many_row_form_scores_far_from_zero(B, keep, dqk, form):
    """Softmax does not change when a head's scores are shifted, so heads whose scores all lie far below or above 0
    (LEVELS: past -128 in base 2, where 2^-score is infinite) are as any other, and so is a row's or a split's first
    chunk (64 slots) that lies far below the rest: 8 splits of 256 slots (9 rows) and one split (300 rows), rows of one
    slot, one chunk, a chunk and one, a split and one, all. Bounds: the file's; for lse 5e-3, what fp32 sums of up to
    32,000 over 36 steps round to (32,000 x 36 x 2^-24 x the scale)."""
    say(f"attention many-row form, scores far from zero, B={B} dqk={dqk} {form}")
    H, L, ps = 64, 2048, 64
    low = torch.cat([torch.arange(0, 64), torch.arange(512, 576), torch.arange(1024, 1300)])
    q, kv, ks, table, scale = _leveled(B, H, dqk, L, ps, low, seed=B + dqk)
    cnt = torch.randint(1, keep + 1, (B,), generator=torch.Generator().manual_seed(B))
    cnt[:7] = torch.tensor([1, 64, 65, keep, min(keep, 513), min(keep, 577), 2])
    idx = torch.where(torch.arange(keep) < cnt.view(-1, 1), torch.arange(keep), 0)
    if form == "rows":
        from trnrt_amd.kernels import dsa_slots_c
        rows = torch.stack([O.token_slots(table[b], idx[b], ps) for b in range(B)])
        bias = torch.where(torch.arange(keep).view(1, -1) < cnt.view(-1, 1), 0.0, O.NEG_INF)
        o, lse = dsa_slots_c.attend(q.cuda(), kv.cuda(), rows.int().cuda(), bias.cuda(), scale, lse=True,
                                    kc_scale=ks.cuda())
    else:
        o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps,
                                          scale)
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, scale)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu(), rl, atol=5e-3, rtol=1e-4)


@pytest.mark.parametrize("B, keep", [(9, 2048), (300, 256)])
def test_many_row_form_reads_no_slot_past_the_count(B, keep):
    """Entries of the selection past a row's count name any token, also one whose cache row was never written (NaN bytes
    and scale): they take no part in the row, in splits or not, whatever its count."""
    say(f"attention many-row form, unwritten cache rows past the count, B={B}")
    g = torch.Generator().manual_seed(B)
    H, L, ps = 64, 4096, 64
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    bad = O.token_slots(table[0], torch.arange(L // 2, L), ps)
    kv.view(torch.uint8)[bad] = 0x7F
    ks[bad] = float("nan")
    cnt = torch.randint(1, keep + 1, (B,), generator=g)
    cnt[:6] = torch.tensor([1, 64, 65, keep, keep - 1, 0])
    idx = torch.stack([torch.randperm(L // 2, generator=g)[:keep].sort().values for _ in range(B)])
    live = torch.arange(keep) < cnt.view(-1, 1).clamp(min=1)  # (a row with none attends its first entry, masked)
    o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), ks.cuda(), torch.where(live, idx, idx + L // 2).cuda(),
                                      cnt.cuda(), table.cuda(), ps, 192 ** -0.5)
    ro, rl = O.sparse_mla_ref(q, kv, ks, torch.where(live, idx, idx[:, :1]), cnt, table, ps, 192 ** -0.5)
    assert torch.isfinite(ro[cnt > 0]).all()
    assert_attention_close(o.cpu()[cnt > 0], ro[cnt > 0])
    torch.testing.assert_close(lse.cpu()[cnt > 0], rl[cnt > 0], atol=1e-3, rtol=1e-4)
    v = O.dequant(kv[O.token_slots(table[0], idx[5, :1], ps)], ks[O.token_slots(table[0], idx[5, :1], ps)])[:, :512]
    assert_attention_close(o.cpu()[5], v.expand(H, -1))


@pytest.mark.parametrize("B, H", [(9, 64), (48, 64), (40, 128), (100, 64)])
def test_many_row_form_reads_no_empty_split(B, H):
    """8, 5, 3 and 2 splits of which a row's short selection fills the first ones (each count of them, 1 and a masked row
    included), in a workspace of NaN bytes: what a split with no slot leaves there does not reach the output."""
    say(f"attention many-row form, empty splits in a NaN workspace, B={B} H={H}")
    g = torch.Generator().manual_seed(B)
    keep, L, ps = 2048, 4096, 64
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    cnt = torch.randint(1, 500, (B,), generator=g)
    cnt[:9] = torch.tensor([0, 1, 256, 257, 769, 1025, 1400, 1793, 2048])
    idx = torch.stack([torch.randperm(L, generator=g)[:keep].sort().values for _ in range(B)])
    idx[0] = 0
    ws = torch.full((_lib.workspace_bytes(_lib.DSA_WS_ATTENTION, B, H, keep, 0, 0),), 0xFF, dtype=torch.uint8,
                    device="cuda")
    o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps,
                                      192 ** -0.5, workspace=ws)
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, 192 ** -0.5)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu()[1:], rl[1:], atol=1e-3, rtol=1e-4)
    assert (lse.cpu()[0] < -1e29).all()


@pytest.mark.parametrize("B, H, keep, form", [
    (8, 64, 256, "split form"), (9, 64, 256, "one"), (5, 128, 256, "one"),  # more than 8 workgroups' rows
    (9, 64, 512, "one"), (10, 64, 512, "split form"), (10, 64, 448, "one"),  # 8 chunks and more of up to 16 rows: by
    (16, 64, 1024, "split form"), (16, 64, 1600, "splits"), (17, 64, 1024, "splits"),  # the split form's rounds
    (17, 64, 640, "one"), (17, 64, 641, "splits"), (23, 64, 768, "splits"), (24, 64, 768, "one"), (24, 64, 769, "splits"),
])
def test_attention_form_by_rows_and_slots(B, H, keep, form):
    """The form that splits 0 takes at the edges of its rule, and its result, against the oracle."""
    from tests._helpers import launched_kernels
    say(f"attention form B={B} H={H} keep={keep}")
    g = torch.Generator().manual_seed(B + keep)
    L, ps = 2048, 64
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    cnt = torch.randint(1, keep + 1, (B,), generator=g)
    cnt[:3] = torch.tensor([keep, 1, keep - 1])
    idx = torch.stack([torch.randperm(L, generator=g)[:keep].sort().values for _ in range(B)])
    args = (q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps, 192 ** -0.5)
    names = launched_kernels(lambda: dsa_decode.attend_tokens(*args))
    assert names == ["sparse_mla_kernel" if form == "split form" else "sparse_mla_wide_kernel"] + \
        ["combine_splits_kernel"] * (form != "one"), names
    o, lse = dsa_decode.attend_tokens(*args)
    ro, rl = O.sparse_mla_ref(q, kv, ks, idx, cnt, table, ps, 192 ** -0.5)
    assert_attention_close(o, ro)
    torch.testing.assert_close(lse.cpu(), rl, atol=1e-3, rtol=1e-4)


def test_many_row_form_error_against_64_bits():
    """The many-row form is no further from 64 bits than the split form with its combine (splits 3: what these rows took
    before): lse, whose error is that of fp32 scores and sums (4.4e-8 of it against 4.1e-8; 5.1e-8 with the scale's product
    and the maximum's rounded), within 1.1 times; the output, where the weights' rounding to bf16 and its own are all,
    within 1.03 (the rounding of a weight depends on its place between two powers of two, so on the maximum in use)."""
    say("attention many-row form, error against 64 bits")
    g = torch.Generator().manual_seed(5)
    B, H, L, ps, keep = 26, 128, 8192, 64, 2048
    kv, ks = W.quantize_rows(torch.randn(L + ps, 576, generator=g))
    table = (torch.randperm(L // ps, generator=g) + 1).to(torch.int32).expand(B, -1).contiguous()
    q = torch.randn(B, H, 576, generator=g).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(L, generator=g)[:keep].sort().values for _ in range(B)])
    cnt = torch.full((B,), keep)
    scale = 192 ** -0.5
    ro, rl = torch.empty(B, H, 512, dtype=torch.float64), torch.empty(B, H, dtype=torch.float64)
    for b in range(B):
        at = O.token_slots(table[b], idx[b], ps)
        K = kv[at].double() * ks[at].double().unsqueeze(1)
        sc = q[b].double() @ K.T.contiguous() * scale
        rl[b] = sc.logsumexp(1)
        ro[b] = (sc - rl[b].unsqueeze(1)).exp() @ K[:, :512].contiguous()
    err = {}
    for splits in (0, 3):
        o, lse = dsa_decode.attend_tokens(q.cuda(), kv.cuda(), ks.cuda(), idx.cuda(), cnt.cuda(), table.cuda(), ps, scale,
                                          splits=splits)
        err[splits] = [float((x.cpu().double() - r).norm() / r.norm()) for x, r in ((o, ro), (lse, rl))]
    say(f"  many-row {err[0]} split form {err[3]}")
    assert err[0][0] <= 1.03 * err[3][0]
    assert err[0][1] <= 1.1 * err[3][1]
