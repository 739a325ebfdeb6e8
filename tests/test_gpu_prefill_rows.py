"""GPU: prompt steps with decoding rows (delta_paged_prefill_rows) against the plain prefill launch and
fp64, and the block-order and page-check edges of the prefill kernel."""
import random

import pytest
import torch

from delta_amd import _lib, kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def build(rows, hq, hkv, dtype, seed, spoil=True):
    """rows: (new tokens, tokens after the step).  Slots past a row's end hold NaN when ``spoil``."""
    rng = random.Random(seed)
    counts = [n // 16 + 1 for _, n in rows]
    perm = list(range(sum(counts) + 3))
    rng.shuffle(perm)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kv = torch.randn((len(perm), 2, 16, hkv, 128), generator=gen, device=DEV).to(dtype)
    ids, ptr, qo = [], [0], [0]
    for (m, n), c in zip(rows, counts):
        pages = perm[len(ids):len(ids) + c]
        if spoil:
            kv[pages[-1], :, n % 16:] = float("nan")
        ids += pages
        ptr.append(len(ids))
        qo.append(qo[-1] + m)
    i32 = dict(dtype=torch.int32, device=DEV)
    q = torch.randn((max(qo[-1], 1), hq, 128), generator=gen, device=DEV).to(dtype)
    return dict(q=q, kv=kv, qo=torch.tensor(qo, **i32), ptr=torch.tensor(ptr, **i32), ids=torch.tensor(ids, **i32),
                last=torch.tensor([n % 16 for _, n in rows], **i32))


def launch(c, rows, max_qo, scale=128 ** -0.5, hints=None):
    q, kv = c["q"], c["kv"]
    hq, hkv, B = q.shape[1], kv.shape[3], c["qo"].numel() - 1
    o = torch.full_like(q, 7.0)
    lse = torch.full(q.shape[:2], 7.0, device=DEV)
    args = [q.data_ptr(), q.stride(0), q.stride(1), kv.data_ptr(), kv.shape[0], c["qo"].data_ptr(), c["ptr"].data_ptr(),
            c["ids"].data_ptr(), c["ids"].numel(), c["last"].data_ptr(), o.data_ptr(), o.stride(0), o.stride(1),
            lse.data_ptr(), B, hq, hkv, 128, K._dtype_code(q), scale, max_qo]
    stream = torch.cuda.current_stream().cuda_stream
    if rows:
        n = _lib.query("delta_paged_prefill_rows_workspace_bytes", B, hq, hkv, c["ids"].numel())
        ws = torch.full((n,), 255, dtype=torch.uint8, device=DEV)  # NaN partials where none are written
        pages = c["ids"].numel()
        hints = (B, pages, pages) if hints is None else hints
        _lib.call("delta_paged_prefill_rows", *args, q.shape[0], *hints, ws.data_ptr(), n, stream)
    else:
        _lib.call("delta_paged_prefill", *args, stream)
    torch.cuda.synchronize()
    return o, lse


CASES = {
    "joins_g4": ([(77, 77)] + [(1, 1 + 97 * i) for i in range(20)], 32, 8, torch.bfloat16),
    "joins_g7_chunked": ([(1, 3000), (40, 1040), (1, 1), (0, 64), (2, 50), (1, 16), (1, 17), (1, 2047)], 28, 4,
                         torch.float16),
    "one_row": ([(1, 5000)], 12, 2, torch.bfloat16),
    "all_single_g1": ([(1, 10 + 300 * i) for i in range(9)], 4, 4, torch.float16),
    "long_row_beside_short_ones_g8": ([(1, 40000)] + [(1, 33)] * 300 + [(5, 5)], 8, 1, torch.bfloat16),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prefill_rows_matches_prefill_and_fp64(name):
    """Rows of other token counts keep the plain launch's bits; single-token rows agree within the two
    kernels' roundings of P (2e-2, the attention tolerance) and with fp64 on sampled rows; lse to fp32."""
    rows, hq, hkv, dtype = CASES[name]
    c = build(rows, hq, hkv, dtype, seed=len(rows))
    mx = max(m for m, _ in rows)
    o0, l0 = launch(c, False, mx)
    o1, l1 = launch(c, True, mx)
    qo = c["qo"].tolist()
    for b, (m, n) in enumerate(rows):
        s = slice(qo[b], qo[b + 1])
        if m != 1:
            assert torch.equal(o0[s], o1[s]) and torch.equal(l0[s], l1[s])
            continue
        assert (o0[s].float() - o1[s].float()).abs().max().item() <= 2e-2
        assert (l0[s] - l1[s]).abs().max().item() <= 1e-4
    singles = [b for b, (m, _) in enumerate(rows) if m == 1]
    for b in singles[:3] + singles[-2:]:
        n = rows[b][1]
        pages = c["ids"][c["ptr"][b]:c["ptr"][b + 1]].long()
        kv = c["kv"][pages].double()
        k, v = (kv[:, i].reshape(-1, hkv, 128)[:n] for i in (0, 1))
        q = c["q"][qo[b]].double().view(hkv, hq // hkv, 128)
        s = torch.einsum("hgd,nhd->hgn", q.cpu(), k.cpu()) * 128 ** -0.5
        o = torch.einsum("hgn,nhd->hgd", s.softmax(-1), v.cpu()).reshape(hq, 128)
        assert (o1[qo[b]].cpu().double() - o).abs().max().item() <= 2e-2


def test_prefill_rows_zero_length_and_invalid_pages():
    """A single-token row without pages gives zeros and -inf; ids outside the cache are masked, in the
    prompt's steps and in the decoding rows, and their neighbours' NaN never reaches the output."""
    rows = [(300, 300), (1, 700), (1, 200), (130, 900)]
    c = build(rows, 32, 8, torch.bfloat16, seed=5)
    ptr = c["ptr"].tolist()
    for b, at in ((0, 3), (0, 18), (1, 40), (3, 0), (3, 30)):
        c["ids"][ptr[b] + at] = -1 if at % 2 else c["kv"].shape[0]
    c["kv"][0] = float("nan")  # page 0 stands in for an invalid id's address
    used = (c["ids"] == 0).nonzero().flatten()
    c["ids"][used] = c["kv"].shape[0] - 1
    o0, l0 = launch(c, False, 300)
    o1, l1 = launch(c, True, 300)
    assert torch.isfinite(o0).all() and torch.isfinite(o1).all()
    assert (o0.float() - o1.float()).abs().max().item() <= 2e-2 and (l0 - l1).abs().max().item() <= 1e-4
    c["ptr"][3:] = c["ptr"][2].clone()  # rows 2 and 3: no pages
    o1, l1 = launch(c, True, 300)
    assert torch.all(o1[301] == 0) and torch.all(l1[301] == float("-inf"))


@pytest.mark.parametrize("lens", [[5000, 4100], [64] * 40, [3, 700, 64, 65, 1, 2000, 511, 4095],
                                  [1024, 1, 1009, 16],                    # by tile, 64 tiles a row
                                  [40] * 63 + [900, 17, 16] + [5] * 70,   # by row, past 64 and 128 rows
                                  [17] * 12, [17] * 13, [1] * 64])        # few slots: by slot
def test_prefill_block_orders_match_a_row_at_a_time(lens):
    """8-wave blocks (4096 tokens and more), 4-wave blocks, blocks by tile (up to 12 rows), by row and by
    slot: each row equals the launch of that row alone, bit for bit where both use the same block size."""
    c = build([(n, n) for n in lens], 28, 4, torch.bfloat16, seed=sum(lens))
    o, lse = launch(c, False, max(lens))
    qo, ptr = c["qo"].tolist(), c["ptr"].tolist()
    for b, n in enumerate(lens):
        one = dict(q=c["q"][qo[b]:qo[b + 1]].contiguous(), kv=c["kv"], qo=torch.tensor([0, n], dtype=torch.int32, device=DEV),
                   ptr=torch.tensor([0, ptr[b + 1] - ptr[b]], dtype=torch.int32, device=DEV),
                   ids=c["ids"][ptr[b]:ptr[b + 1]].contiguous(), last=c["last"][b:b + 1].contiguous())
        o1, l1 = launch(one, False, max(lens) if max(lens) < 4096 else max(n, 4096))
        assert torch.equal(o1, o[qo[b]:qo[b + 1]]) and torch.equal(l1, lse[qo[b]:qo[b + 1]])


def test_prefill_grid_of_more_slots_than_one_dimension_holds():
    """max_qo_len may exceed every row: 300 rows x 188 tiles are 56400 slots, most without a block, over two grid
    layers; the same bits as with the rows' own maximum."""
    c = build([(40, 40)] * 250 + [(7, 90)] * 50, 28, 4, torch.bfloat16, seed=9)
    o0, l0 = launch(c, False, 40)
    o1, l1 = launch(c, False, 3000)
    assert torch.equal(o0, o1) and torch.equal(l0, l1)


@torch.inference_mode()  # as the engine captures: torch's graph state must not change mode between captures
def test_paged_prefill_takes_the_rows_path_where_it_should():
    assert K._prefill_has_decode_rows(808, 32, 777, 32 * 300)
    assert K._prefill_has_decode_rows(4, 4, 1, 4 * 84)
    assert not K._prefill_has_decode_rows(4, 4, 1, 4 * 84 - 1)     # short rows
    assert K._prefill_has_decode_rows(131, 32, 100, 7 + 31 * 64)
    assert not K._prefill_has_decode_rows(131, 32, 100, 6 + 31 * 64)
    assert not K._prefill_has_decode_rows(8192, 1, 8192, 513)      # one prompt
    assert not K._prefill_has_decode_rows(8 * 1024, 8, 1024, 8 * 65)  # equal prompts
    rows, hq, hkv, dtype = CASES["joins_g7_chunked"]
    rows = [(m, n + 600 * (m > 0)) for m, n in rows]
    c = build(rows, hq, hkv, dtype, seed=4)
    args = (c["q"], c["kv"], c["qo"], c["ptr"], c["ids"], c["last"])
    assert K._prefill_has_decode_rows(c["q"].shape[0], len(rows), 40, c["ids"].numel())
    o = K.paged_prefill(*args, max_qo_len=40)
    total = c["ids"].numel() - 3  # the guess: all rows but the longest prompt
    assert torch.equal(o, launch(c, True, 40, hints=(7, total, min(total, 4 * -(-total // 7))))[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        og = K.paged_prefill(*args, max_qo_len=40)
    for _ in range(3):
        og.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(og, o)


def test_paged_prefill_takes_the_callers_word_for_the_decoding_rows(monkeypatch):
    """With ``single_pages`` nothing is guessed: prompts alone get no split launch, one long decoding row
    beside longer prompts does, on the caller's workspace and without an allocation; what does not fit in
    memory is not needed."""
    sent = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (sent.append((name, a)), real(name, *a))[1])
    gave_workspace = lambda: sent[-1][1][-3]
    prompts = build([(400, 400), (150, 150)], 8, 2, torch.bfloat16, seed=1)
    joined = build([(300, 300), (290, 290), (1, 6000), (1, 20)], 8, 2, torch.bfloat16, seed=2)
    singles = [6000 // 16 + 1, 20 // 16 + 1]
    call = lambda c, mx, **kw: K.paged_prefill(c["q"], c["kv"], c["qo"], c["ptr"], c["ids"], c["last"], max_qo_len=mx, **kw)

    o = call(prompts, 400, single_pages=[])
    assert gave_workspace() is None and torch.equal(o, launch(prompts, False, 400)[0])
    plain, split = launch(joined, False, 300)[0], launch(joined, True, 300, hints=(2, sum(singles), singles[0]))[0]
    assert not torch.equal(plain, split)
    ws = torch.empty(K.paged_prefill_workspace_bytes(4, 8, 2, joined["ids"].numel()), dtype=torch.uint8, device=DEV)
    out = torch.empty_like(joined["q"])
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    call(joined, 300, single_pages=singles, workspace=ws, out=out)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
    assert gave_workspace() == ws.data_ptr() and torch.equal(out, split)
    assert torch.equal(call(joined, 300, single_pages=singles), split)
    with pytest.raises(ValueError, match="workspace too small"):
        call(joined, 300, single_pages=singles, workspace=ws[:1024])
    with pytest.raises(ValueError, match="single_pages names"):
        call(joined, 300, single_pages=[10 ** 6])

    def full(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*a, **kw)

    empty = torch.empty
    monkeypatch.setattr(torch, "empty", full)
    assert torch.equal(call(joined, 300, single_pages=singles), plain)
    assert gave_workspace() is None


def test_engine_names_the_decoding_rows_of_its_prompt_steps(monkeypatch):
    """Requests that join a running one: each prompt step passes the pages of the rows that decode and the
    engine's own workspace, which is large enough for a step over the whole pool."""
    from delta_amd.backend import LMBackend
    be = LMBackend(dtype=torch.bfloat16, device=DEV, cuda_graph_decode=True)
    be.is_main_process = False
    be.load_model("random:tiny-test", n_layer=2, seed=1)
    be.setup_caches(max_batch_size=2, max_seq_length=400)
    seen = []
    real = K.paged_prefill
    monkeypatch.setattr(K, "paged_prefill", lambda q, kv, qo, *a, **kw: (seen.append((qo.tolist(), a, kw)),
                                                                        real(q, kv, qo, *a, **kw))[1])
    be.add_requests([torch.arange(1, n) for n in (90, 30, 55)], [200, 36, 70], [])
    be.run_scheduler_loop()
    joins = 0
    for qo, (ptr, ids, last), kw in seen:
        n = [b - a for a, b in zip(qo, qo[1:])]
        pages = [b - a for a, b in zip(ptr.tolist(), ptr.tolist()[1:])]
        assert kw["single_pages"] == [p for p, m in zip(pages, n) if m == 1]
        assert kw["workspace"] is be.workspace
        joins += bool(kw["single_pages"])
    assert joins
    assert be.workspace.numel() >= K.paged_prefill_workspace_bytes(2, 4, 2, be.max_num_pages)
