"""GPU: the row argmax's vector and scalar paths, and the split plans of small attention launches."""
import pytest
import torch

from delta_amd import kernels as K
from delta_amd.workloads import make_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols,stride", [(3, 151936, 151936), (2, 8, 8), (2, 7, 8), (4, 1001, 1008), (4, 1001, 1001),
                                              (1, 260, 264), (5, 2055, 2056), (2, 65543, 65544)])
def test_argmax_rows_vector_and_scalar_paths(dtype, rows, cols, stride):
    """Aligned strides take 16-byte loads (partial last units included), odd strides 2-byte ones; ties,
    all -inf rows and NaN as torch.argmax decides them."""
    gen = torch.Generator(device=DEV).manual_seed(rows * 7 + cols)
    buf = torch.full((rows, stride), 1e4, device=DEV, dtype=dtype)  # what lies past cols must not win
    x = buf[:, :cols]
    x.copy_(torch.randn(rows, cols, generator=gen, device=DEV).clamp(-3, 2).to(dtype))  # many ties at 2
    x[0, cols // 2:] = 2
    assert torch.equal(K.argmax_rows(x), torch.argmax(x.float(), -1))
    x[0] = float("-inf")
    assert int(K.argmax_rows(x)[0]) == 0
    for at in {0, cols - 1, cols // 3}:
        x[-1, at] = float("nan")
        assert int(K.argmax_rows(x)[-1]) == int(torch.argmax(x[-1].float()))


@pytest.mark.parametrize("batch,hq,hkv,lens", [
    (64, 12, 2, [8200] * 64),                            # 128 pairs, 9 units of 57 pages, split by split
    (8, 32, 8, [16384 - 900 * i for i in range(8)]),     # 64 pairs, ragged, units of 65
    (13, 40, 8, [16 * (1 + 31 * i) + i for i in range(13)]),  # 104 pairs, rows of 1-13 units
    (100, 4, 1, [2400] * 99 + [3]),                      # 100 pairs, one kv head
    (4, 32, 8, [700, 16, 5000, 1]),                      # 32 pairs, row by row, most rows one unit
    (15, 28, 4, [33 * 16 + i for i in range(15)]),       # 60 pairs, 4-wave units, partial last pages
    (31, 16, 8, [3000] * 31),                            # 248 pairs, 5 units of 38 pages
    (31, 16, 8, [1279] * 30 + [17]),                     # 248 pairs, two units of 40 pages
])
def test_small_attention_plans_match_the_dump_launch(batch, hq, hkv, lens):
    """Attention launches of 32-255 (row, kv head) pairs split into units of one kv head; the dump launch of
    the same rows splits page-major.  Both round P to bf16 from sums in another order: 2e-2, the attention
    tolerance; lse in fp32."""
    c = make_case(batch=batch, hq=hq, hkv=hkv, kv_lens=lens, seed=batch, k=4, L=2).to(DEV)
    args = (c.q, c.kv_cache, c.kv_indptr, c.kv_indices, c.kv_last_page_len)
    lse, lse2 = (torch.zeros(batch, hq, device=DEV) for _ in range(2))
    o = K.paged_decode(*args, max_pages_per_row=c.max_pages, lse=lse)
    dump = torch.empty(batch, hq, c.max_pages * 16, device=DEV)
    o2 = K.paged_decode(*args, max_pages_per_row=c.max_pages, lse=lse2, logits_dump=dump)
    torch.cuda.synchronize()
    assert (o.float() - o2.float()).abs().max().item() <= 2e-2
    assert (lse - lse2).abs().max().item() <= 1e-4
    for b in range(batch):
        n = lens[b]
        assert (torch.logsumexp(dump[b, :, :n].double(), -1) - lse[b]).abs().max().item() <= 1e-4


@pytest.mark.parametrize("batch,hq,hkv,lens", [(13, 40, 8, [16 * (1 + 31 * i) + i + 1 for i in range(13)]),
                                               (100, 4, 1, [2400] * 99 + [3])])
def test_fused_append_on_units_numbered_split_by_split(batch, hq, hkv, lens):
    """RoPE and the KV append in the launch equal rope_append and the plain launch bit for bit, cache included."""
    c = make_case(batch=batch, hq=hq, hkv=hkv, kv_lens=lens, seed=batch, k=4, L=2).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(1)
    k, v = (torch.randn(batch, hkv, 128, generator=gen, device=DEV).to(c.q.dtype) for _ in range(2))
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV)
    kv0, kv1 = c.kv_cache.clone(), c.kv_cache.clone()
    qo = torch.arange(batch + 1, dtype=torch.int32, device=DEV)
    q = K.rope_append(c.q, k, v, qo, pos, kv0, c.kv_indices, c.kv_indptr, c.kv_last_page_len)
    o0 = K.paged_decode(q, kv0, c.kv_indptr, c.kv_indices, c.kv_last_page_len, max_pages_per_row=c.max_pages)
    o1 = K.paged_decode(c.q, kv1, c.kv_indptr, c.kv_indices, c.kv_last_page_len, max_pages_per_row=c.max_pages,
                        append=K.DecodeAppend(k, v, pos, c.kv_indptr, c.kv_indices))
    assert torch.equal(o0, o1) and torch.equal(kv0, kv1)
