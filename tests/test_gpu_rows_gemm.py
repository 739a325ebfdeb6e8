"""GPU: the 33-128 row decode GEMM (delta_gemm_rows128, _silu) at the edges of its tiles and splits."""
import pytest
import torch

from delta_amd import _lib, kernels as K, model
from delta_amd.model import FeedForward, ModelArgs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,Kd,bias", [
    (33, 1536, 1536, False),    # 64-column blocks, split
    (64, 5120, 640, True),      # 128-column blocks, 10 k steps over 2 splits
    (64, 16, 64, True),         # one tile, one k step
    (37, 1040, 8960, True),     # N past a whole number of blocks, uneven splits
    (65, 4096, 1024, False),    # first size of the 128-row tile
    (128, 5120, 4160, True),    # 192-column blocks, N past a whole number of them, 65 k steps
    (100, 16400, 320, True),    # unsplit, rows and columns ragged
    (1, 208, 192, False),
    (64, 33296, 1536, False),   # unsplit, 24 k steps (four x slabs), columns past a whole number of blocks
])
def test_gemm_rows128_matches_fp32_reference(dtype, M, N, Kd, bias):
    """Partials sum to the product (fp32 sums of Kd products: 1e-5 of the sum of magnitudes, as for
    delta_gemm_rows32); the unsplit output is it rounded once.  Rows past M stay unwritten."""
    gen = torch.Generator(device=DEV).manual_seed(M * 3 + N + Kd)
    x = torch.randn(M, Kd, generator=gen, device=DEV).to(dtype)
    w = (torch.randn(N, Kd, generator=gen, device=DEV) * 0.05).to(dtype)
    b = (torch.randn(N, generator=gen, device=DEV) * 0.1).to(dtype) if bias else None
    S = K.gemm_rows128_splits(M, N, Kd)
    guard = torch.full((M + 1, N), 7.0, dtype=dtype, device=DEV)
    r = K.gemm_rows128(x, w, b, out=guard[:M] if S == 1 else None)
    r2 = K.gemm_rows128(x, w, b)
    torch.cuda.synchronize()
    ref = x.float() @ w.float().T + (b.float() if bias else 0.0)
    mag = x.float().abs() @ w.float().abs().T
    if S == 1:
        assert r.dtype == dtype and torch.all(guard[M] == 7.0)
        err = (r.float() - ref).abs()
        assert torch.all(err <= torch.finfo(dtype).eps * ref.abs() + 1e-5 * mag + 1e-6), f"max err {err.max().item()}"
    else:
        assert r.dtype == torch.float32 and tuple(r.shape) == (S, M, N)
        err = (r.sum(0) - ref).abs()
        assert torch.all(err <= 1e-5 * mag + 1e-6), f"max err {err.max().item()}"
    assert torch.equal(r, r2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,inter,Kd", [(64, 8960, 1536), (40, 16400, 192), (33, 48, 64), (128, 1040, 640),
                                        (65, 13824, 320)])
def test_gemm_rows128_silu_matches_gemm_then_silu_mul(dtype, M, inter, Kd):
    """silu(gate) * up with the roundings of the GEMM followed by delta_silu_mul: a gate or up value
    within fp32 summation noise of a rounding boundary moves by one ulp of the dtype."""
    gen = torch.Generator(device=DEV).manual_seed(M + inter + Kd)
    x = torch.randn(M, Kd, generator=gen, device=DEV).to(dtype)
    w13 = (torch.randn(2 * inter, Kd, generator=gen, device=DEV) * 0.03).to(dtype)
    got = K.gemm_rows128_silu(x, w13).float()
    ref = K.silu_mul((x.float() @ w13.float().T).to(dtype)).float()
    torch.cuda.synchronize()
    eps = torch.finfo(dtype).eps
    g, u = (x.float() @ w13.float().T).split(inter, -1)
    # one ulp of g (|silu'| <= 1.1), of silu(g), of u and of the product
    bound = eps * (1.1 * g.abs() * u.abs() + 3 * (torch.nn.functional.silu(g) * u).abs()) + 1e-5
    assert torch.all((got - ref).abs() <= bound)
    assert (got != ref).float().mean().item() < 0.02  # and few of them do


def test_ffn_at_33_to_128_rows_matches_the_library_path(monkeypatch):
    """The fused FFN on the row-major weight (kernel, partials or output) against the library GEMMs
    and delta_silu_mul, a strided x included, which keeps the library's path."""
    cfg = ModelArgs.from_name("tiny-test")
    cfg.intermediate_size = 9216
    with torch.device(DEV):
        ff = FeedForward(cfg).to(torch.bfloat16)
    fused = []
    silu = K.gemm_rows128_silu
    monkeypatch.setattr(K, "gemm_rows128_silu", lambda x, w: (fused.append(x.shape[1]), silu(x, w))[1])
    with torch.inference_mode():
        gen = torch.Generator(device=DEV).manual_seed(3)
        for p in ff.parameters():
            p.data.normal_(0, 0.05, generator=gen)
        ff.use_row_major_w13()
        for rows in (33, 64, 65, 128, 129):
            wide = torch.randn(1, rows, 520, device=DEV, generator=gen).to(torch.bfloat16)
            x = wide[..., :512].contiguous()
            ref = ff.w2(K.silu_mul(torch.nn.functional.linear(x, ff.w13))).float().view(rows, 512)
            for t in (x, wide[..., :512]):
                y = ff.forward_fused(t)
                y = (y.sum(0) if y.dtype == torch.float32 else y.float()).view(rows, 512)
                # both round silu(g) * u and the output to bf16: a few ulps of the row's magnitude
                assert (y - ref).abs().max().item() <= 4 * 2 ** -8 * ref.abs().max().item()
    assert fused == [33, 64, 65, 128]


@torch.inference_mode()
@pytest.mark.parametrize("N,Kd,rows", [(120016, 1024, (32, 33, 64, 65)), (32768, 2048, (33, 64))])
def test_lm_head_on_the_kernel_only_where_it_is_wide(N, Kd, rows, monkeypatch):
    """dense() on either side of the lm_head rule against fp32 products rounded once."""
    ran = []
    gemm = K.gemm_rows128
    monkeypatch.setattr(K, "gemm_rows128", lambda x, *a: (ran.append(x.shape[1]), gemm(x, *a))[1])
    gen = torch.Generator(device=DEV).manual_seed(N)
    layer = torch.nn.Linear(Kd, N, bias=False, device=DEV, dtype=torch.bfloat16)
    layer.weight.normal_(0, 0.05, generator=gen)
    for m in rows:
        x = torch.randn(1, m, Kd, generator=gen, device=DEV).bfloat16()
        y = model.dense(x, layer)[0].float()
        ref, mag = x[0].float() @ layer.weight.float().T, x[0].float().abs() @ layer.weight.float().abs().T
        assert torch.all((y - ref).abs() <= 2 ** -8 * ref.abs() + 1e-5 * mag + 1e-6)
    assert ran == ([33, 64] if N >= 120000 else [])


@torch.inference_mode()
@pytest.mark.parametrize("N,Kd,partial_rows", [(1536, 8960, (33, 64, 65, 128)), (4096, 4096, (33, 64)), (5120, 5120, (33, 64, 65, 128))])
def test_dense_to_norm_form_and_values(N, Kd, partial_rows):
    """Rows either side of 32, 64 and 128: fp32 partials where the kernel runs (here all split), else the rounded
    output; both the fp32 products."""
    gen = torch.Generator(device=DEV).manual_seed(Kd)
    layer = torch.nn.Linear(Kd, N, bias=False, device=DEV, dtype=torch.bfloat16)
    layer.weight.normal_(0, 0.02, generator=gen)
    for m in (33, 64, 65, 128, 129):
        x = torch.randn(1, m, Kd, generator=gen, device=DEV).bfloat16()
        y = model.dense_to_norm(x, layer)
        ref, mag = x[0].float() @ layer.weight.float().T, x[0].float().abs() @ layer.weight.float().abs().T
        if m in partial_rows:
            assert y.dtype == torch.float32 and torch.all((y.sum(0) - ref).abs() <= 1e-5 * mag + 1e-6)
        else:
            assert y.dtype == torch.bfloat16 and tuple(y.shape) == (1, m, N)
            assert torch.all((y[0].float() - ref).abs() <= 2 ** -8 * ref.abs() + 1e-5 * mag + 1e-6)


def test_a_layer_with_a_forward_of_its_own_is_called():
    """Hooks, a subclass' or an instance's forward and a trained bias act at 33-128 rows as at any other."""
    class Doubled(torch.nn.Linear):
        def forward(self, x):
            return 2 * super().forward(x)

    x = torch.randn(1, 40, 256, device=DEV).bfloat16()
    make = lambda cls=torch.nn.Linear: cls(256, 128, device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    assert not model._own_forward(make())
    hooked, wrapped, trained = make(), make(), make()
    seen = []
    hooked.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    model.dense_to_norm(x, hooked)
    assert seen == [(1, 40, 128)]
    doubled = make(Doubled)
    assert torch.equal(model.dense_to_norm(x, doubled), 2 * torch.nn.functional.linear(x, doubled.weight, doubled.bias))
    wrapped.forward = lambda t: t
    assert model.dense_to_norm(x, wrapped) is x
    trained.bias.requires_grad_(True)
    model.dense_to_norm(x, trained).float().sum().backward()
    assert torch.all(trained.bias.grad == 40)


def test_gemm_rows128_errors():
    x = torch.zeros(33, 64, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(64, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="does not take"):
        K.gemm_rows128(x, w[:40])
    with pytest.raises(ValueError, match="does not take"):
        K.gemm_rows128(torch.zeros(129, 64, dtype=torch.bfloat16, device=DEV), w)
    with pytest.raises(_lib.DeltaHipError, match="multiple of 16"):
        K.gemm_rows128_silu(x, w[:48])
    assert not K.gemm_rows128_ok(x[:, :32], w)
    assert not K.gemm_rows128_ok(x.t(), w)
