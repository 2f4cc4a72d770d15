"""mhip_gemm_sums (shares of K as fp32 sums) against the same sums in 64 bits at the edges of its tiles (64, 128) and
stages (64 k), and GPT-2 over token counts on both sides of the lines between its three forms."""
import pytest
import torch

from metalhlo_amd import _lib, kernels

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 72, 520), (193, 768, 768), (200, 136, 3080), (513, 768, 3072), (1000, 64, 72)])
@pytest.mark.parametrize("parts", [0, 1, 3, 8])
def test_sums(dtype, M, N, K, parts):
    """parts = 0: the number that is recommended; more parts than stages leave some empty."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, b = torch.randn(M, K, generator=g, device="cuda").to(dtype), torch.randn(K, N, generator=g, device="cuda").to(dtype)
    parts = parts or kernels.matmul_sums_parts(M, N, K, dtype)
    sums = kernels.matmul_sums(a, b, parts)
    assert sums.shape == (parts, M, N)
    a64, b64 = a.double().cpu(), b.double().cpu()
    bound = (K + parts) * 2.0 ** -24 * (a64.abs() @ b64.abs())          # every product and sum in fp32
    assert ((sums.double().cpu().sum(0) - a64 @ b64).abs() <= bound).all()


def test_refusals():
    bf = torch.bfloat16
    assert not kernels.matmul_sums_parts(64, 60, 64, bf) and not kernels.matmul_sums_parts(64, 64, 60, bf) and not kernels.matmul_sums_parts(64, 64, 64, torch.float32)
    x = torch.zeros(64, 64, dtype=bf, device="cuda")
    for a, b, parts in ((x, x, 0), (x, x, 9), (x, torch.zeros(64, 60, dtype=bf, device="cuda"), 1), (x, x.float(), 1)):
        with pytest.raises((_lib.MhipError, ValueError, TypeError)):
            kernels.matmul_sums(a, b, parts)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,few,parts", [(1, 96, True, True), (1, 97, False, True), (2, 150, False, True), (1, 768, False, True), (1, 769, False, False)])
def test_gpt2_forms_agree(dtype, B, S, few, parts):
    """The form a token count takes against the one for many tokens: the same roundings, fp32 sums in another order.  Where
    those differ a value rounds the other way and carries on, at most a few units by the second layer."""
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=2, vocab=1000, n_pos=1040)
    model = GPT2(cfg, init_params(cfg, seed=3), compute_dtype=dtype)
    ids = torch.randint(0, cfg.vocab, (B, S), generator=torch.Generator().manual_seed(1), dtype=torch.int32).cuda()
    assert model._few_tokens(B * S) == few and (model._sum_parts(B * S) != (0, 0)) == parts
    got = model.forward(ids)
    model._few_tokens, model._full_tiles = (lambda tokens: False), 0
    whole = model.forward(ids)
    err = (got.double() - whole.double()).norm() / whole.double().norm()
    assert err <= 2 * EPS[dtype], float(err)
    if not few and not parts:
        assert torch.equal(got, whole)


@pytest.mark.parametrize("d_model,d_ff", [(256, 1024), (512, 2048), (768, 3072), (1024, 2048)])
def test_a_sequence_has_the_same_bits_in_any_batch_of_more_than_768_tokens(d_model, d_ff):
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=2, d_model=d_model, n_head=d_model // 64, d_ff=d_ff, vocab=1000)
    model = GPT2(cfg, init_params(cfg, seed=5))
    ids = torch.randint(0, cfg.vocab, (8, 257), generator=torch.Generator().manual_seed(2), dtype=torch.int32).cuda()
    whole = model.forward(ids)
    for batch in (3, 5):                                         # 771 and 1285 tokens
        assert torch.equal(model.forward(ids[:batch]), whole[:batch])


def test_gpt2_in_parts_from_a_graph():
    """Replays with eager work between them give the eager bits."""
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=2, vocab=1000)
    model = GPT2(cfg, init_params(cfg, seed=4))
    ids = [torch.randint(0, cfg.vocab, (2, 150), generator=torch.Generator().manual_seed(i), dtype=torch.int32).cuda() for i in range(3)]
    step = model.capture(ids[0])
    for x in ids + ids:
        got = step(x).clone()
        assert torch.equal(got, model.forward(x))
        torch.cuda.synchronize()
