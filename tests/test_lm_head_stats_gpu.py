"""Log-probabilities without a backward pass: the statistics of logits that are not written."""
import pytest
import torch

from areal_vllm_amd import ops
from areal_vllm_amd.ops import logprob as lp, train_gemm as tg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,first,temperature", [(600, 65536, 128, 0, 1.0), (700, 65536 + 4, 256, 1000, 0.7),
                                                     (1030, 75968, 1536, 75968, 1.0), (769, 65600 + 252, 384, 0, 1.9)])
def test_stats_are_those_of_the_written_logits(M, N, K, first, temperature):
    torch.manual_seed(M)
    x = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, device="cuda") * 4 * K ** -0.5).bfloat16()
    labels = torch.randint(0, first + N + 500, (M,), device="cuda")  # also ids outside the shard
    labels[:4] = torch.tensor([first, first + N - 1, first + N, -100], device="cuda")
    assert tg.stats_supported(x, w, temperature)
    out = torch.full((4, M + 3), float("nan"), device="cuda")[:, :M]
    tg.logit_stats(x, w, labels, temperature, first, out)
    ref = torch.stack(lp.logprob_stats(lp._aligned_copy(tg.tgemm_tn(x, w)), labels, temperature, first))
    assert torch.equal(out[3], ref[3])  # the same products in the same order
    assert torch.allclose(out[0], ref[0], rtol=2.0 ** -23, atol=0)  # one product with 1 / temperature on either side
    # every exponential has an argument of up to 50 with a rounding of 2^-24 of it in both, and sums of N terms in fp32 trees
    assert ((out[1] - ref[1]).abs() <= ref[1] * 2.0 ** -16).all()
    big = torch.stack([ref[1] * ref[0].abs(), ref[2].abs()]).amax(0)
    assert ((out[2] - ref[2]).abs() <= big * 2.0 ** -16).all()


def test_a_block_of_forbidden_ids():
    torch.manual_seed(3)
    M, N, K = 600, 65536, 128
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    x[:, 0] = 1.0
    w[39936:40064, 0] = float("-inf")  # two whole blocks of 64 columns
    w[50000, 0] = float("-inf")
    labels = torch.randint(0, 39936, (M,), device="cuda")
    labels[0] = 40000
    assert tg.stats_supported(x, w, 1.0)
    out = torch.empty(4, M, device="cuda")
    tg.logit_stats(x, w, labels, 1.0, 0, out)
    ref = torch.stack(lp.logprob_stats(tg.tgemm_tn(x, w), labels))
    assert torch.equal(out[3], ref[3]) and out[3, 0] == float("-inf")
    assert torch.equal(out[0], ref[0])
    assert ((out[1] - ref[1]).abs() <= ref[1] * 2.0 ** -16).all()  # as above
    assert out[2].isnan().all() and ref[2].isnan().all()  # 0 times -inf, in either form


def test_no_grad_head_equals_the_one_with_logits():
    torch.manual_seed(0)
    T, N, K = 1300, 65536, 256
    x = torch.randn(T, K, device="cuda").bfloat16()
    w = torch.nn.Parameter((torch.randn(N, K, device="cuda") * 4 * K ** -0.5).bfloat16())
    labels = torch.randint(0, N, (T,), device="cuda")
    with torch.no_grad():
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        logp, ent = ops.lm_head_logprobs(x, w, labels, chunk=700)
        assert torch.cuda.max_memory_allocated() - before < T * N * 2 // 4  # no logits
    glogp, gent = ops.lm_head_logprobs(x, w, labels, chunk=700)
    assert glogp.requires_grad and not logp.requires_grad
    # log of a sum that agrees to 2^-16, and differences of numbers up to 30 in fp32
    assert (logp - glogp).abs().max() < 2e-5 and (ent - gent).abs().max() < 4e-5


def test_a_last_few_rows_do_not_bring_all_logits_back(monkeypatch):
    torch.manual_seed(1)
    T, N, K, chunk = 860, 65536, 256, 100  # 800 rows at once, then 60
    x = torch.randn(T, K, device="cuda").bfloat16()
    w = torch.nn.Parameter((torch.randn(N, K, device="cuda") * 4 * K ** -0.5).bfloat16())
    labels = torch.randint(0, N, (T,), device="cuda")
    rows, stats = [], tg.logit_stats
    monkeypatch.setattr(tg, "logit_stats", lambda h, *a: (rows.append(h.shape[0]), stats(h, *a)))
    with torch.no_grad():
        logp, ent = ops.lm_head_logprobs(x, w, labels, chunk=chunk)
    assert rows == [800]
    glogp, gent = ops.lm_head_logprobs(x, w, labels, chunk=chunk)
    assert (logp - glogp).abs().max() < 2e-5 and (ent - gent).abs().max() < 4e-5  # as above
