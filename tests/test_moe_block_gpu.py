"""A layer of routed experts (``models/moe.py``) on both sides of the rules that choose its kernels."""
import pytest
import torch

from symmetry_amd import ops
from symmetry_amd.models import model_class
from symmetry_amd.models.config import ModelConfig
from symmetry_amd.models.weights import ModelWeights, ShardSpec

pytestmark = pytest.mark.gpu


def _block(E, k, d, F):
    cfg = ModelConfig("moe", 256, d, F, 1, d // 128, d // 128, num_experts=E, top_k=k, bos_token_id=1, eos_token_ids=(2,))
    g = torch.Generator(device="cuda").manual_seed(E + F)

    def rnd(*shape):
        return (torch.randn(*shape, device="cuda", generator=g) * shape[-1] ** -0.5).bfloat16()

    one = torch.ones(d, device="cuda", dtype=torch.bfloat16)
    w = {"embed": rnd(256, d), "lm_head": rnd(256, d), "norm": one, "layers.0.ln1": one, "layers.0.ln2": one,
         "layers.0.wqkv": rnd(3 * d, d), "layers.0.wo": rnd(d, d), "layers.0.router": rnd(E, d) * 4,
         "layers.0.w13": rnd(E, 2 * F, d), "layers.0.w2": rnd(E, d, F)}
    model = model_class(cfg)(ModelWeights(cfg, ShardSpec(), w), torch.device("cuda", 0), max_decode_ctx=512)
    return model.moe, w


# (experts, choices, width, expert width, tokens, gathers, down products on grouped_gemm)
@pytest.mark.parametrize("E,k,d,F,T,gathers,grouped", [
    (16, 4, 256, 4096, 16, True, False), (16, 4, 256, 4352, 16, False, False),     # decode rows: experts up to 4096
    (16, 4, 2048, 256, 8, True, False), (16, 4, 2304, 256, 8, False, False),       # and widths up to 2048
    (16, 4, 384, 4352, 16, True, False),                                           # (a width that the skinny GEMM does not take)
    (32, 4, 256, 192, 40, True, False), (33, 4, 256, 192, 40, True, True),         # prompts: narrow experts among many
    (64, 8, 256, 1024, 70, True, True), (64, 8, 256, 1088, 70, True, False),
    (64, 8, 384, 768, 8, True, False), (64, 2, 128, 64, 700, True, True), (16, 4, 256, 1024, 300, True, False),
])
def test_routed_experts(gpu, monkeypatch, E, k, d, F, T, gathers, grouped):
    """Against 64-bit products of the chosen experts.  The gated rows are rounded to bf16, 2^-9 of themselves at most, and
    so is the sum of all other roundings (fp32): under 2^-8 of the result's 2-norm."""
    monkeypatch.setenv("SYMMETRY_MOE_PRESHUFFLE", "0")
    moe, w = _block(E, k, d, F)
    x = torch.randn(T, d, device="cuda", generator=torch.Generator(device="cuda").manual_seed(T)).bfloat16()
    calls, plain = [], ops.grouped_gemm
    monkeypatch.setattr(ops, "grouped_gemm", lambda *a: calls.append(a[-1]) or plain(*a))
    assert moe._gathers(0, T * k, d) == gathers
    got = moe._forward_local(0, x, False).double()
    assert calls == ([ops.GROUPED_F32] if grouped else [])
    logits = x.double() @ w["layers.0.router"].double().t()
    p, pick = logits.topk(k, -1)
    p = p.softmax(-1)
    want = torch.zeros(T, d, dtype=torch.float64, device="cuda")
    for e in range(E):
        t, j = (pick == e).nonzero(as_tuple=True)
        gate, up = (x[t].double() @ w["layers.0.w13"][e].double().t()).split(F, 1)
        want.index_add_(0, t, p[t, j, None] * ((torch.nn.functional.silu(gate) * up) @ w["layers.0.w2"][e].double().t()))
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("E,k,d,F,T,walks", [(16, 4, 1536, 1536, 8, True), (64, 4, 2048, 2048, 16, True), (9, 1, 1536, 3072, 64, True),
                                             (16, 4, 1024, 1536, 8, False), (16, 4, 1536, 1024, 8, False)])
def test_down_products_of_few_rows(gpu, monkeypatch, E, k, d, F, T, walks):
    """One fp32 product by the walk against the skinny GEMM's slabs, bounds as above."""
    monkeypatch.setenv("SYMMETRY_MOE_PRESHUFFLE", "0")
    moe, w = _block(E, k, d, F)
    calls, plain = [], ops.grouped_skinny
    monkeypatch.setattr(ops, "grouped_skinny", lambda *a, **kw: calls.append(1) or plain(*a, **kw))
    x = torch.randn(T, d, device="cuda", generator=torch.Generator(device="cuda").manual_seed(T)).bfloat16()
    got = moe._forward_local(0, x, False).double()
    assert calls == ([] if walks else [1])
    p, pick = (x.double() @ w["layers.0.router"].double().t()).topk(k, -1)
    p = p.softmax(-1)
    want = torch.zeros(T, d, dtype=torch.float64, device="cuda")
    for e in range(E):
        t, j = (pick == e).nonzero(as_tuple=True)
        gate, up = (x[t].double() @ w["layers.0.w13"][e].double().t()).split(F, 1)
        want.index_add_(0, t, p[t, j, None] * ((torch.nn.functional.silu(gate) * up) @ w["layers.0.w2"][e].double().t()))
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("T", [1, 3, 8])
def test_decode_off_the_residual(gpu, monkeypatch, T):
    """A decode step's block (norm, routing, experts, residual, next norm's input) at one row and more, in one routing launch."""
    monkeypatch.setenv("SYMMETRY_MOE_PRESHUFFLE", "0")
    E, k, d, F = 16, 4, 1536, 1536
    moe, w = _block(E, k, d, F)
    g = torch.Generator(device="cuda").manual_seed(T)
    resid = torch.randn(T, d, device="cuda", generator=g)
    norm, after = (torch.rand(d, device="cuda", generator=g).bfloat16() + 0.5 for _ in range(2))
    x = (resid.double() * (resid.double().square().mean(-1, keepdim=True) + 1e-5).rsqrt() * norm.double())
    p, pick = (x @ w["layers.0.router"].double().t()).topk(k, -1)
    p = p.softmax(-1)
    want = resid.double().clone()
    for e in range(E):
        t, j = (pick == e).nonzero(as_tuple=True)
        gate, up = (x[t] @ w["layers.0.w13"][e].double().t()).split(F, 1)
        want.index_add_(0, t, p[t, j, None] * ((torch.nn.functional.silu(gate) * up) @ w["layers.0.w2"][e].double().t()))
    xw = torch.empty(T, d, device="cuda", dtype=torch.bfloat16)
    start = resid.clone()
    moe.forward_decode(0, resid, norm, 1e-5, after, xw, None)
    # x and the gated rows rounded to bf16, and the routing weights' logits off x by its rounding: under 2^-7 of the block's part
    assert float((resid.double() - want).norm() / (want - start.double()).norm()) <= 2.0 ** -7
    assert float((xw.double() - resid.double() * after.double()).abs().max()) <= 2.0 ** -8 * float((resid.double() * after.double()).abs().max())
