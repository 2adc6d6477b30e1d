"""Layers of a few tokens, on both sides of the rule that hands them from the
fused decode launches to the grouped GEMMs."""
import pytest
import torch

from inferno_amd import Q2_K, Q3_K, Q4_K, Q8_0, SCORE_SOFTMAX, ops

H, E, I, TOP_K, IS = 3072, 32, 1024, 6, 1024


def _weights(quant, seed, rows, cols):
    return ops.synth_quantized(quant, seed, 0.02, rows, cols, torch.device("cuda:0"))


def _layer(quant, shared, T, router_std=0.02):
    g = torch.Generator(device="cuda").manual_seed(2)
    kw = {}
    if shared:
        kw = dict(shared_gate=_weights(Q8_0, 9, IS, H), shared_up=_weights(Q8_0, 10, IS, H),
                  shared_down=_weights(Q8_0, 11, H, IS))
    mats = dict(gate=_weights(quant, 0, E * I, H), up=_weights(quant, 1, E * I, H),
                down=_weights(quant, 2, E * H, I))
    layer = ops.MoELayer(
        hidden=H, experts=E, intermediate=I, top_k=TOP_K, quant=quant, down_quant=quant,
        score_fn=SCORE_SOFTMAX, norm_topk_prob=True, routed_scaling_factor=1.0,
        router=torch.randn(E, H, generator=g, device="cuda") * router_std, router_bias=None,
        shared_intermediate=IS if shared else 0, max_tokens=T, **mats, **kw)
    return layer, mats, kw


def _exact(quant, mats, kw, x, ids, w):
    """The layer in 64 bits for the ids and weights that the layer chose."""
    deq = {n: ops.dequantize(quant, m).view(E, -1, I if n == "down" else H).double()
           for n, m in mats.items()}
    x = x.double()

    def ffn(v, gate, up, down):
        a = v @ gate.T
        return (a * torch.sigmoid(a) * (v @ up.T)) @ down.T

    out = torch.zeros(x.shape[0], H, dtype=torch.float64, device="cuda")
    for t in range(x.shape[0]):
        for e, wt in zip(ids[t].tolist(), w[t].tolist()):
            out[t] += wt * ffn(x[t], deq["gate"][e], deq["up"][e], deq["down"][e])
    if kw:
        sg, su = (ops.dequantize(Q8_0, kw[n]).view(IS, H).double() for n in ("shared_gate", "shared_up"))
        out += ffn(x, sg, su, ops.dequantize(Q8_0, kw["shared_down"]).view(H, IS).double())
    return out


def _both_sides(quant, shared, x, monkeypatch, **kw):
    """Relative error of each token's row against fp64, by the rule and on the
    decode launches (a threshold that no batch reaches)."""
    T = x.shape[0]
    layer, mats, sh = _layer(quant, shared, T, **kw)
    ids = torch.empty(T * TOP_K, dtype=torch.int32, device="cuda")
    w = torch.empty(T * TOP_K, device="cuda")
    by_rule = layer.forward(x, None, ids=ids, weights=w)
    ref = _exact(quant, mats, sh, x, ids.view(T, TOP_K), w.view(T, TOP_K))
    monkeypatch.setenv("INFERNO_PREFILL_MIN_ASSIGNMENTS", "100000")
    decode = layer.forward(x)

    def err(y):
        return ((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()

    return err(by_rule), err(decode), by_rule, decode


# The decode launches round weights times scales and h to f16, in units that
# each 16 values choose; per row (the layers' own 2e-3 is per batch).
BOUND = 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 4, 6])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
def test_fp32_tokens_keep_their_bits(quant, shared, T, monkeypatch):
    # fp32 tokens enter the decode launches as two f16 terms (22 bits); one f16
    # term of the grouped GEMMs would hold 11, so the rule leaves them there
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, H, generator=g, device="cuda")
    _, decode, y, z = _both_sides(quant, shared, x, monkeypatch)
    assert decode < BOUND and torch.equal(y, z)
