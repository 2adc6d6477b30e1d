"""Layers of a few tokens, on both sides of the rule that hands them from the
fused decode launches to the grouped GEMMs: tokens of any size (h grows with
their square, so that plain f16 rows would lose it at either end), one
activation far above the others, fp32 tokens, more than one tile of rows."""
import pytest
import torch

from inferno_amd import Q2_K, Q3_K, Q4_K, Q8_0, SCORE_SOFTMAX, ops

H, E, I, TOP_K, IS = 3072, 32, 1024, 6, 1024


def _weights(quant, seed, rows, cols):
    return ops.synth_quantized(quant, seed, 0.02, rows, cols, torch.device("cuda:0"))


def _layer(quant, shared, T, router_std=0.02, E=E, k=TOP_K, tensors=None):
    g = torch.Generator(device="cuda").manual_seed(2)
    kw = {}
    if shared:
        kw = dict(shared_gate=_weights(Q8_0, 9, IS, H), shared_up=_weights(Q8_0, 10, IS, H),
                  shared_down=_weights(Q8_0, 11, H, IS))
    mats = dict(gate=_weights(quant, 0, E * I, H), up=_weights(quant, 1, E * I, H),
                down=_weights(quant, 2, E * H, I))
    layer = ops.MoELayer(
        hidden=H, experts=E, intermediate=I, top_k=k, quant=quant, down_quant=quant,
        score_fn=SCORE_SOFTMAX, norm_topk_prob=True, routed_scaling_factor=1.0,
        router=torch.randn(E, H, generator=g, device="cuda") * router_std, router_bias=None,
        shared_intermediate=IS if shared else 0, max_tokens=T, **(tensors or dict(mats, **kw)))
    return layer, mats, kw


def _exact(quant, mats, kw, x, ids, w):
    """The layer in 64 bits for the ids and weights that the layer chose."""
    deq = {n: ops.dequantize(quant, m).view(-1, *((H, I) if n == "down" else (I, H))).double()
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


def _sides(monkeypatch, layer, x):
    """The layer by the rule, on the decode launches, on the grouped GEMMs."""
    out = [layer.forward(x)]
    for side in ("0", "1"):
        monkeypatch.setenv("INFERNO_DECODE_GROUPED", side)
        out.append(layer.forward(x))
    monkeypatch.delenv("INFERNO_DECODE_GROUPED")
    return out


def _row_errors(monkeypatch, quant, shared, x, **kw):
    """Largest error of a token's row against fp64: decode, grouped."""
    T = x.shape[0]
    layer, mats, sh = _layer(quant, shared, T, **kw)
    ids = torch.empty(T * layer.top_k, dtype=torch.int32, device="cuda")
    w = torch.empty(T * layer.top_k, device="cuda")
    layer.forward(x, None, ids=ids, weights=w)
    ref = _exact(quant, mats, sh, x, ids.view(T, -1), w.view(T, -1))
    _, decode, grouped = _sides(monkeypatch, layer, x)
    assert not torch.equal(decode, grouped)  # two paths ran
    return [((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
            for y in (decode, grouped)]


# Grouped: f16 holds bf16 tokens and the integers of the weights, so that what
# is rounded is h, by at most 2^-11 of each value. Decode: the products of
# weights and scales too (the layers' own bound).
GROUPED, DECODE = 2.0 ** -11, 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 4, 6])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
@pytest.mark.parametrize("scale", [1e-3, 0.02, 1.0, 200.0])
def test_token_scale(quant, shared, T, scale, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = (torch.randn(T, H, generator=g, device="cuda") * scale).bfloat16()
    decode, grouped = _row_errors(monkeypatch, quant, shared, x, router_std=1e-4)
    assert grouped < GROUPED and decode < DECODE, (grouped, decode)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 6])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
def test_one_large_activation(quant, shared, T, monkeypatch):
    # 1e5 in one token (past f16's range); a router of 1e-6 hardly sees it
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, H, generator=g, device="cuda")
    x[T - 1, 5] = 1e5
    decode, grouped = _row_errors(monkeypatch, quant, shared, x.bfloat16(), router_std=1e-6)
    assert grouped < GROUPED and decode < DECODE, (grouped, decode)


@pytest.mark.gpu
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
def test_more_than_one_tile(quant, monkeypatch):
    # 40 tokens over two experts: tiles of 16 rows and a remainder of each
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(40, H, generator=g, device="cuda").bfloat16()
    decode, grouped = _row_errors(monkeypatch, quant, True, x, E=2, k=1)
    assert grouped < GROUPED and decode < DECODE, (grouped, decode)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 4, 6])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
def test_fp32_tokens_keep_their_bits(quant, shared, T, monkeypatch):
    # fp32 tokens enter the decode launches as two f16 terms (22 bits); one f16
    # term of the grouped GEMMs would hold 11, so the rule leaves them there
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, H, generator=g, device="cuda")
    layer, _, _ = _layer(quant, shared, T)
    by_rule, decode, forced = _sides(monkeypatch, layer, x)
    assert torch.equal(by_rule, decode) and torch.equal(forced, decode)


@pytest.mark.gpu
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant,T,hands_over", [
    (Q3_K, 3, False),  # 18 assignments
    (Q2_K, 6, False),  # 36 assignments of 110 MiB
    (Q3_K, 6, True),   # 145 MiB
    (Q4_K, 5, True)])  # 158 MiB
def test_rule(quant, T, hands_over, shared, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    layer, _, _ = _layer(quant, shared, T)
    by_rule, decode, grouped = _sides(monkeypatch, layer, x)
    assert not torch.equal(decode, grouped)
    assert torch.equal(by_rule, grouped if hands_over else decode)


@pytest.mark.gpu
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
@pytest.mark.parametrize("moved,shift", [("gate", 2), ("up", 4), ("down", 8), ("shared_gate", 2),
                                         ("shared_down", 8)])
def test_matrices_off_the_dma(quant, moved, shift, monkeypatch):
    # a matrix that the LDS DMA cannot take (routed: whole words, Q4_K 16 bytes;
    # shared: 16 bytes) keeps the layer on the decode launches, also when asked
    # for the GEMMs; one that it can take does not
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(6, H, generator=g, device="cuda").bfloat16()
    _, mats, sh = _layer(quant, True, 6)
    t = dict(mats, **sh)
    buf = torch.empty(t[moved].numel() + 16, dtype=torch.uint8, device="cuda")
    buf[shift:shift + t[moved].numel()] = t[moved]
    t[moved] = buf[shift:shift + t[moved].numel()]
    layer, _, _ = _layer(quant, True, 6, tensors=t)
    by_rule, decode, forced = _sides(monkeypatch, layer, x)
    taken = shift % 4 == 0 and quant != Q4_K and not moved.startswith("shared")
    assert torch.equal(forced, decode) == (not taken)
    assert torch.equal(by_rule, forced if quant == Q3_K or not taken else decode)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 5])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
@pytest.mark.parametrize("bf16", [False, True])
def test_vanishing_routing_weights(quant, shared, T, bf16):
    # router logits of a standard deviation of 60: softmax weights down to
    # 1e-38 and below, whose runs of h are subnormal or nearly so
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, H, generator=g, device="cuda")
    x = x.bfloat16() if bf16 else x
    layer, mats, sh = _layer(quant, shared, T, router_std=60 / H ** 0.5)
    ids = torch.empty(T * TOP_K, dtype=torch.int32, device="cuda")
    w = torch.empty(T * TOP_K, device="cuda")
    y = layer.forward(x, None, ids=ids, weights=w)
    assert 0 < float(w[w > 0].min()) < 1e-33  # such weights are there
    ref = _exact(quant, mats, sh, x, ids.view(T, TOP_K), w.view(T, TOP_K))
    assert float(((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max()) < DECODE


@pytest.mark.gpu
@pytest.mark.parametrize("shared", [False, True])
def test_replayed_graph(shared):
    # the launches of a captured layer read each replay's tokens
    g = torch.Generator(device="cuda").manual_seed(3)
    layer, _, _ = _layer(Q3_K, shared, 6)
    x = torch.randn(6, H, generator=g, device="cuda").bfloat16()
    out = torch.empty(6, H, device="cuda")
    layer.forward(x, out=out)  # the kernels' first launches are not captured
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer.forward(x, out=out)
    for _ in range(3):
        x.copy_((torch.randn(6, H, generator=g, device="cuda") * 50).bfloat16())
        graph.replay()
        got = out.clone()
        assert torch.equal(got, layer.forward(x))


@pytest.mark.gpu
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("T", [1, 5, 33, 130])
def test_router_logits_in_the_down_rows(T, bf16):
    # the narrowest down rows for the most experts: as many chunks of logits as
    # their region holds (one, two), ids and weights as the router alone gives
    from inferno_amd import SCORE_SIGMOID
    g = torch.Generator(device="cuda").manual_seed(3)
    for Hn, k in ((256, 1), (256, 2), (512, 1)):
        x = torch.randn(T, Hn, generator=g, device="cuda")
        x = x.bfloat16() if bf16 else x
        router = torch.randn(256, Hn, generator=g, device="cuda") * 0.05
        layer = ops.MoELayer(
            hidden=Hn, experts=256, intermediate=256, top_k=k, quant=Q4_K, down_quant=Q4_K,
            score_fn=SCORE_SIGMOID, norm_topk_prob=False, routed_scaling_factor=1.0, router=router,
            router_bias=None, gate=_weights(Q4_K, 0, 256 * 256, Hn), up=_weights(Q4_K, 1, 256 * 256, Hn),
            down=_weights(Q4_K, 2, 256 * Hn, 256), max_tokens=T)
        ids = torch.empty(T * k, dtype=torch.int32, device="cuda")
        w = torch.empty(T * k, device="cuda")
        layer.forward(x, None, ids=ids, weights=w)
        score = torch.sigmoid(x.double() @ router.double().T)
        top = score.topk(k, dim=1)
        # the chosen experts' own scores, and no better one left out (1e-6: ties)
        got = score.gather(1, ids.view(T, k).long())
        assert float((got - w.view(T, k)).abs().max()) < 1e-6
        assert float((top.values - got.sort(dim=1, descending=True).values).abs().max()) < 1e-6
