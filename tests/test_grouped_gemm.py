"""The grouped GEMM's DMA kernels (inferno_amd/csrc/grouped_gemm.hpp): source
addresses of the weight copies (CPU, tests/weight_dma_check.hip replays the
kernel's own offsets), and on the GPU the tile edges (15, 16, 17, 32, 33, 63,
64, 65 rows of one expert beside experts of 0, 1 and 2 rows), odd and even
super-block counts, every format pair, and weights that the DMA cannot take."""
import os
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

from inferno_amd import Q2_K, Q3_K, Q4_K, Q6_K, ops

ROOT = Path(__file__).resolve().parent.parent
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_weight_dma_addresses(tmp_path):
    if not (Path(HIPCC).exists() or shutil.which(HIPCC)):
        pytest.skip("hipcc not found")
    exe = tmp_path / "dmacheck"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'inferno_amd' / 'csrc'}", str(ROOT / "tests" / "weight_dma_check.hip"),
                    "-o", str(exe)], check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.startswith("OK "), r.stdout[-2000:] + r.stderr


def _ids(rows, E):
    """One expert per assignment (k = 1): expert e takes rows[e] tokens, shuffled."""
    ids = np.concatenate([np.full(n, e) for e, n in enumerate(rows)]).astype(np.uint32)
    return np.random.default_rng(3).permutation(ids)


D_AT = {Q2_K: (84, 80, 82), Q3_K: (110, 108, None), Q4_K: (144, 0, 2)}  # block, d, dmin


def _spread_d(q, mat, seed):
    """The blocks' d (and dmin) times 2^-8 .. 2^1 each, one in six zero."""
    nbytes, *at = D_AT[q]
    b = mat.cpu().numpy().copy().reshape(-1, nbytes)
    rng = np.random.default_rng(seed)
    for o in at:
        if o is not None:
            d = b[:, o:o + 2].copy().view(np.float16)[:, 0]
            f = np.exp2(rng.integers(-8, 2, len(d))) * (rng.integers(0, 6, len(d)) > 0)
            b[:, o:o + 2] = (d * f).astype(np.float16)[:, None].view(np.uint8)
    return torch.from_numpy(b.reshape(-1)).to(mat.device)


def _run(quant, down, H, I, rows, bf16, shift=0, spread=False):
    dev = torch.device("cuda:0")
    E = len(rows)
    ids = _ids(rows, E)
    T = len(ids)
    mats = [ops.synth_quantized(q, 5 + i, 0.02, E * r, c, dev)
            for i, (q, r, c) in enumerate(((quant, I, H), (quant, I, H), (down, H, I)))]
    if spread:
        mats = [_spread_d(q, m, 20 + i) for i, (q, m) in enumerate(zip((quant, quant, down), mats))]
    placed = []
    for m in mats:  # the same bytes at an address that is `shift` past an aligned one
        buf = torch.empty(m.numel() + 16, dtype=torch.uint8, device=dev)
        buf[shift:shift + m.numel()] = m
        placed.append(buf[shift:shift + m.numel()])
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn(T, H, generator=g, device=dev)
    x = x.bfloat16() if bf16 else x
    w = torch.rand(T, generator=g, device=dev) + 0.5
    args = (quant, down, *placed, x, torch.from_numpy(ids.view(np.int32)).to(dev), w, 1, E, I)
    out = ops.gguf_moe(*args)
    again = ops.gguf_moe(*args)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    # fp64, expert by expert (the values' own tests compare dequantize with the oracle)
    deq = [ops.dequantize(q, m).view(E, r, c) for q, m, r, c in
           ((quant, mats[0], I, H), (quant, mats[1], I, H), (down, mats[2], H, I))]
    ref = torch.zeros(T, H, dtype=torch.float64, device=dev)
    for e in range(E):
        at = torch.from_numpy(np.nonzero(ids == e)[0]).to(dev)
        gg, uu = (x[at].double() @ d[e].double().T for d in deq[:2])
        ref[at] = (gg * torch.sigmoid(gg) * uu * w[at, None].double()) @ deq[2][e].double().T
    return float((out.double() - ref).norm() / ref.norm())


# h is rounded to f16 and so are fp32 tokens (2^-12 of a value each, at random);
# Q6_K weights too: 2e-3 is the bound of the layers' own tests
BOUND = 2e-3
PAIRS = [(Q2_K, Q2_K), (Q3_K, Q3_K), (Q4_K, Q4_K), (Q4_K, Q6_K), (Q2_K, Q3_K)]


# small layers take 16-row tiles only; these widths (with the rows of MORE, one
# expert's) the tiles of every size
WIDE = [(512, 3584), (768, 3840), (256, 3584)]
MORE = (650,)


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("H,I", WIDE + [(512, 512), (768, 256), (256, 768)])
@pytest.mark.parametrize("rows", [(15, 0, 16, 17), (32, 33, 1, 0), (63, 2, 64, 65)],
                         ids=["to16", "to32", "to64"])
def test_tile_edges(quant, down, H, I, rows):
    assert _run(quant, down, H, I, rows + MORE, bf16=True) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("H,I", WIDE)
def test_tile_edges_128(quant, down, H, I):
    # whole and partial tiles of 128 rows, one expert with two and a remainder
    assert _run(quant, down, H, I, (65, 127, 128, 129, 0, 275), bf16=True) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", [(Q2_K, Q2_K), (Q3_K, Q3_K), (Q4_K, Q4_K)])
@pytest.mark.parametrize("rows", [(128, 100, 0), (64, 32, 16)], ids=["to128", "to64"])
@pytest.mark.parametrize("I", [3584, 1024], ids=["wide", "narrow"])
def test_blocks_of_unlike_or_zero_scale(quant, down, rows, I):
    # running sums change their unit from block to block, and a block of d = 0
    # (or dmin = 0) has none
    assert _run(quant, down, 1280, I, rows + MORE, bf16=True, spread=True) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("rows", [(160, 0, 1), (31, 17, 200, 48)])
def test_small_layer_tiles(quant, down, rows):
    # many 16-row tiles of one expert, against the same rows of weights that
    # the 16-row rule (like the DMA) leaves to the general kernels
    a = _run(quant, down, 512, 512, rows, bf16=True)
    b = _run(quant, down, 512, 512, rows, bf16=True, shift=2)
    assert a < BOUND and b < BOUND and a <= 1.05 * b


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
def test_sixteen_row_tiles_only(quant, down):
    # 70 rows over 9 experts: the batch takes 16-row tiles only, the first
    # expert two of them
    assert _run(quant, down, 512, 512, (20, 16, 15, 8, 5, 3, 2, 1, 0), bf16=False) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("shift", [2, 4])
@pytest.mark.parametrize("H,I", [(512, 256), (768, 1280), (256, 768)])
def test_weights_at_any_address(quant, down, shift, H, I):
    # 2 bytes past a word (and 4 past 16 bytes for Q4_K): not the DMA's rows;
    # even and odd super-block counts, tiles of 32, 64 and 128 rows
    assert _run(quant, down, H, I, (18, 30, 4, 0), bf16=True, shift=shift) < BOUND
    assert _run(quant, down, H, I, (40, 150, 17, 77), bf16=True, shift=shift) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 16, 17, 33])
@pytest.mark.parametrize("H,Is", [(256, 24), (768, 200), (4608, 256)])
@pytest.mark.parametrize("bf16", [True, False])
def test_dense_q8_rows(T, H, Is, bf16):
    # row counts that do not fill a workgroup (8 gate / 8 up rows, 16 rows),
    # one to 18 K units over four to eight wavefronts, values over 24 binary
    # orders within a row; the products are fp32-accurate: 1e-5 against fp64
    dev = torch.device("cuda:0")
    from inferno_amd import Q8_0
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.randn(T, H, generator=g, device=dev)
    x = x * torch.exp2(-24 * torch.rand(T, H, generator=g, device=dev)) * 1e3
    x = x.bfloat16() if bf16 else x
    wg, wu = (ops.synth_quantized(Q8_0, s, 0.02, Is, H, dev) for s in (1, 2))
    h = ops.q8_0_gate_up_swiglu(wg, wu, x, Is)
    a = x.double() @ ops.dequantize(Q8_0, wg).view(Is, H).double().T
    b = x.double() @ ops.dequantize(Q8_0, wu).view(Is, H).double().T
    ref = a * torch.sigmoid(a) * b
    assert float((h - ref).norm() / ref.norm()) < 1e-5
    O, In = Is, H
    wd = ops.synth_quantized(Q8_0, 3, 0.02, O, In, dev)
    inp = torch.randn(T, In, generator=g, device=dev) * 1e-4
    ra = torch.randn(T, O, generator=g, device=dev) * 1e-5
    for rb in (None, ra * 0.5):
        out = ops.q8_0_matvec_add2(wd, inp, ra, rb, O)
        ref = ra.double() + (0 if rb is None else rb.double()) + \
            inp.double() @ ops.dequantize(Q8_0, wd).view(O, In).double().T
        assert float((out - ref).norm() / ref.norm()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 16, 40])
@pytest.mark.parametrize("bf16", [True, False])
def test_dense_q8_rows_beside_a_large_value(T, bf16):
    # one activation of 1e10 per row that meets weight blocks of d = 0: what it
    # takes from f16's range is its own 32 values', not the row's (1e-5 as above)
    dev = torch.device("cuda:0")
    from inferno_amd import Q8_0
    H, Is, at = 1024, 200, 330
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.randn(T, H, generator=g, device=dev)
    x[:, at] = 1e10
    x = x.bfloat16() if bf16 else x

    def weights(seed, rows):
        w = ops.synth_quantized(Q8_0, seed, 0.02, rows, H, dev).view(rows, H // 32, 34).clone()
        w[:, at // 32, :2] = 0
        return w.view(-1)

    wg, wu, wd = (weights(s, Is) for s in (1, 2, 3))
    a, b, c = (x.double() @ ops.dequantize(Q8_0, w).view(Is, H).double().T for w in (wg, wu, wd))
    ref = a * torch.sigmoid(a) * b
    h = ops.q8_0_gate_up_swiglu(wg, wu, x, Is)
    assert float((h - ref).norm() / ref.norm()) < 1e-5
    ra = torch.randn(T, Is, generator=g, device=dev)
    if not bf16:  # (the matvec takes fp32 rows)
        out = ops.q8_0_matvec_add2(wd, x, ra, None, Is)
        assert float((out - ra - c).norm() / c.norm()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 3, 4, 6])
@pytest.mark.parametrize("shared", [0, 1024])
@pytest.mark.parametrize("quant", [Q2_K, Q3_K, Q4_K])
def test_layer_decode_and_grouped_agree(quant, shared, T, monkeypatch):
    # the three paths of a few tokens: the fused decode launches (a threshold no
    # batch reaches; the rule keeps these there but for Q3_K and Q4_K of six
    # tokens), the grouped GEMMs over scaled rows and over plain ones (a
    # threshold of 1); outputs within the rounding of h to f16 (2^-12 each)
    from inferno_amd import Q8_0, SCORE_SOFTMAX
    dev = torch.device("cuda:0")
    H, E, I, k = 3072, 32, 1024, 6
    mats = [ops.synth_quantized(quant, i, 0.02, E * r, c, dev)
            for i, (r, c) in enumerate(((I, H), (I, H), (H, I)))]
    sh = [ops.synth_quantized(Q8_0, 9 + i, 0.02, r, c, dev)
          for i, (r, c) in enumerate(((1024, H), (1024, H), (H, 1024)))]
    g = torch.Generator(device=dev).manual_seed(2)
    layer = ops.MoELayer(
        hidden=H, experts=E, intermediate=I, top_k=k, quant=quant, down_quant=quant,
        score_fn=SCORE_SOFTMAX, norm_topk_prob=True, routed_scaling_factor=1.0,
        router=torch.randn(E, H, generator=g, device=dev) * 0.02, router_bias=None, gate=mats[0],
        up=mats[1], down=mats[2], shared_intermediate=shared, shared_gate=sh[0], shared_up=sh[1],
        shared_down=sh[2], max_tokens=T)
    x = torch.randn(T, H, generator=g, device=dev).bfloat16()
    by_rule = layer.forward(x)
    monkeypatch.setenv("INFERNO_DECODE_GROUPED", "1")
    scaled = layer.forward(x)
    monkeypatch.delenv("INFERNO_DECODE_GROUPED")
    monkeypatch.setenv("INFERNO_PREFILL_MIN_ASSIGNMENTS", "100000")
    decode = layer.forward(x)
    monkeypatch.setenv("INFERNO_PREFILL_MIN_ASSIGNMENTS", "1")
    grouped = layer.forward(x)
    assert torch.equal(by_rule, scaled if T == 6 and quant != Q2_K else decode)
    assert not torch.equal(scaled, decode) and not torch.equal(grouped, decode)
    assert float((scaled - decode).norm() / decode.norm()) < 2e-3
    assert float((grouped - decode).norm() / decode.norm()) < 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("T,H,Is", [(16, 512, 256), (65, 256, 768), (300, 1024, 2048),
                                    (1030, 1280, 1024), (2100, 1280, 1536),
                                    (2100, 1024, 4096)])
def test_dense_expert_tiles(quant, down, T, H, Is):
    # the layer's shared expert over token tiles of 16, 32, 64 and 128 rows
    # with remainders: what it adds to the same layer without it
    from inferno_amd import SCORE_SOFTMAX
    dev = torch.device("cuda:0")
    E, I, k = 8, 256, 2
    mats = [ops.synth_quantized(Q4_K, i, 0.02, E * r, c, dev)
            for i, (r, c) in enumerate(((I, H), (I, H), (H, I)))]
    sh = [ops.synth_quantized(q, 9 + i, 0.05, r, c, dev)
          for i, (q, r, c) in enumerate(((quant, Is, H), (quant, Is, H), (down, H, Is)))]
    g = torch.Generator(device=dev).manual_seed(2)
    router = torch.randn(E, H, generator=g, device=dev) * 0.02
    x = torch.randn(T, H, generator=g, device=dev).bfloat16()
    out = []
    for shared in (0, Is):
        kw = dict(shared_gate=sh[0], shared_up=sh[1], shared_down=sh[2], shared_quant=quant,
                  shared_down_quant=down) if shared else {}
        layer = ops.MoELayer(
            hidden=H, experts=E, intermediate=I, top_k=k, quant=Q4_K, down_quant=Q4_K,
            score_fn=SCORE_SOFTMAX, norm_topk_prob=True, routed_scaling_factor=1.0,
            router=router, router_bias=None, gate=mats[0], up=mats[1], down=mats[2],
            shared_intermediate=shared, max_tokens=T, **kw)
        out.append(layer.forward(x).double())
    a, b = (x.double() @ ops.dequantize(quant, sh[i]).view(Is, H).double().T for i in (0, 1))
    ref = (a * torch.sigmoid(a) * b) @ ops.dequantize(down, sh[2]).view(H, Is).double().T
    assert float((out[1] - out[0] - ref).norm() / ref.norm()) < BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("quant,down", PAIRS)
@pytest.mark.parametrize("shift", [0, 2])
def test_few_experts_take_all_rows(quant, down, shift):
    # at most ten rows per expert on average, but two experts hold nearly all:
    # 128-row tiles with remainders of 1 to 128 rows beside 16-row ones (64
    # experts of 3072 make more workgroups than the rule of small layers takes)
    rows = [0] * 64
    rows[3], rows[17], rows[40], rows[41], rows[63] = 321, 192, 65, 33, 1
    assert _run(quant, down, 512, 3072, tuple(rows), bf16=True, shift=shift) < BOUND
