"""GPU parity of the whole per-layer path on the benchmark workloads.

c1 (fp32) is compared with the float64 oracle at 1e-5; the fp16 workloads are
compared at the north-star tolerance (max-abs <= 2e-3 against the fp32 oracle
on the attention context, and the LayerNorm output within one fp16 rounding
step of it).  c2 runs at full size here; c3/c4 run at full size through
size-independent properties (bit-exact pack round trips, rows of probabilities
summing to one, LayerNorm row statistics) plus an oracle comparison on a
subset of sequences, so the CPU side stays within seconds.
"""
import ctypes

import pytest
import torch

from gpu_util import BASE, announce, assert_stored_close, max_abs
from oracle import eager

pytestmark = pytest.mark.gpu


def _mods():
    from energonai_amd import layer, workloads
    return layer, workloads


def _run_and_compare(w, inp, acc_dtype, tol_ctx, tol_y, storage_dtype=None):
    layer, _ = _mods()
    dev = {k: (v.cuda() if isinstance(v, torch.Tensor) else v) for k, v in inp.items()}
    got = layer.padding_removal_layer(dev["hidden_padded"], dev["qkv_packed"], dev["lens"], w.heads, w.head_dim,
                                      dev["gamma"], dev["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                      dense_out=dev["dense_out"], keep=True)
    want = eager.layer_unpadded(inp["hidden_padded"], inp["qkv_packed"], inp["lens_list"], w.heads, w.head_dim,
                                inp["gamma"], inp["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                dense_out=inp["dense_out"], acc_dtype=acc_dtype, storage_dtype=storage_dtype)
    assert torch.equal(got["x"].cpu(), want["x"].to(w.dtype)), "depad must be bit-exact"
    assert torch.equal(got["qkv"].cpu(), want["qkv"].to(w.dtype)), "transpose_pad must be bit-exact"
    err_ctx = max_abs(got["ctx_packed"].cpu(), want["ctx_packed"])
    assert err_ctx <= tol_ctx, err_ctx
    if tol_y is None:       # 2e-3 (fp16) on top of half an ulp of the stored value
        assert_stored_close(got["y"].cpu(), want["y"], w.dtype, what="LayerNorm output")
    else:
        err_y = max_abs(got["y"].cpu(), want["y"])
        assert err_y <= tol_y, err_y
    return got, want


def test_layer_c1_fp32_full():
    _, wl = _mods()
    w = wl.BY_NAME["c1"]
    announce("layer c1")
    inp = wl.make_inputs(w)
    assert inp["total"] == 698
    _run_and_compare(w, inp, torch.float64, 1e-5, 2e-5)


def test_layer_c1_matches_padded_layer():
    """The unpadded path equals the ordinary padded layer on valid tokens (examples/bert/bert.py:100-126)."""
    layer, wl = _mods()
    w = wl.BY_NAME["c1"]
    announce("layer c1 vs padded")
    inp = wl.make_inputs(w)
    got = layer.padding_removal_layer(inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(),
                                      w.heads, w.head_dim, inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale,
                                      w.causal, w.left_padded).cpu()
    lens = inp["lens_list"]
    qkv_padded = torch.zeros(w.batch, w.seq, w.heads, 3 * w.head_dim)
    t = 0
    for b, n in enumerate(lens):
        qkv_padded[b, :n] = inp["qkv_packed"][0, t:t + n]
        t += n
    y_pad = eager.layer_padded(inp["hidden_padded"], qkv_padded, lens, w.heads, w.head_dim, inp["gamma"],
                               inp["beta"], 1e-5, w.scale, w.causal, acc_dtype=torch.float64)
    want = eager.depad(y_pad, w.batch, lens)
    assert max_abs(got, want) <= 2e-5


def test_layer_c2_fp16_full():
    _, wl = _mods()
    w = wl.BY_NAME["c2"]
    announce("layer c2")
    inp = wl.make_inputs(w)
    assert inp["total"] == 8538
    # Against the fp32 oracle that rounds scores / probabilities / context to fp16 where the API stores
    # them (the reference materialises the same fp16 tensors): 2e-3 on the context; 2e-3 plus half an fp16
    # ulp of the stored value on the LayerNorm output (|y| reaches ~5, where that rounding alone is 1.95e-3).
    _run_and_compare(w, inp, torch.float32, 2e-3, None, storage_dtype=torch.float16)


def test_layer_c2_unfused_path_misses_2e3_against_the_unrounded_oracle_by_the_fp16_score_rounding():
    """Against the oracle that rounds nothing in between, the three-kernel path cannot meet 2e-3: the score
    tensor it must materialise in fp16 (as the reference does) perturbs every score by up to half an fp16 ulp,
    d = half_ulp(max|score|), so every probability by a factor within exp(+-2 * scale * d) and the context by
    at most 2 * scale * d * max|v|.  The bound below is that worst case on top of the 2e-3; the fused kernel,
    which stores no scores, meets the plain 2e-3 (test_layer_c2_fused_attention)."""
    layer, wl = _mods()
    from gpu_util import half_ulp
    w = wl.BY_NAME["c2"]
    announce("layer c2 vs unrounded oracle")
    inp = wl.make_inputs(w)
    got = layer.padding_removal_layer(inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(),
                                      w.heads, w.head_dim, inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale,
                                      w.causal, w.left_padded, keep=True)
    want = eager.layer_unpadded(inp["hidden_padded"], inp["qkv_packed"], inp["lens_list"], w.heads, w.head_dim,
                                inp["gamma"], inp["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                acc_dtype=torch.float32)
    valid = torch.zeros_like(want["scores"], dtype=torch.bool)
    for b, n in enumerate(inp["lens_list"]):
        valid[b, :, :n, :n] = True
    d = float(half_ulp(want["scores"][valid].abs().max(), torch.float16))
    v_max = float(inp["qkv_packed"][..., 2 * w.head_dim:].abs().max())
    err = max_abs(got["ctx_packed"].cpu(), want["ctx_packed"])
    print(f"max|ctx err| vs unrounded oracle {err:.3e}; score rounding allows {2 * w.scale * d * v_max:.3e} more than 2e-3")
    assert err <= 2e-3 + 2 * w.scale * d * v_max


@pytest.mark.parametrize("name,total", [("c3", 9244), ("c4", 20142)])
def test_layer_large_fp16_properties(name, total):
    layer, wl = _mods()
    w = wl.BY_NAME[name]
    announce("layer", name)
    inp = wl.make_inputs(w)
    assert inp["total"] == total
    from energonai_amd import kernel as k
    lens_l = inp["lens_list"]
    lens_g = inp["lens"].cuda()
    hp = inp["hidden_padded"].cuda()
    qkvp = inp["qkv_packed"].cuda()
    got = layer.padding_removal_layer(hp, qkvp, lens_g, w.heads, w.head_dim, inp["gamma"].cuda(), inp["beta"].cuda(),
                                      1e-5, w.scale, w.causal, w.left_padded,
                                      dense_out=None if inp["dense_out"] is None else inp["dense_out"].cuda(),
                                      keep=True)
    T, B, S, H, D = total, w.batch, w.seq, w.heads, w.head_dim
    # pack round trips at full size, bit-exact
    assert torch.equal(got["x"].cpu(), eager.depad(inp["hidden_padded"], B, lens_l, left_padded=w.left_padded))
    back = k.transpose_depad(got["qkv"], B, T, S, lens_g, H, 3 * D)
    assert torch.equal(back, qkvp)
    # padding of the padded tensor is zero
    for b in (0, B - 1):
        assert bool((got["qkv"][b, :, lens_l[b]:, :] == 0).all())
    # probabilities: valid rows sum to one, nothing above the diagonal
    probs = got["probs"]
    for b in (0, B // 2, B - 1):
        n = lens_l[b]
        sums = probs[b, :, :n].float().sum(-1)
        assert float((sums - 1).abs().max()) < 5e-3
        assert float(probs[b, :, :n].float().triu(1).abs().max()) == 0.0
    # LayerNorm: rows of (y - beta) / gamma have zero mean and unit variance
    y = got["y"].float()[0]
    z = (y - inp["beta"].cuda().float()) / inp["gamma"].cuda().float()
    assert float(z.mean(-1).abs().max()) < 2e-3
    assert float((z.var(-1, unbiased=False) - 1).abs().max()) < 5e-3
    # oracle on the two shortest sequences (keeps the CPU side small)
    order = sorted(range(B), key=lambda b: lens_l[b])[:2]
    cu = [0]
    for n in lens_l:
        cu.append(cu[-1] + n)
    for b in order:
        n = lens_l[b]
        sl = slice(cu[b], cu[b] + n)
        sub_qkv = inp["qkv_packed"][:, sl]
        sub_hidden = inp["hidden_padded"][b:b + 1]
        sub_dense = None if inp["dense_out"] is None else inp["dense_out"][:, sl]
        want = eager.layer_unpadded(sub_hidden, sub_qkv, [n], H, D, inp["gamma"], inp["beta"], 1e-5, w.scale,
                                    w.causal, w.left_padded, dense_out=sub_dense, acc_dtype=torch.float32,
                                    storage_dtype=torch.float16)
        assert_stored_close(got["ctx_packed"][0, sl].cpu(), want["ctx_packed"][0], w.dtype, what="context")
        assert_stored_close(got["y"][0, sl].cpu(), want["y"][0], w.dtype, what="LayerNorm output")


@pytest.mark.parametrize("name,total", [("c3", 9244), ("c4", 20142)])
def test_layer_large_fp16_one_call_path_against_the_oracle(name, total):
    """The forms the benchmark times, through the one-call entry point at full size: the default form (fused
    attention on the packed projections, depad folded into the LayerNorm) and the three-kernel forms (scores in the
    packed causal layout or in [B,H,S,S]; padding rows never written, no softmax tail).  Context and output of the
    longest, the median and the shortest sequence against the oracle run on that sequence alone (attention and
    LayerNorm are independent per sequence), and bit-equality of the three-kernel forms with the op-by-op
    sequence of public calls and with the reference's own sequence of ops.

    Bounds: 2e-3 on top of half an fp16 ulp of the stored value.  The three-kernel forms are held against the
    float32 oracle that rounds scores and probabilities to fp16 where the API stores them (the reference
    materialises the same fp16 tensors, examples/gpt/gpt.py:108-125); the fused kernel never stores them and is
    held against the oracle that rounds nothing in between."""
    layer, wl = _mods()
    w = wl.BY_NAME[name]
    announce("layer one-call", name)
    inp = wl.make_inputs(w)
    assert inp["total"] == total
    T, B, H, D = total, w.batch, w.heads, w.head_dim
    lens_l = inp["lens_list"]
    dense = None if inp["dense_out"] is None else inp["dense_out"].cuda()
    args = (inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(), H, D, inp["gamma"].cuda(),
            inp["beta"].cuda(), 1e-5, w.scale, w.causal, w.left_padded)
    # the default form: fused attention on the packed projections, depad folded into the LayerNorm
    assert layer.default_attention_form(w.causal, w.dtype, w.seq, D, w.scale) == "packed"
    ctx = torch.full((1, T, H, D), float("nan"), dtype=w.dtype, device="cuda")
    y = layer.padding_removal_layer(*args, dense_out=dense, sum_seq=T, ctx_out=ctx)
    # the three kernels on packed operands, scores in the packed causal layout
    assert layer.three_kernel_form(w.causal, w.dtype, w.seq) == "varlen_packed"
    ctx_p = torch.full((1, T, H, D), float("nan"), dtype=w.dtype, device="cuda")
    y_p = layer.padding_removal_layer(*args, dense_out=dense, sum_seq=T, ctx_out=ctx_p, fused_attention="varlen_packed")
    # the same with [B,H,S,S] scores, in one call and op by op through the public functions
    ctx_v = torch.full((1, T, H, D), float("nan"), dtype=w.dtype, device="cuda")
    y_v = layer.padding_removal_layer(*args, dense_out=dense, sum_seq=T, ctx_out=ctx_v, fused_attention="varlen")
    steps = layer.padding_removal_layer(*args, dense_out=dense, sum_seq=T, keep=True, fused_attention="varlen")
    assert torch.equal(y_v, steps["y"]) and torch.equal(ctx_v, steps["ctx_packed"])
    # the reference's sequence of ops (transpose_pad ... transpose_depad on padded tensors): the same bits
    ref = layer.padding_removal_layer(*args, dense_out=dense, sum_seq=T, keep=True, fused_attention=False)
    assert torch.equal(y_v, ref["y"]) and torch.equal(ctx_v, ref["ctx_packed"])
    # packed causal scores: the same bits while the softmax gives a row the same lanes in both layouts
    if w.seq <= 1024:
        assert torch.equal(y_p, y_v) and torch.equal(ctx_p, ctx_v)
    routes = [("default form (fused attention)", y.cpu(), ctx.cpu(), None),
              ("three kernels, packed scores", y_p.cpu(), ctx_p.cpu(), torch.float16),
              ("three kernels, [B,H,S,S] scores", y_v.cpu(), ctx_v.cpu(), torch.float16)]
    del steps, ref, y_v, ctx_v, y_p, ctx_p
    order = sorted(range(B), key=lambda b: lens_l[b])
    cu = [0]
    for n in lens_l:
        cu.append(cu[-1] + n)
    for b in (order[-1], order[B // 2], order[0]):
        n = lens_l[b]
        announce("  sequence", b, "length", n)
        sl = slice(cu[b], cu[b] + n)
        sub_dense = None if inp["dense_out"] is None else inp["dense_out"][:, sl]
        # the fused kernel keeps scores and probabilities in fp32 registers: its oracle rounds nothing in between
        wants = {st: eager.layer_unpadded(inp["hidden_padded"][b:b + 1], inp["qkv_packed"][:, sl], [n], H, D,
                                          inp["gamma"], inp["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                          dense_out=sub_dense, acc_dtype=torch.float32, storage_dtype=st)
                 for st in (None, torch.float16)}
        for route, y_r, ctx_r, st in routes:
            want = wants[st]
            # the LayerNorm passes the error of its input on, scaled by gamma * invvar, and rounds once more
            amp = max(1.0, float(want["invvar"].max()) * float(inp["gamma"].float().abs().max())) if dense is None else 0.0
            assert_stored_close(ctx_r[0, sl].reshape(n, H * D), want["ctx_packed"].reshape(n, H * D), w.dtype,
                                what=f"context, {route}")
            assert_stored_close(y_r[0, sl], want["y"][0], w.dtype, base=BASE[w.dtype] * max(amp, 1.0),
                                what=f"LayerNorm output, {route}")


def test_decode_layer_c5_reduced_and_full():
    layer, wl = _mods()
    w = wl.BY_NAME["c5"]
    announce("layer c5")
    lens = wl.make_lens(w)
    assert int(lens.sum()) == 70929
    # full-size run: caches drawn on the device, oracle on a subset of sequences
    inp = wl.make_decode_inputs(w, device="cuda", cache_on_device=True)
    got = layer.decode_layer(inp["q"], inp["k_cache"], inp["v_cache"], inp["lens"].cuda(), inp["residual"],
                             inp["gamma"], inp["beta"], 1e-5, w.scale, dense_out=inp["dense_out"], keep=True)
    lens_l = inp["lens_list"]
    pick = sorted(range(w.batch), key=lambda b: lens_l[b])
    pick = [pick[0], pick[len(pick) // 2], pick[-1]]
    for b in pick:
        _, probs, ctx = eager.decode_attention(inp["q"][b:b + 1].cpu(), inp["k_cache"][b:b + 1].cpu(),
                                               inp["v_cache"][b:b + 1].cpu(), [lens_l[b]], w.scale)
        assert max_abs(got["ctx"][b:b + 1].cpu(), ctx) <= 2e-3
        assert max_abs(got["scores_probs"][b:b + 1].cpu(), probs) <= 2e-3
    want_y, _, _, _ = eager.layer_norm(inp["dense_out"].cpu(), inp["gamma"].cpu(), inp["beta"].cpu(), 1e-5,
                                       residual=inp["residual"].cpu(), out_dtype=torch.float32)
    assert_stored_close(got["y"].cpu(), want_y, w.dtype, what="LayerNorm output")
    # the attention output feeds the residual directly when no dense output is given
    got2 = layer.decode_layer(inp["q"], inp["k_cache"], inp["v_cache"], inp["lens"].cuda(), inp["residual"],
                              inp["gamma"], inp["beta"], 1e-5, w.scale, keep=True)
    want2, _, _, _ = eager.layer_norm(got2["ctx_packed"].reshape(1, w.batch, -1).cpu(), inp["gamma"].cpu(),
                                      inp["beta"].cpu(), 1e-5, residual=inp["residual"].cpu(),
                                      out_dtype=torch.float32)
    assert_stored_close(got2["y"].cpu(), want2, w.dtype, what="LayerNorm output")
    # the default form of the step: one pass over the caches, then the LayerNorm.  The context against the oracle
    # on nine sequences (the shortest, the longest, and seven spread between them) at the stated bound.
    got3 = layer.decode_layer(inp["q"], inp["k_cache"], inp["v_cache"], inp["lens"].cuda(), inp["residual"],
                              inp["gamma"], inp["beta"], 1e-5, w.scale, single_pass=True, keep=True)
    by_len = sorted(range(w.batch), key=lambda b: lens_l[b])
    assert lens_l[by_len[0]] == 3 and lens_l[by_len[-1]] == 1989
    for b in [by_len[i * (w.batch - 1) // 8] for i in range(9)]:
        _, _, ctx = eager.decode_attention(inp["q"][b:b + 1].cpu(), inp["k_cache"][b:b + 1].cpu(),
                                           inp["v_cache"][b:b + 1].cpu(), [lens_l[b]], w.scale)
        assert_stored_close(got3["ctx"][b:b + 1].cpu(), ctx, w.dtype, what=f"single-pass context, sequence {b}")
    want3, _, _, _ = eager.layer_norm(got3["ctx_packed"].reshape(1, w.batch, -1).cpu(), inp["gamma"].cpu(),
                                      inp["beta"].cpu(), 1e-5, residual=inp["residual"].cpu(),
                                      out_dtype=torch.float32)
    assert_stored_close(got3["y"].cpu(), want3, w.dtype, what="LayerNorm output")
    y_default = layer.decode_layer(inp["q"], inp["k_cache"], inp["v_cache"], inp["lens"].cuda(), inp["residual"],
                                   inp["gamma"], inp["beta"], 1e-5, w.scale)
    assert torch.equal(y_default, got3["y"])


@pytest.mark.parametrize("mode", [True, "packed"])
def test_layer_c2_fused_attention(mode):
    """The optional fused-attention form of the step: no fp16 score tensor, so it meets the
    north-star tolerance against the oracle that rounds nothing but the stored context."""
    layer, wl = _mods()
    w = wl.BY_NAME["c2"]
    announce("layer c2 fused")
    inp = wl.make_inputs(w)
    got = layer.padding_removal_layer(inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(),
                                      w.heads, w.head_dim, inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale,
                                      w.causal, w.left_padded, keep=True, fused_attention=mode)
    want = eager.layer_unpadded(inp["hidden_padded"], inp["qkv_packed"], inp["lens_list"], w.heads, w.head_dim,
                                inp["gamma"], inp["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                acc_dtype=torch.float32)
    assert max_abs(got["ctx_packed"].cpu(), want["ctx_packed"]) <= 2e-3
    assert_stored_close(got["y"].cpu(), want["y"], w.dtype, what="LayerNorm output")


@pytest.mark.parametrize("name,form", [("c1", False), ("c1", "varlen"), ("c2", False), ("c2", True), ("c2", "packed"),
                                       ("c2", "varlen"), ("c2", "varlen_packed")])
def test_layer_single_call_equals_the_op_by_op_sequence(name, form):
    """padding_removal_layer without keep= goes through the one-call entry point of the library; it must give
    bit for bit what the same ops give when called one by one."""
    layer, wl = _mods()
    w = wl.BY_NAME[name]
    announce("layer one call", name, form)
    inp = wl.make_inputs(w)
    args = (inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(), w.heads, w.head_dim,
            inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale, w.causal, w.left_padded)
    dense = inp.get("dense_out")
    dense = None if dense is None else dense.cuda()
    steps = layer.padding_removal_layer(*args, dense_out=dense, keep=True, fused_attention=form)
    once = layer.padding_removal_layer(*args, dense_out=dense, fused_attention=form)
    assert torch.equal(once, steps["y"])
    twice = layer.padding_removal_layer(*args, dense_out=dense, fused_attention=form, sum_seq=int(inp["lens"].sum()))
    assert torch.equal(twice, once)
    if form in ("varlen", "varlen_packed"):
        # the contractions on packed tokens compute what the reference's sequence of ops computes, bit for bit
        ref = layer.padding_removal_layer(*args, dense_out=dense, keep=True, fused_attention=False)
        assert torch.equal(once, ref["y"]) and torch.equal(steps["ctx_packed"], ref["ctx_packed"])


@pytest.mark.parametrize("name,want_form", [("c1", "packed"), ("c2", "packed")])
def test_layer_default_form(name, want_form):
    """With no form named the step runs the fused kernel on the packed projections where it applies (16-bit
    storage; fp32), else the three kernels on packed operands; depad is folded
    into the LayerNorm either way."""
    layer, wl = _mods()
    w = wl.BY_NAME[name]
    announce("layer default form", name)
    assert layer.default_attention_form(w.causal, w.dtype, w.seq, w.head_dim, w.scale) == want_form
    inp = wl.make_inputs(w)
    args = (inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(), w.heads, w.head_dim,
            inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale, w.causal, w.left_padded)
    dense = inp.get("dense_out")
    dense = None if dense is None else dense.cuda()
    default = layer.padding_removal_layer(*args, dense_out=dense)
    named = layer.padding_removal_layer(*args, dense_out=dense, fused_attention=want_form, fold_depad=True)
    assert torch.equal(default, named)
    # fp32 heads of 65..128 channels have a kernel of their own; what neither takes goes to the three kernels on packed operands
    assert layer.default_attention_form(False, torch.float32, 128, 128, 0.1) == "packed_f32_wide"
    assert layer.default_attention_form(False, torch.float32, 128, 70, 0.1) == "varlen"
    assert layer.default_attention_form(True, torch.float32, 128, 64, 0.1) == "packed"
    # and the default form meets the bound against the oracle that rounds nothing in between
    want = eager.layer_unpadded(inp["hidden_padded"], inp["qkv_packed"], inp["lens_list"], w.heads, w.head_dim,
                                inp["gamma"], inp["beta"], 1e-5, w.scale, w.causal, w.left_padded,
                                dense_out=inp.get("dense_out"))
    assert_stored_close(default.cpu(), want["y"], w.dtype,
                        base=BASE[w.dtype] * (max(1.0, float(want["y"].abs().max())) if w.dtype == torch.float32 else 1.0),
                        what="LayerNorm output of the default form")


@pytest.mark.parametrize("name,form", [("c1", False), ("c2", False), ("c2", "packed"), ("c2", "varlen_packed")])
def test_layer_with_depad_folded_into_layernorm(name, form):
    """fold_depad: no depad launch, the LayerNorm reads its residual rows from the padded activations through
    per-token row offsets (right-padded c1, left-padded c2).  Same bits as the step with the depad copy."""
    layer, wl = _mods()
    w = wl.BY_NAME[name]
    announce("layer fold depad", name, form)
    inp = wl.make_inputs(w)
    args = (inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda(), inp["lens"].cuda(), w.heads, w.head_dim,
            inp["gamma"].cuda(), inp["beta"].cuda(), 1e-5, w.scale, w.causal, w.left_padded)
    dense = inp.get("dense_out")
    dense = None if dense is None else dense.cuda()
    plain = layer.padding_removal_layer(*args, dense_out=dense, fused_attention=form, fold_depad=False)
    folded = layer.padding_removal_layer(*args, dense_out=dense, fused_attention=form, fold_depad=True)
    assert torch.equal(folded, plain)


@pytest.mark.parametrize("name,form", [("c1", False), ("c2", False), ("c2", "packed"), ("c1", None), ("c2", None)])
def test_layer_recorded_into_a_hip_graph_replays_the_eager_result(name, form):
    """The step allocates through torch only and never synchronises, so a caller may record it into a HIP graph.
    Each of three replays, with eager launches and synchronisations between them, must give the eager bits, and
    new input written into the recorded buffers must be picked up."""
    layer, wl = _mods()
    from energonai_amd.seqinfo import seq_info
    w = wl.BY_NAME[name]
    announce("layer graph replay", name, form)
    inp = wl.make_inputs(w)
    dev = torch.device("cuda", 0)
    hidden, qkv = inp["hidden_padded"].cuda(), inp["qkv_packed"].cuda()
    gamma, beta = inp["gamma"].cuda(), inp["beta"].cuda()
    dense = inp.get("dense_out")
    dense = None if dense is None else dense.cuda()
    info = seq_info(inp["lens"], w.batch, dev)       # lengths reach the device before the recording starts

    def step():
        return layer.padding_removal_layer(hidden, qkv, info, w.heads, w.head_dim, gamma, beta, 1e-5, w.scale,
                                           w.causal, w.left_padded, dense_out=dense, sum_seq=inp["total"],
                                           fused_attention=form)
    eager_y = step().clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = step()
    torch.cuda.synchronize()
    for i in range(3):
        y.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager_y), f"replay {i}"
        assert torch.equal(step(), eager_y)          # eager work between the replays
        torch.cuda.synchronize()
    hidden.mul_(0.5)
    qkv.mul_(-1)
    eager_y2 = step().clone()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, eager_y2)
    assert not torch.equal(eager_y2, eager_y)


@pytest.mark.parametrize("left", [True, False])
def test_padding_offsets_against_closed_form(left):
    from energonai_amd.seqinfo import seq_info
    lens = [5, 0, 9, 1, 9]
    B, S = len(lens), 9
    announce("padding offsets", left)
    info = seq_info(torch.tensor(lens, dtype=torch.int32).cuda(), B, torch.device("cuda"))
    got = info.row_offsets(S, left).cpu().tolist()
    want = []
    for b, n in enumerate(lens):
        for i in range(n):
            row = b * S + (S - n if left else 0) + i
            want.append(row - len(want))
    assert got[:len(want)] == want


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,S,D", [
    (1, 2, 1100, 64),       # 32 vectors of four channels on 1024 lanes
    (3, 32, 1024, 128),     # exactly one vector per lane
    (2, 33, 1030, 128),     # a second vector for some lanes
    (5, 72, 2048, 128),     # 2.25 vectors
    (1, 128, 1500, 128),    # four, the most the one-pass form takes
    (1, 130, 1024, 128),    # wider: combine and LayerNorm as two launches
    (2, 4, 300, 80),        # nothing is shared
])
def test_decode_layer_one_native_call(dtype, B, H, S, D):
    """Decode step through ``en_decode_layer`` where the shares of a unit are combined inside the LayerNorm and where they
    are not, against the float64 oracle; the LayerNorm bound is BASE plus half an ulp of the stored value."""
    from energonai_amd import layer
    announce("decode layer native", dtype, B, H, S, D)
    g = torch.Generator().manual_seed(S + H)
    kv = [S, 1, 513, 700, 64][:B] if B > 1 else [S - 3]
    kv = [min(n, S) for n in kv]
    q = torch.randn(B, H, 1, D, generator=g).to(dtype)
    kc, vc = (torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(2))
    res = torch.randn(1, B, H * D, generator=g).to(dtype)
    gamma, beta = (1 + 0.02 * torch.randn(H * D, generator=g)).to(dtype), (0.02 * torch.randn(H * D, generator=g)).to(dtype)
    _, _, ctx = eager.decode_attention(q, kc, vc, kv, D ** -0.5, acc_dtype=torch.float64)
    want = torch.nn.functional.layer_norm(ctx.view(1, B, H * D) + res.double(), (H * D,), gamma.double(), beta.double(), 1e-5)
    got = layer.decode_layer(q.cuda(), kc.cuda(), vc.cuda(), torch.tensor(kv, dtype=torch.int32).cuda(), res.cuda(), gamma.cuda(),
                             beta.cuda(), 1e-5)
    assert got.shape == want.shape
    assert_stored_close(got.cpu(), want, dtype)
    # a projection in between: its output takes the context's place
    dense = torch.randn(1, B, H * D, generator=g).to(dtype)
    got = layer.decode_layer(q.cuda(), kc.cuda(), vc.cuda(), torch.tensor(kv, dtype=torch.int32).cuda(), res.cuda(), gamma.cuda(),
                             beta.cuda(), 1e-5, dense_out=dense.cuda())
    want = torch.nn.functional.layer_norm(dense.double() + res.double(), (H * D,), gamma.double(), beta.double(), 1e-5)
    assert_stored_close(got.cpu(), want, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,S,D", [
    (1, 1, 40, 64),         # one workgroup is the last one
    (3, 5, 300, 80),        # lanes past the head size
    (16, 20, 100, 64),      # one key a lane group and step; sequences ranked
    (15, 32, 250, 128),     # 4096 channels, as many as 256 lanes take (fp32: more than that)
    (2, 33, 250, 128),      # one head more
    (5, 8, 700, 96),        # four keys a lane group
    (2, 16, 1100, 128),     # two shares, fewer workgroups than CUs: 512 lanes, 2048 channels, as many as they take
    (2, 17, 1100, 128),     # one head more
    (30, 16, 1500, 64),     # two shares of 480 units: 256 lanes, 1024 channels
    (3, 10, 5000, 64),      # nine shares, more than are sent for at once
])
def test_decode_layer_in_one_launch(dtype, B, H, S, D):
    """``en_decode_layer_norm`` against the float64 oracle, empty sequences among them; the same bits again and again, and the words
    back at zero.  The bound is that of ``test_decode_layer_one_native_call``."""
    from energonai_amd import _lib
    announce("decode layer, one launch", dtype, B, H, S, D)
    g = torch.Generator().manual_seed(S + H)
    kv = ([S, 0, 1, 513, 700, 64, 65] * 5)[:B] if B > 1 else [S - 3]
    kv = [min(n, S) for n in kv]
    q = torch.randn(B, H, 1, D, generator=g).to(dtype)
    kc, vc = (torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(2))
    res = torch.randn(1, B, H * D, generator=g).to(dtype)
    gamma, beta = (1 + 0.02 * torch.randn(H * D, generator=g)).to(dtype), (0.02 * torch.randn(H * D, generator=g)).to(dtype)
    args = [t.cuda() for t in (q, kc, vc, res, gamma, beta)]
    lens = torch.tensor(kv, dtype=torch.int32).cuda()
    words = torch.zeros(_lib.fn.en_decode_layer_norm_words(), dtype=torch.int32, device="cuda")
    need = _lib.fn.en_decode_attn_workspace_bytes(B, H, S, D)
    ws = torch.full((max(need, 16),), 0xff, dtype=torch.uint8, device="cuda")       # NaN wherever nothing is written
    strides = (ctypes.c_int64 * 3)(H * S * D, S * D, D)
    out = []
    for _ in range(3):
        ctx, y = torch.empty(B, H, 1, D, dtype=dtype, device="cuda"), torch.empty(1, B, H * D, dtype=dtype, device="cuda")
        rc = _lib.fn.en_decode_layer_norm(args[0].data_ptr(), args[1].data_ptr(), args[2].data_ptr(), ctx.data_ptr(), lens.data_ptr(), B, H,
                                          S, D, strides, strides, D ** -0.5, args[3].data_ptr(), args[4].data_ptr(), args[5].data_ptr(),
                                          y.data_ptr(), 1e-5, _lib.dtype_tag(q, "test"), ws.data_ptr(), need, words.data_ptr(),
                                          _lib.stream_of(args[0]))
        if H in (17, 33) or (dtype == torch.float32 and H == 32):
            assert rc == -5
            return
        assert rc == 0
        out.append(y)
    assert not words.any() and torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    _, _, ctx = eager.decode_attention(q, kc, vc, kv, D ** -0.5, acc_dtype=torch.float64)
    want = torch.nn.functional.layer_norm(ctx.view(1, B, H * D) + res.double(), (H * D,), gamma.double(), beta.double(), 1e-5)
    assert_stored_close(out[0].cpu(), want, dtype)
    # rows that the call's own output overlaps are for the two launches
    assert _lib.fn.en_decode_layer_norm(args[0].data_ptr(), args[1].data_ptr(), args[2].data_ptr(), out[0].data_ptr(), lens.data_ptr(), B, H, S,
                                        D, strides, strides, D ** -0.5, args[3].data_ptr(), args[4].data_ptr(), args[5].data_ptr(),
                                        out[0].data_ptr(), 1e-5, _lib.dtype_tag(q, "test"), ws.data_ptr(), need, words.data_ptr(),
                                        _lib.stream_of(args[0])) == -5


def test_decode_layer_is_spoilt_by_one_launch_only():
    """Lengths that change under a launch may leave its words off zero (here they are set so): no later step meets them."""
    from energonai_amd import _lib, layer
    from energonai_amd.seqinfo import SeqInfo
    announce("decode layer, words off zero")
    B, H, S, D = 3, 4, 300, 64
    g = torch.Generator(device="cuda").manual_seed(8)
    q, kc, vc = (torch.randn(B, H, n, D, generator=g, device="cuda").half() for n in (1, S, S))
    res, gamma, beta = (torch.randn(n, H * D, generator=g, device="cuda").half() for n in (B, 1, 1))
    lens = torch.tensor([300, 0, 17], dtype=torch.int32, device="cuda")
    a = (q, kc, vc, SeqInfo(lens, None, B, None, lens), res.view(1, B, H * D), gamma[0], beta[0])
    want = layer.decode_layer(*a)
    bad = torch.full((_lib.fn.en_decode_layer_norm_words(),), 1000, dtype=torch.int32, device="cuda")     # nobody would be the last

    def step():
        # outputs and scratch of the call are allocated where these were: what nobody writes is NaN
        del [torch.full((B * H * D,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(8)][:]
        return layer.decode_layer(*a)

    for _ in range(3):
        words = _lib.front.decode_words(kc)
        assert _lib.fn.en_copy_bytes(bad.data_ptr(), words, bad.numel() * 4, _lib.stream_of(kc)) == 0
        assert all(torch.equal(step(), want) for _ in range(70))


@pytest.mark.parametrize("H,S,D,turns", [(72, 2048, 128, 1), (4, 300, 64, 2)])
def test_only_a_decode_layer_of_one_launch_takes_words(H, S, D, turns):
    """A row too wide for one launch is known by its sizes, before words are looked up and a call is refused."""
    from energonai_amd import _lib, layer
    announce("decode layer, words", H, S, D)
    q, kc, vc = (torch.zeros(1, H, n, D, dtype=torch.float16, device="cuda") for n in (1, S, S))
    row, lens = torch.zeros(1, 1, H * D, dtype=torch.float16, device="cuda"), torch.tensor([S], dtype=torch.int32, device="cuda")
    first = _lib.front.decode_words(kc)
    layer.decode_layer(q, kc, vc, lens, row, row[0, 0], row[0, 0])
    size = 4 * _lib.fn.en_decode_layer_norm_words()
    assert (_lib.front.decode_words(kc) - first) % (64 * size) == turns * size


def test_decode_layer_words_belong_to_their_stream():
    """Steps of different operands that overlap on several streams, and one in a graph beside them, each give what a step alone gives.
    No two streams have words in common; a stream of somebody else's and a capture have none and take two launches."""
    from energonai_amd import _lib, layer
    from energonai_amd.seqinfo import SeqInfo
    announce("decode layer, words of a stream")
    B, H, S, D = 2, 12, 1500, 64
    g = torch.Generator(device="cuda").manual_seed(5)

    def operands(*kv):
        def rand(*shape):
            return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)
        lens = torch.tensor(kv, dtype=torch.int32, device="cuda")
        return (rand(B, H, 1, D), rand(B, H, S, D), rand(B, H, S, D), SeqInfo(lens, None, B, None, lens), rand(1, B, H * D), rand(H * D),
                rand(H * D))

    need = _lib.fn.en_decode_attn_workspace_bytes(B, H, S, D)
    zeros = torch.zeros(_lib.fn.en_decode_layer_norm_words(), dtype=torch.int32, device="cuda")
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    strides = (ctypes.c_int64 * 3)(H * S * D, S * D, D)

    def one_launch(a, ctx, y):
        return _lib.fn.en_decode_layer_norm(a[0].data_ptr(), a[1].data_ptr(), a[2].data_ptr(), ctx.data_ptr(), a[3].lens.data_ptr(), B, H, S, D,
                                            strides, strides, D ** -0.5, a[4].data_ptr(), a[5].data_ptr(), a[6].data_ptr(), y.data_ptr(), 1e-5,
                                            _lib.dtype_tag(a[0], "test"), ws.data_ptr(), need, zeros.data_ptr(), _lib.stream_of(a[0]))

    steps = [operands(*kv) for kv in ((1500, 700), (3, 1500), (1024, 1), (600, 0))]
    ctx, y = torch.empty(B, H, 1, D, dtype=torch.float16, device="cuda"), torch.empty(1, B, H * D, dtype=torch.float16, device="cuda")
    want = []
    for a in steps:
        want.append(layer.decode_layer(*a))
        assert one_launch(a, ctx, y) == 0 and torch.equal(y, want[-1])
    streams = [torch.cuda.default_stream()] + [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.ExternalStream(streams[1].cuda_stream)):
        assert _lib.front.decode_words(steps[0][1]) is None
        two_launches = layer.decode_layer(*steps[0])
    words = []
    for s in streams:
        with torch.cuda.stream(s):
            words.append({_lib.front.decode_words(steps[0][1]) for _ in range(128)})      # every set, whichever was next
    assert [len(w) for w in words] == [64] * 4 and len(set().union(*words)) == 256
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        refused = one_launch(steps[0], ctx, y)
        recorded = layer.decode_layer(*steps[0])
    assert refused == -5
    got = [[] for _ in streams]
    for _ in range(8):
        recorded.fill_(float("nan"))
        for s, a, out in zip(streams, steps, got):
            with torch.cuda.stream(s):
                torch.cuda._sleep(200_000)                       # all four are queued before the first runs
                for n in (need, B * H * D * 2, B * H * D * 2):   # scratch and outputs are allocated where these were
                    torch.full((n // 2,), float("nan"), dtype=torch.float16, device="cuda")
                for _ in range(3):
                    out.append(layer.decode_layer(*a))
        graph.replay()
        torch.cuda.synchronize()
        # bit for bit the two launches, which add up in another order
        assert torch.equal(recorded, two_launches)
    for w, out in zip(want, got):
        assert all(torch.equal(y, w) for y in out)


@pytest.mark.parametrize("lens,S,H,left", [([1], 17, 1, False), ([64, 0, 300, 7, 128, 129], 300, 5, True),
                                           ([5] * 1030, 40, 2, False)])
def test_layer_tables_in_one_launch(lens, S, H, left):
    """Row offsets and tile table built together are the ones that their own kernels build."""
    from energonai_amd.seqinfo import build_seq_info
    announce("layer tables", len(lens), S, H, left)
    t = torch.tensor(lens, dtype=torch.int32).cuda()
    for kv_bytes in (1 << 10, 1 << 30):
        both, one = build_seq_info(t, len(lens), total=sum(lens)), build_seq_info(t, len(lens), total=sum(lens))
        off, tab = both.layer_tables(S, left, H, kv_bytes)
        assert torch.equal(off[:sum(lens)], one.row_offsets(S, left)[:sum(lens)])
        assert torch.equal(tab, one.tile_table(H, S, kv_bytes))
        assert both.row_offsets(S, left) is off and both.tile_table(H, S, kv_bytes) is tab


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,S,H,D,causal,left", [
    ([1], 17, 1, 64, True, False),                          # one workgroup meets nobody
    ([41], 64, 12, 64, True, True),                         # fewer rows than waves
    ([127, 128, 129, 0, 65], 130, 4, 64, False, True),      # edges of the 128- and 64-row tiles, a sequence of no rows
    ([300, 7, 256], 300, 20, 80, True, False),              # four vectors per lane (16-bit), ragged first tiles
    ([200, 64, 63], 200, 16, 96, True, True),
    ([140, 1], 257, 48, 16, True, False),                   # the most shares a word has room for
    ([140, 30], 257, 49, 16, True, False),                  # one more: two launches
    ([130, 3], 140, 16, 128, False, False),
    ([128, 77], 128, 3, 64, False, True),                   # eleven rows a wave: rounds of three, the last one of two
    ([129, 300], 300, 9, 128, True, True),                  # three vectors a lane, four rows a wave: rounds of two
    ([100] * 200, 128, 16, 64, True, False),                # more than one round of workgroups: two launches
])
def test_attention_and_layernorm_in_one_launch(dtype, lens, S, H, D, causal, left):
    """The step in one launch against the same step in two, with workgroups that wait for each other and (``polls`` = 0)
    with none that does: the context is bit-identical; y differs by at most one rounding of the stored value (rows of more
    than 192 vectors are added up in another order, and where the compiler fuses the last multiply-add with the conversion
    one of two roundings is left out).  The meeting words return to zero."""
    from energonai_amd import _lib, layer
    from energonai_amd.seqinfo import build_seq_info
    announce("one launch", dtype, lens[:5], S, H, D, causal, left)
    if dtype == torch.float32 and D > 64:
        pytest.skip("the fp32 kernel with the LayerNorm in its launch takes heads of up to 64 channels")
    g = torch.Generator().manual_seed(S + H)
    B, T, hid, scale = len(lens), sum(lens), H * D, D ** -0.5
    hidden, qkv = torch.randn(B, S, hid, generator=g).to(dtype).cuda(), torch.randn(1, T, H, 3 * D, generator=g).to(dtype).cuda()
    gamma, beta = (1 + 0.1 * torch.randn(hid, generator=g)).to(dtype).cuda(), torch.randn(hid, generator=g).to(dtype).cuda()
    info = build_seq_info(torch.tensor(lens, dtype=torch.int32).cuda(), B, total=T)
    offs, table = info.layer_tables(S, left, H, 2 * S * D * hidden.element_size())
    words, f32 = info.arrivals(S), dtype == torch.float32
    assert words is not None and int(words.abs().max()) == 0
    want_ctx = torch.empty(1, T, H, D, dtype=dtype, device="cuda")
    want = _lib.front.layer(hidden, qkv, None, gamma, beta, want_ctx, info.cu_seqlens, info.lens, offs, None if f32 else table, H, D,
                            T, scale, 1e-5, causal, left, 2, None).float()
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -18}[dtype]

    def close(y):
        return bool(((y.float() - want).abs() <= ulp * want.abs().clamp_min(2.0 ** -6)).all())

    one_launch = H <= 48 and hid * hidden.element_size() <= 4096 and B < 200
    for polls in (64, 0, 0, 64):
        ctx, y = torch.full_like(want_ctx, 7.0), torch.full((1, T, hid), 7.0, dtype=dtype, device="cuda")
        rc = _lib.fn.en_attn_fused_norm(qkv.data_ptr(), ctx.data_ptr(), info.lens.data_ptr(), info.cu_seqlens.data_ptr(), B, H, S, D, T,
                                        scale, int(causal), _lib.dtype_tag(qkv, "test"), None if f32 else table.data_ptr(),
                                        hidden.data_ptr(), offs.data_ptr(), gamma.data_ptr(), beta.data_ptr(), y.data_ptr(), 1e-5,
                                        words.data_ptr(), polls, _lib.stream_of(qkv))
        if not one_launch:
            assert rc == -5, rc     # EN_ERR_UNSUPPORTED
            assert bool((y == 7.0).all())
            return
        assert rc == 0, rc
        torch.cuda.synchronize()
        assert torch.equal(ctx, want_ctx)
        assert close(y)
        assert int(words.abs().max()) == 0
    got = layer.padding_removal_layer(hidden, qkv, info, H, D, gamma, beta, 1e-5, scale, causal, left)
    assert close(got)
    with torch.cuda.stream(torch.cuda.Stream()):            # the words are the first stream's: two launches here
        assert info.arrivals(S) is None
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        again = layer.padding_removal_layer(hidden, qkv, info, H, D, gamma, beta, 1e-5, scale, causal, left)
        torch.cuda.current_stream().synchronize()
    assert torch.equal(again.float(), want)


@pytest.mark.parametrize("dtype,lens,S,H,D,hid", [
    (torch.float16, [256, 256, 256], 256, 3, 64, 8),               # every tile of the launch a real one; a vector a row
    (torch.bfloat16, [1], 17, 1, 64, 512),                         # fewer rows than a workgroup has waves
    (torch.float16, [130, 0, 7], 130, 5, 64, 520),                 # a wave per row, more than one vector a lane
    (torch.bfloat16, [127, 128, 129], 140, 4, 80, 1536),
    (torch.float16, [33, 65], 70, 9, 96, 1544),                    # a workgroup per row
    (torch.bfloat16, [512], 512, 2, 128, 4104),
    (torch.float16, [40, 3], 64, 8, 128, 8200),
    (torch.bfloat16, [21], 32, 2, 128, 12288),
    (torch.float16, [21], 32, 2, 128, 12296),                      # wider than a workgroup holds: two launches
    (torch.float16, [100] * 60, 1000, 4, 64, 768),                 # a bucket that is mostly empty
])
def test_layernorm_of_a_projection_beside_the_attention(dtype, lens, S, H, D, hid):
    """With ``dense_out`` the LayerNorm shares the attention's launch: the context is that of the attention alone bit for bit,
    y differs from the LayerNorm's own call by at most one rounding of the stored value (the order of a row's sums).  A context
    written over the projection is read by the LayerNorm as two launches do."""
    from energonai_amd import layer
    from energonai_amd.kernel import attn_fused_packed, depad, layer_norm_forward
    from energonai_amd.seqinfo import build_seq_info
    announce("beside", dtype, lens[:5], S, H, D, hid)
    g = torch.Generator().manual_seed(S + hid)
    B, T = len(lens), sum(lens)
    hidden, qkv = torch.randn(B, S, hid, generator=g).to(dtype).cuda(), torch.randn(1, T, H, 3 * D, generator=g).to(dtype).cuda()
    dense = torch.randn(1, T, hid, generator=g).to(dtype).cuda()
    gamma, beta = (1 + 0.1 * torch.randn(hid, generator=g)).to(dtype).cuda(), torch.randn(hid, generator=g).to(dtype).cuda()
    info = build_seq_info(torch.tensor(lens, dtype=torch.int32).cuda(), B, total=T)
    want_ctx = attn_fused_packed(qkv, B, S, info, H, D, scale=D ** -0.5)
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    for left in (False, True):
        x = depad(hidden, B, info, left_padded=left, sum_seq=T)
        want = layer_norm_forward(dense, gamma, beta, (hid,), 1e-5, residual=x).float()
        for fold in (True, False):
            ctx = torch.full_like(want_ctx, 7.0)
            y = layer.padding_removal_layer(hidden, qkv, info, H, D, gamma, beta, 1e-5, left_padded=left, dense_out=dense, ctx_out=ctx,
                                            fold_depad=fold)
            assert torch.equal(ctx, want_ctx)
            assert bool(((y.float() - want).abs() <= ulp * want.abs().clamp_min(2.0 ** -6)).all())
    if hid <= H * D:
        both = torch.zeros_like(want_ctx)
        y = layer.padding_removal_layer(hidden, qkv, info, H, D, gamma, beta, 1e-5, left_padded=True, ctx_out=both,
                                        dense_out=both.view(-1)[:T * hid].view(1, T, hid))
        want = layer_norm_forward(want_ctx.view(-1)[:T * hid].view(1, T, hid), gamma, beta, (hid,), 1e-5, residual=x)
        assert torch.equal(y, want)


def test_decode_layer_operands_outside_the_native_call():
    """A projection's output in fp32 behind fp16 caches, with more rows than new tokens, or no residual: the step takes them
    as the separate calls do."""
    from energonai_amd import kernel as K, layer
    announce("decode layer, other operands")
    g = torch.Generator().manual_seed(7)
    B, H, S, D = 2, 4, 40, 64
    q, kc, vc = (torch.randn(B, H, n, D, generator=g).half().cuda() for n in (1, S, S))
    lens = torch.tensor([S, 9], dtype=torch.int32).cuda()
    gamma, beta = torch.randn(H * D, generator=g).half().cuda(), torch.randn(H * D, generator=g).half().cuda()
    ctx = K.decode_attn(q, kc, vc, lens).view(1, B, H * D)
    assert torch.equal(layer.decode_layer(q, kc, vc, lens, None, gamma, beta), K.layer_norm_forward(ctx, gamma, beta, (H * D,)))
    for dense in (torch.randn(1, B, H * D, generator=g).cuda(), torch.randn(3, B, H * D, generator=g).half().cuda()):
        res = torch.randn(dense.shape, generator=g).to(dense.dtype).cuda()
        got = layer.decode_layer(q, kc, vc, lens, res, gamma, beta, dense_out=dense)
        assert torch.equal(got, K.layer_norm_forward(dense, gamma, beta, (H * D,), residual=res))
    with pytest.raises(RuntimeError, match="kv_lens must hold"):
        layer.decode_layer(q, kc.view(B * H, 1, S, D), vc.view(B * H, 1, S, D), lens, torch.zeros(1, B, H * D).half().cuda(), gamma, beta)


def test_layer_that_does_not_fit_raises_out_of_memory():
    """A step whose intermediates do not fit raises what torch's allocator raises, the error that callers shrink a batch on."""
    from energonai_amd import layer
    from energonai_amd.seqinfo import build_seq_info
    announce("layer out of memory")
    S, D = 1 << 20, 8                                       # scores of one head: 2 TiB
    hidden, gamma = torch.zeros(1, S, D, dtype=torch.float16, device="cuda"), torch.ones(D, dtype=torch.float16, device="cuda")
    info = build_seq_info(torch.tensor([1], dtype=torch.int32).cuda(), 1, total=1)
    with pytest.raises(torch.OutOfMemoryError):
        layer.padding_removal_layer(hidden, torch.zeros(1, 1, 1, 3 * D, dtype=torch.float16, device="cuda"), info, 1, D, gamma, gamma,
                                    fused_attention=False)
