"""GPU tests of the host side of the boundary: the stand-ins for the reference's compiled extension modules
called exactly as the reference's Python wrappers call them, and the per-batch offset cache under the
conditions of the reference worker (inference mode, lengths given as lists, more than one stream)."""
import pytest
import torch

from gpu_util import announce, max_abs, packed_randn
from oracle import eager

pytestmark = pytest.mark.gpu


def _ref_shape(ref_test_shape):
    r = ref_test_shape
    return r["batch"], r["seq"], r["heads"], r["head_dim"], r["lens"]


@pytest.mark.parametrize("lens_dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_transpose_pad_extension_stand_in(ref_test_shape, dtype, lens_dtype):
    """energonai_transpose_pad.*_wrapper with the argument pattern of
    energonai/kernel/cuda_native/transpose_pad.py:12-87 (contiguous inputs, positional arguments, 0-d tensor
    totals) on the shape of the reference's own kernel test."""
    import energonai_amd.ext.energonai_transpose_pad as ext
    B, S, H, D, lens = _ref_shape(ref_test_shape)
    T = sum(lens)
    announce("ext transpose_pad", dtype, lens_dtype)
    seq_len_list = torch.tensor(lens, dtype=lens_dtype).cuda()
    src = packed_randn(T, H * D, dtype, 3).reshape(1, T, H, D)
    # transpose_pad / transpose_depad
    dst = ext.transpose_pad_wrapper(src.cuda().contiguous(), B, S, seq_len_list, H, D)
    want = eager.transpose_pad(src, B, S, lens, H, D)
    assert dst.shape == (B, H, S, D) and torch.equal(dst.cpu(), want)
    back = ext.transpose_depad_wrapper(dst.contiguous(), B, T, S, seq_len_list, H, D)
    assert back.shape == (1, T, H, D) and torch.equal(back.cpu(), src)
    # the FasterTransformer family: build offsets -> remove -> rebuild; transpose_rebuild -> transpose_remove
    lens32 = torch.tensor(lens, dtype=torch.int32).cuda()
    valid_word_num = torch.zeros(1, dtype=torch.int32, device="cuda")
    tmp_mask_offset = torch.zeros(B * S, dtype=torch.int32, device="cuda")
    mask_offset = torch.zeros(B * S, dtype=torch.int32, device="cuda")
    ext.ft_build_padding_offsets_wrapper(lens32.contiguous(), B, S, valid_word_num, tmp_mask_offset)
    want_valid, want_off = eager.ft_build_padding_offsets(lens, B, S)
    assert int(valid_word_num[0].item()) == int(want_valid[0]) == T
    assert torch.equal(tmp_mask_offset[:T].cpu(), want_off[:T].to(torch.int32))
    hid = H * D
    padded = torch.zeros(B, S, hid, dtype=dtype)
    flat = src.reshape(T, hid)
    t = 0
    for b, n in enumerate(lens):
        padded[b, :n] = flat[t:t + n]
        t += n
    removed = ext.ft_remove_padding_wrapper(padded.cuda().contiguous(), tmp_mask_offset, mask_offset,
                                            valid_word_num[0].item(), hid)
    assert removed.shape == (1, T, hid) and torch.equal(removed.cpu().reshape(T, hid), flat)
    assert torch.equal(mask_offset[:T], tmp_mask_offset[:T])
    rebuilt = ext.ft_rebuild_padding_wrapper(removed.contiguous(), mask_offset, T, hid, B, S)
    assert torch.equal(rebuilt.cpu(), padded)
    q_buf = torch.zeros(B, H, S, D, dtype=dtype, device="cuda")
    k_buf, v_buf = torch.zeros_like(q_buf), torch.zeros_like(q_buf)
    Q = src.reshape(T, H, D).cuda().contiguous()
    ext.ft_transpose_rebuild_padding_wrapper(Q, (2 * Q).contiguous(), (3 * Q).contiguous(), q_buf, k_buf, v_buf, B, S,
                                             H, D, T, mask_offset)
    assert torch.equal(q_buf.cpu(), want) and torch.equal(k_buf.cpu(), 2 * want) and torch.equal(v_buf.cpu(), 3 * want)
    flat_back = ext.ft_transpose_remove_padding_wrapper(q_buf.contiguous(), T, B, S, H, D, mask_offset)
    assert flat_back.shape == (1, T, hid) and torch.equal(flat_back.cpu().reshape(T, hid), flat)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_scale_mask_extension_stand_in(ref_test_shape, dtype):
    """energonai_scale_mask.scale_mask_softmax_wrapper(batch, seq, heads, correlation, real_seq_len) as in
    energonai/kernel/cuda_native/scale_mask_softmax.py:10-13: in place, its input returned."""
    import energonai_amd.ext.energonai_scale_mask as ext
    B, S, H, _, lens = _ref_shape(ref_test_shape)
    announce("ext scale_mask", dtype)
    g = torch.Generator().manual_seed(4)
    src = (2.0 * torch.randn(B, H, S, S, generator=g)).to(dtype)
    x = src.cuda().contiguous()
    dst = ext.scale_mask_softmax_wrapper(B, S, H, x, torch.tensor(lens, dtype=torch.int32).cuda())
    assert dst.data_ptr() == x.data_ptr()
    want = eager.scale_mask_softmax(B, S, H, src.float(), lens, out_dtype=torch.float32)
    got = dst.cpu()
    for b, n in enumerate(lens):
        assert max_abs(got[b, :, :n].float(), want[b, :, :n]) <= (2e-3 if dtype == torch.float16 else 1e-5)
        assert torch.equal(got[b, :, n:], src[b, :, n:])


@pytest.mark.parametrize("in_dtype,out_dtype", [(torch.float32, torch.float32), (torch.float32, torch.float16),
                                                (torch.float16, torch.float16)])
def test_layer_norm_extension_stand_in(in_dtype, out_dtype):
    """energonai_layer_norm.forward_affine(input_, normalized_shape, weight_, bias_, eps) -> [output, mean,
    invvar] as FusedLayerNormAffineFunction.forward unpacks it (energonai/kernel/cuda_native/layer_norm.py:24-28;
    the reference casts the input to fp32 first, so (fp32 in, 16-bit gamma) is its mixed case)."""
    import energonai_amd.ext.energonai_layer_norm as ext
    n1, n2 = 96, 768
    announce("ext layer_norm", in_dtype, out_dtype)
    g = torch.Generator().manual_seed(5)
    x = (1.5 * torch.randn(4, n1 // 4, n2, generator=g) + 0.25).to(in_dtype)
    gamma = (1 + 0.02 * torch.randn(n2, generator=g)).to(out_dtype)
    beta = (0.02 * torch.randn(n2, generator=g)).to(out_dtype)
    output, mean, invvar = ext.forward_affine(x.cuda().contiguous(), torch.Size([n2]), gamma.cuda().contiguous(),
                                              beta.cuda().contiguous(), 1e-5)
    want, want_mean, want_invvar, _ = eager.layer_norm(x, gamma, beta, 1e-5, acc_dtype=torch.float64,
                                                       out_dtype=torch.float64)
    assert output.shape == x.shape and output.dtype == out_dtype
    assert mean.dtype == torch.float32 and mean.shape == (n1,) and invvar.shape == (n1,)
    bound = 1e-5 if out_dtype == torch.float32 else 2e-3 + float(want.abs().max()) * 2.0 ** -11
    assert max_abs(output.cpu(), want) <= bound
    assert max_abs(mean.cpu(), want_mean.reshape(-1)) <= 1e-5
    assert float(((invvar.cpu().double() - want_invvar.reshape(-1).double()).abs() / want_invvar.reshape(-1).double()).max()) <= 1e-5
    with pytest.raises(RuntimeError, match="inference-only"):
        ext.backward_affine()


def test_extension_names_resolve_to_the_stand_ins_after_install():
    import importlib
    import sys
    from energonai_amd import ext
    announce("ext install")
    names = ("energonai_transpose_pad", "energonai_scale_mask", "energonai_layer_norm", "energonai_linear_func")
    saved = {n: sys.modules.pop(n, None) for n in names}
    try:
        ext.install()
        # the lookup the reference wrappers perform (cuda_native/transpose_pad.py:4-7)
        mod = importlib.import_module("energonai_transpose_pad")
        x = torch.arange(2 * 3 * 4, dtype=torch.float32).reshape(1, 2, 3, 4).cuda()
        out = mod.transpose_pad_wrapper(x, 2, 2, torch.tensor([1, 1]).cuda(), 3, 4)
        assert out.shape == (2, 3, 2, 4) and torch.equal(out[:, :, 0].cpu(), x[0].cpu())
    finally:
        for n in names:
            sys.modules.pop(n, None)
            if saved[n] is not None:
                sys.modules[n] = saved[n]


def test_lengths_created_in_inference_mode():
    """The reference worker runs the whole forward under torch.inference_mode() (energonai/worker.py:79); lengths
    made there carry no version counter.  Every wrapper must still work, and an in-place edit of such a tensor
    must be seen by the next call (nothing is cached for it)."""
    from energonai_amd import kernel as K
    B, S, H, D = 3, 16, 2, 8
    announce("inference-mode lens")
    x = torch.randn(B, S, H * D, generator=torch.Generator().manual_seed(6))
    with torch.inference_mode():
        lens = torch.tensor([5, 16, 1]).cuda()
        assert torch.is_inference(lens)
        packed = K.depad(x.cuda(), B, lens)
        assert torch.equal(packed.cpu(), eager.depad(x, B, [5, 16, 1]))
        padded = K.transpose_pad(packed.view(1, -1, H, D), B, S, lens, H, D)
        assert torch.equal(padded.cpu(), eager.transpose_pad(packed.cpu().view(1, -1, H, D), B, S, [5, 16, 1], H, D))
        lens[0] = 7
        packed2 = K.depad(x.cuda(), B, lens)
        assert torch.equal(packed2.cpu(), eager.depad(x, B, [7, 16, 1]))


def test_query_lengths_given_as_a_list():
    """q_len_list as a Python list lives in a device tensor owned by the call alone; the output tensor allocated
    right after must not be handed its memory before the kernel has run."""
    from energonai_amd import kernel as K
    B, H, Sq, Sk, D = 4, 2, 8, 64, 32
    kl, ql = [64, 40, 9, 33], [8, 8, 3, 1]
    announce("q_len_list as list")
    g = torch.Generator().manual_seed(7)
    q = torch.randn(B, H, Sq, D, generator=g).half().cuda()
    k = torch.randn(B, H, Sk, D, generator=g).half().cuda()
    v = torch.randn(B, H, Sk, D, generator=g).half().cuda()
    kl_t, ql_t = torch.tensor(kl, dtype=torch.int32).cuda(), torch.tensor(ql, dtype=torch.int32).cuda()
    for _ in range(3):      # repeated so that freed blocks are there to be reused
        s_list = K.attn_qk(q, k, kl, q_len_list=ql)
        s_tens = K.attn_qk(q, k, kl_t, q_len_list=ql_t)
        p_list = K.scale_mask_softmax(B, Sq, H, s_list, kl, scale=D ** -0.5, k_seq_len=Sk, q_len_list=ql)
        p_tens = K.scale_mask_softmax(B, Sq, H, s_tens, kl_t, scale=D ** -0.5, k_seq_len=Sk, q_len_list=ql_t)
        c_list = K.attn_pv(p_list, v, kl, q_len_list=ql)
        c_tens = K.attn_pv(p_tens, v, kl_t, q_len_list=ql_t)
        f_list = K.attn_fused(q, k, v, kl, q_len_list=ql)
        f_tens = K.attn_fused(q, k, v, kl_t, q_len_list=ql_t)
        for b in range(B):
            assert torch.equal(c_list[b, :, :ql[b]], c_tens[b, :, :ql[b]])
            assert torch.equal(f_list[b, :, :ql[b]], f_tens[b, :, :ql[b]])
    want = eager.attn_pv(eager.scale_mask_softmax(B, Sq, H, eager.attn_qk(q.cpu(), k.cpu(), torch.float32), kl,
                                                  scale=D ** -0.5, k_seq_len=Sk, q_lens=ql), v.cpu(), torch.float32)
    for b in range(B):
        assert max_abs(c_list[b, :, :ql[b]].cpu(), want[b, :, :ql[b]]) <= 2e-3


def test_cached_offsets_used_on_another_stream():
    """The offsets of a batch are computed by a kernel on the stream of first use and cached; a later call on
    another stream must be ordered behind that kernel."""
    from energonai_amd import _lib
    from energonai_amd import kernel as K
    from energonai_amd.seqinfo import clear_cache, seq_info
    B, S, hid = 6, 64, 256
    lens = [64, 1, 30, 17, 0, 55]
    announce("offsets across streams")
    x = torch.randn(B, S, hid, generator=torch.Generator().manual_seed(8))
    xg = x.cuda()
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()
    want = eager.depad(x, B, lens)
    torch.cuda.synchronize()
    clear_cache()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        info = seq_info(lens_t, B, xg.device)                  # prefix kernel launched on `side`
        assert _lib.stream_of(xg) in info._ordered
    main_raw = _lib.stream_of(xg)
    assert main_raw not in info._ordered
    got = K.depad(xg, B, lens_t, sum_seq=sum(lens))          # cache hit on the main stream
    assert seq_info(lens_t, B, xg.device) is info and main_raw in info._ordered
    assert torch.equal(got.cpu(), want)
    off = info.row_offsets(S, True)                           # produced on the main stream ...
    with torch.cuda.stream(side):                             # ... and consumed on the other one
        y = K.layer_norm_forward(torch.zeros(1, sum(lens), hid, device="cuda"), torch.ones(hid, device="cuda"),
                                 torch.zeros(hid, device="cuda"), (hid,), 1e-5, residual=xg,
                                 residual_row_offsets=info.row_offsets(S, True))
    side.synchronize()
    left = torch.cat([x[b, S - n:] for b, n in enumerate(lens)])
    assert max_abs(y.cpu()[0], torch.nn.functional.layer_norm(left, (hid,))) <= 1e-5
    assert off.data_ptr() == info.row_offsets(S, True).data_ptr()


def test_yardstick_kernels_touch_exactly_their_pattern():
    """The bandwidth yardsticks are measuring sticks, but a stick that moved other bytes than it claims would
    mislead: the copy copies, the write-only pass writes its whole range, the prefix passes write the causal
    prefixes of the valid rows (whole 16-byte vectors) and nothing else."""
    import torch
    from energonai_amd import _lib
    from energonai_amd.kernel.attention import packed_scores_elems
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    n = 1 << 20
    a = torch.randint(0, 255, (n,), dtype=torch.uint8, device="cuda")
    for nt in (0, 1):
        b = torch.zeros(n, dtype=torch.uint8, device="cuda")
        _lib.check(lib.en_stream_yardstick(a.data_ptr(), b.data_ptr(), n, 0, nt, stream), "copy")
        assert torch.equal(a, b)
        b.fill_(7)
        _lib.check(lib.en_stream_yardstick(None, b.data_ptr(), n, 2, nt, stream), "write")
        assert bool((b == 0).all())
        b.fill_(7)
        _lib.check(lib.en_stream_yardstick(a.data_ptr(), b.data_ptr(), n, 1, nt, stream), "read")
        assert bool((b == 7).all())
    B, H, S = 3, 2, 200
    lens = [200, 0, 77]
    lens_t = torch.tensor(lens, dtype=torch.int32, device="cuda")
    for packed in (0, 1):
        numel = packed_scores_elems(B, H, S, torch.float16) if packed else B * H * S * S
        src = torch.randn(numel, device="cuda").half()
        for mode in (0, 1, 2, 3, 4, 5, 6, 7):
            buf = src.clone()
            out = torch.full_like(src, 5.0)
            _lib.check(lib.en_prefix_yardstick(buf.data_ptr(), out.data_ptr(), lens_t.data_ptr(), B, H, S, packed, mode, 0, 2,
                                               stream), "prefix")
            touched = torch.zeros(numel, dtype=torch.bool)
            for b in range(B):
                for h in range(H):
                    unit = b * H + h
                    if packed:       # a unit's valid rows are one contiguous range: rows back to back, 128-byte groups
                        t = lens[b] // 64
                        end = 64 * (64 * t * (t + 1) // 2 + (lens[b] - 64 * t) * (t + 1))
                        touched[unit * (numel // (B * H)):unit * (numel // (B * H)) + end] = True
                        continue
                    for q in range(lens[b]):
                        start = (unit * S + q) * S
                        touched[start:start + -(-(q + 1) // 8) * 8] = True
            if mode in (0, 2, 4, 5, 6, 7):     # 4..7: read only, a 128-row tile at a time along the keys
                assert torch.equal(buf, src) and bool((out == 5.0).all())
            if mode == 1:
                assert bool((buf.cpu()[touched] == 0).all()) and torch.equal(buf.cpu()[~touched], src.cpu()[~touched])
            if mode == 3:
                assert torch.equal(out.cpu()[touched], src.cpu()[touched]) and bool((out.cpu()[~touched] == 5.0).all())


NATIVE_OPS = ("layer_norm", "kv_pages_append", "decode_attn_paged", "depad", "transpose_pad", "transpose_depad", "scale_mask_softmax",
              "attn_qk", "attn_pv")


class _Sub(torch.Tensor):
    pass


class _General:
    """The native module without the single operations: the Python calls do all of it."""

    def __init__(self, front):
        self._front = front

    def __getattr__(self, name):
        return (lambda *args: None) if name in NATIVE_OPS else getattr(self._front, name)


class _Watched:
    """The native module, noting the operands and results of the single operations."""

    def __init__(self, front):
        self._front, self.seen = front, {name: [] for name in NATIVE_OPS}

    def __getattr__(self, name):
        native = getattr(self._front, name)
        if name not in NATIVE_OPS:
            return native

        def call(*args):
            result = native(*args)
            self.seen[name].append((args, result))
            return result
        return call


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form", ["plain", "strided", "subclass", "side stream", "function mode", "dispatch mode"])
def test_single_operations_give_the_same_natively_and_in_python(dtype, form, monkeypatch):
    """Each call that has a native form against the same call with that form turned off, bit for bit, over what either accepts; what
    one refuses the other refuses in the same words.  The native forms do run where operands are plain, and leave a subclass's and a
    mode's calls alone."""
    from energonai_amd import _lib, kernel as K
    from energonai_amd.seqinfo import build_seq_info
    announce("native single ops", dtype, form)
    g = torch.Generator().manual_seed(11)
    B, S, H, D, P, lens = 3, 23, 5, 64, 16, [23, 1, 17]
    T, hid = sum(lens), 5 * 64

    def rnd(*shape):
        t = torch.randn(*shape, generator=g).to(dtype).cuda()
        if form == "strided" and len(shape) > 1:      # rows further apart than they are long
            return torch.cat([t, t], -1)[..., :shape[-1]]
        return t.as_subclass(_Sub) if form == "subclass" else t

    x, qkv, w, b = rnd(B, S, hid), rnd(1, T, H, 3 * D), rnd(hid), rnd(hid)
    q1, kn, vn = rnd(B, H, 1, D), rnd(B, H, D), rnd(B, H, D)
    pools = [torch.randn(7, H, P, D, generator=g).to(dtype).cuda() for _ in range(2)]
    table = torch.tensor([[3, 5], [0, -1], [6, 1]], dtype=torch.int32).cuda()
    lens_gpu = torch.tensor(lens, dtype=torch.int32).cuda()
    over = torch.zeros(1, dtype=torch.int32).cuda()

    def run():
        info = build_seq_info(lens_gpu, B, total=T)
        if form == "side stream":      # the lengths are ready on another stream than the one the calls run on
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                out = ops(info)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            return out
        if form == "function mode":
            class Seen(torch.overrides.TorchFunctionMode):
                def __torch_function__(self, func, types, args=(), kwargs=None):
                    return func(*args, **(kwargs or {}))
            with Seen():
                return ops(info)
        if form == "dispatch mode":
            from torch.utils._python_dispatch import TorchDispatchMode

            class SeenBelow(TorchDispatchMode):
                def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                    return func(*args, **(kwargs or {}))
            with SeenBelow():
                return ops(info)
        return ops(info)

    def ops(info):
        rows = K.depad(x, B, info, left_padded=True, sum_seq=T)
        q, k, v = torch.chunk(K.transpose_pad(qkv, B, S, info, H, 3 * D), 3, dim=-1)
        probs = K.scale_mask_softmax(B, S, H, K.attn_qk(q, k, info, alpha=0.5).nan_to_num(0, 0, 0), info, scale=0.125)
        ctx = K.transpose_depad(K.attn_pv(probs, v, info), B, T, S, info, H, D)
        mine = [p.clone() for p in pools]
        K.kv_pages_append(kn, vn, *mine, info, table, over)
        paged = K.decode_attn_paged(q1, *mine, info, table)
        y = K.layer_norm_forward(ctx.view(1, T, hid), w, b, (hid,), 1e-5, residual=rows)
        plain_y = K.layer_norm_forward(rows, w, b, hid)
        wide = K.layer_norm_forward(rows.float(), w, b, torch.Size([hid]), 1e-3)
        refused = []
        for call in (lambda: K.layer_norm_forward(rows, w, b, (hid + 8,)), lambda: K.layer_norm_forward(rows, w.double(), b.double(), (hid,)),
                     lambda: K.layer_norm_forward(rows, w, b, (hid,), residual=rows[:, :-1]), lambda: K.attn_qk(q, k[:, :-1], info),
                     lambda: K.attn_pv(probs, v.double(), info), lambda: K.transpose_pad(qkv.cpu(), B, S, info, H, 3 * D),
                     lambda: K.transpose_depad(ctx, B, T, S, info, H, D), lambda: K.depad(rows[0], B, info, sum_seq=T),
                     lambda: K.depad(x[:B - 1], B, info, sum_seq=T),      # fewer sequences than the batch has
                     lambda: K.decode_attn_paged(q1, mine[0], mine[1][:-1], info, table), lambda: K.kv_pages_append(kn[:2], vn, *mine, info, table),
                     lambda: K.decode_attn_paged(q1, *mine, info, table.long()), lambda: K.scale_mask_softmax(B, S, H + 1, probs, info)):
            with pytest.raises(RuntimeError) as e:
                call()
            refused.append(str(e.value))
        return [rows, ctx, *mine, paged, y, plain_y, wide], refused

    front = _lib.front
    watched = _Watched(front)
    monkeypatch.setattr(_lib, "front", watched)
    native, native_refused = run()
    monkeypatch.setattr(_lib, "front", _General(front))
    general, general_refused = run()
    torch.cuda.synchronize()
    for name, calls in watched.seen.items():
        assert calls, name
        if form in ("plain", "side stream"):
            assert any(result is not None for _, result in calls), name
        for args, result in calls:
            if form in ("function mode", "dispatch mode") or any(type(a) is _Sub for a in args):
                assert result is None, name
    assert native_refused == general_refused
    for got, want in zip(native, general):
        assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(torch.Tensor(got), torch.Tensor(want))


def test_single_operations_word_odd_flags_and_numbers_as_the_python_calls(monkeypatch):
    """A flag that is an array of several values, a number past 64 bits or past a double: the error of the Python call."""
    import numpy as np
    from energonai_amd import _lib, kernel as K
    from energonai_amd.seqinfo import build_seq_info
    announce("native odd flags")
    B, S, H, D = 2, 8, 2, 64
    info = build_seq_info([8, 3], B)
    q, rows = torch.randn(B, H, S, D).half().cuda(), torch.randn(B, S, H * D).half().cuda()
    probs, w = torch.rand(B, H, S, S).half().cuda(), torch.ones(H * D).half().cuda()
    two, many, huge = np.array([True, False]), 2 ** 70, 10 ** 400
    calls = (lambda: K.attn_qk(q, q, info, causal=two), lambda: K.attn_pv(probs, q, info, causal=two),
             lambda: K.scale_mask_softmax(B, S, H, probs, info, causal=two), lambda: K.depad(rows, B, info, left_padded=two, sum_seq=11),
             lambda: K.attn_qk(q, q, info, alpha=huge), lambda: K.scale_mask_softmax(B, S, H, probs, info, scale=huge),
             lambda: K.layer_norm_forward(rows, w, w, (H * D,), huge), lambda: K.layer_norm_forward(rows, w, w, (many,)),
             lambda: K.depad(rows, many, info, sum_seq=11), lambda: K.transpose_pad(rows, many, S, info, H, D),
             lambda: K.scale_mask_softmax(many, S, H, probs, info), lambda: K.transpose_depad(q, B, 11, many, info, H, D))

    def refusals():
        out = []
        for call in calls:
            with pytest.raises(Exception) as e:
                call()
            out.append((e.type, str(e.value)))
        return out

    native = refusals()
    monkeypatch.setattr(_lib, "front", _General(_lib.front))
    assert native == refusals()
    assert [t for t, _ in native[:4]] == [ValueError] * 4


def test_which_operands_a_native_operation_takes():
    """The native forms take plain operands and leave everything else, with nothing launched, to the Python calls."""
    from energonai_amd import _lib
    announce("native operands")
    x, w = torch.randn(4, 64).half().cuda(), torch.randn(64).half().cuda()
    take = lambda *a: _lib.front.layer_norm(*a) is not None
    assert take(x, w, w, (64,), 1e-5, None) and take(x, w, w, 64, 1e-5, x) and take(x.float(), w, w, (64,), 1, None)
    for args in ((x.t().contiguous().t(), w, w, (64,), 1e-5, None), (x.as_subclass(_Sub), w, w, (64,), 1e-5, None), (x.cpu(), w, w, (64,), 1e-5, None),
                 (x, w.float(), w.float(), (64,), 1e-5, None), (x, w, w.float(), (64,), 1e-5, None), (x, w, w, (4, 64), 1e-5, None),
                 (x, w, w, (32,), 1e-5, None), (x, w, w, (64,), "1e-5", None), (x, w, w, (64,), 1e-5, x.float()), (x[:0], w, w, (64,), 1e-5, None)):
        assert not take(*args)


def test_which_operands_the_other_native_operations_take():
    """Each with operands that it takes and, one at a time, with one that it leaves to the Python call."""
    from energonai_amd import _lib
    from energonai_amd.seqinfo import build_seq_info
    announce("native operands of the other operations")
    B, S, H, D, P, lens = 2, 24, 3, 64, 16, [24, 5]
    T = sum(lens)
    info, other = build_seq_info(lens, B), build_seq_info([3, 4, 5], 3)
    half = lambda *shape: torch.randn(*shape).half().cuda()
    strided = lambda *shape: torch.randn(*shape, 2).half().cuda()[..., 0]
    x, qkv, q, ctx, probs = half(B, S, H * D), half(1, T, H, D), half(B, H, S, D), half(B, H, S, D), torch.rand(B, H, S, S).half().cuda()
    kn, pool, q1 = half(B, H, D), half(4, H, P, D), half(B, H, 1, D)
    table, over = torch.tensor([[0, 1], [2, 3]], dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
    cases = {
        "depad": ((x, info, B, True, T), {0: [strided(B, S, H * D), x.cpu(), x.double(), x[0], x[:1], x.as_subclass(_Sub)], 1: [other], 2: [3, 0], 3: [None, "left"],
                                          4: [0, 2 ** 40]}),
        "transpose_pad": ((qkv, info, B, S, H, D), {0: [strided(1, T, H, D), qkv.cpu(), qkv.double(), qkv.as_subclass(_Sub)], 1: [other], 2: [3], 3: [0], 4: [H + 1],
                                                    5: [0, 2 ** 40]}),
        "transpose_depad": ((ctx, info, B, T, S, H, D), {0: [strided(B, H, S, D), ctx.cpu(), ctx.double(), ctx[:1].clone()], 1: [other], 2: [3], 3: [0], 4: [S + 1],
                                                         5: [H + 1], 6: [D + 1]}),
        "scale_mask_softmax": ((probs.clone(), info, B, S, H, 0.5, True, 1), {0: [strided(B, H, S, S), probs.cpu(), probs.double(), probs[:1].clone()], 1: [other],
                                                                               2: [3], 3: [S + 1], 4: [H + 1], 5: ["1"], 6: [None], 7: [-1]}),
        "attn_qk": ((q, q, info, 1.0, True), {0: [strided(B, H, S, D), q.cpu(), q[0], q.double()], 1: [q[:, :2], q.float(), q[..., :32]], 2: [other], 3: ["1"], 4: [None]}),
        "attn_pv": ((probs, q, info, False), {0: [strided(B, H, S, S), probs.cpu(), probs[0]], 1: [q[:, :2], q.float(), q[:, :, :8]], 2: [other], 3: [None]}),
        "kv_pages_append": ((kn, kn, pool.clone(), pool.clone(), info, table, over), {
            0: [strided(B, H, D), kn.cpu(), kn[:1], kn.float()], 1: [kn[:, :2], kn.float()], 2: [pool[:2], pool.cpu()], 3: [pool[:2], pool.float()], 4: [other],
            5: [table.long(), table[:1], table.cpu()], 6: [over.long(), over.cpu()]}),
        "decode_attn_paged": ((q1, pool, pool, info, table, None), {0: [strided(B, H, 1, D), q1.cpu(), q1.float(), q1[:1]], 1: [pool[:2], pool.float()],
                                                                     2: [pool[:2], pool.float()], 3: [other], 4: [table.long(), table[:1]], 5: ["1"]}),
    }
    assert set(cases) == set(NATIVE_OPS) - {"layer_norm"}
    for name, (args, others) in cases.items():
        native = getattr(_lib.front, name)
        assert native(*args) is not None, name
        for i, values in others.items():
            for value in values:
                assert native(*args[:i], value, *args[i + 1:]) is None, (name, i, value if not isinstance(value, torch.Tensor) else value.shape)
    torch.cuda.synchronize()
