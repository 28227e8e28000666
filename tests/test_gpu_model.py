"""Model glue (attention / MLP / block modules, K/V cache, repad) against the padded eager oracle."""
import pytest
import torch
import torch.nn.functional as F

from gpu_util import announce, max_abs
from oracle import eager, models

pytestmark = pytest.mark.gpu


def _mods():
    import energonai_amd.kernel as K
    import energonai_amd.model as M
    return K, M


def _fp32_params(module):
    return {k: v.detach().float().cpu() for k, v in module.state_dict().items()}


def _padded_batch(B, S, hid, lens, left, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, S, hid, generator=g).to(dtype)
    valid = torch.zeros(B, S)
    for b, n in enumerate(lens):
        if left:
            valid[b, S - n:] = 1
        else:
            valid[b, :n] = 1
    return x * valid.unsqueeze(-1).to(dtype), valid


def _init(module, seed):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for name, prm in module.named_parameters():
            if name.endswith("weight") and prm.dim() == 1:
                prm.copy_(1.0 + 0.05 * torch.randn(prm.shape, generator=g))
            elif prm.dim() == 1:
                prm.copy_(0.05 * torch.randn(prm.shape, generator=g))
            else:
                prm.copy_(torch.randn(prm.shape, generator=g) / prm.shape[1] ** 0.5)


def _valid_rows(t, lens, left):
    S = t.shape[1]
    return torch.cat([t[b, S - n:] if left else t[b, :n] for b, n in enumerate(lens)])


@pytest.mark.parametrize("left", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_repad_is_inverse_of_depad(dtype, left):
    K, _ = _mods()
    B, S, hid = 5, 37, 96
    lens = [37, 1, 0, 20, 36]
    announce("repad", dtype, left)
    x, _ = _padded_batch(B, S, hid, lens, left, dtype, 11)
    lens_t = torch.tensor(lens, dtype=torch.int64).cuda()
    packed = K.depad(x.cuda(), B, lens_t, left_padded=left)
    back = K.repad(packed, B, S, lens_t, left_padded=left).cpu()
    assert torch.equal(back, x)
    assert torch.equal(back, eager.repad(packed.cpu(), B, S, lens, left_padded=left))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_kv_cache_fill_and_append_bit_exact(dtype):
    K, M = _mods()
    B, H, D, Smax = 3, 4, 64, 50
    lens = [7, 30, 1]
    T = sum(lens)
    announce("kv cache", dtype)
    g = torch.Generator().manual_seed(12)
    kvq = torch.randn(T, 3 * H, D, generator=g).to(dtype)
    info_lens = torch.tensor(lens, dtype=torch.int32).cuda()
    cache = M.KVCache(B, H, Smax, D, dtype, "cuda")
    from energonai_amd.seqinfo import seq_info
    info = seq_info(info_lens, B, torch.device("cuda"))
    cache.fill(kvq.cuda(), kvq.cuda(), info, 0, H, longest=max(lens))
    want_k = torch.zeros(B, H, Smax, D, dtype=dtype)
    want_v = torch.zeros_like(want_k)
    start = 0
    for b, n in enumerate(lens):
        want_k[b, :, :n] = kvq[start:start + n, :H].permute(1, 0, 2)
        want_v[b, :, :n] = kvq[start:start + n, H:2 * H].permute(1, 0, 2)
        start += n
    assert torch.equal(cache.k.cpu(), want_k) and torch.equal(cache.v.cpu(), want_v)
    assert cache.lens.cpu().tolist() == lens
    for step in range(3):
        new = torch.randn(B, 3 * H, D, generator=g).to(dtype)
        new_g = new.cuda()
        cache.append(new_g[:, :H], new_g[:, H:2 * H])
        for b, n in enumerate(lens):
            want_k[b, :, n + step] = new[b, :H]
            want_v[b, :, n + step] = new[b, H:2 * H]
        assert torch.equal(cache.k.cpu(), want_k) and torch.equal(cache.v.cpu(), want_v)
        assert cache.lens.cpu().tolist() == [n + step + 1 for n in lens]
    # a cache that may be full refuses the next row instead of dropping it silently
    small = M.KVCache(B, H, max(lens) + 2, D, dtype, "cuda")
    small.fill(kvq.cuda(), kvq.cuda(), info, 0, H, longest=max(lens))
    new_g = torch.randn(B, 3 * H, D, generator=g).to(dtype).cuda()
    small.append(new_g[:, :H], new_g[:, H:2 * H])
    small.append(new_g[:, :H], new_g[:, H:2 * H])
    with pytest.raises(RuntimeError, match="max_seq_len"):
        small.append(new_g[:, :H], new_g[:, H:2 * H])
    assert small.lens.cpu().tolist() == [n + 2 for n in lens]
    # a caller of the C entry point itself (no host-side bound of the lengths) is told through a device counter:
    # sequence 1 is full now, the other two take the row
    overflow = torch.zeros(1, dtype=torch.int32, device="cuda")
    before_k = small.k.clone()
    K.kv_cache_append(new_g[:, :H], new_g[:, H:2 * H], small.k, small.v, small.info, overflow=overflow)
    assert overflow.item() == 1
    assert torch.equal(small.k[1], before_k[1])
    for b in (0, 2):
        assert torch.equal(small.k[b, :, lens[b] + 2], new_g[b, :H])
    K.kv_cache_append(new_g[:, :H], new_g[:, H:2 * H], small.k, small.v, small.info, overflow=overflow)
    assert overflow.item() == 2


@pytest.mark.parametrize("dtype,activation,heads,D,bias,page,lens", [
    (torch.float16, torch.nn.functional.relu, 4, 64, True, None, [7, 30, 1]),
    (torch.bfloat16, torch.nn.GELU(), 3, 80, True, 16, [1]),
    (torch.float16, torch.nn.GELU(approximate="tanh"), 2, 128, False, None, [33, 0, 16]),
    (torch.float16, torch.nn.functional.gelu, 5, 24, False, None, [4, 4]),
    (torch.float16, torch.nn.SiLU(), 2, 64, True, None, [5]),             # no code for it: the general form
    (torch.float16, torch.nn.functional.relu, 2, 136, True, None, None),  # heads the fused kernel does not take
])
def test_native_prefill_gives_the_general_forms_bits(monkeypatch, dtype, activation, heads, D, bias, page, lens):
    """A prefill through the native call against the same block op by op: output, caches, lengths and the steps behind them."""
    _, M = _mods()
    from energonai_amd import _lib
    from energonai_amd.model import endecoder
    announce("native prefill", dtype, activation, heads, D, bias, page, lens)
    hid, S = heads * D, 40
    torch.manual_seed(heads + D)
    blocks = [M.Block1D(hid, heads, 2.0, activation=activation, dtype=dtype, bias=bias, max_seq_len=64, kv_page_size=page) for _ in range(2)]
    stack = M.PackedStack(blocks).cuda()
    calls = []
    real = _lib.load_front().block_prefill
    monkeypatch.setattr(_lib.front, "block_prefill", lambda *args: calls.append(real(*args)) or calls[-1], raising=False)
    if lens is None:
        with torch.no_grad(), pytest.raises(RuntimeError):
            stack(torch.randn(1, S, hid, device="cuda").to(dtype), first_cache=True, seq_lens=torch.tensor([5], dtype=torch.int32).cuda())
        assert calls == [None]
        return
    x = torch.randn(len(lens), S, hid, device="cuda").to(dtype)
    tokens = [torch.randn(len(lens), 1, hid, device="cuda").to(dtype) for _ in range(2)]
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()

    def run():
        with torch.no_grad():
            out = [stack(x, first_cache=True, seq_lens=lens_t)]
            state = [t.clone() for b in blocks for t in (b.attn.kv_cache.k, b.attn.kv_cache.v, b.attn.kv_cache.lens)]
            out += [stack(t).clone() for t in tokens]
            out.append(blocks[0](x, first_cache=True, seq_lens=lens_t).clone())       # a block by itself
        return out + state

    got = run()
    native = endecoder.activation_code(activation, blocks[0].mlp._epilogue)
    assert len(calls) == (3 if native is not None else 0) and all(c is not None for c in calls)
    monkeypatch.setattr(M.Block1D, "_native_prefill", lambda *args: None)
    want = run()
    assert len(got) == len(want) and all(torch.equal(g, w) for g, w in zip(got, want))


def test_native_prefill_takes_the_lengths_that_the_general_form_takes(monkeypatch):
    """Packed rows with a lengths tensor or a list in place of the SeqInfo; lengths of another batch never reach a launch."""
    _, M = _mods()
    from energonai_amd import _lib
    from energonai_amd.seqinfo import seq_info
    announce("native prefill, lengths")
    torch.manual_seed(6)
    blk = M.Block1D(128, 2, 2.0, dtype=torch.float16, max_seq_len=64).cuda()
    x, lens = torch.randn(1, 37, 128, device="cuda").half(), [7, 30]
    lens_t, calls = torch.tensor(lens, dtype=torch.int32).cuda(), []
    native = _lib.load_front().block_prefill
    monkeypatch.setattr(_lib.front, "block_prefill", lambda *args: calls.append(args) or native(*args), raising=False)
    with torch.no_grad():
        want = blk.forward_packed(x, seq_info(lens_t, 2, x.device), 2, 32)
        for given in (lens_t, lens):
            assert torch.equal(blk.forward_packed(x, given, 2, 32), want)
        assert len(calls) == 3
        for batch in (1, 3):
            with pytest.raises(RuntimeError, match="SeqInfo was built for batch 2"):
                blk.forward_packed(x, seq_info(lens_t, 2, x.device), batch, 32)
            args = list(calls[0])
            args[22] = batch
            assert native(*args) is None
    assert len(calls) == 3


@pytest.mark.parametrize("activation", [torch.nn.functional.relu, torch.nn.GELU()])
@pytest.mark.parametrize("fill", [True, False])
def test_native_prefill_holds_no_more_memory_than_the_general_form(monkeypatch, activation, fill):
    """Peaks of torch's allocator over one block, in bytes: a batch that fits the general form fits the native call."""
    _, M = _mods()
    from energonai_amd.seqinfo import seq_info
    announce("native prefill, peak memory", activation, fill)
    torch.manual_seed(7)
    blk = M.Block1D(512, 8, 4.0, activation=activation, dtype=torch.float16, max_seq_len=512).cuda()
    x = torch.randn(1, 2048, 512, device="cuda").half()
    info = seq_info(torch.tensor([512] * 4, dtype=torch.int32).cuda(), 4, x.device)

    def peak():
        with torch.no_grad():
            for _ in range(2):                      # the first pass makes what is kept: tables, the GEMMs' scratch
                blk.attn.kv_cache = None
                torch.cuda.synchronize()
                torch.cuda.reset_peak_memory_stats()
                before = torch.cuda.memory_allocated()
                y = blk.forward_packed(x, info, 4, 512, fill)
                torch.cuda.synchronize()
                bytes_ = torch.cuda.max_memory_allocated() - before
                assert y.shape == x.shape
                del y
        return bytes_

    native = peak()
    monkeypatch.setattr(M.Block1D, "_native_prefill", lambda *args: None)
    general = peak()
    announce("peak, rows of hidden", native / (2048 * 512 * 2), general / (2048 * 512 * 2))
    assert native <= general


@pytest.mark.parametrize("dtype,H,D,Smax,lens", [
    (torch.float16, 4, 64, 50, [7, 30, 1]), (torch.bfloat16, 3, 80, 129, [129, 0, 64, 65]), (torch.float32, 2, 64, 700, [700, 3]),
    (torch.float16, 3, 10, 20, [20, 5]),                 # rows of 20 bytes: no 16-byte pieces, two launches
    (torch.float16, 24, 128, 4096, [4096, 17, 0, 1]),    # 96 MB a cache: two launches
])
def test_kv_caches_filled_from_scratch_in_one_launch(dtype, H, D, Smax, lens):
    """A cache allocated without zeros is filled with the rows and the zeros behind them: the same buffers as zeros and two movers."""
    K, M = _mods()
    from energonai_amd.seqinfo import seq_info
    announce("kv start", dtype, H, D, Smax, lens)
    B, T = len(lens), sum(lens)
    g = torch.Generator().manual_seed(33)
    kvq = torch.randn(T, 3 * H, D, generator=g).to(dtype).cuda()
    info = seq_info(torch.tensor(lens, dtype=torch.int32).cuda(), B, torch.device("cuda"))
    want = M.KVCache(B, H, Smax, D, dtype, "cuda")
    want.fill(kvq, kvq, info, 0, H, longest=max(lens))
    for k_src, v_src, v_first in ((kvq, kvq, H), (kvq, kvq[:, H:2 * H].contiguous(), 0)):
        got = M.KVCache(B, H, Smax, D, dtype, "cuda", zeroed=False)
        got.k.fill_(7.0), got.v.fill_(7.0), got.lens.fill_(7)
        got.fill(k_src, v_src, info, 0, v_first, longest=max(lens))
        assert torch.equal(got.k, want.k) and torch.equal(got.v, want.v) and torch.equal(got.lens, want.lens)
        assert got._longest == want._longest


@pytest.mark.parametrize("left", [False, True])
def test_repad_into_a_longer_buffer(left):
    K, _ = _mods()
    lens, S, hid = [5, 0, 9], 9, 40
    g = torch.Generator().manual_seed(34)
    x = torch.randn(1, sum(lens), hid, generator=g).half().cuda()
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()
    buf = torch.full((3, 13, hid), 7.0, dtype=torch.float16, device="cuda")
    assert K.repad(x, 3, S, lens_t, left_padded=left, out=buf) is buf
    assert torch.equal(buf[:, :S], K.repad(x, 3, S, lens_t, left_padded=left)) and bool((buf[:, S:] == 7.0).all())
    for bad in (buf[:, :8].contiguous(), buf[:2], buf.float(), buf[:, :, :32].contiguous()):
        with pytest.raises(RuntimeError, match="out must be"):
            K.repad(x, 3, S, lens_t, left_padded=left, out=bad)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_kv_cache_fill_without_zero_fill_leaves_padding_untouched(dtype):
    """zero_padding=False: rows below each length are written, every other row keeps the bits it had
    (tiles that lie wholly in the padding are skipped, tiles that straddle a length are written in part)."""
    K, _ = _mods()
    B, H, D, Smax = 4, 3, 64, 700
    lens = [700, 0, 129, 64]
    T = sum(lens)
    announce("kv fill no zero", dtype)
    g = torch.Generator().manual_seed(31)
    src = torch.randn(T, 2 * H, D, generator=g).to(dtype)
    sentinel = torch.full((B, H, Smax, D), 123.0, dtype=dtype)
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()
    got = K.kv_cache_fill(src.cuda(), sentinel.clone().cuda(), B, lens_t, head_first=H, zero_padding=False).cpu()
    full = K.kv_cache_fill(src.cuda(), sentinel.clone().cuda(), B, lens_t, head_first=H).cpu()
    want = sentinel.clone()
    start = 0
    for b, n in enumerate(lens):
        want[b, :, :n] = src[start:start + n, H:].permute(1, 0, 2)
        start += n
    assert torch.equal(got, want)
    for b, n in enumerate(lens):
        assert torch.equal(full[b, :, :n], want[b, :, :n]) and not full[b, :, n:].any()


@pytest.mark.parametrize("fused_qkv", [True, False])
@pytest.mark.parametrize("is_decoder", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_attention_module_prefill(dtype, is_decoder, fused_qkv):
    """MultiHeadAttention1D.forward on a padded batch equals the reference forward on valid positions."""
    _, M = _mods()
    B, S, hid, heads = 4, 160, 256, 4
    lens = [160, 33, 97, 128]
    left = is_decoder
    announce("mha prefill", dtype, is_decoder, fused_qkv)
    attn = M.MultiHeadAttention1D(hid, heads, dtype=dtype, max_seq_len=192, fused_qkv=fused_qkv,
                                  is_decoder=is_decoder, disable_past_cache=True).cuda()
    _init(attn, 21)
    x, valid = _padded_batch(B, S, hid, lens, left, dtype, 22)
    mask = models.additive_mask(valid)
    got = attn(x.cuda(), attention_mask=mask.to(dtype).cuda()).float().cpu()
    want = models.mha_forward(x, _fp32_params(attn), heads, is_decoder, mask, fused_qkv)
    tol = {torch.float16: 4e-3, torch.bfloat16: 3e-2, torch.float32: 2e-4}[dtype]
    assert max_abs(_valid_rows(got, lens, left), _valid_rows(want, lens, left)) <= tol
    pad = torch.cat([got[b, :S - n] if left else got[b, n:] for b, n in enumerate(lens)])
    assert bool((pad == 0).all())          # padding rows come back as zeros


@pytest.mark.parametrize("post", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_block_prefill_and_incremental_decode(dtype, post):
    """Block1D: prefill with first_cache=True, then three decode steps; the newest position of each
    step equals the reference block recomputed on the whole extended (left-padded) batch."""
    _, M = _mods()
    B, S, hid, heads = 3, 70, 128, 2
    lens = [70, 9, 41]
    announce("block decode", dtype, post)
    blk = M.Block1D(hid, heads, 4.0, dtype=dtype, apply_post_layernorm=post, max_seq_len=96).cuda()
    _init(blk, 31)
    p = _fp32_params(blk)
    x, valid = _padded_batch(B, S, hid, lens, True, dtype, 32)
    tol = {torch.float16: 1.5e-2, torch.float32: 5e-4}[dtype]
    mask = models.additive_mask(valid)
    got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=True).float().cpu()
    want = models.block_forward(x, p, heads, 1e-5, post, True, mask)
    assert max_abs(_valid_rows(got, lens, True), _valid_rows(want, lens, True)) <= tol
    g = torch.Generator().manual_seed(33)
    for step in range(3):
        x = torch.cat((x, torch.randn(B, 1, hid, generator=g).to(dtype)), 1)
        valid = torch.cat((valid, torch.ones(B, 1)), 1)
        mask = models.additive_mask(valid)
        got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=False).float().cpu()
        want = models.block_forward(x, p, heads, 1e-5, post, True, mask)
        assert got.shape == want.shape
        assert max_abs(got[:, -1], want[:, -1]) <= tol, step


def test_block_with_tuned_gemms_matches_the_reference_block():
    """set_gemm_tuning(True): every projection of the block runs on the fastest hipBLASLt candidate for its
    shape (prefill shapes and the skinny decode shapes are separate problems); same tolerances as untuned."""
    _, M = _mods()
    from energonai_amd.kernel.cuda_native import linear_func as lf
    B, S, hid, heads = 3, 70, 128, 2
    lens = [70, 9, 41]
    dtype = torch.float16
    announce("block tuned gemms")
    blk = M.Block1D(hid, heads, 4.0, activation=F.relu, dtype=dtype, max_seq_len=96).cuda()
    _init(blk, 35)
    p = _fp32_params(blk)
    x, valid = _padded_batch(B, S, hid, lens, True, dtype, 36)
    mask = models.additive_mask(valid)
    lf._tuned.clear()
    M.set_gemm_tuning(True)
    try:
        assert M.gemm_tuning()
        got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=True).float().cpu()
        n_prefill = len(lf._tuned)
        assert n_prefill == 4                 # qkv, dense, fc1 (+ReLU), fc2 at the packed row count
        want = models.block_forward(x, p, heads, 1e-5, False, True, mask, activation=F.relu)
        assert max_abs(_valid_rows(got, lens, True), _valid_rows(want, lens, True)) <= 1.5e-2
        g = torch.Generator().manual_seed(37)
        for step in range(2):
            x = torch.cat((x, torch.randn(B, 1, hid, generator=g).to(dtype)), 1)
            valid = torch.cat((valid, torch.ones(B, 1)), 1)
            mask = models.additive_mask(valid)
            got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=False).float().cpu()
            want = models.block_forward(x, p, heads, 1e-5, False, True, mask, activation=F.relu)
            assert max_abs(got[:, -1], want[:, -1]) <= 1.5e-2, step
        assert len(lf._tuned) == 2 * n_prefill        # the decode shapes were searched once, not per step
    finally:
        M.set_gemm_tuning(False)
    assert not M.gemm_tuning()


@pytest.mark.parametrize("act_name", ["relu", "gelu_tanh", "gelu"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_mlp_with_gemm_epilogues(dtype, act_name):
    """MLP1D: ReLU and tanh-GELU ride in the first GEMM's epilogue, erf-GELU stays a separate op; all
    three equal the reference MLP forward."""
    import functools
    _, M = _mods()
    hid, rows = 256, 77
    announce("mlp", dtype, act_name)
    act = {"relu": F.relu, "gelu_tanh": functools.partial(F.gelu, approximate="tanh"), "gelu": F.gelu}[act_name]
    mlp = M.MLP1D(hid, 4.0, act, dtype=dtype, disable_past_cache=True).cuda()
    assert (mlp._epilogue is None) == (act_name == "gelu")
    _init(mlp, 51)
    g = torch.Generator().manual_seed(52)
    x = torch.randn(1, rows, hid, generator=g).to(dtype)
    got = mlp(x.cuda()).float().cpu()
    want = models.mlp_forward(x, _fp32_params(mlp), act)
    tol = {torch.float16: 6e-3, torch.float32: 2e-4}[dtype]
    assert max_abs(got, want) <= tol * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_packed_stack_prefill_and_decode(dtype):
    """Three blocks with the padding dropped once for all of them, then two decode steps, against the
    reference blocks chained on the padded batch."""
    _, M = _mods()
    B, S, hid, heads, L = 3, 48, 128, 2, 3
    lens = [48, 5, 30]
    announce("stack", dtype)
    blocks = [M.Block1D(hid, heads, 4.0, activation=F.relu, dtype=dtype, max_seq_len=64) for _ in range(L)]
    stack = M.PackedStack(blocks).cuda()
    for i, blk in enumerate(stack.blocks):
        _init(blk, 60 + i)
    ps = [_fp32_params(blk) for blk in stack.blocks]
    x, valid = _padded_batch(B, S, hid, lens, True, dtype, 70)
    tol = {torch.float16: 4e-2, torch.float32: 2e-3}[dtype]

    def reference(x, valid):
        h = x.float()
        for p in ps:
            h = models.block_forward(h, p, heads, 1e-5, False, True, models.additive_mask(valid), F.relu)
        return h

    mask = models.additive_mask(valid)
    got = stack(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=True).float().cpu()
    want = reference(x, valid)
    scale = max(1.0, float(_valid_rows(want, lens, True).abs().max()))
    assert max_abs(_valid_rows(got, lens, True), _valid_rows(want, lens, True)) <= tol * scale
    g = torch.Generator().manual_seed(71)
    for step in range(2):
        x = torch.cat((x, torch.randn(B, 1, hid, generator=g).to(dtype)), 1)
        valid = torch.cat((valid, torch.ones(B, 1)), 1)
        got = stack(x.cuda(), attention_mask=models.additive_mask(valid).to(dtype).cuda(), first_cache=False)
        want = reference(x, valid)
        assert got.shape == want.shape
        assert max_abs(got[:, -1].float().cpu(), want[:, -1]) <= tol * scale, step


@pytest.mark.parametrize("seed", list(range(10)))
def test_block_random_shapes(seed):
    """Block1D on drawn shapes (head sizes 32 / 64 / 80 / 128, pre- or post-LN, ReLU / tanh-GELU / erf-GELU,
    fused or separate projections): prefill, then two incremental steps, against the reference block."""
    import functools
    _, M = _mods()
    g = torch.Generator().manual_seed(9100 + seed)
    ri = lambda lo, hi: int(torch.randint(lo, hi + 1, (1,), generator=g))
    heads, D = ri(1, 4), [32, 64, 80, 128][ri(0, 3)]
    hid = heads * D
    B, S = ri(1, 5), ri(2, 90)
    dtype = [torch.float16, torch.float32, torch.bfloat16][ri(0, 2)]
    post, fused_qkv = bool(ri(0, 1)), bool(ri(0, 1))
    act_name = ["relu", "gelu_tanh", "gelu"][ri(0, 2)]
    act = {"relu": F.relu, "gelu_tanh": functools.partial(F.gelu, approximate="tanh"), "gelu": F.gelu}[act_name]
    lens = [ri(1, S) for _ in range(B)]
    lens[ri(0, B - 1)] = S
    announce("block random", seed, B, S, heads, D, dtype, post, fused_qkv, act_name, lens)
    blk = M.Block1D(hid, heads, 4.0, activation=act, dtype=dtype, apply_post_layernorm=post, max_seq_len=S + 8,
                    fused_qkv=fused_qkv).cuda()
    _init(blk, 9200 + seed)
    p = _fp32_params(blk)
    x, valid = _padded_batch(B, S, hid, lens, True, dtype, 9300 + seed)
    tol = {torch.float16: 2e-2, torch.bfloat16: 1.5e-1, torch.float32: 1e-3}[dtype]
    mask = models.additive_mask(valid)
    got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=True).float().cpu()
    want = models.block_forward(x, p, heads, 1e-5, post, True, mask, activation=act, fused_qkv=fused_qkv)
    ref_scale = max(1.0, float(want.abs().max()))
    assert max_abs(_valid_rows(got, lens, True), _valid_rows(want, lens, True)) <= tol * ref_scale
    for step in range(2):
        x = torch.cat((x, torch.randn(B, 1, hid, generator=g).to(dtype)), 1)
        valid = torch.cat((valid, torch.ones(B, 1)), 1)
        mask = models.additive_mask(valid)
        got = blk(x.cuda(), attention_mask=mask.to(dtype).cuda(), first_cache=False).float().cpu()
        want = models.block_forward(x, p, heads, 1e-5, post, True, mask, activation=act, fused_qkv=fused_qkv)
        assert max_abs(got[:, -1], want[:, -1]) <= tol * ref_scale, step


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,heads,D,ratio,act,bias,page", [
    (1, 1, 64, 4.0, "relu", True, None),          # one row, one step of 64 channels
    (3, 12, 64, 4.0, "gelu", True, 16),           # 768 channels: three steps on four waves; pages
    (16, 3, 80, 4.0, "gelu_tanh", True, None),    # a full row tile; 240 channels end inside a step
    (17, 5, 40, 2.6, "relu", False, None),        # a second row tile of one row; 200 channels, no bias, an odd MLP width
    (32, 8, 128, 1.0, "relu", True, 32),          # the most rows; 1024 channels
    (2, 16, 128, 4.0, "gelu", True, None),        # 2048 channels, 8192 in the MLP
    (2, 17, 128, 1.0, "relu", True, None),        # too wide: the general path
    (33, 2, 64, 1.0, "relu", True, None),         # too many rows: the general path
])
def test_block_decode_in_one_native_call(dtype, B, heads, D, ratio, act, bias, page, monkeypatch):
    """Decode steps of a pre-LN block through ``en_block_decode`` (where it applies) against the block recomputed over the
    whole extended batch in fp32, at the tolerance of the block's general path; lengths, caches and history move on alike."""
    _, M = _mods()
    hid, S = heads * D, 20
    fn = {"relu": F.relu, "gelu": F.gelu, "gelu_tanh": torch.nn.GELU(approximate="tanh")}[act]
    announce("block decode native", dtype, B, heads, D, ratio, act, bias, page)
    blk = M.Block1D(hid, heads, ratio, activation=fn, dtype=dtype, bias=bias, max_seq_len=32, kv_page_size=page).cuda()
    _init(blk, 41)
    p = _fp32_params(blk)
    lens = [S - (3 * b) % S for b in range(B)]
    x, valid = _padded_batch(B, S, hid, lens, True, dtype, 42)
    g = torch.Generator().manual_seed(43)
    tol = {torch.float16: 1.5e-2, torch.bfloat16: 1.2e-1}[dtype]
    with torch.no_grad():
        blk(x.cuda(), attention_mask=models.additive_mask(valid).to(dtype).cuda(), first_cache=True)
        native = B <= 32 and hid <= 2048
        from energonai_amd import _lib
        taken, call = [], _lib.front.block_decode      # the call itself must be what runs where it applies
        monkeypatch.setattr(_lib.front, "block_decode", lambda *a: (lambda y: (taken.append(y is not None), y)[1])(call(*a)))
        for step in range(3):
            new = torch.randn(B, 1, hid, generator=g).to(dtype)
            x, valid = torch.cat((x, new), 1), torch.cat((valid, torch.ones(B, 1)), 1)
            before = blk.attn.kv_cache.lens._version
            # the newest position of a longer, strided view, as the block before hands it on
            wide = torch.zeros(B, 3, hid + 8, dtype=dtype)
            wide[:, 2:, :hid] = new
            got = blk(wide.cuda()[:, :, :hid], first_cache=False)
            assert taken == [True] * native
            del taken[:]
            want = models.block_forward(x, p, heads, 1e-5, False, True, models.additive_mask(valid), activation=fn)
            assert got.shape == want.shape
            assert max_abs(got[:, -1].float().cpu(), want[:, -1]) <= tol, step
            assert blk.attn.kv_cache.lens.tolist() == [n + step + 1 for n in lens]
            assert blk.attn.kv_cache.lens._version > before


@pytest.mark.parametrize("how", ["global_hook", "dense_2", "norm1", "forward_rows", "forward_last", "cache", "activation_hook",
                                 "weight_subclass"])
def test_block_decode_sees_what_a_caller_put_in(how):
    """Decode steps of a block whose modules a caller has instrumented run what the caller put there."""
    _, M = _mods()
    blk = M.Block1D(128, 2, 2.0, activation=torch.nn.GELU(), dtype=torch.float16, max_seq_len=32).cuda()
    _init(blk, 51)
    calls = []

    class Counted(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            calls.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})

    lin, handle = blk.mlp.dense_2, None
    announce("block decode instrumented", how)
    x = torch.randn(2, 8, 128, dtype=torch.float16, device="cuda")
    with torch.no_grad():
        blk(x, first_cache=True, seq_lens=torch.tensor([8, 5], dtype=torch.int32, device="cuda"))
        if how == "global_hook":
            handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, y: calls.append(m))
        elif how in ("dense_2", "norm1", "forward_rows", "forward_last", "cache"):
            owner, name = {"dense_2": (lin, "forward"), "norm1": (blk.norm1, "forward"), "forward_rows": (blk.mlp, "forward_rows"),
                           "forward_last": (blk.attn, "forward_last"), "cache": (blk.attn.kv_cache, "attend")}[how]
            method = getattr(owner, name)
            setattr(owner, name, lambda *a, **k: (calls.append(name), method(*a, **k))[1])
        elif how == "activation_hook":
            blk.mlp.activation.register_forward_pre_hook(lambda m, a: calls.append(m))
        else:
            lin._parameters["weight"] = lin.weight.detach().as_subclass(Counted)
        try:
            out = blk._native_decode(x[:, :1])
            assert out is None and blk._history.cur == 8 and blk.attn.kv_cache.lens.tolist() == [8, 5]
            del calls[:]
            blk(x[:, :1], first_cache=False)
        finally:
            if handle is not None:
                handle.remove()
    assert calls and blk._history.cur == 9 and blk.attn.kv_cache.lens.tolist() == [9, 6]


@pytest.mark.parametrize("act", [F.relu, F.gelu, torch.nn.GELU(approximate="tanh")])
def test_block_decode_keeps_nan(act):
    """A NaN that appears inside the MLP is in the decode step's output, whatever the activation."""
    _, M = _mods()
    blk = M.Block1D(128, 2, 2.0, activation=act, dtype=torch.float16, max_seq_len=32).cuda()
    _init(blk, 52)
    announce("block decode NaN", act)
    x = torch.randn(2, 8, 128, dtype=torch.float16, device="cuda")
    with torch.no_grad():
        blk.mlp.dense_1.bias[5] = float("nan")
        blk(x, first_cache=True, seq_lens=torch.tensor([8, 5], dtype=torch.int32, device="cuda"))
        out = blk._native_decode(x[:, :1])
    assert out[:, -1].isnan().all()


@pytest.mark.parametrize("how", ["gelu_subclass", "relu_subclass", "replaced_after_construction"])
def test_block_decode_applies_the_activation_that_prefill_applies(how):
    """Prompt and decode steps of a block go through one function: a module derived from GELU or ReLU runs its own forward,
    and an activation put in later leaves the epilogue that the MLP was built with."""
    _, M = _mods()
    announce("block decode activation", how)
    if how == "replaced_after_construction":
        act = F.relu
    else:
        base = torch.nn.GELU if how == "gelu_subclass" else torch.nn.ReLU
        act = type("Own", (base,), {"forward": lambda self, h: 1.5 * torch.sigmoid(h)})()
    blk = M.Block1D(128, 2, 2.0, activation=act, dtype=torch.float16, max_seq_len=32).cuda()
    _init(blk, 53)
    if how == "replaced_after_construction":
        blk.mlp.activation = F.gelu
    p, lens = _fp32_params(blk), [8, 5]
    x, valid = _padded_batch(2, 8, 128, lens, True, torch.float16, 54)
    new = torch.randn(2, 1, 128, generator=torch.Generator().manual_seed(55)).half()
    with torch.no_grad():
        blk(x.cuda(), attention_mask=models.additive_mask(valid).half().cuda(), first_cache=True)
        got = blk(new.cuda(), first_cache=False)
    x, valid = torch.cat((x, new), 1), torch.cat((valid, torch.ones(2, 1)), 1)
    want = models.block_forward(x, p, 2, 1e-5, False, True, models.additive_mask(valid), activation=act)
    assert max_abs(got[:, -1].float().cpu(), want[:, -1]) <= 1.5e-2      # the bound of the block's decode steps above


@pytest.mark.parametrize("shape", [(2, 0, 128), (0, 1, 128)])
def test_block_decode_refuses_a_batch_without_a_newest_position(shape):
    """No newest position: nothing is launched on a pointer in front of the tensor, and the general step refuses the call."""
    _, M = _mods()
    announce("block decode, empty", shape)
    blk = M.Block1D(128, 2, 2.0, activation=F.relu, dtype=torch.float16, max_seq_len=32).cuda()
    with torch.no_grad():
        blk(torch.randn(2, 8, 128, device="cuda").half(), first_cache=True,
            seq_lens=torch.tensor([8, 5], dtype=torch.int32, device="cuda"))
        empty = torch.empty(shape, dtype=torch.float16, device="cuda")
        assert blk._native_decode(empty) is None
        with pytest.raises(RuntimeError):
            blk(empty, first_cache=False)
    assert blk._history.cur == 8 and blk.attn.kv_cache.lens.tolist() == [8, 5]


@pytest.mark.parametrize("name", ["attn.query_key_value", "mlp.dense_1", "mlp.dense_2"])
def test_block_decode_refuses_weights_laid_out_the_other_way(name):
    """A weight of [in, out] has as many elements as one of [out, in] and is refused, as the library's projection refuses it."""
    _, M = _mods()
    announce("block decode, transposed weight", name)
    blk = M.Block1D(128, 2, 2.0, activation=F.gelu, dtype=torch.float16, max_seq_len=32).cuda()
    with torch.no_grad():
        x = torch.randn(2, 8, 128, device="cuda").half()
        blk(x, first_cache=True, seq_lens=torch.tensor([8, 5], dtype=torch.int32, device="cuda"))
        lin = blk.get_submodule(name)
        lin.weight = torch.nn.Parameter(lin.weight.t().contiguous())
        assert blk._native_decode(x[:, -1:]) is None
        with pytest.raises(RuntimeError):
            blk(x[:, -1:], first_cache=False)
