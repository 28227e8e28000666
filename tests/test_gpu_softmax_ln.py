"""GPU parity: scale_mask_softmax and the fused LayerNorm against the fp32/fp64 oracle.

Tolerance (from the north-star statement): max-abs error <= 2e-3 against the
fp32 oracle for fp16 storage; fp32 storage must reach 1e-5.  bf16 storage is
held to its own rounding step (2^-8 relative).
"""
import pytest
import torch

from gpu_util import BASE, announce, assert_stored_close, max_abs, ragged_lens
from oracle import eager

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 3.2e-2}


def _kernel():
    from energonai_amd import kernel
    return kernel


def _valid_row_mask(B, H, Sq, Sk, q_lens):
    m = torch.zeros(B, H, Sq, Sk, dtype=torch.bool)
    for b, n in enumerate(q_lens):
        m[b, :, :n] = True
    return m


SOFTMAX_CASES = [
    # B, H, S, lens
    (8, 12, 128, [24, 127, 31, 65, 24, 127, 31, 65]),
    (2, 3, 8, [8, 1]),
    (3, 2, 40, [40, 0, 7]),
    (2, 2, 512, [300, 512]),
    (2, 1, 1024, [1024, 513]),
    (1, 2, 2048, [1500]),          # above the reference's 1024 limit
    (1, 1, 4096, [4096]),
    (2, 2, 37, [37, 5]),           # row length not a multiple of the vector
    (1, 1, 8200, [8200]),          # too long for registers (fp32): generic kernel
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,S,lens", SOFTMAX_CASES)
def test_softmax_reference_semantics(dtype, B, H, S, lens):
    """Five-argument call: causal, no scale, padded rows untouched, in place, same tensor returned."""
    k = _kernel()
    announce("softmax ref", dtype, B, H, S, lens)
    g = torch.Generator().manual_seed(S + B)
    src = (3.0 * torch.randn(B, H, S, S, generator=g)).to(dtype)
    want = eager.scale_mask_softmax(B, S, H, src.float(), lens, out_dtype=torch.float32)
    x = src.clone().cuda()
    out = k.scale_mask_softmax(B, S, H, x, torch.tensor(lens, dtype=torch.int32).cuda())
    assert out.data_ptr() == x.data_ptr(), "must be in place and return its input"
    got = out.cpu()
    valid = _valid_row_mask(B, H, S, S, lens)
    err = max_abs(got[valid].float(), want[valid])
    assert err <= TOL[dtype], err
    # padded query rows hold their raw scores, bit for bit (csrc/scale_mask_softmax_kernel.cu:14-17)
    assert torch.equal(got[~valid], src[~valid])
    # the zero tail is exact and valid rows sum to one
    for b, n in enumerate(lens):
        for q in (0, n // 2, n - 1):
            if 0 <= q < n:
                assert bool((got[b, :, q, q + 1:] == 0).all())
                assert abs(got[b, :, q].float().sum(-1) - 1).max() < 4 * TOL[dtype] + 1e-3 * (dtype != torch.float32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_softmax_scale_and_noncausal(dtype, causal):
    k = _kernel()
    B, H, S = 4, 3, 96
    lens = [96, 1, 50, 17]
    scale = 0.125
    announce("softmax scale", dtype, causal)
    g = torch.Generator().manual_seed(5)
    src = (8.0 * torch.randn(B, H, S, S, generator=g)).to(dtype)
    want = eager.scale_mask_softmax(B, S, H, src.float(), lens, scale=scale, causal=causal, out_dtype=torch.float32)
    got = k.scale_mask_softmax(B, S, H, src.clone().cuda(), torch.tensor(lens).cuda(), scale=scale,
                               causal=causal).cpu()
    valid = _valid_row_mask(B, H, S, S, lens)
    assert max_abs(got[valid].float(), want[valid]) <= TOL[dtype]
    if not causal:
        for b, n in enumerate(lens):
            assert bool((got[b, :, :n, n:] == 0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_softmax_rectangular_decode(dtype):
    """One query row per sequence against a longer ragged key axis."""
    k = _kernel()
    B, H, Sk = 5, 4, 640
    kv = [640, 1, 333, 64, 65]
    announce("softmax decode", dtype)
    g = torch.Generator().manual_seed(6)
    src = (4.0 * torch.randn(B, H, 1, Sk, generator=g)).to(dtype)
    want = eager.scale_mask_softmax(B, 1, H, src.float(), kv, scale=0.5, causal=True, k_seq_len=Sk,
                                    q_lens=[1] * B, out_dtype=torch.float32)
    got = k.scale_mask_softmax(B, 1, H, src.clone().cuda(), torch.tensor(kv, dtype=torch.int32).cuda(), scale=0.5,
                               k_seq_len=Sk, q_len_list=torch.ones(B, dtype=torch.int32).cuda()).cpu()
    assert max_abs(got.float(), want) <= TOL[dtype]
    # q_len_list omitted: defaults to min(k_len, Sq) = 1
    got2 = k.scale_mask_softmax(B, 1, H, src.clone().cuda(), torch.tensor(kv, dtype=torch.int32).cuda(), scale=0.5,
                                k_seq_len=Sk).cpu()
    assert torch.equal(got, got2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])                       # elements between a 16-byte boundary and the first row
@pytest.mark.parametrize("Sq,Sk,lens", [
    (1, 1, [1]), (7, 7, [7, 3]), (301, 301, [301, 40, 0]),      # shorter than a vector; all bands of 16-bit rows
    (5, 8, [8, 5]), (6, 509, [509, 6]), (6, 511, [511, 128]),
    (4, 513, [513]), (4, 1023, [1023, 4]), (4, 1025, [1025]), (4, 2047, [2047]), (4, 2049, [2049, 1024]),
    (3, 4097, [4096]), (3, 8191, [8191, 17]), (2, 8193, [8193]),    # up to and past what the registers hold
    (9, 9, [30, 9]), (130, 130, [5000, 77]),                        # key lengths past the row
])
def test_softmax_rows_off_the_16_byte_boundaries(dtype, shift, Sq, Sk, lens):
    """Rows at any element's address against float64, the tail zeroed to the row's end and nothing else touched.

    Bound: half an ulp of a probability of at most one (2^-12, 2^-9) for 16 bits; in fp32 the argument of the exponential
    is rounded at its size (|x| <= 16: 2^-20) and the sum once per addition."""
    k = _kernel()
    H = 2
    B = len(lens)
    announce("softmax unaligned", dtype, shift, Sq, Sk, lens)
    g = torch.Generator().manual_seed(Sq * Sk + shift)
    n = B * H * Sq * Sk
    flat = (3.0 * torch.randn(n + 32, generator=g)).clamp(-16, 16).to(dtype)
    buf = flat.clone().cuda()
    src = flat[shift:shift + n].view(B, H, Sq, Sk)
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()
    ql = [min(x, Sq) for x in lens]
    k.scale_mask_softmax(B, Sq, H, buf[shift:shift + n].view(B, H, Sq, Sk), lens_t, scale=0.37, k_seq_len=Sk,
                         q_len_list=torch.tensor(ql, dtype=torch.int32).cuda())
    after = buf.cpu()
    assert torch.equal(after[:shift], flat[:shift]) and torch.equal(after[shift + n:], flat[shift + n:])
    got = after[shift:shift + n].view(B, H, Sq, Sk)
    tol = {torch.float32: 2e-6, torch.float16: 2.0 ** -12 + 2e-6, torch.bfloat16: 2.0 ** -9 + 2e-6}[dtype]
    for b in range(B):
        assert torch.equal(got[b, :, ql[b]:], src[b, :, ql[b]:])
        for q in range(ql[b]):
            vis = q + min(lens[b], Sk) - ql[b] + 1
            want = torch.softmax(src[b, :, q, :vis].double() * 0.37, -1)
            assert max_abs(got[b, :, q, :vis].double(), want) <= tol, (b, q)
            assert not got[b, :, q, vis:].any()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("scale", [0.5, -0.5])                  # a scale that is not positive: the general kernel
@pytest.mark.parametrize("Sq,Sk", [(9, 9), (16, 16), (40, 24), (3, 1031), (2, 2056), (2, 8200)])
def test_softmax_of_key_lengths_past_the_row(Sq, Sk, scale, causal):
    """A key length past the row means the whole row, in every kernel: the bits of the length cut to it."""
    k = _kernel()
    announce("softmax lengths past the row", Sq, Sk, scale, causal)
    src = torch.randn(2, 2, Sq, Sk, generator=torch.Generator().manual_seed(Sk)).half().cuda()
    for q_lens in (None, torch.tensor([Sq, 1], dtype=torch.int32).cuda()):
        got, want = (k.scale_mask_softmax(2, Sq, 2, src.clone(), torch.tensor(lens, dtype=torch.int32).cuda(), scale=scale, causal=causal,
                                          k_seq_len=Sk, q_len_list=q_lens) for lens in ([Sk + 21, 5000], [Sk, min(5000, Sk)]))
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [9, 515])
def test_softmax_odd_rows_of_extreme_scores(dtype, S):
    """Rows of the type's lowest value, of -inf, and with one of either: as the definition has it."""
    k = _kernel()
    announce("softmax extremes", dtype, S)
    low = torch.finfo(dtype).min
    src = torch.zeros(1, 1, S, S, dtype=dtype)
    src[..., 4, :] = low
    src[..., 5, :] = -float("inf")
    src[..., 6, 1:] = low
    src[..., 7, 2:] = -float("inf")
    got = k.scale_mask_softmax(1, S, 1, src.clone().cuda(), torch.tensor([S], dtype=torch.int32).cuda(), scale=0.5,
                               causal=False).cpu()[0, 0]
    want = torch.full((S, S), 1.0 / S, dtype=torch.float64)
    want[5] = 0                                     # nothing to see: zeros, no NaN
    want[6], want[7] = 0, 0
    want[6, 0], want[7, :2] = 1, 0.5
    assert max_abs(got.double(), want) <= {torch.float32: 1e-6, torch.float16: 2e-4, torch.bfloat16: 2e-3}[dtype]


def test_softmax_rectangular_chunked_prefill():
    """Sq < Sk with several query rows: queries are the last q_len positions."""
    k = _kernel()
    B, H, Sq, Sk = 3, 2, 16, 128
    kl, ql = [128, 40, 9], [16, 8, 9]
    announce("softmax chunk")
    g = torch.Generator().manual_seed(8)
    src = torch.randn(B, H, Sq, Sk, generator=g)
    want = eager.scale_mask_softmax(B, Sq, H, src, kl, causal=True, k_seq_len=Sk, q_lens=ql)
    got = k.scale_mask_softmax(B, Sq, H, src.clone().cuda(), torch.tensor(kl, dtype=torch.int32).cuda(),
                               k_seq_len=Sk, q_len_list=torch.tensor(ql, dtype=torch.int32).cuda()).cpu()
    valid = _valid_row_mask(B, H, Sq, Sk, ql)
    assert max_abs(got[valid], want[valid]) <= 1e-5
    assert torch.equal(got[~valid], src[~valid])


LN_CASES = [
    # n1, n2
    (698, 768), (64, 9216), (33, 7168), (20, 12288), (5, 1024), (7, 8), (3, 16384),
    (4, 40000),      # wide row: 1024-lane kernel
    (4100, 7168),    # 896 fp16 vectors and many rows: 512 lanes x 2 vectors (fp32: 1792 vectors, 512 x 4)
    (4097, 4000),    # fp32: 1000 vectors and many rows: 512 lanes x 2; fp16: 500 vectors on 256 lanes
    (3, 100),        # fp16: 100 % 8 != 0 -> generic kernel
    (2, 70001),      # too wide / odd: generic kernel
]
LN_DTYPES = [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
             (torch.float32, torch.float16), (torch.float32, torch.bfloat16)]


@pytest.mark.parametrize("in_dtype,out_dtype", LN_DTYPES)
@pytest.mark.parametrize("n1,n2", LN_CASES)
@pytest.mark.parametrize("with_residual", [False, True])
def test_layernorm(in_dtype, out_dtype, n1, n2, with_residual):
    k = _kernel()
    announce("layernorm", in_dtype, out_dtype, n1, n2, with_residual)
    g = torch.Generator().manual_seed(n2 % 1000 + n1)
    x = (torch.randn(1, n1, n2, generator=g) * 1.5 + 0.3).to(in_dtype)
    r = torch.randn(1, n1, n2, generator=g).to(in_dtype) if with_residual else None
    gamma = (1 + 0.02 * torch.randn(n2, generator=g)).to(out_dtype)
    beta = (0.02 * torch.randn(n2, generator=g)).to(out_dtype)
    want, mean, invvar, xsum = eager.layer_norm(x, gamma, beta, 1e-5, residual=r, acc_dtype=torch.float64,
                                                out_dtype=torch.float64)
    res = k.layer_norm_forward(x.cuda(), gamma.cuda(), beta.cuda(), (n2,), 1e-5,
                               residual=None if r is None else r.cuda(), return_stats=True, return_sum=True)
    y, m, iv, s = (t.cpu() for t in res)
    assert y.dtype == out_dtype and y.shape == x.shape
    assert m.dtype == torch.float32 and m.shape == (n1,)
    # fp32 arithmetic (1e-5 relative to the row's largest value) on top of the one rounding of the stored output
    assert_stored_close(y, want, out_dtype, base=1e-5 * max(1.0, float(want.abs().max())), what="LayerNorm output")
    assert max_abs(m, mean) <= 1e-5
    assert ((iv.double() - invvar.double()).abs() / invvar.double()).max() <= 1e-5
    # the emitted residual stream is the fp32 sum rounded once to the input dtype
    xsum32 = x.float() if r is None else x.float() + r.float()
    assert torch.equal(s, xsum32.to(in_dtype))
    assert max_abs(s, xsum) <= TOL[in_dtype] * max(1.0, float(xsum.abs().max()) / 2)


def test_layernorm_fp16_single_rounding():
    """fp16 output equals the fp64 result rounded once to fp16 in all but a sliver of entries."""
    k = _kernel()
    n1, n2 = 256, 12288
    announce("layernorm single rounding")
    g = torch.Generator().manual_seed(12)
    x = torch.randn(n1, n2, generator=g).half()
    gamma = (1 + 0.02 * torch.randn(n2, generator=g)).half()
    beta = (0.02 * torch.randn(n2, generator=g)).half()
    want64, _, _, _ = eager.layer_norm(x, gamma, beta, 1e-5, acc_dtype=torch.float64, out_dtype=torch.float64)
    y = k.layer_norm_forward(x.cuda(), gamma.cuda(), beta.cuda(), (n2,), 1e-5).cpu()
    assert_stored_close(y, want64, torch.float16, base=1e-5 * float(want64.abs().max()), what="LayerNorm output")
    frac_exact = (y == want64.half()).double().mean().item()
    assert frac_exact > 0.995, frac_exact


def test_layernorm_module_matches_reference_interface():
    from energonai_amd.kernel.cuda_native import LayerNorm
    announce("layernorm module")
    ln = LayerNorm(768, eps=1e-5, dtype=torch.float16).cuda()
    assert repr(ln) == "MixedFusedLayerNorm(normalized_shape=torch.Size([768]), eps=1e-05)"
    assert torch.equal(ln.weight.detach().cpu(), torch.ones(768, dtype=torch.float16))
    assert torch.equal(ln.bias.detach().cpu(), torch.zeros(768, dtype=torch.float16))
    x = torch.randn(2, 5, 768, generator=torch.Generator().manual_seed(1)).half()
    with torch.inference_mode():
        y = ln(x.cuda()).cpu()
    want = torch.nn.functional.layer_norm(x.float(), (768,), eps=1e-5)
    assert_stored_close(y, want, torch.float16, base=1e-5 * float(want.abs().max()), what="LayerNorm module")
    # constant row -> beta (here zero)
    with torch.inference_mode():
        z = ln(torch.full((3, 768), 2.5, dtype=torch.float16).cuda()).cpu()
    assert bool((z == 0).all())
    with pytest.raises(RuntimeError, match="expected input with shape"):
        ln(torch.zeros(2, 100, dtype=torch.float16).cuda())


@pytest.mark.parametrize("tile", [128, 32, 1])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("scale", [0.5, -0.5])
def test_softmax_tiled_tail(dtype, causal, tile, scale):
    """tail_rows=t: valid entries identical to the full-tail result, zeros up to the extent of the row's
    t-row query tile (completed to a whole 16-byte vector), everything beyond left untouched.  t = 1 (the form
    in the step) writes no tail beyond that vector.  A negative scale takes the three-pass kernel, which must
    leave the same bytes."""
    k = _kernel()
    B, H, S = 3, 2, 512
    lens = [512, 130, 300]
    announce("softmax tiled tail", dtype, causal, tile, scale)
    g = torch.Generator().manual_seed(21)
    src = (3.0 * torch.randn(B, H, S, S, generator=g)).to(dtype)
    lens_t = torch.tensor(lens, dtype=torch.int32).cuda()
    epv = 16 // src.element_size()
    full = k.scale_mask_softmax(B, S, H, src.clone().cuda(), lens_t, scale=scale, causal=causal).cpu()
    tiled = k.scale_mask_softmax(B, S, H, src.clone().cuda(), lens_t, scale=scale, causal=causal, tail_rows=tile).cpu()
    want = eager.scale_mask_softmax(B, S, H, src.float(), lens, scale=scale, causal=causal, out_dtype=torch.float32)
    valid = _valid_row_mask(B, H, S, S, lens)
    assert max_abs(full[valid].float(), want[valid]) <= TOL[dtype]
    for b, n in enumerate(lens):
        for q0 in range(0, n, tile):
            rows = min(tile, n - q0)
            lim = min(n, q0 + rows) if causal else n
            lim_v = -(-lim // epv) * epv   # whole vectors are written
            assert torch.equal(tiled[b, :, q0:q0 + rows, :lim], full[b, :, q0:q0 + rows, :lim])
            assert bool((tiled[b, :, q0:q0 + rows, lim:lim_v] == 0).all())
            assert torch.equal(tiled[b, :, q0:q0 + rows, lim_v:], src[b, :, q0:q0 + rows, lim_v:])
        assert torch.equal(tiled[b, :, n:], src[b, :, n:])


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("vectors", [1, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 512, 513, 768, 769, 1024, 1025, 1536,
                                     1537, 2048, 2049, 3073, 4097, 6145, 8192, 8193])
def test_layernorm_at_the_edges_of_its_lane_configurations(dtype, vectors):
    """Row widths on either side of every lanes x vectors instance, with residual, row offsets, sum and statistics; the
    reference is LayerNorm in float64 and the bound the module's: BASE plus half an ulp of the stored value."""
    from energonai_amd import kernel as K
    epv = 16 // torch.empty(0, dtype=dtype).element_size()
    width, rows = vectors * epv, 7
    announce("layernorm lane edges", dtype, width)
    g = torch.Generator().manual_seed(vectors)
    x, res = torch.randn(rows, width, generator=g).to(dtype), torch.randn(rows + 5, width, generator=g).to(dtype)
    gamma, beta = (1 + 0.02 * torch.randn(width, generator=g)).to(dtype), (0.02 * torch.randn(width, generator=g)).to(dtype)
    off = torch.tensor([0, 0, 1, 1, 3, 5, 5], dtype=torch.int32)
    s = x.double() + res[torch.arange(rows) + off].double()
    want = torch.nn.functional.layer_norm(s, (width,), gamma.double(), beta.double(), 1e-5)
    y, mean, inv, total = K.layer_norm_forward(x.cuda(), gamma.cuda(), beta.cuda(), (width,), 1e-5, residual=res.cuda(),
                                               return_stats=True, return_sum=True, residual_row_offsets=off.cuda())
    assert_stored_close(y.cpu(), want, dtype)
    assert torch.equal(total.cpu(), (x.float() + res[torch.arange(rows) + off].float()).to(dtype))
    assert max_abs(mean.cpu(), s.mean(-1)) <= 1e-5
    assert max_abs(inv.cpu() * s.var(-1, unbiased=False).add(1e-5).sqrt(), torch.ones(rows)) <= 1e-5


@pytest.mark.parametrize("with_residual", [False, True])
@pytest.mark.parametrize("dtype,rows,width", [
    (torch.float16, 6000, 9216),        # 105 MB: written past the memory-side cache; read out of it without a residual
    (torch.float16, 1001, 65536),       # the same with eight vectors on each of 1024 lanes
    (torch.float32, 4000, 8192),        # four vectors on 512 lanes
    (torch.float32, 1000, 36864),       # 147 MB: input and output together pass the cache's 256 MB
])
def test_layernorm_of_tensors_around_the_size_of_the_memory_side_cache(dtype, rows, width, with_residual):
    """Outputs of 96 MB and more, with inputs that fit the cache beside them and inputs that do not, in every lane of a row;
    reference and bound as above (the reference in float32: its own error is a few 1e-7 of values up to 6)."""
    from energonai_amd import kernel as K
    announce("layernorm large", dtype, rows, width, with_residual)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, res = (torch.randn(rows, width, generator=g, device="cuda").to(dtype) for _ in range(2))
    gamma, beta = ((c + 0.02 * torch.randn(width, generator=g, device="cuda")).to(dtype) for c in (1.0, 0.0))
    got = K.layer_norm_forward(x, gamma, beta, (width,), 1e-5, residual=res if with_residual else None)
    s = x.float() + res.float() if with_residual else x.float()
    want = torch.nn.functional.layer_norm(s, (width,), gamma.float(), beta.float(), 1e-5)
    for part in (slice(0, 64), slice(rows // 2, rows // 2 + 64), slice(rows - 64, rows)):
        assert_stored_close(got[part].cpu(), want[part].cpu(), dtype)
    assert float((got.float() - want).abs().max()) <= BASE[dtype] + 2.0 ** -9 * float(want.abs().max())
