"""The quantizers' and producers' kernels at the sizes and values where each branch can go wrong, against the
CPU oracle (or, for a call that several routes can take, against the general route)."""
import numpy as np
import pytest
import torch

from helpers import FP8_DT, TORCH_DT, f32
from oracle import formats as OF


def _u8(t):
    return t.contiguous().view(torch.uint8).cpu().numpy()


def _edge_floats():
    """fp32 values at the fp8 formats' edges: every 16-bit pattern as the upper half, the midpoints between
    neighbouring codes and one ulp to each side, both signs, infinities and NaNs of both signs."""
    top = (np.arange(1 << 16, dtype=np.uint32) << 16)
    mid = top | 0x8000
    parts = [top, top + 1, top - 1, mid, mid + 1, mid - 1, np.array([0x7FC00000, 0xFFC00000, 0x7F800001, 0xFF800001], np.uint32)]
    return np.concatenate(parts).view(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["e4m3fn", "e5m2"])
def test_fp8_bytes_of_edge_values(gpu, fmt):
    """base = fp8(k) byte for byte, NaN signs included (the residual of a NaN or an overflow is a NaN whose
    sign the subtraction does not define: compared where the base is finite)."""
    from ffa_mi355x import kfmt_quant as KQ

    x = _edge_floats()
    base, res = KQ.quantize_fp8fp8(torch.from_numpy(x.copy()).to(gpu), FP8_DT[fmt])
    with np.errstate(invalid="ignore", over="ignore"):
        ob, orr = OF.quantize_fp8fp8(x, fmt)
    assert np.array_equal(_u8(base), ob)
    fine = (ob & 0x7F) < (0x7F if fmt == "e4m3fn" else 0x7C)
    assert np.array_equal(_u8(res)[fine], orr[fine])


# ------------------------------------------------------------------- per-channel 2-bit quantizer
def _misaligned(k):
    """The same values at an address that is no multiple of 16 bytes (the scalar kernels' route)."""
    flat = torch.empty(k.numel() + 1, dtype=k.dtype, device=k.device)
    flat[1:] = k.reshape(-1)
    return flat[1:].view(k.shape)


def _next(x, tau, n):
    """x moved by n representable values of tau (x positive)."""
    if tau == "fp32":
        return (x.view(torch.int32) + n).view(torch.float32)
    return (x.view(torch.int16) + n).view(x.dtype)


def test_q2_code_turning_points():
    """The closed form the vector quantizer compares against (the middles of the tau values around 0.5, 1.5 and
    2.5, times the scale) gives, for every 16-bit scale and a sample of fp32 ones, the code that the division gives
    on both sides of every turn."""
    g = torch.Generator().manual_seed(5)
    for tau in ("bf16", "fp16", "fp32"):
        dt, p = TORCH_DT[tau], {"bf16": 8, "fp16": 11, "fp32": 24}[tau]
        if tau == "fp32":
            sc = torch.rand(20000, generator=g) * torch.exp2(torch.randint(-20, 20, (20000,), generator=g).float())
            sc = torch.cat([sc.clamp_min(3e-7), torch.exp2(torch.arange(-20, 20).float())])
        else:
            sc = torch.arange(1, 0x7C00 if tau == "fp16" else 0x7F00, dtype=torch.int16).view(dt)
            sc = sc[(sc.float() >= 3e-7) & (sc.float() < 1e4)]
        h = 2.0 ** -p
        for i, q in enumerate((0.5 + h / 2, 1.5 - h, 2.5 + 2 * h)):
            v = sc.double() * q
            t = v.float()
            up = t.double() < v if i == 1 else t.double() <= v
            t = torch.where(up, (t.view(torch.int32) + 1).view(torch.float32), t)
            near = (sc.float() * (i + 0.5)).to(dt)
            for n in range(-3, 4):
                x = _next(near, tau, n)
                code = torch.round(x / sc).clamp(0, 3)  # the reference's ops in tau
                assert torch.equal(x.float() >= t, code.float() >= i + 1), (tau, i, n)



@pytest.mark.gpu
@pytest.mark.parametrize("tau", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("fmt", ["e4m3fn", "e5m2"])
def test_q2_quantizer_turning_points_bit_exact(gpu, tau, fmt):
    """Keys on and next to every code's turning point of 4096 scales, against the oracle."""
    from ffa_mi355x.quant import quantize_per_channel
    from oracle import q2fp8 as OQ

    dt = TORCH_DT[tau]
    g = torch.Generator().manual_seed(11)
    sc = (torch.rand(4, 8, 128, generator=g) * 4 + 0.01).to(dt)
    rows = [torch.zeros_like(sc), (sc.float() * 3).to(dt)]  # zero 0, scale tau(tau(3 sc) / 3)
    s1 = (rows[1] / 3.0)
    for mid in (0.5, 1.5, 2.5):
        rows += [_next((s1.float() * mid).to(dt), tau, n) for n in range(-3, 4)]
    k = torch.stack(rows, 1)  # [4, T, 8, 128]
    kq, ks, kz, kr = quantize_per_channel(k.to(gpu), FP8_DT[fmt])
    oq, os_, oz, orr = OQ.quantize_per_channel(f32(k), tau, fmt)
    assert np.array_equal(_u8(kq), oq) and np.array_equal(_u8(kr), orr)
    assert np.array_equal(f32(ks), os_) and np.array_equal(f32(kz), oz)


@pytest.mark.gpu
@pytest.mark.parametrize("tau", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("B,T,HKV,D", [(1, 1, 1, 8), (2, 257, 3, 24), (1, 300, 2, 12), (3, 17, 5, 64), (1, 2500, 8, 128),
                                       (2, 129, 9, 128)])
def test_q2_quantizer_vector_route_equals_scalar_route(gpu, tau, B, T, HKV, D):
    """Every byte of the vector kernels' route equals the scalar route's, tails of columns, rows and splits,
    infinities and NaNs among them."""
    from ffa_mi355x.quant import quantize_per_channel

    g = torch.Generator().manual_seed(B * 1000 + T)
    k = (torch.randn(B, T, HKV, D, generator=g) * 3).to(TORCH_DT[tau])
    if T > 16:
        k[0, 3, 0, 1], k[0, 5, 0, 2], k[-1, 7, HKV - 1, 3], k[0, 9, 0, 4] = float("inf"), float("-inf"), float("nan"), 0.0
        k[0, 11, 0, 5:7] = 6e4
        k[0, 12, 0, 6] = -6e4
    k = k.to(gpu)
    for fp8 in (torch.float8_e5m2, torch.float8_e4m3fn):
        a, b = quantize_per_channel(k, fp8), quantize_per_channel(_misaligned(k), fp8)
        for x, y in zip(a, b):
            assert np.array_equal(_u8(x), _u8(y))


# ------------------------------------------------------------------- K projection + RoPE
@pytest.mark.gpu
@pytest.mark.parametrize("h_dt", ["bf16", "fp16"])
@pytest.mark.parametrize("B,T,HKV,D,H,cs32,bias", [
    (1, 4100, 8, 128, 1088, True, False),   # 128 x 64 tiles (33 x 16), 17 steps folded by 2, ragged last tile row
    (1, 6200, 8, 128, 1088, True, False),   # 128 x 128 (49 x 8), the same
    (2, 2048, 8, 128, 2112, False, True),   # 128 x 128, 33 steps folded by 4, two sequences
    (1, 4200, 35, 32, 1216, True, True),    # 128 x 128 (33 x 9), a ragged last column, grid not a multiple of 8
    (3, 700, 8, 128, 4160, True, True),     # 128 x 64 (17 x 16), 65 steps folded by 8
    (1, 1030, 8, 128, 1024, False, False),  # 64 x 64 (17 x 16), the shortest K of the tiles
    (1, 290, 7, 128, 1152, True, False),    # 32 x 64 (10 x 14)
    (1, 4100, 8, 128, 64, True, False),     # H below 1024: the 16 x 32 kernel
    (2, 2048, 8, 128, 576, False, True),
    (1, 300, 8, 96, 1056, True, False),     # H no multiple of 64: the 16 x 32 kernel
])
def test_kproj_rope_tiles(gpu, h_dt, B, T, HKV, D, H, cs32, bias):
    """Every tile size of the projection against fp64.  The projection is rounded to h's type from fp32 sums: equal
    to the rounding of the fp64 product but where that lies within the sums' error of a rounding boundary, which
    moves it by one ulp of h's type (2^-8 or 2^-11 relative, at most 2^-7 / 2^-10 of the pair through RoPE, and
    one rounding more to a 16-bit result).  The sums' error is about 2^-22 of the terms' size: fewer than 1 in 100
    elements can be so near."""
    from ffa_mi355x import kfmt_quant as KQ

    dt = TORCH_DT[h_dt]
    g = torch.Generator().manual_seed(T)
    h = torch.randn(B, T, H, generator=g).to(dt).to(gpu)
    w = (torch.randn(HKV * D, H, generator=g) / H ** 0.5).to(dt).to(gpu)
    bv = torch.randn(HKV * D, generator=g).to(dt).to(gpu) if bias else None
    ang = torch.rand(T, D, generator=g) * 6.28
    cos, sin = (x.to(torch.float32 if cs32 else dt).to(gpu) for x in (ang.cos(), ang.sin()))
    k = KQ.kproj_rope(h, w, cos, sin, HKV, D, bias=bv)
    lin = h.double() @ w.double().t().contiguous()
    lin = (lin if bv is None else lin + bv.double()).to(dt).view(B, T, HKV, D)
    rot = torch.stack((-lin[..., 1::2], lin[..., ::2]), -1).flatten(-2)
    ref = lin * cos[None, :, None] + rot * sin[None, :, None]
    assert k.dtype == ref.dtype
    off = (k.double() - ref.double()).abs()
    pair = lin.double().abs() + rot.double().abs()
    ulp = 2.0 ** (-7 if h_dt == "bf16" else -10)
    assert float((off > 0).float().mean()) < 1e-2
    assert bool((off <= ulp * pair * (1 if cs32 else 2) + 1e-30).all())


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1024, 2048, 4096])
def test_kproj_rope_tiles_round_as_the_split(gpu, H):
    """The tiles' sums are as exact as the split kernel's (taken for misaligned cos): of the 2 M products, as many
    round to another fp16 value than the 64-bit ones do.  The counts are 1500 to 2600, so that their difference has
    a standard deviation of at most 3.6 % (sqrt(2 n)); chains twice as long gave 36 % more at H = 1024."""
    from ffa_mi355x import kfmt_quant as KQ

    T = 2048
    g = torch.Generator(device=gpu).manual_seed(H)
    h = torch.randn((1, T, H), generator=g, device=gpu).half()
    w = (torch.randn((1024, H), generator=g, device=gpu) * 0.02).half()
    cos, sin = torch.ones((T, 128), device=gpu), torch.zeros((T, 128), device=gpu)
    ref = (h[0].double() @ w.double().t().contiguous()).half().float()
    tile, split = (int((KQ.kproj_rope(h, w, c, sin, 8, 128).view(T, 1024) != ref).sum())
                   for c in (cos, _misaligned(cos)))
    assert tile <= 1.15 * split


# ------------------------------------------------------------------- paged cache -> contiguous
@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["e4m3fn", "e5m2"])
@pytest.mark.parametrize("v_dt", ["fp16", "bf16"])
def test_paged_dequantize_every_type(gpu, fmt, v_dt):
    """Every residual, V and output type, lengths at page edges (0, 1, 63, 64, 65 tokens of the last page): fp32
    fma(code, scale, zero) + residual of the pool's own bytes, rounded once."""
    from ffa_mi355x.paged import CODES_ORDER, GSCALE_ORDER, RES_ORDER, VT_ORDER, PagedQ2Cache, scale_pos, to_logical

    lens = [192, 129, 127, 65, 64, 1, 0]
    B, HKV, npg = len(lens), 3, 3
    g = torch.Generator().manual_seed(4)
    cache = PagedQ2Cache(B * npg, HKV, gpu, res_dtype=FP8_DT[fmt], v_dtype=TORCH_DT[v_dt])
    bt = torch.randperm(B * npg, generator=g).view(B, npg).int()
    k, v = (torch.randn(B, 192, HKV, 128, generator=g).to(gpu) for _ in range(2))
    cache.append(k, v, torch.zeros(B, dtype=torch.int32, device=gpu), bt.to(gpu))
    codes = to_logical(cache.k_q.cpu().numpy(), CODES_ORDER, 8)  # [P, H, 4, 64, 8]
    bits = (codes[..., None] >> np.array([0, 2, 4, 6], np.uint8)) & 3
    c = bits.reshape(codes.shape[:-1] + (32,)).transpose(0, 1, 3, 2, 4).astype(np.float32)  # [P, H, 64, 4, 32]
    sz = [to_logical(x.cpu().numpy(), GSCALE_ORDER)[..., scale_pos(np.arange(64))].transpose(0, 1, 3, 2)[..., None]
          .astype(np.float32) for x in (cache.k_scale, cache.k_zero)]
    res = to_logical(_u8(cache.k_res), RES_ORDER).reshape(c.shape)
    rf = torch.from_numpy(res).view(FP8_DT[fmt]).float().numpy()
    kf = torch.from_numpy(((c * sz[0] + sz[1]) + rf).reshape(B * npg, HKV, 64, 128))  # c * s is exact
    vf = torch.from_numpy(to_logical(cache.v.view(torch.int16).cpu().numpy(), VT_ORDER)).view(TORCH_DT[v_dt]).float()
    keep = (torch.arange(192)[None] < torch.tensor(lens)[:, None])[..., None, None]
    want = [x.view(B, npg, HKV, 64, 128).permute(0, 1, 3, 2, 4).reshape(B, 192, HKV, 128) * keep
            for x in (kf[bt.long()], vf.transpose(-1, -2)[bt.long()])]
    for out in (torch.float32, torch.float16, torch.bfloat16):
        got = cache.dequantize(bt.to(gpu), 192, torch.tensor(lens, dtype=torch.int32), out_dtype=out)
        for x, y in zip(got, want):
            assert torch.equal(x.cpu(), y.to(out))


@pytest.mark.gpu
@pytest.mark.parametrize("out", [torch.float32, torch.float16, torch.bfloat16])
def test_paged_dequantize_into_any_address(gpu, out):
    """Outputs at addresses that are multiples of an element's size alone (the C entry takes any) get the same values."""
    from ffa_mi355x import _native as N
    from ffa_mi355x.paged import PagedQ2Cache

    B, HKV, T, lens = 2, 3, 128, torch.tensor([128, 65], dtype=torch.int32, device=gpu)
    g = torch.Generator().manual_seed(6)
    cache = PagedQ2Cache(B * 2, HKV, gpu)
    bt = torch.arange(B * 2, dtype=torch.int32, device=gpu).view(B, 2)
    k, v = (torch.randn(B, T, HKV, 128, generator=g).to(gpu) for _ in range(2))
    cache.append(k, v, torch.zeros(B, dtype=torch.int32, device=gpu), bt)
    want = cache.dequantize(bt, T, lens, out_dtype=out)
    for ko, vo in ((1, 1), (0, 1), (3, 0)):
        bufs = [torch.zeros(k.numel() + 8, dtype=out, device=gpu) for _ in range(2)]
        got = [b[o:o + k.numel()] for b, o in zip(bufs, (ko, vo))]
        N.check(N.lib().ffa_q2_paged_dequant(
            cache.k_q.data_ptr(), cache.k_scale.data_ptr(), cache.k_zero.data_ptr(), cache.k_res.data_ptr(),
            N.dtype_code(cache.res_dtype), cache.v.data_ptr(), N.dtype_code(cache.v_dtype), bt.data_ptr(), 2, B * 2,
            lens.data_ptr(), B, T, HKV, got[0].data_ptr(), got[1].data_ptr(), N.dtype_code(out), N.stream_of(gpu)),
            "ffa_q2_paged_dequant")
        for x, y, b, o in zip(got, want, bufs, (ko, vo)):
            assert torch.equal(x, y.reshape(-1))
            assert not b[:o].any() and not b[o + k.numel():].any()


# ------------------------------------------------------------------- paged appends
def _pools(fmt, P, HKV, gpu, fill, v_dtype=torch.float16):
    """A cache whose bytes start as given, and its pools as bytes."""
    from ffa_mi355x.paged import PagedQ2Cache
    from ffa_mi355x.paged_kfmt import PagedKfmtCache

    c = (PagedQ2Cache(P, HKV, gpu, v_dtype=v_dtype) if fmt == "q2" else
         PagedKfmtCache(fmt, P, HKV, gpu, v_dtype=v_dtype))
    pools = [c.k_q, c.k_scale, c.k_zero, c.k_res, c.v] if fmt == "q2" else [c.k, c.k_scale, c.k_res, c.v]
    for t in pools:
        t.view(torch.uint8).fill_(fill)
    return c, pools


def _odd_groups(k):
    """Zero, constant, tiny and wide groups, infinities and NaNs among the keys [B, T, H, 128]."""
    k[0, 3, 0, :32], k[0, 4, 0, 32:64] = 0.0, 1.5
    k[0, 5, 0, 7], k[0, 6, 0, 70], k[0, 7, 0, 100] = float("inf"), float("nan"), float("-inf")
    k[0, 8, 0, :64], k[0, 9, 0, :64] = 1e-7, torch.linspace(-6e4, 6e4, 64).to(k.dtype)
    if k.dtype != torch.float16:
        k[0, 2, 0, :32] = 1e38
        k[0, 2, 0, 32:64] = torch.linspace(-1e38, 1e38, 32).to(k.dtype)
        k[0, 1, 0, :] = torch.linspace(-1e-44, 1e-44, 128).to(k.dtype)
        k[0, 1, 0, 5], k[0, 1, 0, 70] = 300.0, -2600.0


def test_nvfp4_and_nf4_code_turning_points():
    """The float that |k| (nvfp4) or k (nf4) has to reach for the next code equals where fl32(k / scale) passes the
    midpoint, for every e4m3 scale and a sample of fp16 / fp32 ones, seven floats to each side."""
    e4 = torch.arange(1, 0x7F, dtype=torch.uint8).view(torch.float8_e4m3fn).float()
    for c in (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0):
        for n in range(-7, 8):
            x = ((e4 * c).view(torch.int32) + n).view(torch.float32)
            assert torch.equal(x >= e4 * c, x / e4 >= c)
    book = torch.from_numpy(OF.NF4_CODEBOOK)
    mids = (book[:-1] + book[1:]) * 0.5
    g = torch.Generator().manual_seed(3)
    sc = torch.cat([torch.arange(17, 0x7C00, 7, dtype=torch.int16).view(torch.float16).float(),
                    torch.rand(5000, generator=g) * torch.exp2(torch.randint(-18, 60, (5000,), generator=g).float())])
    sc = sc[sc >= 1e-6]
    for mid in mids:
        up = torch.nextafter(mid, torch.tensor(1.0))
        v = sc.double() * (0.5 * (mid.double() + up.double()))
        t = v.float()
        odd = bool(mid.view(torch.int32) & 1)
        t = torch.where(t.double() < v if odd else t.double() <= v, torch.nextafter(t, torch.full_like(t, 1e38)), t)
        for n in range(-7, 8):
            x = (t.view(torch.int32) + n).view(torch.float32)
            assert torch.equal(x >= t, x / sc > mid)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["q2", "nvfp4", "nf4"])
@pytest.mark.parametrize("k_dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("B,Tn,HKV,pos", [
    (1, 1024, 2, [0]),                    # whole pages
    (1, 1100, 3, [63]),                   # one slot of the first page, a ragged last page
    (2, 1025, 1, [1, 127]),
    (33, 32, 2, [7 * i for i in range(33)]),  # half a page each, across a page edge for some
    (5, 1, 2, [0, 1, 63, 64, 130]),       # single tokens (whole pages for the 4-bit formats only)
    (1, 1024, 5, [0]),                    # the same with rows enough for the 2-bit pages
    (1, 1100, 5, [63]),
    (3, 1025, 2, [1, 127, 64]),
    (33, 32, 5, [7 * i for i in range(33)]),
])
def test_page_append_equals_token_append(gpu, fmt, k_dt, B, Tn, HKV, pos):
    """Appending whole pages writes the bytes that the per-token kernel (which takes keys at any address) writes, and
    leaves every other byte of the pools as it was; infinities, NaNs, zero and constant groups among the keys."""
    g = torch.Generator().manual_seed(Tn)
    npg = (max(pos) + Tn + 63) // 64 + 1
    k = (torch.randn(B, Tn, HKV, 128, generator=g) * 2).to(TORCH_DT[k_dt])
    if Tn > 9:
        _odd_groups(k)
    k = k.to(gpu)
    v = torch.randn(B, Tn, HKV, 128, generator=g).to(TORCH_DT[k_dt]).to(gpu)  # cast by the kernels, or before
    bt = torch.randperm(B * npg, generator=g).view(B, npg).int().to(gpu)
    p = torch.tensor(pos, dtype=torch.int32, device=gpu)
    whole, wp = _pools(fmt, B * npg, HKV, gpu, 0x5A)
    parts, pp = _pools(fmt, B * npg, HKV, gpu, 0x5A)
    whole.append(k, v, p, bt)
    if fmt == "q2" and Tn == 1:  # the per-token kernel's own cast
        parts.append(_misaligned(k), v, p, bt)
        assert all(np.array_equal(_u8(x), _u8(y)) for x, y in zip(wp, pp))
        pp[-1].zero_()
        whole.v.zero_()
        whole.append(k, v, p, bt)
    parts.append(_misaligned(k), v.to(torch.float16), p, bt)
    for x, y in zip(wp, pp):
        assert np.array_equal(_u8(x), _u8(y))
    assert any((_u8(x) != 0x5A).any() for x in wp)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["q2", "nvfp4", "nf4"])
@pytest.mark.parametrize("pool", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Tn,HKV", [(2, 300, 9), (5, 1, 3)])  # whole pages for all formats; tokens for q2
def test_append_casts_v_as_a_cast_does(gpu, fmt, pool, rows, B, Tn, HKV):
    """V rows of another type than the pool's get the bytes of torch's cast, on the page and the per-token route:
    ties, overflow, subnormals, infinities, NaNs of both signs among them."""
    from ffa_mi355x.paged import VT_ORDER, to_logical

    g = torch.Generator().manual_seed(Tn)
    n = B * Tn * HKV * 128
    bits = torch.randint(-2 ** 31, 2 ** 31, (n,), generator=g).to(torch.int32)  # every exponent, some NaNs
    x = torch.where(torch.rand(n, generator=g) < 0.5, bits.view(torch.float32), torch.randn(n, generator=g))
    inf, nan = float("inf"), float("nan")
    x[:12] = torch.tensor([inf, -inf, nan, -nan, 65504.0, 65519.9, 65520.0, -65520.0, 2.0 ** -24, 2.0 ** -25, 3.39e38, 0.0])
    x[12:14] = torch.tensor([0x3F808000, 0x3F818000], dtype=torch.int32).view(torch.float32)  # bf16 ties
    v = x.view(B, Tn, HKV, 128).to(rows).to(gpu)
    k = torch.randn(B, Tn, HKV, 128, generator=g).to(gpu)
    npg = Tn // 64 + 2
    bt = torch.randperm(B * npg, generator=g).view(B, npg).int()
    pos = torch.tensor([(17 * b) % 64 for b in range(B)], dtype=torch.int32)
    want = v.to(pool).view(torch.int16).cpu()
    for keys in (k, _misaligned(k)):
        cache, _ = _pools(fmt, B * npg, HKV, gpu, 0x5A, v_dtype=pool)
        cache.append(keys, v, pos.to(gpu), bt.to(gpu))
        got = to_logical(cache.v.view(torch.int16).cpu().numpy(), VT_ORDER)  # [P, HKV, 128, 64]
        for b in range(B):
            t = np.arange(Tn) + int(pos[b])
            assert np.array_equal(got[bt[b].numpy()[t // 64], :, :, t % 64], want[b].numpy())


# ------------------------------------------------------------------- nvfp4 / nf4 / fp8 in the reference layouts
@pytest.mark.gpu
@pytest.mark.parametrize("tau", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("B,T,HKV,D,page", [(1, 1, 1, 8, 128), (2, 130, 3, 24, 128), (1, 300, 2, 128, 64),
                                            (1, 700, 2, 128, 512), (1, 77, 5, 64, 16), (2, 129, 8, 128, 128)])
def test_nvfp4_quantizer_vector_route_equals_scalar_route(gpu, tau, B, T, HKV, D, page):
    """Every byte of the vector kernel's route equals the scalar route's (keys at an odd address): pages held in
    registers and read again, ragged last pages, keys on the codes' turning points, zeros, infinities, NaNs."""
    from ffa_mi355x import kfmt_quant as KQ

    dt = TORCH_DT[tau]
    g = torch.Generator().manual_seed(T + page)
    k = (torch.randn(B, T, HKV, D, generator=g) * 3).to(dt)
    if T > 16:
        k[0, :4, 0, :8] = 0.0
        s = torch.tensor(3.7).to(dt)
        k[:, 4] = k[:, 4].clamp(-1, 1) * s  # below the page's maximum
        mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0])
        k[0, 5, 0, :7], k[0, 6, 0, :7] = (mids * 2).to(dt), -(mids * 2).to(dt)
        k[0, :page, HKV - 1] = k[0, :page, HKV - 1].clamp(-11, 11)
        k[0, 7, HKV - 1, 0] = 12.0  # scale 2: the row of midpoints is exact
        k[0, 5, HKV - 1, :7], k[0, 6, HKV - 1, :7] = (mids * 2).to(dt), -(mids * 2).to(dt)
        k[-1, -1, 0, 1], k[-1, -1, 0, 2], k[-1, -2, 0, 3] = float("nan"), 1e-8, -1e-8
        if B > 1:
            k[0, 2, 1, 4] = float("inf")
    k = k.to(gpu)
    for fp8 in (torch.float8_e5m2, torch.float8_e4m3fn):
        a, b = KQ.encode_nvfp4(k, fp8, page), KQ.encode_nvfp4(_misaligned(k), fp8, page)
        for x, y in zip(a, b):
            assert np.array_equal(_u8(x), _u8(y))


@pytest.mark.parametrize("limit", [16384, 0])
@pytest.mark.parametrize("pos,Tn,table,pages,error", [
    ([0, 70], 58, [[3, 1], [0, 2]], 4, None),
    ([0, 70], 59, [[3, 1], [0, 2]], 4, "positions exceed"),
    ([-1, 0], 1, [[3, 1], [0, 2]], 4, "positions exceed"),
    ([0, 1], 5, [[3, -1], [0, 9]], 4, None),   # the second column is not reached
    ([0, 60], 5, [[3, -1], [0, 2]], 4, "outside the pool"),
    ([0, 60], 5, [[3, 1], [0, 4]], 4, "outside the pool"),
    ([0], 1, [[0], [1]], 4, "one row per sequence"),
])
def test_append_bounds_check(monkeypatch, limit, pos, Tn, table, pages, error):
    """The append's bounds check, with the table read whole or reduced where it lies."""
    from ffa_mi355x import paged

    monkeypatch.setattr(paged, "_CHECK_ON_HOST", limit)
    args = torch.tensor(pos, dtype=torch.int32), Tn, torch.tensor(table, dtype=torch.int32), pages
    if error is None:
        paged.check_append_fits(*args)
    else:
        with pytest.raises(ValueError, match=error):
            paged.check_append_fits(*args)
