"""Groups of more than four query rows over many workgroups: the build that decides before it loads and shares a KV
head's data between its quads, against the same sequences decoded one by one (few workgroups: the other build)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HQ,HKV", [(64, 8), (24, 4), (32, 2)])
@pytest.mark.parametrize("SBS", [16, 64, 128, 1024])
@pytest.mark.parametrize("case", ["probe", "threshold", "mean", "no_residual"])
def test_many_workgroups_equal_single_sequences(gpu, HQ, HKV, SBS, case):
    from ffa_mi355x import synth
    from ffa_mi355x.decode import DecodeWorkspace
    from ffa_mi355x.paged import PagedQ2Cache

    lens = [9000, 1, 700, 4097, 64, 8191, 0, 5000, 9000, 3333] * (2 if HKV < 8 else 1)
    B, T = len(lens), max(lens)
    q = torch.randn(B, HQ, 128, generator=torch.Generator().manual_seed(HQ + SBS)).to(gpu)
    bt, P = synth.page_tables([max(n, 1) for n in lens], seed=SBS)
    bt = torch.nn.functional.pad(bt, (0, -(-T // 64) - bt.shape[1])).to(gpu)
    cache = PagedQ2Cache(P, HKV, gpu)
    for b, n in enumerate(lens):
        if n:
            k, v = synth.sequence_inputs_device(q[b], n, HKV=HKV, seed=b, n_heavy=4)
            cache.append(k, v, torch.zeros(1, dtype=torch.int32, device=gpu), bt[b:b + 1])
    sl = torch.tensor(lens, dtype=torch.int32, device=gpu)
    kw = dict(T=T, BS=max(SBS, 64), SBS=SBS, delta=5.0)
    if case == "threshold":
        kw["precomputed_threshold"] = torch.rand(B, HQ, device=gpu) * 10
    if case == "mean":
        kw["v_mean"] = cache.value_mean(bt, sl, out_dtype=torch.float32)
    if case == "no_residual":
        kw["use_fp8_residual"] = False
    ws = DecodeWorkspace(B, HQ, HKV, T, kw["BS"], SBS, gpu, torch.float32)
    for t in (ws.m_buf, ws.l_buf, ws.o_buf):
        t.fill_(float("nan"))  # every slot that the merge reads is written
    ws.mask_buf.fill_(7)
    cache.decode(q, bt, sl, workspace=ws, **kw)
    for b in range(B):
        one = {k: (v[b:b + 1] if torch.is_tensor(v) else v) for k, v in kw.items()}
        w1 = cache.decode(q[b:b + 1], bt[b:b + 1], sl[b:b + 1], **one)
        assert torch.equal(ws.mask_buf[b], w1.mask_buf[0]), b
        assert torch.equal(ws.threshold_buf[b], w1.threshold_buf[0]), b
        # the same sums in the same order, but for what the compilers of two builds contract: fp32 rounding
        assert torch.allclose(ws.o[b], w1.o[0], rtol=2e-5, atol=2e-6), (b, (ws.o[b] - w1.o[0]).abs().max())


@pytest.mark.parametrize("HQ,HKV", [(64, 8), (24, 4), (32, 2), (32, 8), (8, 8)])
@pytest.mark.parametrize("SBS", [16, 64, 128, 1024])
@pytest.mark.parametrize("case", ["probe", "threshold", "mean", "no_residual"])
def test_contiguous_many_workgroups_equal_single_sequences(gpu, HQ, HKV, SBS, case):
    """The contiguous per-channel builds for many workgroups (V staged a quarter at a time) likewise."""
    import attn_kernel.attn_kernel_v1210_fused_bsz_q2fp8 as K
    from ffa_mi355x import synth
    from ffa_mi355x.quant import quantize_per_channel

    if case == "mean":
        from ffa_mi355x.dropins import _ROOT, _load

        K = _load("ffa_mi355x_meanv_dropin", _ROOT / "ffa-q2fp8-meanv" / "attn_kernel" / "attn_kernel_v1210_meanv_bsz_q2fp8.py")
    lens = [9000, 1, 700, 4097, 64, 8191, 8999, 5000, 9000, 3333] * (4 if SBS == 1024 or HKV < 8 else 2)
    B, T = len(lens), max(lens)
    dt = torch.float16 if SBS == 64 else torch.bfloat16
    q = torch.randn(B, HQ, 128, generator=torch.Generator().manual_seed(HQ + SBS)).to(gpu, dt)
    k = torch.zeros(10, T, HKV, 128, dtype=dt, device=gpu)
    v = torch.zeros_like(k)
    for b in range(10):
        n = lens[b]
        k[b, :n], v[b, :n] = synth.sequence_inputs_device(q[b], n, HKV=HKV, seed=b, n_heavy=4, dtype=dt)
    kq, ks, kz, kr = (t.repeat(B // 10, *[1] * (t.dim() - 1)) for t in quantize_per_channel(k, torch.float8_e5m2))
    q, v = q[:, None], v.repeat(B // 10, 1, 1, 1)
    sl = torch.tensor(lens, dtype=torch.int32, device=gpu)
    BS = max(SBS, 64)
    kw = dict(BS=BS, SBS=SBS, delta=5.0)
    th = torch.rand(B, HQ, device=gpu) * 10 if case == "threshold" else None

    def decode(lo, hi):
        ws = K.allocate_q2fp8_decode_workspace(q[lo:hi], kq[lo:hi], v[lo:hi], BS=BS, SBS=SBS)
        for t in (ws.m_buf, ws.l_buf, ws.o_buf):
            t.fill_(float("nan"))  # every slot that the merge reads is written
        ws.mask_buf.fill_(7)
        o = K.attn_forward_decode_quantized(q[lo:hi], kq[lo:hi], ks[lo:hi], kz[lo:hi], v[lo:hi], k_residual=kr[lo:hi],
                                            precomputed_threshold=None if th is None else th[lo:hi],
                                            use_fp8_residual=case != "no_residual", workspace=ws, seq_lens=sl[lo:hi], **kw)
        return o, ws

    o, ws = decode(0, B)
    ulp = 2.0 ** (-10 if dt == torch.float16 else -7)
    for b in range(B):
        o1, w1 = decode(b, b + 1)
        assert torch.equal(ws.mask_buf[b], w1.mask_buf[0]), b
        if th is None:
            assert torch.equal(ws.threshold_buf[b], w1.threshold_buf[0]), b
        # the same sums but for what two builds contract (fp32 rounding): one step of the output type at most
        assert torch.allclose(o[b].float(), o1[0].float(), rtol=ulp, atol=2e-6), (b, (o[b].float() - o1[0].float()).abs().max())
