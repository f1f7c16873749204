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
