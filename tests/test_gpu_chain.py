"""The fp32 matrix-core kernels at the edges of their blocks, stages and
dispatch rule, bit for bit against the oracle's FMA chains."""
import numpy as np
import pytest
import torch

import oracle
from aps2026_amd import attention, moe, synth

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[chain] {msg}", flush=True)


def dev(a, d):
    return torch.from_numpy(np.ascontiguousarray(a)).to(d)


# k: below, at and past the ring's stages of 32 k (eight, four and two slots),
# with and without a half stage; rows and columns: one-wave tiles, the 32 x 32,
# 32 x 64 and 64 x 64 blocks, the 128-row blocks of 64 and 128 columns, with
# remainders of each
@pytest.mark.parametrize("rows,k,n", [
    (1, 16, 4), (16, 32, 16), (17, 48, 20), (16, 224, 36), (9, 256, 36), (16, 288, 68), (33, 480, 48), (16, 528, 32),
    (600, 96, 260), (600, 128, 256), (601, 112, 256), (601, 160, 252), (590, 288, 256),
    (333, 32, 4096), (321, 80, 4092), (333, 192, 2048), (333, 48, 2044), (300, 288, 2048),
    (1000, 32, 2048), (1023, 96, 2044), (1023, 128, 2044), (1000, 160, 2048), (1000, 192, 2044), (1000, 48, 2048), (4095, 32, 1024), (4096, 64, 1020), (4001, 160, 1024)])
def test_linear_block_and_stage_edges(gpu_device, rows, k, n):
    note(f"linear edges rows={rows} k={k} n={n}")
    rng = np.random.default_rng(rows + 3 * k + 7 * n)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (0.02 * rng.standard_normal((n, k))).astype(np.float32)
    b = (0.1 * rng.standard_normal(n)).astype(np.float32)
    got = attention.linear_gpu(dev(x, gpu_device), dev(w, gpu_device), dev(b, gpu_device)).cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), oracle.linear(x, w, b).view(np.uint32))


# tokens and experts on both sides of the dispatch's lines (8, 96 and 192
# positions per expert for w1||w3, 16 and 192 for w2), ffn widths that deal an
# uneven number of column blocks to the XCDs, k = 64 .. 512 through the rings
@pytest.mark.parametrize("T,E,H,F", [(5, 16, 256, 64), (64, 16, 512, 192), (65, 16, 256, 64), (130, 16, 512, 320),
                                     (97, 2, 256, 192), (192, 2, 512, 64), (193, 2, 256, 448), (700, 3, 256, 64),
                                     (900, 3, 512, 192)])
def test_fp32_experts_block_edges(gpu_device, T, E, H, F):
    note(f"fp32 experts T={T} E={E} H={H} F={F}")
    inp = synth.make_moe_inputs(T=T, H=H, E=E, F=F, dtype="f32", seed=T + E + F)
    d = lambda a: [dev(a[e], gpu_device) for e in range(E)]
    w = moe.register_moe_weights_gpu(d(inp.w1), d(inp.w2), d(inp.w3), torch.float32)
    moe.moe_forward_gpu(dev(inp.x, gpu_device), dev(inp.gate, gpu_device), w)
    plan = w.plan_views(T)
    plan["y"].fill_(float("nan"))   # a row or column that no block writes stays NaN
    plan["act"].fill_(float("nan"))
    out = moe.moe_forward_gpu(dev(inp.x, gpu_device), dev(inp.gate, gpu_device), w)
    ref = oracle.reference_path(inp.x, inp.gate, inp.w1, inp.w3, inp.w2)
    y, got = plan["y"].cpu().numpy(), out.cpu().numpy()
    w.release()
    # the chains are exact; SiLU's exp in double is the GPU's against glibc's,
    # at most the last fp32 bit of a hidden value: 2^-23 of it, row by row
    for a, b in ((y, ref["y"]), (got, ref["out"])):
        err = np.linalg.norm(a.astype(np.float64) - b, axis=1) / np.linalg.norm(b.astype(np.float64), axis=1)
        assert err.max() <= 2.0 ** -23


# k = 16 mod 32 on both sides of the rule that sends short k to SIMT blocks (k up
# to 144, 96 blocks and more, out of 64 and more): whole and partly filled blocks
@pytest.mark.parametrize("rows,k,n", [(6144, 16, 64), (6080, 16, 64), (6100, 16, 60), (700, 48, 1100), (1000, 144, 2600),
                                      (2800, 80, 516), (1000, 176, 2600), (1000, 208, 2600)])
@pytest.mark.parametrize("bias", [True, False])
def test_linear_short_half_stage(gpu_device, rows, k, n, bias):
    note(f"linear short k rows={rows} k={k} n={n} bias={bias}")
    rng = np.random.default_rng(rows + k + n)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = (0.02 * rng.standard_normal((n, k))).astype(np.float32)
    b = (0.1 * rng.standard_normal(n)).astype(np.float32) if bias else None
    out = torch.full((rows, n), float("nan"), device=gpu_device)
    attention.linear_gpu(dev(x, gpu_device), dev(w, gpu_device), dev(b, gpu_device) if bias else None, out=out)
    np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), oracle.linear(x, w, b).view(np.uint32))


def test_linear_multi_short_half_stage(gpu_device):
    """Outputs of different widths in one call, by SIMT blocks, and (a narrow
    one among them) in one grid."""
    from aps2026_amd import capi
    import ctypes
    rows, k = 2000, 48
    rng = np.random.default_rng(k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    for ns in ((512, 256, 640), (512, 32)):
        ws = [(0.02 * rng.standard_normal((n, k))).astype(np.float32) for n in ns]
        bs = [(0.1 * rng.standard_normal(n)).astype(np.float32) for n in ns]
        xd, wd, bd = dev(x, gpu_device), [dev(w, gpu_device) for w in ws], [dev(b, gpu_device) for b in bs]
        ys = [torch.full((rows, n), float("nan"), device=gpu_device) for n in ns]
        vp = ctypes.c_void_p * len(ns)
        ptr = lambda ts: vp(*[t.data_ptr() for t in ts])
        rc = capi.lib().aps_linear_multi(xd.data_ptr(), rows, k, len(ns), ptr(wd), ptr(bd),
                                         (ctypes.c_int32 * len(ns))(*ns), ptr(ys), moe._stream(gpu_device))
        assert rc == 0, capi.last_error()
        for w, b, y in zip(ws, bs, ys):
            np.testing.assert_array_equal(y.cpu().numpy().view(np.uint32), oracle.linear(x, w, b).view(np.uint32))


def off4(a):
    """The same values 4 bytes past a 16-byte boundary."""
    b = torch.empty(a.numel() + 1, dtype=a.dtype, device=a.device)
    b[1:] = a.reshape(-1)
    out = b[1:].view(a.shape)
    assert out.data_ptr() % 16 == 4
    return out


# tokens: the few-token router's and the token-major router's, one to several
# 64-row blocks per expert; an expert without rows among the staged offsets
@pytest.mark.parametrize("T,E,H,F", [(1, 2, 512, 64), (40, 3, 512, 192), (300, 16, 256, 64), (257, 2, 768, 320)])
def test_fp32_experts_unaligned(gpu_device, T, E, H, F):
    """fp32 arrays that are only 4-byte aligned: the block, the staged GEMMs
    (x, act and y alone and together) and the dense FFN give the bits that
    the aligned arrays give."""
    from aps2026_amd import capi
    note(f"fp32 experts unaligned T={T} E={E} H={H} F={F}")
    inp = synth.make_moe_inputs(T=T, H=H, E=E, F=F, dtype="f32", seed=T + H)
    x, gate = dev(inp.x, gpu_device), dev(inp.gate, gpu_device)
    d = lambda a: [dev(a[e], gpu_device) for e in range(E)]
    bits = lambda a: a.view(torch.int32)
    w = moe.register_moe_weights_gpu(d(inp.w1), d(inp.w2), d(inp.w3), torch.float32)
    want = moe.moe_forward_gpu(x, gate, w)
    assert torch.equal(bits(moe.moe_forward_gpu(off4(x), gate, w)), bits(want))
    logits = w.plan_views(T)["logits"].clone()
    assert torch.equal(bits(moe.moe_forward_grouped_gpu(off4(x), logits, w)), bits(want))
    L, s = capi.lib(), moe._stream(gpu_device)
    rng = np.random.default_rng(T)
    cuts = np.sort(rng.integers(0, 2 * T + 1, E - 1))
    cuts[0] = 0   # expert 0 has no row
    offsets = dev(np.concatenate([[0], cuts, [2 * T]]).astype(np.int32), gpu_device)
    arows = dev(rng.integers(0, T, 2 * T).astype(np.int32), gpu_device)

    def staged(xs, act, y):
        act.fill_(float("nan"))
        y.fill_(float("nan"))
        assert L.aps_moe_ffn_up(w.handle, xs.data_ptr(), capi.DTYPE_F32, T, offsets.data_ptr(), arows.data_ptr(),
                                act.data_ptr(), None, s) == 0, capi.last_error()
        assert L.aps_moe_ffn_down(w.handle, act.data_ptr(), None, T, offsets.data_ptr(), y.data_ptr(), s) == 0
        return act.clone(), y.clone()

    act, y = torch.empty(2 * T, F, device=gpu_device), torch.empty(2 * T, H, device=gpu_device)
    ref = staged(x, act, y)
    assert all(torch.isfinite(t).all() for t in ref)
    for xs, a, o in ((off4(x), act, y), (x, off4(act), y), (x, act, off4(y)), (off4(x), off4(act), off4(y))):
        for got, r in zip(staged(xs, a, o), ref):
            assert torch.equal(bits(got), bits(r))
    w.release()
    one = moe.register_moe_weights_gpu(d(inp.w1)[:1], d(inp.w2)[:1], d(inp.w3)[:1], torch.float32)
    n = L.aps_mlp_workspace_size(one.handle, T)
    ws = torch.empty(n, dtype=torch.uint8, device=gpu_device)
    out = []
    for xs, o in ((x, torch.empty_like(x)), (off4(x), torch.empty_like(x)), (x, off4(torch.empty_like(x)))):
        assert L.aps_mlp_forward(one.handle, xs.data_ptr(), capi.DTYPE_F32, T, o.data_ptr(), ws.data_ptr(), n, s) == 0
        out.append(o.clone())
    one.release()
    assert torch.equal(bits(out[1]), bits(out[0])) and torch.equal(bits(out[2]), bits(out[0]))
