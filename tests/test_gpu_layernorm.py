"""GPU parity of the decoder-layer LayerNorm (aps_layer_norm /
aps_add_layer_norm, the producer of the MoE block's input) against the CPU
oracle, through the C ABI.  Bar: bit-exact (y, the updated x, and therefore
the routing of its output), because the reference keeps both row sums serial
precisely so that routing does not move (src/tensor.cu:2010-2014)."""
import sys

import numpy as np
import pytest
import torch

import oracle
from aps2026_amd import moe, synth

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


def _inputs(rows, h, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, h)).astype(np.float32)
    r = rng.standard_normal((rows, h)).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(h)).astype(np.float32)
    b = (0.1 * rng.standard_normal(h)).astype(np.float32)
    return x, r, w, b


def _dev(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 333])
@pytest.mark.parametrize("h", [256, 1280, 4096])
@pytest.mark.parametrize("add", [False, True])
def test_layer_norm_bit_exact(gpu_device, rows, h, add):
    note(f"layer norm rows={rows} h={h} add={add}")
    x, r, w, b = _inputs(rows, h, 11 * rows + h + add)
    xd, rd, wd, bd = (_dev(a, gpu_device) for a in (x, r, w, b))
    y = torch.empty_like(xd)
    if add:
        moe.add_layer_norm_gpu(xd, rd, wd, bd, moe.NORM_EPS, y)
    else:
        moe.layer_norm_gpu(xd, wd, bd, moe.NORM_EPS, y)
    torch.cuda.synchronize()
    want_y, want_v, _, _ = oracle.layer_norm(x, w, b, eps=moe.NORM_EPS, residual=r if add else None)
    np.testing.assert_array_equal(y.cpu().numpy().view(np.uint32), want_y.view(np.uint32))
    np.testing.assert_array_equal(xd.cpu().numpy().view(np.uint32), (want_v if add else x).view(np.uint32))


@pytest.mark.parametrize("rows,h", [(2, 4096), (4, 4096), (6, 512), (3, 768)])
def test_layer_norm_row_groups(gpu_device, rows, h):
    """Rows per wave: partly and exactly filled waves, an even and an odd
    number of streamed 256-column chunks; with the residual, values of large
    and small magnitude so that the order of the sums shows.  Bit-exact."""
    note(f"layer norm groups rows={rows} h={h}")
    x, r, w, b = _inputs(rows, h, rows + h)
    x *= np.exp2(np.random.default_rng(h).integers(-12, 13, (rows, h))).astype(np.float32)
    xd, rd, wd, bd = (_dev(a, gpu_device) for a in (x, r, w, b))
    y = torch.empty_like(xd)
    moe.add_layer_norm_gpu(xd, rd, wd, bd, moe.NORM_EPS, y)
    torch.cuda.synchronize()
    want_y, want_v, _, _ = oracle.layer_norm(x, w, b, eps=moe.NORM_EPS, residual=r)
    np.testing.assert_array_equal(y.cpu().numpy().view(np.uint32), want_y.view(np.uint32))
    np.testing.assert_array_equal(xd.cpu().numpy().view(np.uint32), want_v.view(np.uint32))


@pytest.mark.parametrize("rows", [3, 9])
@pytest.mark.parametrize("h", [256, 512, 768, 1024, 1792, 2048, 5120, 8192])
@pytest.mark.parametrize("add", [False, True])
def test_layer_norm_streamed_widths(gpu_device, rows, h, add):
    """One, two and four chunks of loads in flight, chunk counts around them;
    a last wave of one and of three rows.  Rows of NaN around the output show a
    store past its rows."""
    note(f"layer norm streamed rows={rows} h={h} add={add}")
    x, r, w, b = _inputs(rows, h, rows * h + add)
    x *= np.exp2(np.random.default_rng(rows).integers(-12, 13, (rows, h))).astype(np.float32)
    guard = torch.full((rows + 4, h), float("nan"), device=gpu_device)
    xd = guard.clone()
    xd[2:-2] = _dev(x, gpu_device)
    rd, wd, bd = (_dev(a, gpu_device) for a in (r, w, b))
    y = guard.clone()
    if add:
        moe.add_layer_norm_gpu(xd[2:-2], rd, wd, bd, moe.NORM_EPS, y[2:-2])
    else:
        moe.layer_norm_gpu(xd[2:-2], wd, bd, moe.NORM_EPS, y[2:-2])
    want_y, want_v, _, _ = oracle.layer_norm(x, w, b, eps=moe.NORM_EPS, residual=r if add else None)
    for got, want in ((y, want_y), (xd, want_v if add else x)):
        got = got.cpu().numpy()
        np.testing.assert_array_equal(got[2:-2].view(np.uint32), want.view(np.uint32))
        assert np.isnan(got[:2]).all() and np.isnan(got[-2:]).all()


def test_layer_norm_known_answer_rows(gpu_device):
    """The oracle's order and fused-variance known-answer rows (the mean of
    [1e8, 1, -1e8, 0...] is 0, that of [1e8, -1e8, 1, 0...] is 2^-12; the
    variance of [a, -a, c, -c, 0...] is the fused chain's), plus a constant
    row (y = bias) and an all-zero row, on the GPU."""
    h = 4096
    x = np.zeros((5, h), np.float32)
    x[0, :3] = [1e8, 1.0, -1e8]
    x[1, :3] = [1e8, -1e8, 1.0]
    x[2, :4] = [np.uint32(1067587382).view(np.float32), -np.uint32(1067587382).view(np.float32),
                np.uint32(1070634225).view(np.float32), -np.uint32(1070634225).view(np.float32)]
    x[3] = 0.5
    _, _, w, b = _inputs(1, h, 5)
    xd, wd, bd = (_dev(a, gpu_device) for a in (x, w, b))
    y = torch.empty_like(xd)
    moe.layer_norm_gpu(xd, wd, bd, moe.NORM_EPS, y)
    torch.cuda.synchronize()
    want, _, mean, _ = oracle.layer_norm(x, w, b, eps=moe.NORM_EPS)
    assert mean[0] == 0.0 and mean[1] == np.float32(2.0 ** -12)
    got = y.cpu().numpy()
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(got[3], b)
    np.testing.assert_array_equal(got[4], b)


def test_decoder_post_attention_norm_then_moe_routes_like_the_oracle(gpu_device):
    """The decoder layer's MoE half (reference PhiDecoderLayer::forward_carry,
    src/layer.cu:292-297): post = add_layer_norm(attn, x); moe(post).  With
    synthetic attention output and residual stream (T = 1024, H = 4096), the
    LayerNorm output and the routing plan of the MoE block on it (fp32 x, bf16
    experts) match the oracle bit for bit; the block output is within the bf16
    bar of the oracle's FFN on the same routes."""
    T, H, E, F = 1024, 4096, 16, 448
    note(f"decoder MoE half T={T}")
    inp = synth.make_moe_inputs(T=T, H=H, E=E, F=F, dtype="bf16", seed=21)
    rng = np.random.default_rng(22)
    resid = (0.5 * rng.standard_normal((T, H))).astype(np.float32)
    attn = (0.5 * rng.standard_normal((T, H))).astype(np.float32)
    w = (1.0 + 0.05 * rng.standard_normal(H)).astype(np.float32)
    b = (0.05 * rng.standard_normal(H)).astype(np.float32)
    ad, xd, wd, bd = (_dev(a, gpu_device) for a in (attn, resid, w, b))
    post = torch.empty_like(ad)
    # reference argument order: add_layer_norm_gpu(attn, x, ...): attn += x, post = LN(attn)
    moe.add_layer_norm_gpu(ad, xd, wd, bd, moe.NORM_EPS, post)
    lists = []
    for nm in ("w1", "w2", "w3"):
        t = torch.from_numpy(np.ascontiguousarray(inp.packed[nm + "_bf16"]).view(np.int16)).to(gpu_device)
        lists.append([t.view(torch.bfloat16)[e].contiguous() for e in range(E)])
    wts = moe.register_moe_weights_gpu(lists[0], lists[1], lists[2], compute_dtype=torch.bfloat16)
    gate = _dev(inp.gate, gpu_device)
    out = moe.moe_forward_gpu(post, gate, wts, out_dtype=torch.float32)
    plan = wts.plan_views(T)
    torch.cuda.synchronize()
    want_post, want_v, _, _ = oracle.layer_norm(attn, w, b, eps=moe.NORM_EPS, residual=resid)
    np.testing.assert_array_equal(post.cpu().numpy().view(np.uint32), want_post.view(np.uint32))
    np.testing.assert_array_equal(ad.cpu().numpy().view(np.uint32), want_v.view(np.uint32))
    logits = oracle.router_logits(want_post, inp.gate)
    routes = oracle.route_top2(logits)
    counts, offsets, arows, rpos = oracle.dispatch(routes, E)
    np.testing.assert_array_equal(plan["logits"].cpu().numpy().view(np.uint32), logits.view(np.uint32))
    np.testing.assert_array_equal(plan["routes"].cpu().numpy().astype(np.int32), routes)
    np.testing.assert_array_equal(plan["assignment_rows"].cpu().numpy().view(np.uint32), arows)
    np.testing.assert_array_equal(plan["route_positions"].cpu().numpy().view(np.uint32), rpos)
    # expert FFN on the bf16 copy of post, a token subset
    toks = np.arange(0, T, 37)
    xb = synth.bf16_bits_to_f32(synth.f32_to_bf16_bits(want_post[toks]))
    y_ref = oracle.ffn_rows(np.repeat(xb, 2, axis=0), routes[toks].reshape(-1), inp.w1, inp.w3, inp.w2)
    out_ref = (0.5 * (y_ref[0::2].astype(np.float64) + y_ref[1::2])).astype(np.float32)
    got = out.cpu().numpy()[toks]
    err = np.linalg.norm(got - out_ref, axis=1) / np.linalg.norm(out_ref, axis=1)
    assert err.max() <= 2e-2
    wts.release()
