"""GPU tests of the few-row expert tiles (ffn_small.hip): a batch small enough
to take them gives, bit for bit, the rows that the same tokens have in a batch
past the rule, which the 128- and 256-row tiles serve (those are held to the
oracle elsewhere).  Batches of one token, around the 32-row tile, at the rule's
edge (2 rows <= 12 experts in bf16, 24 in fp8) and one past it; experts with
several tiles, one and no row; K shorter and longer than the stages in flight,
F of one to seven column blocks."""
import sys

import numpy as np
import pytest
import torch

from aps2026_amd import moe, synth

pytestmark = pytest.mark.gpu
BIG = 700


def weights(dtype, E, H, F, dev, seed):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    w = [torch.randn((E,) + s, generator=g, device=dev) * 0.05 for s in ((F, H), (H, F), (F, H))]
    if dtype == "bf16":
        return moe.register_moe_weights_gpu(*[list(t.bfloat16().unbind(0)) for t in w], compute_dtype=torch.bfloat16)
    scales = [t.abs().amax(dim=-1) / synth.FP8_E4M3_MAX for t in w]
    codes = [(t / s[..., None]).to(torch.float8_e4m3fn) for t, s in zip(w, scales)]
    return moe.register_moe_weights_gpu(*[list(t.unbind(0)) for t in codes], compute_dtype=torch.float8_e4m3fn,
                                        scales=tuple(list(s.contiguous().unbind(0)) for s in scales))


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("E,H,F,skew", [(16, 4096, 448, False), (16, 512, 448, True), (8, 256, 64, True),
                                        (24, 768, 192, False), (16, 1024, 320, True)])
def test_few_rows_equal_the_row_tiles(gpu_device, dtype, E, H, F, skew):
    edge = (24 if dtype == "fp8" else 12) * E // 2
    print(f"[gpu-case] few rows {dtype} E={E} H={H} F={F} skew={skew} edge={edge}", flush=True)
    sys.stdout.flush()
    w = weights(dtype, E, H, F, gpu_device, E + H)
    g = torch.Generator(device=gpu_device)
    g.manual_seed(F)
    x = torch.randn((BIG, H), generator=g, device=gpu_device)
    gate = torch.randn((E, H), generator=g, device=gpu_device) * 0.05
    if skew:   # nearly every token to the same two experts
        x[:, 0] = 4.0
        gate[1, 0], gate[E - 1, 0] = 8.0, 4.0
    x = x.bfloat16()
    big = moe.moe_forward_gpu(x, gate, w).clone()
    for n in (1, 2, 31, 33, edge, edge + 1):
        got = moe.moe_forward_gpu(x[:n].contiguous(), gate, w)
        torch.cuda.synchronize()
        assert torch.isfinite(got).all()
        assert torch.equal(got.view(torch.int16), big[:n].view(torch.int16)), n
    w.release()


@pytest.mark.parametrize("E,H,F", [(16, 4096, 448), (16, 512, 64), (8, 256, 320), (24, 768, 512)])
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_w2_tiles_between_the_rules(gpu_device, dtype, E, H, F):
    """w2 stays on the one-wave tiles past the w1||w3 rule, up to 24 (bf16) or
    32 (fp8) routes per expert: that edge and one past it, against a batch of
    row tiles."""
    edge = (32 if dtype == "fp8" else 24) * E // 2
    print(f"[gpu-case] w2 tiles {dtype} E={E} H={H} F={F} edge={edge}", flush=True)
    w = weights(dtype, E, H, F, gpu_device, E * F)
    g = torch.Generator(device=gpu_device)
    g.manual_seed(H)
    x = torch.randn((BIG, H), generator=g, device=gpu_device).bfloat16()
    gate = torch.randn((E, H), generator=g, device=gpu_device) * 0.05
    for out in (torch.bfloat16, torch.float32):
        bits = torch.int16 if out == torch.bfloat16 else torch.int32
        big = moe.moe_forward_gpu(x, gate, w, out_dtype=out).clone()
        for n in (edge - 31, edge, edge + 1):
            got = moe.moe_forward_gpu(x[:n].contiguous(), gate, w, out_dtype=out)
            torch.cuda.synchronize()
            assert torch.equal(got.view(bits), big[:n].view(bits)), n
    w.release()


@pytest.mark.parametrize("E,H,F", [(24, 512, 448), (17, 256, 512), (64, 256, 128), (64, 256, 192)])
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_many_experts_leave_the_small_tiles_early(gpu_device, dtype, E, H, F):
    """w1||w3 past 8192 columns over all experts: 8 experts' worth of rows, that
    edge and one past it, and the mean's own edge, against a batch of row
    tiles; up to 8192 columns (64 x 128) the mean alone.  512 tokens is w2's own
    line for bf16."""
    per = 24 if dtype == "fp8" else 12
    print(f"[gpu-case] many experts {dtype} E={E} H={H} F={F}", flush=True)
    w = weights(dtype, E, H, F, gpu_device, E + F)
    g = torch.Generator(device=gpu_device)
    g.manual_seed(E)
    x = torch.randn((1100, H), generator=g, device=gpu_device)
    gate = torch.randn((E, H), generator=g, device=gpu_device) * 0.05
    x[:, 0], gate[:, 0] = 1.0, -1.1 * torch.log(torch.arange(1, E + 1, device=gpu_device).float())
    x = x.bfloat16()
    big = moe.moe_forward_gpu(x, gate, w).clone()
    for n in (4 * per, 4 * per + 1, E * per // 2, E * per // 2 + 1, 512, 513):
        got = moe.moe_forward_gpu(x[:n].contiguous(), gate, w)
        assert torch.equal(got.view(torch.int16), big[:n].view(torch.int16)), n
    w.release()


def test_few_rows_plan_past_two_assignments_per_row(gpu_device):
    """The staged w1||w3 call with a plan of more positions than 2 rows: the
    grid covers the rest in further rounds."""
    from aps2026_amd import capi
    E, H, F, rows, A = 16, 512, 448, 20, 1500
    w = weights("bf16", E, H, F, gpu_device, 3)
    rng = np.random.default_rng(4)
    x = torch.from_numpy(rng.standard_normal((rows, H)).astype(np.float32)).to(gpu_device).bfloat16()
    big = x.repeat(40, 1).contiguous()      # 800 rows: the row tiles
    arows = torch.from_numpy(rng.integers(0, rows, A).astype(np.int32)).to(gpu_device)
    cuts = np.sort(rng.integers(0, A + 1, E - 1))
    offsets = torch.from_numpy(np.concatenate([[0], cuts, [A]]).astype(np.int32)).to(gpu_device)
    out = []
    for xs in (x, big):
        act = torch.full((A, F), float("nan"), dtype=torch.bfloat16, device=gpu_device)
        rc = capi.lib().aps_moe_ffn_up(w.handle, xs.data_ptr(), capi.DTYPE_BF16, xs.shape[0], offsets.data_ptr(),
                                       arows.data_ptr(), act.data_ptr(), None,
                                       torch.cuda.current_stream(gpu_device).cuda_stream)
        assert rc == 0, capi.last_error()
        torch.cuda.synchronize()
        out.append(act)
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
    w.release()


@pytest.mark.parametrize("dtype,x32", [("bf16", False), ("bf16", True), ("fp8", False), ("f32", True)])
@pytest.mark.parametrize("E,H", [(16, 4096), (5, 1536), (16, 512), (2, 1024)])
def test_few_token_router_equals_the_token_major_router(gpu_device, dtype, x32, E, H):
    """Up to 256 tokens the router takes a workgroup per token and the dispatch
    counts the routes itself: logits, routes and block outputs are, bit for
    bit, those of the same tokens in a larger batch, and the plan is the
    stable sort of the routes (one, full and partly filled 64-token tiles)."""
    F = 64
    print(f"[gpu-case] few-token router {dtype} x32={x32} E={E} H={H}", flush=True)
    sys.stdout.flush()
    g = torch.Generator(device=gpu_device)
    g.manual_seed(E * H)
    if dtype == "f32":
        ws = [list((torch.randn((E,) + sh, generator=g, device=gpu_device) * 0.05).unbind(0))
              for sh in ((F, H), (H, F), (F, H))]
        w = moe.register_moe_weights_gpu(*ws, compute_dtype=torch.float32)
    else:
        w = weights(dtype, E, H, F, gpu_device, E + H)
    x = torch.randn((BIG, H), generator=g, device=gpu_device)
    gate = torch.randn((E, H), generator=g, device=gpu_device) * 0.05
    if not x32:
        x = x.bfloat16()
    big = moe.moe_forward_gpu(x, gate, w).clone()
    view = w.plan_views(BIG)
    logits, routes = view["logits"].clone(), view["routes"].clone()
    for n in (1, 3, 64, 65, 200, 256, 257):
        got = moe.moe_forward_gpu(x[:n].contiguous(), gate, w)
        view = w.plan_views(n)
        torch.cuda.synchronize()
        assert torch.equal(view["logits"].view(torch.int32), logits[:n].view(torch.int32)), n
        assert torch.equal(view["routes"], routes[:n]), n
        r = routes[:n].cpu().numpy().astype(np.int64).reshape(-1)
        order = np.argsort(r, kind="stable")
        assert np.array_equal(view["assignment_rows"].cpu().numpy(), order // 2), n
        assert np.array_equal(view["route_positions"].cpu().numpy().reshape(-1)[order], np.arange(2 * n)), n
        assert np.array_equal(view["offsets"].cpu().numpy(), np.searchsorted(r[order], np.arange(E + 1))), n
        bits = torch.int32 if got.dtype == torch.float32 else torch.int16
        assert torch.equal(got.view(bits), big[:n].view(bits)), n
    w.release()


@pytest.mark.parametrize("H", [512, 1024])
@pytest.mark.parametrize("dtype,E,F", [("fp8", 16, 448), ("fp8", 5, 512), ("bf16", 16, 448), ("bf16", 3, 64)])
def test_tile_histograms_of_few_tokens(gpu_device, dtype, E, F, H):
    """The tile histograms of the published plan after a forward, whatever made
    the plan: the w1||w3 launch, the counting dispatch (hidden 1024) or the
    router (257 tokens, and at hidden 512 from where w1||w3 makes no plan); the
    slot-0 histogram with an fp8 set."""
    print(f"[gpu-case] tile histograms {dtype} E={E} F={F} H={H}", flush=True)
    w = weights(dtype, E, H, F, gpu_device, E + F)
    g = torch.Generator(device=gpu_device)
    g.manual_seed(E)
    x = torch.randn((257, H), generator=g, device=gpu_device).bfloat16()
    gate = torch.randn((E, H), generator=g, device=gpu_device) * 0.05
    for n in (1, 16, 17, 63, 64, 65, 130, 256, 257):
        ws, L = w.workspace(n)
        ws.fill_(0xEE)
        moe.moe_forward_gpu(x[:n].contiguous(), gate, w)
        routes = w.plan_views(n)["routes"].cpu().numpy()
        tiles = (n + 63) // 64
        want = np.zeros((2, tiles, E, 4), np.uint8)
        for t in range(n):
            for slot in range(2):
                want[0, t // 64, routes[t, slot], t % 64 // 16] += 1
            want[1, t // 64, routes[t, 0], t % 64 // 16] += 1
        size = tiles * E * 4
        for off, ref in ((L.tile_counts, want[0]), (L.tile_counts0, want[1])):
            if off == L.tile_counts0 and dtype != "fp8":
                continue
            assert np.array_equal(ws[off:off + size].cpu().numpy().reshape(tiles, E, 4), ref), n
    w.release()


@pytest.mark.parametrize("H,F", [(4096, 448), (512, 64), (256, 320)])
def test_dense_ffn_of_few_rows(gpu_device, H, F):
    """The bf16 one-expert set (aps_mlp_forward): w1||w3 on the one-wave tiles up
    to 6 rows, w2 up to 12, against the same rows of a batch of row tiles."""
    from aps2026_amd import capi
    print(f"[gpu-case] dense ffn few rows H={H} F={F}", flush=True)
    g = torch.Generator(device=gpu_device)
    g.manual_seed(H + F)
    ws = [[(torch.randn(sh, generator=g, device=gpu_device) * 0.05).bfloat16()] for sh in ((F, H), (H, F), (F, H))]
    w = moe.register_moe_weights_gpu(*ws, compute_dtype=torch.bfloat16)
    x = torch.randn((300, H), generator=g, device=gpu_device).bfloat16()
    L = capi.lib()

    def run(n):
        size = L.aps_mlp_workspace_size(w.handle, n)
        scratch = torch.empty(size, dtype=torch.uint8, device=gpu_device)
        out = torch.full((n, H), float("nan"), dtype=torch.bfloat16, device=gpu_device)
        rc = L.aps_mlp_forward(w.handle, x.data_ptr(), capi.DTYPE_BF16, n, out.data_ptr(), scratch.data_ptr(), size,
                               moe._stream(gpu_device))
        assert rc == 0, capi.last_error()
        return out

    big = run(300)
    for n in (1, 5, 6, 7, 12, 13):
        assert torch.equal(run(n).view(torch.int16), big[:n].view(torch.int16)), n
    w.release()
