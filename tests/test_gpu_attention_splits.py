"""Automatic splits of decode attention: how many the rules pick, shown by the
result, which is bit for bit that of the same explicit count (another count, or
splits that follow the lengths, round differently), and the workspace that the
plan of splits that follow the lengths needs."""
import ctypes
import math

import pytest

pytestmark = pytest.mark.gpu


def _cache(torch, B, T, H, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    scale = torch.randn(H, 128, device="cuda", generator=g).exp_()
    return torch.randn(B, T, H, 128, device="cuda", generator=g).mul_(scale).to(torch.bfloat16)


def _inputs(torch, layout, B, T, Hkv, H, spread):
    import zipserv_asplos26_amd.attention as za
    q = torch.randn(B, 1, H, 128, device="cuda").to(torch.bfloat16)
    kv = [_cache(torch, B, T, Hkv, s) for s in (1, 2)]
    if layout != "dense":
        kv = [za.compress_kv(x, layout, retiled=True) for x in kv]
    lens = torch.arange(1, B + 1, device="cuda").mul(T).div(B, rounding_mode="floor").clamp(min=1)
    return q, kv, lens.to(torch.int32) if spread else None


def _call(layout, q, kv, Hkv, T, lens, splits):
    import zipserv_asplos26_amd.attention as za
    if layout == "dense":
        return za.flash_attn_with_kvcache_dense(q, *kv, lens, num_splits=splits)
    return za.flash_attn_with_kvcache_zipserv(q, *kv, Hkv, T, lens, num_splits=splits)


# (layout, B, T, Hkv, H, lengths spread evenly up to T, splits of every sequence)
CASES = [
    # equal ones although there are lengths: short splits, two splits of few
    # tokens, more sequences than the plan takes, the dense mode
    ("by_kv_head", 8, 1000, 8, 64, True, 8),
    ("token_major", 128, 128, 8, 64, True, 2),
    ("by_kv_head", 257, 1500, 1, 8, True, 2),
    ("dense", 8, 4000, 8, 64, True, 4),
    # one wave an item where a round of shared ones is mostly start-up
    ("by_kv_head", 256, 128, 8, 64, False, 1),
    ("by_kv_head", 384, 128, 8, 64, False, 1),
    ("by_kv_head", 384, 300, 8, 64, True, 1),
    # no more splits than leave 64 tokens a wave
    ("by_kv_head", 8, 1500, 8, 64, False, 8),
    ("by_kv_head", 2, 6000, 8, 64, False, 32),
]


@pytest.mark.parametrize("layout,B,T,Hkv,H,spread,count", CASES)
def test_automatic_splits_are_the_explicit_count(torch_cuda, layout, B, T, Hkv, H, spread, count):
    torch = torch_cuda
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the counts are those of 256 CUs")
    q, kv, lens = _inputs(torch, layout, B, T, Hkv, H, spread)
    auto, same = (_call(layout, q, kv, Hkv, T, lens, n) for n in (0, count))
    other = _call(layout, q, kv, Hkv, T, lens, 2 * count)
    torch.cuda.synchronize()
    assert torch.equal(auto.view(torch.int16), same.view(torch.int16))
    assert not torch.equal(auto.view(torch.int16), other.view(torch.int16))


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major"])
def test_workspace_without_room_for_the_plan_keeps_equal_splits(torch_cuda, layout):
    import zipserv_asplos26_amd as zs
    import zipserv_asplos26_amd.attention as za
    torch = torch_cuda
    B, T, Hkv, H = 4, 8000, 8, 64
    q, kv, lens = _inputs(torch, layout, B, T, Hkv, H, True)
    if layout == "by_kv_head":
        splits = min(64, 3 * torch.cuda.get_device_properties(0).multi_processor_count // (B * Hkv))
    else:
        splits = 64  # one workgroup per CU
    L = zs.lib()
    need = B * H * splits * (128 + 2) * 4
    ws = torch.empty(need + 8 * B, dtype=torch.uint8, device="cuda")
    desc = [za._retiled_desc(c, name="kv", device=q.device, batch_size=B, num_heads_k=Hkv) for c in kv]
    outs = []
    for room, count in ((need + 8 * B, 0), (need, 0), (need, splits), (need - 1, 0)):
        out = torch.empty(B, H, 128, dtype=torch.bfloat16, device="cuda")
        rc = L.zs_decode_attention_retiled(
            int(torch.cuda.current_stream().cuda_stream), q.data_ptr(), ctypes.byref(desc[0]),
            ctypes.byref(desc[1]), lens.data_ptr(), T, B, H, Hkv, 128, 1 / math.sqrt(128),
            out.data_ptr(), None, ws.data_ptr(), room, count)
        assert (rc == 0) == (room >= need)
        outs.append(out.view(torch.int16))
    torch.cuda.synchronize()
    # the plan, written behind the partial results: every sequence's first
    # piece follows the last one's, and longer sequences have no fewer
    plan = ws[need:].view(torch.int32).view(B, 2).cpu().tolist()
    first = 0
    for b, (at, n) in enumerate(plan):
        assert at == first and n >= 1 and (b == 0 or n >= plan[b - 1][1])
        first += n
    assert first <= B * splits
    assert not torch.equal(outs[0], outs[1])
    assert torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("layout", ["by_kv_head", "token_major"])
def test_replays_follow_the_lengths(torch_cuda, layout):
    # a captured call reads the lengths, and makes its plan of them, on every replay
    import zipserv_asplos26_amd.attention as za
    torch = torch_cuda
    B, T, Hkv, H = 6, 6000, 8, 32
    q, kv, lens = _inputs(torch, layout, B, T, Hkv, H, True)
    held = lens.clone()
    call = lambda: za.flash_attn_with_kvcache_zipserv(q, *kv, Hkv, T, held)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for step in range(4):
        held.copy_(lens.flip(0) if step % 2 else lens.clamp(max=1000 * (step + 1)))
        graph.replay()
        got = out.clone()
        want = call()
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
