"""Decode attention over ragged batches with automatic splits, against the fp64
oracle within zs_testutil.attention_tolerance: equal splits (short sequences),
compressed against dense bit for bit where both cut the same pieces, and splits
that follow the sequences' lengths (one chunk for the whole call, as many splits
as a sequence needs), which long splits of a compressed cache have."""
import numpy as np
import pytest

from test_gpu_attention import _check, _run

pytestmark = pytest.mark.gpu


def _lens(B, T, seed):
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, T + 1, B)
    lens[0], lens[-1] = T, 0
    return [int(v) for v in lens]


CASES = [
    (2, 500, [500, 1]),                      # one long, one token
    (3, 1100, [0, 1100, 0]),                 # all pieces in one sequence
    (4, 2000, [2000] * 4),                   # equal lengths: the even split
    (4, 2000, [0, 0, 0, 0]),                 # no tokens at all
    (5, 640, [640, 16, 17, 15, 9999]),       # band edges, a length past the cache
    (64, 260, _lens(64, 260, 1)),            # one wave's lanes of lengths
    (65, 260, _lens(65, 260, 2)),            # one more than a wave holds
    (130, 150, _lens(130, 150, 3)),          # three chunks of lengths
]


@pytest.mark.parametrize("B,T,lens", CASES)
@pytest.mark.parametrize("retiled", [False, True])
def test_ragged_head_major(torch_cuda, B, T, lens, retiled):
    used = [min(v, T) for v in lens]
    res = _run(torch_cuda, B, T, 2, 8, seqlens=used, splits=0, seed=B, retiled=retiled, passed=lens)
    # the dense kernel cuts the same pieces where its split count is the same
    # (short sequences: the minimum split length decides in both)
    _check(res, used, exact=B <= 5 and T < 1000)


@pytest.mark.parametrize("B,T,lens", CASES)
def test_ragged_token_major(torch_cuda, B, T, lens):
    used = [min(v, T) for v in lens]
    _check(_run(torch_cuda, B, T, 8, 16, seqlens=used, splits=0, seed=B + 1, retiled=True,
                layout="token_major", passed=lens), used, exact=False)


# (layout, B, T, Hkv, H, lengths), all with splits that follow the lengths
BALANCED = [
    ("by_kv_head", 2, 9000, 8, 64, [9000, 1]),                # nearly all pieces in one sequence
    ("by_kv_head", 3, 9000, 4, 8, [0, 9000, 20000]),          # an empty one, one past the cache
    ("by_kv_head", 4, 16000, 2, 8, [0, 0, -7, 0]),            # no tokens at all
    ("by_kv_head", 64, 2000, 2, 8, _lens(64, 2000, 1)),       # one wave's lanes of lengths
    ("by_kv_head", 65, 1700, 2, 8, _lens(65, 1700, 2)),       # one more
    ("by_kv_head", 256, 1000, 1, 4, _lens(256, 1000, 3)),     # as many as the plan takes
    ("by_kv_head", 154, 960, 5, 10, _lens(154, 960, 4)),      # one wave an item: idle and busy waves
                                                              # share the last workgroups
    ("token_major", 3, 9000, 8, 16, [9000, 16, 17]),
    ("token_major", 2, 700, 8, 16, [700, 90]),                # one workgroup a CU
    ("token_major", 64, 512, 8, 8, _lens(64, 512, 5)),
    ("token_major", 65, 530, 8, 8, _lens(65, 530, 6)),
    ("token_major", 200, 500, 8, 8, _lens(200, 500, 7)),      # fewer pieces than batch * splits
    ("token_major", 256, 520, 8, 8, _lens(256, 520, 8)),
]


@pytest.mark.parametrize("layout,B,T,Hkv,H,lens", BALANCED)
def test_splits_that_follow_the_lengths(torch_cuda, layout, B, T, Hkv, H, lens):
    used = [min(max(v, 0), T) for v in lens]
    _check(_run(torch_cuda, B, T, Hkv, H, seqlens=used, splits=0, seed=B, retiled=True,
                layout=layout, passed=lens), used, exact=False)


@pytest.mark.parametrize("B,T,lens", [(3, 9000, [9000, 40, 5000]), (40, 1600, _lens(40, 1600, 9))])
def test_splits_that_follow_the_lengths_canonical(torch_cuda, B, T, lens):
    _check(_run(torch_cuda, B, T, 2, 8, seqlens=lens, splits=0, seed=B), lens, exact=False)


def test_ragged_large_grid(torch_cuda):
    # a full round of shared items, the last workgroups past the last piece
    lens = [4096, 100, 2048, 3000, 1, 0, 4000, 511] * 2
    _check(_run(torch_cuda, 16, 4096, 8, 32, seqlens=lens, splits=0, seed=9, retiled=True), lens,
           exact=False)


def test_ragged_lengths_past_the_cache_are_clamped(torch_cuda):
    import zipserv_asplos26_amd.attention as za
    torch = torch_cuda
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = [torch.randn(3, 600, 8, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in "kv"]
    q = torch.randn(3, 1, 64, 128, device="cuda", generator=g).to(torch.bfloat16)
    for layout in ("by_kv_head", "token_major"):
        k, v = (za.compress_kv(t, layout=layout, retiled=True) for t in x)
        outs = [za.flash_attn_with_kvcache_zipserv(
            q, k, v, 8, 600, torch.tensor(s, dtype=torch.int32, device="cuda"))
            for s in ([600, 0, 77], [1 << 30, -5, 77])]
        torch.cuda.synchronize()
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("B,T,Hkv,H,ragged", [
    (40, 600, 8, 16, False),    # 320 units: two shared splits, 640 of 768 places
    (50, 1500, 8, 16, False),   # 400 units: one-wave items (a shared split fills half a round)
    (50, 1500, 8, 16, True),
    (97, 300, 8, 8, False),     # 776 units: just over one round of shared items
    (3, 4000, 1, 8, False),     # three units: splits at their smallest
])
def test_automatic_splits_of_larger_grids(torch_cuda, B, T, Hkv, H, ragged):
    lens = _lens(B, T, B) if ragged else None
    _check(_run(torch_cuda, B, T, Hkv, H, seqlens=lens, splits=0, seed=B, retiled=True), lens,
           exact=False)
