"""The persistent scorer's dealing of its tiles: of a wide head group, dealt round (evened out over the rounds they take, or full
where all sequences of a stretch are short), and of a group in one part, a stretch to a workgroup.  Every token of every row scored,
bit for bit the definition's sum."""
import pytest
import torch

from socket_amd import hash_cache

pytestmark = pytest.mark.gpu
DEV, L, P, G = "cuda", 16, 8, 7


@pytest.mark.parametrize("B,Hkv,T,lengths", [
    (3, 4, 90001, "full"),        # a little more than a round of full tiles
    (3, 4, 90001, "ragged"),
    (1, 1, 131072, "full"),       # a row over all XCDs, fewer tiles than workgroups
    (1, 3, 33000, "full"),
    (13, 5, 40000, "short"),      # rows of no, one and a few units
    (64, 9, 1501, "full"),        # short rows, and many
    (20, 4, 12000, "full"),       # 80 rows, three sequences to a stretch
    (52, 2, 20000, "short"),      # stretches of many sequences, all lengths among them
    (64, 1, 5000, "ragged"),      # eight sequences to a stretch
    (64, 9, 1501, "one"),         # all but one of them empty
    (64, 1, 9000, "ragged"),      # about eight rows
    (64, 1, 3001, "one"),
    (40, 1, 30000, "short"),      # rows of very different lengths: a stretch of many, one of a few
])
def test_every_token_is_scored(B, Hkv, T, lengths):
    _check(B, Hkv, G, T, lengths)


@pytest.mark.parametrize("group", [2, 4])
@pytest.mark.parametrize("B,Hkv,T,lengths", [
    (1, 8, 131072, 12000),        # one and a half units of 256 a workgroup, rows and stretches ending together
    (1, 8, 131072, 4000),         # fewer units than workgroups
    (1, 8, 131072, 1),            # one a row
    (2, 5, 131072, "ragged"),
    (1, 8, 131072, "full"),
    (9, 8, 8192, "short"),        # rows of no, one and a few units, empty ones first and last
    (64, 1, 9000, "one"),
    (7, 5, 30001, "short"),
])
def test_a_stretch_to_a_workgroup(B, Hkv, T, lengths, group):
    assert hash_cache.lib().socket_score_persistent_serves(B, Hkv * group, Hkv, T, 0, L, P, 1 << P) == 1
    assert hash_cache.lib().socket_score_lanes_serve(B, Hkv * group, Hkv, T, 0, L, P, 1 << P) == 0
    _check(B, Hkv, group, T, lengths)


def _check(B, Hkv, G, T, lengths):
    g = torch.Generator(device=DEV).manual_seed(B + T)
    table = torch.rand(B, Hkv * G, L, 1 << P, generator=g, device=DEV)
    codes = torch.randint(0, 1 << P, (B, Hkv, L, T), generator=g, device=DEV, dtype=torch.int16)
    Tcap = (T + 7) // 8 * 8
    words = torch.zeros(B, Hkv, hash_cache.words_per_key(L, P), Tcap, dtype=torch.int32, device=DEV)
    hash_cache.pack_codes_into(codes, words, P, t0=0)
    norms = torch.rand(B, Hkv, Tcap, generator=g, device=DEV).half()
    lens = torch.full((B,), T, dtype=torch.int32, device=DEV)
    if lengths == "ragged":
        lens = torch.randint(0, T + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    elif lengths == "short":
        lens = torch.tensor(([0, 1, 255, 256, 257, 511, 512, 513, 1024, 8192, 8193, T, 0] * 4)[:B], dtype=torch.int32, device=DEV)
    elif isinstance(lengths, int):
        lens = torch.full((B,), lengths, dtype=torch.int32, device=DEV)
    elif lengths == "one":
        lens = torch.zeros_like(lens)
        lens[B // 2] = T - 1
    want = torch.zeros(B, Hkv * G, T, device=DEV)
    wide = codes.long().repeat_interleave(G, 1)
    for l in range(L):
        want += table[:, :, l].gather(2, wide[:, :, l])
    want *= norms[..., :T].float().repeat_interleave(G, 1)
    for dt, tol in ((torch.float32, 0.0), (torch.bfloat16, 2e-6)):
        t = table.to(dt)
        if dt != torch.float32:      # the definition on the rounded table; the matrix core's adds differ in the last place
            want.zero_()
            for l in range(L):
                want += t[:, :, l].float().gather(2, wide[:, :, l])
            want *= norms[..., :T].float().repeat_interleave(G, 1)
        out = torch.full((B, Hkv * G, (T + 3) // 4 * 4), 123.0, device=DEV)
        got = hash_cache.score_packed(hash_cache.group_q_probs(t, Hkv), words, norms, T, P, lens=lens, n_heads=Hkv * G, out=out,
                                      skip_masked=True)
        for b, n in enumerate(lens.tolist()):
            assert ((got[b, :, :n] - want[b, :, :n]).abs() <= tol * want[b, :, :n]).all(), (dt, b)
            assert (out[b, :, (n + 3) // 4 * 4:T] == 123.0).all(), (dt, b)
