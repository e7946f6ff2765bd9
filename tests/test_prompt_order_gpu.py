"""Prompt attention where its workgroups are between one and two to a CU, whose second ones come shortest first: every tile
is computed, for any number of heads."""
import pytest
import torch

from tests.test_prompt_attention_gpu import test_causal_over_a_cache as against_softmax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,first,H,G,dt", [
    (1, 2048, 65, 32, 8, torch.bfloat16),        # two to every CU
    (1, 1028, 3, 32, 8, torch.float16),          # one tile of each head more than one to a CU, 33 in all
    (3, 1700, 0, 7, 7, torch.bfloat16),          # heads that do not divide the CUs
    (2, 8500, 0, 2, 2, torch.bfloat16),          # few heads, many tiles
])
def test_every_tile_is_computed(B, T, first, H, G, dt):
    against_softmax(B, T, first, H, G, 64, dt, True)
