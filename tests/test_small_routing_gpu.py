"""Routing metadata at the borders of its one-workgroup form (four steps of 64 slots to a wavefront, 16 wavefronts: 4096
slots; 512 experts) and of the three passes behind it: bit for bit the stable sort of the oracle."""

import numpy as np
import pytest
import torch

from oracle import routing as R

pytestmark = pytest.mark.gpu
KEYS = ("expert_frequency", "expert_frequency_offset", "x_gather_idx", "s_scatter_idx", "s_reverse_scatter_idx",
        "num_activated_expert_per_token_offset")


@pytest.mark.parametrize("E", [1, 8, 100, 512, 513])
@pytest.mark.parametrize("TK", [1, 63, 64, 65, 1023, 1024, 1025, 2047, 3072, 3073, 4095, 4096, 4097, 8191, 8192, 8193])
def test_metadata_borders(dev, TK, E):
    from sonicmoe.functional import _build_metadata

    rng = np.random.default_rng(TK * 1000 + E)
    experts = (E * rng.random(TK) ** 2).astype(np.int32)  # low experts get more, some get none
    T = TK // 3 + 2
    tokens = np.sort(rng.integers(0, T - 1, TK)).astype(np.int32)  # tokens without a slot, the last one among them
    on_gpu = torch.from_numpy(experts).to(dev)
    general = _build_metadata(on_gpu, torch.from_numpy(tokens).to(dev), T, E, 1)
    ref = R.general_routing_router_metadata(tokens, experts, T, E)
    for key, got in zip(KEYS, general):
        np.testing.assert_array_equal(got.cpu().numpy(), ref[key], err_msg=key)
    K = next(k for k in (4, 3, 1) if TK % k == 0)
    choice = _build_metadata(on_gpu, None, TK // K, E, K)
    ref = R.tc_topk_router_metadata(experts.reshape(-1, K), E)
    for key, got in zip(KEYS, choice):
        np.testing.assert_array_equal(got.cpu().numpy(), ref[key], err_msg=key)


@pytest.mark.parametrize("E", [8, 256, 257, 4096])
@pytest.mark.parametrize("TK", [1, 8193, 9216, 9471, 33333])
def test_metadata_segments(dev, TK, E):
    """The three passes: segments of 1024 slots, wavefronts of 256, scans of 256 experts, LDS beyond 64 KiB at E = 4096."""
    from sonicmoe.functional import _build_metadata

    rng = np.random.default_rng(TK + E)
    experts = (E * rng.random(TK) ** 2).astype(np.int32)
    K = next(k for k in (7, 3, 1) if TK % k == 0)
    choice = _build_metadata(torch.from_numpy(experts).to(dev), None, TK // K, E, K)
    ref = R.tc_topk_router_metadata(experts.reshape(-1, K), E)
    for key, got in zip(KEYS, choice):
        np.testing.assert_array_equal(got.cpu().numpy(), ref[key], err_msg=key)
