"""The cuts of the Mamba2 correction backward: token blocks of the unit kernel below 4096 and
heads of the dC kernel split over workgroups, which few token tiles take."""

import itertools

import pytest

from ringmaster_amd import abi


@pytest.mark.gpu
@pytest.mark.parametrize("Bsz,T,H,d,G,n", [
    (2, 2600, 24, 64, 2, 64),    # 44 tiles: 12 heads of a group in 5 uneven splits, 1024-token blocks
    (3, 513, 16, 128, 1, 128),   # 9 tiles: a split per head, a last block of one token
    (1, 256, 4, 64, 1, 128),     # one tile, one block
    (1, 8192, 4, 64, 1, 64),     # 32 tiles: 4 splits, 32 blocks of 256
])
def test_split_backward_matches_oracle(Bsz, T, H, d, G, n):
    from tests.test_gpu_mamba import _check_bwd, _inputs

    print(f"case {(Bsz, T, H, d, G, n)}", flush=True)
    _check_bwd(_inputs(Bsz, T, H, d, G, n, seed=160), H, d)


def test_split_keeps_within_the_scratch_array():
    """A shape whose whole cut (4096-token blocks, no head split) fits the allocation-free
    entry's array fits it with its own cut too, and no other shape's workspace grows."""
    most = 96 << 20
    for b, T, H, d, G, n in itertools.product((1, 2, 8, 16, 64), (1, 255, 512, 4097, 8192, 100000),
                                              (4, 24, 64, 128), (64, 128), (1, 2), (64, 128)):
        got = abi.lib().rmx_mamba2_cp_correction_bwd_workspace(b, T, H, d, G, n)
        if not got:
            continue
        state = b * H * d * n
        whole = -(-T // 4096) * state * 4 + 6 * state + 4 * b * H * T + 256
        assert whole <= got <= max(whole, most), (b, T, H, d, G, n, got, whole)
