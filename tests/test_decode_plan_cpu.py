"""Which form a decoded step's launches take: rules on sizes alone, no launch."""
import os

import pytest

from voice_enabled_browser_automation_amd.ops import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.KERNEL_SO), reason="the kernel library is not built")


@pytest.fixture(scope="module")
def E():
    import torch  # noqa: F401  (the HIP runtime comes with it)

    from voice_enabled_browser_automation_amd.ops import _vwa_kernels as E

    return E


@pytest.mark.parametrize("D,G,nkv", [(128, 4, 8), (128, 8, 2), (64, 4, 8)])
@pytest.mark.parametrize("P", [16, 64, 256, 1008])
def test_sessions_behind_a_prompt_share_a_chunk_where_it_is_ahead(E, D, G, nkv, P):
    """A wave to a session's own keys: always for so few of them that one wave step holds them, never where every session's chunk has a
    CU and more than a wave's steps of keys, nor for very long ones; its prefix chunks are some that the partials have room for."""
    for rows in (1, 2, 4, 8, 12, 16, 24, 32, 48, 64):
        forms = [E.decode_wave_runs(D, G, nkv, rows, P, own, 16) for own in (1, 32, 110, 300, 900)]
        assert forms[0] and forms[1] and all(0 <= f < 16 for f in forms) and not forms[4]
        groups = -(-rows // (16 // G)) * nkv
        if groups * (-(-P // 128) + 16 // G) <= 256:
            assert forms[2:] == [0, 0, 0]
        assert E.decode_wave_runs(D, G, nkv, rows, P, 32, 16 // G) == 0  # (no room for another chunk)
    assert E.decode_wave_runs(128, 4, 8, 32, P, 110, 16) and E.decode_wave_runs(128, 4, 8, 64, P, 300, 16)
    assert E.decode_wave_runs(128, 1, 8, 32, P, 1, 16) == 0          # (more runs to a group than waves)


def test_a_blocks_channels_are_split_by_the_bytes_of_their_gates(E):
    """RG-LRU of decoded rows: parts of at least 128 KB of gates and four tiles; every part has some of the block's tiles."""
    for f32, size in ((False, 2), (True, 4)):
        for bs in range(16, 1025, 16):
            tiles, n = bs // 16, E.rglru_parts(bs, f32)
            per = -(-tiles // n)
            assert n >= 1 and (n - 1) * per < tiles and (n == 1 or per >= 4)
            assert n == 1 or -(-tiles // (n - 1)) * 32 * bs * size >= 128 * 1024
    assert [E.rglru_parts(bs, False) for bs in (64, 80, 128, 256)] == [1, 1, 1, 2]
    assert [E.rglru_parts(bs, True) for bs in (64, 80, 128, 256)] == [1, 1, 1, 4]
    assert E.rglru_parts(768, True) == 12 and E.rglru_parts(8, True) == 0


def test_places_are_counted_where_many_of_few_experts_are_chosen(E):
    """Router: up to 32 experts, and 16 for every one chosen."""
    for n in range(1, 257):
        for top in range(1, min(n, 8) + 1):
            assert E.moe_ranks(n, top) == (n <= 32 and n <= 16 * top)


def test_rows_of_talking_heads_share_their_chunks(E):
    """Scores of a decoded step: a workgroup a chunk of few rows, some 768 of them of more, and three at least to a row's long context."""
    for n in (1, 4, 48, 192, 256, 384, 512, 1024):
        for chunks in (1, 2, 4, 17, 128):
            per = E.talk_step_wgs(n, chunks)
            assert min(chunks, 3) <= per <= chunks and (per <= 3 or n * per <= 768) and (per == chunks or n * (per + 1) > 768)
