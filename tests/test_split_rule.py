"""Which launches go to the split attention kernels."""
import pytest

from warpir_amd import api


@pytest.mark.parametrize("part", ["forward", "backward"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_one_program_per_cu_splits_at_every_length(part, d, causal):
    for programs in (1, 32, 255, 256):
        assert all(api._split_wins(part, programs, seq, d, causal) for seq in (64, 128, 576, 8192))
    assert not api._split_wins(part, 0, 0, d, causal) and not api._split_wins(part, 513, 8192, d, causal)


# heads, S, D, causal, whether the forward and the backward are faster split (measured, with 5% or more between them)
MEASURED = [(256, 64, 64, True, False, False), (128, 128, 128, True, False, False), (85, 192, 64, True, False, False),
            (64, 256, 128, True, False, False), (51, 320, 64, True, False, False), (32, 320, 128, True, True, True),
            (42, 384, 128, True, False, False), (22, 384, 64, True, True, True), (32, 512, 64, True, True, True),
            (21, 768, 128, True, False, True), (16, 1024, 128, True, True, True), (8, 2048, 64, True, True, True),
            (128, 128, 64, False, None, False), (42, 384, 64, False, None, False), (17, 512, 64, False, None, True),
            (32, 512, 128, False, None, False), (12, 1280, 128, False, None, True), (8, 2048, 64, False, None, True)]


@pytest.mark.parametrize("heads,seq,d,causal,forward,backward", MEASURED)
def test_a_second_round_of_programs_needs_long_sequences(heads, seq, d, causal, forward, backward):
    programs = heads * seq // 32
    assert 256 < programs <= 512
    assert api._split_wins("backward", programs, seq, d, causal) == backward
    if forward is not None:
        assert api._split_wins("forward", programs, seq, d, causal) == forward
