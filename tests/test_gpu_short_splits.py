"""The scan's form for short splits (one chunk of 64 positions per wavefront at most): around its limit of 64 positions per
wavefront, with wavefronts that have no chunk, a chunk of one position, empty splits and sequences shorter than the batch's
longest, for every key and value format; against the oracle, with the same positions selected by other split lengths."""
import pytest
import torch

from tests.helpers import make_case, to_device
from tests.test_gpu_fused import SCHEME_GEOMETRY, check_against_oracle, run_fused

pytestmark = pytest.mark.gpu


# sixteen wavefronts up to four query heads per kv-head, eight beyond: the limit is 1024 and 512 positions
@pytest.mark.parametrize("G,S,lens,split_len", [
    (4, 63, [63, 1], 256), (4, 64, [64, 0], 256), (4, 1000, [1000, 130], 256), (4, 1025, [1025, 1024], 1024),
    (4, 1100, [1100, 1024], 1280), (1, 1024, [1024, 961], 1024), (8, 513, [513, 512], 512), (8, 600, [600, 449], 768)])
@pytest.mark.parametrize("scheme", sorted(SCHEME_GEOMETRY))
def test_short_splits_match_the_oracle(scheme, G, S, lens, split_len):
    from jetfire_amd import _lib
    kb, vb, gs = SCHEME_GEOMETRY[scheme]
    c = make_case(31 + S + G, 2, G, 1, S, kb, vb, gs, lens=lens, extra_blocks=2, k_asym=scheme.startswith("a"))
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        out = [t.clone() for t in run_fused(scheme, c, d, S, 64)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    check_against_oracle(scheme, c, S, 64, out)
    again = run_fused(scheme, c, d, S, 64)
    assert torch.equal(out[4], again[4]) and torch.equal(out[7], again[7])


# (four emission segments of L / 4 positions each: the short form works through 256 of each)
@pytest.mark.parametrize("G,S,lens,split_len,K", [
    (4, 1000, [1000, 513], 1280, 64), (4, 1000, [1000, 257], 1280, 512), (4, 700, [700, 641], 2048, 64),
    (1, 300, [300, 257], 2048, 64), (2, 1024, [1024, 770], 4096, 256)])
@pytest.mark.parametrize("scheme", ["k3v2", "k4v4", "b4v4", "a2v2"])
def test_a_split_longer_than_the_sequence_keeps_every_position(scheme, G, S, lens, split_len, K):
    """Split lengths beyond one chunk per wavefront for a sequence that has no more positions than that."""
    from jetfire_amd import _lib
    kb, vb, gs = SCHEME_GEOMETRY[scheme]
    c = make_case(57 + S + G, 2, G, 1, S, kb, vb, gs, lens=lens, extra_blocks=2, k_asym=scheme.startswith("a"))
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        out = [t.clone() for t in run_fused(scheme, c, d, S, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    check_against_oracle(scheme, c, S, K, out)
