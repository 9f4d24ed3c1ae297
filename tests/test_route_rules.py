"""The rules that choose between kernels, where they can be checked without a GPU."""
import pytest

from agave_amd.ops import sequence as S


@pytest.mark.parametrize("n_new,heads,dk,dv,least", [
    ([500], 64, 128, 64, 0), ([48], 64, 128, 64, 0), ([64] * 4, 64, 128, 64, 0),
    ([65], 64, 128, 64, S.WHOLE_STEP),                      # one token behind a whole chunk
    ([64] + [1] * 30, 64, 128, 64, S.WHOLE_STEP), ([64] + [1] * 100, 64, 128, 64, S.WHOLE_STEP),
    ([500] + [1] * 30, 64, 128, 64, S.SSD_CHUNKS_FROM), ([1500] + [1] * 30, 128, 128, 64, S.SSD_CHUNKS_FROM),
    ([500] + [40] * 20, 64, 128, 64, 0), ([100] * 8 + [30] * 8, 64, 128, 64, 0), ([64] + [1] * 30, 2, 64, 16, 0)])
def test_which_sequences_go_through_the_state_space_form_in_chunks(n_new, heads, dk, dv, least):
    """A step of a prompt beside sequences of one token does not pay for a chunk per sequence."""
    assert S.ssd_chunked_from(tuple(n_new), heads * dv // 16, dk) == least
