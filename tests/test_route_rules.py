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


@pytest.mark.parametrize("n_new", [[1], [5, 1, 1, 1, 7], [1] * 20, [16, 16, 1, 15, 3], [40, 2, 2, 2, 2, 2, 90]])
@pytest.mark.parametrize("run", [2, 4, 5, 16])
def test_sequences_among_neighbouring_rows(n_new, run):
    from agave_amd.engine.step import Step
    cu = [sum(n_new[:i]) for i in range(len(n_new) + 1)]
    step = Step(**{**dict.fromkeys(Step.__dataclass_fields__), "cu": cu, "n_new": n_new, "seqs_a_run": {}})
    seq = [i for i, n in enumerate(n_new) for _ in range(n)]
    assert step.most_seqs(run) == step.most_seqs(run) == max(len(set(seq[a:a + run])) for a in range(0, len(seq), run))


@pytest.mark.parametrize("pairs,experts,ff,hidden,rows", [
    (8192, 16, 2048, 2048, 128), (2048, 16, 2048, 2048, 128), (2047, 16, 2048, 2048, 64), (256, 16, 2048, 2048, 64), (255, 16, 2048, 2048, 16),
    (6002, 16, 32, 32, 64), (9003, 12, 96, 64, 64), (6002, 8, 512, 512, 64), (2048, 4, 2048, 1024, 64), (8192, 64, 512, 2048, 128),
    (31, 1, 512, 512, 16), (32, 1, 512, 512, 64)])
def test_rows_of_a_tile_of_sorted_pairs(pairs, experts, ff, hidden, rows):
    """The largest tiles only where their workgroups fill the chip: small experts' tiles would be mostly empty."""
    from agave_amd.ops import routed
    tm, tiles, cap = routed.tile_plan(pairs, experts, True, ff, hidden)
    assert tm == rows and cap == tiles * tm and tiles >= -(-pairs // tm) + experts
    assert routed.tile_plan(pairs, experts)[0] == (64 if pairs >= 32 * experts else 16)


@pytest.mark.parametrize("n,experts,top,ff,hidden,among", [
    (1, 16, 4, 2048, 2048, True), (32, 16, 4, 2048, 2048, True), (512, 16, 4, 2048, 2048, True), (700, 16, 4, 2048, 2048, False),
    (1024, 16, 4, 2048, 2048, True), (3001, 16, 4, 2048, 2048, True), (64, 8, 2, 1536, 1536, True), (2048, 8, 2, 1536, 1536, False),
    (400, 4, 1, 4096, 4096, False), (1300, 32, 4, 1024, 2048, False), (1300, 64, 4, 1024, 2048, True), (40, 1, 1, 64, 64, True)])
def test_where_a_shared_expert_is_one_of_the_experts(n, experts, top, ff, hidden, among):
    from agave_amd.parts.routed_ffn import merges
    assert merges(n, experts, top, ff, hidden) == among


def test_a_shared_expert_of_a_small_test_goes_both_ways():
    """The sizes that the GPU test of the shared expert runs."""
    from agave_amd.parts.routed_ffn import merges
    assert {merges(n, 6, 2, 1024, 1024) for n in (1, 6, 40, 130, 700, 1010)} == {True, False}


def test_how_a_steps_tokens_lie():
    """The kernels that take four positions at a time are told whether a step is one sequence from a multiple of four on."""
    from types import SimpleNamespace as Step
    from agave_amd.ops.attention import tokens_apart
    assert tokens_apart(Step(n_seqs=1, pos0=[0])) == 0 == tokens_apart(Step(n_seqs=1, pos0=[512]))
    assert tokens_apart(Step(n_seqs=1, pos0=[153])) == 1 and tokens_apart(Step(n_seqs=3, pos0=[0, 0, 0])) == 3


@pytest.mark.parametrize("m,n,k,slices", [
    (16, 4096, 8192, 1), (17, 2048, 4092, 1), (17, 2048, 4096, 8), (17, 4096, 4096, 1), (33, 2048, 1024, 1), (33, 1024, 1024, 1), (33,
    2048, 2048, 8), (48, 512, 1100, 1), (64, 1024, 1100, 1), (64, 6144, 1024, 4), (64, 2048, 1020, 1), (64, 2048, 5376, 8), (100, 2048,
    1024, 1), (192, 840, 1036, 1), (150, 6144, 2048, 1), (400, 2048, 1280, 4), (400, 2048, 2048, 4), (700, 3072, 2048, 4), (777, 2048,
    5376, 4), (300, 10752, 4096, 2), (1200, 6144, 8192, 1), (64, 10752, 2048, 4), (200, 2048, 5376, 8), (100, 512, 2048, 8), (17, 2304,
    9216, 8), (17, 4096, 8192, 8), (777, 2048, 2048, 4), (777, 3072, 2048, 4), (64, 2050, 2048, 1), (64, 2048, 2046, 1), (900, 3072, 2048, 2), (1400, 2048, 2048, 2), (2000, 2048, 5376, 2), (1400, 3072, 2048, 2)])
def test_where_32_bit_products_are_shared_out_along_their_columns(m, n, k, slices):
    """Only where both were measured and the slices with their sum were faster."""
    from agave_amd.ops import kernels
    assert kernels.lib("gemm").agave_gemm_slices_for(m, n, k) == slices


@pytest.mark.parametrize("n,top,hidden,adds_up", [
    (1, 5, 2048, True), (6, 64, 4096, True), (1, 10, 8192, True), (1, 12, 7168, False), (6, 16, 8192, False), (6, 5, 16384, True), (6, 6, 14000, True),
    (6, 7, 16384, False), (47, 16, 12288, False), (48, 16, 12288, True), (48, 24, 16384, False), (300, 24, 12288, True), (300, 25, 5120, False),
    (3001, 9, 16384, True)])
def test_where_the_norm_adds_up_a_tokens_pairs(n, top, hidden, adds_up):
    """Only where the two kernels were measured to take longer."""
    from agave_amd.ops.routed import norm_adds_up
    assert norm_adds_up(n, top, hidden) == adds_up


def test_which_steps_hand_on_their_projections_in_slices(monkeypatch):
    """17 to 64 tokens of a packed product in at most as many slices as the kernels add up: decode steps whose heads the one kernel
    takes, and prompts of one sequence whatever their heads."""
    import os
    import re
    from types import SimpleNamespace as Some
    import agave_amd
    from agave_amd.ops import attention, gemm_mfma, kernels
    slices = {}
    monkeypatch.setattr(gemm_mfma, "slices_for", lambda n, out, k: slices.setdefault("made", 4))
    linear = Some(packed=object(), out_features=4096, in_features=2560)

    def takes(n, seqs, head=256, of=linear):
        return attention.adds_slices(Some(n_tokens=n, n_seqs=seqs, is_decode=seqs == n), of, head)
    assert [n for n in (1, 16, 17, 33, 64, 65) if takes(n, n)] == [17, 33, 64] == [n for n in (16, 17, 33, 64, 65, 128) if takes(n, 1)]
    assert not takes(40, 2) and not takes(40, 39)                    # prompts of several sequences
    assert takes(40, 40, 64) and takes(40, 40, 128) and not takes(40, 40, 80) and takes(40, 1, 80)
    assert not takes(40, 40, of=Some(packed=None, out_features=4096, in_features=2560))
    slices["made"] = kernels.QK_MAX_SLICES + 1
    assert not takes(40, 40) and not takes(40, 1)
    with open(os.path.join(os.path.dirname(agave_amd.__file__), "csrc", "qk_rope.h")) as f:
        assert int(re.search(r"#define QK_MAX_SLICES (\d+)", f.read()).group(1)) == kernels.QK_MAX_SLICES
