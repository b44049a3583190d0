"""Which steps go through the mLSTM's matrix memory in chunks: never one whose token-by-token kernels were measured clearly
faster, always one where chunks were."""
import pytest

from arle_amd.kernels import ops

# (portions, rows of a portion, decoded rows, heads, head size) and what was faster by a tenth and more (us a layer on MI355X,
# token by token / in chunks)
MEASURED = [
    ((1, 96, 0, 20, 128), True), ((1, 96, 16, 20, 128), True),          # 53 / 34, 84 / 69
    ((1, 96, 32, 20, 128), False), ((1, 96, 64, 20, 128), False),       # 112 / 126, 164 / 224
    ((1, 96, 256, 20, 128), False), ((1, 128, 16, 20, 128), True),      # 502 / 1,331, 98 / 70
    ((1, 128, 64, 20, 128), False), ((1, 256, 48, 20, 128), True),      # 177 / 225, 215 / 181
    ((1, 256, 128, 20, 128), False), ((1, 512, 64, 20, 128), True),     # 342 / 537, 352 / 252
    ((1, 512, 128, 20, 128), False), ((1, 1024, 128, 20, 128), True),   # 468 / 557, 691 / 619
    ((1, 1024, 256, 20, 128), False), ((1, 2048, 128, 20, 128), True),  # 986 / 1,402, 1,168 / 679
    ((64, 100, 0, 20, 128), True), ((16, 512, 64, 20, 128), True),      # 1,078 / 412, 1,523 / 593
    ((1, 96, 128, 8, 64), False), ((1, 128, 128, 8, 64), False),        # 60 / 110, 72 / 111
    ((1, 192, 128, 8, 64), False), ((1, 512, 128, 8, 64), True),        # 95 / 112, 211 / 123
    ((1, 1024, 256, 8, 64), True), ((64, 128, 0, 8, 64), True),         # 417 / 296, 167 / 92
    ((1, 96, 128, 4, 128), False), ((1, 128, 64, 4, 128), True),        # 91 / 142, 84 / 75
    ((1, 128, 128, 4, 128), False), ((1, 1024, 256, 4, 128), True),     # 104 / 142, 500 / 336
]


@pytest.mark.parametrize("step,chunks", MEASURED)
def test_the_faster_form_is_taken(step, chunks):
    portions, rows, decoded, heads, size = step
    assert ops.mlstm_chunks_preferred(rows, portions * rows + decoded, portions + decoded, heads, size, size) == chunks


def test_decoded_rows_and_other_head_sizes_go_row_by_row():
    assert not ops.mlstm_chunks_preferred(1, 8, 8, 20, 128, 128)
    assert not ops.mlstm_chunks_preferred(95, 95, 1, 20, 128, 128)
    for sizes in ((48, 64), (64, 160), (130, 70)):
        assert not ops.mlstm_chunks_preferred(2048, 2048, 1, 20, *sizes)


def test_a_step_whose_chunks_would_not_fit_the_workspace_goes_row_by_row():
    """20 heads of 128 x 128: a state of 1.31 MB a chunk, so 4 GiB are 3,276 of them."""
    assert ops.mlstm_chunks_preferred(40960, 40960, 1, 20, 128, 128)
    assert not ops.mlstm_chunks_preferred(220000, 220000, 1, 20, 128, 128)
    assert not ops.mlstm_chunks_preferred(60000, 60000, 1, 96, 128, 128)
