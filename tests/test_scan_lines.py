"""Which sequences of a step the matrix recurrences walk in chunks, on both sides of every line."""
from types import SimpleNamespace

from servelab_amd.kernels import recurrent_ops
from servelab_amd.kernels.recurrent_ops import RecurrentOps

DECAY, DELTA, LSTM, SSD, FORGET, HEAD = (recurrent_ops._SCAN_DECAY, recurrent_ops._SCAN_DELTA, recurrent_ops._SCAN_LSTM,
                                         recurrent_ops._SCAN_SSD, recurrent_ops._SCAN_FORGET, recurrent_ops._SCAN_DELTA_HEAD)


class Table(RecurrentOps):
    _num_cus = 256


def split(mode, lens, H=8, G=8, D=128, Dv=256, told=True):
    batch = SimpleNamespace(num_seqs=len(lens), max_q_len=max(lens))
    if told:
        batch.q_lens = lens
    return Table()._scan_chunks(mode, batch, sum(lens), H, G, D, Dv)


NONE = (0, 0, 0, 0, True)


def test_one_sequence():
    for mode, line in ((DECAY, 80), (DELTA, 80), (LSTM, 80), (FORGET, 100), (HEAD, 96)):
        assert split(mode, [line - 1]) == NONE and split(mode, [line]) == (1, line, line, line, False)
    # state space: the later the more heads a group has
    for heads, line in ((8, 67), (32, 112), (56, 157), (64, 171), (112, 261)):
        assert split(SSD, [line - 1], heads, 8, 128, 64) == NONE
        assert split(SSD, [line], heads, 8, 128, 64) == (1, line, line, line, False)


def test_several_sequences():
    # 8 heads of 256 value channels are 128 blocks a sequence: 53,248 / 128 = 416 tokens together
    assert split(DECAY, [52] * 7 + [51]) == NONE and split(DECAY, [52] * 8) == (8, 416, 52, 48, False)
    assert split(DECAY, [47] * 20) == NONE and split(DECAY, [48] * 9) == (9, 432, 48, 48, False)
    # (the matrix LSTM's blocks have 15 columns; a state-space group's heads count)
    assert split(LSTM, [50] * 7) == NONE and split(LSTM, [50] * 8)[0] == 8
    assert split(SSD, [60] * 5, 64, 8, 128, 64) == NONE and split(SSD, [60] * 7, 64, 8, 128, 64)[0] == 7
    assert split(SSD, [48] * 16, 8, 1, 16, 16) == NONE and split(DECAY, [48] * 16, 16, 4, 32, 32) == NONE


def test_long_and_short_sequences():
    assert split(DECAY, [1] * 64) == NONE and split(DECAY, [79] + [1] * 64) == NONE
    assert split(DECAY, [200] + [1] * 64) == (1, 200, 200, 80, True)
    assert split(DECAY, [5, 90, 3, 80, 79, 1]) == (4, 178, 90, 80, True)
    assert split(DECAY, [48] * 9 + [47] * 2 + [1]) == (9, 432, 48, 48, True)


def test_a_bound_for_the_longest_sequence():
    batch = SimpleNamespace(num_seqs=3, max_q_len=512, q_lens=[70, 20, 1])
    assert Table()._scan_chunks(DECAY, batch, 91, 8, 8, 128, 256) == NONE
    batch.q_lens = [90, 20, 1]
    assert Table()._scan_chunks(DECAY, batch, 111, 8, 8, 128, 256) == (1, 90, 90, 80, True)


def test_a_batch_that_does_not_say():
    assert split(DECAY, [79], told=False) == NONE and split(DECAY, [80, 1], told=False) == (2, 81, 80, 1, False)
