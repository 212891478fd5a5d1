"""What the sampler hands to the library, on the CPU."""
import torch

from yalis_amd import SamplingParams
from yalis_amd.sampling.sampler import Sampler


class Calls:
    sample_takes_most_top_k = True

    def __init__(self):
        self.seen = []

    def sample(self, logits, *rows, **word):
        self.seen.append((rows, word))
        return rows[4]

    def argmax(self, logits):
        return logits.argmax(-1)


def test_prepared_rows_are_five_tensors():
    """As a program may keep them, unpack them or make them itself; what is known beside them (the largest top_k) goes along where it is."""
    ops = Calls()
    sampler, logits = Sampler(ops, "cpu"), torch.zeros(3, 11)
    prepared = sampler.prepare([SamplingParams(top_k=5), SamplingParams(temperature=0.0), SamplingParams(top_k=7, top_p=0.5, seed=3)], [0, 1, 2])
    temperature, top_k, top_p, seeds, draws = prepared
    assert temperature.tolist() == [1.0, 0.0, 1.0] and top_k.tolist() == [5, 0, 7] and top_p.tolist() == [1.0, 1.0, 0.5]
    assert seeds.tolist() == [1234, 1234, 3] and draws.tolist() == [0, 1, 2]
    assert sampler.sample_prepared(logits, prepared, 4).tolist() == [4, 5, 6]
    assert sampler.sample_prepared(logits, (temperature, top_k, top_p, seeds, draws), 4).tolist() == [4, 5, 6]
    index = torch.tensor([2, 0], dtype=torch.int32)
    for rows in (prepared, tuple(prepared)):
        assert [t.tolist() for t in sampler.narrow(rows, index)] == [[1.0, 1.0], [7, 5], [0.5, 1.0], [3, 1234], [2, 0]]
    sampler.sample_prepared(logits[:2], sampler.narrow(prepared, index), 0)
    sampler.sample_prepared(logits[:2], sampler.narrow(tuple(prepared), index), 0)
    assert [word for _, word in ops.seen] == [{"most_top_k": 7}, {}, {"most_top_k": 7}, {}]


def test_a_row_without_top_k_gives_no_word():
    ops = Calls()
    sampler = Sampler(ops, "cpu")
    prepared = sampler.prepare([SamplingParams(top_k=5), SamplingParams()], [0, 0])
    assert prepared.most_top_k == 0
    sampler.sample_prepared(torch.zeros(2, 11), prepared, 0)
    assert ops.seen[0][1] == {}
    assert sampler.prepare([SamplingParams(temperature=0.0)], [0]) is None
    assert sampler.sample_prepared(torch.eye(3), None, 0).tolist() == [0, 1, 2]
