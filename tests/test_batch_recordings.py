"""A batch records its graph once and replays it on whatever buffers a call passes, also when calls on
several sets of buffers are queued one after the other; only changed launch shapes or a new plan of a tree
record it again."""
import pytest

import pvfmm_amd as P

from test_batch import clouds

pytestmark = pytest.mark.gpu


def _batch(sizes, seed):
    import torch

    fmm = P.PtFMM("laplace_poten", 6, "mixed")
    cs = clouds(sizes, seed)
    trees = [P.PtFMMTree(x, x, 64).setup(fmm) for x, _ in cs]
    return trees, P.PtFMMBatch(trees), [torch.tensor(q, device="cuda:0") for _, q in cs]


def test_other_buffers_replay_the_recorded_graph(gpu):
    import torch

    trees, batch, den = _batch([3000, 9000, 700], 7)
    sets = [[d * (k + 1) + 0.1 * k for d in den] for k in range(3)]
    ref = [[t.evaluate_device(d) for t, d in zip(trees, dens)] for dens in sets]
    batch.evaluate_device(sets[0])
    assert batch.recordings() == 1
    for rep in range(3):
        outs = [[torch.zeros_like(d) for d in den] for _ in sets]
        torch.cuda.synchronize()
        for dens, out in zip(sets, outs):  # queued back to back
            batch.evaluate_device(dens, out, sync=False)
        torch.cuda.ExternalStream(batch.stream_handle()).synchronize()
        for k in range(len(sets)):
            for o, r in zip(outs[k], ref[k]):
                assert torch.equal(o, r), (rep, k)
        trees[0].evaluate_device(torch.ones_like(den[0]))
    assert batch.recordings() == 1
    batch.evaluate_device(sets[1])
    assert batch.recordings() == 1
    trees[1].setup(P.PtFMM("laplace_poten", 8, "mixed"))
    batch.evaluate_device(sets[1])
    assert batch.recordings() == 2


def test_changed_launch_shapes_record_the_graph_again(gpu):
    """Every change of a shape that the launches use, whatever the value without effect beside it: a
    key that adds the two up takes (1024, 16) and (1023, 80) for the same shapes."""
    trees, batch, den = _batch([3000, 5000], 8)
    batch.evaluate_device(den)
    trees[0].set_tuning(hadamard_tiles_per_block=16, gemm_split_blocks=1024, hadamard_vec_targets_per_wave=16)
    batch.evaluate_device(den)
    assert batch.recordings() == 1
    trees[0].set_tuning(hadamard_tiles_per_block=16, gemm_split_blocks=1023, hadamard_vec_targets_per_wave=80)
    batch.evaluate_device(den)
    assert batch.recordings() == 2
    trees[0].set_tuning(hadamard_tiles_per_block=16, gemm_split_blocks=1023, hadamard_vec_targets_per_wave=3)
    batch.evaluate_device(den)
    assert batch.recordings() == 2
    trees[1].set_tuning(hadamard_tiles_per_block=8, gemm_split_blocks=1024)
    batch.evaluate_device(den)
    assert batch.recordings() == 3
