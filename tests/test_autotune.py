"""The tile autotuner times the flux kernel that has brick shapes: sparse Euler
evaluations run the fused kernel, so its batches need WENO on every cell."""
import pytest


def test_timed_batches_run_the_kernel_with_shapes(monkeypatch):
    import kfvm_amd
    from kfvm_amd import autotune

    class Stop(Exception):
        pass

    texts = []

    def solver(init_text, seeds):
        texts.append(init_text)
        raise Stop

    monkeypatch.setattr(kfvm_amd, "Solver", solver)
    for shape in autotune.SHAPES:
        with pytest.raises(Stop):
            autotune.time_shape(64, shape, problems=2, steps=1)
    assert len(texts) == 3
    for text in texts:
        assert kfvm_amd.parse_init(text)["wenothresh"] < 0.0
