"""The step's bump allocator: buffers of any shape and type lie one behind the other, whole and apart, whatever chunk they are in."""

import pytest
import torch

from nanospec_amd.engine.arena import Arena

SHAPES = [((), torch.float32), ((0,), torch.int64), ((3, 0, 5), torch.bfloat16), ((1,), torch.int32), ((7, 13), torch.float32),
          ([2, 3, 5], torch.bfloat16), ((257,), torch.int64), ((64, 1), torch.float32)]


@pytest.mark.parametrize("nbytes,fixed", [(0, False), (512, False), (1 << 16, True)])
def test_buffers_are_whole_and_apart(nbytes, fixed):
    a = Arena("cpu", nbytes, fixed)
    for _ in range(2):  # (the second time in the chunks merged by reset)
        a.reset()
        got = []
        for i, (shape, dtype) in enumerate(SHAPES):
            t = a.take(shape, dtype)
            assert tuple(t.shape) == tuple(shape) and t.dtype == dtype and t.is_contiguous()
            assert t.storage_offset() * t.element_size() % 256 == 0
            got.append(t.fill_(i + 1))
        assert all(bool((t == i + 1).all()) for i, t in enumerate(got))
        assert a.high_water >= 256 * len(SHAPES) and a.capacity >= a.high_water
    mark = a.mark()
    first = a.take((5,), torch.float32)
    a.release(mark)
    assert a.take((5,), torch.float32).data_ptr() == first.data_ptr()


def test_a_fixed_arena_ends():
    a = Arena("cpu", 1024, fixed=True)
    a.take((256,), torch.float32)
    with pytest.raises(RuntimeError, match="exhausted"):
        a.take((1,), torch.float32)


def test_a_merge_that_finds_no_memory_leaves_an_arena_that_works(monkeypatch):
    a = Arena("cpu")
    a.take((1 << 18,), torch.float32)
    a.take((1 << 20,), torch.float32)  # (a second chunk)
    empty = torch.empty

    def none(*args, **kwargs):
        raise torch.OutOfMemoryError("none left")

    monkeypatch.setattr(torch, "empty", none)
    with pytest.raises(torch.OutOfMemoryError):
        a.reset()
    with pytest.raises(torch.OutOfMemoryError):  # (still none: the allocation's own error, not one of the arena's books)
        a.take((4,), torch.float32)
    monkeypatch.setattr(torch, "empty", empty)
    assert a.take((4,), torch.float32).fill_(1).sum() == 4 and a.capacity >= 16
    a.reset()
    assert a.take((4,), torch.float32).storage_offset() == 0
