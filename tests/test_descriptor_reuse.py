"""Descriptors that the einsum call reuses by content equal freshly made ones for every shape
and stride order, and a rank mismatch is refused on each call."""
import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib, core


def _same(a, b):
    return bytes(a) == bytes(b)


def test_reused_descriptor_equals_a_new_one():
    base = torch.empty(4, 6, 8)
    views = [base, base.transpose(0, 2), base[:, ::2], base[1:3, :, 1:5], base.permute(2, 0, 1), base[0], base[0, 0, 0],
             base.expand(4, 6, 8), torch.empty(6, 4, 8), base[:, :, :1].expand(4, 6, 8)]
    for t in views * 2:
        for labels in ("ijk"[:t.dim()], "kji"[:t.dim()], "iii"[:t.dim()]):
            assert _same(core._desc(t, labels), _lib.make_desc(labels, t.shape, t.stride()))


def test_bounded():
    for n in range(core._DESCS_KEPT + 10):
        core._desc(torch.empty(n), "i")
    assert len(core._descs) <= core._DESCS_KEPT


def test_rank_mismatch_is_refused_each_time():
    for _ in range(2):
        with pytest.raises(core.RankError):
            core._desc(torch.empty(2, 2), "ijk")
