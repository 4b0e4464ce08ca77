"""Index labels given as a sequence (list, tuple, numpy array; of characters or numbers) name
the same descriptor as the string of their characters."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from einsums_amd import _lib, core


def _as_sequences(labels):
    return [list(labels), tuple(labels), np.array(list(labels)), [ord(ch) for ch in labels], np.array([ord(ch) for ch in labels])]


def test_descriptors():
    t = torch.empty(4, 6)
    for labels in _as_sequences("ij"):
        assert bytes(core._desc(t, labels)) == bytes(_lib.make_desc(labels, t.shape, t.stride()))
        assert bytes(core._desc(t, labels)) == bytes(core._desc(t, "ij"))
        with pytest.raises(core.RankError):
            core._desc(torch.empty(4, 6, 8), labels)


@pytest.mark.gpu
def test_plans_and_einsum():
    rng = np.random.default_rng(1)
    A, B = rng.uniform(-1, 1, (5, 7)), rng.uniform(-1, 1, (7, 6))
    dA, dB = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    for c, a, b in zip(_as_sequences("ij"), _as_sequences("ik"), _as_sequences("kj")):
        for call in ("plan", "einsum", "contract"):
            C = torch.zeros((5, 6), dtype=torch.float64, device="cuda")
            if call == "plan":
                core.compile_plan(c, a, b).execute(0.0, C, 1.0, dA, dB)
            elif call == "einsum":
                core.einsum(c, C, a, dA, b, dB)
            else:
                core.contract(c, C, a, dA, b, dB)
            assert np.allclose(C.cpu().numpy(), A @ B, rtol=0, atol=7 * np.finfo(float).eps * 7)
