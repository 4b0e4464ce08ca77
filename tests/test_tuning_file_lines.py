"""Lines of a GEMM tuning file that no call can use are refused with their number, whatever
they hold, and nothing of the file is kept."""
import pytest

pytest.importorskip("torch")

from einsums_amd import core


@pytest.mark.parametrize("key", ["8 64 64 64 0 1 1", "8 64 64 64 -3 1 1", "8 0 64 64 1 1 1", "8 64 -1 64 1 1 1",
                                 "8 64 64 0 1 1 1", "4 9223372036854775807 64 64 1 1 1",
                                 "8 16 16 16 9223372036854775807 0 0", "8 100000 100000 8 100 0 0"])
def test_unusable_wave_entry_is_refused(tmp_path, key):
    before = core.lib.ein_gemm_tuning_count()
    f = tmp_path / "t.txt"
    f.write_text(f"# table\n8 7 7 7 1 0 0 : 64 64 0 0\n{key} : 16 16 0 0\n")
    with pytest.raises(ValueError, match="line 3"):
        core.load_gemm_tuning(f)
    assert core.lib.ein_gemm_tuning_count() == before
