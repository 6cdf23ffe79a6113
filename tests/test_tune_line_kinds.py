"""Line entries of the launch-shape cache per kind of line (x lines; y and z
lines): the text file and what set and get make of them (host code, no GPU)."""
import pytest


@pytest.fixture
def tune():
    from compact_schemes_amd import tune as t
    t.clear()
    yield t
    t.clear()


def _body(path):
    return sorted(ln for ln in path.read_text().splitlines() if ln and not ln.startswith("#"))


def test_entries_per_kind_round_trip(tune, tmp_path):
    src = tmp_path / "kinds.txt"
    lines = ["line 0 300 1 1 0 8 0", "line 1 300 0 0 0 16 1", "line 1 96 0 0 0 32",
             "line 0 200 0 0 0 16 0", "line 0 200 0 0 0 32 1"]
    src.write_text("\n".join(lines) + "\n")
    tune.load(src)
    assert tune.get_line(0, 300, 1, 1) == 8             # x lines
    assert tune.get_line(1, 300) == 16                  # y/z lines: x lines have none
    assert tune.get_line(1, 96) == 32
    assert tune.get_line(0, 200) == 16
    tune.save(tmp_path / "again.txt")
    assert _body(tmp_path / "again.txt") == sorted(lines)
    tune.set_line(0, 200, 8)                            # by hand: both kinds
    tune.set_line(1, 300, 0)                            # clears both kinds
    assert tune.get_line(1, 300) == 0
    tune.save(tmp_path / "again.txt")
    assert _body(tmp_path / "again.txt") == sorted([lines[0], lines[2], "line 0 200 0 0 0 8"])


@pytest.mark.parametrize("text", ["line 0 64 0 0 0 8 2\n", "line 0 64 0 0 0 8 -1\n", "line 0 64 0 0 0 8 0 1\n",
                                  "line 0 1024 0 0 0 8 0\n", "line 0 64 0 0 0 12 1\n"])
def test_bad_kinds_rejected(tune, tmp_path, text):
    import compact_schemes_amd as cs
    path = tmp_path / "bad.txt"
    path.write_text(text)
    with pytest.raises(cs.CsError) as err:
        tune.load(path)
    assert f"{path}:1:" in str(err.value)
    assert tune.get_line(0, 64) == 0
