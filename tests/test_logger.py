"""The log of the operator's ratios: a line a message, appended, whatever stands at the path before."""
import os

import pytest

import my_utils


@pytest.mark.parametrize("place", ["plain.log", os.path.join("a", "b", "made.log")])
def test_lines_are_appended_and_the_folder_made(monkeypatch, tmp_path, capsys, place):
    log, path = my_utils.Logger, tmp_path / place
    monkeypatch.setattr(log, "enabled", True)
    monkeypatch.setattr(log, "log_file_path", str(path))
    log.log("first")
    log.log(lambda: "second")
    log.log_warning("third")
    assert [line.split(" - ", 1)[1] for line in path.read_text().splitlines()] == ["first", "second", "WARNING: third"]
    path.unlink()
    if path.parent != tmp_path:
        path.parent.rmdir()  # (gone between two lines)
    log.log("fourth")
    assert path.read_text().endswith(" - fourth\n") and path.read_text().count("\n") == 1

    def fails():
        raise ValueError("no number")
    descriptors = len(os.listdir("/proc/self/fd"))
    with pytest.raises(ValueError):
        log.log(fails)
    assert len(os.listdir("/proc/self/fd")) == descriptors and path.read_text().count("\n") == 1
    monkeypatch.setattr(log, "log_file_path", str(tmp_path))
    log.log("nowhere")
    assert "Unable to write" in capsys.readouterr().out
    monkeypatch.setattr(log, "log_file_path", str(path))
    monkeypatch.setattr(log, "enabled", False)
    log.log("off")
    assert path.read_text().count("\n") == 1
