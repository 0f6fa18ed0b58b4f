"""build() takes the targets that compile the reference's sources only where
those sources are: an empty folder in their place is the same as none."""
import pytest


@pytest.mark.parametrize("sources", ["none", "empty", "present"])
def test_reference_targets_need_the_sources(monkeypatch, tmp_path, sources):
    import __graft_entry__ as entry
    ref = tmp_path / "reference"
    if sources != "none":
        ref.mkdir()
    if sources == "present":
        (ref / "PIMD.f90").write_text("end\n")
    made = []
    monkeypatch.setattr(entry, "REFERENCE", str(ref))
    monkeypatch.setattr(entry.subprocess, "check_call", made.append)
    entry.build()
    asked = [t for cmd in made for t in cmd if t in ("ref", "dropin")]
    assert asked == (["ref", "dropin"] if sources == "present" else [])
    assert any("-B" in cmd and entry.PKG in cmd for cmd in made)
