"""Where the kernel library may be written to and loaded from (no compiler involved)."""

from __future__ import annotations

import os

from tinyserve_llm_amd.csrc import build


def test_a_fallback_folder_must_be_the_users_own(tmp_path, monkeypatch):
    """The per-user folder under the shared temporary directory has a name anyone can guess, and a
    library found in it is loaded into the process: it is made closed to others, and one that is
    open to others, or is a link to somewhere else, is neither searched nor written to."""
    mine = tmp_path / "mine"
    assert build._usable(str(mine), create=True) and (os.stat(mine).st_mode & 0o777) == 0o700
    assert build._usable(str(mine), create=False)
    shared = tmp_path / "shared"
    shared.mkdir()
    os.chmod(shared, 0o777)
    assert not build._usable(str(shared), create=False) and not build._usable(str(shared), create=True)
    link = tmp_path / "link"
    link.symlink_to(mine)
    assert not build._usable(str(link), create=False)
    assert not build._usable(str(tmp_path / "missing"), create=False)
    # a library with the right stamp in a folder that is open to others is not found
    monkeypatch.setattr(build, "candidate_dirs", lambda: [str(shared)])
    (shared / build.LIB_NAME).write_bytes(b"")
    (shared / (build.LIB_NAME + ".hash")).write_text(build.source_hash())
    assert build.find_current() is None
    os.chmod(shared, 0o700)
    assert build.find_current() == str(shared / build.LIB_NAME)


def test_the_source_folder_is_taken_as_it_is():
    assert build.candidate_dirs()[0] == build.HERE and build._usable(build.HERE, create=False)


def test_a_library_of_another_torch_or_python_is_stale(tmp_path, monkeypatch):
    """calls.cpp takes torch's tensors and Python's objects as their headers lay them out: a library built against others is not loaded."""
    first, second = tmp_path / "torch", tmp_path / "other" / "torch"
    for folder in (first, second):
        folder.mkdir(parents=True)
        (folder / "version.py").write_text("__version__ = '2.10.0'\ngit_version = 'a1'\n")
    monkeypatch.setattr(build, "_torch_folder", lambda: str(first))
    monkeypatch.setattr(build, "candidate_dirs", lambda: [str(tmp_path)])
    monkeypatch.setattr(build, "_usable", lambda folder, create: True)
    (tmp_path / build.LIB_NAME).write_bytes(b"")
    (tmp_path / (build.LIB_NAME + ".hash")).write_text(build.source_hash())
    assert build.find_current() == str(tmp_path / build.LIB_NAME)
    (first / "version.py").write_text("__version__ = '2.10.0'\ngit_version = 'b2'\n")
    assert build.find_current() is None
    (first / "version.py").write_text("__version__ = '2.10.0'\ngit_version = 'a1'\n")
    assert build.find_current() is not None
    with monkeypatch.context() as m:
        m.setattr(build, "_torch_folder", lambda: str(second))
        assert build.find_current() is None
    with monkeypatch.context() as m:
        m.setattr(build.sysconfig, "get_config_var", lambda name: "cpython-399-x86_64-linux-gnu")
        assert build.find_current() is None
    assert build.find_current() is not None
