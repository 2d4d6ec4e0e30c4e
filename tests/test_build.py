"""The incremental build's dependencies: every output lists each source and
header that it is compiled from."""

from __future__ import annotations

import os
import re

from rollfast_amd import build


def _included(path, seen):
    """The repository's own files that `path` includes, itself among them."""
    path = os.path.normpath(path)
    if path in seen:
        return seen
    seen.add(path)
    for name in re.findall(r'^\s*#\s*include\s+"([^"]+)"', open(path).read(), re.M):
        for folder in (os.path.dirname(path), build.CSRC, os.path.join(build.REPO, "include")):
            if os.path.exists(os.path.join(folder, name)):
                _included(os.path.join(folder, name), seen)
                break
    return seen


def test_sources_of_cover_every_included_header():
    for cmd, obj in build._compile_jobs() + [build._pyhost_job()]:
        root = next(a for a in cmd if a.endswith((".hip", ".cpp")))
        missing = _included(root, set()) - set(build._sources_of(obj))
        assert not missing, (os.path.basename(obj), sorted(missing))
