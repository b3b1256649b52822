"""CPU build of the beam walk (lyceanem-python_amd/csrc/lem_beam_walk.h), checked ray by
ray against the oracle's brute force: tests/native/beam_walk_host.cpp casts wavefronts
of 64 rays with a common end over the grid traversal test's scenes, walked from either
end, closest hit, any hit and the native predicate, with macro blocks of 1 to 8 cells a
side; a second build runs under AddressSanitizer and UndefinedBehaviorSanitizer."""
import os

import test_grid_walk_host as walk

SRC = os.path.join(walk.NATIVE, "beam_walk_host.cpp")


def _run(tmp_path, monkeypatch, name, opt, extra, *args):
    monkeypatch.setattr(walk, "SRC", SRC)
    exe = walk._build(str(tmp_path), name, opt, ["-Wno-unused-function", *extra])
    r, lines, _ = walk._run(exe, *args)
    total = lines[-1].split()
    assert "runtime error" not in r.stderr and "AddressSanitizer" not in r.stderr, r.stderr[-3000:]
    assert r.returncode == 0 and lines[-1].endswith(" 0 mismatches"), r.stdout[-3000:]
    return int(total[1]), int(total[4]), int(total[6])


def test_beam_walk_host_matches_oracle(tmp_path, monkeypatch):
    rays, beams, refused = _run(tmp_path, monkeypatch, "beam", "-O2", ["-fopenmp"])
    assert rays > 5_000_000 and beams // 100 < refused < beams // 2


def test_beam_walk_host_sanitizers(tmp_path, monkeypatch):
    san = ["-g", "-fno-omit-frame-pointer",
           "-fsanitize=address,undefined,float-cast-overflow", "-fno-sanitize-recover=all"]
    rays, beams, refused = _run(tmp_path, monkeypatch, "beam_san", "-O1", san, "quick")
    assert rays > 100_000
