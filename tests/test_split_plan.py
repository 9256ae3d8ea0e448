"""Row parts and column chunks of a step's projection and delta stages
(engine._split_plan): whatever the cut, the tasks cover every block once and
keep what each kernel variant promises.  CPU only."""

from __future__ import annotations

import sys

import pytest
import torch

from scao_amd import _lib as L
from scao_amd import engine as E
from scao_amd.preconditioner import SparsePreconditioner


def _items(shapes, k, dim, half):
    out = []
    for shp in shapes:
        p = torch.zeros(shp, dtype=torch.bfloat16 if half else torch.float32)
        pre = SparsePreconditioner(p, k_min=k, k_max=k, max_precond_dim=dim)
        out.append(E.PItem(p=p, graw=p, gmom=None, st={}, group={}, pre=pre, phase2=True, step=3,
                           lars=True, leaves=pre.step_leaf_list(), fp32=not half, half=int(half)))
    return out


SHAPES = [[(64, 64)], [(33, 257)], [(1000, 1537), (513, 2049)], [(2048, 2048)] * 4,
          [(4096, 300)], [(2048, 2048)] * 40, [(128, 8192), (8192, 128)], [(31, 31)]]


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("k", [8, 64, 100, 256, 320])
@pytest.mark.parametrize("shapes", SHAPES)
def test_tasks_cover_blocks_once(shapes, k, half):
    items = _items(shapes, k, 2048, half)
    arrays, _, _, leaves = E._build_structure(items)
    tab = E._leaf_table(leaves, items, E.Workspace(torch.device("cpu")))
    cover = {}
    for kind, arr in arrays.items():
        if not kind.startswith("proj"):
            continue
        var = int(kind[4:])
        for t in arr:
            li, j0, c0, part = int(t["idx"]), int(t["a"]), int(t["b"]) & 0xffff, int(t["b"]) >> 16
            e = tab[li]
            m, n, kp = int(e["m"]), int(e["n"]), int(e["k"])
            parts = max(1, (int(e["flags"]) >> L.LF_NSPLIT_SHIFT) & 255)
            assert part < parts
            rows = -(-m // (E.PROJ_CHUNK * parts)) * E.PROJ_CHUNK      # the kernel's split_rows
            i0, i1 = part * rows, min(m, (part + 1) * rows)
            assert i0 < i1                                              # no empty part
            height = 256 if var & 8 else 128 if var & 4 else 64
            assert c0 % height == 0 and c0 + height <= kp
            assert bool(var & 2) == (c0 == 0)
            if var & 1:
                assert (i1 - i0) % E.PROJ_CHUNK == 0 and j0 + L.PROJ_COLS <= n
                assert (var >> 4) == (1 if half else 0)
            else:
                assert height == 64 and var < 4
            for c in range(c0, c0 + height, 64):
                key = (li, j0, c, part)
                assert key not in cover
                cover[key] = 1
    want = 0
    for li, (lf, *_) in enumerate(leaves):
        if not lf.use_kronecker:
            continue
        e = tab[li]
        parts = max(1, (int(e["flags"]) >> L.LF_NSPLIT_SHIFT) & 255)
        chunks = (int(e["flags"]) >> L.LF_DCHUNK_SHIFT) & 255
        kp = int(e["k"])
        want += parts * -(-lf.n // L.PROJ_COLS) * (kp // 64)
        assert parts == 1 or chunks                    # planes of T are added by the chunks
        part_tasks = [t for t in arrays["dpart"] if int(t["idx"]) == li]
        seen = {(int(t["a"]), int(t["b"]) & 0xffff, int(t["b"]) >> 16) for t in part_tasks}
        assert len(seen) == len(part_tasks) == chunks * (kp // 64) ** 2
        if chunks:
            assert (chunks - 1) * kp < lf.n <= chunks * kp          # the kernel's delta_cols
        tiles = sorted((int(t["a"]), int(t["b"])) for t in arrays["delta"] if int(t["idx"]) == li)
        step = 16 if chunks else 64
        assert tiles == sorted((a, b) for a in range(0, kp, step) for b in range(0, kp, 64))
    assert len(cover) == want


def test_cut_follows_the_number_of_tasks():
    """Few blocks are cut to at least 128 rows a part; a step that fills the
    chip is not cut."""
    small = _items([(2048, 2048)], 64, 2048, False)
    big = _items([(2048, 2048)] * 128, 64, 2048, False)
    plan = E._split_plan([lf for it in small for lf, _, _ in it.leaves])
    assert plan.rows == E.SPLIT_MIN_ROWS and plan.chunks
    assert E._split_plan([lf for it in big for lf, _, _ in it.leaves]).rows == 0


@pytest.mark.parametrize("shapes", [[(768, 2304), (768, 768)], [(2048, 2048)] * 4])
def test_structure_costs_no_python_call_per_task(shapes):
    """A step structure is array arithmetic: the Python calls of building it
    grow with its blocks (some fifty each, and the helpers of a type), not with
    its thousands of task rows; the block table takes the splits the structure
    was built with instead of working them out again."""
    items = _items(shapes, 64, 2048, False)
    arrays, _, _, leaves = E._build_structure(items)
    rows = sum(len(a) for a in arrays.values())
    calls = 0

    def count(frame, event, arg):
        nonlocal calls
        calls += event == "call"

    sys.setprofile(count)
    try:
        E._build_structure(items)
    finally:
        sys.setprofile(None)
    assert calls < 600 + 60 * len(leaves) < rows, (calls, rows)
    splits = E._leaf_splits(leaves)
    ws = E.Workspace(torch.device("cpu"))
    want = E._leaf_table(leaves, items, ws)
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(E, "_split_plan", None)
        mp.setattr(E, "_leaf_split", None)
        assert E._leaf_table(leaves, items, ws, splits).tobytes() == want.tobytes()


@pytest.mark.parametrize("first", [True, False])
def test_slots_of_mixed_parameters(first):
    """Parameters with and without LARS, ragged ones among them, in either
    order: each reduction slot is written once (a strip run writes several)."""
    shapes = [(100, 300), (512, 768), (33, 257), (640, 512)]
    for k in (64, 128, 256):
        items = _items(shapes, k, 512, False)
        for i, it in enumerate(items):
            it.lars = (i % 2 == 0) == first
        arrays, ranges, nslots, leaves = E._build_structure(items)
        writes = [0] * nslots
        for kind, arr in arrays.items():
            var = int(kind[5:]) if kind.startswith("apply") else 0
            for t in arr:
                s = int(t["slot"])
                if s < 0:
                    continue
                n = 1
                if var & 16:
                    tr = 64 if var & 32 else 128
                    m = leaves[int(t["idx"])][0].m
                    n = min(L.APPLY_GROUP, (m - m % tr - int(t["a"])) // tr)
                for q in range(s, s + n):
                    writes[q] += 1
        assert writes == [1] * nslots
        assert ranges[-1][3] == nslots


def test_a_task_type_without_a_launch_is_an_error(monkeypatch):
    """Tasks filed under a variant that the step does not launch would leave
    their part of a parameter as it was, silently."""
    items = _items([(300, 300)], 64, 512, False)
    E._build_structure(items)
    plain = E._apply_tasks

    def misfiled(*args):
        tasks, slots = plain(*args)
        return [("apply9" if kind == "apply2" else kind, t) for kind, t in tasks], slots

    monkeypatch.setattr(E, "_apply_tasks", misfiled)
    with pytest.raises(RuntimeError, match="apply9"):
        E._build_structure(items)
