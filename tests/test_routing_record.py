"""The layer call's routing record is the dataclass it was: dataclasses.replace and copies of it work."""

import copy
import dataclasses
import types

import torch

from abacus_amd.moe import Routing, _PlanRouting


def _record():
    T, E, K = 3, 4, 2
    at = dict(logits=0, weights=256, indices=512, counts=768, offsets=1024, pos=1280, perm=1536)
    route = torch.arange(1792, dtype=torch.int64).to(torch.uint8)
    return _PlanRouting(route, types.SimpleNamespace(at=at, sizes=(T, 8, E, K)), torch.float32)


def test_replace_gives_a_record_with_the_other_fields():
    r = _record()
    new = torch.full((3, 2), 0.5)
    s = dataclasses.replace(r, weights_TK=new)
    assert isinstance(s, Routing) and s.weights_TK is new
    for f in dataclasses.fields(Routing):
        if f.name != "weights_TK":
            assert torch.equal(getattr(s, f.name).view(torch.uint8), getattr(r, f.name).view(torch.uint8)), f.name


def test_copies():
    r = _record()
    for c in (copy.copy(r), copy.deepcopy(r)):
        assert isinstance(c, Routing) and torch.equal(c.pos_TK, r.pos_TK) and torch.equal(c.counts_E, r.counts_E)
