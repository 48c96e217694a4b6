"""Kept small-triangle keys are asked for by JR_PART_KEEP_KEYS in jr_frame.part and by
nothing else: bytes behind jr_frame's last field, which a caller that fills the struct
field by field leaves as they were, mean nothing."""
import ctypes
import re

import numpy as np
import pytest
import torch

from jaxrenderer_amd import _hip, _plan, _raster
from oracle.oracle import run_oracle_plan
from tests.parity import assert_parity
from tests.test_abi import HEADER
from tests.test_gpu_keys import small_triangles

F = _hip.JrFrame
BEHIND = F.part.offset + F.part.size


def test_frame_ends_with_part():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    body = re.search(r"typedef struct jr_frame \{(.*?)\}", text, flags=re.S).group(1)
    assert body.split(";")[-2].split()[-1] == "part"
    assert F._fields_[-1][0] == "part"
    # the padding is there all the same, so the size is the one that it always was
    assert ctypes.sizeof(F) == _hip.lib().jr_sizeof(3) == BEHIND + 4


def test_parts_and_flag_that_are_taken():
    keep = _hip.PART_KEEP_KEYS
    fr = _raster.make_frame(width=84, height=84, n_scenes=2, shader=0)
    size = _hip.lib().jr_workspace_size(ctypes.byref(fr), 10)
    assert size > 0
    for part in (0, 1, 2, keep, keep + 1, keep + 2):
        fr.part = part
        assert _hip.lib().jr_workspace_size(ctypes.byref(fr), 10) == size, part
    for part in (3, 4, -1, keep + 3, keep // 2, 2 * keep, 3 * keep):
        fr.part = part
        assert _hip.lib().jr_workspace_size(ctypes.byref(fr), 10) == -1, part


def test_make_frame_sets_the_flag():
    for part in (_hip.PART_ALL, _hip.PART_BIN, _hip.PART_RASTER):
        for keep in (False, True):
            fr = _raster.make_frame(width=8, height=8, n_scenes=1, shader=0, part=part,
                                    keep_keys=keep)
            assert fr.part == part + (_hip.PART_KEEP_KEYS if keep else 0)


@pytest.mark.gpu
def test_padding_asks_for_nothing(monkeypatch):
    """A workspace whose key state looks in order and is not (its epoch set back, as
    recycled memory could have it), a frame with its padding set: the keys are cleared, as
    for any workspace that nobody vouches for."""
    size = (1024, 1024)
    make = _raster.make_frame

    def frame(**kw):
        fr = make(**kw)
        ctypes.memset(ctypes.addressof(fr) + BEHIND, 0x5A, ctypes.sizeof(fr) - BEHIND)
        return fr

    calls = [small_triangles(k, size) for k in (0, 1)]
    ref = run_oracle_plan([calls[1]])["main"]
    assert int((ref["prim_id"] >= 0).sum()) > 200
    dev = torch.device("cuda")
    cap = _raster.default_capacity(calls[0].n_tris, _raster.n_tiles(*size, 1))
    ws = torch.zeros(_raster.workspace_size(width=size[0], height=size[1], n_scenes=1,
                                            n_tris=calls[0].n_tris, capacity=cap),
                     dtype=torch.uint8, device=dev)

    def run(call, keep):
        out = {"zbuffer": torch.empty((1,) + size, device=dev),
               "canvas": torch.empty((1,) + size + (3,), device=dev),
               "prim_id": torch.empty((1,) + size, dtype=torch.int32, device=dev),
               "bary": torch.empty((1,) + size + (3,), device=dev)}
        _raster.forward(shader=call.shader, width=size[0], height=size[1],
                        scenes=_raster.scenes_to_device(call.scenes, dev), n_scenes=1,
                        inputs=_plan.device_inputs(call, dev), n_slots=call.n_slots,
                        n_tris=call.n_tris, init_buffers=call.init_buffers,
                        zbuffer_default=call.zbuffer_default,
                        colour_default=call.colour_default, capacity=cap, workspace=ws,
                        keep_keys=keep, **out)
        torch.cuda.synchronize()
        return out

    for _ in range(20):
        run(calls[0], True)
    state = ws[:64].view(torch.int32)
    assert int(state[5]) == 20  # the epoch
    state[5] = 3
    monkeypatch.setattr(_raster, "make_frame", frame)
    assert_parity(run(calls[1], False), ref, label="padding")
