"""Small-triangle keys that stay in the workspace from call to call: the binnings of a
workspace take epochs 1 to 254, then the buffer is filled again.  Two scenes of many
small triangles in turn, past that, with a call of another form and one of another
size in between; against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from jaxrenderer_amd import _plan
from jaxrenderer_amd.shaders import DepthShader, GouraudShader
from oracle.oracle import run_oracle_plan
from tests import scenes
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


def small_triangles(seed, size, shader=GouraudShader):
    """A soup shrunk triangle by triangle to a few pixels, over tile edges."""
    call = scenes.soup_call(shader, seed, *size, 120)[-1]
    pos = np.array(call.inputs["positions"], np.float32)
    for f in np.asarray(call.inputs["faces"]):
        c = pos[f].mean(0)
        pos[f] = (c + 0.015 * (pos[f] - c)).astype(np.float32)
    call.inputs["positions"] = pos
    return call


# either side of the 2^20 pixels from which the wide form's keys are tagged
@pytest.mark.parametrize("size", [(1024, 1024), (1021, 1024)], ids=str)
def test_keys_over_many_calls(size):
    ref = [run_oracle_plan([small_triangles(k, size)])["main"] for k in (0, 1)]
    assert int((ref[0]["prim_id"] >= 0).sum()) > 200
    calls = [small_triangles(k, size) for k in (0, 1)]
    other = [small_triangles(2, (96, 80)), small_triangles(3, size, DepthShader)]
    for n in range(520):
        got = _plan.run(calls[n % 2], prim_id=True, bary=True)
        if n in (0, 1, 2, 252, 253, 254, 255, 256, 299, 300, 301, 302, 510, 519):
            torch.cuda.synchronize()
            assert_parity(got, ref[n % 2], label=f"keys/{size}/{n}")
        if n == 299:
            _plan.run(other[0])
        if n == 300:
            _plan.run(other[1])
