"""Early termination decides from the FP32 field's last bits, so single-pass
views with it evaluate the same field as the coarse pass of hierarchical ones."""
import numpy as np
import pytest
import torch

from _cases import shell, shell_rays
from nsvf_amd.render import DeviceScene, Renderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [512, 4096])
def test_one_field_for_both(device, chunk):
    rs, rd = (torch.from_numpy(x).to(device) for x in shell_rays(width=48, seed=9))
    dsc = DeviceScene(shell(), device)
    kept = []
    for hierarchical in (False, True):
        r = Renderer(device, precision="fp32", hierarchical=hierarchical, compat=False,
                     tolerance=1e-2, chunk_size=chunk)
        r.render(dsc, rs, rd, keep=True)
        torch.cuda.synchronize()
        kept.append({k: r.kept[k].cpu().numpy() for k in ("c_field", "c_eval", "c_active")})
    assert kept[0]["c_eval"].any()
    for k in kept[0]:
        np.testing.assert_array_equal(kept[0][k], kept[1][k], err_msg=k)
