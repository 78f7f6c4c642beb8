"""mh_upload_device / mh_download_device of the compensated form: the conversion works on the caller's
device array in place where it can (8-byte aligned, the context's own device, one allocation) and
through a copy elsewhere; both give the bits of the host transfers."""
import numpy as np
import pytest
import torch

import mosscap_amd as M
from mosscap_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 64, 333])
@pytest.mark.parametrize("shift", [0, 8, 4, 2])
def test_device_transfers_equal_host_transfers(n, shift):
    cfg = problems.kh_config(n)
    q0 = problems.kh_band(cfg)
    with M.HydroContext(cfg, precision_form=M.FP32C) as a, M.HydroContext(cfg, precision_form=M.FP32C) as b:
        raw = torch.zeros(q0.nbytes + 64, dtype=torch.uint8, device="cuda:0")
        raw[shift:shift + q0.nbytes] = torch.from_numpy(q0.view(np.uint8).reshape(-1)).cuda()
        out = torch.zeros_like(raw)
        torch.cuda.synchronize()
        a.upload(q0)
        b.upload_device(raw.data_ptr() + shift)
        for c in (a, b):
            c.fill_bcs()
            c.run(2)
        b.download_device(out.data_ptr() + shift)
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[shift:shift + q0.nbytes].view(np.float64).reshape(q0.shape), a.download())
        assert not got[:shift].any() and not got[shift + q0.nbytes:].any()
