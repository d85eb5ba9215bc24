"""The fused cache query at the edges of its split (16 queries a wave, eight
waves a block, 768 blocks a pass): equal to encode + infer bit for bit, and
within the bf16 network's 1 % of the oracle's largest output
(test_gpu_nrc.py), for values whose inputs are not finite as well."""
import ctypes as C

import numpy as np
import pytest

from oracle import nrc_ref as R
from test_gpu_nrc import HptNrc, Net, _check, lib, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 129, 768 * 128 + 17])
def test_query_of_any_length(n):
    L = lib()
    L.hpt_nrc_query.argtypes = [C.POINTER(HptNrc), C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p,
                                C.c_void_p, C.c_void_p]
    L.hpt_nrc_query.restype = C.c_int
    net = Net()
    params = R.init_params(31)
    net.set_params(params)
    rng = np.random.default_rng(n)
    rec = rng.uniform(-1, 1, (n + 3, 16)).astype(np.float32)
    queue = rng.permutation(n + 3)[:n].astype(np.uint32)
    if n > 16:  # one record of NaN, one of an infinite normal
        rec[queue[3], 0], rec[queue[n - 1], 8] = np.nan, np.inf
    contrib = rng.uniform(0, 1, (n + 3, 4)).astype(np.float32)
    lo, hi = np.full(3, -1, np.float32), np.full(3, 1, np.float32)
    rec_d, q_d, c_d = (torch.tensor(a, device="cuda") for a in (rec, queue.astype(np.int32), contrib))
    _check(L.hpt_nrc_query(C.byref(net.s), rec_d.data_ptr(), q_d.data_ptr(), n, lo.ctypes.data, hi.ctypes.data,
                           c_d.data_ptr(), None))
    raw = np.ascontiguousarray(rec[queue][:, [0, 1, 2, 4, 5, 6, 8, 9, 10, 12, 13, 14]])
    raw_d = torch.tensor(raw, device="cuda")
    X = torch.zeros(n * R.N_IN, dtype=torch.bfloat16, device="cuda")
    _check(L.hpt_nrc_encode(raw_d.data_ptr(), n, lo.ctypes.data, hi.ctypes.data, X.data_ptr(), None))
    y = net.infer(X.view(n, R.N_IN))
    expect = contrib.copy()
    with np.errstate(invalid="ignore"):
        expect[queue, :3] = contrib[queue, :3] + rec[queue][:, [3, 7, 11]] * np.fmax(y, np.float32(0))
    assert np.array_equal(c_d.cpu().numpy(), expect, equal_nan=True)
    finite = np.isfinite(raw).all(1)
    sub = np.flatnonzero(finite)[:2000]
    ref, _ = R.forward(params, X.view(n, R.N_IN)[torch.tensor(sub, device="cuda")].float().cpu().numpy().astype(np.float64),
                       bf16=True)
    assert np.max(np.abs(y[sub] - ref)) <= 1e-2 * np.max(np.abs(ref))
