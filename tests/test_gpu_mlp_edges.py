"""The gradient kernels at the edges of their 64-row blocks, 64-column tiles and
splits of the rows, and with a work buffer of the least size and off 16-byte
alignment, against the FP64 oracle in its BF16 rounding mode: every block to
1e-3 in relative norm, as the other gradient tests (FP32 sums of BF16 products;
one operand that rounds the other way, 2^-8 of one of a row's 64 activations,
is 5e-4), plus 1e-6 absolute for gradients that vanish (a head of one bin).
"""
import ctypes as C

import numpy as np
import pytest

from dnsmc_amd import learned
from dnsmc_amd._lib import check, lib
from dnsmc_amd.devarray import DeviceArray
from test_gpu_mlp import _oracle_params, _random_net, t

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbin", [1, 64, 65, 1600])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 1000])
@pytest.mark.parametrize("shift", [0, 1])
def test_gradients_at_block_edges(oracle, nbin, n, shift):
    net = _random_net(nbin, 7)
    rng = np.random.default_rng(n)
    X = rng.normal(0, 1, (n, 6)).astype(np.float32)
    td = rng.integers(0, 64, n).astype(np.int32)
    tb = rng.integers(0, nbin, n).astype(np.int32)
    wt = rng.uniform(0.1, 2.0, n).astype(np.float32)
    P = net.L["P"]
    nwork = ((n + 63) // 64) * (P + 1) + P + 2          # the least the call takes
    work = DeviceArray(nwork + shift, np.float32)
    loss = C.c_float(0.0)
    d = [t(a) for a in (X, td, tb, wt)]
    check(lib().dnsmc_mlp_grad(nbin, net.theta.c, net.W1b.c, net.W2b.c, net.W3b.c, *[a.c for a in d], n,
                               C.c_void_p(work.ptr + 4 * shift), nwork, net.grad.c, C.byref(loss)))
    g = net.grad.numpy()
    p = _oracle_params(net)
    ref_loss, ref = oracle.mlp_loss_grad(X.astype(np.float64), *p, 64, td, tb, wt.astype(np.float64), bf16=True)
    assert abs(loss.value - ref_loss) <= 1e-4 * abs(ref_loss)
    L, no = net.L, net.L["noutp"]
    nout = 64 + nbin
    got = [g[L["W1"]:L["b1"]].reshape(6, 64), g[L["b1"]:L["W2"]], g[L["W2"]:L["b2"]].reshape(64, 64), g[L["b2"]:L["W3"]],
           g[L["W3"]:L["b3"]].reshape(64, no), g[L["b3"]:P]]
    for k, (a, b) in enumerate(zip(got, ref)):
        if k >= 4:
            assert not np.any(a[..., nout:])             # padding columns
            a = a[..., :nout]
        assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b) + 1e-6, (k, np.linalg.norm(a - b), np.linalg.norm(b))
