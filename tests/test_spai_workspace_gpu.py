"""The learned preconditioner's kept workspace: matrices of different sizes in
turn give what a network of their own gives, and calls of several threads on one
network do not share it."""
import threading

import numpy as np
import pytest
import torch

from tnl_amd import spai

pytestmark = pytest.mark.gpu


def _net():
    p = spai.init_parameters(3)
    p[-65:] = 0.02 * np.random.default_rng(4).standard_normal(65)
    return spai.Network(p)


def _probes(A):
    g = torch.Generator(device="cuda").manual_seed(A.rows)
    return torch.randint(0, 2, (2, A.rows), generator=g, device="cuda").double() * 2 - 1


def test_sizes_in_turn():
    mats = [spai.convdiff_matrix(m, 5)[0] for m in (9, 40, 3, 24, 40)]
    net = _net()
    for A in mats:
        loss, M = net.loss_grad(A, _probes(A))
        fresh = _net()
        loss1, M1 = fresh.loss_grad(A, _probes(A))
        assert loss == loss1
        assert torch.equal(M, M1)
        np.testing.assert_array_equal(net.gradients(), fresh.gradients())
        assert torch.equal(net.inverse(A).values, fresh.inverse(A).values)


def test_threads_on_one_network():
    mats = [spai.convdiff_matrix(m, 6)[0] for m in (20, 33, 48)]
    net = _net()
    want = [net.inverse(A).values.clone() for A in mats]
    wrong = []

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(10):
                got = net.inverse(mats[k]).values
                torch.cuda.current_stream().synchronize()
                if not torch.equal(got, want[k]):
                    wrong.append(k)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
