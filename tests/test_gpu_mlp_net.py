"""The surrogate network's passes at the edges of their launch shapes: rows that take 16, 32, 64 and 128
rows a workgroup, an odd number of 64-row tiles, unaligned buffers, batches whose row slices end in a
half step, and the update with its packed weights.  A row's output is the same bits whatever the batch;
gradients against the oracle with the bars of tests/test_gpu_mlp.py."""
import numpy as np
import pytest

from oracle import mlp_oracle as M
from tests.test_gpu_mlp import dev_bf16, inputs, mech, network, torch  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [64, 4096, 4160, 8192, 8256, 16384, 16448, 65600])
def test_forward_independent_of_batch(torch, mech, rows):
    from fortrancfd_amd.lib import Surrogate
    s = Surrogate(mech)
    flat = network()
    s.set_params(flat)
    base = inputs(1024, 21)
    X = dev_bf16(torch, base)[torch.arange(rows, device="cuda") % 1024].contiguous()
    Y = torch.full((rows, 64), float("nan"), dtype=torch.float32, device="cuda")
    print(f"forward {rows} rows", flush=True)
    s.forward(X, Y)
    small = torch.empty((1024, 64), dtype=torch.float32, device="cuda")
    for r in range(0, 1024, 64):
        s.forward(X[:64] if rows == 64 else dev_bf16(torch, base[r:r + 64]), small[r:r + 64])
        if rows == 64:
            break
    n = 64 if rows == 64 else 1024
    assert torch.equal(Y, small[torch.arange(rows, device="cuda") % n])
    ref, _ = M.forward(flat, base[:n], bf16_acts=True)
    got = Y[:n].cpu().numpy().astype(np.float64)[:ref.shape[0]]
    assert np.linalg.norm(got - ref[:got.shape[0]]) <= 1e-2 * np.linalg.norm(ref[:got.shape[0]])


@pytest.mark.parametrize("rows", [128, 16448])
def test_forward_unaligned(torch, mech, rows):
    from fortrancfd_amd.lib import Surrogate
    s = Surrogate(mech)
    s.set_params(network())
    X = dev_bf16(torch, inputs(rows, 22))
    Y = torch.empty((rows, 64), dtype=torch.float32, device="cuda")
    s.forward(X, Y)
    xb = torch.empty(rows * 64 + 1, dtype=X.dtype, device="cuda")
    yb = torch.empty(rows * 64 + 1, dtype=torch.float32, device="cuda")
    x1, y1 = xb[1:].view(rows, 64), yb[1:].view(rows, 64)
    x1.copy_(X)
    print(f"forward {rows} rows, buffers off by one element", flush=True)
    s.forward(x1, y1)
    assert torch.equal(y1, Y)


@pytest.mark.parametrize("rows", [64, 192, 4160, 16448])
def test_gradients(torch, mech, rows):
    from fortrancfd_amd.lib import Surrogate
    s = Surrogate(mech)
    flat = network(6)
    s.set_params(flat)
    X = inputs(rows, 23)
    T = np.random.default_rng(24).normal(size=(rows, M.OUTP)).astype(np.float32)
    T[:, M.OUT:] = 0
    print(f"train step lr=0, {rows} rows", flush=True)
    idx = torch.arange(rows, dtype=torch.int32, device="cuda")
    loss = s.train_step(dev_bf16(torch, X), torch.from_numpy(T).cuda(), idx, 0.0, want_loss=True)
    g = s.get_grads().astype(np.float64)
    ref_loss, ref_g = M.loss_and_grads(flat, X, T.astype(np.float64), bf16_acts=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    for a2, b2 in zip(M.unpack(g), M.unpack(ref_g)):
        for a, b in zip(a2, b2):
            assert np.linalg.norm(a - b) <= 3e-2 * np.linalg.norm(b)
            assert (a * b).sum() >= 0.999 * np.linalg.norm(a) * np.linalg.norm(b)


def test_update_and_packed_weights(torch, mech):
    """One Adam step against its formula (eight FP32 operations: 2e-6 of the step, half an ulp of the
    weight), and the packed weights it leaves: a network set to its parameters gives the same bits."""
    from fortrancfd_amd.lib import Surrogate
    s = Surrogate(mech)
    w0 = network(6).astype(np.float32)
    s.set_params(w0)
    X = dev_bf16(torch, inputs(256, 25))
    T = torch.zeros((256, 64), dtype=torch.float32, device="cuda")
    T[:, :54] = torch.randn((256, 54), device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    print("one Adam step", flush=True)
    s.train_step(X, T, torch.arange(256, dtype=torch.int32, device="cuda"), 1e-3)
    w1, g = s.get_params(), s.get_grads().astype(np.float64)
    step = 1e-3 * g / (np.abs(g) + 1e-8)
    assert np.all(np.abs(w1 - (w0 - step)) <= 2e-6 * 1e-3 + 1.2e-7 * np.abs(w0))
    s2 = Surrogate(mech)
    s2.set_params(w1)
    a, b = (torch.empty((256, 64), dtype=torch.float32, device="cuda") for _ in range(2))
    s.forward(X, a)
    s2.forward(X, b)
    assert torch.equal(a, b)
    s.train_step(X, T, torch.arange(256, dtype=torch.int32, device="cuda"), 0.0)
    s2.train_step(X, T, torch.arange(256, dtype=torch.int32, device="cuda"), 0.0)
    np.testing.assert_array_equal(s.get_grads(), s2.get_grads())
