"""One training step and one backward pass of the proposal network at the sizes where the training kernels' blocks,
row ranges and half-filled row blocks end: 1 to 67 groups, groups with non-finite labels, against the
oracle (loss, gradient). Bounds as in test_gpu_learned: the gradient's error against the oracle's bf16 restatement within
2 % of its norm, the loss within 2e-3 relative."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def dptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 31, 63, 64, 65, 67])
def test_backward_and_loss_sizes(gpu, n):
    import torch
    from unidock_engine import proposal as LP
    print(f"training kernels: {n} groups", flush=True)
    rng = np.random.default_rng(90 + n)
    p = LP.init_params(3)
    p[:gpu.MLP_NPARAM] += rng.normal(0, 0.02, gpu.MLP_NPARAM).astype(np.float32)
    x = rng.normal(0.2, 0.8, (n * 16, 80)).astype(np.float32)
    bits = O.bf16_bits(x)
    xd = torch.from_numpy(bits.astype(np.int16)).cuda()
    label = rng.normal(-5, 2, n * 16).astype(np.float32)
    label[3] = np.inf
    if n > 2:
        label[16:32] = np.nan  # a group without a label
    y = O.mlp_forward(p, bits)
    loss_ref, dy = O.group_loss(y, label)
    ref = O.mlp_backward(p, bits, dy)
    m = gpu.Mlp(p)
    grad = torch.zeros(gpu.MLP_NPARAM, device="cuda")
    dyd = torch.from_numpy(np.ascontiguousarray(dy, np.float32)).cuda()
    gpu.check(gpu.lib().ud2_mlp_backward(m.h, dptr(xd), None, n, dptr(dyd), dptr(grad), gpu.stream_ptr()))
    loss = torch.zeros(1, device="cuda")
    opt = gpu.Adam(1e-3, 0.9, 0.999, 1e-8)
    ld = torch.from_numpy(label).cuda()
    gpu.check(gpu.lib().ud2_mlp_train_step(m.h, dptr(xd), dptr(ld), None, n, C.byref(opt), dptr(loss), gpu.stream_ptr()))
    torch.cuda.synchronize()
    g = grad.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(g - ref) <= 0.02 * np.linalg.norm(ref)
    assert abs(float(loss.item()) - loss_ref) <= 2e-3 * abs(loss_ref)
    # the first Adam step moves a parameter by lr against its gradient's sign, where that is not tiny
    moved = m.params()[:gpu.MLP_NPARAM].astype(np.float64) - p[:gpu.MLP_NPARAM]
    big = np.abs(g) > 1e-5
    assert np.allclose(moved[big], -1e-3 * np.sign(g[big]), atol=2e-5)
