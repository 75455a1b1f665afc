"""The fused training kernels (kernels/mlp.hip: mlp_forward, mlp_backward, mlp_weights) at the edges of their ranges:
networks of an odd and an even number of layers (the last launch of the backward pass takes one or two), of one wave's and
of several rounds of columns, batches around one block of 64 states and around one and several ranges of the weight sums;
and 640 features, which run layer by layer. Against the oracle, which rounds to BF16 where the kernels do. FP32 sums of at
most 640 terms are 1e-5 off at the worst; an activation that such a difference carries over a rounding boundary of BF16
moves by 2^-8 of itself, and reaches an output or gradient as one of at least 55 terms: the bars are those of the existing
test, 1e-3 of the largest value for 99 of 100 values and 2e-2 for all."""
import numpy as np
import pytest

from oracle import mlp as omlp


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,width,depth,n_out,n", [
    (55, 256, 3, 55, 1), (55, 256, 3, 55, 63), (55, 256, 3, 55, 65), (55, 256, 3, 55, 3001), (55, 256, 3, 55, 4097),
    (10, 64, 1, 7, 300), (10, 64, 1, 7, 5000), (70, 128, 2, 130, 1500), (55, 320, 4, 55, 200), (130, 576, 2, 64, 130),
    (55, 640, 2, 55, 130)])
def test_training_step_matches_oracle(n_in, width, depth, n_out, n, gpu):
    import torch
    from combustion_amd.native import Network
    net = Network(n_in, width, depth, n_out)
    rng = np.random.default_rng(n + width)
    params = np.zeros(net.n_params, np.float32)
    for l, (w, b, o, i) in enumerate(net.layers):
        W = np.zeros((o, i), np.float32)
        rows, cols = (n_out if l == depth else o), (n_in if l == 0 else i)
        W[:rows, :cols] = rng.normal(0, 1.0 / np.sqrt(cols), (rows, cols))
        params[w:w + o * i] = W.ravel()
        params[b:b + rows] = rng.normal(0, 0.1, rows)
    x, t = np.zeros((n, net.in_pad), np.float32), np.zeros((n, net.out_pad), np.float32)
    x[:, :n_in] = rng.normal(size=(n, n_in))
    t[:, :n_out] = rng.normal(size=(n, n_out))
    p, xd, td = (torch.from_numpy(a).to(gpu) for a in (params, x, t))
    p16 = p.to(torch.bfloat16)
    y = torch.full((n, net.out_pad), float("nan"), device=gpu)
    grad = torch.full((net.n_params,), float("nan"), device=gpu)
    ws = torch.empty(net.workspace_bytes(n) + 256, dtype=torch.uint8, device=gpu).fill_(0xAB)
    net.forward(p, p16, xd, y, ws[:-256])
    net.backward_mse(p16, y, td, ws[:-256], grad)
    first = grad.clone()
    net.backward_mse(p16, y, td, ws[:-256], grad)  # the forward pass's values are still there
    assert torch.equal(first, grad)
    assert (ws[-256:] == 0xAB).all()
    ref_grad, ref_y = omlp.backward_mse(params, net.layers, x, t, n_out)

    def check(name, got, ref):
        e = np.abs(got - ref) / np.abs(ref).max()
        print(n_in, width, depth, n_out, n, name, np.percentile(e, 99), e.max(), flush=True)
        assert np.percentile(e, 99) < 1e-3 and e.max() < 2e-2

    y, grad = y.cpu().numpy(), grad.cpu().numpy()
    check("output", y[:, :n_out], ref_y[:, :n_out])
    assert np.all(y[:, n_out:] == 0)
    for l, (w, b, o, i) in enumerate(net.layers):
        check(f"layer {l} dW", grad[w:w + o * i], ref_grad[w:w + o * i])
        check(f"layer {l} db", grad[b:b + o], ref_grad[b:b + o])
