"""The network's kernels on tensors that start in the middle of a buffer, aligned to their elements only: the fused kernels
read and write them 16 bytes at a time, and give what they give on tensors of their own, to the bit."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [1, 3])
def test_training_step_on_views(offset, gpu):
    import torch
    from combustion_amd.native import Network
    net, n = Network(55, 256, 3, 55), 200
    rng = np.random.default_rng(4)

    def tensors(offset):
        def place(a, dtype):
            flat = torch.from_numpy(a).to(gpu).to(dtype).flatten()
            buf = torch.zeros(len(flat) + 8, dtype=dtype, device=gpu)
            buf[offset:offset + len(flat)] = flat
            return buf[offset:offset + len(flat)].view(a.shape)
        return place

    x, t = np.zeros((n, net.in_pad), np.float32), np.zeros((n, net.out_pad), np.float32)
    x[:, :55], t[:, :55] = rng.normal(size=(2, n, 55))
    params = np.zeros(net.n_params, np.float32)
    for w, b, o, i in net.layers:
        params[w:w + o * i] = rng.normal(0, 1 / np.sqrt(i), o * i)
    results = []
    for place in (tensors(0), tensors(offset)):
        p, xd, td = (place(a, torch.float32) for a in (params, x, t))
        p16 = place(params, torch.bfloat16)
        y, grad = place(np.zeros((n, net.out_pad), np.float32), torch.float32), place(np.zeros(net.n_params, np.float32), torch.float32)
        ws = torch.empty(net.workspace_bytes(n), dtype=torch.uint8, device=gpu)
        net.forward(p, p16, xd, y, ws)
        net.backward_mse(p16, y, td, ws, grad)
        results.append((y.clone(), grad.clone()))
    print(offset, float(results[0][1].abs().max()), flush=True)
    for a, b in zip(*results):
        assert float(a.abs().max()) > 0 and torch.equal(a, b)
