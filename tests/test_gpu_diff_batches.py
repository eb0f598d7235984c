"""Gradients of large differentiable batches, whose hashed levels go through
per-slice records, equal the sum over small batches, which add every level
with atomics: table sizes of one slice, several, and more than the records
take; batches of several chunks; rays crowded into few table entries, more
than a slice's share of records."""
import numpy as np
import pytest
import torch

from frustumvolumecaching_amd import lib
from frustumvolumecaching_amd import synthetic as S

pytestmark = pytest.mark.gpu

# FP32 sums in another order: unit roundoff 6e-8 times the square root of the
# at most 1e5 rounded additions behind one value
TOL = 2e-5


def gradients(r, rm, pix, params, d_rgb):
    rgb = torch.empty(len(pix), 3, device="cuda")
    st = r.diff_forward(rm, pix, params, rgb)
    grads = tuple(torch.zeros_like(p) for p in params)
    r.diff_backward(d_rgb, grads)
    torch.cuda.synchronize()
    return grads, st.n_samples


@pytest.mark.parametrize("log2_t, rays, small, crowd", [
    (10, 2000, 250, False), (13, 2000, 250, False), (14, 90000, 700, False), (19, 2200, 300, False),
    (22, 2000, 250, False), (19, 400, 50, True)])
def test_large_batch_is_the_sum_of_small_ones(log2_t, rays, small, crowd):
    wl = S.small_plain(800, 800, log2_hashmap_size=log2_t)
    model = lib.NerfNetwork.from_workload(wl)
    r = lib.Renderer(model)
    rm = wl.rm()
    g = torch.Generator().manual_seed(5)
    pix = torch.randperm(800 * 800, generator=g)[:rays].to(torch.int32)
    if crowd:
        pix[:] = 400 * 800 + 400
    pix = pix.cuda()
    d_rgb = torch.randn(rays, 3, generator=g).cuda()
    params = tuple(torch.from_numpy(np.asarray(p, np.uint16).view(np.float16).astype(np.float32)).cuda()
                   for p in wl.params)
    got, n = gradients(r, rm, pix, params, d_rgb)
    print(f"[diff batch] T 2^{log2_t}: {rays} rays, {n} samples", flush=True)
    assert n > 1 << 16
    want = [torch.zeros_like(p, dtype=torch.float64) for p in params]
    total = 0
    for a in range(0, rays, small):
        part, k = gradients(r, rm, pix[a:a + small].contiguous(), params, d_rgb[a:a + small].contiguous())
        assert k < 1 << 16
        total += k
        for w, q in zip(want, part):
            w += q.double()
    assert total == n
    for b, (x, w) in enumerate(zip(got, want)):
        rel = float(torch.linalg.norm(x.double() - w) / torch.linalg.norm(w))
        print(f"[diff batch] block {b}: {rel:.2e}", flush=True)
        assert rel < TOL, (b, rel)
    r.close()
    model.close()
