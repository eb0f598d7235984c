"""The hash-grid encoder over every layout of a lane group's four levels: read
from vertex copies, hashed, or a mix, in the order of the common models and in
others (the encoding bit for bit, the networks by the network parity's bar)."""
import numpy as np
import pytest
import torch

from frustumvolumecaching_amd import lib
from frustumvolumecaching_amd import synthetic as S

from .gpu_util import dev, empty, host_f16
from .test_gpu_parity import _positions, assert_fp16_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2_size, base, finest", [
    (19, 16, 2048),   # two quads copied, two hashed
    (10, 16, 2048),   # the same without a dense level
    (19, 4, 12),      # all dense
    (14, 16, 300),    # three quads copied, one hashed
    (14, 200, 2048),  # all hashed
    (20, 100, 1540),  # a dense level among hashed ones too fine to copy
])
def test_layouts(oracle_mod, log2_size, base, finest):
    wl = S.small_plain(8, 8, stepsize_setup=lib.stepsize_setup)
    wl.net = S.net_desc(log2_hashmap_size=log2_size, base_resolution=base, max_resolution=finest)
    wl.params = S.make_params(wl.net)
    model, ref = lib.NerfNetwork.from_workload(wl), oracle_mod.Model.from_workload(wl)
    p = _positions(2049, log2_size + base)
    # grid vertices and their neighbours in single precision, on both sides
    at = ((np.arange(512) % base + 0.5) / (base - 1)).astype(np.float32)
    p[64:576, 0] = np.nextafter(at, np.float32(0))
    p[64:576, 1] = at
    p[320:832, 2] = np.nextafter(at, np.float32(1))
    d01 = np.full((len(p), 3), 0.25, np.float32)
    enc, lat, out = (empty((len(p), k), torch.int16) for k in (32, 16, 4))
    model.encode(dev(p), len(p), enc)
    model.inferenceLatents(dev(p), len(p), lat)
    model.inference(dev(p), dev(d01), len(p), out)
    torch.cuda.synchronize()
    assert np.array_equal(host_f16(enc), ref.encode(p, oracle_mod.EMU16))
    assert_fp16_close(host_f16(lat)[:, :9], ref.latents(p, oracle_mod.EMU16)[:, :9])
    assert_fp16_close(host_f16(out), ref.inference(p, d01, oracle_mod.EMU16))
    model.close()


# launches below, at and above the lines between the orders in which the blocks
# take their samples, and past the largest grid
@pytest.mark.parametrize("n", [1, 32767, 65537, 262143, 262145, 524289, (1 << 21) + 1, (1 << 22) + 65])
def test_every_sample_is_taken(n):
    model = lib.NerfNetwork.from_workload(S.small_plain(8, 8, stepsize_setup=lib.stepsize_setup))
    period = 4099
    p = dev(_positions(period, 7))
    d = torch.full((period, 3), 0.25, device="cuda")
    at = torch.arange(n, device="cuda") % period
    got = []
    for pos, dirs in ((p, d), (p[at].contiguous(), d[at].contiguous())):
        lat, out = empty((len(pos), 16), torch.int16).fill_(-1), empty((len(pos), 4), torch.int16).fill_(-1)
        model.inferenceLatents(pos, len(pos), lat)
        model.inference(pos, dirs, len(pos), out)
        got.append((lat, out))
    torch.cuda.synchronize()
    for one, all_ in zip(*got):
        assert torch.equal(all_, one[at])
    model.close()
