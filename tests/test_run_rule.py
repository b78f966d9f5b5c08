"""Where a sampling run takes the whole-run kernel: the rule against what both routes took on an MI355X (us per layer
and step)."""

import ctypes

import pytest

from ar_nanotabpfn_amd import _lib

BF16, F32 = _lib.ARTAB_BF16, _lib.ARTAB_F32

# dtype, d_model, trajectories, context rows, layers, whole run, step by step
MEASURED = [
    (BF16, 512, 1, 2048, 12, 90.6, 139.5), (BF16, 512, 1, 8192, 12, 254.5, 144.7), (BF16, 512, 16, 2048, 12, 123.8, 141.1),
    (BF16, 512, 16, 4096, 12, 195.4, 141.2), (BF16, 512, 64, 1024, 12, 90.8, 142.4), (BF16, 512, 64, 2048, 12, 127.4, 140.7),
    (BF16, 512, 64, 4096, 12, 206.7, 152.9), (BF16, 512, 200, 1024, 12, 114.8, 150.6), (BF16, 512, 256, 512, 12, 87.7, 139.1),
    (BF16, 256, 1, 8192, 12, 122.7, 141.6), (BF16, 256, 1, 12288, 12, 176.4, 142.5), (BF16, 256, 16, 4096, 12, 91.0, 138.8),
    (BF16, 256, 64, 4096, 12, 99.8, 139.5), (BF16, 256, 128, 2048, 12, 67.9, 139.3), (BF16, 256, 256, 1024, 12, 56.8, 140.3),
    (BF16, 256, 512, 512, 12, 58.4, 139.1), (BF16, 128, 1, 16384, 12, 117.5, 143.0), (BF16, 128, 64, 8192, 12, 95.0, 182.7),
    (BF16, 128, 64, 16384, 12, 180.9, 326.5), (BF16, 128, 256, 4096, 12, 92.4, 134.4), (F32, 256, 1, 2048, 12, 116.7, 279.2),
    (F32, 256, 1, 4096, 12, 199.8, 280.7), (F32, 256, 16, 4096, 12, 232.8, 279.2), (F32, 256, 64, 2048, 12, 138.8, 274.4),
    (F32, 256, 256, 1024, 12, 125.5, 274.9), (F32, 128, 1, 8192, 12, 177.2, 292.5), (F32, 128, 1, 16384, 12, 346.4, 300.3),
    (F32, 128, 64, 8192, 12, 213.1, 291.8), (F32, 128, 256, 2048, 12, 95.8, 287.7), (BF16, 512, 1, 8192, 2, 272.1, 345.6),
    (BF16, 512, 1, 16384, 2, 492.6, 343.2), (BF16, 512, 64, 16384, 2, 733.1, 505.4), (BF16, 256, 1, 16384, 2, 242.1, 338.0),
    (F32, 256, 1, 8192, 2, 380.2, 484.4), (F32, 256, 1, 16384, 2, 716.8, 491.7), (F32, 256, 64, 16384, 2, 828.0, 612.1)]


@pytest.mark.parametrize("dtype,D,B,Nc,layers,run,steps", MEASURED)
def test_own_contexts_take_the_faster_route(dtype, D, B, Nc, layers, run, steps):
    lib = _lib.load()
    group = lib.artab_trajectory_group_layers(B, Nc, 6, D // 32, D, 256, layers, 1, dtype)
    assert (group > 0) == (run < steps)
    if layers == 12:
        assert lib.artab_trajectory_group(B, Nc, 6, D // 32, D, 256, 1, dtype) == group


# shared contexts, 4 layers: as above
SHARED = [
    (F32, 128, 8, 2048, 57.0, 111.0), (F32, 128, 8, 8192, 176.5, 119.8), (F32, 128, 64, 2048, 55.2, 146.7), (F32, 128, 256, 64, 18.3, 135.6),
    (F32, 128, 256, 2048, 54.5, 156.1), (F32, 128, 256, 8192, 166.6, 188.6), (F32, 128, 1024, 2048, 108.7, 160.1),
    (F32, 128, 1024, 8192, 347.6, 261.8), (F32, 256, 8, 512, 56.5, 119.3), (F32, 256, 8, 8192, 361.7, 131.5), (F32, 256, 64, 2048, 112.6, 212.2),
    (F32, 256, 64, 8192, 344.3, 225.6), (F32, 256, 256, 2048, 112.1, 188.7), (F32, 256, 256, 8192, 337.0, 220.9), (F32, 256, 1024, 512, 106.9, 145.1),
    (F32, 256, 1024, 2048, 225.6, 169.3), (F32, 256, 1024, 8192, 698.3, 268.3), (BF16, 128, 64, 2048, 21.3, 31.6), (BF16, 128, 64, 8192, 58.5, 32.6),
    (BF16, 128, 1024, 2048, 26.0, 32.7), (BF16, 256, 8, 512, 21.7, 32.9), (BF16, 256, 64, 2048, 39.3, 33.9), (BF16, 256, 1024, 512, 24.9, 34.1),
    (BF16, 256, 1024, 2048, 47.0, 36.2)]


@pytest.mark.parametrize("dtype,D,B,Nc,run,steps", SHARED)
def test_shared_contexts_take_the_faster_route(dtype, D, B, Nc, run, steps):
    group = _lib.load().artab_trajectory_group_layers(B, Nc, 12, D // 32, D, 256, 4, 0, dtype)
    assert (group > 0) == (run < steps)


# several workgroups to a trajectory: dtype, d_model, trajectories, context rows, own contexts, us per layer and step with
# 1, 2, 4 and 8 of them, step by step (4 layers; None: not built, or not measured)
PARTS = [
    (BF16, 128, 64, 16000, 0, (102.9, 61.4, 33.4, None), 31.9), (BF16, 128, 32, 4000, 0, (30.7, 19.1, 13.2, None), 25.2),
    (BF16, 128, 100, 200, 0, (10.0, 10.4, None, None), 33.1), (BF16, 128, 128, 3000, 0, (28.7, 20.5, None, None), 32.9),
    (BF16, 256, 32, 300, 0, (15.7, 12.1, 9.9, 10.5), 24.3), (BF16, 256, 32, 16000, 0, (203.8, 120.4, 65.6, 37.7), 36.1),
    (BF16, 256, 64, 16000, 0, (200.6, 116.7, 61.7, None), 35.1), (BF16, 256, 8, 4000, 0, (66.4, 39.1, 22.7, 16.8), 28.8),
    (BF16, 256, 64, 600, 1, (21.7, 15.7, 15.7, None), None), (BF16, 256, 64, 2500, 1, (72.6, 42.6, 35.9, None), None),
    (BF16, 512, 8, 300, 0, (44.1, 33.9, 27.9, 23.4), 45.4), (BF16, 512, 32, 16000, 0, (420.4, 267.5, 137.3, 80.3), 68.5),
    (BF16, 512, 64, 2500, 1, (144.6, 106.5, 86.5, None), None), (F32, 128, 64, 32, 0, (15.7, 16.3, 16.2, None), 124.2),
    (F32, 128, 8, 4000, 0, (84.2, 46.4, 29.3, None), 85.7), (F32, 256, 32, 300, 0, (40.6, 30.5, 26.8, 26.9), 136.8),
    (F32, 256, 128, 16000, 0, (588.7, 304.0, None, None), 356.7), (F32, 256, 64, 2500, 1, (154.5, 103.3, 78.1, None), None)]


@pytest.mark.parametrize("dtype,D,B,Nc,own,times,steps", PARTS)
def test_workgroups_per_trajectory(dtype, D, B, Nc, own, times, steps):
    lib = _lib.load()
    parts = lib.artab_trajectory_parts(B, Nc, 24, D // 32, D, 256, 4, own, dtype)
    assert parts * B <= 256 or parts == 1
    taken = times[parts.bit_length() - 1]
    if parts == 1 and not lib.artab_trajectory_group_layers(B, Nc, 24, D // 32, D, 256, 4, own, dtype):
        taken = steps
    assert taken <= 1.1 * min(t for t in (*times, steps) if t is not None)


def test_workgroups_per_trajectory_are_checked():
    lib = _lib.load()
    a = _lib.ArtabTrajectoryArgs()
    for name, kind in a._fields_:  # (pointers that nobody follows: the calls end in front of the launch)
        if kind is ctypes.c_void_p:
            setattr(a, name, 4096)
    a.n_layers, a.n_ctx, a.ctx_rows, a.own_rows, a.K, a.bs, a.B, a.Nt, a.group, a.D, a.F = 2, 8, 8, 8, 3, 4, 4, 4, 1, 128, 256
    call = lambda parts, exchange: lib.artab_trajectory_decode_parts(ctypes.byref(a), parts, exchange, BF16, None)  # noqa: E731
    assert call(3, 4096) == call(8, 4096) == call(0, 4096) == call(-2, 4096) == _lib.ARTAB_ERR_UNSUPPORTED
    assert call(2, None) == _lib.ARTAB_ERR_NULL_POINTER and call(2, 4104) == _lib.ARTAB_ERR_BAD_STRIDE
    a.group = 2
    assert call(2, 4096) == _lib.ARTAB_ERR_UNSUPPORTED
    assert lib.artab_trajectory_exchange_bytes(4, 128, BF16) == 2 * 4 * 128 * 8 and lib.artab_trajectory_exchange_bytes(0, 128, BF16) == 0
