"""recon_mc_extract_noalloc (marching cubes with a static device scratch,
for callers that cannot allocate) against recon_mc_extract through the
C-ABI: identical triangle counts, vertex bits and index lists on two calls
in a row, the second on a smaller field (the static scratch keeps the first
call's contents).  The refusal above its size limit is a host check, tested
without a GPU in test_abi.py."""
import ctypes as C

import numpy as np
import pytest

import oracle_ffi as O
import recon
from helpers import assert_bitexact
from recon import ffi, scenes

pytestmark = pytest.mark.gpu


def _field(torch, w):
    vol = recon.TSDFVolume(w.config())
    dev = torch.from_numpy(w.render()).cuda()
    for f in range(w.num_frames):
        vol.integrate(dev[f], w.poses[f])
    torch.cuda.synchronize()
    D, _ = vol.download()
    info = vol.info
    vol.close()
    return torch.from_numpy(D).cuda(), list(info.grid), list(info.voxel_size), list(info.global_offset)


def _extract(torch, fn, field, grid, vs, off, cap):
    verts = torch.full((max(cap, 1), 3, 3), -7.0, dtype=torch.float32, device="cuda")
    tris = torch.full((max(cap, 1), 3), -7, dtype=torch.int32, device="cuda")
    n = C.c_int64()
    st = fn(field.data_ptr(), ffi.i32x3(grid), ffi.f32x3(vs), ffi.f32x3(off), verts.data_ptr(),
            tris.data_ptr(), cap, C.byref(n), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return st, int(n.value), verts[:n.value].cpu().numpy(), tris[:n.value].cpu().numpy()


def test_noalloc_equals_allocating_extract(cuda):
    lib = ffi.load()
    big = scenes.plain_small()                     # 128^3, 10 frames
    small = scenes.tiny(grid=(40, 36, 28), voxel_size=0.025, image=(64, 48), num_frames=3)
    for name, w in (("128^3", big), ("40x36x28", small)):
        field, grid, vs, off = _field(cuda, w)
        n_ref = C.c_int64()
        assert lib.recon_mc_count(field.data_ptr(), ffi.i32x3(grid), ffi.f32x3(vs), ffi.f32x3(off),
                                  C.byref(n_ref), None) == 0
        cap = int(n_ref.value)
        assert cap > 1000, (name, cap)
        print(f"no-alloc marching cubes on {name}: {cap} triangles", flush=True)
        st0, n0, v0, t0 = _extract(cuda, lib.recon_mc_extract, field, grid, vs, off, cap)
        st1, n1, v1, t1 = _extract(cuda, lib.recon_mc_extract_noalloc, field, grid, vs, off, cap)
        assert st0 == 0 and st1 == 0, (st0, st1, lib.recon_last_error())
        assert n0 == n1 == cap
        assert np.array_equal(v0.view(np.uint32), v1.view(np.uint32)), f"{name}: vertices differ"
        assert np.array_equal(t0, t1), f"{name}: indices differ"
        # too small an output: the count is reported with RECON_ERR_CAPACITY
        st2, n2, _, _ = _extract(cuda, lib.recon_mc_extract_noalloc, field, grid, vs, off, cap - 1)
        assert st2 == ffi.ERR_CAPACITY and n2 == cap


def _noise(grid):
    gx, gy, gz = grid
    rng = np.random.default_rng(sum(grid))
    f = rng.standard_normal((gz, gy, gx)).astype(np.float32)
    f[rng.random(f.shape) < 0.1] = 0.0           # exact zeros: not < 0
    f[rng.random(f.shape) < 0.05] = -0.0         # negative zero: not < 0
    f[rng.random(f.shape) < 0.05] = 1e-41        # denormals
    return f


def _few_chunks():
    # 35 chunks a cube row, surface voxels in a few of them, at chunk
    # boundaries and row ends
    gx, gy, gz = 2200, 6, 4
    f = np.full((gz, gy, gx), 0.5, np.float32)
    for k, x in enumerate([0, 5, 7 * 64 + 10, 30 * 64 + 63, 31 * 64, 31 * 64 + 3, 33 * 64 + 40, gx - 1]):
        f[k % gz, (2 * k) % gy, x] = -0.25 - 0.01 * k
    f[2, 5, 32 * 64 + 1] = -1.0
    return f


def _many_tiles():
    # 65536 tiles of 16 cube rows: eight passes of the tile scan
    gx, gy, gz = 8, 1025, 1025
    y = np.arange(gy, dtype=np.float32)[None, :, None]
    z = np.arange(gz, dtype=np.float32)[:, None, None]
    f = (np.sqrt((y - 500.0) ** 2 + (z - 480.0) ** 2) - 300.0 + np.zeros(gx)).astype(np.float32)
    f[-64:] = np.random.default_rng(11).standard_normal((64, gy, gx)).astype(np.float32)
    return f


# The passes by chunk counts, which only this entry takes: rows of 3, 70, 65
# and 129 voxels, and an unaligned field, use the count's 4-byte loads; rows of
# a multiple of 4 its 16-byte loads, 256 cubes a span: one span cut short (4,
# 64, 68), two (260) and three (516)
@pytest.mark.parametrize("case", [(3, 2, 2), (70, 3, 5), (65, 66, 7), (129, 2, 3), (4, 3, 3), (64, 5, 9),
                                  (68, 7, 6), (260, 9, 4), (516, 6, 5), "unaligned", "few chunks",
                                  "many tiles"])
def test_noalloc_equals_oracle(cuda, case):
    f = _noise(case) if isinstance(case, tuple) else \
        {"unaligned": lambda: _noise((68, 7, 6)), "few chunks": _few_chunks, "many tiles": _many_tiles}[case]()
    grid = f.shape[::-1]
    vs, off = (0.01, 0.02, 0.03), (0.1, -0.2, 0.3)
    ov, ot, _, _ = O.mc_extract(f, grid, vs, off)
    shift = 1 if case == "unaligned" else 0
    buf = cuda.zeros(f.size + shift, dtype=cuda.float32, device="cuda")
    buf[shift:] = cuda.from_numpy(f.ravel()).cuda()
    assert buf[shift:].data_ptr() % 16 == 4 * shift
    print(f"no-alloc marching cubes on {case}: {len(ot)} triangles", flush=True)
    st, n, v, t = _extract(cuda, ffi.load().recon_mc_extract_noalloc, buf[shift:], grid, vs, off, len(ot))
    assert st == 0 and n == len(ot) > 0
    assert_bitexact(v, ov, "vertices")
    assert np.array_equal(t, ot)
