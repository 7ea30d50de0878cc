"""The one-pass step's psi addresses (step3_face, step3_psi_offset) against the
index the two-pass kernels form, on the CPU: the far faces of grids whose
nodes pass 2^32 bytes, and long grids along each axis.  A face that 32-bit
offsets do not reach has to be turned away (step3_face_fits), and only such
a face."""
import os
import subprocess

import pytest

from xfdtd_cuda_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("step3") / "step3_offsets")
    r = subprocess.run([build.HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-o", out,
                        os.path.join(HERE, "cpp", "step3_offsets.cpp")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.parametrize("nx,ny,nz,layers,size", [
    (24, 20, 28, 4, 8),
    (536, 536, 536, 12, 8),
    (820, 820, 820, 10, 8),      # FP64: a component of 4.4e9 bytes
    (1100, 1100, 1100, 8, 4),    # 32-bit psi: 5.3e9
    (1100, 1100, 1100, 8, 8),
    (70000, 100, 100, 6, 8),     # long along each axis
    (100, 70000, 100, 6, 8),
    (100, 100, 70000, 6, 8),
    (8, 11000, 11000, 2, 8),     # flat: x faces of 2 layers, 1.9e9 bytes each
])
def test_addresses_are_the_two_pass_kernels(program, nx, ny, nz, layers, size):
    out = subprocess.run([program, f"{nx},{ny},{nz},{layers},{size}"], capture_output=True, text=True, check=True).stdout
    reached, faces, wrong = map(int, out.split())
    assert (reached, faces, wrong) == (12, 12, 0)


@pytest.mark.parametrize("nx,ny,nz,layers,size,most", [
    # x faces of 2 layers and y faces biased by 24000 rows: 4.6e9 bytes and more; the z faces are small
    (4, 24000, 24000, 2, 8, 8),
    # 32-bit rows: nothing along x or y is reached
    (2, 60000, 60000, 2, 4, 6),
])
def test_faces_out_of_reach_are_turned_away(program, nx, ny, nz, layers, size, most):
    out = subprocess.run([program, f"{nx},{ny},{nz},{layers},{size}"], capture_output=True, text=True, check=True).stdout
    reached, faces, wrong = map(int, out.split())
    assert 0 < reached <= most and faces == 12 and wrong == 0
