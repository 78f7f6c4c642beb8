"""Registers of the built kernels, read from the library's code-object metadata: a kernel that grows past
a step of the register file silently halves the wavefronts that hide its latency."""
import struct

import pytest

import mosscap_amd as M

msgpack = pytest.importorskip("msgpack")

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, p)


def _kernels(elf):
    (shoff,) = struct.unpack_from("<Q", elf, 40)
    entsize, num = struct.unpack_from("<HH", elf, 58)
    for k in range(num):
        sh = struct.unpack_from("<IIQQQQ", elf, shoff + k * entsize)
        if sh[1] != 7:  # SHT_NOTE
            continue
        p, end = sh[4], sh[4] + sh[5]
        while p < end:
            namesz, descsz, kind = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if kind == 32:  # NT_AMDGPU_METADATA
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    blob = M.LIB_PATH.read_bytes()
    return {k[".name"]: k for elf in _code_objects(blob) for k in _kernels(elf)}


def _instances(kernels, name, recon, solver, *rest, form="7FormF64"):
    """Instances of `name`, scheme enums as in the bindings, `rest` the further template arguments."""
    tail = "".join(f"Lb{int(r)}E" if isinstance(r, bool) else f"Li{r}E" for r in rest)
    found = [k for n, k in kernels.items()
             if f"{name}INS_{form}" in n and f"ReconstructionE{M.RECONSTRUCTION[recon]}E" in n
             and f"RiemannSolverE{M.RIEMANN_SOLVER[solver]}E{tail}" in n]
    assert found, (name, recon, solver, rest)
    return found


def _waves(kernel):
    return 512 // ((kernel[".vgpr_count"] + 7) // 8 * 8)


@pytest.mark.parametrize("copies", [True, False])
@pytest.mark.parametrize("recon", ["fog", "muscl", "ppm", "weno5z"])
@pytest.mark.parametrize("solver", ["rusanov", "hll", "hllc"])
def test_fp64_general_instance_two_waves_per_simd(kernels, recon, solver, copies):
    """Gravity, tracers and large grids: an instance that lets two wavefronts share a SIMD."""
    every = _instances(kernels, "stage2d_kernel", recon, solver, 2, copies)
    limiters = {"fog": 1, "muscl": 3, "ppm": 3, "weno5z": 1}[recon]
    assert sum(_waves(k) >= 2 for k in every) == limiters


@pytest.mark.parametrize("copies", [True, False])
def test_fp64_general_3d_march_spills(kernels, copies):
    """Held to two wavefronts per SIMD, WENO5-Z + HLLC spills; no more than before ghosts were mirrored."""
    (k,) = _instances(kernels, "stage3d_kernel", "weno5z", "hllc", True, copies)
    assert _waves(k) >= 2 and k[".vgpr_spill_count"] <= 60


# the wavefronts per SIMD that the division into spans counts on (four) or that the scheme had
@pytest.mark.parametrize("copies", [True, False])
@pytest.mark.parametrize("name,recon,solver,waves", [("stage2d_kernel", "muscl", "rusanov", 4),
                                                     ("stage3d_kernel", "fog", "rusanov", 4),
                                                     ("stage3d_kernel", "fog", "hllc", 4),
                                                     ("stage3d_kernel", "ppm", "rusanov", 3),
                                                     ("stage3d_kernel", "ppm", "hll", 3)])
def test_fp32c_general_instances(kernels, name, recon, solver, waves, copies):
    every = _instances(kernels, name, recon, solver, 2 if name.startswith("stage2d") else True, copies,
                       form="8FormF32c")
    assert all(_waves(k) >= waves and k[".vgpr_spill_count"] == 0 for k in every)


@pytest.mark.parametrize("copies", [True, False])
def test_fp64_plain_ppm_rusanov_three_waves_per_simd(kernels, copies):
    every = _instances(kernels, "stage2d_kernel", "ppm", "rusanov", 0, copies)
    assert len(every) == 3 and all(_waves(k) >= 3 for k in every)
