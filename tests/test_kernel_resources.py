"""What the compiler made of the matrix-core kernels, read from the code objects in libkx_hip.so (no GPU needed): scratch
memory and registers where they decide how a launch runs."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 code objects of a host library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        entry = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, entry)
            if size and data[entry + 24:entry + 24 + name].endswith(b"gfx950"):
                yield data[at + offset:at + offset + size]
            entry += 24 + name
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Template arguments of each awq_gemv_mfma_kernel (waves, steps, rows per round, rounds, prologue, epilogue, odd words,
    walks, crosses groups, plain of which three fit a compute unit) -> its bytes of scratch memory, its vector registers and its
    bytes of LDS."""
    from mykuiperllama_amd.build import KX_LIB
    if not os.path.exists(READELF):
        pytest.skip("llvm-readelf is not installed")
    found = {}
    path = tmp_path_factory.mktemp("code") / "object"
    with open(KX_LIB, "rb") as f:
        data = f.read()
    for code in code_objects(data):
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n *- \.agpr_count", notes)[1:]:
            field = lambda name: re.search(r"\." + name + r": +(\S+)", block).group(1)
            m = re.search(r"awq_gemv_mfma_kernelI(.*?)EEv", field("name"))
            if m:
                args = tuple(int(v) for v in re.findall(r"L[ib](\d+)E", m.group(1) + "E"))
                found[args] = int(field("private_segment_fixed_size")), int(field("vgpr_count")), int(field("group_segment_fixed_size"))
    assert found, "no matrix-core kernel in the library"
    return found


def test_short_waves_at_sixteen_rows_fit_three_to_a_compute_unit(kernels):
    # three workgroups leave 168 registers; what does not fit goes to memory and back in the workgroup that finishes a column tile
    short = {args: found for args, found in kernels.items() if args[1] <= 2 and args[2] * args[3] == 16 and args[5] == 0}
    assert short and not [args for args, (scratch, registers, _) in short.items() if scratch or registers > 168]


def test_walking_kernels_keep_their_addresses(kernels):
    # A few words of a walking launch at sixteen rows behind SwiGLU still go to memory; with the addresses of the staged rows
    # among them every block waited for its weights before it could produce its activations.
    walking = {args: scratch for args, (scratch, _, _) in kernels.items() if args[7]}
    assert max(walking.values()) <= 40
    assert not [args for args, scratch in walking.items() if scratch and not (args[4] and args[2] * args[3] == 16)]


def test_two_rows_into_the_residual_stream_leave_room_for_six_workgroups(kernels):
    # one step per wave: 512 registers a lane and six waves per SIMD are 80 registers a wave
    few = {args: registers for args, (_, registers, _) in kernels.items() if args[1:4] == (1, 2, 1) and args[5] == 2 and not args[8]}
    assert few and max(few.values()) <= 80


def test_four_steps_behind_a_norm_fit_three_to_a_compute_unit(kernels):
    # Their workgroups wait for each other in grids of up to three per compute unit: 168 registers, a third of 160 KB of LDS.  The
    # compiler keeps to the registers by sending to memory what does not fit: at sixteen rows behind a norm what the read-back of a
    # single reader holds, in the plain form, which has no such reader, two words.
    three = {args: found for args, found in kernels.items()
             if args[1] == 4 and args[2] * args[3] >= 8 and args[5] == 0 and not args[7] and not args[8] and (args[4] == 5 or args[9])}
    assert len(three) >= 4
    for args, (scratch, registers, lds) in three.items():
        assert registers <= 168 and 3 * lds <= 160 * 1024, args
        assert scratch <= (8 if args[9] else (80 if args[2] * args[3] == 16 else 0)), args
