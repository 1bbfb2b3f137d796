"""Kernels that wait for their memory requests by count hold no spilled vector registers.  A spilled register is reloaded by
a memory operation, and since such operations complete in order, the wait for it is a wait for every request made before it:
the weights and activations requested ahead would be waited for where the reload stands and no longer be ahead.  The
compiler spills silently; what it did stands in the metadata of the code objects in the built library."""
import struct
import subprocess

import pytest

from llmxabe_amd import _ffi

msgpack = pytest.importorskip("msgpack")

EM_AMDGPU, NT_AMDGPU_METADATA, SHT_NOTE = 224, 32, 7


def _code_objects(blob):
    at = blob.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == EM_AMDGPU:
            yield at
        at = blob.find(b"\x7fELF", at + 1)


def _kernels(blob, at):
    sections, = struct.unpack_from("<Q", blob, at + 40)
    size, count = struct.unpack_from("<HH", blob, at + 58)
    for i in range(count):
        head = at + sections + i * size
        if struct.unpack_from("<I", blob, head + 4)[0] != SHT_NOTE:
            continue
        start, length = struct.unpack_from("<QQ", blob, head + 24)
        note, end = at + start, at + start + length
        while note < end:
            name_len, desc_len, kind = struct.unpack_from("<III", blob, note)
            desc = note + 12 + (name_len + 3) // 4 * 4
            if kind == NT_AMDGPU_METADATA:
                yield from msgpack.unpackb(blob[desc:desc + desc_len])["amdhsa.kernels"]
            note = desc + (desc_len + 3) // 4 * 4


@pytest.fixture(scope="module")
def spilled():
    """Kernel -> spilled vector registers, of every kernel in the library."""
    _ffi.lib()
    blob = open(_ffi.LIB_PATH, "rb").read()
    found = {k[".name"]: k[".vgpr_spill_count"] for at in _code_objects(blob) for k in _kernels(blob, at)}
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.split("\n")
    return {name.split("(")[0].split("xabe::")[-1]: n for name, n in zip(names, found.values())}


@pytest.mark.parametrize("kernel,forms", [("k_mfma_rows", 16), ("k_decode_up", 24), ("k_decode_up_shared", 4), ("k_decode_down", 12),
                                          ("k_mfma_parts", 4), ("k_mfma_with_shared", 8), ("k_digit_columns", 4), ("k_digit_down", 5), ("k_digit_up", 4),
                                          ("k_head_tiles_bf16", 1), ("k_head_tiles_q8", 4), ("k_head_tiles_q6", 2)])
def test_no_vector_register_is_spilled(spilled, kernel, forms):
    got = {name: n for name, n in spilled.items() if name.split("<")[0] == kernel}
    assert len(got) == forms, sorted(spilled)
    assert not any(got.values()), {name: n for name, n in got.items() if n}
