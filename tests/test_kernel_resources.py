"""Registers of the kernels as built (no GPU needed), from the metadata of libnmx.so's code objects.
attn_pvl_k's two workgroups of a CU (5 or more rows of 8 heads) are resident together only at 128
vector registers; at 140 the second waited for the first and short contexts lost 2 us a layer. No
kernel spills registers to memory."""
from __future__ import annotations

import struct

import msgpack

from nibblemac_amd.nmx import library_path


def kernels() -> dict[str, dict]:
    """Mangled name -> metadata map, from the NT_AMDGPU_METADATA notes."""
    data, out, at = library_path().read_bytes(), {}, 0
    name = b"AMDGPU\0\0"
    while (at := data.find(name, at)) >= 0:
        namesz, descsz, kind = struct.unpack_from("<III", data, at - 12)
        at += len(name)
        if (namesz, kind) == (7, 32):
            for k in msgpack.unpackb(data[at:at + descsz])["amdhsa.kernels"]:
                out[k[".name"]] = k
    return out


def test_long_attention_fits_twice():
    ks = {n: k for n, k in kernels().items() if "attn_pvl_k" in n}
    assert len(ks) == 3, sorted(ks)  # the three cache formats
    for n, k in ks.items():
        assert k[".max_flat_workgroup_size"] == 320 and k[".vgpr_count"] <= 128, (n, k[".vgpr_count"])


def test_no_kernel_spills():
    ks = kernels()
    assert len(ks) > 50
    spilled = {n: k[".vgpr_spill_count"] for n, k in ks.items() if k[".vgpr_spill_count"]}
    assert not spilled, spilled
