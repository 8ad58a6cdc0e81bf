"""Arguments of the library's kernels, from the metadata of the code objects inside libtab_amd.so: below the 120 bytes from which a launch
takes 0.6-0.8 us longer, and none of the compiler's hidden ones (gridDim, blockDim and the like: 256 bytes more)."""
import re
import struct

import msgpack

from tab_amd import _capi

NOTE, AMDGPU_METADATA = 7, 32


def kernels(path):
    """The metadata of every gfx950 kernel: offload bundles, their ELF files, the AMDGPU note."""
    data, magic = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__"
    bundle = data.find(magic)
    while bundle >= 0:
        entry = bundle + 32
        for _ in range(struct.unpack_from("<Q", data, bundle + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" not in target:
                continue
            elf = data[bundle + offset:bundle + offset + size]
            sections, (width, count) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
            for i in range(count):
                header = sections + i * width
                if struct.unpack_from("<I", elf, header + 4)[0] != NOTE:
                    continue
                at = struct.unpack_from("<Q", elf, header + 24)[0]
                name, length, kind = struct.unpack_from("<III", elf, at)
                if kind == AMDGPU_METADATA:
                    at += 12 + (name + 3) // 4 * 4
                    yield from msgpack.unpackb(elf[at:at + length])["amdhsa.kernels"]
        bundle = data.find(magic, bundle + 1)


def test_arguments_are_short_and_no_hidden_ones():
    seen = 0
    for k in kernels(_capi.LIB_PATH):
        seen += 1
        hidden = [a[".value_kind"] for a in k[".args"] if a[".value_kind"].startswith("hidden")]
        assert not hidden, (k[".name"], hidden)
        # (the mixed launch takes the arguments of two tilings)
        assert k[".kernarg_segment_size"] <= (208 if re.search(r"\d+conv_mfma_tail", k[".name"]) else 112), (k[".name"], k[".kernarg_segment_size"])
    assert seen > 500
