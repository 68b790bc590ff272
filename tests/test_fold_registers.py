"""The fold kernels hold their tables in registers, none in scratch memory: a loop over
the candidate tiles that the compiler does not unroll puts the table of their slots there.
Read from the kernels' metadata in the built library.
"""
import struct

import msgpack

import cunfft_amd


def kernels():
    """{mangled name: metadata} of every gfx950 kernel in the library."""
    blob = open(cunfft_amd.LIB_PATH, "rb").read()
    out, at = {}, 0
    while (at := blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", blob, entry)
            target = blob[entry + 24:entry + 24 + n]
            entry += 24 + n
            if b"gfx950" not in target or size == 0:
                continue
            obj = blob[at + off:at + off + size]
            name = obj.find(b"AMDGPU\0\0")   # the note's name; its header is 12 bytes before
            descsz = struct.unpack_from("<I", obj, name - 8)[0]
            meta = msgpack.unpackb(obj[name + 8:name + 8 + descsz], strict_map_key=False)
            out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
        at += 24
    return out


def test_no_fold_uses_scratch_memory():
    cunfft_amd.lib()
    folds = {k: v for k, v in kernels().items() if "k_tile_fold" in k}
    assert len(folds) > 100
    assert {k for k, v in folds.items() if v[".private_segment_fixed_size"] > 0} == set()
