"""What the compiler gave the built kernels, read from their code objects' metadata."""
import os
import struct

import pytest

from flexible_llm_sharding_amd import _native

msgpack = pytest.importorskip("msgpack")
NOTE, BUNDLE = 7, b"__CLANG_OFFLOAD_BUNDLE__"


def kernels(path):
    """{mangled name: its metadata} of all device code in a library."""
    with open(path, "rb") as f:
        data = f.read()
    out, at = {}, data.find(BUNDLE)
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" not in target or not size:
                continue
            elf = data[at + offset:at + offset + size]
            sections, (entry, count) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
            for i in range(count):
                _, kind, _, _, o, _ = struct.unpack_from("<IIQQQQ", elf, sections + i * entry)
                if kind == NOTE:
                    name, desc, _ = struct.unpack_from("<III", elf, o)
                    start = o + 12 + (name + 3) // 4 * 4
                    for k in msgpack.unpackb(elf[start:start + desc])["amdhsa.kernels"]:
                        out[k[".name"]] = k
        at = data.find(BUNDLE, at + len(BUNDLE))
    return out


def test_products_keep_their_accumulators_in_registers():
    """No kernel of the stateful models' products has scratch memory: a loop over accumulators that is not unrolled puts them there, and halves the speed
    (1,011 rows x 6416 x 1760 104 us, 217 with them in scratch)."""
    if not os.path.exists(_native._SEQ):
        pytest.skip("the library is not built")
    products = {n: k for n, k in kernels(_native._SEQ).items() if "gemm_" in n}
    assert len(products) > 50
    assert not {n: k[".private_segment_fixed_size"] for n, k in products.items() if k[".private_segment_fixed_size"]}
