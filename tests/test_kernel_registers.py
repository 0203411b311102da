"""CPU check of the built library's kernel metadata: the kernels listed here
keep everything in registers (no scratch memory per lane)."""
import re
import struct

import msgpack

EM_AMDGPU, SHT_NOTE = 224, 7


def kernels(path):
    """Metadata records of every device kernel in the library."""
    data = open(path, "rb").read()
    out = []
    for m in re.finditer(b"\x7fELF\x02\x01\x01\x40", data):
        o = m.start()
        if struct.unpack_from("<H", data, o + 18)[0] != EM_AMDGPU:
            continue
        shoff, = struct.unpack_from("<Q", data, o + 40)
        entsize, count = struct.unpack_from("<HH", data, o + 58)
        for i in range(count):
            sh = o + shoff + i * entsize
            if struct.unpack_from("<I", data, sh + 4)[0] != SHT_NOTE:
                continue
            at = o + struct.unpack_from("<Q", data, sh + 24)[0]
            name, size, _ = struct.unpack_from("<III", data, at)
            at += 12 + ((name + 3) & ~3)
            note = msgpack.unpackb(data[at:at + size], strict_map_key=False)
            out += note.get("amdhsa.kernels", [])
    return out


def test_one_launch_external_product_keeps_its_registers():
    import cfft_amd  # noqa: F401  (builds nothing; fails if the library is absent)
    from cfft_amd._lib import LIB_PATH
    fused = [k for k in kernels(LIB_PATH) if "k_extprod_fused" in k[".name"]]
    assert len(fused) == 36
    spilled = {k[".name"]: k[".private_segment_fixed_size"] for k in fused
               if k[".private_segment_fixed_size"]}
    assert not spilled, spilled


def test_eight_point_products_keep_their_registers():
    """n = 2048 ... 8192, every algo but Dif16 (whose radix-16 lane pairs keep
    12 to 20 bytes)."""
    from cfft_amd._lib import LIB_PATH
    found, spilled = 0, {}
    for k in kernels(LIB_PATH):
        m = re.search(r"k_polymul_fixed8ILi(\d+)ELi(\d+)E", k[".name"])
        if not m or int(m.group(1)) == 6 or int(m.group(2)) < 11:
            continue
        found += 1
        if k[".private_segment_fixed_size"]:
            spilled[k[".name"]] = k[".private_segment_fixed_size"]
    assert found == 36 and not spilled, (found, spilled)
