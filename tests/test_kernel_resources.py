"""What the compiled kernels take of a compute unit, read from the metadata of
the gfx950 code objects in the engine library (no device)."""
import os
import re
import struct

import msgpack

import alps_amd as A

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels():
    """Metadata of every gfx950 kernel: name -> dict."""
    with open(A.LIB_PATH, "rb") as f:
        d = f.read()
    out = {}
    at = d.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", d, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", d, p)
            triple = d[p + 24:p + 24 + tl].decode()
            p += 24 + tl
            if "gfx950" in triple and size:
                out.update(metadata(d[at + off:at + off + size]))
        at = d.find(MAGIC, at + 1)
    return out


def metadata(elf):
    (shoff,) = struct.unpack_from("<Q", elf, 40)
    shsize, shnum = struct.unpack_from("<HH", elf, 58)
    for s in range(shnum):
        sh = shoff + s * shsize
        if struct.unpack_from("<I", elf, sh + 4)[0] == 7:  # SHT_NOTE
            (o,) = struct.unpack_from("<Q", elf, sh + 24)
            name, desc, _ = struct.unpack_from("<III", elf, o)
            md = msgpack.unpackb(elf[o + 12 + (name + 3) // 4 * 4:][:desc])
            return {k[".name"]: k for k in md["amdhsa.kernels"]}
    return {}


def test_table_kernel_keeps_eight_waves():
    # short segments: the kernel with low-low target tables lives on waves in
    # flight (512 registers per lane and SIMD, eight waves of 64)
    ks = {n: k for n, k in kernels().items() if "hv_ranked_kernel" in n}
    assert any(re.search("hv_ranked_kernelId", n) for n in ks)
    for n, k in ks.items():
        if re.search("hv_ranked_kernelId", n):
            assert k[".vgpr_count"] + k[".agpr_count"] <= 64 and k[".vgpr_spill_count"] == 0, n


def test_every_schedule_is_a_kernel():
    # six FP32 schedules (ALPS_ED_HV_SCHEDULES) with and without the dot, of
    # the page kernel (gathered and staged; and its 512-thread form) and of the
    # table kernel
    ks = [n for n in kernels() if "9hv_kernelIf" in n or "hv_ranked_kernelIf" in n]
    assert sum("hv_ranked_kernelIf" in n for n in ks) == 2 * A.Operator.HV_SCHEDULES
    assert sum("9hv_kernelIf" in n for n in ks) == 4 * (A.Operator.HV_SCHEDULES + 1)


def test_reorthogonalization_launches_the_updates_threads():
    # its grid is the update's (one norm partial per block): so are its blocks
    ks = kernels()
    sizes = {kind: {k[".max_flat_workgroup_size"] for n, k in ks.items() if kind in n}
             for kind in ("update_fused_kernel", "reorth_update_kernel")}
    assert sizes["update_fused_kernel"] == sizes["reorth_update_kernel"] != set()


def test_kernels_that_address_lds_hold_no_static_lds():
    # lds_ld / lds_st (ed_device.hpp) take addresses from 0 on, where the
    # dynamic allocation starts only if the kernel has no __shared__ variable
    ks = kernels()
    for kind in ("9hv_kernelI", "hv_ranked_kernelI", "batch_hv_kernelI", "batch_plain_hv_kernel", "flip_gram_kernelI"):
        found = {n: k[".group_segment_fixed_size"] for n, k in ks.items() if kind in n}
        assert found and not any(found.values()), (kind, found)
    # the metadata does tell: kernels that have such variables report them
    assert any(k[".group_segment_fixed_size"] for n, k in ks.items() if "update_fused_kernel" in n)
