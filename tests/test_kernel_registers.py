"""Registers of built kernels, from the notes of their code objects: as many
blocks fit a CU as a kernel's comments and the rules that choose it count on,
nothing that was asked for early is spilled, and where a kernel spills it is no
more than its comment says."""

import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def kernels(lib, tmp):
    """Name -> (vector registers, spilled ones) of a library's kernels."""
    fat = os.path.join(tmp, "fat")
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin",
                    "--set-section-flags", ".hip_fatbin=alloc", lib, fat],
                   check=True)
    data, out = open(fat, "rb").read(), {}
    for m in re.finditer(MAGIC, data):
        i = m.start()
        (n,), at = struct.unpack_from("<Q", data, i + 24), i + 32
        for _ in range(n):
            off, size, name = struct.unpack_from("<QQQ", data, at)
            target, at = data[at + 24:at + 24 + name], at + 24 + name
            if b"gfx950" not in target:
                continue
            co = os.path.join(tmp, "co")
            with open(co, "wb") as f:
                f.write(data[i + off:i + off + size])
            text = subprocess.run([READELF, "--notes", co], check=True,
                                  capture_output=True, text=True).stdout
            for k in text.split("\n  - .agpr_count:")[1:]:
                get = lambda s: re.search(rf"\.{s}:\s+(\S+)", k).group(1)
                out[get("name")] = (int(get("vgpr_count")),
                                    int(get("vgpr_spill_count")))
    return out


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    from csrc.build import ensure_built
    return {n: kernels(lib, str(tmp_path_factory.mktemp(n))) for n, lib in
            zip(("gqa", "llmops"), ensure_built(names=["gqa", "llmops"]))}


def waves(registers):
    """Waves that a SIMD holds; registers go out in eights."""
    return min(8, 512 // (-(-registers // 8) * 8))


# keys and values that are asked for ahead of the norms, of each padded size; a
# block has a wave on each SIMD
@pytest.mark.parametrize("kind,DP,VP,least", [
    ("f", 64, 64, 3), ("f", 64, 128, 2), ("f", 128, 64, 2), ("f", 128, 128, 1),
    ("f", 256, 256, 1), ("t", 64, 64, 4), ("t", 64, 128, 2), ("t", 128, 64, 3),
    ("t", 128, 128, 2), ("t", 256, 256, 1)])
def test_new_tokens_attention(built, kind, DP, VP, least):
    found = [v for n, v in built["gqa"].items()
             if f"k_gqa_tokenI{kind}Li{DP}ELi{VP}E" in n]
    assert len(found) == 1
    registers, spilled = found[0]
    assert spilled == 0 and waves(registers) >= least


def test_product_tiles(built):
    """Two waves on each SIMD: a block of eight, or two blocks of four."""
    found = {n: v for n, v in built["llmops"].items()
             if "k_gemm_promptI" in n or "k_gemm_wideI" in n}
    assert any("k_gemm_promptILb0ELi128ELi128ELi2ELi2ELi2ELb1ELb0ELb1E" in n
               for n in found)                          # beside MXFP4
    for n, (registers, spilled) in found.items():
        assert spilled == 0 and waves(registers) >= 2, n


# dims, keys a tile, waves that share the rows, groups of them, e4m3 pool, cap:
# registers that are spilled
ROWS_SPILL = {(64, 64, 4, 2, 0, 0): 1,
              (256, 32, 1, 1, 1, 0): 6, (256, 32, 1, 1, 1, 1): 6,
              (256, 32, 4, 1, 1, 0): 28, (256, 32, 4, 1, 1, 1): 29}


def test_prompt_attention(built):
    """Four waves or two groups of four: two blocks a CU, of 128 dims by two
    groups one; blocks of one wave have what LDS leaves of the registers."""
    found = {}
    for n, v in built["llmops"].items():
        m = re.search(r"k_attn_rowsILi(\d+)ELi(\d+)ELi(\d)ELi(\d)ELb(\d)ELb(\d)E",
                      n)
        if m:
            found[tuple(map(int, m.groups()))] = v
    assert set(ROWS_SPILL) <= set(found)
    assert {k[0] for k in found} == {64, 128, 256}
    for k, (registers, spilled) in found.items():
        hd, _, nw, groups = k[:4]
        least = 1 if nw == 1 else 4 if groups == 2 and hd == 64 else 2
        assert waves(registers) >= least, k
        assert spilled <= ROWS_SPILL.get(k, 0), k
