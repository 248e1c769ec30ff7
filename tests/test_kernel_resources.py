"""What the compiler reports for the kernels of the built library (the metadata of its
gfx950 code objects): scratch memory and registers of the tile passes."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name with its template arguments -> (VGPRs, bytes of scratch a lane)"""
    with open(os.path.join(PKG, "libpbd.so"), "rb") as f:
        data = f.read()
    found, at = {}, 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, name = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + name] and size:
                obj = tmp_path_factory.mktemp("co") / "kernels.o"
                obj.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
                for k in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
                    get = lambda key: re.search(r"\." + key + r":\s+(\S+)", k).group(1)  # noqa: E731
                    found[get("name")] = (int(get("vgpr_count")), int(get("private_segment_fixed_size")))
            entry += 24 + name
        at += 24
    names = subprocess.run(["c++filt"], input="\n".join(found), check=True, capture_output=True, text=True).stdout
    out = {re.sub(r"^void pbd::(\(anonymous namespace\)::)?", "", n).split(">(")[0]: v
           for n, v in zip(names.split("\n"), found.values())}
    assert out, "no gfx950 kernels in the library"
    return out


def _of(kernels, *names):
    return {k: v for k, v in kernels.items() if k.split("<")[0] in names}


def test_tile_passes_use_no_scratch(kernels):
    """A list walk in scratch memory waits for it in every chunk of eight pairs."""
    passes = _of(kernels, "k_tile_lambda", "k_tile_delta", "k_tile_omega", "k_tile_final", "k_wide_lambda",
                 "k_wide_omega", "k_tile_adjlist_forward")
    assert len(passes) > 50
    bad = {k: v[1] for k, v in passes.items() if v[1]}
    assert not bad, bad


def test_capped_grid_passes_keep_four_waves(kernels):
    """The passes whose workgroups take tile after tile (batches, large boxes) hold at most
    128 registers a lane: four waves on a SIMD."""
    stride = {"k_tile_lambda": r"<5, \w+, true, ", "k_tile_delta": r"<5, \w+, \d, true, ",
              "k_tile_omega": r"<5, \w+, true, ", "k_tile_final": r"<5, \w+, \w+, true, "}
    vgprs = {k: v[0] for k, v in kernels.items() for n, args in stride.items() if re.match(n + args, k)}
    assert len(vgprs) == 12, sorted(vgprs)
    bad = {k: v for k, v in vgprs.items() if v > 128}
    assert not bad, bad


def test_reverse_list_builders_keep_four_waves(kernels):
    built = _of(kernels, "k_tile_adjlist", "k_tile_adjlist_redo", "k_tile_adjlist_wide")
    assert len(built) == 3, sorted(built)
    bad = {k: v for k, v in built.items() if v[0] > 128 or v[1]}
    assert not bad, bad
