"""C ABI: the library loads, exports every symbol include/lfh.h declares, and
rejects bad input with status codes and messages (no GPU needed: every case
here fails before any device work)."""
import ctypes as C
import re

import numpy as np
import pytest

from lavaframe_amd import lfh, scenes


def test_exports_every_declared_symbol(lib):
    declared = lfh.header_symbols()
    assert len(declared) > 40
    missing = [s for s in declared if not hasattr(lib, s)]
    assert missing == []
    assert lib.lfh_abi_version() == 1


def test_native_library_is_in_tree():
    assert lfh.LIB_PATH.exists()
    assert lfh.LIB_PATH.parent.parent.name == "lavaframe_amd"


def test_device_clears_name_their_stream():
    """Contexts and servers work on non-blocking streams, which the null stream
    is not ordered with: a clear queued on the null stream could land after
    the first kernel that counts on it (or writes what it clears)."""
    csrc = lfh.LIB_PATH.parent.parent / "csrc"
    files = [f for f in csrc.iterdir() if f.suffix in (".cpp", ".hip", ".h")]
    assert len(files) > 20
    on_null = [f"{f.name}: {line.strip()}" for f in files for line in f.read_text().splitlines()
               if re.search(r"\bhipMemset(D8|D16|D32|2D|3D)?\(", line)]
    assert on_null == []


def test_null_arguments_return_invalid(lib):
    assert lib.lfh_scene_create(None) == -1
    assert b"NULL" in lib.lfh_last_error(None)
    assert lib.lfh_create(None, None, None) == -1
    assert lib.lfh_scene_load(None, None) == -1


def test_missing_scene_file_is_io_error(lib):
    s = lfh.Scene(lib)
    with pytest.raises(lfh.LfhError) as e:
        s.load("/nonexistent/scene.lfs")
    assert e.value.code == -5


def _desc(arr):
    return lfh.desc_from_arrays(arr)


def _bad_create(lib, arr, opts=None):
    d, keep = _desc(arr)
    o = opts or lfh.Options(width=8, height=8, max_depth=2, kahan=1)
    h = C.c_void_p()
    code = lib.lfh_create(C.byref(d), C.byref(o), C.byref(h))
    return code, lib.lfh_last_error(None).decode()


def test_create_rejects_bad_layouts(lib):
    arr = scenes.soup(50).arrays()
    bad = dict(arr)
    bad["top_level_index"] = arr["nodes"].shape[0] + 5
    code, msg = _bad_create(lib, bad)
    assert code == -1 and "top_level_index" in msg
    # a child pointing back at its parent would make traversal loop
    bad = dict(arr)
    nodes = arr["nodes"].copy()
    internal = np.nonzero(nodes[:, 8] == 0)[0]
    nodes[internal[1], 6] = internal[0]
    bad["nodes"] = nodes
    code, msg = _bad_create(lib, bad)
    assert code == -1
    # vertex indices out of range
    bad = dict(arr)
    vi = arr["vert_indices"].copy()
    vi[0, 0] = 10**7
    bad["vert_indices"] = vi
    code, msg = _bad_create(lib, bad)
    assert code == -1 and "vertex index" in msg
    # leaf with too many triangles for the packed encoding
    bad = dict(arr)
    nodes = arr["nodes"].copy()
    leaf = np.nonzero(nodes[:, 8] > 0)[0][0]
    nodes[leaf, 7] = 9
    bad["nodes"] = nodes
    code, msg = _bad_create(lib, bad)
    assert code == -1
    # no materials
    bad = dict(arr)
    bad["materials"] = np.zeros((0, 28), np.float32)
    code, msg = _bad_create(lib, bad)
    assert code == -1 and "material" in msg
    # bad resolution
    code, msg = _bad_create(lib, arr, lfh.Options(width=0, height=8, max_depth=2))
    assert code == -1


def test_scene_builder_errors(lib):
    s = lfh.Scene(lib)
    with pytest.raises(lfh.LfhError):
        s.add_instance(3, None, 0)            # no such mesh
    with pytest.raises(lfh.LfhError):
        s.build()                              # no instances
    m = s.add_mesh(scenes.unit_cube_tris())
    s.add_instance(m, None, 5)                 # material 5 does not exist
    with pytest.raises(lfh.LfhError):
        s.build()
