"""lv_decode_attn_store is exported and rejects bad arguments on the host, before any launch."""
import ctypes
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_header_and_arguments():
    from light_vllm_amd import _lib
    lib = _lib.load()
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "lv_decode_store.h")).read(), flags=re.S)
    args = re.search(r"lv_decode_attn_store\s*\(([^;]*?)\)\s*;", text, flags=re.S).group(1)
    assert args.count(",") + 1 == len(_lib.STORE_SIGNATURES["lv_decode_attn_store"][1])
    buf = ctypes.create_string_buffer(256)
    p = (ctypes.addressof(buf) + 15) & ~15

    def call(q=p, key=p, value=p, ks=1024, vs=1024, slots=p, nslots=512, B=1, Hq=16, Hkv=8, splits=1, scale=0.1):
        return lib.lv_decode_attn_store(q, key, value, ks, vs, p, p, slots, nslots, p, 2048, 2048, p, p, 2, B, 2, 256, Hq, Hkv, 128, scale,
                                        None, 0, splits, None, 0, None)

    assert call(B=0) == 0
    for bad in (dict(key=None), dict(value=None), dict(slots=None), dict(q=None), dict(ks=512), dict(vs=1000), dict(nslots=-1), dict(Hq=20),
                dict(scale=-1.0)):
        assert call(**bad) == -1, bad
    assert call(ks=1028) == -2 and call(key=p + 2) == -2
    assert call(splits=4) < 0                       # splits without a workspace
