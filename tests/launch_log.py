"""What libprichs_hip.so launches, seen on the CPU: a call runs in a fresh
process over tests/cpp/launch_log.cpp, which notes each kernel instead of
running it."""
import collections
import ctypes as C
import json
import os
import re
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

# kernel: its name with template arguments, without namespaces and parameters.
Launch = collections.namedtuple("Launch", "kernel symbol grid block lds device")
_so = None


def _build():
    global _so
    if _so is None:
        _so = tempfile.NamedTemporaryFile(suffix=".so")
        subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-fPIC", "-shared", "-w",
                        "-I", os.path.join(ROCM, "include"),
                        os.path.join(ROOT, "tests", "cpp", "launch_log.cpp"), "-o", _so.name],
                       check=True)
    return _so.name


def run(body, **env):
    """Runs `body` (Python text that sets `result`) with `lib`, `L`, `C`,
    `engine(...)` and `launches()` at hand, and returns `result`.  env: further
    environment variables."""
    code = "import sys; sys.path.insert(0, %r)\nfrom tests.launch_log import *\n" \
           "lib, L = start(%r)\n%s\nprint('RESULT' + json.dumps(result))\n" % (ROOT, _build(), body)
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, **env},
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    out = json.loads(r.stdout[r.stdout.index("RESULT") + 6:])
    return out


def as_launches(rows):
    return [Launch(*r) for r in rows]


# ------------------------------------------------- in the process of a call --
_log = None
P = 1 << 20  # a 16-byte aligned address; nothing dereferences it


def start(so):
    global _log
    _log = C.CDLL(so, mode=C.RTLD_GLOBAL)
    _log.launch_log_take.restype = C.c_char_p
    from prichs_amd import _lib as L

    return L.load(), L


def hip():
    """The stand-in library (hipSetDevice)."""
    return _log


def raw_events():
    """The log since the last call: rows of text, launches and raised limits."""
    return [ln.split("\t") for ln in _log.launch_log_take().decode().splitlines()]


def _short(name):
    name = name.replace("(anonymous namespace)::", "").replace("prichs::", "")
    name = re.sub(r"^void ", "", name)
    depth = 0
    for i, ch in enumerate(name):  # up to the parameter list
        depth += (ch == "<") - (ch == ">")
        if ch == "(" and depth == 0:
            return name[:i]
    return name


def launches():
    """The kernels launched since the last call, as Launch rows."""
    return [[_short(r[0]), r[1], [int(v) for v in r[2:5]], int(r[5]), int(r[6]), int(r[7])]
            for ev, *r in raw_events() if ev == "launch"]


def engine(d, f, E, k, dtype, max_tokens, backward=False):
    """An uploaded engine with one shared expert (all weights zero)."""
    from prichs_amd import _lib as L

    lib, h = L.load(), C.c_void_p()
    L.check(lib.prichs_moe_engine_create(d, f, E, k, 1, dtype, max_tokens, C.byref(h)))
    z = (C.c_float * (d * f))()
    ptrs = (C.c_void_p * (E + 1))(*[C.addressof(z)] * (E + 1))
    w, b = (C.c_float * (d * E))(), (C.c_float * E)()
    if backward:
        L.check(lib.prichs_moe_engine_enable_backward(h))
    L.check(lib.prichs_moe_engine_upload(h, w, b, ptrs, ptrs, ptrs))
    return h


def _unpack(b, i):
    """The MessagePack value at b[i] and the index past it (what code object
    metadata holds: maps, arrays, texts, whole numbers, truth values)."""
    t = b[i]
    i += 1

    def number(n):
        return int.from_bytes(b[i:i + n], "big"), i + n

    if t < 0x80:
        return t, i
    if t in (0xc2, 0xc3):
        return t == 0xc3, i
    if 0xcc <= t <= 0xcf:
        return number(1 << (t - 0xcc))
    if t >> 5 == 5:
        n = t & 31
    elif t >> 5 == 4:
        n = t & 15
    else:
        n, i = number({0xd9: 1, 0xda: 2, 0xdb: 4, 0xdc: 2, 0xdd: 4, 0xde: 2, 0xdf: 4}[t])
    if t >> 5 == 5 or 0xd9 <= t <= 0xdb:
        return b[i:i + n].decode(), i + n
    is_map, items = t >> 4 == 8 or t >= 0xde, []
    for _ in range(2 * n if is_map else n):
        v, i = _unpack(b, i)
        items.append(v)
    return (dict(zip(items[::2], items[1::2])) if is_map else items), i


def static_lds(library=os.environ.get("PRICHS_HIP_LIB") or os.path.join(
        ROOT, "prichs_amd", "libprichs_hip.so")):
    """Bytes of LDS that each kernel of the library has at launch (besides its
    dynamic LDS), by symbol, from its code objects' metadata."""
    data, out, at = open(library, "rb").read(), {}, 0
    key = b"\xaeamdhsa.kernels"
    while (at := data.find(key, at)) >= 0:
        kernels, _ = _unpack(data, at + len(key))
        for k in kernels:
            out[k[".name"]] = k[".group_segment_fixed_size"]
        at += len(key)
    return out
