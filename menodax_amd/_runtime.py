"""ctypes binding of ``libmenodax_hip.so`` and the code-object cache.

The library is the C ABI declared in ``include/menodax_hip.h``. It is loaded
after ``torch`` so that both share one HIP runtime (they link the same
``libamdhip64.so.7`` soname; the first one loaded serves the process), which is
what lets a launch run on a torch stream and write into torch-allocated memory.

A missing library is an error, never a reason to fall back: there is no CPU
path in the product.
"""

from __future__ import annotations

import ctypes
import hashlib
import os
import re
import struct
import threading

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmenodax_hip.so")
KERNEL_DIR = os.path.join(_HERE, "kernels")
ARCH = "gfx950"

KERNEL_PERSISTENT = 1
KERNEL_UNIT_WEIGHTS = 2
KERNEL_ADJOINT = 4
KERNEL_HOOK = 8
KERNEL_WAVE = 16
KERNEL_RESUMABLE = 32
#: wavefronts per workgroup of a team kernel, in bits 8..12 of the flags
KERNEL_TEAM_SHIFT = 8

# Every kernel is compiled with contraction off (the fused multiply-adds are
# explicit in the source) and without packed FP32 instructions.
COMPILE_OPTIONS = (
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
)

#: Added where ``spills_ahead_of_exec`` finds a kernel wrong: no splitting of live
#: ranges over regions of blocks. Where registers run out, splitting puts scalar
#: copies at the head of a join block, ahead of the instruction that widens EXEC
#: again, and this compiler then puts vector copies and spills ahead of the scalar
#: ones, where only the lanes of the branch execute them, or none when it is
#: skipped: the joint Robertson solve (FP64, a controller with three terms) spilled
#: its second to last error inside the rarely taken redo of a back substitution and
#: read it back uninitialised, and a 19-variable rolled Tsit5 step went wrong the
#: same way. Kernels that are in order keep the code with splitting, which is
#: mostly faster (value and gradient of the 64-variable ring, one direction, 1,000
#: trajectories: 2.99 ms, without splitting 3.33; a row a lane, 32 variables FP64:
#: 1,665 us, without 1,732).
NO_REGION_SPLITTING = ("-mllvm", "-grow-region-complexity-budget=0")

_lib = None
_lock = threading.Lock()


class NativeError(RuntimeError):
    """A call into libmenodax_hip.so failed."""


def lib():
    """The loaded library, built on demand if this tree has never built it."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        import torch  # noqa: F401  (first: its HIP runtime is the process's)

        if not os.path.exists(LIB_PATH):
            raise NativeError(
                f"{LIB_PATH} is not built; run `python -m menodax_amd.build` "
                "(or __graft_entry__.build()) first"
            )
        L = ctypes.CDLL(LIB_PATH)
        i32, i64, vp, cp, dbl, sz = (
            ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p, ctypes.c_char_p,
            ctypes.c_double, ctypes.c_size_t,
        )
        L.mdx_abi_version.restype = i32
        L.mdx_last_error.restype = cp
        L.mdx_free.argtypes = [vp]
        L.mdx_free.restype = None
        L.mdx_rtc_compile.argtypes = [
            cp, cp, i32, ctypes.POINTER(cp), ctypes.POINTER(cp), i32, ctypes.POINTER(cp),
            ctypes.POINTER(vp), ctypes.POINTER(sz), ctypes.POINTER(ctypes.c_char_p),
        ]
        L.mdx_rtc_compile.restype = i32
        L.mdx_kernel_create.argtypes = [vp, sz, cp, i32, i32, ctypes.POINTER(i64)]
        L.mdx_kernel_create.restype = i32
        L.mdx_kernel_info.argtypes = [i64] + [ctypes.POINTER(i32)] * 4
        L.mdx_kernel_info.restype = i32
        L.mdx_persistent_grid.argtypes = [i64, ctypes.POINTER(i32)]
        L.mdx_persistent_grid.restype = i32
        L.mdx_workspace_bytes.argtypes = [i64, i64]
        L.mdx_workspace_bytes.restype = i64
        L.mdx_solve_launch.argtypes = [
            i64, vp, i32, i64, i32, i32, i32, i32,
            vp, vp, vp, dbl, dbl, dbl, i32, vp,
            vp, vp, vp, vp, vp, i32, vp, i64,
        ]
        L.mdx_solve_launch.restype = i32
        L.mdx_solve_launch_ordered.argtypes = L.mdx_solve_launch.argtypes + [vp]
        L.mdx_solve_launch_ordered.restype = i32
        L.mdx_cost_pilot_launch.argtypes = [
            i64, vp, i64, i32, i32, i32, i32, vp, vp, vp, dbl, dbl, dbl, i32, vp,
            vp, vp, vp, vp, vp,
        ]
        L.mdx_cost_pilot_launch.restype = i32
        L.mdx_cost_pilot_launch_resumable.argtypes = L.mdx_cost_pilot_launch.argtypes + [vp]
        L.mdx_cost_pilot_launch_resumable.restype = i32
        L.mdx_solve_launch_resumed.argtypes = [
            i64, vp, i32, i64, i32, i32, i32, i32, vp, vp, vp, dbl, dbl, dbl, i32, vp,
            vp, vp, vp, vp, vp, i64, vp, vp,
        ]
        L.mdx_solve_launch_resumed.restype = i32
        L.mdx_adjoint_workspace_bytes.argtypes = [i64, i32, i32, i32]
        L.mdx_adjoint_workspace_bytes.restype = i64
        L.mdx_adjoint_launch.argtypes = [
            i64, vp, i64, i32, i32, i32, i32, vp, vp, vp, dbl, dbl, dbl, i32, vp,
            vp, vp, vp, vp, i32, i32, vp, i64,
        ]
        L.mdx_adjoint_launch.restype = i32
        L.mdx_adjoint_launch_static.argtypes = L.mdx_adjoint_launch.argtypes[:-2]
        L.mdx_adjoint_launch_static.restype = i32
        L.mdx_device_info.argtypes = [ctypes.c_char_p, sz, ctypes.POINTER(i32)]
        L.mdx_device_info.restype = i32
        if L.mdx_abi_version() != 1:
            raise NativeError("libmenodax_hip.so has an unexpected ABI version; rebuild it")
        _lib = L
        return L


def _check(rc, what):
    if rc != 0:
        msg = lib().mdx_last_error().decode(errors="replace")
        raise NativeError(f"{what} failed ({rc}): {msg}")


def headers():
    """The kernel headers, as (name, text) pairs handed to hipRTC in memory."""
    out = []
    for name in sorted(os.listdir(KERNEL_DIR)):
        if name.endswith(".hpp"):
            with open(os.path.join(KERNEL_DIR, name)) as f:
                out.append((name, f.read()))
    return out


def _included(source: str, hdrs) -> list:
    """The headers ``source`` includes, directly or through one another, so
    that a kernel's cache key depends on nothing it does not read."""
    texts = dict(hdrs)
    seen, stack = set(), [source]
    while stack:
        for name in re.findall(r'^\s*#include "([^"]+)"', stack.pop(), re.M):
            if name in texts and name not in seen:
                seen.add(name)
                stack.append(texts[name])
    return [(n, t) for n, t in hdrs if n in seen]


#: code objects compiled ahead of time by ``build`` travel with the tree here
PACKAGE_CACHE = os.path.join(_HERE, "_kcache")


def _cache_dirs():
    """Lookup order for compiled code objects; the first writable one is where
    a fresh compile is stored."""
    dirs = []
    env = os.environ.get("MENODAX_KERNEL_CACHE")
    if env:
        dirs.append(env)
    dirs.append(PACKAGE_CACHE)
    dirs.append(os.path.join(os.path.expanduser("~"), ".cache", "menodax_amd", "kernels"))
    return dirs


def cache_key(source: str, hdrs, options) -> str:
    hdrs = _included(source, hdrs)
    h = hashlib.sha256()
    h.update(b"mdx-code-object-v3\0")
    h.update(source.encode())
    for name, text in hdrs:
        h.update(b"\0" + name.encode() + b"\0" + text.encode())
    for o in options:
        h.update(b"\0" + o.encode())
    return h.hexdigest()


def rtc_compile(source: str, name: str = "mdx_kernel.hip", hdrs=None, options=COMPILE_OPTIONS) -> bytes:
    """Compile with hipRTC (no cache)."""
    L = lib()
    hdrs = headers() if hdrs is None else hdrs
    n_h = len(hdrs)
    h_src = (ctypes.c_char_p * max(n_h, 1))(*[t.encode() for _, t in hdrs])
    h_nam = (ctypes.c_char_p * max(n_h, 1))(*[n.encode() for n, _ in hdrs])
    opts = (ctypes.c_char_p * len(options))(*[o.encode() for o in options])
    code = ctypes.c_void_p()
    size = ctypes.c_size_t()
    log = ctypes.c_char_p()
    rc = L.mdx_rtc_compile(
        source.encode(), name.encode(), n_h, h_src, h_nam, len(options), opts,
        ctypes.byref(code), ctypes.byref(size), ctypes.byref(log),
    )
    text = ""
    if log.value is not None:
        text = log.value.decode(errors="replace")
        L.mdx_free(ctypes.cast(log, ctypes.c_void_p))
    if rc != 0:
        raise NativeError(f"hipRTC compilation of {name} failed:\n{text}\n--- source ---\n{source}")
    try:
        return ctypes.string_at(code, size.value)
    finally:
        L.mdx_free(code)


_memory_cache: dict[str, bytes] = {}


def code_object(source: str, name: str = "mdx_kernel.hip", store_in: str | None = None) -> bytes:
    """Compile through the cache: memory, then disk (keyed on source, headers
    and options), then hipRTC. ``store_in`` forces a copy into that directory."""
    hdrs = headers()
    key = cache_key(source, hdrs, COMPILE_OPTIONS)
    if store_in is not None:
        data = code_object(source, name)
        os.makedirs(store_in, exist_ok=True)
        path = os.path.join(store_in, key + ".co")
        if not os.path.exists(path):
            tmp = f"{path}.{os.getpid()}.tmp"
            with open(tmp, "wb") as f:
                f.write(data)
            os.replace(tmp, path)
        return data
    hit = _memory_cache.get(key)
    if hit is not None:
        return hit
    for d in _cache_dirs():
        path = os.path.join(d, key + ".co")
        if os.path.exists(path):
            with open(path, "rb") as f:
                data = f.read()
            _memory_cache[key] = data
            return data
    data = rtc_compile(source, name, hdrs)
    if spills_ahead_of_exec(data):
        data = rtc_compile(source, name, hdrs, COMPILE_OPTIONS + NO_REGION_SPLITTING)
    _memory_cache[key] = data
    for d in _cache_dirs():
        try:
            os.makedirs(d, exist_ok=True)
            tmp = os.path.join(d, f"{key}.{os.getpid()}.tmp")
            with open(tmp, "wb") as f:
                f.write(data)
            os.replace(tmp, os.path.join(d, key + ".co"))
            break
        except OSError:
            continue
    return data


def spills_ahead_of_exec(code: bytes) -> bool:
    """Whether, where a branch for an empty EXEC lands or such a loop ends, some
    kernel of ``code`` spills or reloads vector registers ahead of the
    instruction that widens EXEC again: the lanes it brings back execute none of
    that."""
    words, start = _instructions(code)
    where = {a: i for i, a in enumerate(start)}
    for i, a in enumerate(start):
        w = words[a]
        if w >> 16 == 0xBF88:  # s_cbranch_execz
            at = where.get(a + 1 + (w & 0x7FFF) - (w & 0x8000))
        elif w >> 16 == 0xBF89:  # s_cbranch_execnz
            at = i + 1
        else:
            continue
        spilled = whole = waves = False
        for b in start[at:at + 400] if at is not None else ():
            w = words[b]
            sop1 = w >> 23 == 0x17D
            if sop1 and w & 0xFFFF == 0x21C1:  # s_or_saveexec_b64 s, -1: scalar registers'
                whole = waves = True           # spills, for the whole wavefront
            elif whole:
                whole = not (sop1 and w >> 8 == 0xBEFE01)  # s_mov_b64 exec, s
            elif w >> 16 == 0x87FE and w & 0xFF == 0x7E:  # s_or_b64 exec, exec, s
                if spilled:
                    return True
                break
            elif (0xBF81 <= w >> 16 <= 0xBF89 and w >> 16 != 0xBF83  # a branch or the end
                  or sop1 and (0x20 <= w >> 8 & 0xFF <= 0x27 or w >> 8 & 0xFF in (0x1D, 0x1E))
                  or w >> 30 == 2 and w >> 28 != 0xB and w >> 16 & 0x7F == 0x7E
                  and not 0x17E <= w >> 23):  # EXEC written otherwise
                break
            elif w >> 16 == 0xD3D9:  # v_accvgpr_write
                spilled = True
            elif w >> 26 == 0x37 and w >> 14 & 3 == 1:  # scratch: opcodes from 24 on store
                spilled |= w >> 18 & 0x7F >= 0x18 or not waves
            elif w >> 16 == 0xD3D8:  # v_accvgpr_read
                spilled |= not waves
    return False


def _instructions(code):
    """The words of an AMD code object's text and the indices its instructions
    start at, by the lengths of their encodings."""
    table, = struct.unpack_from("<Q", code, 40)
    entry, n = struct.unpack_from("<HH", code, 58)
    words, start = [], []
    for k in range(n):
        _, kind, flags, _, off, size = struct.unpack_from("<IIQQQQ", code, table + k * entry)
        if kind != 1 or not flags & 4:
            continue
        words += struct.unpack_from(f"<{size // 4}I", code, off)
    i = 0
    while i < len(words):
        start.append(i)
        w = words[i]
        if w >> 31 == 0:  # VOP1, VOP2, VOPC: a literal, SDWA or DPP; fused with a constant
            long = w & 0x1FF in (0xFF, 0xF9, 0xFA) or w >> 25 in (0x17, 0x18, 0x24, 0x25)
        elif w >> 28 == 0xB and w >> 23 not in (0x17D, 0x17E, 0x17F):
            long = w >> 23 & 0x1F == 0x14  # SOPK: s_setreg_imm32
        elif w >> 30 == 2:
            long = (w >> 23 != 0x17F and w & 0xFF == 0xFF
                    or w >> 23 not in (0x17D, 0x17F) and w >> 8 & 0xFF == 0xFF)
        else:
            long = w >> 26 != 0x35
        i += 1 + long
    return words, start


def kernel_registers(code: bytes) -> dict:
    """Per kernel of a code object, from its metadata (a MessagePack map per
    kernel, keys in alphabetical order): a lane's vector registers, the
    accumulation registers among them, those spilled and its scratch bytes, and
    the workgroup's most threads."""
    def number(key, after):
        at = code.index(key, after) + len(key)
        head = code[at]
        if head < 0x80:
            return head
        size = {0xCC: 1, 0xCD: 2, 0xCE: 4}[head]
        return int.from_bytes(code[at + 1:at + 1 + size], "big")

    out, key = {}, b".symbol"
    at = code.find(key)
    while at >= 0:
        at += len(key)
        # a string: its length in the head byte, or in the byte after it
        short = code[at] != 0xD9
        size, start = (code[at] - 0xA0, at + 1) if short else (code[at + 1], at + 2)
        name = code[start:start + size].decode().removesuffix(".kd")
        before = {k: number(k, code.rindex(k, 0, at)) for k in (
            b".agpr_count", b".max_flat_workgroup_size", b".private_segment_fixed_size")}
        out[name] = dict(vgprs=number(b".vgpr_count", at), agprs=before[b".agpr_count"],
                         spills=number(b".vgpr_spill_count", at),
                         scratch=before[b".private_segment_fixed_size"],
                         threads=before[b".max_flat_workgroup_size"])
        at = code.find(key, at)
    return out


def kernel_create(code: bytes, entry: str, block: int, flags: int) -> int:
    handle = ctypes.c_int64()
    buf = ctypes.create_string_buffer(code, len(code))
    _check(
        lib().mdx_kernel_create(buf, len(code), entry.encode(), int(block), int(flags), ctypes.byref(handle)),
        f"mdx_kernel_create({entry})",
    )
    return int(handle.value)


def kernel_info(handle: int) -> dict:
    v, s, l, b = (ctypes.c_int32() for _ in range(4))
    _check(
        lib().mdx_kernel_info(handle, ctypes.byref(v), ctypes.byref(s), ctypes.byref(l), ctypes.byref(b)),
        "mdx_kernel_info",
    )
    return dict(vgprs=v.value, scratch_bytes=s.value, lds_bytes=l.value, blocks_per_cu=b.value)


def persistent_grid(handle: int) -> int:
    g = ctypes.c_int32()
    _check(lib().mdx_persistent_grid(handle, ctypes.byref(g)), "mdx_persistent_grid")
    return int(g.value)


def workspace_bytes(handle: int, n_traj: int) -> int:
    v = lib().mdx_workspace_bytes(handle, n_traj)
    if v < 0:
        _check(1, "mdx_workspace_bytes")
    return int(v)


def device_info():
    buf = ctypes.create_string_buffer(128)
    n_cu = ctypes.c_int32()
    _check(lib().mdx_device_info(buf, 128, ctypes.byref(n_cu)), "mdx_device_info")
    return buf.value.decode(), int(n_cu.value)


def adjoint_workspace_bytes(n_traj, n_vars, ckpt_every, max_ckpt) -> int:
    v = lib().mdx_adjoint_workspace_bytes(int(n_traj), int(n_vars), int(ckpt_every), int(max_ckpt))
    if v < 0:
        raise ValueError("mdx_adjoint_workspace_bytes: bad extents")
    return int(v)


def adjoint_launch(handle, stream, n_traj, n_vars, n_params, n_save, layout, y0, times, params,
                   dt0, rtol, atol, max_steps, weights, gbar, grad_y0, grad_p, status,
                   ckpt_every, max_ckpt, workspace, workspace_bytes):
    """Launch through ``mdx_adjoint_launch``; pointers are plain integers."""
    _check(
        lib().mdx_adjoint_launch(
            handle, stream, int(n_traj), int(n_vars), int(n_params), int(n_save), int(layout),
            y0, times, params or None, float(dt0), float(rtol), float(atol), int(max_steps),
            weights or None, gbar, grad_y0, grad_p or None, status, int(ckpt_every),
            int(max_ckpt), workspace, int(workspace_bytes),
        ),
        "mdx_adjoint_launch",
    )


#: bytes of the static device scratch behind ``adjoint_launch_static``
#: (``MDX_STATIC_SCRATCH_BYTES`` in include/menodax_hip.h)
STATIC_SCRATCH_BYTES = 64 << 20


def adjoint_launch_static(handle, stream, n_traj, n_vars, n_params, n_save, layout, y0, times,
                          params, dt0, rtol, atol, max_steps, weights, gbar, grad_y0, grad_p,
                          status, ckpt_every, max_ckpt):
    """Launch through ``mdx_adjoint_launch_static``: as ``adjoint_launch``, with
    the checkpoints in the library's static device scratch instead of a
    workspace (nothing is allocated)."""
    _check(
        lib().mdx_adjoint_launch_static(
            handle, stream, int(n_traj), int(n_vars), int(n_params), int(n_save), int(layout),
            y0, times, params or None, float(dt0), float(rtol), float(atol), int(max_steps),
            weights or None, gbar, grad_y0, grad_p or None, status, int(ckpt_every),
            int(max_ckpt),
        ),
        "mdx_adjoint_launch_static",
    )


def solve_launch(handle, stream, grid, n_traj, n_vars, n_params, n_save, layout, y0, times, params,
                 dt0, rtol, atol, max_steps, weights, hist, accepted, rejected, loop_steps,
                 hook_out=0, hook_size=0, workspace=0, workspace_bytes=0, order=0, resume=0):
    """Launch through ``mdx_solve_launch`` (``mdx_solve_launch_ordered`` when a
    claim ``order`` pointer is given, ``mdx_solve_launch_resumed`` when a
    pilot's step-state buffer ``resume`` is); pointers are plain integers."""
    if resume:
        if hook_out or hook_size:
            raise ValueError("a resumed solve runs no save hook")
        _check(lib().mdx_solve_launch_resumed(
            handle, stream, int(grid), int(n_traj), int(n_vars), int(n_params), int(n_save),
            int(layout), y0, times, params, float(dt0), float(rtol), float(atol),
            int(max_steps), weights or None, hist, accepted, rejected, loop_steps,
            workspace or None, int(workspace_bytes), order or None, resume),
            "mdx_solve_launch_resumed")
        return
    args = (handle, stream, int(grid), int(n_traj), int(n_vars), int(n_params), int(n_save),
            int(layout), y0, times, params, float(dt0), float(rtol), float(atol), int(max_steps),
            weights or None, hist, accepted, rejected, loop_steps, hook_out or None,
            int(hook_size), workspace or None, int(workspace_bytes))
    if order:
        _check(lib().mdx_solve_launch_ordered(*args, order), "mdx_solve_launch_ordered")
    else:
        _check(lib().mdx_solve_launch(*args), "mdx_solve_launch")


def cost_pilot_launch(handle, stream, n_traj, n_vars, n_params, n_save, layout, y0, times, params,
                      dt0, rtol, atol, steps, weights, hist, accepted, rejected, loop_steps, cost,
                      resume=0):
    """Launch through ``mdx_cost_pilot_launch`` (``_resumable`` when a
    step-state buffer ``resume`` is given); pointers are plain integers."""
    args = (handle, stream, int(n_traj), int(n_vars), int(n_params), int(n_save), int(layout),
            y0, times, params, float(dt0), float(rtol), float(atol), int(steps),
            weights or None, hist, accepted, rejected, loop_steps, cost)
    if resume:
        _check(lib().mdx_cost_pilot_launch_resumable(*args, resume),
               "mdx_cost_pilot_launch_resumable")
    else:
        _check(lib().mdx_cost_pilot_launch(*args), "mdx_cost_pilot_launch")
