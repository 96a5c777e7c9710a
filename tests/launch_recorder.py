"""What the library would launch, seen without a GPU: record() runs calls of the C ABI in a child process in which
tests/launch_recorder.c stands in for the HIP runtime's launch entry points."""
import ctypes as C
import functools
import json
import os
import re
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# variant bits of fwd_kernel.h, as they appear in a kernel's name
VEC, ALIBI, DROPOUT, FULL_D, STAMP, ALIBI_LEFT, KV_ONCE, EVERY, NARROW, FOLD, PAIR = (1 << i for i in range(11))


@functools.lru_cache(maxsize=None)
def _recorder():
    """The stand-in, built once per test run."""
    folder = tempfile.mkdtemp(prefix="launch_recorder_")
    so = os.path.join(folder, "recorder.so")
    subprocess.check_call(["gcc", "-std=c11", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(HERE, "launch_recorder.c"), "-o", so])
    return so


def record(calls):
    """calls: dicts of flash_params fields (pointers that a call needs are filled in with made-up, aligned addresses), plus
    "entry" ("forward" or "splitkv").  Per call a dict: rc; launches [{kernel, variant, groups, threads, split_count}]; and what the
    size queries say of the same fields without the buffers they are about: splits, workspace (bytes of both parts),
    stamp_bytes."""
    out = subprocess.run([sys.executable, os.path.abspath(__file__), _recorder()], input=json.dumps(calls), capture_output=True,
                         text=True, timeout=600)
    assert out.returncode == 0, out.stderr[-3000:]
    return json.loads(out.stdout)


def form(launch):
    """What a tiled launch's work-groups are: "narrow" (32 rows), "paired" (two halves of four waves), "tall" (256 rows, four waves),
    "8-wave" (256 rows) or "plain" (128 rows)."""
    if "fwd_pp_kernel" in launch["kernel"]:
        return "8-wave"
    if launch["variant"] & (NARROW | PAIR):
        return "narrow" if launch["variant"] & NARROW else "paired"
    return "tall" if launch["kernel"].split("ELi")[1] == "2" else "plain"


def call(B, H, Hk, Nq, Nk, d, p=0.0, causal=False, window=(-1, -1), alibi=False, num_splits=1, kernel_hint=0):
    """A call in the words of the GPU tests, for record()."""
    c = dict(entry="splitkv" if num_splits != 1 else "forward", B=B, H=H, H_kv=Hk, Nq=Nq, Nk=Nk, d=d, is_causal=int(causal),
             window_left=window[0], window_right=window[1], dropout_p=p, num_splits=num_splits, kernel_hint=kernel_hint)
    return dict(c, alibi_slopes=0xA00000) if alibi else c


def _child(so):
    sys.path.insert(0, ROOT)
    sys.modules["torch"] = None  # (the binding loads torch's HIP runtime first where there is one)
    rec = C.CDLL(so, mode=C.RTLD_GLOBAL)
    rec.recorder_name.restype = C.c_char_p
    rec.recorder_groups.restype = rec.recorder_threads.restype = C.c_ulonglong
    from flash_attn_amd import binding

    L = binding.lib()
    res = []
    for call in json.load(sys.stdin):
        entry = call.pop("entry")
        split = entry == "splitkv"
        p = binding.FlashParams()
        L.flash_params_init(C.byref(p))
        p.softmax_scale = 0.125
        for name, value in call.items():
            setattr(p, name, value)
        # sizes first, as a caller asks for them
        stamps, p.stage_stamps_out = p.stage_stamps_out, None
        o, l, s = C.c_size_t(), C.c_size_t(), C.c_size_t()
        L.flash_splitkv_workspace_bytes(C.byref(p), C.byref(o), C.byref(l))
        L.flash_stage_stamps_bytes(C.byref(p), int(split), C.byref(s))
        splits = L.flash_splitkv_resolve_splits(C.byref(p))
        p.Q, p.K, p.V, p.O, p.LSE, p.O_partial, p.LSE_partial = (0x100000 * (i + 1) for i in range(7))
        p.stage_stamps_out = stamps
        rec.recorder_clear()
        rc = (L.flash_forward_splitkv if split else L.flash_forward)(C.byref(p), None)
        launches = []
        for i in range(rec.recorder_count()):
            name = rec.recorder_name(i).decode()
            m = re.search(r"fwd_(?:pp_)?kernelILi\d+E(?:Li\d+E)?Li(\d+)E", name)
            launches.append(dict(kernel=name, variant=int(m.group(1)) if m else None, groups=rec.recorder_groups(i),
                                 threads=rec.recorder_threads(i), split_count=rec.recorder_split_count(i)))
        res.append(dict(rc=rc, launches=launches, splits=splits, workspace=(o.value, l.value), stamp_bytes=s.value))
    json.dump(res, sys.stdout)


if __name__ == "__main__":
    _child(sys.argv[1])
