"""Build step: turn the compiler's per-kernel resource report for the fused
kernels (hipcc -Rpass-analysis=kernel-resource-usage on csrc/fa_fused.hip)
into csrc/fa_resources.hpp's table, written as a C++ source file that is
compiled into libfa_mi355x.so.

Used by _build.py (which passes the remarks of its own compile of
fa_fused.hip) and, as a script, by the CMake build (which runs a device-only
compile of fa_fused.hip just for the report):

    python kernel_resources.py --hipcc HIPCC --source fa_fused.hip --out table.cpp -- <hipcc flags>
"""
from __future__ import annotations

import argparse
import re
import subprocess
import sys

_NAME = re.compile(r"remark: Function Name: (\S+)")
_FIELD = re.compile(r"remark:\s+(VGPRs|AGPRs|TotalSGPRs|LDS Size \[bytes/block\]|ScratchSize \[bytes/lane\]): (\d+)")
# fused_attention_kernel<D, kWpg, kCausal, kGroups, kList> in the Itanium mangling
_FUSED = re.compile(r"fused_attention_kernelILi(\d+)ELi(\d+)ELb([01])ELi(\d+)ELb([01])EE")
# (kWpg carries 16 more for two LDS stages per tensor)


def parse(remarks: str) -> list[dict]:
    """Resource records of every fused kernel instance in the text."""
    entries, current = [], None
    for line in remarks.splitlines():
        m = _NAME.search(line)
        if m:
            t = _FUSED.search(m.group(1))
            current = None
            if t:
                waves = int(t.group(2))
                current = {"head_dim": int(t.group(1)), "waves_per_group": waves % 16,
                           "causal": int(t.group(3)), "groups": int(t.group(4)), "list": int(t.group(5)),
                           "stages": 2 if waves >= 16 else 3}
                entries.append(current)
            continue
        f = _FIELD.search(line)
        if f and current is not None:
            key = {"VGPRs": "vgprs", "AGPRs": "agprs", "TotalSGPRs": "sgprs", "LDS Size [bytes/block]": "lds_bytes",
                   "ScratchSize [bytes/lane]": "scratch_bytes"}[f.group(1)]
            current[key] = int(f.group(2))
    fields = ("vgprs", "agprs", "sgprs", "lds_bytes", "scratch_bytes")
    return [e for e in entries if all(k in e for k in fields)]


def render(entries: list[dict]) -> str:
    rows = ",\n".join(
        "    {{{head_dim}, {waves_per_group}, {causal}, {groups}, {list}, {stages}, {vgprs}, {agprs}, {sgprs}, {lds_bytes}, "
        "{scratch_bytes}}}".format(**e) for e in sorted(entries, key=lambda e: (e["head_dim"], e["waves_per_group"],
                                                                               e["groups"], e["list"], e["stages"],
                                                                               e["causal"])))
    body = rows if rows else "    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}"
    return ("// Generated by cuda_fused_attention_amd/kernel_resources.py from the compiler's\n"
            "// resource report of csrc/fa_fused.hip. Do not edit.\n"
            "#include \"fa_resources.hpp\"\n\n"
            "namespace fa {\n\n"
            "const KernelResources kFusedKernelResources[] = {\n" + body + "\n};\n"
            f"const int kFusedKernelResourceCount = {len(entries)};\n\n"
            "}  // namespace fa\n")


def write(entries: list[dict], path: str) -> None:
    with open(path, "w") as fh:
        fh.write(render(entries))


def main(argv=None) -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--hipcc", required=True)
    ap.add_argument("--source", required=True)
    ap.add_argument("--out", required=True)
    ap.add_argument("flags", nargs="*")
    args = ap.parse_args(argv)
    cmd = [args.hipcc, *args.flags, "--cuda-device-only", "-c", "-x", "hip", args.source, "-o", "/dev/null",
           "-Rpass-analysis=kernel-resource-usage"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stderr)
        return proc.returncode
    entries = parse(proc.stderr)
    if not entries:
        sys.stderr.write("no fused_attention_kernel resource remarks found\n")
        return 1
    write(entries, args.out)
    return 0


if __name__ == "__main__":
    sys.exit(main())
