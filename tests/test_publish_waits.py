"""Kernels that publish their results from inside (to the host, or to the last
block of their own grid) have one thread write the word that others wait for.
A workgroup barrier does not wait for the other waves' stores on this target,
and a fence waits for its own wave's only, so every wave has to have waited for
its stores before the barrier in front of that word.  Read off the built
library's gfx950 code: from the publishing instruction back to the barriers
that come right before it, no path may reach one with a store still in flight."""
import os
import re
import subprocess

import pytest

from voxelmapplus_fastlio2_amd import build

LLVM = "/opt/rocm/llvm/bin"
STORE = re.compile(r"^(global|flat|buffer)_store_")
# the counted finish of a block, and a store past every cache
PUBLISH = re.compile(r"^global_atomic_add |^(global|flat)_store_dword .* sc0 sc1$")


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    lib = os.path.join(build.OUT, "libvmp.so")
    if not os.path.exists(lib):
        build.build_all()
    d = tmp_path_factory.mktemp("code")
    fat, co = str(d / "fat"), str(d / "co")
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", lib, os.devnull], check=True)
    subprocess.run(
        [f"{LLVM}/clang-offload-bundler", "--unbundle", "--type=o", f"--input={fat}", f"--output={co}",
         "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"],
        check=True,
    )
    return co


def kernels(co, name):
    """{symbol: [(address, text, branch target or None)]} of the kernels called `name`."""
    out = subprocess.run([f"{LLVM}/llvm-objdump", "-d", co], check=True, capture_output=True, text=True).stdout
    found, cur = {}, None
    mangled = re.compile(rf"{len(name)}{name}")
    for line in out.splitlines():
        m = re.match(r"^([0-9a-f]+) <(\w+)>:$", line)
        if m:
            base = int(m[1], 16)
            cur = found.setdefault(m[2], []) if mangled.search(m[2]) else None
            continue
        m = re.match(r"^\t(.*?)\s*// ([0-9A-F]{12}):[0-9A-F ]*(?:<\w+(?:\+0x([0-9a-f]+))?>)?$", line)
        if cur is not None and m:
            target = base + int(m[3] or "0", 16) if re.match(r"s_c?branch", m[1]) else None
            cur.append((int(m[2], 16), m[1].strip(), target))
    return found


def successors(ins):
    at = {a: i for i, (a, _, _) in enumerate(ins)}
    nxt = []
    for i, (_, text, target) in enumerate(ins):
        n = []
        if not text.startswith(("s_branch", "s_endpgm")) and i + 1 < len(ins):
            n.append(i + 1)
        if target is not None:
            n.append(at[target])
        nxt.append(n)
    return nxt


def barriers_with_stores_in_flight(ins):
    """(publishing instructions, those of the barriers right before them that
    a wave can reach without having waited for its stores)"""
    nxt = successors(ins)
    prev = [[] for _ in ins]
    for i, n in enumerate(nxt):
        for j in n:
            prev[j].append(i)
    # may a wave have stores in flight before instruction i
    flight = [False] * len(ins)
    work = list(range(len(ins)))
    while work:
        i = work.pop()
        text = ins[i][1]
        after = flight[i]
        if STORE.match(text):
            after = True
        elif text.startswith("s_waitcnt") and "vmcnt(0)" in text:
            after = False
        for j in nxt[i]:
            if after and not flight[j]:
                flight[j] = True
                work.append(j)
    publish = [i for i, (_, text, _) in enumerate(ins) if PUBLISH.match(text)]
    bad = set()
    for p in publish:
        seen, work = set(), list(prev[p])
        while work:
            i = work.pop()
            if i in seen:
                continue
            seen.add(i)
            if ins[i][1].startswith("s_barrier"):
                if flight[i]:
                    bad.add(i)
            else:
                work.extend(prev[i])
    return publish, sorted(bad)


@pytest.mark.parametrize("name", ["k_finish", "k_obs_reduce", "k_check_points"])
def test_results_for_the_host_are_stored_before_the_signal(code_object, name):
    found = kernels(code_object, name)
    assert found
    for symbol, ins in found.items():
        publish, bad = barriers_with_stores_in_flight(ins)
        assert publish, symbol
        assert not bad, (symbol, [hex(ins[i][0]) for i in bad])


@pytest.mark.parametrize("name", ["k_select1", "k_rs_pass", "k_spec_eval"])
def test_a_tile_is_stored_before_it_counts_itself_done(code_object, name):
    found = kernels(code_object, name)
    assert found
    for symbol, ins in found.items():
        publish, bad = barriers_with_stores_in_flight(ins)
        assert publish, symbol
        assert not bad, (symbol, [hex(ins[i][0]) for i in bad])
