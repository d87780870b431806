"""The tile cull's early-exit flag as the compiler builds it (CPU only: hipcc
cross-compiles gfx950).

Every wave of a k_tile_cull block reads, after the last barrier of a batch of
candidates, whether some tile still takes lights, and leaves the batch loop by
that word.  A clear of the word for a later batch that no barrier separates
from those reads lets a late wave see the cleared word, leave alone and pair
its barriers with the others' wrongly.  This test compiles hl_cull.hip to LLVM
IR with the library's own flags and follows the control flow from every read
of the flag words: no store to them may be reached before a barrier.  A GPU
test runs several batches past tiles that never fill.
"""
import re
import shutil
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from helio_amd import abi, build, synth
from helio_amd.device import LightCullPass, upload_scene
from test_gpu_parity import check_tile_lists

SCALARS = {"i8": 1, "i16": 2, "i32": 4, "float": 4}
BARRIER = "@llvm.amdgcn.s.barrier("


@pytest.fixture(scope="module")
def cull_ir(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not shutil.which(hipcc):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("ir") / "hl_cull.ll"
    cmd = [hipcc, *build.HIPCC_FLAGS, "--cuda-device-only", "-S", "-emit-llvm",
           str(build.CSRC / "hl_cull.hip"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


def size_of(ir, t):
    if t in SCALARS:
        return SCALARS[t]
    if t.startswith("["):
        n, of = re.fullmatch(r"\[(\d+) x (.*)\]", t).groups()
        return int(n) * size_of(ir, of)
    body = re.search("^" + re.escape(t) + r" = type \{ (.*) \}$", ir, re.M).group(1)
    return sum(size_of(ir, f) for f in fields(body))


def fields(body):
    out, depth, cur = [], 0, ""
    for ch in body:
        depth += {"[": 1, "]": -1}.get(ch, 0)
        if ch == "," and depth == 0:
            out.append(cur.strip())
            cur = ""
        else:
            cur += ch
    return out + [cur.strip()]


def flag_range(ir, sm):
    """Byte range of the flag words in the block's LDS record: its only pair of words (every field before
    it is a multiple of its successors' alignment, so sizes add up)."""
    t = re.search("^" + re.escape(sm) + r" = .*addrspace\(3\) global (%\"[^\"]+\")", ir, re.M).group(1)
    at = 0
    found = []
    for f in fields(re.search("^" + re.escape(t) + r" = type \{ (.*) \}$", ir, re.M).group(1)):
        n = size_of(ir, f)
        if f == "[2 x i32]":
            found.append((at, at + n))
        at += n
    assert len(found) == 1
    return found[0]


def blocks_of(body):
    """{label: instructions}, the entry block first."""
    out, label = {"": []}, ""
    for line in body.splitlines()[1:-1]:
        m = re.match(r"^([\w.]+):", line)
        if m:
            label = m.group(1)
            out[label] = []
        elif line.strip():
            out[label].append(line.strip())
    return out


def flag_accesses(blocks, sm, lo, hi):
    """Places (block, index) of the reads and of the plain stores of the flag words."""
    const = re.escape(sm) + r", i32 (\d+)\)"
    flags = set()
    for ins in (i for b in blocks.values() for i in b):
        m = re.match(r"(%\S+) = getelementptr .*" + const, ins)
        if m and lo <= int(m.group(2)) < hi:
            flags.add(m.group(1))

    def hits(ins):
        m = re.search(const, ins)
        return (m and lo <= int(m.group(1)) < hi) or any(
            re.search(r"ptr addrspace\(3\) " + re.escape(f) + r"\b", ins) for f in flags)

    reads, stores = [], []
    for label, code in blocks.items():
        for k, ins in enumerate(code):
            if re.match(r"%\S+ = load ", ins) and hits(ins):
                reads.append((label, k))
            elif ins.startswith("store ") and hits(ins):
                stores.append((label, k))
    return reads, stores


def reached_before_barrier(blocks, start):
    seen, todo, out = set(), [start], []
    while todo:
        label, k = todo.pop()
        code = blocks[label]
        stopped = False
        while k < len(code):
            if BARRIER in code[k]:
                stopped = True
                break
            out.append((label, k))
            k += 1
        if stopped:
            continue
        for nxt in re.findall(r"label %([\w.]+)", " ".join(code)):
            if nxt not in seen:
                seen.add(nxt)
                todo.append((nxt, 0))
    return out


def test_no_flag_store_races_with_a_read(cull_ir):
    kernels = re.findall(r"^define [^\n]*@(_ZN2hl11k_tile_cull\S*?)\(.*?^}", cull_ir, re.M | re.S)
    assert len(kernels) == 2
    checked = {}
    for name in kernels:
        body = re.search(r"^define [^\n]*@" + re.escape(name) + r"\(.*?^}", cull_ir, re.M | re.S).group(0)
        sm = "@_ZZ" + name[2:] + "E2sm"
        lo, hi = flag_range(cull_ir, sm)
        blocks = blocks_of(body)
        reads, stores = flag_accesses(blocks, sm, lo, hi)
        assert stores, name
        for r in reads:
            bad = set(reached_before_barrier(blocks, (r[0], r[1] + 1))) & set(stores)
            assert not bad, f"{name}: a store to the flag words without a barrier after their read: {bad}"
        checked[name] = len(reads)
    assert any("j16384" in k and v for k, v in checked.items()), checked


@pytest.mark.gpu
def test_batches_past_tiles_that_never_fill(ctx):
    """1500 small lights in one super-tile of 8 x 8 tiles: three batches of candidates, tiles that are full
    after the first one beside tiles that never fill."""
    sc = synth.make_scene("c2_1080p_1k", width=3850, height=2170, num_lights=1500)
    rng = np.random.default_rng(5)
    sc.lights["light_type"] = abi.HL_LIGHT_POINT
    sc.lights["position_range"][:, :3] = np.array((0.45, 2.3, 0.0)) + rng.normal(0, 0.15, (1500, 3))
    sc.lights["position_range"][:, 3] = 0.05
    ol, oc = O.cull_tiles(sc)
    tiles = np.zeros((136, 248), np.uint32)
    tiles[:, :241] = oc.reshape(136, 241)
    supers = tiles.reshape(17, 8, 31, 8)
    full = (supers == 64).any(axis=(1, 3))
    assert (full & (supers < 64).any(axis=(1, 3))).any() and full.sum() == 1
    print("[tile flag] 3850x2170, 1500 lights in one super-tile", flush=True)
    ds = upload_scene(ctx, sc)
    cull = LightCullPass(ctx, sc.width, sc.height)
    cull.prepare(ds)
    for _ in range(2):  # the second call meets the first one's scratch
        cull.tiles.lists.fill_u32(0xFFFFFFFF)
        cull.execute(ds)
    check_tile_lists(cull.tiles.lists.download(np.uint32).reshape(-1, 64), cull.tiles.counts.download(np.uint32),
                     ol, oc)
