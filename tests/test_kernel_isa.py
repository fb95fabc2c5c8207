"""A property of the built kernels that neither the source nor a run shows: libfrhip.so's code objects, taken apart."""
import os
import re
import shutil
import struct
import subprocess

import pytest

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(HERE, "faster-rwkv_amd", "libfrhip.so")
OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin") or shutil.which("llvm-objdump")


def code_objects(data):
    """The gfx950 code objects of the offload bundles in a library"""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", -1
    while (at := data.find(magic, at + 1)) >= 0:
        n, pos = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            offset, size, length = struct.unpack_from("<3Q", data, pos)
            target = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in target and size:
                yield data[at + offset:at + offset + size]


def functions(listing):
    """name -> [(address, instruction text, 16-bit branch offset)]"""
    out, body = {}, None
    for line in listing.splitlines():
        head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if head:
            body = out.setdefault(head.group(1), [])
            continue
        m = re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+): ([0-9A-F]{8})", line)
        if m and body is not None:
            offset = int(m.group(3), 16) & 0xffff
            body.append((int(m.group(2), 16), m.group(1), offset - 0x10000 if offset & 0x8000 else offset))
    return out


def reads_outstanding_at_barriers(body):
    """Addresses of barriers that some path reaches with an LDS read issued and not waited for.  LDS answers a wave in order, so lgkmcnt(n)
    leaves at most the last n accesses outstanding.  The state: which of the last 64 accesses, bit 0 the last one, can be such a read."""
    place = {addr: i for i, (addr, _, _) in enumerate(body)}
    state, work, found = {0: 0}, [0], set()
    while work:
        i = work.pop()
        mask = state[i]
        addr, text, offset = body[i]
        op = text.split()[0]
        if op.startswith("ds_"):
            mask = (mask << 1 | op.startswith("ds_read")) & (1 << 64) - 1
        wait = re.search(r"lgkmcnt\((\d+)\)", text)
        if wait:
            mask &= (1 << int(wait.group(1))) - 1
        elif op == "s_waitcnt" and "cnt" not in text.split(None, 1)[1]:
            mask = 0  # printed as a plain 0: all counters
        if op == "s_barrier" and mask:
            found.add(addr)
        follow = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if op == "s_branch" or op.startswith("s_cbranch"):
            follow.append(place[addr + 4 + 4 * offset])
        for j in follow:
            if j < len(body) and (j not in state or state[j] | mask != state[j]):
                state[j] = state.get(j, 0) | mask
                work.append(j)
    return found


@pytest.mark.parametrize("n,barriers", [(0, set()), (1, set()), (2, {0})])
def test_the_analysis_finds_a_read_that_is_not_waited_for(n, barriers):
    """A loop over a barrier, a read, a write and lgkmcnt(n)"""
    assert reads_outstanding_at_barriers([(0, "s_barrier", 0), (4, "ds_read_b128 v[0:3], v8", 0), (12, "ds_write_b32 v9, v8", 0),
                                          (20, "s_waitcnt lgkmcnt(%d)" % n, 0), (24, "s_cbranch_scc1 65529", -7), (28, "s_endpgm", 0)]) == barriers


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_no_fragment_read_is_outstanding_at_a_barrier(tmp_path):
    """The product kernels' MFMA waves meet the waves that load at bare barriers, behind which the LDS that they have read is written again.
    Their reads have to be complete there.  The compiler waits for them ahead of the MFMAs that take them, which stand ahead of the barrier; a
    wait of its own there made uint8 products up to 2.4 % slower (0.3 % on average), so what it built is checked instead."""
    seen = {}
    for i, obj in enumerate(code_objects(open(LIB, "rb").read())):
        if b"gemm_ring_kernel" not in obj and b"gemm_q8_kernel" not in obj and b"gemm_vw_kernel" not in obj:
            continue
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(obj)
        listing = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(path)], capture_output=True, text=True, check=True).stdout
        for name, body in functions(listing).items():
            kind = re.search(r"gemm_(ring|q8|vw|vw256)_kernel", name)
            if kind:
                assert any(t == "s_barrier" for _, t, _ in body) and any("mfma" in t for _, t, _ in body), name
                seen[name] = kind.group(1)
                assert not reads_outstanding_at_barriers(body), name
    assert sorted(set(seen.values())) == ["q8", "ring", "vw", "vw256"], seen
