"""CPU test of the K-split projections' exchange of operands between the lanes of a wave
through LDS (engine-mlx_amd/csrc/qgemm_ks.hip): between a lane's writes to a slot and its reads
of what other lanes wrote there, the source must order the two for the compiler
(wave_lds_fence). The hardware keeps a wave's LDS operations in order, so a missing fence shows
in no run until a compiler tells the two addresses apart; it is looked for in the source."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "engine-mlx_amd", "csrc")


def source(name):
    text = open(os.path.join(CSRC, name)).read()
    return re.sub(r"//[^\n]*", "", text)


def events(body):
    """The kernel's slot accesses and fences in source order: 'w', 'r' and 'f'."""
    found = []
    for m in re.finditer(r"wave_lds_fence\(\)|reinterpret_cast<(const )?u32x4\*>\(sl \+", body):
        found.append("f" if m.group(0).startswith("wave") else "r" if m.group(1) else "w")
    return found


def kernels():
    text = source("qgemm_ks.hip")
    for name in ("qgemm_ks_kernel", "qmv_ks_kernel"):
        start = text.index(f"void {name}(")
        yield name, text[start:text.index("\n}\n", start)]


def test_every_exchange_through_a_slot_is_fenced():
    for name, body in kernels():
        ev = events(body)
        # 4-bit weights, 8-bit weights, x
        assert ev.count("r") == 3, (name, ev)
        for i, e in enumerate(ev):
            if e == "r":
                assert ev[i - 1] == "f" and ev[i - 2] == "w", f"{name}: slot read without a fence after the write: {ev}"


def test_a_slot_is_reused_behind_a_fence():
    """A slot is written again kSlots exchanges later, so with two or more slots the fence of
    another exchange lies between its read and that write."""
    assert int(re.search(r"kSlots = (\d+)", source("qgemm_ks.hip")).group(1)) >= 2


def test_the_fence_orders_memory_and_lanes():
    text = source("qmatmul_common.hpp")
    start = text.index("void wave_lds_fence()")
    body = text[start:text.index("\n}\n", start)]
    calls = re.findall(r"__builtin_amdgcn_\w+\([^)]*\)", body)
    assert calls == ['__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront")', "__builtin_amdgcn_wave_barrier()",
                     '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront")'], calls
