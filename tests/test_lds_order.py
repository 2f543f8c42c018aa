"""Lanes of a wave that exchange data through LDS without a workgroup barrier: the
hardware keeps a wave's LDS accesses in order, the compiler only where it is told to
(wave_phase, stride_amd/csrc/tc_common.hpp). A race of this kind does not show in
results until a compiler reorders, so the source is checked (CPU)."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stride_amd", "csrc")


def source(name):
    """The file without comments."""
    return re.sub(r"//[^\n]*", "", open(os.path.join(CSRC, name)).read())


def test_matrix_gemm_weight_slot():
    """sum() stores this lane's pieces of the slot, reads other lanes' in slot_step, and
    the next call overwrites them: stores, phase, reads, phase."""
    text = source("exact.hip")
    body = text[text.index("auto sum = [&](const Batch& B"):text.index("constexpr int kTurns")]
    kinds = re.findall(r"(aw\[wave\]\[[^;]*\] = )|(slot_step\()|(wave_phase\(\))", body)
    order = "".join("s" if store else "r" if read else "p" for store, read, _ in kinds)
    assert re.fullmatch(r"s+pr+p", order), order


def test_wave_phase_orders_lds():
    text = source("tc_common.hpp")
    body = text[text.index("void wave_phase() {"):]
    body = body[:body.index("}")]
    assert re.search(r'fence\(__ATOMIC_RELEASE, "wavefront", "local"\).*wave_barrier\(\).*'
                     r'fence\(__ATOMIC_ACQUIRE, "wavefront", "local"\)', body, re.S)


def test_attention_tile_tail_weights():
    """The tile kernel's last positions: lanes store their weights in the wave's wb and
    read other lanes' (each turn of the loop overwrites them)."""
    text = source("tc_aux.hip")
    body = text[text.index("for (int c0 = 4 * whole_steps;"):]
    body = body[:body.index("auto record =")]
    kinds = re.findall(r"(wb\[wave\]\[[^;]*\] = )|(&wb\[wave\])|(wave_phase\(\))", body)
    order = "".join("s" if store else "r" if read else "p" for store, read, _ in kinds)
    assert order == "pspr", order
