"""Waves per SIMD of the forward sweeps that share the chip.

A batch's width buckets run side by side on streams of their own.  The FP32
widths 9..16 leave room for a wave of the next bucket: seven waves a SIMD, by
scalar registers, of 64 vector registers each (512 a SIMD), so that what one
of them frees and the unused 64 hold a wave of widths 17..24."""

import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _kernels(name):
    path = os.path.join(ROOT, "piquasso_amd", "lib", "obj", name)
    if not os.path.exists(path):
        pytest.skip("no resource records (library not built by piquasso_amd/csrc/Makefile)")
    out, cur = {}, None
    for line in open(path):
        key, _, value = line.partition(":")
        if key == "Function Name":
            cur = out.setdefault(value.strip(), {})
        else:
            cur[key.split(" [")[0].strip()] = int(value)
    return out


def _static(name):
    (res,) = [r for k, r in _kernels(name).items() if "perm_static_kernel" in k]
    return res


def test_a_wave_of_the_next_width_fits_beside_the_fp32_widths_9_to_16():
    here, next_ = _static("perm_fwd_b1_v2.o.res"), _static("perm_fwd_b2_v2.o.res")
    held = -(-here["VGPRs"] // 8) * 8
    assert here["Occupancy"] == 7
    # one of them ends: its registers and those no wave holds are enough
    assert held + 512 - here["Occupancy"] * held >= -(-next_["VGPRs"] // 8) * 8
