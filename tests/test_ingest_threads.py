"""Load-time repack with its rows split over threads (CPU): shapes on either side of the split, rows that do not divide over
the threads, padded and unpadded contractions, into memory that holds other bytes before -- against the oracle."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import quant
from reinstinct_amd._lib import check, lib
from oracle import orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PTR = C.c_void_p
SHAPES = [(1024, 1), (1024, 2049), (1280, 1639), (256, 8193)]          # one thread; two, padded; two, not padded; two, one superblock a row


@pytest.mark.parametrize("fmt", [rein.Q4_0, rein.Q8_0, rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.IQ4_XS, rein.Q5_1, rein.IQ3_S])
@pytest.mark.parametrize("in_dim,out_dim", SHAPES)
def test_repack_writes_every_byte(fmt, in_dim, out_dim):
    raw = np.random.default_rng(fmt).integers(0, 256, in_dim * out_dim // orc.block_size(fmt) * orc.bytes_per_block(fmt), dtype=np.uint8)
    got = np.full(quant.repacked_len(fmt, in_dim, out_dim), 0xA5, np.uint8)
    check(lib.rein_repack_for_matvec(fmt, raw.ctypes.data_as(PTR), in_dim, out_dim, got.ctypes.data_as(PTR)))
    assert np.array_equal(got, orc.repack_for_matvec(fmt, raw, in_dim, out_dim))


@pytest.mark.parametrize("in_dim,out_dim", SHAPES)
def test_q3k_rows_are_the_transcoded_tensor(in_dim, out_dim):
    raw = np.random.default_rng(3).integers(0, 256, in_dim * out_dim // 256 * 110, dtype=np.uint8)
    slab, fmt = quant.ingest_for_matvec(quant.GGML_Q3_K, raw, in_dim, out_dim)
    assert fmt == rein.Q6_K
    assert np.array_equal(slab, orc.repack_for_matvec(rein.Q6_K, quant.transcode_q3_k_to_q6_k(raw, in_dim * out_dim), in_dim, out_dim))


@pytest.mark.parametrize("in_dim,out_dim", SHAPES + [(32 * 9, 8000)])
def test_bf16_rows_with_half_steps_and_extremes(in_dim, out_dim):
    g = np.random.default_rng(4)
    w = g.standard_normal(in_dim * out_dim).astype(np.float32)
    w[:32] = np.arange(32) * 4 + 0.5                    # with the 127 below: scale 1, half steps round away from zero
    w[31] = 127
    w[32:64] = 0
    w[64:96] = np.copysign(np.float32(1e-38), w[64:96])  # a subnormal scale has no finite reciprocal
    w[96:128] *= np.float32(1e38)
    bf = (w.view(np.uint32) >> 16).astype(np.uint16)
    slab, _ = quant.ingest_for_matvec(quant.GGML_BF16, bf.view(np.uint8), in_dim, out_dim)
    want = orc.repack_for_matvec(rein.Q8_0, orc.q8_0_quantize_from_f32(orc.bf16_to_f32(bf)), in_dim, out_dim)
    assert np.array_equal(slab, want)


def test_no_thread_to_be_had():
    """a process at its limits gets the same bytes from the calling thread alone (a child whose address space has no room for a
    thread's stack)"""
    code = ("import resource, numpy as np\n"
            "from reinstinct_amd import quant\n"
            "from reinstinct_amd._lib import lib\n"
            "raw = np.random.default_rng(1).integers(0, 256, 2048 * 2304 // 32 * 18, dtype=np.uint8)\n"
            "got = np.full(quant.repacked_len(2, 2048, 2304), 0xA5, np.uint8)\n"
            "args = (2, raw.ctypes.data, 2048, 2304, got.ctypes.data)\n"
            "size = int(open('/proc/self/statm').read().split()[0]) * resource.getpagesize()\n"
            "before = resource.getrlimit(resource.RLIMIT_AS)\n"
            "resource.setrlimit(resource.RLIMIT_AS, (size + (1 << 20), before[1]))\n"
            "rc = lib.rein_repack_for_matvec(*args)\n"
            "resource.setrlimit(resource.RLIMIT_AS, before)\n"
            "assert rc == 0 and np.array_equal(got, quant.repack_for_matvec(2, raw, 2048, 2304))\n"
            "print('same')\n")
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, cwd=ROOT)
    assert run.stdout.strip() == "same", (run.returncode, run.stderr[-500:])
