"""Build-time guard of the register budgets the kernels' speed depends on (CPU only: hipcc cross-compiles for gfx950).

The d = 64 kernels are tuned to the register counts at which one more wave fits a SIMD (128 VGPRs: four waves, 168: three).
One extra live register in a main loop silently costs a wave per SIMD or turns into scratch traffic, so the counts the
compiler reports (-Rpass-analysis=kernel-resource-usage) are pinned here for the variants the headline workloads run.
"""
import os
import re
import subprocess
import sys
import threading
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "flash-attention_amd"))
import build as fa_build  # noqa: E402


_UNITS = ["fa_%s_d%d.hip" % (w, d) for w in ("bwd", "fwd") for d in (128, 64, 32, 16)] + ["fa_bwd_fused.hip", "fa_decode.hip"]
_pool, _compiled, _compiled_lock = ThreadPoolExecutor(8), {}, threading.Lock()


def _resources(src):
    """What the compiler reports of a unit's kernels.  Units take up to two minutes: the first call asks for all of them, unless other processes do, too."""
    with _compiled_lock:
        for unit in [src] + (_UNITS if "PYTEST_XDIST_WORKER" not in os.environ else []):
            if unit not in _compiled:
                _compiled[unit] = _pool.submit(_compile, unit)
    return _compiled[src].result()


def _compile(src):
    cmd = [fa_build.HIPCC] + fa_build.FLAGS + ["-Rpass-analysis=kernel-resource-usage", "-c",
                                               os.path.join(fa_build.CSRC, src), "-o", os.devnull]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    out, name = {}, None
    for line in r.stdout.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            out[name] = {}
            continue
        m = re.search(r"remark:\s+([A-Za-z ]+?)(?: \[[^\]]*\])?: (\d+)", line)
        if m and name:
            out[name][m.group(1).strip()] = int(m.group(2))
    return out


def _pick(res, *parts):
    hits = [v for k, v in res.items() if all(p in k for p in parts)]
    assert len(hits) == 1, (parts, [k for k in res if parts[0] in k])
    return hits[0]


@pytest.mark.timeout(600)
def test_d64_kernels_keep_their_waves_per_simd():
    fwd = _resources("fa_fwd_d64.hip")
    bwd = _resources("fa_bwd_d64.hip")
    # <f16, 64, ..., causal, dropout, sparse, alibi, key split> mangled as ...IDF16_Li64E...Lb{0,1}E x3, Li{0,1,2}E for the score bias, Li{1,2}E
    # (the dK/dV kernel has no key-split parameter)
    plain, causal, dropout = "Lb0ELb0ELb0ELi0E", "Lb1ELb0ELb0ELi0E", "Lb0ELb1ELb0ELi0E"
    full = "Li1EEEv"
    # (the forward's last parameter: the dropout variant that also leaves its keep decisions for the backward)
    for flags, want in ((plain, 4), (causal, 4), (dropout, 3)):
        k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", flags + "Li1ELb0EEEv")
        # (the plain variant parks one register pair in scratch across its main loop: stored before, reloaded after)
        assert k["Occupancy"] >= want and k["VGPRs Spill"] <= (2 if flags == plain else 0), ("forward", flags, k)
        k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", flags + "Li2ELb0EEEv")  # half-size tiles
        assert k["Occupancy"] >= 4 and k["VGPRs Spill"] == 0, ("forward, key split", flags, k)
    k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", dropout + "Li1ELb1EEEv")
    assert k["Occupancy"] >= 3 and k["VGPRs Spill"] == 0, ("forward, keep words", k)
    k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", dropout + "Li2ELb1EEEv")
    # (scalar registers that do not fit are parked in lanes of a vector register, outside the main loop: a handful is fine)
    assert k["Occupancy"] >= 4 and k["VGPRs Spill"] == 0 and k["SGPRs Spill"] <= 8, ("forward, keep words, key split", k)
    # backward kernels: <..., causal, dropout mode (0 none, 1 drawn with Philox, 2 read from the forward's keep words),
    # sparse, alibi, ...>
    bplain, bcausal, bdrawn, bread = "Lb0ELi0ELb0ELi0E", "Lb1ELi0ELb0ELi0E", "Lb0ELi1ELb0ELi0E", "Lb0ELi2ELb0ELi0E"
    for flags, want in ((bplain, 3), (bcausal, 3), (bdrawn, 3), (bread, 3)):
        k = _pick(bwd, "fa_bwd_dq_kernelIDF16_Li64E", flags + full)
        assert k["Occupancy"] >= want and k["VGPRs Spill"] == 0, ("dq", flags, k)
        k = _pick(bwd, "fa_bwd_dq_kernelIDF16_Li64E", flags + "Li2EEEv")
        assert k["Occupancy"] >= 3 and k["VGPRs Spill"] == 0, ("dq, key split", flags, k)
    for flags, want, spill in ((bplain, 3, 2), (bcausal, 3, 2), (bdrawn, 2, 0), (bread, 2, 0)):
        k = _pick(bwd, "fa_bwd_dkdv_kernelIDF16_Li64E", flags + "Lb0EEEv")  # (last flag: the variant that turns dK back, rotary)
        assert k["Occupancy"] >= want and k["VGPRs Spill"] <= spill, ("dkdv", flags, k)
    # the ALiBi variants (fourth flag set) keep the waves per SIMD of their plain counterparts in the backward
    for flags, bflags in (("Lb0ELb0ELb0ELi1E", "Lb0ELi0ELb0ELi1E"), ("Lb1ELb0ELb0ELi1E", "Lb1ELi0ELb0ELi1E")):
        assert _pick(fwd, "fa_fwd_kernelIDF16_Li64E", flags + "Li1ELb0EEEv")["Occupancy"] >= 3, flags  # (the bias costs the fourth)
        assert _pick(bwd, "fa_bwd_dq_kernelIDF16_Li64E", bflags + full)["Occupancy"] >= 3, bflags
        k = _pick(bwd, "fa_bwd_dkdv_kernelIDF16_Li64E", bflags + "Lb0EEEv")
        assert k["Occupancy"] >= 3 and k["VGPRs Spill"] <= 4, (bflags, k)


@pytest.mark.timeout(600)
def test_d64_bias_tensor_and_one_kernel_backward_variants():
    """The variants that read a bias tensor run at three (forward without dropout) and two waves per SIMD; the dK/dV variant
    that also draws dropout decisions is at the register limit and may spill a few registers, the others must not.  The
    one-kernel backward runs two workgroups per compute unit: two waves per SIMD, nothing spilled, at most 80 KB of LDS."""
    fwd = _resources("fa_fwd_d64.hip")
    bwd = _resources("fa_bwd_d64.hip")
    for causal in ("Lb0E", "Lb1E"):
        k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", causal + "Lb0ELb0ELi2ELi1ELb0EEEv")
        assert k["Occupancy"] >= 3 and k["VGPRs Spill"] <= 3, ("forward, bias tensor", causal, k)
        for drop, words in (("Lb1E", "Lb0E"), ("Lb1E", "Lb1E")):
            k = _pick(fwd, "fa_fwd_kernelIDF16_Li64E", causal + drop + "Lb0ELi2ELi1E" + words + "EEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0, ("forward, bias tensor, dropout", causal, words, k)
        for drop, spill in (("Li0E", 0), ("Li2E", 4), ("Li1E", 16)):
            k = _pick(bwd, "fa_bwd_dq_kernelIDF16_Li64E", causal + drop + "Lb0ELi2ELi1EEEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0, ("dq, bias tensor", causal, drop, k)
            k = _pick(bwd, "fa_bwd_dkdv_kernelIDF16_Li64E", causal + drop + "Lb0ELi2ELb0EEEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] <= spill, ("dkdv, bias tensor", causal, drop, k)
    # dQ and dK/dV in one launch (short launches): the register count of the dK/dV part, two waves per SIMD, nothing spilled
    for dt in ("IDF16_", "IDF16b"):
        for flags in ("Lb0ELi0E", "Lb0ELi2E", "Lb1ELi0E", "Lb1ELi2E"):
            k = _pick(bwd, "fa_bwd_merged_kernel" + dt, flags + "EEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 80 * 1024, ("merged backward", dt, flags, k)
    fused = _resources("fa_bwd_fused.hip")
    for dt in ("IDF16_", "IDF16b"):
        k = _pick(fused, "fa_bwd_fused_kernel%sLi64ELi0E" % dt)
        assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 80 * 1024, ("one-kernel backward", dt, k)


@pytest.mark.timeout(600)
def test_d128_backward_keeps_two_waves_per_simd():
    """d = 128: the dK/dV kernel holds its V tile in LDS so that K, the two accumulators and the scores fit 256 registers
    (two waves per SIMD, nothing spilled: a spill's scratch load would wait behind the tile prefetch on every step)."""
    bwd = _resources("fa_bwd_d128.hip")
    for dt in ("IDF16_", "IDF16b"):
        # plain, causal, both with a block layout, and the two without that read the dropout decisions from keep words
        for flags in ("Lb0ELi0ELb0ELi0E", "Lb1ELi0ELb0ELi0E", "Lb0ELi0ELb1ELi0E", "Lb1ELi0ELb1ELi0E", "Lb0ELi2ELb0ELi0E",
                      "Lb1ELi2ELb0ELi0E"):
            k = _pick(bwd, "fa_bwd_dkdv_kernel%sLi128E" % dt, flags + "Lb0EEEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 80 * 1024, (dt, flags, k)
            k = _pick(bwd, "fa_bwd_dq_kernel%sLi128E" % dt, flags + "Li1EEEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] <= (1 if "Lb1ELi0E" in flags[8:] else 0), ("dq", dt, flags, k)
        # the dK/dV kernel of wave pairs (launch policy 0x40) is built for three waves per SIMD and three workgroups' LDS
        for flags in ("Lb0ELb0E", "Lb1ELb0E", "Lb0ELb1E", "Lb1ELb1E"):
            k = _pick(bwd, "fa_bwd_dkdv_pair_kernel%s" % dt, flags + "EEv")
            assert k["Occupancy"] >= 3 and k["VGPRs Spill"] <= 2 and k["LDS Size"] <= 160 * 1024 // 3, (dt, flags, k)


@pytest.mark.timeout(600)
def test_forward_and_decode_variants_keep_their_waves_per_simd():
    """The forward at every head dimension but the headline's, over block layouts, with ALiBi and with dropout, the dQ variants that
    draw dropout decisions, and the decode kernel: (waves per SIMD at least, spilled registers at most) of each."""
    with ThreadPoolExecutor(6) as ex:
        d16, d32, d64, d128, dec, bwd = ex.map(_resources, ("fa_fwd_d16.hip", "fa_fwd_d32.hip", "fa_fwd_d64.hip", "fa_fwd_d128.hip",
                                                            "fa_decode.hip", "fa_bwd_d64.hip"))
    T, F = "Lb1E", "Lb0E"

    def flags(causal, dropout, sparse, bias, ks=1, words=F):
        return causal + dropout + sparse + "Li%dELi%dE" % (bias, ks) + words + "EEv"

    for dt in ("IDF16_", "IDF16b"):
        for causal in (F, T):
            for what, res, d, variant, waves, spills in (
                    ("plain", d128, 128, flags(causal, F, F, 0), 3, 0),
                    ("block layout", d128, 128, flags(causal, F, T, 0), 3, 2 if causal == F else 0),
                    ("block layout", d64, 64, flags(causal, F, T, 0), 4, 8 if causal == F else 5),
                    ("block layout", d16, 16, flags(causal, F, T, 0), 5, 0),
                    ("ALiBi", d16, 16, flags(F, F, F, 1), 4, 0),
                    ("dropout, half-size", d16, 16, flags(causal, T, F, 0, 2), 6, 0),
                    ("dropout, block layout", d32, 32, flags(causal, T, T, 0), 4, 0),
                    ("dropout, block layout, ALiBi", d32, 32, flags(causal, T, T, 1), 3, 0)):
                k = _pick(res, "fa_fwd_kernel%sLi%dELi%dELb0E" % (dt, d, 32 if d == 128 else 64), variant)
                assert k["Occupancy"] >= waves and k["VGPRs Spill"] <= spills, (what, d, dt, causal, k)
            k = _pick(d128, "fa_fwd_kernel%sLi128ELi32ELb1E" % dt, flags(causal, F, F, 0))  # launches short of workgroups
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0, ("roomy", dt, causal, k)
            for sparse, alibi, spills in ((F, 0, 0), (F, 1, 0), (T, 0, 1), (T, 1, 3)):
                k = _pick(bwd, "fa_bwd_dq_kernel%sLi64E" % dt, causal + "Li1E" + sparse + "Li%dELi1EEEv" % alibi)
                assert k["Occupancy"] >= 3 and k["VGPRs Spill"] <= spills, ("dq, drawn dropout", dt, causal, sparse, alibi, k)
        for d in (16, 32, 64, 128):  # two workgroups of two waves (64 KB of tiles at d = 128) on a compute unit need one per SIMD
            k = _pick(dec, "fa_decode_kernel%sLi%dE" % (dt, d))
            assert k["Occupancy"] >= 1 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 64 * 1024 + 64, ("decode", dt, d, k)


@pytest.mark.timeout(600)
def test_key_words_of_the_dropout_forward_only_where_they_pay():
    """The Philox key words kept in LDS (1 KB of LDS, dense dropout forward): in the full-size tiles of d = 32 and 64, not in the half-size ones nor
    where a causal mask's keep words are left, which they slow down; (waves per SIMD at least) of the variants, and no vector register spilled."""
    with ThreadPoolExecutor(2) as ex:
        d32, d64 = ex.map(_resources, ("fa_fwd_d32.hip", "fa_fwd_d64.hip"))
    for dt in ("IDF16_", "IDF16b"):
        for causal in ("Lb0E", "Lb1E"):
            for words in ("Lb0E", "Lb1E"):
                for res, d, waves in ((d32, 32, 3), (d64, 64, 3)):
                    name = "fa_fwd_kernel%sLi%dELi64ELb0E" % (dt, d)
                    full = _pick(res, name, causal + "Lb1ELb0ELi0ELi1E" + words + "EEv")
                    half = _pick(res, name, causal + "Lb1ELb0ELi0ELi2E" + words + "EEv")
                    tiles = 64 * d * 2 * 4  # two K and two V tiles of 64 keys
                    key_words = 0 if causal == "Lb1E" and words == "Lb1E" else 1024
                    assert full["Occupancy"] >= waves and full["VGPRs Spill"] == 0 and full["LDS Size"] == tiles + key_words, (dt, d, causal, words, full)
                    assert half["Occupancy"] >= 4 and half["VGPRs Spill"] == 0 and half["LDS Size"] == tiles, (dt, d, causal, words, half)


@pytest.mark.timeout(600)
def test_padded_rows_and_d128_half_size_variants_keep_their_waves_per_simd():
    """The forward over a padded batch (three as score-bias parameter) keeps the waves per SIMD of the dense variant it is bounded like, nothing in
    scratch; the half-size tiles of d = 128, forward and dQ, run two waves per SIMD and two workgroups' LDS on a compute unit."""
    with ThreadPoolExecutor(5) as ex:
        d16, d32, d64, d128, bwd = ex.map(_resources, ("fa_fwd_d16.hip", "fa_fwd_d32.hip", "fa_fwd_d64.hip", "fa_fwd_d128.hip", "fa_bwd_d128.hip"))
    for dt in ("IDF16_", "IDF16b"):
        for causal in ("Lb0E", "Lb1E"):
            rows, dense = causal + "Lb0ELb0ELi3ELi%dELb0EEEv", causal + "Lb0ELb0ELi0ELi2ELb0EEEv"
            for res, d, bn, roomy, ks, waves in ((d16, 16, 64, 0, 1, 5), (d16, 16, 64, 0, 2, 7), (d32, 32, 64, 0, 1, 4), (d32, 32, 64, 0, 2, 6),
                                                 (d64, 64, 64, 0, 1, 4), (d64, 64, 64, 0, 2, 4), (d128, 128, 32, 0, 1, 3), (d128, 128, 32, 1, 1, 2),
                                                 (d128, 128, 64, 0, 2, 2)):
                k = _pick(res, "fa_fwd_kernel%sLi%dELi%dELb%dE" % (dt, d, bn, roomy), rows % ks)
                assert k["Occupancy"] >= waves and k["VGPRs Spill"] == 0, ("padded rows", d, dt, causal, roomy, ks, k)
            k = _pick(d128, "fa_fwd_kernel%sLi128ELi64ELb0E" % dt, dense)
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 80 * 1024, ("forward, half-size", dt, causal, k)
            k = _pick(bwd, "fa_bwd_dq_kernel%sLi128E" % dt, causal + "Li0ELb0ELi0ELi2EEEv")
            assert k["Occupancy"] >= 2 and k["VGPRs Spill"] == 0 and k["LDS Size"] <= 80 * 1024, ("dq, half-size", dt, causal, k)


@pytest.mark.timeout(600)
def test_block_layout_dkdv_keeps_its_block_list_in_registers():
    """dK/dV over a block layout at d = 16, whose tiles gather four 16-row blocks: the list is neither in scratch nor in LDS beside the tiles."""
    bwd = _resources("fa_bwd_d16.hip")
    for dt in ("IDF16_", "IDF16b"):
        for causal in ("Lb0E", "Lb1E"):
            for drop in ("Li0E", "Li1E"):
                lds = []
                for bias in ("Li0E", "Li1E", "Li2E"):
                    k = _pick(bwd, "fa_bwd_dkdv_kernel%sLi16E" % dt, "Li16E" + causal + drop + "Lb1E" + bias + "Lb0EEEv")
                    assert k["ScratchSize"] == 0, (dt, causal, drop, bias, k)
                    lds.append(k["LDS Size"])
                # two buffers of 64 rows of Q and dO, 16 elements of 2 bytes, and the rows' statistics, and less than the list's 32 bytes a thread more
                assert lds[0] == lds[1] < 2 * 64 * (2 * 16 * 2 + 2 * 4) + 256 * 32 and lds[2] > lds[0], (dt, causal, drop, lds)


@pytest.mark.timeout(600)
def test_live_order_variants_are_bounded_like_the_slot_order():
    """The kernels whose workgroups enumerate the tiles that hold rows keep the waves per SIMD of the same variant in the slot order and put at most
    two registers more in scratch (the first step over the keys peeled off the loop took 20 to 50); at d = 16 dQ with a bias under a causal mask takes two
    registers more than its waves allow.  The merged causal backward, which has no such variant, does not carry its code: few of its scalars are parked."""
    units = ["fa_fwd_d64.hip", "fa_fwd_d128.hip", "fa_fwd_d16.hip", "fa_bwd_d64.hip", "fa_bwd_d128.hip", "fa_bwd_d16.hip"]
    with ThreadPoolExecutor(6) as ex:
        all_res = dict(zip(units, ex.map(_resources, units)))
    pairs = 0
    for unit, res in all_res.items():
        for name, k in res.items():
            if "_live_kernel" not in name:
                continue
            m = re.match(r"_ZN2fa\d+fa_(fwd|bwd_dq|bwd_dkdv|bwd_merged)_live_kernelI(.*)EEEvNS", name)
            kind, args = m.group(1), m.group(2)
            if kind == "bwd_dq":
                args = re.sub(r"^(\w+?Li\d+ELi\d+ELb[01]ELi\d)E(Li\dELi\d)$", r"\1ELb0E\2", args)
            elif kind == "bwd_dkdv":
                args = re.sub(r"^(\w+?Li\d+ELb[01]ELi\d)E(Li\dELb[01])$", r"\1ELb0E\2", args)
            elif kind == "bwd_merged":
                args = re.sub(r"Li", "Lb0ELi", args, count=1)
            slot = _pick(res, "fa_%s_kernelI%sEEEv" % (kind, args))
            waves = slot["Occupancy"] - (1 if kind == "bwd_dq" and re.search(r"Li16ELi64ELb1ELi0ELb0ELi[12]E", args) else 0)
            assert k["Occupancy"] >= waves and k["VGPRs Spill"] <= slot["VGPRs Spill"] + 2 and k["LDS Size"] == slot["LDS Size"], (unit, name, k, slot)
            pairs += 1
    assert pairs > 200, pairs
    for dt in ("IDF16_", "IDF16b"):
        for drop in ("Li0E", "Li2E"):
            k = _pick(all_res["fa_bwd_d64.hip"], "fa_bwd_merged_kernel" + dt, "Lb1E" + drop + "EEv")
            assert k["VGPRs Spill"] == 0 and k["SGPRs Spill"] <= 20, ("merged causal", dt, drop, k)


@pytest.mark.timeout(600)
def test_small_head_dkdv_variants_keep_four_waves():
    """dK/dV over a block layout at d = 16: four waves per SIMD without dropout, as with ALiBi; the LDS of all its variants is two buffers of a pair of 64 x 16
    tiles, 64 bytes that the wider transposed reads run past a row and the rows' statistics, with a bias tensor 4 KB a wave more and nothing for
    the block list (2 KB or more wherever it was).  With keep words and rotary at d = 32: four waves."""
    with ThreadPoolExecutor(2) as ex:
        d16, d32 = ex.map(_resources, ("fa_bwd_d16.hip", "fa_bwd_d32.hip"))
    tiles = 2 * 2 * 64 * 16 * 2 + 64 + 2 * 2 * 64 * 4
    for dt in ("IDF16_", "IDF16b"):
        for causal in ("Lb0E", "Lb1E"):
            for bias, waves in (("Li0E", 4), ("Li1E", 4), ("Li2E", 3)):
                for drop in ("Li0E", "Li1E"):
                    k = _pick(d16, "fa_bwd_dkdv_kernel%sLi16E" % dt, "Li16E" + causal + drop + "Lb1E" + bias + "Lb0EEEv")
                    assert k["LDS Size"] == tiles + (4 * 64 * 32 * 2 if bias == "Li2E" else 0), (dt, causal, drop, bias, k)
                    if drop == "Li0E":
                        assert k["Occupancy"] >= waves and k["VGPRs Spill"] == 0, (dt, causal, bias, k)
        for name, flags in (("fa_bwd_dkdv_kernel%sLi32E", "Lb0ELi2ELb0ELi0ELb1EEEv"), ("fa_bwd_dkdv_live_kernel%sLi32E", "Lb0ELi2ELi0ELb1EEEv")):
            k = _pick(d32, name % dt, flags)
            assert k["Occupancy"] >= 4 and k["VGPRs Spill"] == 0, (name, dt, k)
