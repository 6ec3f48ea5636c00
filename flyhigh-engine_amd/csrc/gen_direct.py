"""Generates the instantiation table of the direct conv kernel (direct_impl.h).

Writes direct_table.h (the host-visible list of configurations; a configuration's index + 128 is its variant code)
and direct_<group>.hip (the instantiations, one translation unit per group so they compile in parallel).
Run after changing the list below:  python gen_direct.py
"""
import os

HERE = os.path.dirname(os.path.abspath(__file__))


def regs(ks, s, cin32, fm, wm, wn, na, wk):
    """Rough register need of one wave, (VGPRs, accumulators): resident weights, two LDS operand sets, the halo
    staging, bias/slope, addressing; the accumulators may live in AGPRs."""
    kw = ks * ks * (cin32 // 32) // wk
    th = fm * wm
    nld = -(-(((th - 1) * s + ks) * (15 * s + ks) * (cin32 // 8)) // (64 * wm * wn * wk))
    return 4 * kw * na + 8 * fm + 4 * nld + 40 + 8 * na, 4 * fm * na


def lds(ks, s, cin32, th, threads):
    """LDS bytes: the halo, padded to whole staging rounds of 8-channel groups"""
    ih, iw = (th - 1) * s + ks, 15 * s + ks
    groups = ih * iw * (cin32 // 8)
    rounds = -(-groups // threads)
    return -(-(rounds * threads) // (cin32 // 8)) * (cin32 + 8) * 2


# configurations the estimate admits but the compiler spills (kernel-resource-usage remarks of hipcc):
# (ks, stride, cin32, fm, wm, wn, na, wk, persist)
SPILL = {(3, 1, 64, 8, 2, 4, 1, 1, 0), (3, 2, 64, 4, 1, 2, 1, 1, 1), (3, 1, 64, 2, 4, 2, 2, 1, 1),
         (3, 2, 64, 1, 4, 2, 2, 1, 1)}


def entries():
    out = []

    def add(ks, s, cin32, fm, wm, wn, wk, persist=0, na=1):
        waves = wm * wn * wk
        if waves > 16:
            return
        per_simd = -(-waves // 4)
        v, acc = regs(ks, s, cin32, fm, wm, wn, na, wk)
        if v > 256 or v + acc > 512 // per_simd or (ks, s, cin32, fm, wm, wn, na, wk, persist) in SPILL:
            return
        if lds(ks, s, cin32, fm * wm, 64 * waves) > 65536:
            return
        out.append((ks, s, cin32, fm, wm, wn, na, wk, persist))

    for cin32 in (32, 64, 96, 128):  # 3x3 stride 1, all channels in one pass
        for wn in (1, 2, 3, 4, 6):
            if wn in (1, 2, 4):
                add(3, 1, cin32, 2 if wn == 1 else 4, 4 if wn == 1 else 2, wn, 1)  # 8 rows
            add(3, 1, cin32, 1, 2, wn, 1)                                      # 2 rows
            if cin32 <= 96 and wn <= 4:
                add(3, 1, cin32, 2, 1, wn, 1)  # 2 rows in one wave row: half the weight loads per tile
        if cin32 <= 64:  # big layers, persistent: the next tile's halo loads while this one computes
            for wn in (2, 4):
                for fm, wm in ((8, 1), (8, 2), (4, 1), (4, 2)):
                    add(3, 1, cin32, fm, wm, wn, 1, 1)
    for cin32 in (160, 288):  # deep: one kernel row of K per wave
        for wn in (1, 2, 3, 4, 5):
            add(3, 1, cin32, 2, 1, wn, 3)  # 2 rows
            add(3, 1, cin32, 4, 1, wn, 3)  # 4 rows
    for cin32 in (64, 96):  # the frame's small layers: a kernel row of K per wave, chains a third as long
        for wn in (1, 2, 3):
            add(3, 1, cin32, 1, 1, wn, 3)  # 1 row
            add(3, 1, cin32, 2, 1, wn, 3)  # 2 rows
    for cin32 in (32, 64):  # 3x3 stride 2
        for wn in (1, 2, 3, 4):
            add(3, 2, cin32, 2, 2, wn, 1)  # 4 rows
            add(3, 2, cin32, 1, 2, wn, 1)  # 2 rows
            if wn in (2, 3, 4):
                add(3, 2, cin32, 2, 1, wn, 1)  # 2 rows in one wave row
        for wn in (2, 4):  # big layers, persistent
            for fm, wm in ((4, 1), (4, 2), (2, 2)):
                add(3, 2, cin32, fm, wm, wn, 1, 1)
    for cin32 in (32, 64, 96, 128):  # 1x1
        for wn in (2, 4):
            add(1, 1, cin32, 1, 2, wn, 1)
            add(1, 1, cin32, 2, 1, wn, 1)
    # big layers over more channels, persistent (their codes follow every earlier one's): one wave row of 4 rows, the
    # weights of up to 8 channel blocks over its waves (by the compiler's register report, not the estimate: the
    # larger ones keep weights in AGPRs, and (128, 8) spills 6 registers and is still the fastest over 80 channels)
    for cin32, wns in ((96, (2, 3, 4, 6, 8)), (128, (2, 3, 4, 6, 8))):
        for wn in wns:
            out.append((3, 1, cin32, 4, 1, wn, 1, 1, 1))
    # wave-stream kernel (wave_impl.h): 4 independent waves, each FM rows x 16 pixels x all 16 * NA channels of
    # the workgroup's channel tile; weights NA * K / 8 VGPRs per lane at one wave per SIMD
    # ((3, 1, 64, 2, 4) spills: 288 weight registers)
    for ks, s, cin32, fm, na in ((3, 1, 32, 4, 2), (3, 1, 32, 4, 4), (3, 1, 32, 8, 2),
                                 (3, 1, 64, 4, 2), (3, 1, 64, 2, 2),
                                 (3, 1, 96, 2, 2), (3, 2, 32, 2, 4), (3, 2, 32, 2, 2)):
        out.append((ks, s, cin32, fm, 1, 1, na, 1, 2))
    return out


def group(e):
    ks, s, cin32 = e[0], e[1], e[2]
    if e[8] == 2:
        return "w"
    if ks == 1:
        return "k1"
    if s == 2:
        return "s2"
    if e[8] == 2:
        return "w"
    if e[8]:
        return "s1p" if cin32 <= 64 else "s1q"
    return {32: "s1a", 64: "s1a", 96: "s1b", 128: "s1c", 160: "s1d", 288: "s1d"}[cin32]


def main():
    order = ["s1a", "s1b", "s1c", "s1d", "s1p", "s2", "k1", "w", "s1q"]
    es = sorted(entries(), key=lambda e: order.index(group(e)))
    assert len(es) <= 383  # variant codes 128 .. 511
    h = ["// Generated by gen_direct.py: the configurations of the direct conv kernel. Do not edit.",
         "#pragma once", "", "namespace fhc {", "",
         "struct DirectCfg {",
         "    int ks, stride, cin32, fm, wm, wn;  // rows per tile = fm * wm, channels = 16 * na * wn",
         "    int na;                             // 16-channel blocks per wave (each LDS read feeds na MFMAs)",
         "    int wk;                             // kernel-row K split; waves = wm * wn * wk",
         "    int persist;                        // 1: resident grid looping over tiles; 2: wave-stream kernel",
         "};", "",
         f"constexpr int kNumDirect = {len(es)};",
         "inline constexpr DirectCfg kDirectCfgs[kNumDirect] = {"]
    for e in es:
        h.append("    {%d, %d, %d, %d, %d, %d, %d, %d, %d}," % e)
    h += ["};", "", "}  // namespace fhc", ""]
    open(os.path.join(HERE, "direct_table.h"), "w").write("\n".join(h))
    groups = {}
    for i, e in enumerate(es):
        groups.setdefault(group(e), []).append((i, e))
    for g, items in groups.items():
        src = [f"// Generated by gen_direct.py: direct conv kernel instantiations, group {g}. Do not edit.",
               '#include "wave_impl.h"' if g == "w" else '#include "direct_impl.h"', "", "namespace fhc {", "",
               f"LaunchFn direct_launcher_{g}(int index, const void** kernel, bool residual) {{", "    switch (index) {"]
        for i, e in items:
            src.append(f"        case {i}:")
            if e[8] == 2:
                args = "%d, %d, %d, %d, %d" % (e[0], e[1], e[2], e[3], e[6])
                src.append(f"            if (kernel) *kernel = wave_kernel<{args}>();")
                src.append(f"            return launch_wave<{args}>;")
                continue
            args = "%d, %d, %d, %d, %d, %d, %d, %d, %s" % (e[:8] + ("true" if e[8] else "false",))
            src.append(f"            if (kernel) *kernel = direct_kernel<{args}>(residual);")
            src.append(f"            return launch_direct<{args}>;")
        src += ["        default: return nullptr;", "    }", "}", "", "}  // namespace fhc", ""]
        open(os.path.join(HERE, f"direct_{g}.hip"), "w").write("\n".join(src))
    disp = ["// Generated by gen_direct.py: index -> launcher of the direct conv kernel. Do not edit.",
            '#include "conv_kernels.h"', '#include "direct_table.h"', "", "namespace fhc {", ""]
    for g in groups:
        disp.append(f"LaunchFn direct_launcher_{g}(int index, const void** kernel, bool residual);")
    disp += ["", "LaunchFn direct_launcher(int index, const void** kernel, bool residual) {",
             "    if (index < 0 || index >= kNumDirect) return nullptr;"]
    for g, items in groups.items():
        idx = [i for i, _ in items]
        disp.append(f"    if (index >= {min(idx)} && index <= {max(idx)}) return direct_launcher_{g}(index, kernel, residual);")
    disp += ["    return nullptr;", "}", "", "}  // namespace fhc", ""]
    open(os.path.join(HERE, "direct_dispatch.cpp"), "w").write("\n".join(disp))
    print(f"{len(es)} direct configurations in {len(groups)} groups: {', '.join(groups)}")


if __name__ == "__main__":
    main()
