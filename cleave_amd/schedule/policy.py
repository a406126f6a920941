"""Launch-plan search space for gfx950 and the model that ranks it.

Stands where the reference's roller-style policy stands
(``python/cleave/schedule/policy/default.py:23-1110``): enumerate tilings, discard the ones
the hardware cannot hold, rank by a traffic x waves model, keep ``topk``.  Nothing of its
CUDA-shaped space is kept (warp 32, 64x32x32 wmma base tile, 164 KB shared memory, 128/256
threads).  The space here is written for one MI355X:

* 64-lane wavefronts, four SIMDs and 512 vector registers per lane per SIMD, up to 160 KiB of
  LDS per workgroup, 256 compute units;
* matrix-core tiles of 16x16x32 (f16/bf16, f32 accumulate), so every tile extent is a
  multiple of 16 and every contraction step a multiple of 32;
* 16-byte (dwordx4) global accesses: eight elements per lane, rows walked so that sixteen
  lanes cover 256 contiguous bytes;
* bandwidth-bound families (few-row matmul, decode attention) stream operands HBM -> registers
  and are tiled by *waves in flight*, not by LDS tiles; the split factor is what fills the
  256 compute units.
"""

from __future__ import annotations

import itertools
import math

from ..arch import Arch
from ..lower.stages import mla_po_elem
from .hint import TileDict

ELEM_BYTES = {"float16": 2, "bfloat16": 2}


def _ceil(a, b):
    return -(-a // b)


def _waves_time(blocks, per_cu, arch: Arch):
    """Number of full passes the grid makes over the machine."""
    return _ceil(blocks, max(1, per_cu * arch.compute_units))


# ----------------------------------------------------------------------------- GEMM
def gemm_lds_bytes(bm, bn, bk, norm=False):
    return 2 * (bm + bn) * bk * 2 + (bm * 4 if norm else 0)


def gemm_candidates(low, role, factor, arch: Arch):
    p = low.problem
    splits = factor or 1
    M, N, K = p["M"], p["N"], p["K"]
    if K % splits:
        return []
    kps = K // splits
    batch = max(p["batch_A"], p["batch_B"])
    norm = low.family == "rmsnorm_matmul"
    out = []
    shapes = (16, 32, 64, 128, 256)
    for bm, bn, bk, (wm, wn), depth in itertools.product(
            shapes, shapes, (64,), ((1, 1), (1, 2), (2, 1), (2, 2), (1, 4), (4, 1), (2, 4), (4, 2)), (1, 2)):
        if bm % (16 * wm) or bn % (16 * wn):
            continue
        if kps % bk and (splits > 1 or K % 8):       # a ragged last step: unsplit, rows of whole 16-byte chunks
            continue
        if bm > max(16, 2 * M) or bn > max(16, 2 * N):
            continue
        threads = wm * wn * 64
        tm, tn = bm // wm // 16, bn // wn // 16
        acc_regs = tm * tn * 4
        if acc_regs > 256:
            continue
        if p["trans_A"] and (bm % 8 or M % 8):
            continue
        if not p["trans_B"] and (bn % 8 or N % 8):
            continue
        # staging registers per thread and step in flight: K-minor tiles move 16-byte chunks (4
        # registers), K-major ones 8x8 blocks (32) or, when those would idle threads, 4x8 halves (16)
        def stage(rows, k_major):
            if not k_major:
                return _ceil(rows * (bk // 8), threads) * 4
            blocks = (rows // 8) * (bk // 8)
            if rows % 64 == 0 and blocks < threads:
                return _ceil(2 * blocks, threads) * 16
            return _ceil(blocks, threads) * 32
        stage_regs = depth * (stage(bm, p["trans_A"]) + stage(bn, not p["trans_B"]))
        frag_regs = (min(tm, 3) + 2 * tn) * 4
        vgprs = acc_regs + stage_regs + frag_regs + 40
        if vgprs > arch.vgprs_per_lane:
            continue
        lds = gemm_lds_bytes(bm, bn, bk, norm)
        if lds > arch.lds_bytes:
            continue
        blocks = _ceil(M, bm) * _ceil(N, bn) * batch * splits
        per_cu = arch.blocks_per_cu(threads, lds, vgprs)
        if per_cu < 1:
            continue
        if depth == 2 and (_ceil(kps, bk) < 4 or per_cu * threads > 512 and vgprs > 128):
            continue
        passes = _waves_time(blocks, per_cu, arch)
        live = min(per_cu, _ceil(blocks, arch.compute_units))         # blocks a CU really holds
        # one pass over the machine: the CU's matrix cores, its L1 path (about 24 B/clk sustained
        # for these access shapes) and its LDS are shared by the blocks it holds
        mfma_clk = live * (bm * bn * kps * 2) / 4096.0 / min(1.0, live * wm * wn / 8.0)
        l1_clk = live * ((bm + bn) * kps * 2) / (24.0 * (1.6 if depth == 2 else 1.0))
        lds_clk = live * (tm + tn) * 16 * wm * wn * kps * 2 / 256.0
        pass_clk = max(mfma_clk, l1_clk, lds_clk) + 2500 + 1200 * _ceil(kps, bk) / max(1, min(live, 2))
        score = passes * pass_clk
        # (where the direct-to-LDS kernel offers the same tile it has measured a quarter to two thirds
        # faster -- 2048 x 4096 x 4096 on 128 x 128 tiles: 67 against 91 us; 512 x 512 x 4096 on 16 x 32 tiles:
        # 14 against 42 -- while this model ranked the register-staged one ahead: its candidates go behind)
        if low.family == "matmul":
            score *= 2.0
        tiling = dict(BM=bm, BN=bn, BK=bk, WM=wm, WN=wn, GDEPTH=depth)
        out.append(TileDict("gemm", role, tiling, output_tile=[bm, bn], rstep_map={"k": bk}, n_threads=threads,
                            split_factor=factor, score=score, lds_bytes=lds, est_vgprs=vgprs))
    return out


def phased_matmul(family, problem, splits, tile) -> bool:
    """Which products run on ``gemm_phased.hip`` (two wave groups alternating between memory and matrix work)
    instead of the lock-step ``gemm_dma.hip``: all that it has a form for.  It needs eight waves (two per SIMD,
    one multiplying while the other reads) with 16 matrix ops each per phase, at least the two K steps its
    pipeline holds, and rows of C that leave as 16-byte pieces; the fused norm, the row-sum walk and the load
    and matrix-op knobs are the lock-step kernel's.  us, lock-step / phased: 8192^3 bf16 (N, K) weight 806 / 701,
    4096 x 14336 x 4096 f16 393 / 352 (with the last half round split), SwiGLU of that size 752 / 676, 3000 x 5000 x 2048
    56 / 52; 128 x 256 tiles (three stages lock-step) 2048 x 4096 x 4096 60.1 / 56.3, 724 x 6272 x 640 13.3 / 10.7; at the
    small end 2999 x 1000 x 192 9.8 / 8.2.  192 x 256 tiles (A's halves of 128 and 64 rows) exist here only, for row-major A."""
    bm, bn, wm, wn = (int(tile[k]) for k in ("BM", "BN", "WM", "WN"))
    sizes = ((bm, bn) == (256, 256) or ((bm, bn) in ((128, 256), (256, 128)) and not int(tile.get("TAIL", 0)))
             or ((bm, bn, wm) == (192, 256, 2) and not problem["trans_A"] and not int(tile.get("TAIL", 0))))
    return (sizes and wm * wn == 8 and bn // 2 // wn % 32 == 0 and bm // 2 // wm % 16 == 0 and family in ("matmul", "swiglu")
            and problem["K"] // splits > 64 and problem["N"] % 8 == 0 and int(tile.get("STAGES", 2)) == 2
            and not {"ASM_LOADS", "ASM_MFMA", "SPREAD_LOADS"} & set(tile))


def gemm_dma_candidates(low, role, factor, arch: Arch, twin_of=None):
    """Tilings of the direct-to-LDS matmul: the plain matmul, and the RMSNorm -> matmul without a
    learned weight, unsplit (the norm then scales the product's rows; with a weight the operand
    would have to pass through registers on its way to LDS).  No staging registers, so the budget is accumulators plus two
    k blocks of operand fragments; tiles whose accumulators would fill a whole register class
    (256) are left out: the compiler then shuffles them on every step."""
    p = low.problem
    splits = factor or 1
    post_norm = low.family == "rmsnorm_matmul" and not p.get("gamma") and not p["trans_A"] and splits == 1 \
        and role == "main"
    if low.family != "matmul" and not post_norm:
        return []
    M, N, K = p["M"], p["N"], p["K"]
    # (unsplit, the last K step may be partly filled: its chunks past K are fetched as zeros)
    if K % (splits * 64 if splits > 1 else 8) or (not p["trans_B"] and N % 8) or (p["trans_A"] and M % 8):
        return []
    kps = _ceil(K // splits, 64) * 64
    batch = max(p["batch_A"], p["batch_B"])
    out = []
    shapes = (16, 32, 64, 128, 256)
    grids = ((1, 1), (1, 2), (2, 1), (2, 2), (1, 4), (4, 1), (2, 4), (4, 2))
    # 192 x 256 tiles, of the two-group kernel only: a round of them takes about 0.9 of one of 256 x 256 ones (0.78 to 0.93), so they are
    # proposed where that many rounds (one workgroup per compute unit) are less.  us a call, f16, 256 x 256 / these: one round each 3479 x
    # 3264 x 1984 44.3 / 40.9, 2300 x 5120 x 2048 46.1 / 41.6, 1536 x 8000 x 4096 83.4 / 77.8, 3916 x 3072 x 384 15.6 / 13.9, two each 2226 x
    # 7296 x 544 35.2 / 29.0; where they cost one round more 3000 x 5000 x 2048 53.5 / 83.6.  Of 24 drawn products that are offered them
    # they were the fastest of the eight tried in all, and none was fastest on the tiling they push out.
    uneven = (192, 256, (2, 4))
    rounds = {bm: _ceil(_ceil(M, bm) * _ceil(N, 256) * batch, arch.compute_units) for bm in (192, 256)}
    fits = (not post_norm and twin_of != "matmul_rowsum" and splits == 1 and 0.9 * rounds[192] < rounds[256]
            and phased_matmul("matmul", p, 1, dict(BM=192, BN=256, WM=2, WN=4)))
    for bm, bn, (wm, wn) in itertools.chain(itertools.product(shapes, shapes, grids), (uneven,) if fits else ()):
        if bm % (16 * wm) or bn % (16 * wn):
            continue
        if bm > max(16, 2 * M) or bn > max(16, 2 * N):
            continue
        threads = wm * wn * 64
        tm, tn = bm // wm // 16, bn // wn // 16
        if (tm & (tm - 1) and bm != 192) or tn & (tn - 1) or tm * tn * 4 > 128:
            continue
        if post_norm and low.dtype == "bfloat16" and tm * tn * 4 > 64 and wm > wn:
            continue      # bf16 squares go through float conversions: beside a 128-register, 4-row-fragment tile they spill
        # every wave must own whole 1 KiB load units of both tiles or none
        units_a, units_b = bm // 8, bn // 8
        vgprs = tm * tn * 4 + (tm + tn) * 6 + -(-units_a // (wm * wn)) + -(-units_b // (wm * wn)) + 24
        if vgprs > arch.vgprs_per_lane:
            continue
        lds = gemm_lds_bytes(bm, bn, 64)
        if lds > arch.lds_bytes:
            continue
        blocks = _ceil(M, bm) * _ceil(N, bn) * batch * splits
        per_cu = arch.blocks_per_cu(threads, lds, vgprs)
        if per_cu < 1:
            continue
        passes = _waves_time(blocks, per_cu, arch)
        live = min(per_cu, _ceil(blocks, arch.compute_units))
        mfma_clk = live * (bm * bn * kps * 2) / 4096.0 / min(1.0, live * wm * wn / 8.0)
        # LDS -> register traffic: about 32 B/clk per SIMD for 16-byte reads, two thirds of that for
        # the transposing reads of a K-major operand
        a_rate = 21.0 if p["trans_A"] else 32.0
        b_rate = 32.0 if p["trans_B"] else 21.0
        waves_per_simd = max(1.0, live * wm * wn / 4.0)
        lds_clk = waves_per_simd * kps * 2 * 16 * (tm / a_rate + tn / b_rate)
        fetch_clk = live * ((bm + bn) * kps * 2) / 24.0
        pass_clk = max(mfma_clk, lds_clk, fetch_clk) + 2500 + 1500 * (kps // 64) / max(1, min(live, 2))
        # (equal tiles: the wave grids with more waves have measured a few per cent faster -- more loads in flight)
        score = passes * pass_clk * (1.0 + 0.03 / (wm * wn))
        tiling = dict(BM=bm, BN=bn, BK=64, WM=wm, WN=wn)
        # 128 x 256 and 256 x 128 tiles whose wave groups alternate between memory and matrix work: 6 to 25 % ahead of
        # the three-stage lock-step form of the same tile (which ranks at 0.85), so a plain product has no use for that
        # one.  SwiGLU's two weights keep both, this one right behind: the search times them.
        phased = bm * bn == 128 * 256 and not post_norm and twin_of != "matmul_rowsum" and phased_matmul("matmul", p, splits, tiling)
        place = score if not phased else math.nextafter(0.85 * score, math.inf) if twin_of else 0.8 * score
        out.append(TileDict("gemm_dma", role, tiling, output_tile=[bm, bn], rstep_map={"k": 64}, n_threads=threads,
                            split_factor=factor, score=place, lds_bytes=lds, est_vgprs=vgprs))
        # Three LDS stages where three images fit beside as many workgroups per compute unit as two
        # allow: the loads of a step asked for two steps ahead and spread over the whole step
        # (256 x 128 tiles on 4096 x 14336 x 4096: 426 us against 526).  The row-sum walk has no such form.
        if (twin_of != "matmul_rowsum" and (twin_of or not phased) and 3 * (bm + bn) * 128 * per_cu <= arch.lds_bytes and units_a % (wm * wn) == 0 and units_b % (wm * wn) == 0
                and not post_norm):
            out.append(TileDict("gemm_dma", role, dict(tiling, STAGES=3), output_tile=[bm, bn], rstep_map={"k": 64},
                                n_threads=threads, split_factor=factor, score=0.85 * score, lds_bytes=3 * lds // 2,
                                est_vgprs=vgprs))
        # A last round that fills at most half of the machine: its tiles as two half-height
        # workgroups each (row-major A, one workgroup per compute unit, unsplit, unbatched).
        tail = blocks % arch.compute_units
        if (blocks > arch.compute_units and 0 < tail <= arch.compute_units // 2 and per_cu == 1 and splits == 1
                and batch == 1 and not p["trans_A"] and tm >= 2 and M % bm == 0 and bm != 192):
            out.append(TileDict("gemm_dma", role, dict(tiling, TAIL=tail), output_tile=[bm, bn], rstep_map={"k": 64},
                                n_threads=threads, split_factor=factor, score=(passes - 0.45) * pass_clk,
                                lds_bytes=lds, est_vgprs=vgprs))
    if not twin_of and not post_norm:
        # Third and fourth at best, behind the two best tilings of one wave grid per tile: the request model below ranks the
        # K-sharing tilings among themselves, and timing, not the model, puts one of them first.
        second = sorted(c.score for c in out)[1:2]
        for c in kwaves_candidates(low, role, factor, arch):
            c.score = max([c.score] + [math.nextafter(s, math.inf) for s in second])
            out.append(c)
    if not twin_of and low.family == "matmul" and splits == 1:
        out += k_range_candidates(low, role, arch)
    if K % 64:
        # (under the name of the template that takes such lengths; DMA picks its direct-to-LDS form)
        for c in out:
            c.template, c.tiling = "gemm", dict(c.tiling, DMA=1)
    return out


def k_range(K, n) -> int:
    """The extent of ``n`` ranges that K is dealt out to inside an unsplit product, or 0 where it cannot be: whole 64-wide steps
    if the last range is then less than a step short, else whole 16-byte chunks.  Every range is walked in the same number of
    steps, two or more, and the kernels fetch zeros for the rest of a range's last step only."""
    if n < 2 or K % 8:
        return 0
    for unit in (64, 8):
        extent = _ceil(_ceil(K, unit), n) * unit
        steps = _ceil(extent, 64)
        if steps >= 2 and K - (n - 1) * extent - (steps - 1) * 64 >= 0:
            return extent
    return 0


def k_range_candidates(low, role, arch: Arch, twin=False):
    """Products of too few tiles for the chip and a long contraction: K dealt out to ranges inside an unsplit operator, f32
    partials in scratch folded by a second launch (SwiGLU's gate there too).  Two tilings, with as many ranges as give
    every compute unit one 128 x 256 tile (two of 128 x 128, at most five ranges) and a range eight steps.  Measured, us, best unsplit /
    ranges: 655 x 3264 x 6912 53.1 / 41.6, 3000 x 1000 x 8000 67.0 / 53.1, 290 x 1968 x 5056 32.6 / 18.8, SwiGLU 156 x 3968 x
    8064 89.8 / 44.3 and 700 x 1024 x 4096 32.4 / 23.5; behind where the contraction is short (906 x 1152 x 1024 9.7 / 13.1)
    or the tiles fill the chip (SwiGLU 507 x 7040 x 2240 32.3 / 49.7)."""
    p = low.problem
    M, N, K = p["M"], p["N"], p["K"]
    width = 2 * N if twin else N
    batch = max(p["batch_A"], p["batch_B"])
    steps = _ceil(K, 64)
    if role != "main" or steps < 24 or K % 8 or (not p["trans_B"] and N % 8) or (p["trans_A"] and M % 8):
        return []
    out = []
    for (bm, bn), fill in (((128, 256), 1), ((128, 128), 2)):
        if twin and N % (bn // 2) or not twin and bn > 2 * N:
            continue
        blocks = _ceil(M, bm) * _ceil(width, bn) * batch
        most = min(fill * arch.compute_units // blocks, 8 if fill == 1 else 5, steps // 8)
        fits = [n for n in range(2, most + 1) if k_range(K, n) and 4 * n * batch * M * width + 512 <= FIXED_SCRATCH]
        # (ranges that start on a 128-byte line ahead of one range more)
        n = max((n for n in fits[-2:] if k_range(K, n) % 64 == 0), default=fits[-1] if fits else 0)
        if n and _ceil(M, 128) * _ceil(width, 256) * batch <= arch.compute_units // 2:
            tiling = dict(BM=bm, BN=bn, BK=64, WM=2, WN=4, KS=n, **({"SWIGLU": 1} if twin else {}))
            out.append(TileDict("gemm_dma", role, tiling, output_tile=[bm, bn // 2 if twin else bn], rstep_map={"k": 64}, n_threads=512,
                                score=float(steps // n), lds_bytes=gemm_lds_bytes(bm, bn, 64), est_vgprs=200, late=True))
    return out


def kwaves_lds_bytes(bm, bn, kw):
    """LDS of the matmul whose waves share K: two images of both tiles per wave, reused for the final sums."""
    return max(kw * 2 * (bm + bn) * 128, kw * bm * bn * 4)


def kwaves_candidates(low, role, factor, arch: Arch):
    """Tilings of the matmul whose waves share K, for products of few tiles and a long contraction (at least eight
    64-wide steps, at most 1024 tiles of 32 x 32): the two the model likes best.  What a step costs a compute unit is
    the 64-byte requests its waves make, one a clock at best (measured alike with two, three and four images per
    wave: 47 bytes a clock): two per K-minor row (three where rows are not whole 128-byte lines), one per 32 columns of
    a K-major row."""
    p = low.problem
    M, N, K = p["M"], p["N"], p["K"]
    batch = max(p["batch_A"], p["batch_B"])
    steps = _ceil(K, 64)
    if (low.family != "matmul" or role != "main" or (factor or 1) > 1 or K % 8 or N % 8 or (p["trans_A"] and M % 8)
            or steps < 8 or _ceil(M, 32) * _ceil(N, 32) * batch > 1024):
        return []

    def requests(extent, k_major):
        return 64 * _ceil(extent, 32) if k_major else extent * (2 if K % 64 == 0 else 3)

    out = []
    for (bm, bn), kw in itertools.product(((16, 16), (16, 32), (32, 16), (32, 32), (32, 64), (64, 32), (64, 64)), (4, 8)):
        lds = kwaves_lds_bytes(bm, bn, kw)
        if lds > arch.lds_bytes or kw > steps or (bm > 16 and bm >= 2 * M) or (bn > 16 and bn >= 2 * N):
            continue
        blocks = _ceil(M, bm) * _ceil(N, bn) * batch
        per_cu = max(1, min(arch.lds_bytes // lds, 32 // kw))
        live = min(per_cu, _ceil(blocks, arch.compute_units))
        step_clk = max(1000.0, live * kw * (requests(bm, p["trans_A"]) + requests(bn, not p["trans_B"])) * 1.3)
        score = _waves_time(blocks, per_cu, arch) * (_ceil(steps, kw) * step_clk + 4000 + 60 * kw)
        out.append(TileDict("gemm_dma", role, dict(BM=bm, BN=bn, BK=64, WM=1, WN=1, KW=kw), output_tile=[bm, bn],
                            rstep_map={"k": 64}, n_threads=kw * 64, split_factor=factor, score=score, lds_bytes=lds,
                            est_vgprs=bm * bn // 64 + 60))
    out.sort(key=lambda c: (c.score, c.key()))
    return out[:2]


def swiglu_candidates(low, role, factor, arch: Arch):
    """SwiGLU runs on the direct-to-LDS matmul with a B tile made of two halves, the same
    columns of the bare weight and of the gate weight: the tilings of a matmul twice as wide in
    which every wave owns an even number of column fragments (half of them per weight)."""
    import copy

    if (factor and factor > 1) or low.problem["K"] % 64:
        return []
    twin = copy.copy(low)
    twin.family, twin.problem = "matmul", dict(low.problem, N=2 * low.problem["N"])
    out = []
    for c in gemm_dma_candidates(twin, role, None, arch, twin_of="swiglu"):
        t = c.tiling
        tn = t["BN"] // t["WN"] // 16
        if tn % 2 or low.problem["N"] % (t["BN"] // 2):
            continue
        c.tiling = dict(t, SWIGLU=1)
        c.output_tile = [t["BM"], t["BN"] // 2]
        out.append(c)
    return out + (k_range_candidates(low, role, arch, twin=True) if out else [])


def rowsum_candidates(low, role, factor, arch: Arch):
    """Matmul + row sum: tilings of the direct-to-LDS matmul in which one workgroup owns BM rows and
    walks all of N (whole column tiles), so the grid is the row tiles alone: ranked by how many
    step sequences of ``(N / BN) * (K / 64)`` steps the machine runs one after another."""
    import copy

    if (factor and factor > 1) or low.problem["K"] % 64:
        return []
    p = low.problem
    twin = copy.copy(low)
    twin.family = "matmul"
    out = []
    for c in gemm_dma_candidates(twin, role, None, arch, twin_of="matmul_rowsum"):
        t = c.tiling
        if p["N"] % t["BN"]:
            continue
        blocks = _ceil(p["M"], t["BM"])
        steps = (p["N"] // t["BN"]) * (p["K"] // 64)
        waves = t["WM"] * t["WN"]
        mfma_clk = (t["BM"] // t["WM"] // 16) * (t["BN"] // t["WN"] // 16) * 2 * 16.4 * max(1.0, waves / 4.0)
        c.score = _waves_time(blocks, 1, arch) * steps * (mfma_clk + 700)
        c.tiling = dict(t, ROWSUM=1)
        c.output_tile = [t["BM"], 1]
        out.append(c)
    return out


def lora_lds_bytes(mt, waves_n, waves_k, rank):
    """The few-row kernel's reduction buffers twice (main and rank-R accumulators) plus the D tile."""
    return 2 * skinny_lds_bytes(mt, waves_n, waves_k) + waves_n * 16 * mt * rank * 4 + 16


def lora_candidates(low, role, factor, arch: Arch):
    """LoRA: the few-row matmul with the rank-R product ``x @ a`` riding along.  Unsplit, the epilogue
    applies the rank update; split over K, the partial kernel writes partial sums of both products
    and the combine applies it (it needs the whole of ``x @ a``)."""
    import copy

    p = low.problem
    if p["R"] % 8 or p["R"] > 64 or ((factor or 1) > 1 and p["N"] % 256):
        return []
    twin = copy.copy(low)
    twin.family = "matmul"
    if not skinny_ok(twin):
        return []
    out = []
    for c in skinny_candidates(twin, role, factor, arch):
        t = c.tiling
        lds = lora_lds_bytes(_ceil(p["M"], 16), t["WAVES_N"], t["WAVES_K"], p["R"])
        if lds > arch.lds_bytes:
            continue
        c.tiling, c.lds_bytes = dict(t, LORA=1), lds
        if t["WAVES_N"] * t["WAVES_K"] > 4:
            # more than four waves have 256 registers each: the ring of tiles (each now carries a block
            # of the rank-R factor too) is one tile shallower so that nothing spills
            c.tiling["PREFETCH"] = 1
        out.append(c)
    return out


def rowsum_only_candidates(low, role, factor, arch: Arch):
    """Row reductions: one wave per row, 1, 2 or 4 rows per workgroup; the cost is the stream."""
    p = low.problem
    if (factor or 1) > 1 or p["N"] % 8:
        return []
    out = []
    for rows in (4, 2, 1):
        blocks = _ceil(p["M"], rows)
        nbytes = p["M"] * p["N"] * 2 * (3 if p["div"] else 1)
        score = nbytes / (arch.hbm_gbps * 1e3 * 0.6) * 2400 + 3000 + 200 * _waves_time(blocks, 8, arch) + rows
        out.append(TileDict("rowsum", role, dict(ROWS_PER_BLOCK=rows), output_tile=[rows, p["N"] if p["div"] else 1],
                            rstep_map={"n": 512}, n_threads=64 * rows, split_factor=factor, score=score, lds_bytes=0,
                            est_vgprs=40))
    return out


# ----------------------------------------------------------------------------- few-row matmul
def skinny_ok(low) -> bool:
    p = low.problem
    return (p["M"] <= 64 and not p["trans_A"] and not p["trans_B"] and p["batch_A"] == 1 and p["batch_B"] == 1
            and p["K"] % 32 == 0 and p["N"] % 8 == 0 and p["N"] >= 8)


def skinny_lds_bytes(mt, waves_n, waves_k):
    return ((waves_k - 1) * waves_n * mt * 32 * 64 + waves_k * mt * 16) * 4 + 16


def skinny_candidates(low, role, factor, arch: Arch):
    p = low.problem
    splits = factor or 1
    M, N, K = p["M"], p["N"], p["K"]
    mt = _ceil(M, 16)
    steps = K // 32
    if steps % splits:
        return []
    out = []
    for waves_n, waves_k in itertools.product((1, 2, 4), (1, 2, 4, 8)):
        threads = waves_n * waves_k * 64
        if threads > 1024:
            continue
        per_split = steps // splits
        if per_split < waves_k:
            continue
        lds = skinny_lds_bytes(mt, waves_n, waves_k)
        if lds > arch.lds_bytes:
            continue
        vgprs = mt * 32 + 3 * 32 + 32 + mt * 4 + 40
        blocks = _ceil(N, 128 * waves_n) * splits
        per_cu = arch.blocks_per_cu(threads, max(lds, 1), vgprs)
        if per_cu < 1:
            continue
        passes = _waves_time(blocks, per_cu, arch)
        waves_live = min(blocks, per_cu * arch.compute_units) * waves_n * waves_k
        # a wave keeps ~3 steps of 8 KiB in flight; HBM wants ~16 MiB outstanding machine-wide
        inflight = waves_live * 24 * 1024
        bw_frac = min(1.0, inflight / (12 * 1024 * 1024))
        stream_us = (K * N * 2) / (arch.hbm_gbps * 1e3 * bw_frac)
        partial_us = (2 * splits * M * N * 4) / (arch.hbm_gbps * 1e3) if splits > 1 else 0.0
        tail = 1.0 + 0.25 * (passes - 1) + 0.02 * waves_k
        score = (stream_us * tail + partial_us) * 2400
        tiling = dict(WAVES_N=waves_n, WAVES_K=waves_k)
        out.append(TileDict("skinny", role, tiling, output_tile=[M, 128 * waves_n], rstep_map={"k": 32},
                            n_threads=threads, split_factor=factor, score=score, lds_bytes=lds, est_vgprs=vgprs))
    return out


# ----------------------------------------------------------------------------- decode attention
def attn_lds_bytes(waves, vdim):
    """LDS of the streaming decode kernel: every wave but the first parks its accumulators (a 16-byte piece per
    lane and accumulator, eight accumulators per 128 value features) and its 16 reference points and sums."""
    return (waves - 1) * (-(-vdim // 128) * 8 * 64 * 16 + 128)


def attn_ok(low) -> bool:
    p = low.problem
    return p["head_dim"] % 32 == 0 and (p["vdim"] % 128 == 0 or p["vdim"] == 64)


def attn_candidates(low, role, factor, arch: Arch, waves_options=(1, 2, 4, 8)):
    p = low.problem
    splits = factor or 1
    rows = p["group"] * p["sq"]
    row_tiles = _ceil(rows, 16)
    d, vd = p["head_dim"], p["vdim"]
    steps = _ceil(p["skv"], 32)
    out = []
    for waves in waves_options:
        lds = attn_lds_bytes(waves, vd)
        if lds > arch.lds_bytes:
            continue
        kv_regs = (2 * (d // 32) + 8 * _ceil(vd, 128)) * 4
        vgprs = 2 * kv_regs + 32 * _ceil(vd, 128) + 4 * (d // 32) + 32 + 48
        if vgprs > arch.vgprs_per_lane:
            continue
        blocks = p["units"] * row_tiles * splits
        per_cu = arch.blocks_per_cu(waves * 64, lds, vgprs)
        if per_cu < 1:
            continue
        passes = _waves_time(blocks, per_cu, arch)
        steps_per_wave = _ceil(_ceil(steps, splits), waves)
        waves_live = min(blocks, per_cu * arch.compute_units) * min(waves, _ceil(steps, splits))
        inflight = waves_live * 2 * kv_regs * 64 * 4 / 2
        # (measured on the 8192-key decode: 512 one-wave workgroups with one 16 KB step in flight each stream at
        # the rate of the box; two and four waves per workgroup take 7 % and 20 % longer)
        bw_frac = min(1.0, inflight / (8 * 1024 * 1024))
        bytes_total = p["units"] * row_tiles * p["skv"] * (d + vd) * 2
        stream_us = bytes_total / (arch.hbm_gbps * 1e3 * bw_frac) * (1.0 + 0.07 * math.log2(waves) ** 1.5)
        ramp_us = 1.5                                    # fixed launch + drain cost
        partial_us = (2 * splits * p["units"] * rows * (vd + 2) * 4) / (arch.hbm_gbps * 1e3) if splits > 1 else 0.0
        score = (stream_us * (1.0 + 0.2 * (passes - 1)) + ramp_us + partial_us + 0.05 * waves) * 2400
        tiling = dict(WAVES=waves)
        out.append(TileDict("attn_decode", role, tiling, output_tile=[16, vd], rstep_map={"kv": 32},
                            n_threads=waves * 64, split_factor=factor, score=score, lds_bytes=lds, est_vgprs=vgprs))
        # split ranges spread over the XCDs and skewed between even and odd ones (measured on the 8192-key
        # decode: with all splits of a unit on one XCD the kernel ends with its slowest XCD, 4-5 % later)
        if splits > 1 and splits % 2 == 0 and waves <= 2 and (p["units"] * row_tiles) % 8 == 0 and steps >= 4 * splits:
            for skew in (30, 60):
                out.append(TileDict("attn_decode", role, dict(WAVES=waves, SKEW=skew), output_tile=[16, vd],
                                    rstep_map={"kv": 32}, n_threads=waves * 64, split_factor=factor,
                                    score=score * (0.96 if skew == 30 else 0.965), lds_bytes=lds, est_vgprs=vgprs))
        # a second step of loads in flight (measured on the 8192-key decode: with about two waves per CU
        # streaming, the deeper ring is worth a few percent; with many waves it is not)
        if waves <= 2 and vgprs + kv_regs <= arch.vgprs_per_lane and steps_per_wave >= 8:
            out.append(TileDict("attn_decode", role, dict(WAVES=waves, PREFETCH=2), output_tile=[16, vd],
                                rstep_map={"kv": 32}, n_threads=waves * 64, split_factor=factor, score=score * 1.001,
                                lds_bytes=lds, est_vgprs=vgprs + kv_regs))
    return out


def attn_many_rows_candidates(low, role, factor, arch: Arch):
    """Units with many query rows (prefill-shaped dense attention): the kernel whose four waves
    share every key tile through LDS, 128 query rows per workgroup, instead of one 16-row tile per
    workgroup streaming all keys.  Key and value widths in 64-feature panels; split over the keys
    (ranges of whole 32-key steps, f32 partials) when there are too few units and rows to fill the chip."""
    p = low.problem
    rows, d = p["group"] * p["sq"], p["head_dim"]
    vd = p["vdim"]
    splits = factor or 1
    # plain softmax attention with few rows per unit belongs to the streaming decode kernel; QK-norm, the
    # chained matmul and widths the streaming kernel has no form for (a 192-wide value) exist in this
    # kernel only, so there it takes units of any height (one workgroup per unit, most of its 128 rows masked)
    only_here = bool(p.get("norm_eps") or p.get("linear")) or not attn_ok(low)
    if (rows < 64 and not only_here) or d % 64 or d > 256 or vd % 64 or vd > 256 or p["skv"] < 1:
        return []
    if splits > 1 and p.get("emit_lse"):
        return []
    if p.get("k_major") and p["skv"] % 32:       # feature-major keys are loaded in whole 32-key steps
        return []
    items = p["units"] * _ceil(rows, 128) * splits
    steps = _ceil(_ceil(p["skv"], 32), splits)
    # a workgroup-step is 32 matrix ops per wave beside as many vector ops; two workgroups per CU
    score = _waves_time(items, 2, arch) * (steps * 2200 + 9000)
    lds = (4 if d > 192 or d + vd == 384 else 3) * 32 * (d + vd) * 2
    out = [TileDict("attn_prefill", role, dict(SHARED=1), output_tile=[128, vd], rstep_map={"kv": 32}, n_threads=256,
                    split_factor=factor, score=score, lds_bytes=lds, est_vgprs=230)]
    # normalised keys: every workgroup of a unit normalises all of its keys again (a quarter more
    # matrix ops per step and the scaling of the scores); with many row blocks per unit a launch
    # that normalises them once into a scratch copy is cheaper
    kpre = "k" in (p.get("norm_eps") or {}) and not p.get("k_major") and d in (64, 128, 256) and rows >= 512
    if kpre:
        out.append(TileDict("attn_prefill", role, dict(SHARED=1, KPRE=1), output_tile=[128, vd], rstep_map={"kv": 32},
                            n_threads=256, split_factor=factor, score=0.8 * score, lds_bytes=lds, est_vgprs=230))
    if role != "main":
        return out
    # 256 rows on two wave groups half a step apart: half the tile bytes per row, but one workgroup per compute unit
    # and nothing beside its first loads.  Measured ahead from about 1000 keys (128 wide, us: 4096 keys 245 -> 228, 1024 keys
    # 67.1 -> 65.4, 512 keys 39.7 -> 40.0) where its workgroups keep most compute units busy, so it is proposed from half of either on.  Where it is ahead for
    # certain -- keys in plenty, wide keys, and rows that fill seven eighths of its rounds of one workgroup per compute unit --
    # instead of the other: a search times each for some milliseconds, in which the clock has not settled where the power cap
    # holds it, and picked the slower one every other time.  us over 2048 keys, 128 wide, the other / this one, by the share of its
    # rounds that 32 / 8 heads fill: 2048 rows (all of one) 66.2 / 61.7, 2112 (0.52 of two) 90.1 / 108.1, 3072 (0.75) 98.4 / 108.6,
    # 3584 (0.88) 115 / 106, 4096 (all) 128.8 / 122.2, 4160 (0.68 of three) 150 / 168, 5120 (0.83) 159.4 / 168.7, 5376 (0.88) 172 / 161,
    # 7200 (0.88 of four) 229 / 217; 3584 rows at 192 / 128, 192 / 64 and 128 / 64 wide 138 / 127, 119 / 105, 94 / 85.
    blocks = p["units"] * _ceil(rows, 256)
    filled = p["units"] * rows / (256 * arch.compute_units * _ceil(blocks, arch.compute_units))
    if attn_phased_ok(p, kpre) and p["skv"] >= 768 and blocks >= arch.compute_units // 2:
        out.append(TileDict("attn_prefill", role, dict(SHARED=1, PHASED=1, **({"KPRE": 1} if kpre else {})), output_tile=[256, vd],
                            rstep_map={"kv": 64}, n_threads=512, split_factor=factor, score=score,
                            lds_bytes=4 * 64 * (d + vd) * 2, est_vgprs=216, late=True,
                            displaces=out[-1].tiling if d >= 128 and p["skv"] >= 2048 and blocks >= arch.compute_units and filled >= 0.875 else None))
    # Too few workgroups for the chip and keys enough to share out among more: the key ranges of the split form inside one
    # operator (partials in scratch, folded by a second launch).  Measured, us, unsplit / ranges: 56 items of 122 steps
    # 61.5 / 31.3 (4), 16 items of 76 steps 40.3 / 17.1 (8; 20.3 with 16), 64 items of 63 steps 64 wide 26.2 / 16.8 (4); behind
    # from about a hundred items on or a range of fewer than six steps: 80 items of 14 steps 11.5 / 16.8.  At most 32 ranges: the
    # combine reads every range's partial of a row at once, and from 64 on that is slower than what they save -- two items of
    # 512 steps, 128 wide, us by ranges: 1 225, 20 30.3, 32 25.2, 48 29.8, 64 59.5, 128 120.  (Where the steps do not divide, the
    # last ranges are empty: eight items of 97 steps take 19.6 in 16 ranges, two of them empty, and 21.6 in 14.)
    if not p.get("emit_lse") and not kpre:
        most = [min(fill // items, steps // 6, 32) for fill in (arch.compute_units, arch.compute_units // 2)]
        for n in (most[0], most[1] if most[1] < most[0] else most[0] // 2):
            if n > 1 and attn_keys_scratch(p, n) <= FIXED_SCRATCH:
                out.append(TileDict("attn_prefill", role, dict(SHARED=1, KEYS=n), output_tile=[128, vd], rstep_map={"kv": 32},
                                    n_threads=256, split_factor=factor, score=score / n, lds_bytes=lds, est_vgprs=230, late=True))
    return out


FIXED_SCRATCH = 64 << 20         # what a call without allocations has for scratch: plans of its own that need more are not proposed


def attn_keys_scratch(p, n) -> int:
    """Bytes of the partials of ``n`` key ranges: reference point, sum and unnormalised values of every row."""
    return n * p["units"] * p["group"] * p["sq"] * (p["vdim"] + 2) * 4 + 3 * 256


def attn_phased_ok(p, kpre) -> bool:
    """Whether the two-group kernel takes an attention: four 64-key images of K and V in 160 KiB of LDS, its accumulators and
    query rows in half a SIMD's registers, row-major keys that need no norm on the way (``kpre``: a launch ahead normalises them)."""
    d, vd = p["head_dim"], p["vdim"]
    return (d % 64 == 0 and vd % 64 == 0 and vd <= 128 and (d + vd) // 64 <= 5 and not p.get("k_major")
            and (kpre or "k" not in (p.get("norm_eps") or {})))


COMBINE_GROUPS = (8, 16)         # of 32 threads, 128 columns; of 16 threads where the values are an odd number of 64s wide


def combine_groups(rows, vdim, splits) -> int:
    """Thread groups that share the splits of a row in the combine of f32 partials, or 1: one thread adds up all of them.  The line
    lies between 256 x 128 values of 32 splits (25.1 us with one thread each, 23.9 with groups) and 256 x 512 of 16 (18.0 / 18.3)."""
    if splits <= 16 or vdim % 64 or rows * vdim > 64 * 1024:
        return 1
    return next(n for n in COMBINE_GROUPS if vdim * n % 1024 == 0)


# ----------------------------------------------------------------------------- MLA decode
def mla_lds_bytes(ckv, kpe, stages=3):
    """`stages` token-major images of a 32-token step: (ckv + kpe) / 64 panels of 32 x 64 elements."""
    return stages * ((ckv + kpe) // 64) * 32 * 64 * 2


def mla_duo_lds_bytes(ckv, kpe, prefill=False):
    """LDS of the score-wave / value-wave kernel: four images, weights and reference points in flight, and for prefill the
    table entries of four steps and the final sums."""
    return mla_lds_bytes(ckv, kpe, 4) + (14 if prefill else 9) * 1024


def mla_duo_fits(ckv, kpe, prefill=False) -> bool:
    """Widths the score-wave / value-wave kernel is written for: two value waves halve the latent row's 64-feature panels,
    and the Q rows in LDS are an odd number of 64-feature runs long (128 bytes off between neighbours: no bank conflicts),
    with four images in a workgroup's LDS.  (A rope width of 128 passed here and failed in the compiler.)"""
    return ckv % 128 == 0 and kpe % 128 == 64 and mla_duo_lds_bytes(ckv, kpe, prefill) <= 160 * 1024


def mla_ok(low) -> bool:
    p = low.problem
    return p["heads"] % 16 == 0 and p["ckv"] % 64 == 0 and p["kpe"] % 64 == 0


def mla_candidates(low, role, factor, arch: Arch):
    p = low.problem
    splits = factor or 1
    out = []
    d = p["ckv"] + p["kpe"]
    for waves, (hg, vsplit), stages in itertools.product((1, 2, 4, 8), ((1, 1), (2, 2)), (2, 3, 4)):
        # 32 heads per wave only with the value features shared out over a wave pair: the
        # accumulators of 32 heads x all features would fill a whole register class
        if waves % vsplit or (p["ckv"] // 16) % (4 * vsplit):
            continue
        heads_per_block = 16 * hg * waves // vsplit
        if p["heads"] % heads_per_block:
            continue
        lds = mla_lds_bytes(p["ckv"], p["kpe"], stages)
        if lds > arch.lds_bytes:
            continue
        units_per = (d // 64) * 4 // min(waves, 4)
        if (stages - 2) * units_per >= 64:        # the wait for a step's loads counts the younger ones
            continue
        # Q fragments and accumulators of a wave's heads stay in registers for the whole split
        # (plus the ring of LDS operand reads and the softmax state); loads use no registers
        vgprs = hg * (d // 32 * 4 + p["ckv"] // 16 * 4 // vsplit + 4) + 32 + 24
        if vgprs > arch.vgprs_per_lane:
            continue
        blocks = p["batch"] * (p["heads"] // heads_per_block) * splits
        per_cu = arch.blocks_per_cu(waves * 64, lds, vgprs)
        if per_cu < 1:
            continue
        passes = _waves_time(blocks, per_cu, arch)
        steps = _ceil(_ceil(p["skv"], 32), splits)
        # per step and wave: the score operands are 1 KiB reads at about 32 B/clk and SIMD, the
        # value operands transposing reads at about two thirds of that; each feeds hg matrix ops
        score_reads, value_reads = 2 * (d // 32), p["ckv"] // 16 // vsplit
        mfma_clk = (score_reads + value_reads + 1) * hg * 18
        lds_clk = (score_reads * 32 + value_reads * 48) * 0.45     # measured: LDS reads hide under the matrix ops
        simd_share = max(1.0, per_cu * waves / 4.0)
        # measured: the matrix ops of a step plus about 1500 clocks that nothing overlaps (barrier,
        # load issue, the softmax between the two products); per workgroup of heads_per_block heads
        step_clk = (max(mfma_clk, lds_clk) * simd_share / per_cu + 1500) * (64.0 / heads_per_block)
        util = min(1.0, blocks / (per_cu * arch.compute_units))
        # a step's loads have (stages - 1) steps of matrix work to arrive in
        latency_clk = 4000.0 / (stages - 1)
        step_clk = max(step_clk, latency_clk)
        # split partials go out and come back once
        partial_bytes = 2 * splits * p["batch"] * p["heads"] * p["ckv"] * (2 if mla_po_elem(p["heads"]) else 4)
        partial_clk = partial_bytes / (arch.hbm_gbps * 1e3 * 0.6) * 2400 if splits > 1 else 0.0
        score = passes * steps * step_clk * (1.0 + 0.3 * (1 - util)) + 8000 + partial_clk
        out.append(TileDict("mla_decode", role, dict(WAVES=waves, HG=hg, VSPLIT=vsplit, STAGES=stages),
                            output_tile=[heads_per_block, p["ckv"]], rstep_map={"kv": 32}, n_threads=waves * 64,
                            split_factor=factor, score=score, lds_bytes=lds, est_vgprs=vgprs))
    # The score-wave / value-wave form: eight waves own 64 heads, every LDS operand feeds two matrix
    # ops.  Measured 25-30 % ahead of the best form above wherever both run, so it is ranked first
    # (with the shorter read-ahead of its value operands as a second candidate).
    duo_lds = mla_duo_lds_bytes(p["ckv"], p["kpe"])
    if out and p["heads"] % 64 == 0 and mla_duo_fits(p["ckv"], p["kpe"]) and duo_lds <= arch.lds_bytes:
        best = min(c.score for c in out)
        # (third: the score waves ask for about half of every image's panels -- a wave that waits for the
        # path into the compute unit does not hold up the other wave of its SIMD, and the value
        # waves are the longer chain of a step; measured 1-2 % ahead)
        shared = max(1, (p["ckv"] + p["kpe"]) // 64 // 2)
        for tiling, rel in ((dict(DUO=1), 0.75), (dict(DUO=1, LDS_AHEAD=4), 0.76),
                            (dict(DUO=1, LDS_AHEAD=4, S_PANELS=shared), 0.755)):
            out.append(TileDict("mla_decode", role, tiling, output_tile=[64, p["ckv"]], rstep_map={"kv": 32},
                                n_threads=512, split_factor=factor, score=rel * best, lds_bytes=duo_lds, est_vgprs=208))
    if role == "main" and not p.get("emit_lse") and out:
        out += mla_key_ranges(p, min(out, key=lambda c: (c.score, c.key())), arch)
    return out


def mla_key_ranges(p, base, arch: Arch):
    """Latent attention of too few workgroups for the chip: the keys dealt out to ranges inside an unsplit operator, f32 partials
    in scratch, folded by a second launch.  As many ranges as give every compute unit the workgroups it holds, and one or half a
    workgroup each: requests x heads x keys, us, one range / ranges: 3 x 16 x 7233 345 / 15.5 (57; 30 with 16), 24 x 16 x 2869 156 / 24.1
    (18; 28.1 with 10, 39.4 with 5), 2 x 16 x 639 34 / 8.2 (20; 9.9 with 10), 6 x 128 x 7649 198 / 28.8 (20; 34.0 as the split form
    at 8).  The split form, where a program asks for it, stays ahead for multiples of 64 heads on few keys, whose partials it halves
    by keeping them in 16 bits: 4 x 64 x 1819 15.7 (8) against 17.7 (12)."""
    rows, steps = p["batch"] * p["heads"], _ceil(p["skv"], 32)
    blocks = p["batch"] * _ceil(p["heads"], base.output_tile[0])
    out, seen = [], set()
    per_cu = min(2, max(1, arch.blocks_per_cu(base.n_threads, base.lds_bytes, base.est_vgprs)))
    for fill in sorted({arch.compute_units * per_cu, arch.compute_units, arch.compute_units // 2}, reverse=True):
        n = min(fill // blocks, steps, 64)
        n = _ceil(steps, _ceil(steps, n)) if n > 1 else 0              # (no empty ranges)
        if n > 1 and n not in seen and n * rows * (p["ckv"] + 2) * 4 + 3 * 256 <= FIXED_SCRATCH:
            seen.add(n)
            tiling = dict(base.tiling, KEYS=n)
            out.append(TileDict(base.template, base.role, tiling, output_tile=base.output_tile, rstep_map=base.rstep_map, n_threads=base.n_threads,
                                score=base.score / n, lds_bytes=base.lds_bytes, est_vgprs=base.est_vgprs, late=True))
    return out


# ----------------------------------------------------------------------------- combine kernels
def combine_candidates(low, factor, arch: Arch):
    """The combine of a split has one shape: one thread per 4 (attention) or 4/8 (matmul)
    output columns, 256 threads; it is memory-trivial next to its partial."""
    family = {"matmul": "gemm", "rmsnorm_matmul": "gemm", "lora": "gemm", "attention": "attn_decode",
              "mla": "mla_decode"}[low.family]
    return [TileDict(family, "combine", {}, output_tile=[1, 256], rstep_map={"split": factor}, n_threads=256,
                     split_factor=factor, score=1.0, lds_bytes=0, est_vgprs=32)]
