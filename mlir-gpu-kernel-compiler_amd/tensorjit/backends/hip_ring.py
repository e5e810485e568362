"""Ring schedule of the MFMA GEMM: a ring of LDS stages filled by DMA (``MatmulConfig.STAGES``).

The direct-to-LDS schedule (``direct_loop_lines``) is built for products that fill the chip
with 128-256 wide tiles: two LDS stages, one wave per SIMD, loads about one K tile ahead.
A product with few output tiles (a batched decode step, a short prompt, a small model's
layers) is bound by how many bytes each CU has in flight against the latency of HBM and L2,
not by the matrix cores.  This schedule takes small tiles, ``STAGES`` K tiles of 128-byte rows
deep in LDS -- so ``STAGES - 1`` tiles are in flight per workgroup -- and splits K over
``KSPLIT`` workgroups where the tiles alone leave CUs idle.  It also takes what the
direct-to-LDS schedule does not: B stored ``[K][N]`` and K that is no multiple of the K tile
(whole 16-byte chunks of the rows are enough).

One barrier per K tile ``t``: every wave first waits for its own loads of tile ``t`` (vmcnt: the
loads of tiles t+1 .. t+STAGES-2 may stay in flight), then the barrier publishes the tile and
frees the stage of tile t-1, whose fragment reads every wave has consumed; the loads of tile
t+STAGES-1 go into that stage, and the MFMAs of tile t run.

LDS layouts (16-byte chunks, applied by choosing which chunk each lane fetches):

* rows of K (A, and B of an NT product): chunk ``c`` of row ``r`` at ``c ^ (r & 7) ^ ((r >> 3) & 3)``
  and k-group g of a sub-step reads chunk 4 ks + sigma(g), sigma swapping g's bits, as the
  direct-to-LDS schedule's 16x16x32 form does (no two lanes of a half wave share a bank).
* rows of N (B of an NN product), 16-bit: the fragment is gathered by two
  ``ds_read_b64_tr_b16`` per 8 k; a half wave reads 8 rows (r & 3, bit 4 of r) x 32 bytes,
  so the 32-byte unit u of row r sits at u ^ swizzle(r) with swizzle taken from those bits:
  the 8 rows land on 8 different units of 256 bytes.
* rows of N, fp32: one 4-byte read per MFMA; unit u (64 bytes) of row r at u ^ ((r >> 2) & 3).
"""
from __future__ import annotations

from ..ir import DType

OOB = "0x80000000u"      # a byte offset past every descriptor's range: the load returns zeros
NW_MAX_VMCNT = 63
WAVE_SYNC = '  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier();'


def ring_ok(cfg, dt: DType) -> bool:
    """Tile constraints of the ring schedule (independent of the product)."""
    vk = 16 // dt.itemsize
    nw = cfg.num_warps
    batch = (cfg.TM + cfg.TN) // (8 * nw)
    return (cfg.MI == 16 and cfg.TK * dt.itemsize == 128 and cfg.SPLIT_K == 1 and nw in (4, 8)
            and not (cfg.PINGPONG or cfg.INTERLEAVE or cfg.DIRECT or cfg.PERSIST) and 3 <= cfg.STAGES <= 4
            and cfg.WM * cfg.WN == nw and cfg.TM % (16 * cfg.WM) == 0 and cfg.TN % (16 * cfg.WN) == 0
            and cfg.TM % (8 * nw) == 0 and cfg.TN % (8 * nw) == 0 and cfg.TN & (cfg.TN - 1) == 0
            and cfg.STAGES * (cfg.TM + cfg.TN) * 128 + 64 <= 160 * 1024
            and batch * (cfg.STAGES - 1) <= NW_MAX_VMCNT
            # epilogue staging: one 16-row block of a wave's columns in one stage array
            and 16 * (cfg.TN // cfg.WN + 4) * 4 <= min(cfg.TM, cfg.TN) * 128 and nw <= 2 * cfg.STAGES
            and (cfg.TN // cfg.WN) % vk == 0)


def ring_fits(cfg, dt: DType, M: int, N: int, K: int, tb: bool, batch: int) -> bool:
    """Does a product of this shape fit the ring schedule: whole 16-byte chunks along the
    contiguous dim of both operands, 31-bit byte offsets, a K split whose every part has a
    K tile, and a workspace within the descriptor's range."""
    e = dt.itemsize
    vk = 16 // e
    if K % vk or (not tb and N % vk):
        return False
    b_bytes = (N + cfg.TN) * K * e if tb else (K + cfg.TK) * N * e
    if (M + cfg.TM) * K * e >= 2**31 or b_bytes >= 2**31:
        return False
    kt = -(-K // cfg.TK)
    S = cfg.KSPLIT
    if S > 1:
        per = -(-kt // S)
        tiles = -(-M // cfg.TM) * -(-N // cfg.TN)
        if (S - 1) * per >= kt or batch * S * tiles * cfg.TM * cfg.TN * 4 >= 2**31:
            return False
    return True


def _wait_barrier(vm: int) -> list[str]:
    """All but this wave's ``vm`` youngest DMA loads have landed and its fragment reads are
    done, then the workgroup barrier (a plain ``s_barrier``: the fence of ``__syncthreads``
    waits for every load in flight)."""
    assert 0 <= vm <= NW_MAX_VMCNT
    imm = (vm & 15) | ((vm >> 4) << 14) | 0x70
    return ["__builtin_amdgcn_sched_barrier(0);", f"__builtin_amdgcn_s_waitcnt({hex(imm)});",
            "__builtin_amdgcn_s_barrier();", "__builtin_amdgcn_sched_barrier(0);"]


def ring_loop_lines(cfg, dt: DType, M: int, N: int, K: int, tb: bool, opvec: str, builtin: str) -> list[str]:
    """Accumulators ``acc[TMW][TNW]`` of this workgroup's tile (its share of K when split)."""
    e = dt.itemsize
    f32 = dt == DType.f32
    vk = 16 // e
    nw, NS, S = cfg.num_warps, cfg.STAGES, cfg.KSPLIT
    BM, BN, BK = cfg.TM, cfg.TN, cfg.TK
    TMW, TNW = BM // cfg.WM // 16, BN // cfg.WN // 16
    KT = -(-K // BK)
    KTs = -(-KT // S)                       # K tiles of one part (the last may run past K: zeros)
    guard_k = K % BK != 0 or KTs * S != KT
    a_cnt, b_cnt = BM // (8 * nw), BN // (8 * nw)
    n_batch = a_cnt + b_cnt
    L = []
    for s in range(NS):
        L.append(f"  __shared__ __attribute__((aligned(1024))) char As{s}[{BM * 128}];")
        L.append(f"  __shared__ __attribute__((aligned(1024))) char Bs{s}[{BN * 128}];")
    L += ["  const unsigned int wv = __builtin_amdgcn_readfirstlane(wave);",
          "  const unsigned int drow = lane >> 3;",
          f"  tj_f32x4 acc[{TMW}][{TNW}];",
          "#pragma unroll", f"  for (int x = 0; x < {TMW}; ++x)", "#pragma unroll",
          f"    for (int y = 0; y < {TNW}; ++y) acc[x][y] = (tj_f32x4)(0.0f);"]
    if S > 1:
        L.append(f"  const unsigned int ksp = blockIdx.z % {S}u, kt0 = ksp * {KTs}u;")
    t0 = "kt0 + " if S > 1 else ""
    # ---- DMA: one instruction fills 1 KiB of LDS (lane i at byte 16 i) ----------------
    b_range = N * K * e
    L.append(f"  const __amdgpu_buffer_rsrc_t rsA = __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, {M * K * e}, 0x00020000);")
    L.append(f"  const __amdgpu_buffer_rsrc_t rsB = __builtin_amdgcn_make_buffer_rsrc((void*)Bb, (short)0, {b_range}, 0x00020000);")
    # rows of K: eight 128-byte rows per instruction; the chunk a lane fetches (and so its k
    # within the tile) is the same for every instruction of a wave, as nw % 4 == 0
    L.append(f"  const unsigned int dk = ((lane & 7u) ^ drow ^ (wv & 3u)) * {vk}u;")
    L.append(f"  unsigned int voA[{a_cnt}], voB[{b_cnt}];")
    for i in range(a_cnt):
        L.append(f"  voA[{i}] = ((m0 + ({i * nw}u + wv) * 8u + drow) * {K}u + dk) * {e}u;")
    if tb:
        for i in range(b_cnt):
            L.append(f"  voB[{i}] = ((n0 + ({i * nw}u + wv) * 8u + drow) * {K}u + dk) * {e}u;")
    else:
        cpr = BN * e // 16                  # 16-byte chunks per row of N
        unit = 4 if f32 else 2              # chunks per swizzle unit (64 / 32 bytes)
        sw = _nn_swizzle("dkr", BN, f32)
        L.append(f"  unsigned int krB[{b_cnt}];")
        for i in range(b_cnt):
            L.append(f"  {{ const unsigned int P = ({i * nw}u + wv) * 64u + lane, dkr = P / {cpr}u, "
                     f"c = (P % {cpr}u) ^ (({sw}) * {unit}u), col = n0 + c * {vk}u;")
            L.append(f"    krB[{i}] = dkr; voB[{i}] = col < {N}u ? (dkr * {N}u + col) * {e}u : {OOB}; }}")

    def dma(t: str, stage: int) -> list[str]:
        out = ["{", f"  const unsigned int kt = {t0}({t});"]
        if guard_k:
            out.append(f"  const unsigned int kleft = kt * {BK}u < {K}u ? {K}u - kt * {BK}u : 0u;")
            if KTs * S > KT:
                # tiles past the end (a part with fewer K tiles): every lane's offset is OOB, and
                # the scalar offset stays inside the descriptor, whose range check may subtract it
                out[1] = out[1].replace("kt = ", "kf = ")
                out[2] = out[2].replace("kt *", "kf *")
                out.append(f"  const unsigned int kt = kf < {KT}u ? kf : {KT - 1}u;")
        for op, cnt in (("A", a_cnt), ("B", b_cnt)):
            row_k = op == "A" or tb
            step = BK * e if row_k else BK * N * e
            for i in range(cnt):
                vo = f"vo{op}[{i}]"
                if guard_k:
                    vo = f"({'dk' if row_k else f'krB[{i}]'} < kleft ? {vo} : {OOB})"
                out.append(f"  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs{op}, (__attribute__((address_space(3))) void*)"
                           f"({op}s{stage} + ({i * nw}u + wv) * 1024u), 16, {vo}, (int)(kt * {step}u), 0, 0);")
        return out + ["}"]

    # ---- fragment reads ------------------------------------------------------------------
    # f(r) of row wave base + 16 x + fr: (fr & 7) ^ ((fr >> 3) | 2 * (bit 4 of the row))
    L += ["  const unsigned int fr = lane & 15u, fh = lane >> 4, fg = ((fh & 1u) << 1) | (fh >> 1);",
          "  const unsigned int fsw = (fr & 7u) ^ (fr >> 3);",
          f"  const unsigned int arow = (wm * {BM // cfg.WM}u + fr) * 128u;"]
    KS = 2                                  # 64-byte sub-steps per 128-byte K row

    def kofs(name: str, tiles: int, wave_id: str) -> list[str]:
        """Byte offsets in a K row of sub-step ks for even / odd 16-row blocks of the wave."""
        odd = f" ^ (({wave_id} & 1u) << 1)" if tiles % 2 else ""
        return [f"  const unsigned int {name}{ks}{par} = (({4 * ks}u + fg) ^ fsw ^ {2 * par}u{odd}) * 16u;"
                for ks in range(KS) for par in range(2)]

    L += kofs("ao", TMW, "wm")
    if tb:
        L.append(f"  const unsigned int brow = (wn * {BN // cfg.WN}u + fr) * 128u;")
        L += kofs("bo", TNW, "wn")
    elif f32:
        L.append(f"  unsigned int bo[{TNW}];      // row 4 sigma(g) (its swizzle is sigma(g)), column 16 y + fr")
        nunit = BN // 16
        L.append("#pragma unroll")
        L.append(f"  for (int y = 0; y < {TNW}; ++y) bo[y] = fg * {4 * BN * 4}u + "
                 f"(((wn * {TNW}u + y) ^ (fg & {min(3, nunit - 1)}u)) * 16u + fr) * 4u;")
    else:
        L.append("  const unsigned int te = (lane & 15u) >> 2, tm_ = lane & 3u, tkr = fg * 8u + te;")
        L.append(f"  unsigned int bo[{TNW}];")
        L.append("#pragma unroll")
        L.append(f"  for (int y = 0; y < {TNW}; ++y) bo[y] = tkr * {BN * 2}u + "
                 f"(((wn * {TNW}u + y) ^ ({_nn_swizzle('tkr', BN, False)})) * 32u) + tm_ * 8u;")

    def compute(stage: int) -> list[str]:
        out = ["{", f"  {opvec} fa[{KS}][{TMW}], fb[{KS}][{TNW}];"]
        for ks in range(KS):
            for x in range(TMW):
                out.append(f"  fa[{ks}][{x}] = *(const {opvec}*)(As{stage} + arow + ao{ks}{x & 1} + {x * 2048}u);")
            for y in range(TNW):
                if tb:
                    out.append(f"  fb[{ks}][{y}] = *(const {opvec}*)(Bs{stage} + brow + bo{ks}{y & 1} + {y * 2048}u);")
                elif f32:
                    for j in range(4):
                        out.append(f"  fb[{ks}][{y}][{j}] = *(const float*)(Bs{stage} + bo[{y}] + {(16 * ks + j) * BN * 4}u);")
                else:
                    rd = ("__builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tj_i16x4*)"
                          f"(Bs{stage} + bo[{y}] + ")
                    base = 32 * ks * BN * 2
                    out.append(f"  {{ const tj_i16x4 lo = {rd}{base}u)), hi = {rd}{base + 4 * BN * 2}u));")
                    out.append(f"    fb[{ks}][{y}] = __builtin_bit_cast({opvec}, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)); }}")
        for ks in range(KS):
            for j in range(4 if f32 else 1):
                el = f"[{j}]" if f32 else ""
                for x in range(TMW):
                    for y in range(TNW):
                        out.append(f"  acc[{x}][{y}] = {builtin}(fa[{ks}][{x}]{el}, fb[{ks}][{y}]{el}, acc[{x}][{y}], 0, 0, 0);")
        return out + ["}"]

    # ---- pipeline ------------------------------------------------------------------------
    ahead = min(NS - 1, KTs)
    for t in range(ahead):
        L += ["  " + x for x in dma(f"{t}u", t)]

    def tile(t: str, tc: int, ind: str) -> list[str]:
        """K tile ``t`` (``tc``: its index, -1 in the loop, whose tiles all load ahead)."""
        left = NS if tc < 0 else KTs - tc                  # tiles not yet computed, this one included
        out = _wait_barrier(n_batch * min(NS - 2, left - 1))
        stage = tc % NS if tc >= 0 else int(t.split("+")[1].rstrip("u")) % NS
        if left >= NS:
            out += dma(f"{t} + {NS - 1}u", (stage + NS - 1) % NS)
            out.append("__builtin_amdgcn_sched_barrier(0);")
        return [ind + x for x in out + compute(stage)]

    nload = max(0, KTs - (NS - 1))                         # tiles that load ahead
    rounds = nload // NS if nload // NS > 1 else 0
    if rounds:
        L.append(f"  for (unsigned int kt_ = 0; kt_ < {rounds * NS}u; kt_ += {NS}u) {{")
        for j in range(NS):
            L += tile(f"kt_ +{j}u", -1, "    ")
        L.append("  }")
    for t in range(rounds * NS, KTs):
        L += tile(f"{t}u", t, "  ")
    return L


def _nn_swizzle(row: str, BN: int, f32: bool) -> str:
    """Swizzle of row ``row`` of an NN product's B stage, in units of 32 bytes (16-bit) or
    64 bytes (fp32)."""
    if f32:
        return f"(({row} >> 2) & {min(3, BN // 16 - 1)}u)"
    if BN >= 128:
        return f"(({row} & 3u) | ((({row} >> 4) & 1u) << 2))"
    if BN == 64:
        return f"((({row} >> 1) & 1u) | ((({row} >> 4) & 1u) << 1))"
    return f"(({row} >> 4) & 1u)"


def ring_split_lines(cfg, ntm: int, ntn: int, batch: int, bi: str) -> list[str]:
    """K split over workgroups: every workgroup stores its accumulators to the workspace as
    they lie in its registers (16 bytes per lane, 1 KiB per wave and store), and the last
    of a tile's workgroups to count itself adds the parts in split order and goes on to the
    epilogue with the sums in ``acc``.

    The stores and loads are agent-coherent (sc1: past this XCD's L2), each wave waits for
    its stores before the workgroup barrier in front of the count, and the counters (at the
    head of the stream's workspace block, zero when it is allocated) wrap to zero at the last
    count of a launch.  They are never stored to: whole launches that overlap in any order, which
    only a caller that breaks run_static's rule can bring about, still leave them at zero, so
    the damage ends with those launches."""
    S, nw = cfg.KSPLIT, cfg.num_warps
    TMW, TNW = cfg.TM // cfg.WM // 16, cfg.TN // cfg.WN // 16
    part = cfg.TM * cfg.TN * 4
    ws_bytes = batch * S * ntm * ntn * part
    L = [f"  const __amdgpu_buffer_rsrc_t rsW = __builtin_amdgcn_make_buffer_rsrc((void*)ws_p, (short)0, {ws_bytes}, 0x00020000);",
         f"  const unsigned int ct_ = ({bi} * {ntm}u + m0 / {cfg.TM}u) * {ntn}u + n0 / {cfg.TN}u;",
         f"  const unsigned int wo_ = ct_ * {S * part}u + tid * 16u;"]
    slot = lambda x, y: (x * TNW + y) * nw * 1024   # noqa: E731
    for x in range(TMW):
        for y in range(TNW):
            L.append(f"  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(tj_u32x4, acc[{x}][{y}]), rsW, "
                     f"(int)(wo_ + ksp * {part}u + {slot(x, y)}u), 0, 16);")
    L += ["  __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): this wave's partial stores are done",
          "  __shared__ unsigned int tj_last_;",
          "  __syncthreads();",
          f"  if (tid == 0u) tj_last_ = atomicInc(&cnt_p[ct_], {S - 1}u) == {S - 1}u ? 1u : 0u;   // {S - 1} wraps to 0",
          "  __syncthreads();",
          "  if (tj_last_ == 0u) return;"]
    for x in range(TMW):
        for y in range(TNW):
            L.append(f"  acc[{x}][{y}] = (tj_f32x4)(0.0f);")
    L += ["#pragma unroll", f"  for (unsigned int s = 0; s < {S}u; ++s) {{"]
    for x in range(TMW):
        for y in range(TNW):
            L.append(f"    {{ const tj_f32x4 p = __builtin_bit_cast(tj_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsW, "
                     f"(int)(wo_ + s * {part}u + {slot(x, y)}u), 0, 16));")
            L.append(f"      acc[{x}][{y}][0] += p[0]; acc[{x}][{y}][1] += p[1]; acc[{x}][{y}][2] += p[2]; acc[{x}][{y}][3] += p[3]; }}")
    L.append("  }")
    return L


def ring_epilogue_lines(cfg, out_dts, N: int, M: int, guard_m: bool, guard_n: bool, idx_t: str, run_lines) -> list[str]:
    """Epilogue: wave w stages its sub-tile through one stage array of its own, a 16-row MFMA
    block at a time (a wave's LDS accesses complete in order: no barrier after the first),
    and each lane takes 16-byte runs of output rows.  ``run_lines(ve, cs)`` gives the
    statements for one run at (i, j)."""
    nw = cfg.num_warps
    TMW, TNW = cfg.TM // cfg.WM // 16, cfg.TN // cfg.WN // 16
    cols = TNW * 16
    ldc = cols + 4
    one = all(d == out_dts[0] for d in out_dts)
    vk = 16 // out_dts[0].itemsize
    ve = vk if one and N % vk == 0 and cols % vk == 0 else 1
    per_row = cols // ve
    arrays = [f"{op}s{s}" for s in range(cfg.STAGES) for op in "AB"][:nw]
    sel = arrays[-1]
    for w in range(nw - 2, -1, -1):
        sel = f"wave == {w}u ? {arrays[w]} : {sel}"
    # lanes exchange values through Cw within a wave: the wave barriers keep the compiler from
    # running one branch of a divergent condition (few runs per row, tile edges) through
    # several blocks before the other lanes' branch
    sync = [WAVE_SYNC]
    L = ["  __syncthreads();", f"  float* Cw = (float*)({sel});"]
    for x in range(TMW):
        L += sync if x else []
        L += ["#pragma unroll", f"  for (int y = 0; y < {TNW}; ++y)", "#pragma unroll", "  for (int r = 0; r < 4; ++r)",
              f"    Cw[((lane / 16u) * 4u + r) * {ldc}u + y * 16u + lane % 16u] = acc[{x}][y][r];",
              *sync, "#pragma unroll", f"  for (unsigned int c = lane; c < {16 * per_row}u; c += 64u) {{",
              f"    const unsigned int lr = c / {per_row}u, cc = (c % {per_row}u) * {ve}u;",
              f"    const {idx_t} i = m0 + wm * {cfg.TM // cfg.WM}u + {x * 16}u + lr;",
              f"    const {idx_t} j = n0 + wn * {cfg.TN // cfg.WN}u + cc;"]
        conds = ([f"i < {M}u"] if guard_m else []) + ([f"j < {N}u"] if guard_n else [])
        if conds:
            L.append(f"    if (!({' && '.join(conds)})) continue;")
        L += run_lines(ve, f"Cw[lr * {ldc}u + cc + q]")
        L.append("  }")
    return L
