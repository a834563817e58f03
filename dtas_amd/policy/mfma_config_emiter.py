"""Tile candidates for the dynamic-M GEMM on the MFMA matrix cores.

Plays the part of the reference's WMMAConfigEmiter (python/dtas/policy/wmma_config_emiter.py:15-353):
enumerate block tiles as i x j wavefronts of micro_x x micro_y matrix-core blocks (:72-115), drop
those that do not fit shared memory / registers (:46-70) and rank by a roofline estimate in which a
tile's throughput is min(matrix-core peak, bandwidth * flops-per-byte of the tile) and the job costs
ceil(tiles / SMs) rounds (:148-262).  The candidate set is what libdtas_gfx950.so has kernels for:
MFMA tiles from 64x64 to 256x256 (16x16x32 on 8 wavefronts, 32x32x16 on 4) with 2 to 4 LDS stages, with K split over up to 4 workgroups
per tile when M x N yields few tiles, plus, for M <= 64, the weight-streaming 16x16x32 kernel whose
wavefronts split K.  The order is the one on-GPU sweeps favoured;
with a GPU present the Engine times the top-k anyway.
"""
from typing import List, Tuple

from ..common.config import MFMAConfig, Range
from .base_config_emiter import BaseConfigEmiter

# (micro_x, micro_y) per wavefront of the 2x2-wavefront kernels
_TILES = [(4, 2), (2, 4), (2, 2), (1, 2), (2, 1), (1, 1)]
# the 8-wavefront kernels: tile -> (wavefronts along M, along N)
_TILES8 = {(256, 256): (2, 4), (224, 256): (2, 4), (192, 256): (2, 4), (160, 256): (2, 4), (128, 256): (2, 4), (96, 256): (2, 4),
           (256, 128): (4, 2), (224, 128): (2, 4), (192, 128): (4, 2), (160, 128): (2, 4), (128, 128): (4, 2), (96, 128): (2, 4), (128, 64): (4, 2)}
# the library's cost model beyond 128 rows (libdtas: kTile8Cost): tile, threads, stages, whether the table's rows name it, and
# a, b, w, r, h0, h1, h2, pitch, pow2, few, pad
_COST8 = [
    (64, 64, 256, 4, True, 3.57, 0.29, 0.478, 0.717, 0.524, 0.734, 0.129, 1.088, 1.009, 0.574, 0.47),
    (128, 64, 512, 0, True, 2.631, 0.403, 1.476, 0.909, 2.034, 0.637, 0.653, 1.108, 0.961, 0.203, 0.153),
    (96, 128, 512, 0, False, 3.519, 0.476, 0.746, 0.809, 1.266, 0.975, 1.735, 1.107, 0.98, 0.614, 0.623),
    (128, 128, 512, 0, True, 3.291, 0.544, 1.551, 0.823, 0.877, 1.463, 2.133, 1.071, 0.951, 0.485, 0.404),
    (160, 128, 512, 0, False, 3.721, 0.611, 0.409, 0.902, 1.024, 1.727, 4.122, 1.08, 0.968, 0.377, 0.217),
    (192, 128, 512, 0, True, 4.008, 0.677, 0.586, 0.909, 1.074, 2.066, 5.196, 1.085, 0.974, 0.301, 0.201),
    (224, 128, 512, 0, False, 4.428, 0.766, 0, 0.849, 2.076, 2.391, 3.818, 1.088, 0.968, 0.232, 0.231),
    (256, 128, 512, 0, True, 5.651, 0.874, 0, 0.737, 1.586, 2.705, 3.646, 1.051, 0.932, 0.223, 0.316),
    (96, 256, 512, 0, False, 3.125, 0.722, 1.919, 0.88, 1.049, 1.981, 2.592, 1.096, 0.96, 0.948, 0.41),
    (128, 256, 512, 0, False, 5.289, 0.846, 0, 0.692, 0.862, 2.651, 2.37, 1.081, 0.954, 0.889, 0.566),
    (160, 256, 512, 0, False, 5.914, 0.99, 0.447, 0.675, -0.599, 3.146, 6.082, 1.054, 0.979, 0.584, 0.593),
    (192, 256, 512, 0, True, 7.283, 1.152, 0.273, 0.69, 0.249, 2.667, 7.583, 1.039, 0.966, 0.497, 0.537),
    (224, 256, 512, 0, False, 7.123, 1.294, 0.808, 0.652, 1.88, 2.796, 4.098, 1.025, 0.983, 0.407, 0.415),
    (256, 256, 512, 2, True, 8.473, 1.449, 0.41, 0.613, -1.316, 4.31, 8.162, 1.011, 0.984, 0.311, 0.395),
    (192, 256, 512, 2, True, 6.715, 1.142, 0.592, 0.663, 2.39, 3.56, 3.96, 1.063, 0.96, 0.508, 0.209),
]
_LDS = 160 * 1024


class MFMAConfigEmiter(BaseConfigEmiter):
    def check_valid(self, c: MFMAConfig) -> bool:
        if c.block_threads == 512:   # the 8-wavefront kernels are built to fit
            return (c.tile_size_m, c.tile_size_n) in _TILES8
        stages = c.stages or 2
        lds = stages * (c.tile_size_m + c.tile_size_n) * c.tile_size_k * 2  # fp16 stages of the load pipeline
        acc = c.micro_shape_x * c.micro_shape_y * 16                         # fp32 accumulators per lane
        return lds <= self.arch.max_smem_per_block and acc <= 256

    @staticmethod
    def max_stages(tile_m: int, tile_n: int) -> int:
        return 2 if tile_m + tile_n >= 512 else 3 if tile_m + tile_n >= 384 else 4

    @staticmethod
    def row_pitch(K: int) -> str:
        """How far apart rows of K lie, as the cost model sees it (libdtas: row_pitch): 'slow' 3 x 2^j or 5 x 2^j KiB, 'pow2' a
        power of two from 4 KiB, '' otherwise."""
        if K >= 2048 and K & (K - 1) == 0:
            return "pow2"
        odd = K
        while odd and odd % 2 == 0:
            odd //= 2
        return "slow" if K % 512 == 0 and odd in (3, 5) else ""

    def tile8_policy(self, M: int, N: int, K: int):
        """(tile_m, tile_n, stages, split_k, threads) of the table's row beyond 128 rows: the cost model of the library's
        tile8_policy, over the tiles and splits the table's rows name (a host test keeps the two alike)."""
        cdiv = lambda a, b: -(-a // b)
        cus, ktiles = self.arch.num_sm, cdiv(K, 64)
        pitch_class = self.row_pitch(K)
        best_us, best = 1e300, None
        for bm, bn, threads, stages, in_table, a, b0, w, r, h0, h1, h2, pitch, pow2, few, pad in _COST8:
            if not in_table or K * 2 * max(bm, bn) >= 1 << 31:
                continue
            tm = cdiv(M, bm)
            ring_192 = bm == 192 and stages == 2
            if ring_192 and pitch_class != "pow2":
                continue
            tiles = tm * cdiv(N, bn)
            if tiles > 0x7fffffff // 8:
                continue
            whole_rounds = bm == 256 and bn == 256
            slots = 2 * cus if bm * bn <= 64 * 64 else cus
            b = b0 * (pitch if pitch_class == 'slow' else pow2 if pitch_class == 'pow2' else 1.0) * (1.0 + few / float(tm) - pad * (1.0 - float(M) / float(tm * bm)))
            for parts in range(1, 2 if ring_192 else 5):
                last_parts = parts
                if whole_rounds:
                    last_parts, _ = self.tail_split_256(M, N, K)
                elif parts > 1 and (tiles * parts > slots or ktiles // parts < 8 or tiles * parts * bm * bn * 4 > 32 << 20):
                    break
                tail = whole_rounds and last_parts > 1
                wgs = tiles if whole_rounds else tiles * parts
                full, rem = divmod(wgs, slots)
                steps = float(ktiles if whole_rounds else cdiv(ktiles, parts))
                share = float(wgs) / cus
                us = float(full) * (a + b * steps) + w * share
                fill = float(rem * last_parts if whole_rounds else rem) / float(slots)
                if slots > cus:     # (64x64: two or more workgroups share a CU)
                    us = a + b * steps * (r + (1.0 - r) * share if wgs <= cus else 0.75 * float(cdiv(wgs, cus))) + w * share
                elif rem > 0:
                    us += a + b * (float(cdiv(ktiles, last_parts)) if whole_rounds else steps) * (r + (1.0 - r) * fill)
                if last_parts > 1:
                    crowd = fill if whole_rounds else share
                    us += h0 + h1 * last_parts + h2 * crowd * crowd * crowd * crowd
                if us < best_us:
                    best_us, best = us, (bm, bn, stages, 0 if tail else parts, threads)
                if whole_rounds:
                    break
        self._model_us = best_us
        return best

    def preferred(self, m_hi: int, N: int, K: int = 4096):
        """(tile_m, tile_n, stages, split_k, threads) under the cost models fitted to sweeps on an MI355X (the same
        ones the library's built-in table uses).  Beyond 128 rows: tile8_policy.  Up to 128 rows: time = rounds of workgroups
        over the chip x time of one k tile x k tiles.  One k tile with every CU busy: 128x128 0.665 us (4 stages, one workgroup
        per CU) or 1.14 us per round of two per CU (2 stages); a partly filled round costs 0.55 + 0.45 * fill of a full
        one (0.8 + 0.2 * fill for 128x128 with 4 stages in a single round); 64x64 0.33 us per k tile up to one workgroup per CU,
        x 0.82 * (workgroups on the fullest CU) beyond; with few tiles K is split over up to 4 workgroups per tile at ~4 us
        (128x128) / ~1 us (64x64; 2.5 us with more than one per CU) per partial tile; 128x64 (4 stages, at most one workgroup
        per CU) 0.47 us per k tile whatever the fill and ~2.5 us per partial tile.  No candidate is faster than W (2NK bytes) streams through it: 3.1 .. 4.3 TB/s
        by tile, measured with 64 rows against a 50280 x 2560 W."""
        if m_hi > 128:
            wide = self.tile8_policy(m_hi, N, K)
            if wide:
                return wide
        cdiv = lambda a, b: -(-a // b)
        cus = self.arch.num_sm
        ktiles = cdiv(K, 64)

        def rounds(wgs, slots):
            full, rem = divmod(wgs, slots)
            return full + ((0.55 + 0.45 * rem / slots) if rem else 0.0)

        tiles = lambda bm, bn: cdiv(m_hi, bm) * cdiv(N, bn)
        w_mb = 2.0 * float(N) * float(K) * 1e-6
        # W streams at 3.1 .. 4.3 TB/s, by tile; candidates that all sit on that floor are told apart by their own estimates
        floored = lambda us, tbs: (us if us > w_mb / tbs else w_mb / tbs) + 1e-3 * us
        cands = [(floored(rounds(tiles(128, 128), 2 * cus) * 1.14 * ktiles, 3.1), (128, 128, 2, 1))]
        for split in (1, 2, 3, 4):
            if split > 1 and (ktiles // split < 8 or ktiles <= 16):    # (K <= 1024: a hand-over costs what the shorter loop saves)
                continue
            steps = cdiv(ktiles, split)
            t128, t64 = tiles(128, 128) * split, tiles(64, 64) * split
            if split == 1 or t128 <= cus:
                cands.append((floored((0.8 + 0.2 * t128 / cus if t128 <= cus else rounds(t128, cus)) * 0.665 * steps
                                      + (4.0 * split if split > 1 else 0.0), 4.1 if split == 1 else 3.5), (128, 128, 4, split)))
            cands.append((floored((1.0 if t64 <= cus else 0.82 * -(-int(t64) // cus)) * 0.33 * steps
                                  + ((1.0 if t64 <= cus else 2.5) * split if split > 1 else 0.0), 4.3),
                          (64, 64, 4, split)))
            t12864 = tiles(128, 64) * split
            if t12864 <= cus:
                cands.append((floored(0.47 * steps + (2.5 * split if split > 1 else 0.0), 3.8), (128, 64, 4, split)))
        best = cands[0]
        for c in cands[1:]:          # first strict minimum, in the library's order of evaluation
            if c[0] < best[0]:
                best = c
        self._model_us = best[0]
        tm, tn, stages, split = best[1]
        return tm, tn, stages, split, 256

    def tail_split_256(self, M: int, N: int, K: int):
        """(parts, tiles left whole) for split_k = 0 on the 8-wavefront 256x256 tile: whole rounds of the chip
        run one workgroup per tile, the tiles of a last, partly filled round are shared by 2..4 workgroups each
        (as many as still fit the chip at once, each keeping 8 k tiles or more) -- unless the parts would fill more
        than three quarters of the chip and K is short (a partly filled round clocks higher; libdtas: tail_split_256)."""
        cdiv = lambda a, b: -(-a // b)
        cus = self.arch.num_sm
        tiles, ktiles = cdiv(M, 256) * cdiv(N, 256), cdiv(K, 64)
        rem = tiles % cus
        if rem == 0:
            return 1, 0
        split = min(cus // rem, 4)
        while split >= 2 and ktiles // split < 8:
            split -= 1
        if split >= 2 and rem * split > 3 * cus // 4 and ktiles < 128:
            return 1, 0
        if split < 2:
            return 1, 0
        return split, tiles - rem

    def prefers_stream(self, m_hi: int, N: int, K: int) -> bool:
        """M <= 32 and at most one workgroup per CU of the W-streaming kernel (M <= 16: 64 columns x 1024 of K each):
        measured 10.9 against 12.8 us at 4096 x 4096, 7.2 against 10.2 at 2560 x 2560; beyond one round of
        workgroups the tiles win again (libdtas: gemm_policy)."""
        if m_hi <= 16:
            return -(-N // 64) * -(-K // 1024) <= self.arch.num_sm
        # 17 .. 32 rows: 32 rows of A and 512 of K per workgroup, between a quarter of a round and one round of them
        # (8.4 against 9.8 us at 2560 x 2560, 11.4 / 13.9 at 1024 x 8192)
        # (from K = 2048 on: at 4096 x 1024 the 64x64 tiles take 7.4 us, this form 8.2)
        return m_hi <= 32 and K >= 2048 and self.arch.num_sm // 4 <= -(-N // 64) * -(-K // 512) <= self.arch.num_sm

    def prefers_stream_loop(self, m_hi: int, N: int, K: int) -> int:
        """Columns per workgroup (16 or 64) of the looping W-streaming kernel where it leads, else 0: M <= 16, K <= 4096
        and its workgroups fill one round of the chip -- two one-wavefront workgroups per CU for 4096 < N <= 8192, one
        4-wavefront workgroup per CU for 8192 <= N <= 16384 (15.9 against 20.2 us at 8192 x 4096, 20.4 / 24.5 at
        11008 x 4096; libdtas: gemm_policy)."""
        if m_hi > 16 or K > 4096 or self.prefers_stream(m_hi, N, K):
            return 0
        cu = self.arch.num_sm
        if cu < -(-N // 16) <= 2 * cu:
            return 16
        if cu // 2 <= -(-N // 64) <= cu:
            return 64
        return 0

    def prefers_skinny(self, m_hi: int, N: int, K: int) -> bool:
        """M <= 32: the W-streaming kernel (about 3.5 TB/s of W, slower as M grows) against the model's
        best MFMA candidate; call after preferred()."""
        if m_hi > 32:
            return False
        us = N * K * 2.0 / 3.5e6 * (0.9 if m_hi <= 8 else 0.95 if m_hi <= 16 else 1.35)
        wgs = -(-N // 16)               # one workgroup per 16 rows of W: fewer than one per CU leave CUs idle
        if wgs < self.arch.num_sm:
            us *= self.arch.num_sm / wgs
        return us <= self._model_us

    def emit_config(self, range_tuple: Tuple[Range, ...], topk: int = 20) -> List[MFMAConfig]:
        params = self.func_info.func.params
        N, K = params[1].shape
        if range_tuple:
            m_hi = range_tuple[0].end
        else:
            m_hi = 1
            for e in params[0].shape[:-1]:
                m_hi *= e
        out: List[MFMAConfig] = []
        stream: List[MFMAConfig] = []
        if m_hi <= 64:
            # the W-streaming kernel: rows of A x columns x K slice, (rows + columns) * slice * 2 bytes of LDS
            for cols, kslice in ((64, 1024), (64, 512), (128, 512)):
                rows = 16 if m_hi <= 16 else 32 if m_hi <= 32 else 64
                if (rows + cols) * kslice * 2 > _LDS or (rows == 64 and cols == 128):
                    continue
                c = MFMAConfig()
                c.stream, c.block_threads = True, 4 * cols
                c.i, c.j, c.micro_shape_x, c.micro_shape_y, c.micro_shape_k = 1, cols // 16, rows // 16, 1, kslice // 32
                c.mfma_m, c.mfma_n, c.mfma_k = 16, 16, 32
                stream.append(c)
        # the share kernel: every workgroup N / (number of CUs) columns over the whole of K.  The second candidate: the library
        # takes it for a call without a config where it leads at the M at hand (libdtas: share_leads), a line that the table's
        # rows, which a first candidate equals, do not draw -- only a timed tuning finds it here
        share: List[MFMAConfig] = []
        rows, cols = self.share_shape(m_hi, N)
        if rows:
            c = MFMAConfig()
            c.share = True
            c.i, c.j, c.micro_shape_x, c.micro_shape_y, c.micro_shape_k = 1, 1, rows // 16, cols // 16, 1
            c.mfma_m, c.mfma_n, c.mfma_k = 16, 16, 32
            share.append(c)
        loop: List[MFMAConfig] = []
        if m_hi <= 16:
            # its looping form (K slice 256 = the segment of the LDS ring; the whole of K per workgroup)
            for cols in (64, 16):
                c = MFMAConfig()
                c.stream, c.block_threads = True, 4 * cols
                c.i, c.j, c.micro_shape_x, c.micro_shape_y, c.micro_shape_k = 1, cols // 16, 1, 1, 8
                c.mfma_m, c.mfma_n, c.mfma_k = 16, 16, 32
                loop.append(c)
            lead = self.prefers_stream_loop(m_hi, N, K)
            loop.sort(key=lambda c: c.tile_size_n != lead)
        if m_hi <= 64:
            for threads in (512, 256):
                c = MFMAConfig()
                c.skinny, c.block_threads = True, threads
                c.i, c.j, c.micro_shape_x, c.micro_shape_y, c.micro_shape_k = 1, 1, -(-m_hi // 16), 1, 1
                c.mfma_m, c.mfma_n, c.mfma_k = 16, 16, 32
                out.append(c)
        pref = self.preferred(m_hi, N, K)
        scored = []
        shapes: List[MFMAConfig] = []
        for (tm, tn), (wm, wn) in _TILES8.items():
            # stages 0: what the LDS holds; 2: the ring of the largest tile, which 192x256 comes with too
            for st in ((2,) if (tm, tn) == (256, 256) else (0, 2) if (tm, tn) == (192, 256) else (0,)):
                c = MFMAConfig()
                c.i, c.j, c.micro_shape_x, c.micro_shape_y, c.micro_shape_k = wm, wn, tm // wm // 16, tn // wn // 16, 2
                c.mfma_m, c.mfma_n, c.mfma_k, c.block_threads, c.stages = 16, 16, 32, 512, st
                shapes.append(c)
        for mx, my in _TILES:
            base = MFMAConfig()
            base.micro_shape_x, base.micro_shape_y = mx, my
            for stages in range(2, self.max_stages(base.tile_size_m, base.tile_size_n) + 1):
                c = MFMAConfig()
                c.micro_shape_x, c.micro_shape_y, c.stages = mx, my, stages
                shapes.append(c)
        for c in shapes:
            tm, tn, stages = c.tile_size_m, c.tile_size_n, c.stages
            if not self.check_valid(c):
                continue
            tiles = -(-m_hi // tm) * -(-N // tn)
            c.num_wave = -(-tiles // self.arch.num_sm)
            splits = [1] + [sk for sk in (2, 3, 4) if tiles * sk <= 4 * self.arch.num_sm and -(-K // 64) // sk >= 8]
            if c.block_threads == 512 and (tm, tn) == (256, 256):
                splits = [0] + splits   # 0: only the tiles of a partly filled last round are split
            for sk in splits:
                cs = MFMAConfig().from_dict(c.to_dict())
                cs.split_k, cs.num_wave = sk, -(-tiles * sk // self.arch.num_sm)
                # rank: the measured preference first, then by distance in tile area, split and stage count
                first = (tm, tn, sk, c.block_threads) == (pref[0], pref[1], pref[3], pref[4]) and \
                    (stages == pref[2] or (c.block_threads == 512 and (tm, tn) != (192, 256)))
                rank = (0 if first else 1, abs(tm * tn - pref[0] * pref[1]),
                        abs(sk - pref[3]), abs(stages - pref[2]), abs(c.block_threads - pref[4]))
                scored.append((rank, cs))
        mfma = [c for _, c in sorted(scored, key=lambda t: t[0])]
        # the W-streaming kernel leads only where it beats the best MFMA candidate under the model
        out = (out + mfma) if self.prefers_skinny(m_hi, N, K) else (mfma[:1] + out + mfma[1:])
        out = (stream + out) if self.prefers_stream(m_hi, N, K) else (out[:1] + stream + out[1:])
        out = (loop + out) if m_hi <= 16 and self.prefers_stream_loop(m_hi, N, K) else (out[:2] + loop + out[2:])
        return (out[:1] + share + out[1:])[:topk]

    def share_shape(self, m_hi: int, N: int) -> Tuple[int, int]:
        """(rows of A, columns per workgroup) of the share kernel for m_hi rows, (0, 0) where there is none: the rows rounded
        up to a kernel's, the fewest columns that give every CU one workgroup (libdtas: share_shape; a host test keeps the
        two alike)."""
        per_cu = -(-N // self.arch.num_sm)
        rows = next((r for r in (16, 32, 48, 64, 96, 128) if m_hi <= r), 0)
        if rows == 16:
            return 16, 16 if per_cu <= 16 else 32 if per_cu <= 56 else 64 if per_cu <= 64 else 128
        cols = next((c for c in (16, 32, 48, 64) if per_cu <= c), 128)
        if rows > 64 and (cols > 48 or (rows == 128 and cols != 48)):
            return 0, 0
        return (rows, cols) if rows else (0, 0)
