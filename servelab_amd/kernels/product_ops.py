"""Matrix products: the layouts a weight is kept in, and the routes a product takes by its rows
(few-rows kernels over the tiled copy, the LDS-staged kernel, tiles over the row-major copy, the
library for the bfloat16 table's large steps; float32 kernels for the float32 table)."""
import contextlib
import ctypes
import os
import re
import tempfile
from typing import Optional

import torch

from .values import (AttentionShares, Deferred, KernelError, LinearWeight, PartialSums, ScaledRows, TiledRows,
                     _c_float, _p, activation_code)


def tuned_shapes(results):
    """(rows, N, K) of the bfloat16 products x w^T among TunableOp's ``results`` (operation, parameters, solution, time)."""
    found = (re.match(r"tn_(\d+)_(\d+)_(\d+)_", r[1]) for r in results if r[0].endswith("_BFloat16_TN"))
    return {(int(m[2]), int(m[1]), int(m[3])) for m in found if m}


class ProductOps:
    def _pair_tiles(self, M, N, K, th=16) -> bool:
        """Whether a few-rows product gives its workgroups two tiles of W (16
        rows each) instead of one.  Two tiles share one pass over x; these
        kernels are bound by what the busiest CU has to pull through its L1
        (45-50 GB/s a CU at most on MI355X, W and the re-read x alike) unless HBM
        is slower still, so the choice goes by the workgroups the busiest CU
        gets times the bytes of one.  Up to 8 rows x is small enough that the
        two forms measured within a few per cent of each other on the 7B, 32B
        and 72B shapes (pairs lose 7 % where K = 8192), so one tile stays; at 16
        rows pairs gain 15-25 % on the large matrices."""
        tiles = -(-N // th)
        if tiles < 2 or M <= 8:
            return False
        w, x = th * K, min(M, 16) * K                     # bytes / 2 of a tile of W and of x
        one = -(-tiles // self._num_cus) * (w + x)
        two = -(-(-(-tiles // 2)) // self._num_cus) * (2 * w + x)
        return two < 0.97 * one

    def _tiles_a_workgroup(self, M, N, K, th, whole, plain=False) -> int:
        """Tiles of W (``th`` rows each) that a workgroup of a few-rows product owns: 2, 1, or 0 for half of one.
        Halves (not where ``whole``: a gate and its up product, a channel and its partner lie in one tile) as long as
        they go round the CUs once: a CU pulls some 50 GB/s whatever the kernel does, and a matrix of 2,048 rows has tiles
        for half of them (us, whole / half: 2048 x 11008 at 1 / 4 rows 10.6 / 12.1 and 9.2 / 9.8, 2048 x 2048 3.8 / 4.0 and
        3.4 / 3.7, 896 x 4864 5.8 and 4.9, 64 x 2048 3.2 and 2.8; products that add to the stream, a copy in tiles of 8 rows / halves,
        at 1 / 8 / 16 rows: 896 x 4864 5.7 / 6.5 / 8.4 and 4.5 / 5.9 / 7.5, 2048 x 11008 10.7 / 11.8 / 15.8 and 9.4 / 10.9 / 14.8, 2048 x
        2048 4.1 / 4.4 / 5.2 and 3.7 / 4.1 / 4.9: a load of a tile of 8 rows brings half as much).  Beyond, the halves' second round costs more than the
        idle CUs (2112 x 2048 3.9 and 4.2, 3584 x 18944 at 8 rows 24.0 and 30.8), until whole tiles are two on some CUs where
        halves are three: up to four rows then (us at 1 / 4 rows 5120 x 27648 56.4 / 58.9 and 53.1 / 57.8, 4608 x 8192 18.9 / 20.2 and 16.8 / 18.7,
        4224 x 2048 6.1 / 6.3 and 5.7 / 6.1; at 8 rows x is read again too often, 34.9 and 37.3 of 5120 x 13824).  ``plain``: not a product that
        adds to the stream, whose readers take 512 sums of squares a row at most."""
        if self._pair_tiles(M, N, K, th):
            return 2
        tiles = -(-N // 16)
        third = plain and M <= 4 and K >= 1024 and self._num_cus < tiles and 2 * tiles <= 3 * self._num_cus
        return 0 if not whole and th == 16 and (2 * tiles <= self._num_cus or third) else 1

    def _skinny(self, x, weight, bias, y, M, N, K, out_f32=False, gated=False, scaled=None,
                resid=None, next_gain=None, out_parts=None, rope=None, y_tiled=False, act=0):
        """One call of the few-rows kernel (at most 16 rows) in any of its forms."""
        parts = scaled.parts if scaled is not None else None
        x_tiled = scaled.tiled if scaled is not None else 0
        if isinstance(x, TiledRows):
            x_tiled, x = x.shape[0], x.data
        # (the product that adds to the stream reads the copy in lower tiles, where the matrix has one)
        wt, th = self._producer_copy(weight, M) if resid is not None else (weight.tiled, 16)
        tiles = self._tiles_a_workgroup(M, N, K, th, gated or scaled is not None or rope is not None, resid is None)
        self._call("gemm", "sl_gemm_skinny", _p(x), _p(wt), _p(bias), _p(y), M, N, K,
                   int(out_f32), int(gated), _p(parts), parts.shape[0] if parts is not None else 0,
                   _c_float(scaled.eps if scaled is not None else 0.0),
                   _p(scaled.rows) if scaled is not None else None, _p(resid), _p(next_gain),
                   _p(out_parts), ctypes.byref(rope) if rope is not None else None,
                   tiles, int(x_tiled), int(y_tiled), th, int(M <= 8 and self.PAIR_X_LOADS),
                   int(act))

    # --------------------------------------------------------------- linear
    def plan_weights(self, total_bytes: int) -> str:
        """Choose the layout for a model whose matrices take ``total_bytes``
        (called before the matrices are loaded)."""
        if self.act_dtype == torch.bfloat16:
            total = torch.cuda.get_device_properties(self.device).total_memory
            self.weight_layout = "dual" if 2 * total_bytes <= self.DUAL_MEMORY_SHARE * total else "tiled"
            # "tiled": as many matrices as fit below ROWS_COPIES_MEMORY_SHARE keep their row-major copy as
            # well, in the order in which they are loaded; the products of many rows of the others go
            # through the scratch buffer
            self._rows_budget = 0 if self.weight_layout == "dual" else \
                max(0, int(self.ROWS_COPIES_MEMORY_SHARE * total) - total_bytes)
            # a third copy of the matrices that add to the stream (about a third of all), in lower tiles
            self.lower_tiles = self.weight_layout == "dual" and 2.35 * total_bytes <= self.LOWER_TILES_MEMORY_SHARE * total
        return self.weight_layout

    def layout_summary(self) -> str:
        """The layout in words, for records: "dual", "rows", or "tiled" with how many of the
        matrices kept a row-major copy as well."""
        if self.weight_layout != "tiled" or not self._matrices_with_rows:
            return self.weight_layout
        return f"tiled, {self._matrices_with_rows} of {self._matrices} matrices also row-major"

    def producer_tile_height(self, N, rows=8):
        """(rows per tile, rows of x from which it pays) for the few-rows product of a matrix of N rows that
        adds to the residual stream.  At 8 rows and more such a product takes as long as its busiest CU needs
        to pull its tiles of W and its re-read of x, so the tiles should go round the CUs evenly: of 16, 14,
        12, 10 and 8 rows the height is taken whose busiest CU pulls least; 16 unless another saves
        LOWER_TILES_MIN_GAIN of it.  Measured on MI355X (us at 1 / 4 / 8 / 16 rows, tiles of 16 against the
        choice): 3584 x 18944, 14 rows (256 tiles on 256 CUs instead of 224): 23.8 / 25.7 / 29.4 / 38.6 against
        25.8 / 26.2 / 28.0 / 33.8; 5120 x 27648, 10 rows (512 tiles instead of 320, two on a quarter of the
        CUs): 57.6 / 61.2 / 68.9 against 54.1 / 52.6 / 56.1.  Where the busiest CU pulls less W (fewer rounds, or
        idle CUs put to work at a lower tile) the lower tiles win from one row on; where only the re-read
        of x per tile of W shrinks (3584), from 8 rows on: below, HBM is the limit, and it streams tiles of
        1 KB a k-step a little faster.  (Timed with x in plain rows; with x laid out by k-step, as the engine
        hands it over, the 3584 case gains nothing end to end, which is why the default minimum gain leaves
        it at 16 rows.  ``prepare_weight`` does not ask about matrices of which halves of tiles of 16 rows go round the CUs once:
        those are as many workgroups.)"""
        def busiest(th, x):
            return -(-(-(-N // th)) // self._num_cus) * (th + x)
        # (a tile is one sum of squares a row for the products that read the stream next: the kernel that keeps
        # x in registers adds up 256 of them, 512 for rows of more than 4,096 values, as the others do)
        most = 256 if N <= 4096 else 512
        heights = [th for th in (16, 14, 12, 10, 8) if th == 16 or -(-N // th) <= most]
        best = min(heights, key=lambda th: (busiest(th, rows), -th))
        if busiest(best, rows) > (1 - self.LOWER_TILES_MIN_GAIN) * busiest(16, rows):
            return 16, 1
        return best, (1 if busiest(best, 0) <= 0.8 * busiest(16, 0) else 8)

    def _producer_copy(self, weight, M):
        """(tiled copy, its tile height) that the product adding ``M`` rows to the stream reads."""
        if weight.lower is not None and M >= weight.lower_from:
            return weight.lower, weight.th
        return weight.tiled, 16

    def prepare_weight(self, w, keep_rows=False, residual_delta=False, _th=None):
        """Called once per matrix at load: returns what ``linear`` takes.
        ``keep_rows``: the caller holds the row-major tensor anyway (a tied
        embedding table), so keeping it costs nothing.  ``residual_delta``: the
        matrix's products are only ever added to the residual stream."""
        N, K = w.shape
        self._check(w, self.act_dtype, None, "weight")
        if self.act_dtype != torch.bfloat16:
            return LinearWeight(w)
        if K % 32 or self.weight_layout == "rows":
            self.graph_rows_limit = min(self.graph_rows_limit, self.ROWS_KERNEL_MAX_M)
            return LinearWeight(w)
        tiled = torch.empty(-(-N // 16) * 16 * K, dtype=torch.bfloat16, device=self.device)
        self._call("gemm", "sl_tile_weight", _p(w), _p(tiled), N, K, 16)
        self._matrices += 1
        if self.weight_layout == "tiled" and not keep_rows and 2 * N * K > self._rows_budget:
            weight = LinearWeight(None, tiled, (N, K))
        else:
            if self.weight_layout == "tiled" and not keep_rows:
                self._rows_budget -= 2 * N * K
            self._matrices_with_rows += 1
            weight = LinearWeight(w, tiled)
        # (halves of tiles of 16 rows, where they go round the CUs once, are as many workgroups and take the same copy as every
        # other product: ``_tiles_a_workgroup``)
        if residual_delta and self.fuse_norms and self.lower_tiles and (_th is not None or 2 * -(-N // 16) > self._num_cus):
            th, lower_from = (_th, 1) if _th is not None else self.producer_tile_height(N)
            if th != 16:
                weight.lower = torch.empty(-(-N // th) * th * K, dtype=torch.bfloat16, device=self.device)
                weight.th, weight.lower_from = th, lower_from
                self._call("gemm", "sl_tile_weight", _p(w), _p(weight.lower), N, K, th)
        self.graph_rows_limit = min(self.graph_rows_limit, self._few_rows_limit(weight))
        return weight

    def rows_of(self, weight):
        """The row-major matrix of a weight; for a tiled-only weight it is
        written into the scratch buffer (valid until the next call)."""
        if weight.w is not None:
            return weight.w
        N, K = weight.shape
        if self._untiled is None or self._untiled.numel() < N * K:
            self._untiled = None
            self._untiled = torch.empty(N * K, dtype=torch.bfloat16, device=self.device)
        out = self._untiled[:N * K].view(N, K)
        self._call("gemm", "sl_untile_weight", _p(weight.tiled), _p(out), N, K, 16)
        return out


    def linear(self, x, weight, bias, out_f32=False, defer=False):
        """y = x W^T (+ bias); ``weight`` is a LinearWeight or a plain [N, K] tensor.
        ``defer``: y will only be added to the residual stream, so the product
        may be left to the norm that adds it: up to 16 rows a ``Deferred`` comes
        back (the norm's kernel runs the product), at 17..64 rows ``PartialSums``
        of a product whose K was split (the norm adds them up).

        bfloat16, by rows of x: 1..16 the few-rows kernel over the tiled weight,
        17..64 the wide or the LDS-staged kernel (by the size of W; the latter
        up to 128 rows), more the kernels in tiles, some of them in shares of K (``_block_plan``, ``_shares_plan``,
        ``_shares_by_estimate``), over the tiled copy where such tiles go round the CUs once (``_even_columns``),
        or the library, or as many rows as the first ones take at a time when the result is wanted in float32.
        float32: ``linear_rows`` up to 16 rows (FMAs, from three on the matrix units), ``linear_f32_mfma`` above where
        K % 16 == 0, else the tiled FMA kernel; never a library product."""
        if not isinstance(weight, LinearWeight):
            weight = LinearWeight(weight)
        if isinstance(x, ScaledRows):
            if weight.tiled is not None and weight.shape == (weight.shape[0], x.shape[1]):
                return self._linear_scaled(x, weight, bias, out_f32, False)
            x = self.finish_scaled_rows(x)      # (a matrix the fused kernels do not take: rows of odd length)
        if isinstance(x, AttentionShares):
            x = self.combine_shares(x)
        M, K = x.shape
        N = weight.shape[0]
        if isinstance(x, TiledRows) and not (defer and self.fuse_norms and not out_f32 and N <= 8192):
            # (rows by k-step are read by the few-rows kernel only, which is where they come from)
            if weight.shape != (N, K):
                raise KernelError(f"weight has shape {list(weight.shape)}, x has {K} columns")
            y = self._new((M, N), torch.float32 if out_f32 else None)
            self._skinny(x, weight, bias, y, M, N, K, out_f32)
            return y
        if (defer and self.fuse_norms and not out_f32 and 0 < M <= self._fused_rows(N)
                and weight.tiled is not None and weight.shape == (N, K) and N <= 8192):
            return Deferred(x, weight, bias)
        self._check(x, self.act_dtype, None, "x")
        if weight.shape != (N, K):
            raise KernelError(f"weight has shape {list(weight.shape)}, x has {K} columns")
        if weight.w is not None:
            self._check(weight.w, self.act_dtype, (N, K), "weight")
        if bias is not None:
            self._check(bias, torch.float32, (N,), "bias")
        if self.act_dtype == torch.float32:
            if K % 4 == 0 and M <= self.ROWS_KERNEL_MAX_M:
                return self.linear_rows(x, weight.w, bias, out_f32)
            if K % 16 == 0 and M >= self.F32_MFMA_MIN_M:
                return self.linear_f32_mfma(x, weight.w, bias)
            return self.linear_tiled(x, weight.w, bias, out_f32)
        limit = self._few_rows_limit(weight)
        plan = self._block_plan(M, N, K, weight) or (
            defer and M > self.BLOCK_SQUARE_MAX_M and self.fuse_norms and not out_f32
            and not self._tuned_for(M, N, K) and self._block_reads(x, weight)
            and (self._shares_plan(M, N, K, weight) or self._shares_by_estimate(M, N, K, weight)))
        if plan:
            # (deferred: the norm adds the partial sums)
            return self.linear_block(x, weight, bias, out_f32, plan[0],
                                     partial=defer and self.fuse_norms and not out_f32, square=plan[1])
        if (defer and self.fuse_norms and not out_f32 and self._wide_from(N) <= M <= limit
                and K % 32 == 0 and N % 4 == 0 and self._takes_mid(M, N, K)):
            return self.linear_mid(x, weight, bias, partial=True,     # the norm adds the partial sums
                                   target=self.MID_DEFERRED_WORKGROUPS)
        if M <= limit:
            return self.linear_skinny(x, weight, bias, out_f32)
        columns = self._even_columns(M, N, K)
        if columns and weight.tiled is not None and not self._tuned_for(M, N, K) and x.data_ptr() % 16 == 0:
            return self.linear_even(x, weight, bias, columns, out_f32)
        if out_f32 and limit:
            # float32 results of many rows (the head for more requests than the few-rows kernels take,
            # logits of every position).  With a row-major copy of W: the library's product with its
            # float32 sums kept, one pass over W (7B shape, the head for 144 requests: 150 us; the
            # few-rows kernels stream W once per `limit` rows, 128 + 16 rows in 236 + 178 us).  Without:
            # those, several times faster than the plain tiled kernel below.
            if weight.w is not None:
                if bias is not None and self._bias_tiles(M, N, K) and self._block_reads(x, weight):
                    return self.linear_block(x, weight, bias, True, square=True)
                sums = self.library_sums(x, weight.w, torch.float32)
                return sums if bias is None else sums.add_(bias)
            return torch.cat([self.linear_skinny(x[i:i + limit], weight, bias, True)
                              for i in range(0, M, limit)])
        w = self.rows_of(weight)
        if M <= self.ROWS_KERNEL_MAX_M and K % 8 == 0:
            return self.linear_rows(x, w, bias, out_f32)
        if K % 8:
            # rows that are no multiple of 16 bytes: the plain tiled kernel for any number of rows (no
            # library call, so that a captured decode step stays clear of it as well)
            return self.linear_tiled(x, w, bias, out_f32)
        if out_f32:
            if M <= 4 * self.ROWS_KERNEL_MAX_M and K % 8 == 0:
                return self.linear_rows(x, w, bias, out_f32)
            return self.linear_tiled(x, w, bias, out_f32)
        return self.linear_library(x, w, bias)

    def _even_columns(self, M, N, K):
        """Columns of y a workgroup takes in the product of tiles that go round the CUs once (``sl_gemm_even``, 128 rows of x), the
        fewest that do, or 0 where the product is not its own: matrices of 512 rows and more with rows of up to EVEN_MAX_K values,
        tiles of up to 192 columns, or 224 on nine tenths of the CUs; with rows of more than EVEN_SHORT_K values seven tenths of the
        CUs busy, in tiles of 128 columns and more 0.76 of them (GPU time, library / here: three quarters, 700 x 4096 x 4096 31.5 / 34.6,
        1,536 x 2048 x 3072 in 1.15 of it; at 0.76 to 0.8 in 0.92).  The call is worth having beyond its GPU time, of which 1,966 such
        products (512 to 6,144 rows, 65 to 8,192 rows of x) take 0.99 of the library's on average: the library's takes the host 20 us,
        and prompts of up to some 450 tokens wait for the host.  Those take tiles also where few CUs have one (256 x 2048 x 2048 11.9 / 18.5;
        whole prompts, library / here: twelve layers of the 1.5B shape, 200 / 400 tokens 2,213 / 1,313 and 2,328 / 1,785, of the 3B shape 256 / 400
        1,674 / 1,670 and 2,044 / 1,999); longer ones with rows of more than EVEN_HOST_K values only on 0.425 of the CUs (the 3B shape at 512
        tokens, o on 0.34 and q/k/v on 0.42: 2,104 / 2,191; 24 layers of the 0.5B shape, rows of 896, at 512 / 1,000 3,582 / 2,819 and 3,505 / 2,805).
        us, library / here: 2,048 rows of x, 3584 x 3584 52 / 48, 2560 x 2048 26 / 24; 527 rows 4608 x 3584 29 / 26.
        Longer rows and idle CUs: 527 rows, 2048 x 8192 43 / 46, 1536 x 8960 37 / 48; 1,500 rows, 4096 x 4096 49 / 54 in 224
        columns on 0.89 of the CUs; two rounds: 2,048 rows, 4608 x 3584 60 / 76."""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or K % 64 or N % 4 or N < self.EVEN_MIN_N
                or K > self.EVEN_MAX_K):
            return 0
        rows = -(-M // 128)
        for columns in range(96, 225, 32):
            fill = rows * -(-N // columns) / self._num_cus
            if fill <= 1:
                least = 0.9 if columns == 224 else 0
                if K > self.EVEN_SHORT_K:
                    least = max(least, 0.7 if columns == 96 else 0.76)
                elif K > self.EVEN_HOST_K and M > self.EVEN_HOST_ROWS:
                    least = max(least, 0.425)
                return columns if fill >= least else 0
        return 0

    def linear_even(self, x, weight, bias, columns, out_f32=False):
        """y = x W^T (+ bias) of many rows over the tiled copy of the weight, tiles of 128 x ``columns``."""
        M, K = x.shape
        N = weight.shape[0]
        self._check(x, self.act_dtype, (M, K), "x")
        y = self._new((M, N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_even", _p(x), _p(weight.tiled), _p(bias), _p(y), M, N, K, int(out_f32), int(columns))
        return y

    def linear_wide(self, x, weight, bias, out_f32=False, gated=False, act=0):
        M, K = x.shape
        N = weight.shape[0]
        if weight.tiled is None:
            raise KernelError("linear_wide needs the tiled copy of the weight")
        y = self._new((M, N // 2 if gated else N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_wide", _p(x), _p(weight.tiled), _p(bias), _p(y), M, N, K,
                   int(out_f32), int(gated), int(act))
        return y

    def _takes_mid(self, M, N, K) -> bool:
        return N * K >= (self.MID_MIN_ELEMENTS if M <= 32 else self.MID_MIN_ELEMENTS_MANY)

    MID_MAX_M = 128               # the LDS-staged kernel takes up to this many rows

    def _few_rows_limit(self, weight) -> int:
        """Up to how many rows of x a product with this weight stays with the
        kernels that stream the tiled copy (more rows: the library): none
        without a tiled copy, SKINNY_MAX_M, or MID_MAX_M where the LDS-staged
        kernel takes the matrix."""
        if weight.tiled is None or self.act_dtype != torch.bfloat16:
            return 0
        N, K = weight.shape
        if K % 32 == 0 and N * K >= self.MID_MIN_ELEMENTS_MANY:
            return self.MID_MAX_M
        return self.SKINNY_MAX_M

    def linear_mid(self, x, weight, bias, out_f32=False, gated=False, ks=None, partial=False,
                   target=None, act=0):
        """17..128 rows with x staged through LDS; K split over workgroups when
        N alone gives too few of them.  ``partial``: a split product comes back
        as ``PartialSums`` for its reader to add up."""
        M, K = x.shape
        N = weight.shape[0]
        if weight.tiled is None:
            raise KernelError("linear_mid needs the tiled copy of the weight")
        wgs = -(-(-(-N // 16)) // 8)
        if ks is None:
            if target is None:
                target = self.MID_PARTIAL_WORKGROUPS if partial else self.MID_TARGET_WORKGROUPS
            ks = 1 if gated or act else max(1, min(16, K // 32 // 4, -(-target // wgs)))
        part = self._new((ks, M, N), torch.float32) if ks > 1 else None
        if partial and ks > 1:
            self._call("gemm", "sl_gemm_mid", _p(x), _p(weight.tiled), None, None, M, N, K,
                       0, 0, int(ks), self.MID_WIDE_WORKGROUPS, self._num_cus, _p(part), 0)
            return PartialSums(part, bias)
        y = self._new((M, N // 2 if gated else N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_mid", _p(x), _p(weight.tiled), _p(bias), _p(y), M, N, K,
                   int(out_f32), int(gated), int(ks), self.MID_WIDE_WORKGROUPS, self._num_cus, _p(part), int(act))
        return y

    def _block_plan(self, M, N, K, weight):
        """How the block kernel takes a product of M rows: (shares of K, square tiles), or None
        when the product is not one of its own: bfloat16, a row-major copy of the weight, K in
        chunks of 64, a matrix of few rows (its tiles alone would leave most CUs idle, which is
        what the split repairs) but of BLOCK_MIN_ELEMENTS elements at least (smaller ones stay
        with the kernels they were measured on).  Tiles of 256 x 128 for BLOCK_MIN_M to BLOCK_MAX_M
        rows of x; tiles of 256 x 256 for matrices with long rows (K of BLOCK_SQUARE_MIN_K and
        more: the down projection) from 257 to BLOCK_SQUARE_MAX_M rows, if their tiles and shares
        fill three quarters of the CUs.  As many shares as give every CU a workgroup, 16 at most,
        of at least 3 chunks each (7B shape, down projection at 256 rows: 70 / 44 / 41 us with 4 / 8
        / 9 shares; q/k/v: 21 / 17 / 26 us with 4 / 7 / 8, the last being more workgroups than CUs;
        down at 527 rows: 84 us in square tiles, 101 us in 256 x 128, 130 us in the library's tuned
        kernel; at 1,024 rows 111 us in 4 shares, 144 us in 6)."""
        w = weight.w if isinstance(weight, LinearWeight) else weight
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or w is None
                or K % 64 or N % 4 or N > self.BLOCK_MAX_N or N * K < self.BLOCK_MIN_ELEMENTS):
            return None
        if K >= self.BLOCK_SQUARE_MIN_K and 256 < M <= self.BLOCK_SQUARE_MAX_M:
            tiles = -(-N // 256) * -(-M // 256)
            shares = min(16, K // 64 // 3, self._num_cus // tiles)
            if shares >= 1 and 4 * tiles * shares >= 3 * self._num_cus:
                return shares, True
        if not self.BLOCK_MIN_M <= M <= self.BLOCK_MAX_M:
            return None
        tiles = -(-N // 128) * -(-M // 256)
        return max(1, min(16, K // 64 // 3, self._num_cus // tiles)), False

    def _shares_plan(self, M, N, K, weight):
        """Like ``_block_plan`` for a product of more rows that the norm adds to the stream: two or
        three shares of K in square tiles where they fill the CUs well, two to seven eighths, three to four fifths (GPU
        time with the norm, library's product / shares: 3584 x 18944, 2,048 rows 387 / 236 us in two; 2560 x 9728, 2,048 rows 121 / 107
        in three, 2560 x 13824 163 / 136; 4096 x 14336, 1,600 / 2,048 rows 344 / 185 and 231 / 212; 4096 x 8192 loses 2 to 5 % but at 1,792)."""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or weight.w is None
                or K % 64 or N % 4 or N > self.BLOCK_MAX_N or K < self.BLOCK_SQUARE_MIN_K
                or not self.BLOCK_SQUARE_MAX_M < M <= self.SHARES_MAX_M):
            return None
        tiles = -(-N // 256) * -(-M // 256)
        shares = self._num_cus // tiles
        fill = tiles * shares / self._num_cus
        return (shares, True) if (shares == 2 and fill >= 0.875) or (shares == 3 and fill >= 0.8) else None

    def _shares_by_estimate(self, M, N, K, weight):
        """The sizes that ``_shares_plan`` leaves: two to eight shares in wide tiles, as many as take the least time by estimate
        (the product's, ``_tiles_us``, and SHARE_US for every million sums written and read again).  us with the norm that adds
        them, the library's product / the shares: 2048 x 11008 at 1,792 / 1,930 / 2,048 rows 111 / 87, 109 / 92 and 115 / 96 in
        four, 2048 x 8192 at 2,048 83 / 79, 1536 x 8960 83 / 71 in five, 3584 x 18944 at 1,664 / 1,792 244 / 203 and 321 / 221 in two,
        64 x 8192 31 / 20 in eight; of 142 sizes from 64 columns on 0.85 of the time on average, 1.05 at worst (one of ``_shares_plan``).  Two shares on
        three quarters of the CUs or fewer lose and are left to the library (3072 x 8192 at 1,930 / 2,048 109 / 115 and 110 / 115, 3328 x 8192 at 1,792
        111 / 115, 2880 x 11520 at 1,930 141 / 149); at 0.77 they do not (3584 x 8192 at 1,792 120 / 117).
        Rows of 5,632 values and less gain nothing (2048 x 5632 at 2,048 64 / 62, 896 x 4864 34 / 33)."""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or weight.w is None
                or K % 64 or N % 4 or N > self.BLOCK_MAX_N or K < self.BLOCK_SQUARE_MIN_K
                or not self.BLOCK_SQUARE_MAX_M < M <= self.SHARES_MAX_M):
            return None
        tiles = -(-N // 256) * -(-M // 256)
        plans = [ks for ks in range(2, 9) if tiles * ks <= self._num_cus]
        if not plans:
            return None
        ks = min(plans, key=lambda ks: self._tiles_us(self._tile_rows(M, N, K, ks), M, N, K, ks) + self.SHARE_US * 1e-6 * ks * M * N)
        if ks == 2 and 4 * 2 * -(-N // 256) * -(-M // self._tile_rows(M, N, K, 2)) <= 3 * self._num_cus:
            return None
        return ks, True

    def _gated_rows(self, M, N, K):
        """Rows of x a workgroup takes (192 or 256) for the gated product of a prompt at sizes that take the tiles whatever their
        estimated rate (``_prompt_tiles``) says, or None.  The kernel saves the pass that gates the library's product and the
        host the library's call, some 25 us a layer.  Rows of up to GATED_SHORT_K values
        therefore always take it: such models' prompts wait for the host at nearly every size (whole passes, pair / kernel as it
        was with sixteen wavefronts: 24 layers of the 0.5B shape, 9728 x 896, 260 / 600 / 1,000 / 1,700 / 2,048 tokens 4,893 / 4,194,
        3,837 / 3,356, 4,116 / 3,604, 4,184 / 3,901 and 4,381 / 4,191 us; 12 layers of 4096 x 1024, 256 and
        2,048 tokens 2,063 / 1,823 and 2,133 / 1,862).  By GPU time alone it wins there as well now (9728 x 896, 300 / 1,000 /
        1,600 / 2,048 rows 35 / 22, 37 / 25, 43 / 42 and 59 / 43 us).  Rows of up to GATED_ONE_ROUND_K values take it where one
        round of tiles is GATED_FILL useful (17920 x 1536, 527 / 640 / 768 rows 38 / 33, 45 / 41 and 47 / 42 us a product), and
        longer ones, up to GATED_LONG_K values at GATED_LONG_ROWS rows of x, in several rounds of tiles of 256 x 256 whose last
        one is filled by GATED_LAST_ROUND where neither 192 nor 224 divides N, at which the library's picks idle (2,048 rows of
        37888 x 3584 543 / 429, of 22016 x 2048 193 / 153).  The sums meet the activation unrounded, so that it
        is the more exact form as well.  Shapes that were tuned may stay with the library (``_tiles_beat_tuned``)."""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or K % 64 or N % 16
                or N < self.GATED_MIN_N or M > self.GATED_MAX_M):
            return None
        columns = -(-N // 256)
        if M >= self.GATED_MIN_M and K <= self.GATED_ONE_ROUND_K:
            rounds = {rows: -(-columns * -(-M // rows) // self._num_cus) for rows in (256, 192)}
            rows = min(rounds, key=lambda r: rounds[r] * (r * K + 65536))
            if K <= self.GATED_SHORT_K or (rounds[rows] == 1 and M * N >= self.GATED_FILL * self._num_cus * rows * 256):
                return rows
        rounds, last = divmod(columns * -(-M // 256), self._num_cus)
        least, most = self.GATED_LAST_ROUND
        fits = (K <= self.GATED_LONG_K and self.GATED_LONG_ROWS[0] <= M <= self.GATED_LONG_ROWS[1] and N % 192 and N % 224
                and rounds and least * self._num_cus <= last <= most * self._num_cus)
        return 256 if fits else None

    # rows of x a tile -> us of a launch, of a round of tiles, of a chunk of 64 values of k with few CUs busy, and what all of
    # them add to a chunk (they share the power): fitted to 168 gated products of 12 shapes, 260 to 2,048 rows of x, with a cheaper activation than is taken
    # now; against 153 of them as they are 4 % rms and 12 % at worst (7 and 15 for the ones of 128 rows, with six halves on the way where
    # the others have four) but for rows of 896 values, which take up to a fifth longer, and no other choice would gain more than 0.1 % on average
    TILE_US = {256: (1.8, 6.0, 0.92, 0.49), 192: (2.5, 4.0, 0.74, 0.39), 128: (1.0, 3.5, 0.68, 0.20)}

    def _tiles_us(self, rows, M, N, K, ks=1):
        """Estimated time of a product in tiles of ``rows`` rows of x by 256 of W."""
        launch, tile, chunk, shared = self.TILE_US[rows]
        items = -(-N // 256) * -(-M // rows) * ks
        rounds = -(-items // self._num_cus)
        return launch + rounds * (tile + K / ks / 64 * (chunk + shared * items / (rounds * self._num_cus)))

    def _tile_rows(self, M, N, K, ks=1):
        """Rows of x a workgroup takes, the ones that take the least time by estimate (of 125 products 0.12 % slower on average than the best height,
        9 % at worst, 1000 x 22016 x 2048; 128 where the others leave CUs idle: 22016 x 2048 at 527 / 640 rows
        75 / 58 us both times, 9216 x 3584 at 768 57 / 48)."""
        return min(self.TILE_US, key=lambda rows: self._tiles_us(rows, M, N, K, ks))

    def _prompt_tiles(self, M, N, K):
        """Rows of x a tile for a product of a prompt whose results the library would leave to a second pass (a gate or an
        activation), or None where its product and the pass are the faster pair: where the tiles' estimated rate is below
        PROMPT_MIN_TFLOPS, which is where they leave CUs idle.  Of 153 products (rows of 896 to 5,120 values) the
        kernel at 750 and more takes 0.91 of the pair's time on average, 1.11 at worst (600 x 27648 x 3584, 128 against 116
        us); at 700 9216 x 3584 with 640 rows of x is among them (56 against 45)."""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or K % 64 or N % 16
                or N < self.GATED_MIN_N or not self.GATED_MIN_M <= M <= self.GATED_MAX_M or K > self.PROMPT_MAX_K):
            return None
        rows = self._tile_rows(M, N, K)
        return rows if 2e-6 * M * N * K >= self.PROMPT_MIN_TFLOPS * self._tiles_us(rows, M, N, K) else None

    def _bias_tiles(self, M, N, K) -> bool:
        """Whether a prompt's product with float32 results and a bias, which the library leaves to a second pass over
        them, goes into the tiles: by their estimated rate, from BIAS_MIN_TFLOPS on.  Of 92 products of twelve matrices at 300 to 2,500
        rows the tiles take 0.87 of the pair's time where this says so, 0.99 at worst (us, library and pass / tiles: 6160 x 2048 at
        1,000 / 2,048 rows 44 / 37 and 75 / 58, 7168 x 3584 at 1,500 / 1,852 85 / 73 and 101 / 92, 10304 x 2048 at 600 / 1,500 44 / 37 and 82 /
        65).  The longer the rows, the less the pass is beside the product, and the higher the line: at 750 and more, but below it,
        10792 x 3584 at 1,500 123 / 133 and 7168 x 3584 at 2,500 134 / 137, 5120 x 5120 at 1,000 62 / 66, 14336 x 4096 at 1,280 148 / 153; 6160 x 2048 at
        768 35 / 37.  (Whether the shape was tuned is not asked: ``library_tuning`` times no product with float32 results.)"""
        if (self.act_dtype != torch.bfloat16 or not self.use_block_products or K % 64 or N % 4 or M < self.GATED_MIN_M):
            return False
        least = next((rate for values, rows, rate in self.BIAS_MIN_TFLOPS if K <= values and M <= rows), None)
        return least is not None and 2e-6 * M * N * K >= least * self._tiles_us(self._tile_rows(M, N, K), M, N, K)

    def _tuned_for(self, M, N, K) -> bool:
        """Whether the library's product of this shape has been timed over its candidates (``library_tuning``; inside
        its block: whether it may be).  Those shapes stay with the library, whose default pick is
        what the rules above were measured against: tuned it is up to a quarter faster."""
        return self._tuning or (self.library_rows(M), N, K) in self._tuned

    def _tiles_beat_tuned(self, M, N, K) -> bool:
        """Whether a gated or activated product that may take the tiles does: a shape that was tuned stays with the library and its
        pass below an estimated rate of PROMPT_TUNED_TFLOPS.  From there on the tiles are the faster pair also against the tuned pick
        (us, tuned / tiles: 37888 x 3584 at 544 / 1,024 / 2,048 rows 176 / 150, 279 / 259 and 469 / 475, 22016 x 2048 at 2,048 187 /
        169, 17920 x 1536 137 / 130, 55296 x 5120 973 / 909, 28672 x 4096 407 / 394, 18944 x 3584 with relu squared 267 / 273)."""
        return not self._tuned_for(M, N, K) or 2e-6 * M * N * K >= self.PROMPT_TUNED_TFLOPS * self._tiles_us(self._tile_rows(M, N, K), M, N, K)

    @staticmethod
    def _block_reads(x, weight) -> bool:
        """Whether the rows lie as the block kernel reads them, from multiples of 16 bytes on (the library takes any)."""
        return x.data_ptr() % 16 == 0 and (weight.w is None or weight.w.data_ptr() % 16 == 0)

    def linear_gated_block(self, x, weight, bias, rows, act):
        """act(gate) * up of many rows over the row-major weight, tiles of ``rows`` x 256."""
        M, K = x.shape
        N = weight.shape[0]
        w = self.rows_of(weight)
        self._check(x, self.act_dtype, (M, K), "x")
        self._check(w, self.act_dtype, (N, K), "weight")
        y = self._new((M, N // 2))
        self._call("gemm", "sl_gemm_block", _p(x), _p(w), _p(bias), _p(y), M, N, K, 0, int(act), 0, 1, int(rows), None)
        return y

    def linear_activated_block(self, x, weight, bias, rows, act):
        """act(x W^T + b) of many rows over the row-major weight, tiles of ``rows`` x 256: the activation meets the float sums, and
        the pass over the library's rounded product is saved (18944 x 3584, relu squared, 900 / 1,536 / 1,852 rows 139 / 126, 170 /
        170 and 288 / 203 us, library and pass / here; 11008 x 2048, 768 / 1,000 / 2,048 rows 47 / 37, 56 / 45 and 93 / 81)."""
        M, K = x.shape
        N = weight.shape[0]
        w = self.rows_of(weight)
        self._check(x, self.act_dtype, (M, K), "x")
        self._check(w, self.act_dtype, (N, K), "weight")
        if bias is not None:
            self._check(bias, torch.float32, (N,), "bias")
        y = self._new((M, N))
        self._call("gemm", "sl_gemm_block", _p(x), _p(w), _p(bias), _p(y), M, N, K, 0, 0, int(act), 1, int(rows), None)
        return y

    def linear_block(self, x, weight, bias, out_f32=False, ks=1, partial=False, square=False):
        """A few hundred rows over the row-major copy of the weight: workgroups
        own a tile of 256 rows of x by 128 rows of W (``square``: of 256, 192 or 128, ``_tile_rows``, by 256) over
        one of ``ks`` shares of K.  ``partial``: the product comes back as
        ``PartialSums`` for its reader to add up."""
        M, K = x.shape
        N = weight.shape[0]
        w = weight.w if isinstance(weight, LinearWeight) else weight
        if w is None:
            raise KernelError("linear_block needs the row-major copy of the weight")
        self._check(x, self.act_dtype, (M, K), "x")
        self._check(w, self.act_dtype, (N, K), "weight")
        rows = self._tile_rows(M, N, K, ks) if square else 0
        part = self._new((ks, M, N), torch.float32) if ks > 1 or partial else None
        if partial:
            if ks > 1:
                self._call("gemm", "sl_gemm_block", _p(x), _p(w), None, None, M, N, K, 0, 0, 0, int(ks), rows,
                           _p(part))
            else:
                self._call("gemm", "sl_gemm_block", _p(x), _p(w), None, _p(part), M, N, K, 1, 0, 0, 1, rows, None)
            return PartialSums(part, bias)
        y = self._new((M, N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_block", _p(x), _p(w), _p(bias), _p(y), M, N, K, int(out_f32),
                   0, 0, int(ks), rows, _p(part))
        return y

    def linear_skinny(self, x, weight, bias, out_f32=False):
        M, K = x.shape
        N = weight.shape[0]
        if weight.tiled is None:
            raise KernelError("linear_skinny needs the tiled copy of the weight")
        if M >= self._wide_from(min(N, K)):       # (the stream is what a projection reads or what it writes)
            if self._takes_mid(M, N, K):
                return self.linear_mid(x, weight, bias, out_f32)
            return self.linear_wide(x, weight, bias, out_f32)
        y = self._new((M, N), torch.float32 if out_f32 else None)
        self._skinny(x, weight, bias, y, M, N, K, out_f32)
        return y

    def _linear_scaled(self, xs, weight, bias, out_f32, gated, y_tiled=False):
        """The consumer of un-normalised rows: one few-rows product that scales
        its result rows by rsqrt(mean x^2 + eps)."""
        M, K = xs.shape
        N = weight.shape[0]
        if weight.tiled is None or weight.shape != (N, K) or M > self.FUSED_NORM_MAX_M:
            raise KernelError("un-normalised rows need a tiled weight and at most 16 rows")
        if bias is not None:
            self._check(bias, torch.float32, (N,), "bias")
        y = self._new((M, N // 2 if gated else N), torch.float32 if out_f32 else None)
        if self._takes_resident(N, K, xs.parts.shape[0]):
            self._call("gemm", "sl_gemm_resident", _p(xs.x), _p(weight.tiled), _p(bias), _p(y), M, N, K,
                       int(out_f32), int(gated), _p(xs.parts), xs.parts.shape[0], _c_float(xs.eps),
                       _p(xs.rows), int(xs.tiled), int(y_tiled))
        else:
            self._skinny(xs.x, weight, bias, y, M, N, K, out_f32, gated, scaled=xs, y_tiled=y_tiled)
        return TiledRows(y, (M, N // 2)) if y_tiled else y

    def finish_scaled_rows(self, xs):
        """Un-normalised rows as plain normed rows in the activation dtype, for a reader whose matrix
        the fused few-rows kernels do not take: every row times rsqrt(mean x^2 + eps) from the sums
        of squares the producer left."""
        x = xs.plain_x()
        sums = xs.parts.sum(0)                                  # by row of the producer's step
        if xs.rows is not None:
            x, sums = x[xs.rows.long()], sums[xs.rows.long()]
        else:
            sums = sums[:x.shape[0]]
        return (x.float() * torch.rsqrt(sums / x.shape[1] + xs.eps)[:, None]).to(self.act_dtype)

    def _takes_resident(self, N, K, parts) -> bool:
        """Whether a consumer product runs on the workgroups that stay and walk the tiles
        (x in registers, row scales computed once): matrices with several tiles per CU whose
        row length the kernel is built for (the library says which: ``sl_gemm_resident_parts``,
        the most sums of squares a row its kernel for K adds up, 0 for no kernel).  Every other
        width takes the workgroup-per-tile kernel: the same result with 9 to 16 rows, and up to the order of the float
        sums with 8 and fewer."""
        if -(-N // 16) < self.RESIDENT_MIN_ROUNDS * self._num_cus:
            return False
        most = self._resident_k.get(K)
        if most is None:
            most = self._resident_k[K] = int(self._lib["gemm"].sl_gemm_resident_parts(K))
        return 0 < parts <= most

    GATE_BLOCK = 8                # gate and up rows alternate in blocks of 8 (half an MFMA tile)

    def gated_linear(self, x, weight, block, _tiled_out=False, activation="silu", bias=None):
        """act(x Wg^T + bg) * (x Wu^T + bu) for a weight whose rows hold gate and up
        interleaved in blocks of ``block`` rows (``block`` = I: plain [Wg; Wu]) and a
        ``bias`` [2 I] (or None) that lies as the rows do;
        ``activation``: "silu", "relu" or "gelu_tanh".  Blocks of 8 and few rows of x over
        a tiled weight, or as many as ``_gated_rows`` takes: one fused kernel."""
        if not isinstance(weight, LinearWeight):
            weight = LinearWeight(weight)
        code = activation_code(activation, ("silu", "relu", "gelu_tanh"))      # (what the kernels take as `gated`)
        if bias is not None:
            self._check(bias, torch.float32, (weight.shape[0],), "bias")
        if isinstance(x, ScaledRows):
            if block == self.GATE_BLOCK and weight.shape[0] % 16 == 0 and weight.tiled is not None:
                return self._linear_scaled(x, weight, bias, False, code, y_tiled=_tiled_out)
            x = self.finish_scaled_rows(x)
            _tiled_out = False
        M, K = x.shape
        N = weight.shape[0]
        if (_tiled_out and M < self._wide_from(K) and M <= self._few_rows_limit(weight)
                and block == self.GATE_BLOCK and N % 16 == 0):
            self._check(x, self.act_dtype, None, "x")
            y = self._new((M, N // 2))
            self._skinny(x, weight, bias, y, M, N, K, gated=code, y_tiled=True)
            return TiledRows(y, (M, N // 2))
        if M <= self._few_rows_limit(weight) and block == self.GATE_BLOCK and N % 16 == 0:
            self._check(x, self.act_dtype, None, "x")
            if M >= self._wide_from(K):
                if self._takes_mid(M, N, K):
                    return self.linear_mid(x, weight, bias, gated=code)
                return self.linear_wide(x, weight, bias, gated=code)
            y = self._new((M, N // 2))
            self._skinny(x, weight, bias, y, M, N, K, gated=code)
            return y
        rows = block == self.GATE_BLOCK and (self._prompt_tiles(M, N, K) or self._gated_rows(M, N, K))
        if rows and self._tiles_beat_tuned(M, N, K) and self._block_reads(x, weight):
            return self.linear_gated_block(x, weight, bias, rows, code)
        return self.gate_mul(self.linear(x, weight, bias), block, activation)

    def gated_mlp(self, x, w_gate_up, block, w_down, defer=False, activation="silu", bias_gate_up=None,
                  bias_down=None):
        """down(act(gate x) * (up x)), with biases when given: ``gated_linear`` followed by ``linear``.  With few rows the
        kernel table keeps what lies between them in the layout its second kernel reads best
        (rows by k-step: the eight rows of a decode step then cost the down product half as many
        cache lines per load of x)."""
        if not isinstance(w_gate_up, LinearWeight):
            w_gate_up = LinearWeight(w_gate_up)
        if not isinstance(w_down, LinearWeight):
            w_down = LinearWeight(w_down)
        M = x.shape[0]
        inner = w_gate_up.shape[0] // 2
        tiled = (self.act_dtype == torch.bfloat16 and self.tile_few_rows and 1 < M <= self._fused_rows(w_down.shape[0])
                 and block == self.GATE_BLOCK and inner % 32 == 0 and w_gate_up.tiled is not None
                 and w_down.tiled is not None and w_down.shape[1] == inner and w_gate_up.shape[0] % 16 == 0)
        h = self.gated_linear(x, w_gate_up, block, _tiled_out=tiled, activation=activation, bias=bias_gate_up)
        return self.linear(h, w_down, bias_down, defer=defer)

    def activated_linear(self, x, weight, activation, bias=None, _tiled_out=False):
        """act(x W^T + b) for an ``activation`` of ``activate``.  Few rows and a tiled weight, or as many as
        ``_prompt_tiles`` takes: the activation sits in the product's epilogue, on its float32 sums."""
        if not isinstance(weight, LinearWeight):
            weight = LinearWeight(weight)
        code = activation_code(activation, ("silu", "relu", "relu2", "gelu_tanh"))
        if isinstance(x, ScaledRows):
            x = self.finish_scaled_rows(x)
        M, K = x.shape
        N = weight.shape[0]
        if M > self._few_rows_limit(weight) or M == 0:
            rows = self._prompt_tiles(M, N, K)
            if rows and weight.shape == (N, K) and self._tiles_beat_tuned(M, N, K) and self._block_reads(x, weight):
                return self.linear_activated_block(x, weight, bias, rows, code)
            return self.activate(self.linear(x, weight, bias), activation)
        self._check(x, self.act_dtype, None, "x")
        if weight.shape != (N, K):
            raise KernelError(f"weight has shape {list(weight.shape)}, x has {K} columns")
        if bias is not None:
            self._check(bias, torch.float32, (N,), "bias")
        if M >= self._wide_from(min(N, K)):
            if self._takes_mid(M, N, K):
                return self.linear_mid(x, weight, bias, act=code)
            return self.linear_wide(x, weight, bias, act=code)
        y = self._new((M, N))
        self._skinny(x, weight, bias, y, M, N, K, act=code, y_tiled=_tiled_out)
        return TiledRows(y, (M, N)) if _tiled_out else y

    def plain_mlp(self, x, w_up, w_down, activation, defer=False):
        """down(act(up x)) without a gate and without biases; with few rows what lies between the two
        products is kept in the layout the second one reads best (rows by k-step)."""
        if not isinstance(w_up, LinearWeight):
            w_up = LinearWeight(w_up)
        if not isinstance(w_down, LinearWeight):
            w_down = LinearWeight(w_down)
        M, inner = x.shape[0], w_up.shape[0]
        tiled = (self.act_dtype == torch.bfloat16 and self.tile_few_rows and 1 < M <= self._fused_rows(w_down.shape[0])
                 and M < self._wide_from(min(w_up.shape)) and inner % 32 == 0 and w_up.tiled is not None
                 and w_down.tiled is not None and w_down.shape[1] == inner)
        h = self.activated_linear(x, w_up, activation, _tiled_out=tiled)
        return self.linear(h, w_down, None, defer=defer)

    def linear_rows(self, x, w, bias, out_f32=False):
        M, K = x.shape
        N = w.shape[0]
        y = self._new((M, N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_rows", _p(x), _p(w), _p(bias), _p(y), M, N, K, int(out_f32),
                   int(self.ROWS_THROUGH_LDS))
        return y

    def linear_tiled(self, x, w, bias, out_f32=False):
        M, K = x.shape
        N = w.shape[0]
        y = self._new((M, N), torch.float32 if out_f32 else None)
        self._call("gemm", "sl_gemm_tiled", _p(x), _p(w), _p(bias), _p(y), M, N, K, int(out_f32))
        return y

    # (library products of fewer than LIBRARY_PADDED_MAX_M rows run on a multiple of LIBRARY_ROW_STEP
    # rows: few distinct shapes, each of which can be tuned)

    def library_rows(self, M: int) -> int:
        """The number of rows a library product of M rows of x runs with."""
        if M >= self.LIBRARY_PADDED_MAX_M:
            return M
        return -(-M // self.LIBRARY_ROW_STEP) * self.LIBRARY_ROW_STEP

    F32_MFMA_MIN_M = 17           # float32 products of this many rows or more run on the matrix cores

    def linear_f32_mfma(self, x, w, bias):
        """Float32 product on the matrix cores, K % 16 == 0: more than 64 rows, K % 32 == 0 and 64 at least by products of
        three bfloat16 terms an operand, which together are the float (gemm_f32_split.h: closer to 64 bits than
        float32 instructions there), else by float32 instructions; float32 sums."""
        if self.act_dtype != torch.float32:
            raise KernelError("linear_f32_mfma is for the float32 table only")
        M, K = x.shape
        N = w.shape[0]
        y = self._new((M, N), torch.float32)
        shares = self._f32_shares(M, N, K)
        part = self._new((shares, M, N), torch.float32) if shares > 1 else None
        self._call("gemm", "sl_gemm_f32_mfma", _p(x), _p(w), _p(bias), _p(y), M, N, K, shares, _p(part))
        return y

    def _f32_shares(self, M, N, K):
        """Into how many shares of K a float32 product on the matrix cores is cut (``sl_gemm_f32_shares``)."""
        return int(self._lib["gemm"].sl_gemm_f32_shares(M, N, K, self._num_cus))

    def library_sums(self, x, w, out_dtype=None):
        """x w^T by the library, in bfloat16 or (``out_dtype`` float32) with the
        float32 sums kept.  Fewer than LIBRARY_PADDED_MAX_M rows are padded to a
        multiple of LIBRARY_ROW_STEP; the rows beyond M hold whatever the buffer
        held: a row of a product depends on its own row of x only (the library
        splits no K across rows), and they are cut off."""
        if self.act_dtype != torch.bfloat16:
            raise KernelError("the library GEMM is for the bfloat16 table only")
        M = x.shape[0]
        rows = self.library_rows(M)
        if rows != M:
            padded = self._new((rows, x.shape[1]))
            padded[:M].copy_(x)
            x = padded
        if out_dtype is None:
            if self._tuning:
                self._tuned.add((rows, w.shape[0], x.shape[1]))
            return torch.mm(x, w.t())[:M]
        return torch.mm(x, w.t(), out_dtype=out_dtype)[:M]

    def linear_library(self, x, w, bias):
        """Many rows: the library's product.  A bias is added to the float32
        sums before the one rounding to bfloat16, as the few-rows kernels do, so
        that a row gives the same values whichever path its step takes."""
        if bias is None:
            return self.library_sums(x, w)
        b16 = self._bias_as_bfloat16(bias)
        if b16 is not None:
            # a bias that bfloat16 holds exactly (one that a bfloat16 checkpoint stored): the library adds it
            # to its float32 sums in the product's epilogue, before the one rounding
            M = x.shape[0]
            rows = self.library_rows(M)
            if rows != M:
                padded = self._new((rows, x.shape[1]))
                padded[:M].copy_(x)
                x = padded
            if self._tuning:
                self._tuned.add((rows, w.shape[0], x.shape[1]))
            return torch.addmm(b16, x, w.t())[:M]
        return self.library_sums(x, w, torch.float32).add_(bias).to(torch.bfloat16)

    def _bias_as_bfloat16(self, bias):
        """``bias`` in bfloat16 when that loses nothing, else None; looked at once per bias (the first many-row
        product that adds it, which no captured step contains)."""
        if not hasattr(bias, "_as_bfloat16"):         # (kept on the tensor itself: it lives as long as the bias)
            b16 = bias.to(torch.bfloat16)
            bias._as_bfloat16 = b16 if bool(torch.equal(b16.float(), bias)) else None
        return bias._as_bfloat16

    @contextlib.contextmanager
    def library_tuning(self, max_ms: int = 30, results_file: Optional[str] = None):
        """Inside the block, every new shape of a library product is timed over
        the library's own candidate kernels (PyTorch's TunableOp, at most
        ``max_ms`` a candidate) and the fastest is kept for that exact shape;
        afterwards tuned shapes keep their choice and every other shape takes
        the library's default.  The choices are also written to
        ``results_file`` (default: a file in the temporary folder), which a
        later process reads instead of timing again.  The library's pick for
        the 7B shape's prompt products measured 26 % slower than the tuned one
        on MI355X."""
        tunable = getattr(torch.cuda, "tunable", None)
        if tunable is None:                      # a PyTorch without TunableOp: the library's defaults stay
            yield
            return
        if results_file is None:
            results_file = os.path.join(tempfile.gettempdir(),
                                        f"servelab_amd_tunableop_{os.getuid()}.csv")
        tunable.set_filename(results_file)
        tunable.set_max_tuning_duration(int(max_ms))
        tunable.enable(True)
        tunable.tuning_enable(True)
        self._tuning = True
        try:
            yield
        finally:
            self._tuning = False
            tunable.tuning_enable(False)           # the choices made stay in use; nothing new is timed
            self._tuned |= tuned_shapes(tunable.get_results())          # (those of the file among them)
