"""Fused SAE encoder: act((x - b_dec) @ W_enc + b_enc) on gfx950 MFMA.

Mirrors saeflow/kernels/encode.py:97-144 (fused_encode, best_config): same signature,
defaults, validation and errors. One prologue pass forms x' = cast(x - b_dec) once per
call (each x row block feeds every feature tile), the MFMA kernel stages x' and W_enc
tiles into LDS, and its epilogue applies b_enc plus ReLU / JumpReLU to the fp32
accumulators and counts each row's nonzeros for the dense -> CSR compaction.
"""

import ctypes
import statistics

import torch

from .. import _lib

ACTIVATIONS = {"relu": 0, "jumprelu": 1}  # encode.py:16

_last_config = None


# GROUP_N (runs of GROUP_N feature tiles, token tile by token tile) extends the reference's
# keys; a config without it (0) orders tiles by GROUP_M as the reference does (encode.py:44-52).
CONFIG_KEYS = ("BLOCK_M", "BLOCK_N", "BLOCK_K", "GROUP_M", "NUM_WAVES", "GROUP_N")


def _config_array(config, w_dtype):
    """`config` dict -> int32[6] {BLOCK_M, BLOCK_N, BLOCK_K, GROUP_M, NUM_WAVES, GROUP_N} (None =
    the default tiling). Missing keys take the defaults of the tiling BLOCK_N names."""
    if config is None:
        return None
    bn = int(config.get("BLOCK_N", 256)) if isinstance(config, dict) else 256
    bk = (32 if w_dtype == torch.float32 else 64) // (2 if bn == 128 else 1)
    try:
        vals = [int(config.get("BLOCK_M", 256)), bn, int(config.get("BLOCK_K", bk)), int(config.get("GROUP_M", 4)),
                int(config.get("NUM_WAVES", 8 if bn == 256 else 4)), int(config.get("GROUP_N", 0))]
    except AttributeError:
        raise ValueError(f"config must be a dict of block sizes, got {config!r}") from None
    return (ctypes.c_int32 * 6)(*vals)


def _vector(t, n, name):
    if t.dim() != 1 or t.numel() != n:
        raise ValueError(f"{name} must have shape [{n}], got {list(t.shape)}")
    return t.contiguous()


# Autotuning (reference encode.py:19-33, 94: triton.autotune keyed on M, N, K): on the first
# call for a shape key without an explicit `config`, the compiled tilings are timed against
# each other and the fastest is kept for the key. All tilings give bit-identical results (the same MFMA
# chain per output element), so the pick changes speed only. Small problems take the
# default tiling untimed.
AUTOTUNE = True
AUTOTUNE_MIN_FLOPS = 1 << 36
AUTOTUNE_ROUNDS = 3
# The 8-wave and 4-wave 256x256 tilings (both persistent on whole tiles) are within about 1% of
# each other at C3 and C5 and 1-3% apart at C4, near the spread between runs: a 2% margin keeps
# the default unless a candidate is clearly faster, so the pick rarely changes from one process
# to the next (results are bit-identical either way).
AUTOTUNE_MARGIN = 0.02
_tuned = {}


def _candidates(w_dtype):
    bk = 32 if w_dtype == torch.float32 else 64
    return [{"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": bk, "GROUP_M": 1, "NUM_WAVES": 8, "GROUP_N": 8},
            {"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": bk, "GROUP_M": 4, "NUM_WAVES": 8, "GROUP_N": 0},
            {"BLOCK_M": 256, "BLOCK_N": 256, "BLOCK_K": bk, "GROUP_M": 1, "NUM_WAVES": 4, "GROUP_N": 8},
            {"BLOCK_M": 256, "BLOCK_N": 128, "BLOCK_K": bk // 2, "GROUP_M": 4, "NUM_WAVES": 4, "GROUP_N": 0}]


def _default_tiling(M, N, K, W_enc):
    """The tiling of a call without `config`, as a config: the 256x256 tile, or the small one that the
    library estimates to be faster for this shape and layout."""
    got = (ctypes.c_int32 * 6)()
    _lib.check(_lib.load().sf_encode_tiling(M, N, K, _lib.ptr(W_enc), W_enc.stride(0), W_enc.stride(1),
                                            _lib.dtype_code(W_enc, "W_enc"), 0, got))
    return dict(zip(CONFIG_KEYS, got))


def _autotune(key, launch, cands, row_nnz, dev):
    """Fastest candidate tiling for `key`. Every candidate is launched once to warm up, then
    timed over AUTOTUNE_ROUNDS interleaved rounds (one launch per candidate per round, so
    clock and power drift spreads over all of them) and ranked by its median; a candidate
    replaces the incumbent, the default first, only when at least AUTOTUNE_MARGIN faster.
    The caller's row_nnz is restored afterwards (the reference zeroes it for its benchmark
    runs, reset_to_zero=["nnz_ptr"])."""
    if key not in _tuned:
        saved = row_nnz.clone() if row_nnz is not None else None
        stream = torch.cuda.current_stream(dev)  # the stream the launches go to
        for cfg in cands:
            launch(cfg)
        events = [[] for _ in cands]
        for _ in range(AUTOTUNE_ROUNDS):
            for i, cfg in enumerate(cands):
                start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record(stream)
                launch(cfg)
                end.record(stream)
                events[i].append((start, end))
        stream.synchronize()
        med = [statistics.median(s.elapsed_time(e) for s, e in ev) for ev in events]
        best = 0
        for i in range(1, len(cands)):
            if med[i] < med[best] * (1.0 - AUTOTUNE_MARGIN):
                best = i
        if saved is not None:
            row_nnz.copy_(saved)
        _tuned[key] = cands[best]
    return _tuned[key]


def _launch(x, W_enc, b_enc, b_dec, threshold, act, out, row_nnz, config):
    M, K = x.shape
    N = W_enc.shape[1]
    dev = _lib.require_gpu(("x", x), ("W_enc", W_enc), ("b_enc", b_enc), ("b_dec", b_dec),
                           ("threshold", threshold), ("row_nnz", row_nnz))
    b_enc = _vector(b_enc, N, "b_enc")
    b_dec = _vector(b_dec, K, "b_dec")
    if threshold is not None:
        threshold = _vector(threshold, N, "threshold")
    if row_nnz is not None:
        if row_nnz.dtype != torch.int32 or row_nnz.dim() != 1 or row_nnz.numel() != M or not row_nnz.is_contiguous():
            raise ValueError(f"row_nnz must be a contiguous int32 tensor of shape [{M}]")
    lib = _lib.load()
    thr_code = _lib.dtype_code(threshold, "threshold") if threshold is not None else 0
    w_code = _lib.dtype_code(W_enc, "W_enc")
    # x' = cast(x - b_dec) scratch (from torch's caching allocator, reused across calls)
    ws = torch.empty(max(_lib.encode_workspace_bytes(M, K, w_code), 16), dtype=torch.uint8, device=x.device)

    def launch(config):
        cfg = _config_array(config, W_enc.dtype)
        with _lib.device(dev):
            _lib.check(lib.sf_encode(
                _lib.ptr(x), x.stride(0), x.stride(1), _lib.dtype_code(x, "x"),
                _lib.ptr(W_enc), W_enc.stride(0), W_enc.stride(1), w_code,
                _lib.ptr(b_enc), _lib.dtype_code(b_enc, "b_enc"), _lib.ptr(b_dec), _lib.dtype_code(b_dec, "b_dec"),
                _lib.ptr(threshold), thr_code,
                _lib.ptr(out), out.stride(0), out.stride(1), _lib.dtype_code(out, "out"),
                _lib.ptr(row_nnz), M, N, K, act, cfg, _lib.ptr(ws), ws.numel(), _lib.stream(dev)))
        return cfg

    explicit = config is not None
    if not explicit and AUTOTUNE and 2 * M * N * K >= AUTOTUNE_MIN_FLOPS:
        # (the alignment decides how W_enc is staged)
        key = (M, N, K, x.dtype, W_enc.dtype, out.dtype, W_enc.stride(), W_enc.data_ptr() % 16 == 0, act)
        config = _tuned.get(key)
        if config is None and not torch.cuda.is_current_stream_capturing():  # no timing under graph capture
            cands, own = _candidates(W_enc.dtype), _default_tiling(M, N, K, W_enc)
            # a small tile (ragged shapes, a W_enc whose rows are not 16-B aligned) is timed with them
            config = _autotune(key, launch, cands if own in cands else [*cands, own], row_nnz, dev)
    cfg = launch(config)
    if explicit:
        return  # a pinned tiling is not a tuning result: best_config() keeps reporting the last one
    global _last_config
    if cfg is None:
        got = (ctypes.c_int32 * 6)()
        _lib.check(lib.sf_encode_config(M, N, K, w_code, got))
        cfg = got
    _last_config = dict(zip(CONFIG_KEYS, list(cfg)))


def fused_encode(x, W_enc, b_enc, b_dec, threshold=None, activation="relu", *,
                 out_dtype=None, row_nnz=None, config=None, allow_tf32=None):
    """The SAE encoder on the matrix cores: returns the [M, d_sae] features
    act((x - b_dec) W_enc + b_enc), with fp32 sums.

    x: tokens [M, d_in] in fp32, bf16 or fp16; W_enc: [d_in, d_sae] with any strides.
    activation: "relu", or "jumprelu" with a per-feature `threshold` [d_sae].
    row_nnz: optional zeroed int32 [M] buffer; receives each row's nonzero count
      (counted on the stored, rounded values).
    config: dict {BLOCK_M, BLOCK_N, BLOCK_K, GROUP_M, NUM_WAVES, GROUP_N} naming a compiled
      tiling: {256, 256, 64 (32 for fp32), G, 8 or 4, GN} (256x256 tiles of 8 waves of 128x64
      or 4 waves of 128x128) or {256, 128, 32 (16), G, 4, GN} (two workgroups per CU), or a small
      tile {32, 64, 64 (32), G, 2, GN}, {128, 64, 64 (32), G, 4, GN}, {128, 128, 32 (16),
      G, 4, GN}, {32 | 64, 128, 64 (32), G, 4, GN}, {160, 256, 64 (32), G, 4, GN}, and its
      tile order: runs of GN feature tiles if GN > 0, else runs of G token tiles (GN 0, the
      default of a dict without it); None = autotuned, or, for problems too small to time, the
      256x256 tile or a small one by an estimate of both.
    allow_tf32: accepted for compatibility; gfx950 has no xf32 matrix path, so fp32 inputs
      always run the IEEE fp32 MFMA path.
    """
    if activation not in ACTIVATIONS:
        raise ValueError(f"fused_encode supports {list(ACTIVATIONS)}, got {activation!r}")
    if activation == "jumprelu" and threshold is None:
        raise ValueError("jumprelu needs a threshold")
    M, K = x.shape
    K_w, N = W_enc.shape
    if K != K_w:
        raise ValueError(f"x has d_in={K} but W_enc has d_in={K_w}")
    out = torch.empty(M, N, device=x.device, dtype=out_dtype or x.dtype)
    if M == 0:
        return out
    _launch(x, W_enc, b_enc, b_dec, threshold if activation == "jumprelu" else None, ACTIVATIONS[activation],
            out, row_nnz, config)
    return out


def encode_pre(x, W_enc, b_enc, b_dec, *, out_dtype=None, config=None):
    """(x - b_dec) @ W_enc + b_enc -> [M, d_sae] (the bare pre-activation, reference.py:36-37)."""
    M, K = x.shape
    K_w, N = W_enc.shape
    if K != K_w:
        raise ValueError(f"x has d_in={K} but W_enc has d_in={K_w}")
    out = torch.empty(M, N, device=x.device, dtype=out_dtype or x.dtype)
    if M == 0:
        return out
    _launch(x, W_enc, b_enc, b_dec, None, _lib.ACT["none"], out, None, config)
    return out


def encode_rows(x, W_enc, b_enc, b_dec, threshold=None, activation="relu", *, cap, out_dtype=None,
                row_floor=None, config=None):
    """Fused encode into per-row candidate lists instead of a dense [M, d_sae] output.

    Returns (cand_cnt int32 [M], cand_idx int32 [M, cap], cand_val [M, cap]): row m's kept
    values (the nonzeros fused_encode would store) as (column, value) pairs in
    cand_idx/cand_val[m, :min(cnt, cap)], in no particular order; cand_cnt[m] counts them
    all, so cand_cnt[m] > cap flags an overflowed row. row_floor (float32 [M], relu only)
    keeps only stored values >= row_floor[m]. Same fused kernels as fused_encode: the
    256x256 tiling with 8 waves and the small tiles.
    """
    if activation not in ACTIVATIONS:
        raise ValueError(f"encode_rows supports {list(ACTIVATIONS)}, got {activation!r}")
    if activation == "jumprelu" and threshold is None:
        raise ValueError("jumprelu needs a threshold")
    M, K = x.shape
    K_w, N = W_enc.shape
    if K != K_w:
        raise ValueError(f"x has d_in={K} but W_enc has d_in={K_w}")
    vdt = out_dtype or x.dtype
    # with features to encode, the call clears the counts itself (without, it checks its arguments)
    cnt = (torch.empty if N else torch.zeros)(M, device=x.device, dtype=torch.int32)
    idx = torch.empty(M, cap, device=x.device, dtype=torch.int32)
    val = torch.empty(M, cap, device=x.device, dtype=vdt)
    if M == 0:
        return cnt, idx, val
    threshold = threshold if activation == "jumprelu" else None
    dev = _lib.require_gpu(("x", x), ("W_enc", W_enc), ("b_enc", b_enc), ("b_dec", b_dec),
                           ("threshold", threshold), ("row_floor", row_floor))
    b_enc = _vector(b_enc, N, "b_enc")
    b_dec = _vector(b_dec, K, "b_dec")
    if threshold is not None:
        threshold = _vector(threshold, N, "threshold")
    if row_floor is not None:
        if row_floor.dtype != torch.float32 or row_floor.dim() != 1 or row_floor.numel() != M:
            raise ValueError(f"row_floor must be a float32 tensor of shape [{M}]")
        row_floor = row_floor.contiguous()
    cfg = _config_array(config, W_enc.dtype)
    lib = _lib.load()
    w_code = _lib.dtype_code(W_enc, "W_enc")
    ws = torch.empty(max(_lib.encode_workspace_bytes(M, K, w_code), 16), dtype=torch.uint8, device=x.device)
    encode = lib.sf_encode_rows_cleared if N else lib.sf_encode_rows
    with _lib.device(dev):
        _lib.check(encode(
            _lib.ptr(x), x.stride(0), x.stride(1), _lib.dtype_code(x, "x"),
            _lib.ptr(W_enc), W_enc.stride(0), W_enc.stride(1), w_code,
            _lib.ptr(b_enc), _lib.dtype_code(b_enc, "b_enc"), _lib.ptr(b_dec), _lib.dtype_code(b_dec, "b_dec"),
            _lib.ptr(threshold), _lib.dtype_code(threshold, "threshold") if threshold is not None else 0,
            _lib.ptr(row_floor), _lib.ptr(cnt), _lib.ptr(idx), _lib.ptr(val), _lib.dtype_code(val, "out"), cap,
            M, N, K, ACTIVATIONS[activation], cfg, _lib.ptr(ws), ws.numel(), _lib.stream(dev)))
    return cnt, idx, val


def encode_gather(x, W_enc, b_enc, b_dec, rows, n_rows, threshold=None, activation="relu", *, row_off=0, out_rows,
                  out_dtype=None):
    """fused_encode of the tokens x[rows[row_off + i]] for i < clamp(n_rows - row_off, 0, out_rows),
    where n_rows is an int32 count in device memory: returns [out_rows, d_sae] whose rows past
    the live ones are unspecified. Values are bit-identical to fused_encode's for the same tokens.
    Nothing is read back to the host, so the count may come from a kernel still in flight."""
    if activation not in ACTIVATIONS:
        raise ValueError(f"encode_gather supports {list(ACTIVATIONS)}, got {activation!r}")
    if activation == "jumprelu" and threshold is None:
        raise ValueError("jumprelu needs a threshold")
    Mx, K = x.shape
    K_w, N = W_enc.shape
    if K != K_w:
        raise ValueError(f"x has d_in={K} but W_enc has d_in={K_w}")
    for name, t in (("rows", rows), ("n_rows", n_rows)):
        if t.dtype != torch.int32 or not t.is_contiguous():
            raise ValueError(f"{name} must be a contiguous int32 tensor")
    out = torch.empty(out_rows, N, device=x.device, dtype=out_dtype or x.dtype)
    if out_rows == 0:
        return out
    threshold = threshold if activation == "jumprelu" else None
    dev = _lib.require_gpu(("x", x), ("W_enc", W_enc), ("b_enc", b_enc), ("b_dec", b_dec), ("threshold", threshold),
                           ("rows", rows), ("n_rows", n_rows))
    b_enc = _vector(b_enc, N, "b_enc")
    b_dec = _vector(b_dec, K, "b_dec")
    if threshold is not None:
        threshold = _vector(threshold, N, "threshold")
    lib = _lib.load()
    w_code = _lib.dtype_code(W_enc, "W_enc")
    ws = torch.empty(max(_lib.encode_workspace_bytes(out_rows, K, w_code), 16), dtype=torch.uint8, device=x.device)
    with _lib.device(dev):
        _lib.check(lib.sf_encode_gather(
            _lib.ptr(x), x.stride(0), x.stride(1), _lib.dtype_code(x, "x"), Mx, _lib.ptr(rows), _lib.ptr(n_rows),
            row_off, _lib.ptr(W_enc), W_enc.stride(0), W_enc.stride(1), w_code,
            _lib.ptr(b_enc), _lib.dtype_code(b_enc, "b_enc"), _lib.ptr(b_dec), _lib.dtype_code(b_dec, "b_dec"),
            _lib.ptr(threshold), _lib.dtype_code(threshold, "threshold") if threshold is not None else 0,
            _lib.ptr(out), out.stride(0), out.stride(1), _lib.dtype_code(out, "out"), out_rows, N, K,
            ACTIVATIONS[activation], _lib.ptr(ws), ws.numel(), _lib.stream(dev)))
    return out


def best_config():
    """Tiling chosen by the most recent launch that chose one, i.e. a call without `config`
    (None until such a call): the autotuner's timed pick for that shape, which may be a small tile,
    or the default tiling of a problem that was not timed (too small, or first met under graph
    capture; encode.py:142-144), which stands for the small tile that such a problem may run instead
    (same bits). Calls that pin `config` leave it unchanged."""
    return None if _last_config is None else dict(_last_config)
