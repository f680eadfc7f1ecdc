"""Zero-copy device path: fused prune+compress into a flat cache, SpMVs with one row per head.

Everything stays on the device, in the order of the current stream; the host waits for a packed size where the caller did
not provide a capacity or asks for it, and for nothing else.  Such a size may be there before the kernel has stored its last
values: a result that another stream is to use, or an input that another stream may write to or free, waits for this one as with
any torch call (an event recorded, or wait_stream called, after the call).
"""
import ctypes
import math
import threading
import weakref

import torch

from ._lib import check, host, lib

class Workspace:
    """Scratch memory for the entry points that need it (split partials, compressor scans), owned by one caller.

    A cache, a decode loop or a benchmark that records its calls into a HIP graph creates one sized for its largest
    call BEFORE capturing and passes it as `ws=`: the buffer then never moves, and calls on different streams with
    different workspaces are independent.  `get` hands out the buffer if it is large enough; growing replaces it but
    keeps the old buffers alive (a captured graph may still point at them), and growing while the current stream is
    being captured is an error - unless it holds the least that an attention call does with, if slower."""

    _status = ()        # status words of the producers, zero between two calls; the last ones are in use
    _spoilt = False     # the last ones are not zero any more

    def __init__(self, device, nbytes=1 << 20):
        self.device = torch.device(device)
        self._bufs = [torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=self.device)]
        self._status = []

    @property
    def tensor(self):
        return self._bufs[-1]

    def reserve(self, nbytes):
        """Makes room for nbytes; to be called outside any graph capture."""
        if self.tensor.numel() < nbytes:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("workspace of %d bytes is too small for a call that needs %d and cannot grow while "
                                   "the stream is being captured: reserve() it before the capture"
                                   % (self.tensor.numel(), nbytes))
            self._bufs.append(torch.empty(int(nbytes), dtype=torch.uint8, device=self.device))
        return self.tensor

    def get(self, nbytes, call=None):
        """call: (tokens, window, rows) of an attention call, which nbytes is the best size for."""
        if (call is not None and attention_workspace_least(*call) <= self.tensor.numel() < nbytes
                and torch.cuda.is_current_stream_capturing()):
            return self.tensor
        return self.reserve(nbytes)

    def status(self, words):
        """`words` kept status words (mstf_status_bytes) for a producer on the current stream, or None where they would have
        to be made while it is being captured."""
        if self._spoilt or not self._status or self._status[-1].numel() < words:
            if torch.cuda.is_current_stream_capturing():
                return None
            # (as the words before them at least, twice that if they were too few: all of them together are bounded)
            last = self._status[-1].numel() if self._status else 0
            room = max(words, 4096, last if words <= last else 2 * last)
            self._status = [*self._status, torch.zeros(room, dtype=torch.int64, device=self.device)]
            self._spoilt = False
        return self._status[-1]

    def status_spoilt(self, words):
        """A producer gave up over these words: they are not zero any more.  The next producer makes others, cleared on its own
        stream, which need not be the one that this is called on."""
        if self._status and self._status[-1] is words:
            self._spoilt = True


def status_words(units, sides=1):
    """mstf_status_bytes in words, of a producer's call over `units` blocks a side."""
    return 16 + sides * (units + 242)


_WS = {}


def _stream():
    # the handle alone: torch.cuda.current_stream() makes an object first, 3 us in front of every launch
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


_LANDING = threading.local()     # a thread's pinned word and the result mstf_read_word fills, see read_word


def read_word(t):
    """The value of a one-element int64 device tensor on the host (a wait for the current stream, as int(t) is)."""
    if not (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == torch.int64 and t.numel() == 1
            and t.device.index == torch._C._cuda_getDevice()):
        return int(t)
    own = _landing_word()
    check(lib().mstf_read_word(_stream(), t.data_ptr(), own[1], own[3]), "mstf_read_word")
    return own[2].value


def _landing_word():
    """This thread's (pinned word, its address, result, its address) for the calls that wait for a word."""
    own = getattr(_LANDING, "own", None)
    if own is None:
        word, value = torch.empty(1, dtype=torch.int64, pin_memory=True), ctypes.c_int64()
        own = _LANDING.own = (word, word.data_ptr(), value, ctypes.addressof(value))
    return own


class _LandingPair:
    """The pinned words that a call which returns without waiting has its two totals stored to (mstf_landing_take)."""
    __slots__ = ("pair", "stream", "device", "ws", "words", "_give")
    EMPTY, NOT_LANDED = -(1 << 63) + 1, -(1 << 63) + 2

    def __init__(self, pair, stream, ws, words, device=None):
        """device: the one that was current at the call, which `stream` is a handle of."""
        self.pair, self.stream, self.device, self._give = pair, stream, device, lib().mstf_landing_give
        self.ws, self.words = ws and weakref.ref(ws), words

    def read(self, side):
        """The total, or None where the call was recorded into a graph."""
        at = self.pair + 8 * side
        value = ctypes.c_int64.from_address(at).value
        if value == self.EMPTY:
            if self.device == torch._C._cuda_getDevice():
                value = self._wait(at)
            else:
                with torch.cuda.device(self.device):    # (a default stream's handle is the same on every device)
                    value = self._wait(at)
        return None if value == self.NOT_LANDED else value

    def _wait(self, at):
        value = ctypes.c_int64()
        check(lib().mstf_landing_wait(self.stream, at, ctypes.addressof(value)), "mstf_landing_wait")
        return value.value

    def spoilt(self):
        ws = self.ws and self.ws()
        if ws is not None:
            ws.status_spoilt(self.words)

    def __del__(self):
        self._give(self.pair)


def attention_workspace_least(tokens, window, rows):
    """Bytes that an attention call over `tokens` compressed tokens and a window demands of its workspace."""
    return (rows * (-(-tokens // 512) + -(-window // 64)) * 520 + 255) // 256 * 256


def workspace(device, nbytes, ws=None, call=None):
    """The scratch tensor for a call that needs nbytes: the caller's Workspace (`ws`) or, for the mirrors of the
    reference's operators, which have no such argument, a default one per (device, stream) - so two streams never
    share a buffer unless the caller passes the same Workspace to both.  call: see Workspace.get."""
    if ws is not None:
        if not isinstance(ws, Workspace):
            return ws
        t = ws.tensor
        return t if t.numel() >= nbytes else ws.get(nbytes, call)
    device = torch.device(device)
    key = (device.type, device.index if device.index is not None else torch.cuda.current_device(), _stream())
    w = _WS.get(key)
    if w is None:
        w = _WS[key] = Workspace(device)
    return w.get(nbytes, call)


def _call(fn, ws, device, call, *args):
    """One of the native calls (csrc/host.cpp), with the scratch memory at hand or, where it answers that it needs more,
    with what `workspace` finds."""
    if ws is None:
        w = _WS.get((device.type, device.index, _stream())) if device.type == "cuda" else None
        t = None if w is None else w._bufs[-1]
    else:
        t = ws._bufs[-1] if isinstance(ws, Workspace) else ws
    r = fn(*args, t, 0)
    if type(r) is int:
        r = fn(*args, workspace(device, r, ws, call), 1)
    return r


def _own_workspace(ws, device):
    """The Workspace that keeps a producer's status words, None where the caller brought a bare buffer or tensors of another
    device than the current one, on whose stream the words are cleared and the launch goes."""
    if device.type != "cuda" or device.index != torch._C._cuda_getDevice():
        return None
    if ws is None:
        key = ("cuda", device.index, _stream())
        ws = _WS.get(key)
        if ws is None:
            ws = _WS[key] = Workspace(device)
    return ws if isinstance(ws, Workspace) and ws.device.type == "cuda" else None


def gave_up(ws, words, what):
    if ws is not None:
        ws.status_spoilt(words)
    raise RuntimeError(what)


def kth_from_sparsity(sparsity, head_dim):
    """Rank of the pruning threshold: max(1, int(target_sparsity * D)) as in dh_prune_key."""
    return max(1, int(sparsity * head_dim))


def _gave_up(total):
    return not 0 <= total <= 1 << 62


_GAVE_UP = "the compressor gave up waiting for an earlier workgroup; the packed values are incomplete"


class CompressedKV:
    """One side (K or V) of the compressed cache, flat on the device.

    bmp int64 [B, T], idx int32 [B, T+1], nz fp16 flat, nz_off int32 [B] (16-byte units)."""

    _landing = None     # _LandingPair that gets the total too; given back once the total is read
    _used = None        # the total, from there

    def __init__(self, bmp, idx, nz, nz_off, tokens, head_dim, is_value, total_halfs=None, landing=None):
        self.bmp, self.idx, self.nz, self.nz_off = bmp, idx, nz, nz_off
        self.tokens, self.head_dim, self.is_value = tokens, head_dim, is_value
        self.total_halfs = total_halfs
        self._landing = landing

    def __getstate__(self):
        # a copy has the total from its own tensor (total_halfs): the words that it landed in go with the call
        return {name: value for name, value in self.__dict__.items() if name != "_landing"}

    @property
    def heads(self):
        return self.bmp.shape[0]

    def used_halfs(self):
        """Number of fp16 values in use (the total is read once; the values themselves may be on their way yet, see above).
        The one-pass compressor reports a wait that ran out - which the dispatch order rules out - as a total of all ones:
        that raises here."""
        landing = self._landing     # (in front of _used, which is set before this one goes: another thread may be between the two)
        if self._used is not None:
            return self._used
        n = landing.read(int(self.is_value)) if landing is not None else None
        landed = n is not None
        if not landed:
            n = read_word(self.total_halfs)
        if _gave_up(n):
            if landed:
                landing.spoilt()
            raise RuntimeError(_GAVE_UP)
        if landed:
            self._used = n
        self._landing = None
        return n

    def packed(self):
        """The used part of the flat value buffer (needs the host-side size), complete in the order of the call's stream."""
        return self.nz[:self.used_halfs()]

    def nbytes(self):
        """Algorithmic size: bitmaps + offsets + packed values actually used."""
        used = self.nz.numel() if self.total_halfs is None else self.used_halfs()
        return self.bmp.numel() * 8 + self.idx.numel() * 4 + used * 2


def prune_rows(x, kth, out=None):
    """dh_prune_key / dh_prune_value on the last axis (D = 128)."""
    assert x.is_cuda and x.dtype == torch.float16 and x.is_contiguous()
    D = x.shape[-1]
    y = torch.empty_like(x) if out is None else out
    check(lib().mstf_prune_rows_f16(_stream(), x.data_ptr(), y.data_ptr(), x.numel() // D, D, int(kth)),
          "mstf_prune_rows_f16")
    return y


def compress(x, is_value, kth=0, capacity_halfs=None, ws=None):
    """Prune (kth > 0) and compress x [B, M, N] into the bitmap format.

    With capacity_halfs=None the packed size is read back once (like the reference's .item()) and the values are stored by
    a launch behind that; with a capacity nothing is waited for and `total_halfs` stays on the device."""
    assert x.is_cuda and x.dtype == torch.float16 and x.dim() == 3
    x = x.contiguous()
    B, M, N = x.shape
    T = M * N // 64
    dev = x.device
    L = lib()
    bmp = torch.empty((B, T), dtype=torch.int64, device=dev)
    idx = torch.empty((B, T + 1), dtype=torch.int32, device=dev)
    nz_off = torch.empty((B,), dtype=torch.int32, device=dev)
    total = torch.empty((1,), dtype=torch.int64, device=dev)
    wsb = L.mstf_compress_workspace_bytes(B, M, N)
    ws = workspace(dev, wsb, ws)
    fn = L.mstf_compress_value_f16 if is_value else L.mstf_compress_key_f16
    name = "mstf_compress_value_f16" if is_value else "mstf_compress_key_f16"
    if capacity_halfs is None:
        check(fn(_stream(), x.data_ptr(), B, M, N, int(kth), bmp.data_ptr(), idx.data_ptr(), nz_off.data_ptr(),
                 total.data_ptr(), None, 0, ws.data_ptr(), ws.numel()), name)
        n = read_word(total)
        nz = torch.empty((max(n, 8),), dtype=torch.float16, device=dev)
        sc = L.mstf_scatter_value_f16 if is_value else L.mstf_scatter_key_f16
        check(sc(_stream(), x.data_ptr(), B, M, N, bmp.data_ptr(), idx.data_ptr(), nz_off.data_ptr(), nz.data_ptr(),
                 n), name.replace("compress", "scatter"))
        if n == 0:
            nz.zero_()
        return CompressedKV(bmp, idx, nz if n == 0 else nz[:n], nz_off, M, N, is_value, n)
    nz = torch.empty((int(capacity_halfs),), dtype=torch.float16, device=dev)
    check(fn(_stream(), x.data_ptr(), B, M, N, int(kth), bmp.data_ptr(), idx.data_ptr(), nz_off.data_ptr(),
             total.data_ptr(), nz.data_ptr(), int(capacity_halfs), ws.data_ptr(), ws.numel()), name)
    return CompressedKV(bmp, idx, nz, nz_off, M, N, is_value, total)


def _capacity(capacity_halfs):
    capacity = int(capacity_halfs)
    if capacity < 0:    # (-1 is 'none given' to the native calls)
        raise RuntimeError("capacity_halfs must not be negative")
    return capacity


def compress_kv(k, v, kth_k=0, kth_v=0, capacity_halfs=None, ws=None):
    """compress(k, False, kth_k) and compress(v, True, kth_v) of the same tokens in one launch (mstf_compress_kv_f16):
    identical outputs, less time - a launch of both sides runs less in lockstep than two launches of one side each.
    k, v: [B, M, N]; capacity_halfs (default: room for the dense rows) sizes both value buffers, the totals stay on
    the device.  Returns (CompressedKV of the keys, CompressedKV of the values)."""
    assert k.dim() == 3
    B, M, N = k.shape
    capacity = -1 if capacity_halfs is None else _capacity(capacity_halfs)
    pair = lib().mstf_landing_take()
    own = _own_workspace(ws, k.device) if pair else None
    words = own.status(status_words(B * (M // 64), 2)) if own else None
    landing = _LandingPair(pair, _stream(), own, words, torch._C._cuda_getDevice()) if pair else None
    kb, ki, ko, kt, kn, vb, vi, vo, vt, vn = _call(host().compress_kv, ws, k.device, None, k, v, int(kth_k), int(kth_v),
                                                   capacity, pair or 0, words)
    return (CompressedKV(kb, ki, kn, ko, M, N, False, kt, landing), CompressedKV(vb, vi, vn, vo, M, N, True, vt, landing))


def proj_source(x, cos=None, sin=None, rot=None):
    """The mstf_proj_source of x [batch, rows, heads, 128] fp16 (any strides with contiguous channels, e.g. a view of
    a projection output [batch, rows, heads * 128]).  cos, sin: [rows, 128] or [batch, rows, 128] fp16 (keys only);
    rot: where the rotated rows go, shaped like x (default: x itself, in place).  Returns (struct, rot)."""
    from ._lib import ProjSource
    assert x.is_cuda and x.dtype == torch.float16 and x.dim() == 4 and x.stride(3) == 1
    src = ProjSource()
    src.x = x.data_ptr()
    src.stride_batch, src.stride_token, src.stride_head = x.stride(0), x.stride(1), x.stride(2)
    src.batch, src.rows, src.heads = x.shape[0], x.shape[1], x.shape[2]
    if cos is not None:
        assert sin is not None and cos.dtype == sin.dtype == torch.float16 and cos.shape == sin.shape
        assert cos.stride(-1) == 1 and sin.stride() == cos.stride() and cos.shape[-2] >= x.shape[1]
        rot = x if rot is None else rot
        assert rot.shape == x.shape and rot.dtype == torch.float16 and rot.stride(3) == 1
        src.cos, src.sin = cos.data_ptr(), sin.data_ptr()
        src.rope_stride_batch = cos.stride(0) if cos.dim() == 3 and cos.shape[0] > 1 else 0
        src.rope_stride_token = cos.stride(-2)
        src.rot = rot.data_ptr()
        src.rot_stride_batch, src.rot_stride_token, src.rot_stride_head = rot.stride(0), rot.stride(1), rot.stride(2)
    return src, rot


def compress_proj(x, is_value, kth, M, cos=None, sin=None, rot=None, capacity_halfs=None, ws=None):
    """Prune and compress the first M tokens of x [batch, rows, heads, 128] where the projection left them, the keys
    rotated first when cos / sin are given (all rows are rotated and written to rot).  Heads are numbered
    batch * heads + head.  Returns (CompressedKV, rot); without a capacity it waits for the size, not for the last values
    and rotated rows."""
    assert x.dim() == 4
    batch, _, heads, N = x.shape
    if cos is not None and rot is None:
        rot = x
    capacity = -1 if capacity_halfs is None else _capacity(capacity_halfs)
    sized = capacity_halfs is None and M != 0
    own = _own_workspace(ws, x.device) if sized else None
    words = own.status(status_words(batch * heads * (M // 64))) if own else None
    bmp, idx, nz_off, total, nz, n = _call(host().compress_proj, ws, x.device, None, x, int(is_value), int(kth), int(M), cos, sin,
                                           rot, capacity, _landing_word()[1] if sized else 0, 1, words)
    if M == 0:
        return None, rot
    if sized and n < 0:
        gave_up(own, words, _GAVE_UP)
    return CompressedKV(bmp, idx, nz, nz_off, M, N, is_value, n if sized else total), rot


def compress_proj_both(kx, vx, kth_k, kth_v, M, cos, sin, ws=None):
    """compress_proj of the keys, rotated in place, and of the values of the same tokens (M > 0), for a caller who wants both: the
    second launch goes out while the first one runs, not behind a wait for its size.  Returns a function to be called
    once, behind the caller's other launches, which waits for both sizes and returns the two CompressedKV, or raises."""
    assert kx.dim() == 4 and vx.dim() == 4 and M > 0
    device = torch._C._cuda_getDevice() if kx.is_cuda else None
    pair = lib().mstf_landing_take() if kx.is_cuda and kx.device.index == device and vx.device == kx.device else None
    if not pair:
        both = compress_proj(kx, False, kth_k, M, cos, sin, ws=ws)[0], compress_proj(vx, True, kth_v, M, ws=ws)[0]
        return lambda: both
    own = _own_workspace(ws, kx.device)
    words = own.status(status_words(max(x.shape[0] * x.shape[2] for x in (kx, vx)) * (M // 64))) if own else None
    landing = _LandingPair(pair, _stream(), own, words, device)
    sides = [_call(host().compress_proj, ws, x.device, None, x, side, int(kth), int(M), *rope, -1, pair + 8 * side, 0, words)
             for side, (x, kth, rope) in enumerate(((kx, kth_k, (cos, sin, kx)), (vx, kth_v, (None,) * 3)))]

    def settle():
        sizes = [landing.read(side) for side in (0, 1)]
        if any(map(_gave_up, sizes)):
            landing.spoilt()
            raise RuntimeError(_GAVE_UP)
        return tuple(CompressedKV(bmp, idx, nz[:n], nz_off, M, x.shape[3], bool(side), n)
                     for side, (n, x, (bmp, idx, nz_off, _, nz, _)) in enumerate(zip(sizes, (kx, vx), sides)))
    return settle


def key_spmv(ck, q, groups, n_rows=1, out=None):
    """scores[bq, n, t] = sum_d K[bq // groups][t, d] * q[bq, n, d]   (unscaled).  q: [Bq, n_rows, D]."""
    assert q.dtype == torch.float16 and q.is_contiguous()
    Bq = q.numel() // (n_rows * ck.head_dim)
    C = torch.empty((Bq, n_rows, ck.tokens), dtype=torch.float16, device=q.device) if out is None else out
    check(lib().mstf_key_spmv_f16(_stream(), ck.bmp.data_ptr(), ck.nz.data_ptr(), ck.idx.data_ptr(),
                                  ck.nz_off.data_ptr(), q.data_ptr(), C.data_ptr(), ck.tokens, ck.head_dim, Bq,
                                  groups, n_rows), "mstf_key_spmv_f16")
    return C


def value_spmv(cv, p, groups, n_rows=1, out=None, ws=None):
    """out[bq, n, d] = sum_t V[bq // groups][t, d] * p[bq, n, t].  p: [Bq, n_rows, Lc]."""
    assert p.dtype == torch.float16 and p.is_contiguous()
    Bq = p.numel() // (n_rows * cv.tokens)
    L = lib()
    C = torch.empty((Bq, n_rows, cv.head_dim), dtype=torch.float16, device=p.device) if out is None else out
    wsb = L.mstf_value_spmv_workspace_bytes(cv.head_dim, cv.tokens, Bq, groups, n_rows)
    ws = workspace(p.device, wsb, ws)
    check(L.mstf_value_spmv_f16(_stream(), cv.bmp.data_ptr(), cv.nz.data_ptr(), cv.idx.data_ptr(),
                                cv.nz_off.data_ptr(), p.data_ptr(), C.data_ptr(), cv.head_dim, cv.tokens, Bq, groups,
                                n_rows, ws.data_ptr(), ws.numel()), "mstf_value_spmv_f16")
    return C


def decode_attention(ck, cv, q, groups, out=None, lse=None, ws=None):
    """Fused key SpMV -> scale+softmax -> value SpMV over the compressed tokens, one query row per head.

    q: [Bq, D] fp16 -> out [Bq, D] fp16.  lse (optional fp32 [Bq, 2]) receives (max, sum) of every row."""
    return _call(host().decode_attention, ws, q.device, (ck.tokens, 0, q.numel() // ck.head_dim), ck.bmp, ck.nz, ck.idx, ck.nz_off,
                 cv.bmp, cv.nz, cv.idx, cv.nz_off, q, groups, ck.tokens, ck.head_dim, out, lse)


def decode_attention_static(ck, cv, q, groups, out=None, lse=None):
    """decode_attention through the entry point that uses the library's own fixed scratch buffer: no workspace is
    passed and nothing is allocated by the library (calls on one GPU must not overlap)."""
    assert q.dtype == torch.float16 and q.is_contiguous()
    D = ck.head_dim
    Bq = q.numel() // D
    o = torch.empty((Bq, D), dtype=torch.float16, device=q.device) if out is None else out
    check(lib().mstf_decode_attention_static_f16(_stream(), ck.bmp.data_ptr(), ck.nz.data_ptr(), ck.idx.data_ptr(),
                                                 ck.nz_off.data_ptr(), cv.bmp.data_ptr(), cv.nz.data_ptr(),
                                                 cv.idx.data_ptr(), cv.nz_off.data_ptr(), q.data_ptr(), o.data_ptr(),
                                                 lse.data_ptr() if lse is not None else None, ck.tokens, D, Bq, groups),
          "mstf_decode_attention_static_f16")
    return o


def decode_attention_window(ck, cv, q, k_win, v_win, win_len, groups, out=None, lse=None, win_len_dev=None, ws=None):
    """Attention of one decode step over [compressed tokens | dense window] under one softmax, three launches.

    ck, cv: CompressedKV or None (nothing compressed yet); q: [Bq, D]; k_win, v_win: [Bkv, win_stride, D] fp16 with
    the first win_len tokens valid.  win_len_dev (int32 tensor of one element): the valid length is read on the
    device and win_len is only its upper bound, so that the call can be captured in a HIP graph."""
    assert q.dtype == torch.float16 and q.is_contiguous()
    assert k_win.dtype == torch.float16 and k_win.is_contiguous() and v_win.is_contiguous() and k_win.shape == v_win.shape
    D = k_win.shape[-1]
    Bq = q.numel() // D
    tokens = ck.tokens if ck is not None else 0
    L = lib()
    o = torch.empty((Bq, D), dtype=torch.float16, device=q.device) if out is None else out
    ws = workspace(q.device, L.mstf_decode_attention_window_workspace_bytes(tokens, int(win_len), D, Bq, groups), ws,
                   (tokens, int(win_len), Bq))
    cp = [t.data_ptr() for t in (ck.bmp, ck.nz, ck.idx, ck.nz_off, cv.bmp, cv.nz, cv.idx, cv.nz_off)] if tokens else [None] * 8
    check(L.mstf_decode_attention_window_f16(_stream(), *cp, q.data_ptr(), k_win.data_ptr(), v_win.data_ptr(), int(win_len),
                                             win_len_dev.data_ptr() if win_len_dev is not None else None,
                                             k_win.shape[1], o.data_ptr(), lse.data_ptr() if lse is not None else None,
                                             tokens, D, Bq, groups, ws.data_ptr(), ws.numel()),
          "mstf_decode_attention_window_f16")
    return o


def decode_attention_window_pool(k_pool, v_pool, q, k_win, v_win, win_len, groups, win_len_dev, out=None, lse=None,
                                 ws=None):
    """decode_attention_window over two cache.CompressedPool sides that grow in place: the pools' pre-allocated
    per-tile arrays are read with their row stride and the number of compressed tokens comes from the pool's device
    counter, so nothing about the call changes when a chunk is appended (a HIP graph holding it stays valid)."""
    assert q.dtype == torch.float16 and q.is_contiguous()
    assert k_win.dtype == torch.float16 and k_win.is_contiguous() and v_win.is_contiguous() and k_win.shape == v_win.shape
    assert k_pool.max_tokens == v_pool.max_tokens
    D = k_win.shape[-1]
    Bq = q.numel() // D
    L = lib()
    o = torch.empty((Bq, D), dtype=torch.float16, device=q.device) if out is None else out
    ws = workspace(q.device, L.mstf_decode_attention_window_workspace_bytes(k_pool.max_tokens, int(win_len), D, Bq,
                                                                           groups), ws,
                   (k_pool.max_tokens, int(win_len), Bq))
    cp = [t.data_ptr() for t in (k_pool.bmp_store, k_pool.nz, k_pool.idx_store, k_pool.nz_off, v_pool.bmp_store, v_pool.nz,
                                 v_pool.idx_store, v_pool.nz_off)]
    check(L.mstf_decode_attention_window_pool_f16(_stream(), *cp, q.data_ptr(), k_win.data_ptr(), v_win.data_ptr(),
                                                  int(win_len), win_len_dev.data_ptr() if win_len_dev is not None else None,
                                                  k_win.shape[1], o.data_ptr(), lse.data_ptr() if lse is not None else None,
                                                  k_pool.max_tokens, k_pool.tokens_dev.data_ptr(), k_pool.tile_capacity, D,
                                                  Bq, groups, ws.data_ptr(), ws.numel()),
          "mstf_decode_attention_window_pool_f16")
    return o


def decode_step_pool(k_pool, v_pool, q_in, k_in, v_in, k_win, v_win, win_len, cos=None, sin=None, win_len_dev=None,
                     overflow=None, out=None, lse=None, ws=None):
    """The cache side of a decode step in two launches (mstf_decode_step_pool_f16): window_append followed by
    decode_attention_window_pool, bit for bit, with rotation, append and the attention over the window inside the
    launch of the compressed tokens.  q_in [bs, n_q * D], k_in / v_in [bs, n_kv * D]: the projection outputs of the
    new token (views with a batch stride are fine); cos, sin [D] or [bs, D] or None; k_win, v_win
    [bs * n_kv, win_stride, D]; win_len bounds the count of valid rows after the step, win_len_dev holds it."""
    assert k_pool.max_tokens == v_pool.max_tokens
    return _call(host().decode_step, ws, q_in.device, (k_pool.max_tokens, int(win_len), q_in.numel() // k_win.shape[-1]),
                 k_pool.bmp_store, k_pool.nz, k_pool.idx_store, k_pool.nz_off, v_pool.bmp_store, v_pool.nz, v_pool.idx_store,
                 v_pool.nz_off, q_in, k_in, v_in, k_win, v_win, int(win_len), cos, sin, win_len_dev, overflow, out, lse,
                 k_pool.max_tokens, k_pool.tokens_dev, k_pool.tile_capacity)


def window_append(k_in, v_in, k_win, v_win, win_len, q_in=None, cos=None, sin=None, q_out=None, win_len_dev=None,
                  overflow=None):
    """The per-token work in front of the attention call in one launch (models/llama_mustafar_kernel.py:363-374, 391,
    430): q_in [bs, n_q * D], k_in / v_in [bs, n_kv * D] fp16 are the projection outputs of the new token (views with
    a batch stride are fine); query and key heads are rotated with cos, sin [D] or [bs, D] (None: no rotation), the
    query rows returned as [bs * n_q, D], key and value rows written to row win_len - 1 of the window buffers
    k_win, v_win [bs * n_kv, win_stride, D].  win_len counts the valid rows after the call, the new token included;
    with win_len_dev (int32 tensor) the count is read on the device.  Returns q_out (None without q_in)."""
    D = k_win.shape[-1]
    bs = k_in.shape[0]
    n_kv = k_in.shape[-1] // D
    for t in (k_in, v_in) + ((q_in,) if q_in is not None else ()):
        assert t.dtype == torch.float16 and t.dim() == 2 and t.stride(1) == 1 and t.shape[0] == bs
    assert k_win.dtype == torch.float16 and k_win.is_contiguous() and v_win.is_contiguous() and k_win.shape == v_win.shape
    assert k_win.shape[0] == bs * n_kv and v_in.shape[-1] == n_kv * D
    n_q = 0
    if q_in is not None:
        n_q = q_in.shape[-1] // D
        if q_out is None:
            q_out = torch.empty((bs * n_q, D), dtype=torch.float16, device=q_in.device)
        assert q_out.dtype == torch.float16 and q_out.is_contiguous() and q_out.numel() == bs * n_q * D
    rope_stride = 0
    if cos is not None:
        assert cos.dtype == torch.float16 and sin.dtype == torch.float16 and cos.shape == sin.shape
        assert cos.shape[-1] == D and cos.stride(-1) == 1 and sin.stride(-1) == 1
        if cos.dim() == 2 and cos.shape[0] > 1:
            assert cos.shape[0] == bs and cos.stride(0) == sin.stride(0)
            rope_stride = cos.stride(0)
    check(lib().mstf_window_append_f16(
        _stream(), q_in.data_ptr() if q_in is not None else None, q_in.stride(0) if q_in is not None else 0,
        k_in.data_ptr(), k_in.stride(0), v_in.data_ptr(), v_in.stride(0), bs, n_q, n_kv, D,
        cos.data_ptr() if cos is not None else None, sin.data_ptr() if sin is not None else None, rope_stride,
        q_out.data_ptr() if q_out is not None else None, k_win.data_ptr(), v_win.data_ptr(), k_win.shape[1], int(win_len),
        win_len_dev.data_ptr() if win_len_dev is not None else None, overflow.data_ptr() if overflow is not None else None),
        "mstf_window_append_f16")
    return q_out


def decode_attention_partial(ck, cv, q, groups, ws=None):
    """First phase of decode_attention: un-normalised outputs and (max, sum) per 512-token split, left in `ws`."""
    assert q.dtype == torch.float16 and q.is_contiguous()
    D = ck.head_dim
    Bq = q.numel() // D
    L = lib()
    ws = workspace(q.device, attention_workspace_least(ck.tokens, 0, Bq), ws)
    check(L.mstf_decode_attention_partial_f16(_stream(), ck.bmp.data_ptr(), ck.nz.data_ptr(), ck.idx.data_ptr(),
                                              ck.nz_off.data_ptr(), cv.bmp.data_ptr(), cv.nz.data_ptr(),
                                              cv.idx.data_ptr(), cv.nz_off.data_ptr(), q.data_ptr(), ck.tokens, D, Bq,
                                              groups, ws.data_ptr(), ws.numel()), "mstf_decode_attention_partial_f16")
    return ws


def decode_attention_merge(ws, tokens, head_dim, Bq, groups, out=None, lse=None):
    """Second phase of decode_attention: combines the splits left in `ws` by decode_attention_partial."""
    o = torch.empty((Bq, head_dim), dtype=torch.float16, device=ws.device) if out is None else out
    check(lib().mstf_decode_attention_merge_f16(_stream(), ws.data_ptr(), ws.numel(), o.data_ptr(),
                                                lse.data_ptr() if lse is not None else None, tokens, head_dim, Bq,
                                                groups), "mstf_decode_attention_merge_f16")
    return o


def scale_softmax(s, head_dim, out=None):
    """softmax(s / sqrt(head_dim), dtype=float32).to(float16) over the last axis."""
    return host().scale_softmax(s, int(head_dim), out)


def sqrt_head_dim(head_dim):
    return math.sqrt(head_dim)
