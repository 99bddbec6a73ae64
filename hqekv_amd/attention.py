"""Host glue between the reference's 42-field cache tuple and the hybrid HIP launches.

The tuple layout is the reference's (quant/quant_matmul_hq.py:34-38):
  0 sixteen_K (B,Hkv,D,T16)  1 sixteen_K_idx  2 sixteen_V (B,Hkv,T16,D)  3 sixteen_V_idx
  K class b at base 4/12/20/28 (8/4/2/1 bit): code, idx, scale, zero;  V class at 8/16/24/32
  36 outliers  37 outliers_idx  38 V_token_norm  39 new_K (B,Hkv,Tn,D)  40 new_V  41 kv_seq_len
Each populated class becomes one ``hqekv_seg``; the kernels read the tensors where they lie.
"""
from __future__ import annotations

import ctypes as C
import os
import weakref
from typing import List, Optional, Tuple

import numpy as np
import torch

from . import _lib

BITS = (8, 4, 2, 1)   # 1: the uniform 1-bit class of the 'uniform_group' strategy (32 codes per word)
K_BASE = {8: 4, 4: 12, 2: 20, 1: 28}
V_BASE = {8: 8, 4: 16, 2: 24, 1: 32}
K16, K16_IDX, V16, V16_IDX = 0, 1, 2, 3
NEW_K, NEW_V, KV_SEQ_LEN = 39, 40, 41


def _idx(t: Optional[torch.Tensor], n: int, dev) -> Optional[torch.Tensor]:
    if t is None:
        return None
    if t.dtype != torch.int64:
        t = t.to(torch.int64)
    if t.device != dev:
        t = t.to(dev)
    t = t.contiguous()
    if t.numel() != n:
        raise ValueError(f"index of length {t.numel()} for a class of {n} tokens")
    return t


def token_major_window(t: torch.Tensor):
    """An fp16 (B,H,n,D) tensor as the kernels read it: -> (tensor whose data_ptr is the first row, token rows between
    two (b, h) slabs or 0 when dense).  The head of a longer buffer -- ``buf[:, :, :n]`` of a capacity-sized residual
    buffer -- is read where it lies; anything else that is not dense is copied."""
    if t.is_contiguous():
        return t, 0
    B, H, n, D = t.shape
    sb, sh, st, sd = t.stride()
    if sd == 1 and st == D and sh % D == 0 and sh >= n * D and (B == 1 or sb == H * sh):
        return t, sh // D
    return t.contiguous(), 0


def ring_order(T: int, weights: torch.Tensor) -> int:
    """How torch's GPU reduction deals the 32 head rows of ``weights`` (B,32,1,T) to threads when it sums them: to two
    threads when rows are a multiple of 4 long, at least 256, and 8-byte aligned, else to one (measured on the
    device; ``hqekv_ring_row`` and the decode step reproduce either order bit for bit)."""
    return 2 if (T % 4 == 0 and T >= 256 and weights.data_ptr() % 8 == 0) else 1


def ring_row_on_device_applies(weights: torch.Tensor) -> bool:
    """Shapes for which the ring row's order is pinned against torch on the device."""
    return (weights.dtype == torch.float16 and weights.dim() == 4 and weights.shape[2] == 1 and weights.shape[1] == 32
            and weights.shape[0] <= 8 and weights.shape[3] >= 256 and weights.is_contiguous())


def _f16_k_item(k16: torch.Tensor, idx, keep: list) -> dict:
    """fp16 K class (B,Hkv,D,T): read channel-major, or token-major if it is a transposed view."""
    B, H, D, T = k16.shape
    if k16.is_contiguous():
        data, tm = k16, 0
    elif k16.stride(2) == 1 and k16.transpose(2, 3).is_contiguous():
        data, tm = k16, 1  # memory is (B,Hkv,T,D)
    else:
        data, tm = k16.contiguous(), 0
    keep.append(data)
    return dict(bits=16, n_tokens=T, data=data, idx=idx, token_major=tm)


def key_segments(pkv: tuple, dev, Tall: int, keep: list, low_uniform: bool = True,
                 residual: bool = True) -> Tuple[List[dict], int, int]:
    """K classes of the tuple in launch order; ``residual=False`` leaves out ``new_K`` (the only segment
    that changes between two compressions)."""
    items = []
    nh_kv = D = None
    if pkv[K16] is not None:
        k = pkv[K16]
        nh_kv, D = k.shape[1], k.shape[2]
        items.append(_f16_k_item(k, _idx(pkv[K16_IDX], k.shape[3], dev), keep))
    for b in BITS:
        base = K_BASE[b]
        if pkv[base] is not None:
            code = pkv[base].contiguous()
            sc, zr = pkv[base + 2].contiguous(), pkv[base + 3].contiguous()
            n = code.shape[3] * (32 // b)
            nh_kv, D = code.shape[1], code.shape[2]
            idx = _idx(pkv[base + 1], n, dev)
            keep += [code, sc, zr, idx]
            # the 1-bit class holds (std, mean) and normal-quantile codes unless the strategy is 'uniform_group'
            layout = _lib.LAYOUT_NORMAL1 if (b == 1 and not low_uniform) else 0
            items.append(dict(bits=b, n_tokens=n, data=code, scale=sc, zero=zr, idx=idx, layout=layout))
    new_K = pkv[NEW_K]
    if residual and new_K is not None and new_K.shape[2] > 0:
        nk, slab = token_major_window(new_K)
        keep.append(nk)
        nh_kv, D = nk.shape[1], nk.shape[3]
        n = nk.shape[2]
        items.append(dict(bits=16, n_tokens=n, data=nk, idx=None, pos_base=Tall - n, token_major=1, slab_tokens=slab))
    return items, nh_kv, D


def value_segments(pkv: tuple, dev, Tall: int, keep: list, low_uniform: bool = True,
                   residual: bool = True) -> Tuple[List[dict], int, int]:
    items = []
    nh_kv = D = None
    if pkv[V16] is not None:
        v = pkv[V16].contiguous()
        nh_kv, D = v.shape[1], v.shape[3]
        idx = _idx(pkv[V16_IDX], v.shape[2], dev)
        keep += [v, idx]
        items.append(dict(bits=16, n_tokens=v.shape[2], data=v, idx=idx))
    for b in BITS:
        base = V_BASE[b]
        if pkv[base] is not None:
            code = pkv[base].contiguous()
            sc, zr = pkv[base + 2].contiguous(), pkv[base + 3].contiguous()
            n = code.shape[2]
            nh_kv, D = code.shape[1], code.shape[3] * (32 // b)
            idx = _idx(pkv[base + 1], n, dev)
            keep += [code, sc, zr, idx]
            # the 1-bit class holds (std, mean) and normal-quantile codes unless the strategy is 'uniform_group'
            layout = _lib.LAYOUT_NORMAL1 if (b == 1 and not low_uniform) else 0
            items.append(dict(bits=b, n_tokens=n, data=code, scale=sc, zero=zr, idx=idx, layout=layout))
    new_V = pkv[NEW_V]
    if residual and new_V is not None and new_V.shape[2] > 0:
        nv, slab = token_major_window(new_V)
        keep.append(nv)
        nh_kv, D = nv.shape[1], nv.shape[3]
        n = nv.shape[2]
        items.append(dict(bits=16, n_tokens=n, data=nv, idx=None, pos_base=Tall - n, slab_tokens=slab))
    return items, nh_kv, D


def value_length(pkv: tuple) -> int:
    """Sum of the V class lengths plus the residual (quant/hqe_matmul.py:379-402)."""
    n = 0
    if pkv[V16] is not None:
        n += pkv[V16].shape[2]
    for b in (8, 4, 2, 1):
        if pkv[V_BASE[b]] is not None:
            n += pkv[V_BASE[b]].shape[2]
    if pkv[NEW_V] is not None:
        n += pkv[NEW_V].shape[2]
    return n


def _cover_on_device(idx_list, n: int):
    """The checks of ``idx_cover_once`` as one launch over a bit per position (it waits for the answer).
    -> (every position once, whole runs of 32 consecutive positions in every array)."""
    dev, k = idx_list[0].device, len(idx_list)
    scratch = torch.zeros(1 + (n + 31) // 32, dtype=torch.int32, device=dev)
    with _lib.on_device(dev):
        rc = _lib.load().hqekv_cover_once((C.c_void_p * k)(*[t.data_ptr() for t in idx_list]), (C.c_int64 * k)(*[t.numel() for t in idx_list]),
                                          k, scratch.data_ptr(), scratch.numel() * 4, _lib.stream_ptr(dev))
    _lib.check(rc, "cover_once")
    status = int(scratch[0])
    return not status & 1, not status & 2 and all(t.numel() % 32 == 0 for t in idx_list)


def _whole_runs(a: np.ndarray) -> bool:
    """Does ``a`` consist of whole runs of 32 consecutive positions?"""
    if a.size % 32:
        return False
    r = a.reshape(-1, 32)
    return bool((r == r[:, :1] + np.arange(32)).all())


def idx_cover_once(idx_list, n: int, may_wait: bool = True) -> bool:
    """True when the class position arrays, taken together, hold every position in [0, n) exactly once -- what
    the softmax fused into the two GEMV launches relies on (a position nobody writes keeps whatever the score
    buffer held, one written twice is counted twice).  Arrays that carry a host copy (the cache policy's) are
    checked there; others on the device, which waits for it once: the verdict is remembered per set of tensors
    until one of them is written to.  Without ``may_wait`` -- the stream is being captured -- a set that has to be looked at
    on the device counts as not covering."""
    idx_list = [t for t in idx_list if t is not None]
    if sum(int(t.numel()) for t in idx_list) != n:
        return False
    if not idx_list:
        return True
    # The verdict rides on the first array and names the others by weak reference: it holds while these very tensor
    # objects are alive, sit where they sat and have not been written through torch since.  (A kernel that writes an
    # array through its raw pointer does not show here: whoever launches one drops `_hq_cover` from the array.)
    key = tuple((t.data_ptr(), int(t.numel()), t._version) for t in idx_list) + (n,)
    hit = getattr(idx_list[0], "_hq_cover", None)
    if hit is not None and hit[0] == key and len(hit[2]) == len(idx_list) and all(r() is t for r, t in zip(hit[2], idx_list)):
        return hit[1]
    trusted = [getattr(t, "_hq_host_version", None) == t._version for t in idx_list]
    blocks = [getattr(t, "_hq_blocks", None) if ok_ else None for t, ok_ in zip(idx_list, trusted)]
    hosts = [getattr(t, "_hq_host", None) if ok_ else None for t, ok_ in zip(idx_list, trusted)]
    if n % 32 == 0 and all(b is not None and b.shape[0] * 32 == t.numel() for b, t in zip(blocks, idx_list)):
        c = np.concatenate(blocks)   # whole aligned 32-token blocks: check the block numbers
        nb = n // 32
        ok, runs = bool(c.size == nb and (c >= 0).all() and (c < nb).all() and (np.bincount(c, minlength=nb) == 1).all()), True
    elif all(h is not None for h in hosts):
        c = np.concatenate(hosts)
        ok = bool(c.size == n and (c >= 0).all() and (c < n).all() and (np.bincount(c, minlength=n) == 1).all())
        runs = all(_whole_runs(h) for h in hosts)
    elif not may_wait:
        return False
    elif idx_list[0].is_cuda and len(idx_list) <= _lib.MAX_SEGS and n < 2 ** 38 and \
            all(t.dtype == torch.int64 and t.is_contiguous() and t.device == idx_list[0].device for t in idx_list):
        ok, runs = _cover_on_device(idx_list, n)
    else:
        c = torch.cat([t.reshape(-1).to(torch.int64) for t in idx_list])
        inside = (c >= 0) & (c < n)
        ok = bool(inside.all() & (torch.bincount(c.clamp(0, n - 1), minlength=n) == 1).all())
        runs = all(_whole_runs(t.cpu().numpy().reshape(-1)) for t in idx_list)
    idx_list[0]._hq_cover = (key, ok, [weakref.ref(t) for t in idx_list], ok and runs)
    return ok


def mark_runs(items: List[dict]) -> None:
    """Name the segments whose index arrays are known -- from ``idx_cover_once``, asked of exactly these arrays just now --
    to consist of whole runs of 32 consecutive positions: the kernels then read one index per run."""
    held = [it for it in items if it.get("idx") is not None]
    hit = getattr(held[0]["idx"], "_hq_cover", None) if held else None
    if hit is not None and hit[3] and len(hit[2]) == len(held) and all(r() is it["idx"] for r, it in zip(hit[2], held)):
        for it in held:
            it["layout"] = int(it.get("layout", 0)) | _lib.LAYOUT_RUNS


def _class_idx(pkv: tuple, base0: int, bases) -> list:
    """Position arrays of the populated classes of one side."""
    out = [pkv[base0 + 1]] if pkv[base0] is not None else []
    return out + [pkv[bases[b] + 1] for b in BITS if pkv[bases[b]] is not None]


def classes_partition_positions(pkv: tuple) -> bool:
    """Both sides' classes cover [0, kept) exactly once each, kept = tokens held by the V classes."""
    v_idx = _class_idx(pkv, V16, V_BASE)
    n = sum(int(t.numel()) for t in v_idx if t is not None)
    if any(t is None for t in v_idx):
        return False
    k_idx = _class_idx(pkv, K16, K_BASE)
    if any(t is None for t in k_idx):
        return False
    return idx_cover_once(k_idx, n) and idx_cover_once(v_idx, n)


def _mask_arg(mask, B: int, Hq: int, Tall: int, dev, keep: list):
    """-> (pointer or None, row stride in elements) for an additive fp16 mask."""
    if mask is None:
        return None, 0
    if not torch.is_tensor(mask):
        if float(mask) == 0.0:
            return None, 0
        mask = torch.full((1, 1, 1, Tall), float(mask), dtype=torch.float16, device=dev)
    mask = mask.to(device=dev, dtype=torch.float16)
    while mask.dim() < 4:
        mask = mask.unsqueeze(0)
    if mask.shape[-1] != Tall or mask.shape[-2] != 1:
        mask = mask.expand(*mask.shape[:-2], 1, Tall) if mask.shape[-1] in (1, Tall) else mask
        if mask.shape[-1] != Tall:
            raise ValueError(f"mask last dim {mask.shape[-1]} != {Tall}")
    if mask.shape[0] == 1 and mask.shape[1] == 1:
        m = mask.reshape(Tall).contiguous()
        keep.append(m)
        return m.data_ptr(), 0
    m = mask.expand(B, Hq, 1, Tall).contiguous()
    keep.append(m)
    return m.data_ptr(), Tall


def workspace_for(v_segs, n_v: int, B: int, Hq: int, Hkv: int, D: int, dev) -> torch.Tensor:
    """Split-K workspace of a stand-alone p.V launch."""
    need = _lib.load().hqekv_pv_workspace_bytes(v_segs, n_v, B, Hq, Hkv, D)
    if need < 0:
        raise ValueError("invalid segment table")
    return torch.empty(max(need, 16) // 4, dtype=torch.float32, device=dev)


def decode_workspace(k_segs, n_k: int, v_segs, n_v: int, B: int, Hq: int, Hkv: int, D: int, dev) -> torch.Tensor:
    """Workspace of a whole decode-attention call (split-K partials and per-tile softmax statistics)."""
    need = _lib.load().hqekv_decode_workspace_bytes(k_segs, n_k, v_segs, n_v, B, Hq, Hkv, D)
    if need < 0:
        raise ValueError("invalid segment table")
    return torch.empty(max(need, 256) // 4, dtype=torch.float32, device=dev)


_environ = os.environ   # (attribute lookups on the module are the slow part of this per-step call)


def default_flags() -> int:
    """Fuse the softmax into the two GEMV launches unless HQEKV_UNFUSED=1 asks for the general path."""
    return 0 if _environ.get("HQEKV_UNFUSED") == "1" else _lib.FUSE_SOFTMAX


class SegmentMemo:
    """One layer's segment tables between two compressions.  Fields 0..38 of the tuple (the classes) stay
    the same tensor objects from one decode step to the next -- the caller only replaces ``new_K``,
    ``new_V`` and the length -- so their table entries are built once and only the residual entry is
    rewritten per step.  The memo holds the class tensors it points into; it is valid for a tuple whose
    first 39 fields ARE the held objects, and rebuilt otherwise.  The workspace is kept as well (calls of
    one layer are ordered on one stream)."""

    def __init__(self):
        self.held: Optional[tuple] = None      # fields 0..38 of the tuple the tables were built from
        self.key = None                        # (device, low_uniform) they were built for
        self.ws: Optional[torch.Tensor] = None
        self.keep: list = []                   # converted / made-contiguous tensors the tables point into
        self.k_arr = self.v_arr = None         # ctypes arrays of hqekv_seg with one spare entry each
        self.n_k = self.n_v = 0
        self.Hkv = None
        self.dims = (None, None)
        self.partition = False                 # the classes' position arrays cover [0, kept) once per side
        self._native = None                    # the class entries as the native step takes them (k_arr is None where
                                               # they were built there: ``build`` makes the rest when it is asked for)

    def lookup(self, pkv: tuple, dev, low_uniform: bool) -> bool:
        held = self.held
        if held is None or self.key != (dev, low_uniform):
            return False
        for a, b in zip(held, pkv):  # zip stops after the 39 held fields
            if a is not b:
                return False
        return True

    def build(self, pkv: tuple, dev, low_uniform: bool) -> None:
        self.keep = []
        k_items, hk, dk = key_segments(pkv, dev, 0, self.keep, low_uniform, residual=False)
        v_items, hv, dv = value_segments(pkv, dev, 0, self.keep, low_uniform, residual=False)
        if len(k_items) + 2 > _lib.MAX_SEGS or len(v_items) + 2 > _lib.MAX_SEGS:
            raise ValueError("too many segments")
        self.partition = classes_partition_positions(pkv)
        if self.partition:
            mark_runs(k_items)
            mark_runs(v_items)
        self.n_k, self.n_v = len(k_items), len(v_items)
        self.k_arr = (_lib.Seg * (self.n_k + 2))()   # two spare entries each: the residual and the step's new token
        self.v_arr = (_lib.Seg * (self.n_v + 2))()
        for dst, src in ((self.k_arr, _lib.make_segs(k_items)), (self.v_arr, _lib.make_segs(v_items))):
            for i in range(len(dst) - 2):
                C.memmove(C.byref(dst[i]), C.byref(src[i]), C.sizeof(_lib.Seg))
        self.need = {}                                # workspace bytes per (residual, tail, B, Hq) of this cache
        self.Hkv = hk if hk is not None else hv
        self.dims = (dk, dv)
        self.held = tuple(pkv[:NEW_K])
        self.key = (dev, low_uniform)
        self._native = None

    @staticmethod
    def _fill(s, t: torch.Tensor, end: int, layout: int, keep: list):
        """Table entry of an fp16 token-major block (B,Hkv,n,D) whose last token sits at position end - 1."""
        tc, slab = token_major_window(t)
        keep.append(tc)
        n = tc.shape[2]
        s.bits, s.layout, s.n_tokens, s.pos_base, s.data, s.slab_tokens = 16, layout, n, end - n, tc.data_ptr(), slab
        return tc.shape[1], tc.shape[3]

    def tables(self, pkv: tuple, Tall: int, keep: list, tail=None):
        """-> (k_segs, n_k, v_segs, n_v, Hkv, (dk, dv), (residual tokens, tail tokens)) with this step's residual
        -- and the tokens of ``tail`` = (k, v), which follow it -- filled in."""
        n_k, n_v, Hkv, (dk, dv) = self.n_k, self.n_v, self.Hkv, self.dims
        n_tail = tail[0].shape[2] if tail is not None else 0
        n_res = 0
        new_K, new_V = pkv[NEW_K], pkv[NEW_V]
        if new_K is not None and new_K.shape[2] > 0:
            n_res = new_K.shape[2]
            Hkv, dk = self._fill(self.k_arr[n_k], new_K, Tall - n_tail, _lib.LAYOUT_TOKEN_MAJOR, keep)
            n_k += 1
        if new_V is not None and new_V.shape[2] > 0:
            Hkv, dv = self._fill(self.v_arr[n_v], new_V, Tall - n_tail, 0, keep)
            n_v += 1
        if n_tail:
            Hkv, dk = self._fill(self.k_arr[n_k], tail[0], Tall, _lib.LAYOUT_TOKEN_MAJOR, keep)
            Hkv, dv = self._fill(self.v_arr[n_v], tail[1], Tall, 0, keep)
            n_k += 1
            n_v += 1
        return self.k_arr, n_k, self.v_arr, n_v, Hkv, (dk, dv), (n_res, n_tail)

    def workspace(self, need: int, dev) -> torch.Tensor:
        if self.ws is None or self.ws.numel() * 4 < need or self.ws.device != dev:
            self.ws = torch.empty(max(need + need // 8, 256) // 4, dtype=torch.float32, device=dev)
        return self.ws

    def steps(self, pkv: tuple, q: torch.Tensor, low_uniform: bool, known: bool):
        """The native tables (``_host.StepTables``) of a cache whose classes cover every position once, else None.
        ``known``: the caller vouches that ``pkv`` carries the class tensors the tables were built from (it is the tuple
        the previous step returned)."""
        dev = q.device
        if not (known and self.held is not None) and not self.lookup(pkv, dev, low_uniform):
            native = _lib.host().step_tables(q, pkv, low_uniform, idx_cover_once)
            if native is not None:
                self.held, self.key, self._native, self.partition = tuple(pkv[:NEW_K]), (dev, low_uniform), native, True
                self.keep, self.need, self.k_arr, self.v_arr = [], {}, None, None
                return native
            self.build(pkv, dev, low_uniform)
        if not self.partition:
            return None
        if self._native is None:
            self._native = _lib.host().StepTables(C.addressof(self.k_arr), self.n_k, C.addressof(self.v_arr), self.n_v)
        return self._native


def decode_attention(q: torch.Tensor, pkv: tuple, mask, Tall: int, zero_init: bool, flags: Optional[int] = None,
                     low_uniform: bool = True, memo: Optional[SegmentMemo] = None, tail=None, step=None):
    """q (B,Hq,1,D) fp16 -> (attn_weights (B,Hq,1,Tall) fp16 probabilities, attn_output (B,Hq,1,D) fp16).

    One q.K^T launch over all K classes and one p.V launch over all V classes with the softmax fused
    into them; or, with a mask / an incomplete cover of the positions / ``flags=0``, the general path
    (q.K^T, scale+mask+clamp+softmax, p.V, fixed-order combine).  Runs on torch's current stream.
    ``memo``: a ``SegmentMemo`` the caller keeps per layer, so that steps between two compressions rebuild
    only the residual's table entry.
    ``tail`` = (k, v), each (B,Hkv,L,D) fp16: tokens that follow the tuple's residual without being part of it yet
    (``Tall`` counts them).  The kernels read them as one more fp16 segment per side, so a caller can start the
    attention of a decode step before it appends the step's key and value to the residual.
    ``step``: what the caller's decode step does around the attention, folded into the call's last launch
    (``hqekv_decode_step``): ``step["ring_line"]`` = a (Tall,) fp16 view that receives ``attn_weights.sum(0).sum(0)``
    in torch's order (only for shapes ``ring_row_on_device_applies`` covers; the caller checks), ``step["append"]`` =
    (K buffer, V buffer, n): the rows of ``tail`` are copied to token row n of the (B,Hkv,cap,D) buffers.
    """
    _lib.require_gpu(q, "q")
    if q.dtype != torch.float16:
        raise TypeError("q must be float16 (the cache is fp16 by definition)")
    if q.dim() != 4 or q.shape[2] != 1:
        raise ValueError("q must be (B, Hq, 1, D): only single-token decode is computed")
    B, Hq, _, D = q.shape
    dev = q.device
    keep: list = []
    use_flags = default_flags() if flags is None else flags
    if memo is not None:
        if not memo.lookup(pkv, dev, low_uniform) or memo.k_arr is None:
            memo.build(pkv, dev, low_uniform)
        k_segs, n_k, v_segs, n_v, Hkv, (dk, dv), res_tail = memo.tables(pkv, Tall, keep, tail)
        covered = memo.partition
    else:
        covered = not (use_flags & _lib.FUSE_SOFTMAX) or mask is not None or classes_partition_positions(pkv)
    if not covered:   # a position nobody writes must read as zero, and the fused softmax must not run
        use_flags &= ~_lib.FUSE_SOFTMAX
        zero_init = True
    if memo is None:
        n_tail = tail[0].shape[2] if tail is not None else 0
        k_items, hk, dk = key_segments(pkv, dev, Tall - n_tail, keep, low_uniform)
        v_items, hv, dv = value_segments(pkv, dev, Tall - n_tail, keep, low_uniform)
        if n_tail:
            tk, tv = tail[0].contiguous(), tail[1].contiguous()
            keep += [tk, tv]
            k_items.append(dict(bits=16, n_tokens=n_tail, data=tk, idx=None, pos_base=Tall - n_tail, token_major=1))
            v_items.append(dict(bits=16, n_tokens=n_tail, data=tv, idx=None, pos_base=Tall - n_tail))
            hk, dk, hv, dv = tk.shape[1], tk.shape[3], tv.shape[1], tv.shape[3]
        Hkv = hk if hk is not None else hv
        if covered and use_flags & _lib.FUSE_SOFTMAX and mask is None:
            mark_runs(k_items)
            mark_runs(v_items)
        k_segs, v_segs, n_k, n_v = _lib.make_segs(k_items), _lib.make_segs(v_items), len(k_items), len(v_items)
    if Hkv is None:
        raise ValueError("invalid past_key_value")
    for d_ in (dk, dv):
        if d_ is not None and d_ != D:
            raise ValueError("head_dim of the cache does not match q")
    qc = q.contiguous()
    weights = (torch.zeros if zero_init else torch.empty)(B, Hq, 1, Tall, dtype=torch.float16, device=dev)
    out = torch.empty(B, Hq, 1, D, dtype=torch.float16, device=dev)
    mptr, mstride = _mask_arg(mask, B, Hq, Tall, dev, keep)
    lib = _lib.load()
    with _lib.on_device(dev):
        if memo is not None:
            need_key = (res_tail, B, Hq)
            need = memo.need.get(need_key)
            if need is None:
                need = memo.need[need_key] = lib.hqekv_decode_workspace_bytes(k_segs, n_k, v_segs, n_v, B, Hq, Hkv, D)
            if need < 0:
                raise ValueError("invalid segment table")
            ws = memo.workspace(need, dev)
        else:
            ws = decode_workspace(k_segs, n_k, v_segs, n_v, B, Hq, Hkv, D, dev)
        if step is None:
            rc = lib.hqekv_decode_attn(
                k_segs, n_k, v_segs, n_v, qc.data_ptr(), mptr, mstride,
                weights.data_ptr(), out.data_ptr(), B, Hq, Hkv, D, Tall, ws.data_ptr(), ws.numel() * 4,
                use_flags, _lib.stream_ptr(dev))
        else:
            x = _lib.StepExtra()
            line = step.get("ring_line")
            if line is not None:
                x.ring_line, x.ring_order = line.data_ptr(), ring_order(Tall, weights)
            app = step.get("append")
            if app is not None:
                kbuf, vbuf, n = app
                tk, tv = tail[0].contiguous(), tail[1].contiguous()
                keep += [tk, tv]
                x.append_rows, x.new_k, x.new_v = tk.shape[2], tk.data_ptr(), tv.data_ptr()
                x.k_dst, x.v_dst = kbuf[0, 0, n].data_ptr(), vbuf[0, 0, n].data_ptr()
                x.k_dst_slab_tokens, x.v_dst_slab_tokens = kbuf.shape[2], vbuf.shape[2]
            rc = lib.hqekv_decode_step(
                k_segs, n_k, v_segs, n_v, qc.data_ptr(), mptr, mstride,
                weights.data_ptr(), out.data_ptr(), B, Hq, Hkv, D, Tall, ws.data_ptr(), ws.numel() * 4,
                use_flags, _lib.stream_ptr(dev), C.byref(x))
    _lib.check(rc, "decode_attention")
    return weights, out


class DecodePlan:
    """Pre-validated launch plan for one layer's cache: segment tables, outputs and the split-K
    workspace are built once, so a decode step is a single C call (three kernel launches, one for
    short caches, or two under stream capture) with no per-step Python work.  Holds references to every tensor it points into.
    """

    def __init__(self, q_like: torch.Tensor, pkv: tuple, mask=None, Tall: Optional[int] = None,
                 flags: Optional[int] = None, low_uniform: bool = True):
        _lib.require_gpu(q_like, "q")
        B, Hq, _, D = q_like.shape
        self.dev = q_like.device
        self.Tall = int(Tall) if Tall is not None else value_length(pkv)
        self._keep: list = []
        k_items, hk, _ = key_segments(pkv, self.dev, self.Tall, self._keep, low_uniform)
        v_items, hv, _ = value_segments(pkv, self.dev, self.Tall, self._keep, low_uniform)
        self.Hkv = hk if hk is not None else hv
        if self.Hkv is None:
            raise ValueError("invalid past_key_value")
        self.flags = default_flags() if flags is None else flags
        if (self.flags & _lib.FUSE_SOFTMAX) and mask is None:
            if classes_partition_positions(pkv):
                mark_runs(k_items)
                mark_runs(v_items)
            else:
                self.flags &= ~_lib.FUSE_SOFTMAX   # weights is zero-initialised below: uncovered positions stay 0
        self.B, self.Hq, self.D = B, Hq, D
        self.n_k, self.n_v = len(k_items), len(v_items)
        self.k_segs, self.v_segs = _lib.make_segs(k_items), _lib.make_segs(v_items)
        self.weights = torch.zeros(B, Hq, 1, self.Tall, dtype=torch.float16, device=self.dev)
        self.out = torch.empty(B, Hq, 1, D, dtype=torch.float16, device=self.dev)
        self.mask_ptr, self.mask_stride = _mask_arg(mask, B, Hq, self.Tall, self.dev, self._keep)
        with _lib.on_device(self.dev):
            self.ws = decode_workspace(self.k_segs, self.n_k, self.v_segs, self.n_v, B, Hq, self.Hkv, D, self.dev)
        self._lib = _lib.load()
        self.inv_sqrt_d = 1.0 / (D ** 0.5)

    def run(self, q: torch.Tensor, stream: Optional[int] = None, only: int = 0):
        """``only`` = _lib.ONLY_QK / ONLY_PV / ONLY_COMBINE runs one part of the step (per-kernel timing)."""
        st = _lib.stream_ptr(self.dev) if stream is None else stream
        rc = self._lib.hqekv_decode_attn(
            self.k_segs, self.n_k, self.v_segs, self.n_v, q.data_ptr(), self.mask_ptr, self.mask_stride,
            self.weights.data_ptr(), self.out.data_ptr(), self.B, self.Hq, self.Hkv, self.D, self.Tall,
            self.ws.data_ptr(), self.ws.numel() * 4, self.flags | only, st)
        if rc:
            _lib.check(rc, "DecodePlan.run")
        return self.weights, self.out

    # the three stages on their own, for per-kernel timing
    def run_qk(self, q: torch.Tensor, stream: Optional[int] = None):
        st = _lib.stream_ptr(self.dev) if stream is None else stream
        _lib.check(self._lib.hqekv_qk_hybrid(self.k_segs, self.n_k, q.data_ptr(), self.weights.data_ptr(), self.B,
                                             self.Hq, self.Hkv, self.D, self.Tall, st), "run_qk")

    def run_softmax(self, stream: Optional[int] = None):
        st = _lib.stream_ptr(self.dev) if stream is None else stream
        _lib.check(self._lib.hqekv_scale_softmax(self.weights.data_ptr(), self.mask_ptr, self.mask_stride,
                                                 self.B * self.Hq, self.Tall, self.inv_sqrt_d, st), "run_softmax")

    def run_pv(self, stream: Optional[int] = None):
        st = _lib.stream_ptr(self.dev) if stream is None else stream
        _lib.check(self._lib.hqekv_pv_hybrid(self.v_segs, self.n_v, self.weights.data_ptr(), self.out.data_ptr(),
                                             self.B, self.Hq, self.Hkv, self.D, self.Tall, self.ws.data_ptr(),
                                             self.ws.numel() * 4, st), "run_pv")
