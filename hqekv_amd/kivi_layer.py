"""The second caller of the path in the reference: its KIVI-style attention (``LlamaAttention.forward`` of
model/llama_kivi.py:96-266; model/qwen3_kivi.py has the same cache logic), without the projections, the
rotary embedding and ``o_proj``.  Every token is kept: K is quantised per channel in blocks of
``residual_length`` tokens, V per token one token at a time, both with an fp16 tail.

Cache tuple, as upstream (model/llama_kivi.py:266):
  0 K codes (B,Hkv,D,Tq/pf) int32   1 K fp16 tail (B,Hkv,r,D)   2 K scale (B,Hkv,D,Tq/32)   3 K zero
  4 V codes (B,Hkv,Tv,D/pf) int32   5 V fp16 tail (B,Hkv,r',D)  6 V scale (B,Hkv,Tv,D/32)   7 V zero
  8 kv_seq_len

Upstream attends with two per-class GEMVs plus two dense matmuls over the tails, a concatenation, the
softmax and an addition (:130-188).  Here a decode step is ONE hybrid launch sequence (q.K^T over the
quantised class and the tail, softmax fused, p.V over both, combine): the tuple's fields are handed to the
hybrid kernels as two segments per side, where they lie.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib
from .attention import K_BASE, NEW_K, NEW_V, V_BASE, SegmentMemo, decode_attention, default_flags
from .decode_layer import gqa_prompt_attention
from .pack_unpack import quantize_pack_into, uniform_group_quantize_pack_last_dim


class KiviAttentionLayer:
    """``k_bits``/``v_bits`` in {1, 2, 4, 8}; ``group_size`` 32; ``residual_length`` a multiple of 32
    (upstream: 2, 2, 32, 128 -- model/llama_kivi.py:72-76)."""

    MIN_V_ROWS = 1024   # least capacity (token rows) of the V class buffers of the in-place decode step

    def __init__(self, head_dim: int, k_bits: int = 2, v_bits: int = 2, group_size: int = 32,
                 residual_length: int = 128):
        if group_size != 32:
            raise ValueError("group_size must be 32")
        if residual_length <= 0 or residual_length % group_size:
            raise ValueError("residual_length must be a positive multiple of the group size")
        if k_bits not in K_BASE or v_bits not in V_BASE:
            raise ValueError("k_bits and v_bits must be 1, 2, 4 or 8")
        self.head_dim, self.k_bits, self.v_bits = head_dim, k_bits, v_bits
        self.group_size, self.residual_length = group_size, residual_length
        self.scaling = head_dim ** -0.5
        self._memo = SegmentMemo()
        self._k_segs = (_lib.Seg * 3)()   # (quantised class, fp16 tail, this step's token) of each side, rewritten every step
        self._v_segs = (_lib.Seg * 3)()
        self._ws: Optional[torch.Tensor] = None
        self._st = None                   # buffers behind the tuple this layer handed out last (a _host.KiviState)
        self.in_place = True              # decode steps append in capacity buffers (False: upstream's cat / slice sequence)

    # ------------------------------------------------------------------ prompt
    def _prefill(self, q, k, v, attention_mask):
        """-> (output, the first eight fields of the tuple, None), or (output, None, the buffers that hold them) where the decode steps
        will append in place: what such a step needs is quantised and copied straight into its capacity buffers."""
        T, R = k.shape[-2], self.residual_length
        out = gqa_prompt_attention(q, k, v, attention_mask, self.scaling)   # grouped heads: no repeat_kv copies
        tail = T % R
        k_quant = k if tail == 0 else (k[:, :, :T - tail, :] if T >= R else None)
        kq = ks = kz = None
        if k_quant is not None:
            # (B,Hkv,D,T) view of token-major memory: the quantiser reads it in place
            kq, ks, kz = uniform_group_quantize_pack_last_dim(k_quant.transpose(2, 3), self.group_size, self.k_bits)
        n_vq = max(0, T - R)
        if self._runs_in_place(q) and k.dtype == v.dtype == torch.float16:
            st = self._buffers(k, n_vq)
            st.kq, st.ks, st.kz = kq, ks, kz
            if tail:
                st.kt[:, :, :tail].copy_(k[:, :, T - tail:])
            st.nk, st.nv, st.n_vq = tail, T - n_vq, n_vq
            st.vt[:, :, :T - n_vq].copy_(v[:, :, n_vq:])
            if n_vq:
                quantize_pack_into(v[:, :, :n_vq], self.v_bits, *(x[:, :, :n_vq] for x in (st.vcode, st.vscale, st.vzero)))
            return out, None, st
        k_full = None if tail == 0 else k[:, :, T - tail:, :].contiguous()
        if n_vq == 0:
            vq, v_full, vs, vz = None, v, None, None
        else:
            v_full = v[:, :, n_vq:, :].contiguous()
            vq, vs, vz = uniform_group_quantize_pack_last_dim(v[:, :, :n_vq, :], self.group_size, self.v_bits)
        return out, (kq, k_full, ks, kz, vq, v_full, vs, vz), None

    # ------------------------------------------------------------------ decode attention
    def _attend(self, q, kq, ks, kz, k_full, vq, vs, vz, v_full, T: int):
        """The step's attention straight from the tuple's fields: per side the quantised class at positions
        [0, n) and the fp16 tail behind it -- two table entries whose pointers and lengths are rewritten in place
        (the class tensors are new objects after every step here, so a memo keyed on them would be rebuilt every
        time).  Both sides cover every position once by construction, so the softmax rides in the two launches."""
        B, Hq, _, D = q.shape
        dev = q.device
        keep = []

        def fill(segs, code, scale, zero, bits, n_class, tail, layout_tail):
            n = 0
            if code is not None:
                code, scale, zero = code.contiguous(), scale.contiguous(), zero.contiguous()
                keep.extend((code, scale, zero))
                e = segs[0]
                e.bits, e.layout, e.n_tokens, e.pos_base = bits, 0, n_class, 0
                e.data, e.scale, e.zero, e.idx = code.data_ptr(), scale.data_ptr(), zero.data_ptr(), None
                n = 1
            if tail is not None and tail.shape[2] > 0:
                tail = tail.contiguous()
                keep.append(tail)
                e = segs[n]
                e.bits, e.layout, e.n_tokens, e.pos_base = 16, layout_tail, tail.shape[2], n_class
                e.data, e.scale, e.zero, e.idx = tail.data_ptr(), None, None, None
                n += 1
            return n

        Hkv = (k_full if k_full is not None else kq).shape[1]
        n_kq = 0 if kq is None else kq.shape[3] * (32 // self.k_bits)
        n_vq = 0 if vq is None else vq.shape[2]
        n_k = fill(self._k_segs, kq, ks, kz, self.k_bits, n_kq, k_full, _lib.LAYOUT_TOKEN_MAJOR)
        n_v = fill(self._v_segs, vq, vs, vz, self.v_bits, n_vq, v_full, 0)
        qc = q.contiguous()
        weights = torch.empty(B, Hq, 1, T, dtype=torch.float16, device=dev)
        out = torch.empty(B, Hq, 1, D, dtype=torch.float16, device=dev)
        lib = _lib.load()
        with _lib.on_device(dev):
            need = lib.hqekv_decode_workspace_bytes(self._k_segs, n_k, self._v_segs, n_v, B, Hq, Hkv, D)
            if need < 0:
                raise ValueError("invalid segment table")
            if self._ws is None or self._ws.numel() * 4 < need or self._ws.device != dev:
                self._ws = torch.empty(max(need + need // 4, 256) // 4, dtype=torch.float32, device=dev)
            rc = lib.hqekv_decode_attn(self._k_segs, n_k, self._v_segs, n_v, qc.data_ptr(), None, 0,
                                       weights.data_ptr(), out.data_ptr(), B, Hq, Hkv, D, T, self._ws.data_ptr(),
                                       self._ws.numel() * 4, default_flags(), _lib.stream_ptr(dev))
        _lib.check(rc, "KiviAttentionLayer")
        return weights, out

    # ------------------------------------------------------------------ a decode step in place
    def _runs_in_place(self, q: torch.Tensor) -> bool:
        return self.in_place and q.is_cuda and q.dtype == torch.float16 and self.head_dim == q.shape[-1] == 128

    def _buffers(self, like: torch.Tensor, n_vq: int):
        """Empty capacity buffers for a sequence with ``n_vq`` value rows in the quantised class."""
        B, H, _, D = like.shape
        dev, R = like.device, self.residual_length
        st = _lib.host().KiviState()
        st.kt = self._tail_buffer(like, R)
        st.vt = self._tail_buffer(like, 2 * R + 32)   # the tail's window slides one row per step
        self._grow_v_class(st, B, H, D, dev, n_vq + 1)
        return st

    @staticmethod
    def _tail_buffer(like: torch.Tensor, rows: int) -> torch.Tensor:
        """Rows for a tail.  A row is written once: views of it are in tuples that the caller may keep, so a buffer that is
        used up is replaced by another."""
        B, H, _, D = like.shape
        return torch.empty(B, H, rows, D, dtype=torch.float16, device=like.device)

    def _adopt(self, pkv: tuple, like: torch.Tensor):
        """Capacity buffers holding what ``pkv`` holds: the K tail, the V tail (a window that slides one row per step)
        and the V class (which grows one row per step).  The K class stays as it is: it changes every
        ``residual_length`` steps only."""
        kq, k_full, ks, kz, vq, v_full, vs, vz, _ = pkv
        n_vq = 0 if vq is None else vq.shape[2]
        st = self._buffers(like, n_vq)
        if kq is not None:
            st.kq, st.ks, st.kz = kq.contiguous(), ks.contiguous(), kz.contiguous()
        st.nk = 0 if k_full is None else k_full.shape[2]
        if st.nk:
            st.kt[:, :, :st.nk].copy_(k_full)
        st.nv = 0 if v_full is None else v_full.shape[2]
        if st.nv:
            st.vt[:, :, :st.nv].copy_(v_full)
        st.n_vq = n_vq
        if n_vq:
            for dst, src in ((st.vcode, vq), (st.vscale, vs), (st.vzero, vz)):
                dst[:, :, :n_vq].copy_(src)
        return st

    def _grow_v_class(self, st, B: int, H: int, D: int, dev, need: int) -> None:
        """Room for ``need`` rows in the V class buffers (doubling)."""
        old = (st.vcode, st.vscale, st.vzero)
        if old[0] is not None and need <= old[0].shape[2]:
            return
        cap = max(self.MIN_V_ROWS, 2 * need)
        code = torch.empty(B, H, cap, D * self.v_bits // 32, dtype=torch.int32, device=dev)
        scale = torch.empty(B, H, cap, D // 32, dtype=torch.float16, device=dev)
        zero = torch.empty_like(scale)
        n = st.n_vq
        if n:
            for dst, src in zip((code, scale, zero), old):
                dst[:, :, :n].copy_(src[:, :, :n])
        st.vcode, st.vscale, st.vzero = code, scale, zero

    def _step_in_buffers(self, q, k, v, pkv: tuple, T: int):
        """One decode step with everything appended in place: ONE call for the attention over (K class, K tail, this
        step's key) and (V class, V tail, this step's value), whose last launch also copies the two rows behind their
        tails and quantises the oldest value row when it leaves the tail (straight into the class buffers); one
        concatenation every ``residual_length`` steps when a block of keys is quantised.  The tuple handed back holds
        views of the buffers, with upstream's shapes and contents [117-266]; later steps write only rows that no tuple
        shows.  None: an input is not what the native step takes."""
        q, k, v = (x if x.is_contiguous() else x.contiguous() for x in (q, k, v))
        R = self.residual_length
        st = self._st
        if st is None or st.returned is not pkv:
            st = self._st = self._adopt(pkv, k)
        if st.nv == R and st.n_vq == st.vcode.shape[2]:   # a value row is about to leave the tail [254-264]
            self._grow_v_class(st, k.shape[0], k.shape[1], k.shape[3], k.device, st.n_vq + 1)
        done = st.step(q, k, v, T, self.k_bits, self.v_bits)
        if done is None:
            self._st = None
            return None
        weights, out = done
        if st.nk == R:   # a full block of fp16 keys: quantise it per channel, straight from its rows [236-252]
            new = uniform_group_quantize_pack_last_dim(st.kt.transpose(2, 3), self.group_size, self.k_bits)
            if st.kq is not None:
                new = [torch.cat((old, x), dim=3) for old, x in zip((st.kq, st.ks, st.kz), new)]
            st.kq, st.ks, st.kz = new
            st.kt, st.nk = self._tail_buffer(k, R), 0
        nv, v0 = st.nv, st.v0
        if v0 + nv == st.vt.shape[2]:   # the window has reached the end of its buffer: on to the start of another
            vt = self._tail_buffer(k, st.vt.shape[2])
            vt[:, :, :nv].copy_(st.vt[:, :, v0:v0 + nv])
            st.vt, st.v0 = vt, 0
        return out, weights, st.fields(T)

    # ------------------------------------------------------------------ one call
    def forward(self, query_states: torch.Tensor, key_states: torch.Tensor, value_states: torch.Tensor,
                attention_mask: Optional[torch.Tensor] = None, past_key_value: Optional[tuple] = None):
        """query (B,Hq,L,D), key/value (B,Hkv,L,D) fp16, rotary applied.
        -> (attn_output (B,Hq,L,D), attn_weights (B,Hq,1,T) for a decode step, None for a prompt -- upstream's
        fused prompt attention returns none either -- , the 9-field tuple)."""
        L = key_states.shape[-2]
        kv_seq_len = L + (past_key_value[-1] if past_key_value is not None else 0)
        if past_key_value is None:
            out, fields, self._st = self._prefill(query_states, key_states, value_states, attention_mask)
            return out, None, fields + (kv_seq_len,) if self._st is None else self._st.fields(kv_seq_len)
        if L != 1:
            raise ValueError("a decode step appends one token")
        if attention_mask is None and self._runs_in_place(query_states):
            done = self._step_in_buffers(query_states, key_states, value_states, past_key_value, kv_seq_len)
            if done is not None:
                return done
        self._st = None
        kq, k_full, ks, kz, vq, v_full, vs, vz, _ = past_key_value
        R = self.residual_length
        k_full = key_states if k_full is None else torch.cat((k_full, key_states), dim=2)
        v_full = value_states if v_full is None else torch.cat((v_full, value_states), dim=2)

        if attention_mask is None and query_states.is_cuda and self.head_dim == query_states.shape[-1]:
            attn_weights, attn_output = self._attend(query_states, kq, ks, kz, k_full, vq, vs, vz, v_full, kv_seq_len)
        else:
            # with a mask: the quantised class and the fp16 tail of each side as fields of the hybrid tuple
            # (positions [0, Tq) are the class -- no index list: it sits at the head of the row --, the tail follows)
            t = [None] * 42
            if kq is not None:
                kb = K_BASE[self.k_bits]
                t[kb], t[kb + 2], t[kb + 3] = kq, ks, kz
            if vq is not None:
                vb = V_BASE[self.v_bits]
                t[vb], t[vb + 2], t[vb + 3] = vq, vs, vz
            t[NEW_K], t[NEW_V], t[41] = k_full, v_full, kv_seq_len
            attn_weights, attn_output = decode_attention(query_states, tuple(t), attention_mask, kv_seq_len,
                                                         zero_init=False, memo=self._memo)

        if k_full.shape[-2] == R:   # a full block of fp16 keys: quantise it per channel, straight from its rows
            c, s, z = uniform_group_quantize_pack_last_dim(k_full.transpose(2, 3), self.group_size, self.k_bits)
            k_full = None
            kq = c if kq is None else torch.cat((kq, c), dim=3)
            ks = s if ks is None else torch.cat((ks, s), dim=3)
            kz = z if kz is None else torch.cat((kz, z), dim=3)
        if v_full.shape[-2] > R:    # the oldest fp16 value row leaves the tail
            c, s, z = uniform_group_quantize_pack_last_dim(v_full[:, :, :1, :].contiguous(), self.group_size,
                                                           self.v_bits)
            v_full = v_full[:, :, 1:, :].contiguous()
            vq = c if vq is None else torch.cat((vq, c), dim=2)
            vs = s if vs is None else torch.cat((vs, s), dim=2)
            vz = z if vz is None else torch.cat((vz, z), dim=2)
        return attn_output, attn_weights, (kq, k_full, ks, kz, vq, v_full, vs, vz, kv_seq_len)

    __call__ = forward
