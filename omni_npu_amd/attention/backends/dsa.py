"""DSA (sparse MLA) attention backend for MI355X behind the reference's vLLM plugin contract.

Mirrors src/omni_npu/attention/backends/dsa.py.  Vendor ops replaced:
  npu_scatter_nd_update_ x2 (dsa.py:359-362)          -> kernels.cache_write
  npu_lightning_indexer (patch_dsv32_indexer.py:133-146,
                         v1/layers/attention/npu_dsa.py:92-103)  -> LightningIndexer: quant + fp8 score MFMA + exact top-k
  npu_sparse_flash_attention (dsa.py:259-291)         -> kernels.build_sparse_rows + kernels.sparse_decode
The third cache tensor holds the indexer keys.  The reference keeps them in bf16; here the same bytes hold float8_e4m3fn
keys and one fp32 scale per key, per page: [page*128 B keys | page*4 B scales | unused], see indexer_cache_views().
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import ClassVar, Optional, Tuple

import torch

from ... import _host
from ... import kernels as K
from .mla import HalfUpProjection, _caller_wrote_cache, _is_its_weight, _persistent_int32
from ..._vllm_compat import (PAD_SLOT_ID, AttentionCGSupport, AttentionType, MLACommonBackend, MLACommonBaseImpl,
                             MLACommonDecodeMetadata, MLACommonMetadata, MLACommonMetadataBuilder,
                             MLACommonPrefillMetadata, QueryLenSupport, get_current_vllm_config)

INDEX_HEAD_DIM = 128
def masked_pairs_per_pick(num_heads: int) -> float:
    """Up to how many visible (token, key) pairs per picked one prompts attend over up-projected keys under a mask of the picks
    instead of gathering the picked latents.

    Scores and values of a pair and head cost 640 flops on up-projected keys and 2176 on latents (the up-projection costs what
    absorbing the queries and up-projecting the outputs does), and the latents have to be gathered per token whatever the heads
    are: a share of the gather that goes with the heads, and one that does not.  Measured with k = 2048, one prompt, bf16 keys, ms
    of selection and attention masked / gathered (visible pairs per pick): 128 heads 4.1 / 6.5 (2.3), 9.5 / 10.9 (3.3),
    12.5 / 12.7 (3.8), 16.0 / 15.0 (4.3); 64 heads 9.3 / 12.1 (4.3), 17.0 / 17.7 (5.8), 19.9 / 19.5 (6.3); 32 heads 22.0 / 26.8
    (8.3), 33.9 / 36.1 (10.3), 47.4 / 46.3 (12.3); 16 heads 15.4 / 32.8 (8.3), 56.7 / 81.4 (16.3, the longest prompt a step
    holds).  They meet at 3.95, 6.1 and 11.5 pairs; the line stays below them."""
    return 1.7 + 269.0 / num_heads


def indexer_cache_views(index_cache: torch.Tensor):
    """(k8 [nblk, page, 128] float8 view, k_scale [nblk, page] fp32 view) of the third cache tensor
    ([nblk, page, 1, 128] in a 2-byte dtype, reference dsa.py:67)."""
    nblk, page = index_cache.shape[0], index_cache.shape[1]
    raw = index_cache.reshape(nblk, -1).view(torch.uint8)                    # [nblk, page*256]
    k8 = raw[:, : page * INDEX_HEAD_DIM].view(nblk, page, INDEX_HEAD_DIM)
    ks = raw[:, page * INDEX_HEAD_DIM: page * (INDEX_HEAD_DIM + 4)].view(torch.float32)
    return k8, ks


# In the place of pick bits between the selection and the attention behind it: the prompts are no longer than the selection, every token
# attends over all the keys it sees
EVERY_KEY = "every key"


def _mask_words(stride: int) -> int:
    """32-bit words of a row of pick bits over ``stride`` scores: whole 64-key tiles."""
    return stride // 64 * 2 + 2


class NPUDSABackend(MLACommonBackend):
    @staticmethod
    def get_name() -> str:
        return "NPUDSA"

    @staticmethod
    def get_metadata_cls() -> type["NPUDSAMetadata"]:
        return NPUDSAMetadata

    @staticmethod
    def get_builder_cls() -> type["NPUDSAMetadataBuilder"]:
        return NPUDSAMetadataBuilder

    @staticmethod
    def get_impl_cls() -> type["NPUDSAImpl"]:
        return NPUDSAImpl

    @staticmethod
    def reshape_kv_cache(raw_tensor: torch.Tensor, num_blocks: int, block_size: int, num_kv_heads: int, head_size: int,
                         dtype: torch.dtype = torch.bfloat16) -> Tuple[torch.Tensor, ...]:
        """Three contiguous tensors out of one raw allocation (reference dsa.py:58-73)."""
        raw_tensor = raw_tensor.view(dtype=dtype)
        shapes = [(num_blocks, block_size, 1, 512), (num_blocks, block_size, 1, 64), (num_blocks, block_size, 1, 128)]
        sizes = [math.prod(shape) for shape in shapes]
        if raw_tensor.numel() != sum(sizes):
            raise RuntimeError(f"Raw tensor has {raw_tensor.numel()} elements, while"
                               f" the expected sizes for KV cache are {sizes}.")
        tensors = torch.split(raw_tensor, sizes)
        return tuple(t.view(shape) for t, shape in zip(tensors, shapes))


@dataclass
class NPUDSAPrefillMetadata(MLACommonPrefillMetadata):
    query_cumlens: torch.Tensor = None
    seq_lens: torch.Tensor = None
    # prompt lengths on the host, where every prefill request starts at its first token (else None)
    prompt_lens: list = None

    def over_up_projected(self, k: int, pairs_per_pick: float) -> bool:
        """Whether the prefill attends over up-projected keys and values with a mask of the k picks instead of gathering
        the picked latents: while there are at most ``pairs_per_pick`` visible (token, key) pairs per picked one."""
        if self.prompt_lens is None or not pairs_per_pick:
            return False
        seen = sum(n * (n + 1) // 2 for n in self.prompt_lens)
        picked = sum(n * (n + 1) // 2 if n <= k else k * (k + 1) // 2 + (n - k) * k for n in self.prompt_lens)
        return seen <= pairs_per_pick * picked


@dataclass
class NPUDSADecodeMetadata(MLACommonDecodeMetadata):
    query_cumlens: torch.Tensor = None
    query_start_loc: torch.Tensor = None
    q_len: int = 1
    mc2_mask: torch.Tensor = None


@dataclass
class NPUDSAMetadata(MLACommonMetadata[NPUDSADecodeMetadata]):
    pass


class NPUDSAMetadataBuilder(MLACommonMetadataBuilder[NPUDSAMetadata]):
    _cudagraph_support: ClassVar[AttentionCGSupport] = AttentionCGSupport.UNIFORM_BATCH
    query_len_support: ClassVar[QueryLenSupport] = QueryLenSupport.VARLEN

    def __init__(self, kv_cache_spec, layer_names, vllm_config, device):
        super().__init__(kv_cache_spec, layer_names, vllm_config, device, NPUDSAMetadata)
        self.prefill_metadata_cls = NPUDSAPrefillMetadata
        if self._use_fi_prefill:
            raise ValueError("Flashinfer should not be enabled.")
        if self._use_cudnn_prefill:
            raise ValueError("CUDNN should not be enabled.")
        if self.dcp_world_size > 1:
            raise ValueError("DCP should not be enabled.")
        if self.aot_schedule:
            raise ValueError("AOT schedule should be enabled.")
        spec = getattr(vllm_config, "speculative_config", None)
        self.uniform_decode_query_len = 1 if not spec else 1 + spec.num_speculative_tokens
        if self.compilation_config is not None:
            cap = getattr(self.compilation_config, "max_cudagraph_capture_size", None) or 0
            self.reorder_batch_threshold = max(cap, self.reorder_batch_threshold, self.uniform_decode_query_len)

    def _build_decode(self, block_table_tensor, seq_lens_cpu, seq_lens_device, query_start_loc_cpu,
                      query_start_loc_device, num_decode_tokens, dcp_tot_seq_lens_device) -> NPUDSADecodeMetadata:
        qlens = query_start_loc_cpu[1:] - query_start_loc_cpu[:-1]
        n = qlens.numel()
        max_q = int(qlens.max()) if n else 1
        uniform = n > 0 and int(qlens.min()) == max_q
        return NPUDSADecodeMetadata(block_table=block_table_tensor, seq_lens=_persistent_int32(self, "_seq_lens_i32", seq_lens_device),
                                    dcp_tot_seq_lens=dcp_tot_seq_lens_device, query_cumlens=query_start_loc_device[1:],
                                    query_start_loc=None if uniform else query_start_loc_device.to(torch.int32).contiguous(),
                                    q_len=max_q)

    def build(self, common_prefix_len: int, common_attn_metadata, fast_build: bool = False) -> NPUDSAMetadata:
        metadata = super().build(common_prefix_len, common_attn_metadata, fast_build)
        if metadata.decode is not None and getattr(self.vllm_config, "kv_transfer_config", None) is not None:
            metadata.slot_mapping = self._align_slot_mapping(metadata.slot_mapping, metadata.num_reqs)
        if metadata.prefill is not None:
            qsl = metadata.prefill.query_start_loc
            metadata.prefill.seq_lens = qsl[1:] - qsl[:-1]
            metadata.prefill.query_cumlens = torch.cumsum(qsl[1:] - qsl[:-1], dim=0)
            # sparse attention over the cache needs each prefill request's total cached length
            nd = metadata.num_decodes
            metadata.prefill.kv_lens = common_attn_metadata.seq_lens[nd:].to(torch.int32)
            done = getattr(common_attn_metadata, "num_computed_tokens_cpu", None)
            if done is not None and not bool((done[nd:nd + metadata.num_prefills] > 0).any()):
                starts = common_attn_metadata.query_start_loc_cpu[nd:nd + metadata.num_prefills + 1]
                metadata.prefill.prompt_lens = (starts[1:] - starts[:-1]).tolist()
        if metadata.prefill is not None and metadata.prefill.chunked_context is not None:
            raise RuntimeError("Chunked prefill is not enabled yet.")
        return metadata

    def _align_slot_mapping(self, slot_mapping: torch.Tensor, num_reqs) -> torch.Tensor:
        num_tokens_padded = num_reqs * self.uniform_decode_query_len
        if slot_mapping.numel() < num_tokens_padded:
            slot_mapping = torch.nn.functional.pad(slot_mapping, (0, num_tokens_padded - slot_mapping.numel()),
                                                   value=PAD_SLOT_ID)
        return slot_mapping


class LightningIndexer:
    """The selection step of the DeepSeek-V3.2 indexer on the GPU: quantise q, quantise-and-cache the new keys, fp8
    score GEMM, exact top-k into ``topk_indices_buffer`` (the tail of the reference's patched Indexer.forward,
    patch_dsv32_indexer.py:104-146; the projections, LayerNorm and RoPE before it are the caller's)."""

    def __init__(self, topk_tokens: int, n_head: int = 64, head_dim: int = INDEX_HEAD_DIM, max_tokens: int = 1,
                 device=None):
        self.topk_tokens, self.n_head, self.head_dim = topk_tokens, n_head, head_dim
        self.topk_indices_buffer = torch.full((max_tokens, topk_tokens), -1, dtype=torch.int32, device=device)
        # what the sparse attention reads: the picks as flat cache rows and their number per token, written by the same
        # launch that writes the positions (the block ids of the three DSA cache tensors are the same)
        self.rows_buffer = torch.zeros((max_tokens, topk_tokens), dtype=torch.int32, device=device)
        self.counts_buffer = torch.zeros((max_tokens,), dtype=torch.int32, device=device)
        self._rows_meta = None       # the metadata object the row buffers were filled for
        # Up to how many visible pairs per pick the attention behind this selection wants a step's prompts as bits over their
        # own keys instead of cache rows (NPUDSAImpl says so once its weights are loaded); the bits, until the attention has
        # used them (drop_mask), and the metadata object they were made for
        self.masked_pairs_per_pick = 0.0
        self._mask, self._mask_meta = None, None
        self._mask_shape = (0, 0)    # of the bits that EVERY_KEY stands for
        self._logits = None
        self._logits_kept = []       # outgrown score buffers: a captured graph may still hold their address, never freed

    def __call__(self, q: torch.Tensor, k: torch.Tensor, weights: torch.Tensor, kv_cache, attn_metadata):
        if attn_metadata is None:                                   # profile run (patch_dsv32_indexer.py:104-112)
            return self.topk_indices_buffer
        assert len(kv_cache) >= 3, f"Expected kv_cache to have at least 3 elements, but got {len(kv_cache)}"
        t = q.shape[0]
        if attn_metadata.num_prefills == 0 and attn_metadata.num_decodes > 0 and self._native_select(q, k, weights, kv_cache[2],
                                                                                                     attn_metadata):
            return self.topk_indices_buffer[:t].view(t, 1, self.topk_tokens)
        p = attn_metadata.prefill if attn_metadata.num_prefills > 0 else None
        masked = (p is not None and self.masked_pairs_per_pick > 0
                  and p.over_up_projected(self.topk_tokens, self.masked_pairs_per_pick))
        # (prompts no longer than the selection: every token takes all the keys it sees)
        whole = masked and p.max_query_len <= self.topk_tokens
        if masked and attn_metadata.num_decodes == 0 and self._native_select_prompts(q, k, weights, kv_cache[2], attn_metadata, whole):
            return self.topk_indices_buffer[:t].view(t, 1, self.topk_tokens)
        k8, ks = indexer_cache_views(kv_cache[2])
        # the new keys into the cache and the queries that are scored into plain buffers: one launch
        if p is not None and self.n_head % 64 == 0:
            ndt = attn_metadata.num_decode_tokens if attn_metadata.num_decodes > 0 else 0
            p_qsl = p.query_start_loc.to(torch.int32).contiguous()
            q8, w = K.quant_qkw_fp8_above(q.reshape(t, self.n_head, self.head_dim), weights, ndt if whole else t,
                                          k.reshape(-1, self.head_dim), k8, ks, attn_metadata.slot_mapping, p_qsl,
                                          p.kv_lens.contiguous(), p.max_query_len, ndt, self.topk_tokens)
            qs = None
        else:
            q8 = torch.empty(t, self.n_head, self.head_dim, dtype=torch.uint8, device=q.device)
            qs = torch.empty(t, self.n_head, dtype=torch.float32, device=q.device)
            K.quant_qk_fp8(q.reshape(t * self.n_head, self.head_dim), q8, qs, k.reshape(-1, self.head_dim), k8, ks,
                           attn_metadata.slot_mapping)
            w = weights.float().contiguous()
        out = self.topk_indices_buffer[:t]
        off = 0
        self._rows_meta = self._mask_meta = self._mask = None
        for meta, nreq in ((attn_metadata.decode, attn_metadata.num_decodes), (attn_metadata.prefill, attn_metadata.num_prefills)):
            if meta is None or nreq == 0:
                continue
            if meta is attn_metadata.decode:
                ntok, lens, q_len, qsl = attn_metadata.num_decode_tokens, meta.seq_lens, meta.q_len, meta.query_start_loc
            else:
                ntok = t - off
                lens, q_len = meta.kv_lens, meta.max_query_len
                qsl = meta.query_start_loc.to(torch.int32).contiguous()
            over_own = masked and meta is p
            max_len = meta.block_table.shape[1] * k8.shape[1]
            if over_own:                                            # (the longest prompt, not the longest the server takes)
                max_len = min(max_len, (q_len + 63) // 64 * 64)
            stride = K.indexer_logits_stride(max_len)
            lg = (self._no_scores if over_own and whole else self._scores_buffer)(ntok, stride, q.device)
            sl = slice(off, off + ntok)
            if not (over_own and whole):
                K.indexer_scores(q8[sl], w[sl], k8, ks, meta.block_table, lens, lg, q_len=q_len, q_scale=None if qs is None else qs[sl],
                                 query_start_loc=qsl, max_seq_len=max_len, skip_up_to=self.topk_tokens)
            if over_own:
                self._mask_meta, self._mask_shape = attn_metadata, (ntok, _mask_words(stride))
                self._mask = EVERY_KEY if whole else torch.empty(self._mask_shape, dtype=torch.int32, device=q.device)
                K.topk(lg, lens, self.topk_tokens, out[sl], q_len=q_len, query_start_loc=qsl, mask=None if whole else self._mask)
            else:
                K.topk(lg, lens, self.topk_tokens, out[sl], q_len=q_len, query_start_loc=qsl, block_table=meta.block_table,
                       page_size=k8.shape[1], num_pages=k8.shape[0], rows=self.rows_buffer[sl],
                       counts=self.counts_buffer[sl])
                self._rows_meta = attn_metadata
            off += ntok
        return out.view(t, 1, self.topk_tokens)

    def _scores_buffer(self, ntok: int, stride: int, device) -> torch.Tensor:
        if self._logits is None or self._logits.shape[0] < ntok or self._logits.shape[1] < stride:
            rows, cols = max(ntok, 1), stride
            if self._logits is not None:
                self._logits_kept.append(self._logits)
                rows, cols = max(rows, self._logits.shape[0]), max(cols, self._logits.shape[1])
            self._logits = torch.empty(rows, cols, dtype=torch.float32, device=device)
        return self._logits[:ntok, :stride]

    @staticmethod
    def _no_scores(ntok: int, stride: int, device) -> torch.Tensor:
        """In the place of scores where every token takes all of its keys: rows as wide as these prompts, by which the kernel is chosen and
        which none of them reads, given back behind the step."""
        return torch.empty(ntok, stride, dtype=torch.float32, device=device)

    def _native_select(self, q, k, weights, index_cache, attn_metadata) -> bool:
        """The selection of a step of decode tokens in one native call; False, with nothing done, where that call does not
        know the case."""
        d, ntok = attn_metadata.decode, attn_metadata.num_decode_tokens
        if not q.is_cuda or self.n_head != 64 or self.head_dim != INDEX_HEAD_DIM or q.dim() != 3:
            return False
        max_len = d.block_table.shape[1] * index_cache.shape[1]
        lg = self._scores_buffer(ntok, K.indexer_logits_stride(max_len), q.device)
        self._rows_meta = self._mask_meta = self._mask = None
        if not _host.load().dsa_select(q, k, weights, index_cache, attn_metadata.slot_mapping, d.block_table, d.seq_lens,
                                       d.query_start_loc, ntok, d.q_len, max_len, self.topk_tokens, lg,
                                       self.topk_indices_buffer, self.rows_buffer, self.counts_buffer):
            return False
        self._rows_meta = attn_metadata
        return True

    def _native_select_prompts(self, q, k, weights, index_cache, attn_metadata, whole: bool) -> bool:
        """The selection of a step of masked prompts in one native call; False, with nothing done, where that call does not know the
        case."""
        t, p = q.shape[0], attn_metadata.prefill
        if not q.is_cuda or self.n_head != 64 or self.head_dim != INDEX_HEAD_DIM or q.dim() != 3:
            return False
        max_len = min(p.block_table.shape[1] * index_cache.shape[1], (p.max_query_len + 63) // 64 * 64)
        stride = K.indexer_logits_stride(max_len)
        lg, mask = (self._no_scores if whole else self._scores_buffer)(t, stride, q.device), None
        if not whole:
            mask = torch.empty(t, _mask_words(stride), dtype=torch.int32, device=q.device)
        self._rows_meta = self._mask_meta = self._mask = None
        if not _host.load().dsa_select_prompts(q, k, weights, index_cache, attn_metadata.slot_mapping, p.block_table, p.kv_lens,
                                               p.query_start_loc, p.max_query_len, max_len, self.topk_tokens, whole, lg,
                                               self.topk_indices_buffer, mask):
            return False
        self._mask_meta, self._mask, self._mask_shape = attn_metadata, EVERY_KEY if whole else mask, (t, _mask_words(stride))
        return True

    def picks_for(self, attn_metadata):
        """What NPUDSAImpl._forward_prompts takes: mask_for's bits, EVERY_KEY where they would all be set, or None."""
        return self._mask if self.masked_prompts(attn_metadata) else None

    def mask_for(self, attn_metadata) -> Optional[torch.Tensor]:
        """The picks of the step's prompt tokens as bits [T, W] (kernels.topk's mask) if the last selection made them for this very
        metadata object and the attention has not used them yet, else None."""
        picks = self.picks_for(attn_metadata)
        if picks is EVERY_KEY:
            return torch.full(self._mask_shape, -1, dtype=torch.int32, device=self.topk_indices_buffer.device)
        return picks

    def masked_prompts(self, attn_metadata) -> bool:
        """Whether the last selection ran for this very metadata object and made its prompts' picks as bits: the row buffers
        then hold the step's decode tokens only."""
        return attn_metadata is not None and self._mask_meta is attn_metadata

    def drop_mask(self) -> None:
        """The attention has queued its use of the bits: their memory (a bit per pair of a prompt, 8 MB for 8k tokens) goes back
        behind it instead of staying with every layer until that layer's next step."""
        if isinstance(self._mask, torch.Tensor) and self._mask.is_cuda:
            self._mask.record_stream(torch.cuda.current_stream(self._mask.device))
        self._mask = None

    def rows_for(self, attn_metadata):
        """(cache rows [max_tokens, k], counts [max_tokens]) of the picks if the last selection ran for this very metadata
        object, else None (the caller then translates ``topk_indices_buffer`` itself)."""
        if attn_metadata is not None and self._rows_meta is attn_metadata:
            return self.rows_buffer, self.counts_buffer
        return None


class NPUDSAImpl(HalfUpProjection, MLACommonBaseImpl[NPUDSAMetadata]):
    can_return_lse_for_decode: bool = False
    cache_written_for = None     # see NPUMLAImpl.cache_written_for
    # Prompts attend in the types that a gather of the cache would: bf16 latents, rope rows, queries and keys.  True makes keys and
    # rope rows fp16 (11 bits instead of 8, at the same speed) for a model whose rope rows, queries, keys and values stay between
    # 2^-14 and 65504.
    prefill_kv_fp16 = False
    # (masked prompts are offered for a plain weight only, whose product W_UK and W_UV stand for everywhere else; a layer with an adapter
    # or hooks is called)
    keys_bf16_values_f16 = True

    def __init__(self, num_heads: int, head_size: int, scale: float, num_kv_heads: int, alibi_slopes: Optional[list],
                 sliding_window: Optional[int], kv_cache_dtype: str, logits_soft_cap: Optional[float], attn_type: str,
                 kv_sharing_target_layer_name: Optional[str], **mla_args) -> None:
        super().__init__(num_heads, head_size, scale, num_kv_heads, alibi_slopes, sliding_window, kv_cache_dtype,
                         logits_soft_cap, attn_type, kv_sharing_target_layer_name, **mla_args)
        cfg = get_current_vllm_config()
        self.chunked_prefill_workspace_size = (
            MLACommonMetadataBuilder.determine_chunked_prefill_workspace_size(cfg) if cfg is not None else 0)
        unsupported_features = [alibi_slopes, sliding_window, logits_soft_cap]
        if any(unsupported_features):
            raise NotImplementedError(
                "NPUDSAImpl does not support one of the following: "
                "alibi_slopes, sliding_window, logits_soft_cap")
        if attn_type != AttentionType.DECODER:
            raise NotImplementedError(
                "Encoder self-attention and "
                "encoder/decoder cross-attention "
                "are not implemented for "
                "NPUDSAImpl")
        if kv_cache_dtype in ("fp8", "fp8_e4m3"):
            raise NotImplementedError("NPUDSAImpl writes the bf16 cache layout (latent, rope, indexer keys) only: "
                                      "an fp8 KV cache is not supported for DSA models")

    def process_weights_after_loading(self, act_dtype: torch.dtype):
        super().process_weights_after_loading(act_dtype)
        self.offer_masked_prompts(getattr(self.indexer, "select", self.indexer))

    def offer_masked_prompts(self, select) -> None:
        """Tells the selection whether, and for how many pairs per pick, this layer attends over masked prompts."""
        if hasattr(select, "masked_pairs_per_pick"):
            select.masked_pairs_per_pick = masked_pairs_per_pick(self.num_heads) if self._plain_up_weight() is not None else 0.0

    def _v_up_proj(self, x: torch.Tensor, out: torch.Tensor):
        """[T,N,512] token-major -> out [T, N*V]  (reference dsa.py:233-240)."""
        x = x.transpose(0, 1)
        out2 = torch.bmm(x, self.W_UV)
        out.copy_(out2.transpose(0, 1).reshape(-1, self.num_heads * self.v_head_dim))

    def _absorb_prolog(self, q: torch.Tensor):
        q_nope, q_pe = q.split([self.qk_nope_head_dim, self.qk_rope_head_dim], dim=-1)
        ql_nope = K.absorb(q_nope, self.W_UK_T)
        return ql_nope, q_pe

    def _fusable_w_uv(self, out: torch.Tensor) -> bool:
        """The fused merge + up-projection kernel takes bf16 W_UV [N,512,128] with contiguous rows and writes rows of 128."""
        w = self.W_UV
        return (w.dtype == torch.bfloat16 and w.dim() == 3 and w.shape[1:] == (512, 128) and w.stride(2) == 1
                and w.stride(0) % 8 == 0 and w.stride(1) % 8 == 0 and w.data_ptr() % 16 == 0
                and out.dtype == torch.bfloat16 and out.stride(-1) == 1 and out.stride(0) % 4 == 0 and out.data_ptr() % 8 == 0)

    def _apply_sparse_attention(self, q_nope, q_pe, kv_cache, meta, lens, q_len, qsl, topk_indices,
                                proj_out: Optional[torch.Tensor] = None, rows_counts=None) -> Optional[torch.Tensor]:
        """Absorbed MLA over the indexer's positions (reference dsa.py:259-291); token-major [T,N,512].  With
        ``proj_out`` ([T, N*V]) the value up-projection (dsa.py:233-240) is fused into the merge of the partials and
        nothing is returned.  ``rows_counts``: the picks of these tokens already translated into cache rows, with their
        counts (LightningIndexer.rows_for); without it the positions are translated here."""
        bs = q_nope.shape[0]
        k = topk_indices.shape[-1]
        nope, rope = kv_cache[0], kv_cache[1]
        if rows_counts is not None:
            rows, counts = rows_counts
        else:
            rows = torch.empty(bs, k, dtype=torch.int32, device=q_nope.device)
            counts = torch.empty(bs, dtype=torch.int32, device=q_nope.device)
            K.build_sparse_rows(topk_indices.reshape(bs, k), meta.block_table, lens, nope.shape[1], nope.shape[0], rows,
                                counts, q_len=q_len, query_start_loc=qsl)
        if proj_out is not None:
            K.sparse_decode(q_nope, q_pe, nope, rope, rows, counts, self.scale, proj_out, w_uv=self.W_UV, counts_bounded=True)
            return None
        out = torch.empty(bs, self.num_heads, self.kv_lora_rank, dtype=q_nope.dtype, device=q_nope.device)
        K.sparse_decode(q_nope, q_pe, nope, rope, rows, counts, self.scale, out, counts_bounded=True)
        return out

    def _forward_prompts(self, q, kv_c_normed, k_pe, prefill, pick, out: torch.Tensor) -> bool:
        """Sparse attention of whole prompts over their own up-projected keys and values, with the picks as a mask
        (NPUDSAPrefillMetadata.over_up_projected); False, and nothing done, where the shapes do not allow it."""
        t, n, w = q.shape[0], self.num_heads, self._plain_up_weight()
        bf16 = torch.bfloat16
        if pick is None or w is None or not (w.dtype == bf16 or self.prefill_kv_fp16) or self.qk_nope_head_dim != 128 or \
                self.v_head_dim != 128 or not (q.dtype == kv_c_normed.dtype == k_pe.dtype == out.dtype == bf16) or \
                q.stride(-1) != 1 or kv_c_normed.stride(-1) != 1 or k_pe.stride(-1) != 1 or out.stride(-1) != 1 or \
                tuple(out.shape) != (t, n * 128) or (q.stride(0) | q.stride(1) | k_pe.stride(0) | out.stride(0)) % 8 or \
                (q.data_ptr() | k_pe.data_ptr() | out.data_ptr()) % 16:
            return False
        bits = None if pick is EVERY_KEY else pick
        if (self.prefill_kv_fp16 or (self.keys_bf16_values_f16 and _is_its_weight(self.kv_b_proj))) and _host.load().prefill(
                q, kv_c_normed, k_pe, 0, t, prefill.query_start_loc, prefill.max_query_len, w, self.prefill_kv_fp16, self.scale, out,
                bits, None, None, None, None, None, None, 0):
            return True
        cu = prefill.query_start_loc.to(torch.int32).contiguous()
        queue = K.prefill_queue(t, cu.numel() - 1, prefill.max_query_len, n, q.device)
        k_nope, pe, v, _ = self._kv_up_rows(kv_c_normed, k_pe, queue)
        K.prefill_varlen(q[..., :128], q[..., 128:], k_nope, pe, v, cu, cu, prefill.max_query_len, self.scale, True,
                         out.view(t, n, 128), pick=bits, queue=queue)
        return True

    def forward(self, layer, q: torch.Tensor, k_c_normed: torch.Tensor, k_pe: torch.Tensor,
                kv_cache: Tuple[torch.Tensor, torch.Tensor, torch.Tensor], attn_metadata: NPUDSAMetadata,
                output: Optional[torch.Tensor] = None, output_scale: Optional[torch.Tensor] = None,
                output_block_scale: Optional[torch.Tensor] = None) -> torch.Tensor:
        assert output is not None, "Output tensor must be provided."
        if output_scale is not None or output_block_scale is not None:
            raise NotImplementedError("fused output quantization is not yet supported for NPUDSAImpl")
        if attn_metadata is None:
            # (beside the up-projection scratch what a step of masked prompts makes and drops again: the fp16 weight, and the
            # picks of one prompt of all the step's tokens as bits)
            toks = max(int(k_c_normed.shape[0]), 1)
            _ = (torch.empty((self.chunked_prefill_workspace_size, self.num_heads,
                              self.qk_nope_head_dim + self.v_head_dim), device=k_c_normed.device, dtype=k_c_normed.dtype),
                 self._half_up_weight(),
                 torch.empty(toks, _mask_words(K.indexer_logits_stride(toks)), dtype=torch.int32, device=k_c_normed.device))
            # the profile run sizes the KV cache: the split-KV scratch a real prefill will need (bounded by
            # SPARSE_WORKSPACE_CAP whatever the chunk size) is allocated now, so that it is counted
            # (for the split count the real steps will pick; scratch is kept per stream, so a runner that captures its graphs
            # on another stream pays this once more there: at most SPARSE_WORKSPACE_CAP per stream that runs steps)
            if k_c_normed.is_cuda:
                k_sel = int(self.indexer.topk_indices_buffer.shape[-1]) if self.indexer is not None else 2048
                splits = K.launch_splits(toks, 1, self.num_heads, k_sel, full=True)
                need = K._lib.load().mla_decode_workspace_bytes(min(toks, 32768), 1, self.num_heads, splits)
                K._workspace(k_c_normed.device, min(need, K.SPARSE_WORKSPACE_CAP))
            return output.fill_(0)

        num_actual_toks = attn_metadata.num_actual_tokens
        assert isinstance(kv_cache, (list, tuple)), f"{type(kv_cache)=}."
        assert len(kv_cache) == 3, f"{len(kv_cache)=}."
        k_nope, k_rope, _ = kv_cache
        assert isinstance(k_nope, torch.Tensor) and isinstance(k_rope, torch.Tensor), f"{type(k_nope)=}, {type(k_rope)=}."
        assert k_nope.numel() > 0 and k_rope.numel() > 0, f"{k_nope.shape=}, {k_rope.shape=}"

        output_padded = output
        output = output[:num_actual_toks, ...]
        q = q[:num_actual_toks, ...]
        assert (attn_metadata.num_decodes is not None and attn_metadata.num_prefills is not None
                and attn_metadata.num_decode_tokens is not None)
        has_decode = attn_metadata.num_decodes > 0
        has_prefill = attn_metadata.num_prefills > 0
        ndt = attn_metadata.num_decode_tokens
        written = _caller_wrote_cache(self, attn_metadata, num_actual_toks)
        select = getattr(self.indexer, "select", self.indexer)     # (what was offered masked prompts, see there)
        rc = select.rows_for(attn_metadata) if hasattr(select, "rows_for") else None
        native = None
        if has_decode and not has_prefill and rc is not None:
            native = lambda *new: _host.load().sparse_decode(q, k_nope, k_rope, rc[0], rc[1], self.W_UK_T, self.W_UV, self.scale,
                                                             ndt, output, *new)
        if written:                                                # (the caller's fused norm + rope launch wrote the rows)
            if native is not None and native(None, None, None):
                return output_padded
        elif K.cache_write(k_c_normed, k_pe, attn_metadata.slot_mapping, k_nope, k_rope, along=native):
            return output_padded
        topk = self.indexer.topk_indices_buffer
        part = lambda a, b: None if rc is None else (rc[0][a:b], rc[1][a:b])
        # (a selection that made bits has left no rows for the prompts, also after the bits are gone)
        masked = hasattr(select, "masked_prompts") and select.masked_prompts(attn_metadata)

        if has_prefill:
            p = attn_metadata.prefill
            assert p is not None
            pick = getattr(select, "picks_for", select.mask_for)(attn_metadata) if masked else None
            if not self._forward_prompts(q[ndt:], k_c_normed[ndt:num_actual_toks], k_pe[ndt:num_actual_toks], p, pick,
                                         output[ndt:]):
                q_nope, q_pe = self._absorb_prolog(q[ndt:])
                fused = output[ndt:] if self._fusable_w_uv(output[ndt:]) else None
                attn_out = self._apply_sparse_attention(q_nope, q_pe, kv_cache, p, p.kv_lens, p.max_query_len,
                                                        p.query_start_loc.to(torch.int32).contiguous(),
                                                        topk[ndt:num_actual_toks], proj_out=fused,
                                                        rows_counts=None if masked else part(ndt, num_actual_toks))
                if fused is None:
                    self._v_up_proj(attn_out, out=output[ndt:])
            if pick is not None:
                select.drop_mask()
        if has_decode:
            d = attn_metadata.decode
            assert d is not None
            q_nope, q_pe = self._absorb_prolog(q[:ndt])
            fused = output[:ndt] if self._fusable_w_uv(output[:ndt]) else None
            attn_out = self._apply_sparse_attention(q_nope, q_pe, kv_cache, d, d.seq_lens, d.q_len, d.query_start_loc,
                                                    topk[:ndt], proj_out=fused, rows_counts=part(0, ndt))
            if fused is None:
                self._v_up_proj(attn_out, out=output[:ndt])
        return output_padded
